"""Kernels in which one lane announces its workgroup's results to other workgroups (an agent fence, then a
counter): a workgroup barrier does not wait for the stores that other wavefronts have in flight, and the
lane's fence covers its own wavefront only, so every wavefront must have waited for its stores before the
barrier.  Looked up in the gfx950 assembly of the library's sources."""
import os
import re
import shlex
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sph_fem_2d_cutting_gpu_amd", "csrc")


def _assembly(source, tmp_path):
    plan = subprocess.run(["make", "-C", CSRC, "-n", "-B", f"build/{source}.o"], check=True, capture_output=True, text=True)
    cmd = shlex.split(next(l for l in plan.stdout.splitlines() if f" -c {source} " in l))
    at = cmd.index("-c")
    out = str(tmp_path / "k.s")
    subprocess.run(cmd[:at] + ["--cuda-device-only", "-S", cmd[at + 1], "-o", out], check=True, cwd=CSRC,
                   capture_output=True)
    with open(out) as f:
        return f.read()


def _body(asm, kernel):
    m = re.search(rf"^_ZN6sphfem\d+{kernel}\w*:.*?s_endpgm$", asm, re.S | re.M)
    assert m, f"{kernel} not found"
    return [l.split(";")[0].strip() for l in m.group(0).splitlines()]


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="no hipcc")
@pytest.mark.parametrize("source,kernel,fenced", [("sphfem_sort.hip", "k_resort", False),
                                                  ("sphfem_tool.hip", "k_near_contact", True)])
def test_every_wavefront_waits_for_its_stores(source, kernel, fenced, tmp_path):
    """fenced: plain stores, written back by the announcing lane's fence; else every store that other
    workgroups read is written through (sc1) and the counter is bumped without a fence."""
    lines = _body(_assembly(source, tmp_path), kernel)

    def announces(k):
        if fenced:
            if not lines[k].startswith("buffer_wbl2"):
                return False
            after = next(l for l in lines[k + 1:] if l.startswith(("s_barrier", "buffer_wbl2", "global_atomic", "s_endpgm")))
            return after.startswith("global_atomic_add")   # else the fence of a workgroup that reads others' results
        return lines[k].startswith("global_atomic_add") and "sc0" not in lines[k]       # returns nothing: the counter

    found = [k for k in range(len(lines)) if announces(k)]
    assert len(found) == 1
    b = max(q for q in range(found[0]) if lines[q] == "s_barrier")
    before = next(l for l in reversed(lines[:b])
                  if l.startswith(("global_", "flat_", "buffer_", "s_branch", "s_cbranch", ".LBB")) or "vmcnt(0)" in l)
    assert "vmcnt(0)" in before, f"{kernel}: the barrier before the announcement follows `{before}`, not a wait"
    if not fenced:
        queue = next(k for k, l in enumerate(lines) if l.startswith("global_atomic_add"))       # the first ticket
        stores = [l for l in lines[queue:] if l.startswith("global_store")]
        through = [l for l in stores if "sc1" in l]
        # the keys of pass 0, the counts, and keys and sources of the scatter; the only other store clears cells
        assert len(through) >= 4 and len(stores) - len(through) <= 1, stores
        assert not any(l.startswith("buffer_wbl2") for l in lines)
