"""A blanked particle adds nothing to any neighbour's sums, whatever its own position and velocity hold.

A live particle with a NaN velocity leaves its step blanked, with a NaN position, and so does every
particle whose 5x5 cells held it; they keep their cells.  From then on they are skipped
(interactions_gpu.cu:232), so the failure stays where it is."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from helpers import assert_close, assert_equal
from oracle.oracle import Oracle
from sph_fem_2d_cutting_gpu_amd import _lib, cases
from sph_fem_2d_cutting_gpu_amd import solver as S
from test_gpu_interactions_window import OUT, STATE, _sorted

pytestmark = pytest.mark.gpu

BAD = {"nan_x": (np.nan, 0.5), "nan_y": (0.5, np.nan), "nan": (np.nan, np.nan), "inf_x": (np.inf, 0.5),
       "inf_y": (0.5, -np.inf), "mixed": (np.inf, np.nan)}


def test_stage_calls_skip_blanked_particles_anywhere():
    """Every seventh particle blanked, with its position and velocity as they were and then non-finite:
    the other particles' outputs are the same bit for bit, equal to the oracle's in the FP64 call."""
    o = _sorted(48, 16)
    sim = S.Simulation(o.case, precision=_lib.FP32C)
    nc = len(o.st["cell_start"])
    cells = [C.c_void_p(), C.c_void_p()]
    for q, name in zip(cells, ("cell_start", "cell_end")):
        sim.ctx.call("sphfem_malloc", C.byref(q), 4 * nc)
        sim.ctx.htod(q.value, o.st[name])
    S.interactions_setup_geometry_constants(sim.grid)
    o.P["blanked"][3::7] = 1.0
    clean = {f: o.P[f].copy() for f in STATE}
    live = clean["blanked"] != 1.0
    o.call("o_interactions_monaghan", "cps")
    want = {}
    for name, bad in [("finite", None)] + list(BAD.items()):
        for which in ("fp64", "fp32c"):
            for f in STATE:
                a = clean[f].copy()
                if bad is not None and f in ("pos", "vel"):
                    a[~live] = bad
                sim.p.upload(f, a)
            print(name, which, flush=True)
            if which == "fp32c":
                S.interactions_monaghan_fp32c(sim.stepper, sim.p, cells[0].value, cells[1].value, nc)
            else:
                S.interactions_monaghan(sim.p, cells[0].value, cells[1].value, nc)
            for f in OUT:
                got = sim.p.download(f)
                assert np.all(np.isfinite(got[live])), f"{name} {which} {f}"
                if bad is None:
                    want[which, f] = got
                    if which == "fp64":
                        assert_equal(f"{f} against the oracle", got[live], o.P[f][live])
                assert_equal(f"{name} {which} {f}", got[live], want[which, f][live])
    for q in cells:
        sim.ctx.call("sphfem_free", q)
    sim.close()


@pytest.mark.parametrize("which", ["chip", "cutting"])
@pytest.mark.parametrize("prec", [_lib.FP64, _lib.FP32C])
def test_one_nan_velocity_stays_in_its_window(prec, which):
    """Without a tool, and with one (the near-tool pass and the tool's end of the step)."""
    if which == "chip":
        case = cases.chip_case(n_target=800)
        at = np.median(case.pos, axis=0)
    else:
        case = cases.perturbed(cases.small_cutting_case(nx=48, ny=16, wear=True))
        at = np.array([0.0140, 0.0590])
    vel = case.vel.copy()
    vel[int(np.argmin(np.hypot(*(case.pos - at).T)))] = [0.0, np.nan]
    case = dataclasses.replace(case, vel=vel)
    o, sim = Oracle(case), S.Simulation(case, precision=prec)
    for step in range(1, 4):
        print(which, prec, "step", step, flush=True)
        o.step(1)
        sim.step(1)
        sim.ctx.check_error()
        a, b = sim.state(), o.P
        for f in ("hash", "idx", "blanked"):
            assert_equal(f"{f} after {step} steps", a[f], b[f])
        live = b["blanked"] != 1.0
        gone = int((~live).sum())
        print("blanked", gone, flush=True)
        assert np.isnan(b["pos"][~live]).any() and 1 < gone < case.N // 2
        if step == 1:
            first = gone
        assert gone == first
        for f in ("pos", "vel", "S", "rho", "T"):
            assert_close(f"{f} after {step} steps", a[f], b[f], 1e-6, mask=live)
        for f in ("pos_t", "vel_t", "rho_t", "S_t"):
            assert_close(f"{f} after {step} steps", a[f], b[f], 1e-5, mask=live)
    sim.close()
