"""interactions_monaghan's choice between the in-support pairs and the reference's full 5x5-cell
window: the sums equal the oracle's bit for bit, with finite inputs and with a NaN, an infinity or a
zero density among them (which spread to every particle whose window holds them), in any order of
calls on one context, for particle counts around the workgroup size and growing workspaces."""
import ctypes as C

import numpy as np
import pytest

from helpers import assert_equal
from oracle.oracle import Oracle
from sph_fem_2d_cutting_gpu_amd import cases
from sph_fem_2d_cutting_gpu_amd import solver as S

pytestmark = pytest.mark.gpu

OUT = ("v_der", "S_der", "vel_t", "pos_t", "T_t")
STATE = ("pos", "vel", "rho", "S", "R", "p", "T", "h", "hash", "blanked", "tool_particle") + OUT


def _sorted(nx, ny):
    o = Oracle(cases.perturbed(cases.small_cutting_case(nx=nx, ny=ny, tool_tris=400)))
    o.call("o_compute_hashes", "cp")
    o.call("o_sort_and_cells", "cps")
    o.call("o_material_eos", "cp")
    o.call("o_artificial_stress", "cp")
    return o


@pytest.mark.parametrize("nx,ny", [(17, 15), (32, 8), (257, 9), (48, 16)])
def test_window_switch(nx, ny):
    o = _sorted(nx, ny)
    sim = S.Simulation(o.case)
    n, nc = o.case.N, len(o.st["cell_start"])
    cells = [C.c_void_p(), C.c_void_p()]
    for q, name in zip(cells, ("cell_start", "cell_end")):
        sim.ctx.call("sphfem_malloc", C.byref(q), 4 * nc)
        sim.ctx.htod(q.value, o.st[name])
    S.interactions_setup_geometry_constants(sim.grid)
    clean = {f: o.P[f].copy() for f in STATE}
    k = n // 2
    for fault in (None, ("S", np.nan), None, ("vel", np.inf), ("rho", 0.0), None):
        for f in STATE:
            o.P[f][...] = clean[f]
        if fault is not None:
            o.P[fault[0]][k] = fault[1]
        print("N", n, "fault", fault, flush=True)
        for f in STATE:
            sim.p.upload(f, o.P[f])
        o.call("o_interactions_monaghan", "cps")
        S.interactions_monaghan(sim.p, cells[0].value, cells[1].value, nc)
        for f in OUT:
            got, want = sim.p.download(f), o.P[f]
            assert_equal(f"{fault} {f} NaN", np.isnan(got), np.isnan(want))
            assert_equal(f"{fault} {f}", np.nan_to_num(got, nan=0.0), np.nan_to_num(want, nan=0.0))
        if fault is not None:
            assert any(np.isnan(o.P[f]).any() for f in OUT)
    for q in cells:
        sim.ctx.call("sphfem_free", q)
    sim.close()
