"""FP32C pair sums where the fast form's assumptions fail, against the FP64 pair sums of the same state:
particles above and below the grid's rows (their keys name cells of the next or previous column: they
meet only each other), two column heights away, on the grid's edge and clustered near coincidence; kernel
widths other than the cell size (smaller, larger, and wide enough to reach the blanked records' place); a support
that starts at 0; grids of few rows.  One step's derivatives agree within 1e-5 of each field's largest
magnitude, the bound of the ordinary form: the general form does the same FP32 terms in the same blocks."""
import ctypes as C

import numpy as np
import pytest

from helpers import assert_equal
from sph_fem_2d_cutting_gpu_amd import _lib, cases
from sph_fem_2d_cutting_gpu_amd import solver as S
from test_gpu_fp32c import DERIVS, TOL_DERIV, _check, normwise
from test_gpu_interactions_window import OUT, STATE, _sorted

pytestmark = pytest.mark.gpu


def _moved(kind, P, geom):
    """the state's fields with the form's condition planted"""
    pos, h, blanked = P["pos"].copy(), P["h"].copy(), P["blanked"].copy()
    dx, ny = geom.dx, geom.ny
    block = np.argsort(pos[:, 1])[-40:]                 # the top rows: a patch that stays together
    if kind in ("above", "below", "two_heights"):
        pos[block, 1] += {"above": 1, "below": -1, "two_heights": 2}[kind] * ny * dx
        # columns back into the grid's keys
        pos[block, 0] += {"above": -1, "below": 1, "two_heights": -2}[kind] * dx
        sel = pos[block, 0]
        inside = (sel > geom.bbmin_x + 3 * dx) & (sel < geom.bbmin_x + (geom.nx - 3) * dx)
        pos[block[~inside]] = P["pos"][block[~inside]]
    elif kind == "edge":
        pos[block, 1] = geom.bbmin_y + ny * dx + np.linspace(-1.0, 1.9, len(block)) * dx
        pos[block[pos[block, 0] > geom.bbmin_x + (geom.nx - 2) * dx], 0] -= 3 * dx
    elif kind == "narrow":
        h[::3] *= 0.8
    elif kind == "wide":
        h[::5] *= 1.9
        blanked[1::7] = 1.0
    elif kind == "reach":
        h[::5] *= 2.6
        blanked[1::7] = 1.0
    elif kind == "close":
        pos[1:-1:9] = pos[:-2:9] + 9e-5 * np.array([1.0, -1.0])
    return {"pos": pos, "h": h, "blanked": blanked}


@pytest.mark.parametrize("nx,ny", [(48, 16), (96, 7)])
@pytest.mark.parametrize("kind", ["above", "below", "two_heights", "edge", "narrow", "wide", "reach", "close", "cutoff"])
def test_pair_forms(kind, nx, ny):
    case = cases.perturbed(cases.small_cutting_case(nx=nx, ny=ny))
    out = []
    for prec in (_lib.FP32C, _lib.FP64):
        sim = S.Simulation(case, precision=prec)
        g = sim.grid.geom
        P = sim.state(("pos", "h", "blanked"))
        for f, a in _moved(kind, P, g).items():
            sim.p.upload(f, a)
        if kind == "cutoff":
            sim.ctx.call("sphfem_set_kernel_cutoff", 1e-17)
        print(kind, nx, ny, prec, flush=True)
        sim.step(1)
        sim.ctx.check_error()
        out.append(sim.state())
        sim.close()
    _check(out[0], out[1], DERIVS, TOL_DERIV, f"{kind} {nx}x{ny}")


def test_blanked_set_changes_between_steps():
    """which particles are blanked is read from the state, not from an earlier step's buffers"""
    case = cases.perturbed(cases.small_cutting_case(nx=48, ny=16))
    out = []
    for prec in (_lib.FP32C, _lib.FP64):
        sim = S.Simulation(case, precision=prec)
        for k in range(4):
            blanked = np.zeros(case.N)
            blanked[k % 2::5] = 1.0
            sim.p.upload("blanked", blanked)
            print("blanked set", k, prec, flush=True)
            sim.step(1)
        sim.ctx.check_error()
        out.append(sim.state())
        sim.close()
    _check(out[0], out[1], DERIVS, TOL_DERIV, "blanked sets")


def test_fp32c_stage_call_form_switch():
    """interactions_monaghan_fp32c in any order of calls with finite and non-finite inputs, for a particle
    count past a workgroup: the same outputs are NaN as with the FP64 call, the others agree to the
    derivative bound, and blanked particles' outputs are left alone."""
    o = _sorted(48, 16)
    sim = S.Simulation(o.case, precision=_lib.FP32C)
    n, nc = o.case.N, len(o.st["cell_start"])
    cells = [C.c_void_p(), C.c_void_p()]
    for q, name in zip(cells, ("cell_start", "cell_end")):
        sim.ctx.call("sphfem_malloc", C.byref(q), 4 * nc)
        sim.ctx.htod(q.value, o.st[name])
    S.interactions_setup_geometry_constants(sim.grid)
    clean = {f: o.P[f].copy() for f in STATE}
    clean["blanked"][5::11] = 1.0
    for fault in (None, ("S", np.nan), None, ("vel", np.nan), ("h", 0.8), ("pos", np.nan), None):
        got = {}
        for which in ("fp32c", "fp64"):
            for f in STATE:
                a = clean[f].copy()
                if fault is not None and f == fault[0]:
                    a[n // 2] = a[n // 2] * fault[1] if f == "h" else fault[1]
                sim.p.upload(f, a)
            print("fault", fault, which, flush=True)
            if which == "fp32c":
                S.interactions_monaghan_fp32c(sim.stepper, sim.p, cells[0].value, cells[1].value, nc)
            else:
                S.interactions_monaghan(sim.p, cells[0].value, cells[1].value, nc)
            got[which] = {f: sim.p.download(f) for f in OUT}
        a, b = got["fp32c"], got["fp64"]
        acc = lambda r: np.stack([r["S_der"][:, 0] + r["S_der"][:, 1] + r["vel_t"][:, 0],
                                  r["S_der"][:, 2] + r["S_der"][:, 3] + r["vel_t"][:, 1]], 1)
        live = clean["blanked"] != 1.0
        for name, x, y in (("v_der", a["v_der"], b["v_der"]), ("pos_t", a["pos_t"], b["pos_t"]),
                           ("T_t", a["T_t"], b["T_t"]), ("acceleration", acc(a), acc(b))):
            assert_equal(f"{fault} {name} non-finite", ~np.isfinite(x[live]), ~np.isfinite(y[live]))
            ok = live & np.isfinite(y.reshape(n, -1)).all(1)
            assert normwise(x, y, ok) <= TOL_DERIV, f"{fault} {name}"
        for f in OUT:
            assert_equal(f"{fault} blanked {f}", a[f][~live], clean[f][~live])
    for q in cells:
        sim.ctx.call("sphfem_free", q)
    sim.close()
