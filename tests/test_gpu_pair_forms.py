"""FP32C pair sums where the fast form's assumptions fail, against the FP64 pair sums of the same state:
particles above and below the grid's rows (their keys name cells of the next or previous column: they
meet only each other), two column heights away, on the grid's edge and clustered near coincidence; kernel
widths other than the cell size (smaller, and wide enough to reach the blanked records' place); a support
that starts at 0; grids of few rows.  One step's derivatives agree within 1e-5 of each field's largest
magnitude, the bound of the ordinary form: the general form does the same FP32 terms in the same blocks."""
import numpy as np
import pytest

from sph_fem_2d_cutting_gpu_amd import _lib, cases
from sph_fem_2d_cutting_gpu_amd import solver as S
from test_gpu_fp32c import DERIVS, TOL_DERIV, _check

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
    elif kind == "close":
        pos[1:-1:9] = pos[:-2:9] + 9e-5 * np.array([1.0, -1.0])
    return {"pos": pos, "h": h, "blanked": blanked}


@pytest.mark.parametrize("nx,ny", [(48, 16), (96, 7)])
@pytest.mark.parametrize("kind", ["above", "below", "two_heights", "edge", "narrow", "wide", "close", "cutoff"])
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
