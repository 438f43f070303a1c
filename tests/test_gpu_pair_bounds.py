"""The FP32C pair kernels on keys and cell tables that do not fit the particles: no access outside the
tables and records, whatever they hold."""
import ctypes as C

import numpy as np
import pytest

from helpers import assert_equal
from sph_fem_2d_cutting_gpu_amd import _lib, cases
from sph_fem_2d_cutting_gpu_amd import solver as S
from test_gpu_interactions_window import OUT

pytestmark = pytest.mark.gpu


class Pass:
    """a sorted chip domain with its cell table, and the FP32C pair sums over it"""

    def __init__(self, n):
        self.sim = sim = S.Simulation(cases.chip_case(n_target=n), precision=_lib.FP32C)
        self.nc = sim.grid.num_cell
        self.cells = [C.c_void_p(), C.c_void_p()]
        for q in self.cells:
            sim.ctx.call("sphfem_malloc", C.byref(q), 4 * self.nc)
        p, g = sim.p, sim.grid
        g.assign_hashes(p)
        g.sort(p)
        g.get_cells(p, self.cells[0].value, self.cells[1].value)
        S.interactions_setup_geometry_constants(g)
        S.material_eos(p)
        S.corrector_artificial_stress(p)

    def sums(self):
        S.interactions_monaghan_fp32c(self.sim.stepper, self.sim.p, self.cells[0].value, self.cells[1].value, self.nc)
        return {f: self.sim.p.download(f) for f in OUT}

    def close(self):
        for q in self.cells:
            self.sim.ctx.call("sphfem_free", q)
        self.sim.close()


@pytest.mark.parametrize("kernel", [_lib.PAIRS_LIST, _lib.PAIRS_STAGED])
def test_keys_outside_the_grid_are_reported(kernel):
    """Some particles' keys name no cell: the call is reported, and with the keys back the sums are as before."""
    s = Pass(5000)
    s.sim.set_tuning(pair_kernel=kernel)
    want = s.sums()
    s.sim.ctx.check_error()
    key = s.sim.p.download("hash")
    bad = np.arange(7, len(key), 101)
    wrong = key.copy()
    wrong[bad] = np.resize(np.array([s.nc, s.nc + 7, 2**30, 2**31 - 1, -1, -5, -2**31], np.int32), len(bad))
    s.sim.p.upload("hash", wrong)
    print("keys outside the grid", kernel, flush=True)
    got = s.sums()
    with pytest.raises(_lib.SphfemError):
        s.sim.ctx.check_error()
    for f in OUT:
        assert np.all(np.isfinite(got[f])), f
    s.sim.p.upload("hash", key)
    got = s.sums()
    for f in OUT:
        assert_equal(f, got[f], want[f])
    s.close()


@pytest.mark.parametrize("chunk", [16, 32, 48])
def test_cell_tables_that_leave_particles_out(chunk):
    """Every third column missing from the table, and some cells of the others: a particle's own column may
    have no records.  The staged kernel's sums equal the list kernel's bit for bit."""
    s = Pass(50_000)
    geo, start = s.sim.grid.geom, s.sim.ctx.dtoh(s.cells[0].value, s.nc, np.int32)
    cell = np.arange(s.nc)
    start[((cell // geo.ny) % 3 == 1) | (cell % 11 == 4)] = -1
    s.sim.ctx.htod(s.cells[0].value, start)
    out = []
    for kernel in (_lib.PAIRS_LIST, _lib.PAIRS_STAGED):
        s.sim.set_tuning(pair_kernel=kernel, pair_chunk=chunk)
        print("partial table", kernel, chunk, flush=True)
        out.append(s.sums())
        s.sim.ctx.check_error()
    for f in OUT:
        assert np.all(np.isfinite(out[0][f])), f
        assert_equal(f, out[1][f], out[0][f])
    s.close()
