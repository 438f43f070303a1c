"""Device memory that the library's objects hold."""
import ctypes as C

import numpy as np
import pytest

from helpers import assert_equal
from sph_fem_2d_cutting_gpu_amd import _lib, cases
from sph_fem_2d_cutting_gpu_amd import solver as S

pytestmark = pytest.mark.gpu


def _free(ctx):
    """free device memory, by the HIP runtime that the library has loaded"""
    ctx.synchronize()
    with open("/proc/self/maps") as f:
        path = next(l.split()[-1] for l in f if "libamdhip64" in l)
    free, total = C.c_size_t(), C.c_size_t()
    assert C.CDLL(path).hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_fp32c_stepper_holds_no_fp64_workspace():
    """An FP32C stepper takes 276 B per particle: the step's initial values (80), the near list (4), records,
    sums and the rates' carry (192); the FP64 form's 200 B are not there before an FP64 step."""
    n = 4_000_000
    ctx = S.Context(0)
    before = _free(ctx)
    h = C.c_void_p()
    ctx.call("sphfem_leap_frog_create", n, 0, 0, C.byref(h))
    ctx.call("sphfem_leap_frog_set_precision", h, _lib.FP32C)
    held = (before - _free(ctx)) / n
    print("bytes per particle", held, flush=True)
    assert 250 < held < 290
    ctx.call("sphfem_leap_frog_destroy", h)
    ctx.close()


def test_forms_switched_between_steps_and_graphs():
    """The FP64 workspace comes with the first FP64 step, also when that follows FP32C ones or is captured."""
    case = cases.perturbed(cases.small_cutting_case(nx=48, ny=16))
    ref = S.Simulation(case)
    ref.step(3)
    sims = [S.Simulation(case), S.Simulation(case, precision=_lib.FP32C)]
    print("first FP64 step eager and captured", flush=True)
    sims[0].step(1)
    sims[0].capture(2).launch(1)
    sims[0].ctx.check_error()
    want, got = ref.state(), sims[0].state()
    for f in ("hash", "idx", "pos", "vel", "S", "T"):
        assert_equal(f, got[f], want[f])
    sims[1].step(1)
    sims[1].ctx.call("sphfem_leap_frog_set_precision", sims[1].stepper.h, _lib.FP64)
    print("captured after FP32C steps", flush=True)
    sims[1].capture(2).launch(1)
    sims[1].ctx.check_error()
    got = sims[1].state()
    for f in ("hash", "idx"):
        assert_equal(f, got[f], want[f])
    for f in ("pos", "vel", "S", "T"):
        assert np.max(np.abs(got[f] - want[f])) <= 1e-6 * np.max(np.abs(want[f])), f


def test_interactions_workspace_goes_with_the_particles():
    """interactions_monaghan's workspace in the context: given back with the particles that it was sized for,
    there again for the next ones."""
    small, large = cases.chip_case(n_target=40_000), cases.chip_case(n_target=2_000_000)
    keep = S.Simulation(small)
    ctx = keep.ctx

    def sums(case, p, g):
        cells = [C.c_void_p(), C.c_void_p()]
        for q in cells:
            ctx.call("sphfem_malloc", C.byref(q), 4 * g.num_cell)
        g.assign_hashes(p)
        g.sort(p)
        g.get_cells(p, cells[0].value, cells[1].value)
        S.interactions_setup_geometry_constants(g)
        S.material_eos(p)
        S.corrector_artificial_stress(p)
        S.interactions_monaghan(p, cells[0].value, cells[1].value, g.num_cell)
        out = p.download("S_der")
        for q in cells:
            ctx.call("sphfem_free", q)
        return out

    print("workspace of", small.N, "then", large.N, "particles", flush=True)
    want = sums(small, keep.p, keep.grid)
    before = _free(ctx)
    init = cases.initial_particles(large)
    p = S.particle_gpu(ctx, large.N, **{f: init[f] for f in ("pos", "vel", "rho", "T", "h", "S")})
    g = S.grid_gpu_green(ctx, large.N, large.grid_bbmin, large.grid_bbmax, large.h)
    sums(large, p, g)
    ctx.call("sphfem_grid_destroy", g.h)
    p.free()
    assert before - _free(ctx) < 16 * large.N
    assert_equal("S_der", sums(small, keep.p, keep.grid), want)
    keep.close()
