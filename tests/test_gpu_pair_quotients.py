"""The FP64 pair sums' quotients by shared reciprocals against the oracle's plain operators, bit for bit, at
operands where the reciprocal alone is not enough: viscous terms that overflow or lie among the subnormal
numbers (velocities of finite but extreme size)."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from helpers import assert_equal
from oracle.oracle import Oracle
from sph_fem_2d_cutting_gpu_amd import cases
from sph_fem_2d_cutting_gpu_amd import solver as S
from test_gpu_interactions_window import OUT, STATE

pytestmark = pytest.mark.gpu


def _columns(rows):
    """two columns of particles, one at x = 0 and one just short of a power of two away: the distance of the
    two particles of a row lies half an ulp class below that power"""
    base = cases.chip_case(n_target=40)
    x = np.ldexp(1.0 - 2.0**-53, int(np.floor(np.log2(base.dx))))
    pos = np.stack([np.tile([0.0, x], rows), np.repeat(1.05 * x * np.arange(rows), 2)], 1)
    rng, n = np.random.default_rng(5), 2 * rows
    Sd = np.zeros((n, 4))
    Sd[:, :3] = rng.standard_normal((n, 3)) * 3e-3
    return dataclasses.replace(base, N=n, pos=pos, vel=rng.standard_normal((n, 2)) * 1e-3, S=Sd,
                               rho=base.const.phys["rho0"] * (1 + 1e-3 * rng.standard_normal(n)),
                               T=300.0 + 50.0 * rng.random(n), hh=np.full(n, base.h), fixed=np.zeros(n),
                               grid_bbmin=pos.min(0) - 3 * base.h, grid_bbmax=pos.max(0) + 3 * base.h)


def _against_oracle(case, label):
    o = Oracle(case)
    for fn, sig in (("o_compute_hashes", "cp"), ("o_sort_and_cells", "cps"), ("o_material_eos", "cp"),
                    ("o_artificial_stress", "cp")):
        o.call(fn, sig)
    sim = S.Simulation(case)
    nc = len(o.st["cell_start"])
    cells = [C.c_void_p(), C.c_void_p()]
    for q, name in zip(cells, ("cell_start", "cell_end")):
        sim.ctx.call("sphfem_malloc", C.byref(q), 4 * nc)
        sim.ctx.htod(q.value, o.st[name])
    S.interactions_setup_geometry_constants(sim.grid)
    for f in STATE:
        sim.p.upload(f, o.P[f])
    print(label, flush=True)
    o.call("o_interactions_monaghan", "cps")
    S.interactions_monaghan(sim.p, cells[0].value, cells[1].value, nc)
    for f in OUT:
        got, want = sim.p.download(f), o.P[f]
        assert_equal(f"{label} {f} NaN", np.isnan(got), np.isnan(want))
        assert_equal(f"{label} {f}", np.nan_to_num(got, nan=0.0, posinf=np.inf, neginf=-np.inf),
                     np.nan_to_num(want, nan=0.0, posinf=np.inf, neginf=-np.inf))
    for q in cells:
        sim.ctx.call("sphfem_free", q)
    sim.close()
    return o


@pytest.mark.parametrize("scale", [1e170, 1e-300, 1e-310, 1e-316])
def test_viscous_terms_at_the_ends_of_the_range(scale):
    case = _columns(60)
    rng = np.random.default_rng(7)
    o = _against_oracle(dataclasses.replace(case, vel=rng.standard_normal((case.N, 2)) * scale), f"velocities {scale}")
    if scale > 1:
        assert np.isinf(o.P["vel_t"]).any()
    else:
        assert np.any(o.P["vel_t"] != 0.0)


def test_distances_just_below_a_power_of_two():
    o = _against_oracle(_columns(400), "below a power of two")
    assert np.all(o.P["T_t"] != 0.0)
