"""The re-sort's three ways to the same order: the ranked changes, the one-launch work queue (an item a tile,
and above 256 tiles several) and the sort known beforehand (the queue, multi-block launches above 2^19
particles), at sizes around a tile and a wavefront.  Each step's order against numpy's stable argsort
of the hashes, and the whole state bit for bit."""
import dataclasses

import numpy as np
import pytest

from helpers import assert_equal
from sph_fem_2d_cutting_gpu_amd import _lib, cases
from sph_fem_2d_cutting_gpu_amd import solver as S

pytestmark = pytest.mark.gpu


def _moving(n):
    base = cases.chip_case(n_target=max(n, 40))
    pick = slice(0, n) if n < base.N else slice(0, base.N)
    cut = {f: getattr(base, f)[pick] for f in ("pos", "vel", "rho", "T", "hh", "fixed", "S")}
    # below 4096 changes a step
    scale = min(0.003, 810.0 / n) * base.h / base.dt / max(float(np.sqrt(np.mean(base.vel ** 2))), 1e-30)
    cut["vel"] = cut["vel"] * scale
    margin = 20 * base.h
    return dataclasses.replace(base, N=len(cut["pos"]), grid_bbmin=base.grid_bbmin - margin,
                               grid_bbmax=base.grid_bbmax + margin, **cut)


@pytest.mark.parametrize("n", [3, 64, 257, 4096, 4097, 60_000, 270_000, 1_100_000])
@pytest.mark.parametrize("prec", [_lib.FP64, _lib.FP32C])
def test_three_ways_one_order(n, prec):
    if prec == _lib.FP64 and n > 100_000:
        pytest.skip("the sort does not depend on the form")
    case = _moving(n)
    sims = {}
    for limit in (4096, 1, 0):
        sims[limit] = S.Simulation(case, precision=prec)
        sims[limit].grid.set_resort_limit(limit)
    seen = []
    for k in range(5):
        out = {}
        before = sims[4096].state(("pos",))["pos"]
        for limit, sim in sims.items():
            print(f"n {n} step {k} limit {limit}", flush=True)
            sim.step(1)
            sim.ctx.check_error()
            out[limit] = sim.state(("hash", "idx", "pos", "vel", "S", "rho"))
        seen.append(sims[4096].grid.resort_stats())
        geo = sims[4096].grid.geom
        key = (((before[:, 0] - geo.bbmin_x) / geo.dx).astype(np.int64) * geo.ny
               + ((before[:, 1] - geo.bbmin_y) / geo.dx).astype(np.int64))
        perm = np.argsort(key, kind="stable")
        assert_equal("idx", out[4096]["idx"], perm.astype(np.int32))
        assert_equal("hash", out[4096]["hash"], key[perm].astype(np.int32))
        for limit in (1, 0):
            for f in out[4096]:
                assert_equal(f"limit {limit} {f}", out[limit][f], out[4096][f])
    print(seen)
    assert all(m == 2 for m, _ in seen[1:])
    if n >= 4096:
        assert max(c for _, c in seen[1:]) > 4          # limit 1 takes the queue
    for sim in sims.values():
        sim.close()


@pytest.mark.parametrize("speed", [0.0003, 0.012, 0.03, 0.05, 0.1, 0.25])
def test_ranked_changes(speed):
    """From a few to more than 4096 changes a step among 60k particles moving together (counted, sorted in
    LDS, and above the limit the full sort): each step's order against numpy's stable argsort."""
    base = _moving(60_000)
    n = base.N
    vel = np.tile([0.8, -0.6], (n, 1)) * speed * base.h / base.dt
    sim = S.Simulation(dataclasses.replace(base, vel=vel, S=np.zeros((n, 4))), precision=_lib.FP32C)
    seen = []
    for k in range(6):
        before = sim.state(("pos",))["pos"]
        print(f"speed {speed} step {k}", flush=True)
        sim.step(1)
        sim.ctx.check_error()
        seen.append(sim.grid.resort_stats())
        geo = sim.grid.geom
        key = (((before[:, 0] - geo.bbmin_x) / geo.dx).astype(np.int64) * geo.ny
               + ((before[:, 1] - geo.bbmin_y) / geo.dx).astype(np.int64))
        perm = np.argsort(key, kind="stable")
        a = sim.state(("hash", "idx"))
        assert_equal("idx", a["idx"], perm.astype(np.int32))
        assert_equal("hash", a["hash"], key[perm].astype(np.int32))
    print(seen, flush=True)
    assert all((m == 2) == (c <= 4096) for m, c in seen[1:]) and any(c > 0 for _, c in seen[1:])
    sim.close()
