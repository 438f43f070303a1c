"""What is measured: the work that a user of this framework has it do, through its public entry points.

A cutting simulation advances a particle workpiece step by step (solver.Simulation, replayed from a
captured graph or launched step by step) with a FEM tool, a rigid tool or none, in the FP64 or the FP32C
form; beside it stand the kernel-only pass (hash, sort, cells, pressure and artificial stress, pair sums), the step assembled from the
reference's own functions, and a batch of independent cases.  Lengths, materials and tools are those of
sph_fem_2d_cutting_gpu_amd/cases.py; the sizes run from its smallest test case to the 4M-particle
benchmark and the 16M-particle chip domain.

The state starts from the lattice of the case with seeded noise on every field (as a cut that has run for
a while carries: part of the material yields) and one step already taken, so that the first full sort and
the first step's records are behind it.
"""
import ctypes as C
import dataclasses
import functools
import math

import numpy as np
import torch

from sph_fem_2d_cutting_gpu_amd import _lib, cases
from sph_fem_2d_cutting_gpu_amd import solver as S

# what a step leaves behind for the particles and for the FEM tool
PARTICLES = ("pos", "vel", "rho", "S", "T", "eps_pl", "eps_pl_dot", "fc", "ft", "n", "blanked", "hash", "idx", "on_seg")
TOOL = (("T", "node_num", ()), ("position", "node_num", (2,)), ("left", "seg_num", (2,)),
        ("heat_exchange", "seg_num", (2,)))
# what a sweep's user looks at, per case
SWEEP = ("pos", "vel", "S", "T")
# what one interaction pass leaves behind, after the sort
PASS = ("pos", "rho", "hash", "idx", "v_der", "S_der", "vel_t", "pos_t", "T_t")
SPEC = {name: (shape, dtype) for name, shape, dtype in cases.PARTICLE_FIELDS}


# ---------------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest run of a user: the reduced cutting case of the tests, a driver that steps one by one
        dict(name="cut_768_f64_eager", kind="cut", nx=48, ny=16, material="Ti6Al4V", tris=600, f32c=False,
             grid="green", wear=True, graph=False),
        # the 6,400-particle Ti6Al4V case, replayed from its graph: launches and latency count
        dict(name="cut_6400_f32c", kind="cut", nx=160, ny=40, material="Ti6Al4V", tris=2000, f32c=True,
             grid="green", wear=False, graph=True),
        # the 160k-particle AISI 1045 case
        dict(name="cut_160k_f32c", kind="cut", nx=800, ny=200, material="AISI1045", tris=8000, f32c=True,
             grid="green", wear=False, graph=True),
        # the 4M-particle Ti6Al4V case with wear: the benchmark's step
        dict(name="cut_4m_f32c_wear", kind="cut", nx=4000, ny=1000, material="Ti6Al4V", tris=8000, f32c=True,
             grid="green", wear=True, graph=True),
        # the FP64 form at a size that is no multiple of a tile
        dict(name="cut_1m_f64", kind="cut", nx=1999, ny=501, material="Ti6Al4V", tris=4000, f32c=False,
             grid="green", wear=False, graph=True),
        # the reference's other grid, which sorts in full at every step
        dict(name="cut_500k_f32c_rothlin", kind="cut", nx=1423, ny=353, material="AISI1045", tris=4000, f32c=True,
             grid="rothlin", wear=False, graph=True),
        # the reference's rigid-tool cut at a fine resolution (3.07M particles, a quarter of them the tool's)
        dict(name="rigid_3m_f32c", kind="rigid", ny=600, f32c=True, graph=True),
        # the impact of a disc on a wall: plasticity, no tool, a grid that follows the particles
        dict(name="impact_131k_f32c", kind="impact", nbox=200, f32c=True, graph=False),
        # kernel-only pass over the 16M-particle chip domain with its 10:1 density range
        dict(name="pass_16m_f32c", kind="pass", n=16_000_000, f32c=True),
        # the same pass with the reference's FP64 interactions_monaghan
        dict(name="pass_2m_f64", kind="pass", n=2_000_003, f32c=False),
        # the step as a caller of the reference writes it, function by function
        dict(name="calls_100k_f64", kind="calls", nx=633, ny=159, material="Ti6Al4V", tris=2000, wear=False),
        # a parameter sweep: 16 independent cases in flight together
        dict(name="batch_16_f32c", kind="batch", cases=16, tris=1000, f32c=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cut", "cut", "cut", "cut", "rigid", "impact", "pass", "pass", "calls", "batch"])
    f32c = rng.random() < 0.65
    material = rng.choice(["Ti6Al4V", "AISI1045"])
    if kind == "cut":
        n = _log(rng, 700, 3_500_000 if f32c else 1_000_000)
        ny = max(14, int(round(math.sqrt(n / rng.uniform(3.0, 5.0)))))
        return dict(kind="cut", nx=max(3 * ny, n // ny), ny=ny, material=material, tris=_log(rng, 500, 8000),
                    f32c=f32c, grid="rothlin" if rng.random() < 0.2 else "green", wear=rng.random() < 0.5,
                    graph=rng.random() < 0.8)
    if kind == "rigid":
        return dict(kind="rigid", ny=_log(rng, 30, 560 if f32c else 320), f32c=f32c, graph=rng.random() < 0.8)
    if kind == "impact":
        return dict(kind="impact", nbox=2 * _log(rng, 10, 130), f32c=f32c, graph=False)
    if kind == "pass":
        return dict(kind="pass", n=_log(rng, 20_000, 12_000_000 if f32c else 2_000_000), f32c=f32c)
    if kind == "calls":
        ny = _log(rng, 16, 300)
        return dict(kind="calls", nx=int(ny * rng.uniform(3.0, 5.0)), ny=ny, material=material,
                    tris=_log(rng, 500, 4000), wear=rng.random() < 0.5)
    return dict(kind="batch", cases=rng.randrange(3, 17), tris=_log(rng, 400, 1000), f32c=f32c)


# ---------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=4)
def _base(key):
    """The lattice, tool and constants of a case (no seed in them)."""
    c = dict(key)
    if c["kind"] in ("cut", "calls"):
        # spacing as the named cases of the same size have it: 2.5 um below 100k particles, 1.25 um below
        # 1M, 1 um above; depth of cut and edge radius in proportion to the height of small workpieces
        n = c["nx"] * c["ny"]
        dx = 2.5e-4 if n < 100_000 else (1.25e-4 if n < 1_000_000 else 1e-4)
        doc = min(5e-3, 0.4 * c["ny"] * dx)
        return cases.cutting_case("cut", c["nx"], c["ny"], dx, c["material"], 200.0, doc, 0.35, 0.0, 7.0,
                                  min(5e-4, 0.125 * doc), c["tris"], wear=c["wear"])
    if c["kind"] == "rigid":
        return cases.ref_cut_sph(ny=c["ny"])
    if c["kind"] == "impact":
        return cases.impact(c["nbox"])
    if c["kind"] == "pass":
        return cases.chip_case(n_target=c["n"])
    return tuple(cases.batch_cases(n_cases=c["cases"], tool_tris=c["tris"]))


def _seeded(case, seed, vel_sd=2e-4):
    """The case with seeded noise: 0.5 % of the spacing on the positions and, on the material that is not
    fixed, velocity, deviatoric stress (a few per cent of the material yields), density and temperature
    (0 to about 100 K of rise)."""
    S_sd = 0.18 * case.const.joco["A"]
    rng = np.random.default_rng(seed)
    n = case.N
    mat = np.ones(n) if case.tool_p is None else 1.0 - case.tool_p
    free = mat * (case.fixed == 0.0)
    pos = case.pos + (mat * case.dx * 5e-3)[:, None] * (2.0 * rng.random((n, 2)) - 1.0)
    # inside the box of the locked grid, as the lattice is
    pos = np.clip(pos, case.pos.min(axis=0), case.pos.max(axis=0))
    vel = case.vel + free[:, None] * rng.standard_normal((n, 2)) * vel_sd
    sd = free[:, None] * rng.standard_normal((n, 3)) * S_sd
    Sn = np.zeros((n, 4)) if case.S is None else case.S.copy()
    Sn[:, :3] += sd
    Sn[:, 3] -= sd[:, 0] + sd[:, 2]
    rho = case.rho * (1.0 + free * rng.standard_normal(n) * 1e-3)
    T = case.T + free * np.abs(rng.standard_normal(n)) * 40.0
    return dataclasses.replace(case, pos=pos, vel=vel, S=Sn, rho=rho, T=T)


def _inputs(case, seed):
    base = _base(tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "f32c", "grid", "graph"))))
    if case["kind"] == "impact":      # SI units
        return _seeded(base, seed, vel_sd=1.0)
    if case["kind"] == "batch":
        return [_seeded(b, seed * 64 + k) for k, b in enumerate(base)]
    return _seeded(base, seed)


class _Owner:
    """Releases a simulation's device memory with the last tensor that looks into it."""

    def __init__(self, sim):
        self.sim = sim

    def __del__(self):
        self.sim.close()


class _Span:
    def __init__(self, owner, ptr, shape, dtype):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=np.dtype(dtype).str, data=(ptr, False),
                                             version=2)


def _view(owner, ptr, shape, dtype):
    """Device memory of the library as a tensor, without a copy."""
    return torch.as_tensor(_Span(owner, int(ptr), shape, dtype), device="cuda")


class _Fields:
    """The fields of a simulation as tensors; the library swaps its arrays, so a view is looked up by address."""

    def __init__(self, owner, sim, names):
        self.owner, self.sim, self.names, self.known = owner, sim, names, {}

    def __call__(self):
        out = {}
        p = self.sim.p
        for name in self.names:
            ptr = p.ptr(name)
            if ptr not in self.known:
                shape, dtype = SPEC[name]
                self.known[ptr] = _view(self.owner, ptr, (p.N,) + shape, dtype)
            out[name] = self.known[ptr]
        if self.sim.tool is not None and "on_seg" in self.names:
            out.update(self.tool())
        return out

    def tool(self):
        if "tool" not in self.known:
            a = self.sim.tool.arrays()
            self.known["tool"] = {"tool_" + name: _view(self.owner, a[name], (a[count],) + shape, np.float64)
                                  for name, count, shape in TOOL}
        return self.known["tool"]


def _precision(case):
    return _lib.FP32C if case.get("f32c") else _lib.FP64


def prepare(case, seed):
    state = dict(case=case)
    inputs = _inputs(case, seed)
    if case["kind"] == "batch":
        batch = S.BatchedSimulation(inputs, precision=_precision(case))
        owner = _Owner(batch)
        batch.step(1)
        batch.capture(one_graph=False)
        state.update(owner=owner, batch=batch, fields=[_Fields(owner, s, SWEEP) for s in batch.sims])
        batch.synchronize()
        return state
    sim = S.Simulation(inputs, precision=_precision(case), grid=case.get("grid", "green"))
    owner = _Owner(sim)
    state.update(owner=owner, sim=sim)
    if case["kind"] in ("pass", "calls"):
        nc = sim.grid.num_cell
        cells = [torch.empty(nc, dtype=torch.int32, device="cuda") for _ in range(2)]
        torch.cuda.synchronize()
        state.update(cells=cells, cs=cells[0].data_ptr(), ce=cells[1].data_ptr(), nc=nc)
        state["fields"] = _Fields(owner, sim, PASS if case["kind"] == "pass" else PARTICLES)
        if case["kind"] == "pass":
            S.interactions_setup_geometry_constants(sim.grid)
        else:
            _calls(state)
    else:
        sim.step(1)
        state["fields"] = _Fields(owner, sim, PARTICLES)
        state["graph"] = sim.capture(2) if case["graph"] else None
    sim.synchronize()
    return state


# ---------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------
def _calls(s):
    """leap_frog::step(particles, grid, tool_FEM) written with the reference's own functions."""
    sim = s["sim"]
    p, g, t, lf, dt = sim.p, sim.grid, sim.tool, sim.stepper, sim.case.dt
    g.assign_hashes(p)
    g.sort(p)
    g.get_cells(p, s["cs"], s["ce"])
    lf.init(p)
    t.reset_FEM_server()
    t.segments_wear_rate_reset()
    lf.predict(p, dt)
    t.calculate_temp(0.5 * dt)
    S.material_eos(p)
    S.corrector_artificial_stress(p)
    S.interactions_setup_geometry_constants(g)
    S.interactions_monaghan(p, s["cs"], s["ce"], s["nc"])
    S.material_stress_rate_jaumann(p)
    S.contmech_continuity(p)
    S.contmech_momentum(p)
    S.contmech_advection(p)
    lf.correct(p, dt)
    S.material_fric_heat_gen_FEM_v2(p, t)
    t.apply_heat_boundary_condition()
    t.calculate_temp_rate()
    t.calculate_temp(dt)
    S.plasticity_johnson_cook(p)
    if sim.case.wear:
        S.wear_adjustment(t)
    t.segments_update(dt)
    t.tool_update_FEM_gpu(dt)
    S.compute_contact_forces_FEM_tool_v3(p, t)
    S.perform_boundary_conditions(p)
    S.perform_boundary_conditions_thermal(p)
    S.debug_invalidate(p)


def run(state):
    kind = state["case"]["kind"]
    if kind == "batch":
        state["batch"].launch(1)
        return [f() for f in state["fields"]]
    sim = state["sim"]
    if kind == "pass":
        p, g = sim.p, sim.grid
        g.assign_hashes(p)
        g.sort(p)
        g.get_cells(p, state["cs"], state["ce"])
        S.material_eos(p)
        S.corrector_artificial_stress(p)
        if state["case"]["f32c"]:
            S.interactions_monaghan_fp32c(sim.stepper, p, state["cs"], state["ce"], state["nc"])
        else:
            S.interactions_monaghan(p, state["cs"], state["ce"], state["nc"])
    elif kind == "calls":
        _calls(state)
    elif state["graph"] is not None:
        state["graph"].launch(1)
    else:
        sim.step(2)
    return state["fields"]()


# ---------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far two right answers may lie apart
# ---------------------------------------------------------------------------------------------------
# bytes per particle of one step: the state read once and written once.  Read: pos, vel, S, fixed, blanked,
# tool_particle, rho, T, eps_pl, eps_pl_dot, h, fc, ft, n, hash, on_seg (200) and the rates (80, or 40 in FP32).
# Written: the same and p, idx (212, rates 80 or 40).
STEP_BYTES = {False: 200 + 212 + 160, True: 200 + 212 + 80}
# one pass: the 20 arrays of the sort read and written (276 each), hash and idx, then p and R, the pair sums' 112
# bytes read and 112 written
PASS_BYTES = 276 * 2 + 12 + 40 + 224
# a pair term is about 90 operations, 28 neighbours a particle; the rest of a step about 400
STEP_FLOPS = 28 * 90 + 400


def _size(case):
    if case["kind"] in ("cut", "calls"):
        return case["nx"] * case["ny"]
    if case["kind"] == "rigid":       # the workpiece's lattice and the tool's samples, in proportion
        return int(case["ny"] ** 2 * 8.536)
    if case["kind"] == "impact":
        return int(case["nbox"] ** 2 * (math.pi / 4 + 2.48))
    if case["kind"] == "pass":
        return case["n"]
    return 115_000 * case["cases"]


def work(case):
    n = _size(case)
    if case["kind"] == "pass":
        return {"bytes": float(PASS_BYTES * n), "flops": float(28 * 90 * n)}
    steps = 1 if case["kind"] == "calls" else 2
    return {"bytes": float(steps * STEP_BYTES[bool(case.get("f32c"))] * n), "flops": float(steps * STEP_FLOPS * n)}


def tolerance(case):
    # FP32C sums pair terms in 32 bits; the FP64 form rounds distances to single precision where the
    # reference does, so an implementation without those roundings differs at 1e-7 too.  A particle at its
    # yield stress may go either way, which a maximum sees.  Both forms lie within 2e-6 of exact() in the
    # plastic strain rate and within 3e-7 in everything else.
    if case.get("f32c"):
        return {"rel": 1e-5, "max": 5e-2, "differ": 1e-5}
    return {"rel": 7e-6, "max": 1e-2, "differ": 1e-5}


# ---------------------------------------------------------------------------------------------------
# the same in 64 bits, without the framework's kernels
# ---------------------------------------------------------------------------------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _kernel(rr2, h, rr2_min):
    """Value and radial factor (gradient over distance vector) of the kernel; zero outside the support."""
    inside = (rr2 < 4 * h * h) & (rr2 >= rr2_min)
    r = torch.sqrt(torch.where(inside, rr2, h * h))
    q = r / h
    fac = 0.454728408833987 / (h * h)
    outer = q > 1
    w = fac * torch.where(outer, 0.25 * (2 - q) ** 6, 1 - 1.5 * q * q * (1 - 0.5 * q))
    g = fac / h / r * torch.where(outer, -0.75 * (2 - q) ** 2, -3.0 * q * (1 - 0.75 * q))
    return w * inside, g * inside, inside


def _pair_sums(c, geom, rr2_min, p, lo, hi):
    """Pair sums of the sorted particles lo..hi of p (no tool particles, none blanked)."""
    const = c.const
    mass, K = const.phys["mass"], const.phys["K"]
    corr, alpha = const.corr, const.trml_wp["alpha"]
    nx, ny = geom["nx"], geom["ny"]
    i = torch.arange(lo, hi, device=p["pos"].device)
    key = p["hash"].long()
    gi = key[lo:hi] // ny
    gj = key[lo:hi] - gi * ny
    me = {f: p[f][lo:hi] for f in ("pos", "vel", "rho", "S", "R", "p", "T", "h")}
    n = hi - lo
    out = {f: torch.zeros(n, dtype=torch.float64, device=i.device)
           for f in ("xx", "xy", "yx", "yy", "sx", "sy", "sz", "sw", "vx", "vy", "px", "py", "T")}
    ci = torch.sqrt(K / me["rho"])
    for d in range(-2, 3):
        col = gi + d
        ok = (col >= 0) & (col < nx)
        first = torch.searchsorted(key, (col * ny + (gj - 2).clamp(min=0)).contiguous())
        last = torch.searchsorted(key, (col * ny + (gj + 3).clamp(max=ny)).contiguous())
        count = torch.where(ok, last - first, torch.zeros_like(first))
        for k in range(int(count.max()) if n else 0):
            j = torch.where(k < count, first + k, i)
            x = me["pos"] - p["pos"][j]
            rr2 = (x * x).sum(1)
            w, g, inside = _kernel(rr2, me["h"], rr2_min)
            on = (inside & (k < count)).double()
            w, g = w * on, g * on
            wx, wy = g * x[:, 0], g * x[:, 1]
            rho, vol = p["rho"][j], mass / p["rho"][j]
            dv = p["vel"][j] - me["vel"]
            out["xx"] += dv[:, 0] * wx * vol
            out["xy"] += dv[:, 0] * wy * vol
            out["yx"] += dv[:, 1] * wx * vol
            out["yy"] += dv[:, 1] * wy * vol
            f = (w / corr["wdeltap"]) ** 4
            a, b = 1 / me["rho"] ** 2, 1 / rho ** 2
            Sj, Rj, pj = p["S"][j], p["R"][j], p["p"][j]
            sxx = (me["S"][:, 0] - me["p"]) * a + (Sj[:, 0] - pj) * b + f * (me["R"][:, 0] + Rj[:, 0])
            sxy = me["S"][:, 1] * a + Sj[:, 1] * b + f * (me["R"][:, 1] + Rj[:, 1])
            syy = (me["S"][:, 2] - me["p"]) * a + (Sj[:, 2] - pj) * b + f * (me["R"][:, 2] + Rj[:, 2])
            out["sx"] += mass * sxx * wx
            out["sy"] += mass * sxy * wy
            out["sz"] += mass * sxy * wx
            out["sw"] += mass * syy * wy
            vr = -(dv * x).sum(1)
            rij, hij = 0.5 * (me["rho"] + rho), 0.5 * (me["h"] + p["h"][j])
            mu = hij * vr / (rr2 + corr["eta"] ** 2 * hij * hij)
            pi = (-corr["alpha"] * 0.5 * (ci + torch.sqrt(K / rho)) * mu + corr["beta"] * mu * mu) / rij * (vr < 0)
            out["vx"] -= mass * pi * wx
            out["vy"] -= mass * pi * wy
            out["px"] += corr["xspheps"] * w * mass / rij * dv[:, 0]
            out["py"] += corr["xspheps"] * w * mass / rij * dv[:, 1]
            if alpha != 0.0:
                out["T"] += 2.0 * vol * (me["T"] - p["T"][j]) * g * (rr2 > 1e-16)
    return out


def _sums(c, geom, rr2_min, p):
    n, step = len(p["hash"]), 2_000_000
    parts = [_pair_sums(c, geom, rr2_min, p, a, min(a + step, n)) for a in range(0, n, step)]
    return {f: torch.cat([x[f] for x in parts]) for f in parts[0]}


def _eos(c, p):
    const = c.const
    p["p"] = const.phys["K"] / const.phys["rho0"] * (p["rho"] - const.phys["rho0"])
    sxx, sxy, syy = p["S"][:, 0] - p["p"], p["S"][:, 1], p["S"][:, 2] - p["p"]
    th = 0.5 * torch.atan2(2 * sxy, sxx - syy)
    co, si = torch.cos(th), torch.sin(th)
    a = co * co * sxx + 2 * co * si * sxy + si * si * syy
    b = si * si * sxx - 2 * co * si * sxy + co * co * syy
    k = -const.corr["stresseps"] / p["rho"] ** 2
    a, b = k * a.clamp(min=0), k * b.clamp(min=0)
    p["R"] = torch.stack([co * co * a + si * si * b, co * si * (a - b), si * si * a + co * co * b, 0 * a], 1)


def _grid(c, p):
    if c.max_cell is None:
        return cases.grid_geometry(c.grid_bbmin, c.grid_bbmax, c.h)
    lo, hi = p["pos"].min(0).values.tolist(), p["pos"].max(0).values.tolist()
    return cases.grid_geometry(lo, hi, float(p["h"].max()))


def _sort(geom, p, keep=()):
    k = ((p["pos"] - torch.tensor([geom["bbmin_x"], geom["bbmin_y"]], dtype=torch.float64, device=p["pos"].device))
         / geom["dx"]).long()
    key = k[:, 0] * geom["ny"] + k[:, 1]
    order = torch.sort(key, stable=True).indices
    for f in list(p):
        if f not in keep:
            p[f] = p[f][order]
    p["hash"] = key[order].int()
    return order


def _yield(j, eps, rate, T):
    theta = ((T - j["Tref"]) / (j["Tmelt"] - j["Tref"])).clamp(max=1.0)
    r = rate / j["eps_dot_ref"]
    b = torch.where(r > 1, 1 + j["C"] * torch.log(r.clamp(min=1.0)), (1 + r) ** j["C"])
    return (j["A"] + j["B"] * eps ** j["n"]) * b * (1 - theta ** j["m"])


def _plastic(c, p, pr):
    j, G, dt, tq = c.const.joco, c.const.phys["G"], c.dt, c.const.trml_wp["tq"]
    s = p["S"]
    x, y, z, xy = s[:, 0] - pr, s[:, 2] - pr, s[:, 3] - pr, s[:, 1]
    svm = torch.sqrt(x * x + y * y + z * z - x * y - x * z - y * z + 3 * xy * xy)
    at = (svm >= _yield(j, p["eps_pl"], p["eps_pl_dot"], p["T"])).nonzero().squeeze(1)
    rate0 = p["eps_pl_dot"][at]
    p["eps_pl_dot"] = torch.zeros_like(p["eps_pl_dot"])
    s, eps, T = s[at], p["eps_pl"][at], p["T"][at]
    norm = torch.sqrt(s[:, 0] ** 2 + s[:, 2] ** 2 + s[:, 3] ** 2 + 2 * s[:, 1] ** 2)
    r23 = math.sqrt(2 / 3)

    def off(d):
        e = r23 * d.clamp(min=0)
        return norm - 2 * G * d - r23 * _yield(j, eps + e, e / dt, T)

    dl = (rate0 * dt * r23).clamp(min=1e-8)
    going = torch.ones_like(dl, dtype=torch.bool)
    for _ in range(102):
        g, g1 = off(dl), off(1.01 * dl)
        new = dl - g / ((g - g1) / (dl - 1.01 * dl))
        new = torch.where(new < 0, -0.1 * new, new)
        new = torch.where(going, new, dl)
        going = going & ((new - dl).abs() >= 1e-6)
        dl = new
        if not bool(going.any()):
            break
    e = r23 * dl.clamp(min=0)
    p["eps_pl"][at] = eps + e
    p["eps_pl_dot"][at] = e / dt
    p["S"][at] = s - s / norm[:, None] * dl[:, None] * 2 * G
    if tq != 0.0:
        T = T + tq / (c.const.trml_wp["cp"] * p["rho"][at]) * e * _yield(j, eps + e, e / dt, T)
        p["T"][at] = T


class _Tool:
    """The FEM tool of a case: nodes, segments and heat conduction (cold: its wear is below 1e-20 cm)."""

    def __init__(self, c, dev):
        t = c.tool

        def f(a):
            return torch.tensor(np.asarray(a, np.float64), device=dev)

        def whole(a):
            return torch.tensor(np.asarray(a, np.int64), device=dev)

        self.c, self.T, self.pos, self.n = c.const.tool, f(t.T), f(t.nodes), f(t.seg_n)
        self.left, self.right, self.ends = f(t.seg_left), f(t.seg_right), whole(t.seg_marks[:, 2:4])
        self.K, self.M, self.f, self.col = f(t.K), f(t.M), f(t.f), whole(t.col_ind)
        self.row = whole(np.repeat(np.arange(len(t.nodes)), np.diff(t.row_ptr)))
        self.vel, self.tl, self.ref = f(c.tool_vel), f(t.tl), t.ref_dist
        self.k = torch.zeros_like(self.T)
        self.exchange = torch.zeros_like(self.left)
        self.fric = torch.zeros(len(self.left), dtype=torch.float64, device=dev)

    def begin(self, dt):
        self.T_old = self.T
        self.T = self.T + 0.5 * dt * self.k

    def end(self, dt):
        load = -torch.zeros_like(self.T).index_add(0, self.row, self.K * self.T[self.col]) + self.f
        hot = (self.exchange[:, 1] != 0).nonzero().squeeze(1)
        length = torch.sqrt(((self.left - self.right)[hot] ** 2).sum(1))
        Tc = self.exchange[hot, 0] / self.exchange[hot, 1]
        for k in range(2):
            node = self.ends[hot, k]
            load = load.index_add(0, node, 0.5 * self.c["h"] * length * (Tc - self.T[node]) + 0.5 * self.fric[hot])
        self.k = load / self.M
        self.T = self.T_old + dt * self.k
        for a in (self.pos, self.left, self.right, self.tl):
            a += dt * self.vel
        self.exchange, self.fric = torch.zeros_like(self.exchange), torch.zeros_like(self.fric)


def _friction(c, t, p):
    """Friction heat of the particles that the last step left on a segment (after the corrector)."""
    at = ((p["on_seg"] != -1) & (p["eps_pl"] <= 20)).nonzero().squeeze(1)
    seg, n = p["on_seg"][at].long(), p["n"][at]
    dv = p["vel"][at] - t.vel
    rel = torch.sqrt(((dv - (dv * n).sum(1)[:, None] * n) ** 2).sum(1))
    heat = t.c["eta"] * torch.sqrt((p["ft"][at] ** 2).sum(1)) * rel * (rel <= 0.03)
    p["T"][at] += heat * (1 - t.c["beta"]) * c.dt / c.const.trml_wp["cp"] / c.const.phys["mass"]
    t.fric.index_add_(0, seg, heat * t.c["beta"])


def _contact(c, t, p):
    """Penalty contact and friction of the particles near the moved tool, and their heat exchange."""
    near = (((p["pos"] - t.tl) ** 2).sum(1).sqrt() < 1.05 * t.ref).nonzero().squeeze(1)
    ft_old = p["ft"][near]
    for f in ("fc", "ft", "n"):
        p[f] = torch.zeros_like(p[f])
    p["on_seg"] = torch.full_like(p["on_seg"], -1)
    q = p["pos"][near][:, None, :]
    lx, ly, rx, ry = t.left[:, 0], t.left[:, 1], t.right[:, 0], t.right[:, 1]

    def single(a):
        return a.float().double()

    # crossings of the ray towards +x, with the ends compared in single precision as the reference does
    band = (q[..., 1] <= single(torch.maximum(ly, ry))) & (q[..., 1] >= single(torch.minimum(ly, ry)))
    flat = ly == ry
    xs = rx + (lx - rx) / torch.where(flat, torch.ones_like(ly), ly - ry) * (q[..., 1] - ry)
    hit = torch.where(flat, q[..., 0] <= torch.maximum(lx, rx), (xs > q[..., 0]) & (xs != lx))
    hit = band & (hit | ((lx == rx) & (q[..., 0] < lx)))
    inside = hit.sum(1) % 2 == 1
    near, q, ft_old = near[inside], q[inside], ft_old[inside]
    if len(near) == 0:
        return
    depth = ((q - t.left) * t.n).sum(2)
    foot = q - depth[..., None] * t.n
    lo, hi = torch.minimum(t.left, t.right), torch.maximum(t.left, t.right)
    ok = ((q > lo - 8e-4) & (q < hi + 8e-4) & (foot >= lo) & (foot <= hi)).all(2) & (depth >= 0)
    depth = torch.where(ok, depth, torch.full_like(depth, 1e30))
    dist, seg = depth.min(1)
    normal = -t.n[seg]
    corner = (dist > 2.5e-4).nonzero().squeeze(1)
    if len(corner):
        away = torch.sqrt(((q[corner] - t.right) ** 2).sum(2))
        dist[corner], seg[corner] = away.min(1)
        for k in corner.tolist():
            s = int(seg[k])
            j = (t.left == t.right[s]).all(1).nonzero()
            m = (t.n[int(j[0])] + t.n[s]) / 2 if len(j) else t.n[s]
            normal[k] = -m / torch.sqrt((m * m).sum())
    dt, m, a = c.dt, t.c["slave_mass"], t.c["contact_alpha"]
    fN = m * dist[:, None] * normal / dt ** 2 * a
    dv = p["vel"][near] - t.vel
    dv = dv - (dv * normal).sum(1)[:, None] * normal
    trial = ft_old - a * m * dv / dt
    size, most = torch.sqrt((trial ** 2).sum(1)), t.c["mu"] * torch.sqrt((fN ** 2).sum(1))
    trial = trial * torch.where(size > most, most / size.clamp(min=1e-300), torch.ones_like(size))[:, None]
    p["fc"][near], p["ft"][near], p["n"][near], p["on_seg"][near] = fN, trial, normal, seg.int()
    T = p["T"][near]
    rise = 0.5 * (t.T[t.ends[seg, 0]] + t.T[t.ends[seg, 1]]) - T
    length = torch.sqrt(m / p["rho"][near])
    t.exchange.index_add_(0, seg, torch.stack([T * length, length], 1))
    step = rise * t.c["h"] * length / c.const.trml_wp["cp"] / m * dt
    p["T"][near] = T + torch.where(step < 0, torch.maximum(step, rise), torch.minimum(step, rise))


def _step(c, t, p, rothlin=False):
    const, dt = c.const, c.dt
    geom = _grid(c, p)
    if t is not None:
        t.begin(dt)
    order = _sort(geom, p, keep=("ft", "n", "hash") if rothlin else ("hash", "idx"))
    if not rothlin:
        p["idx"] = order.int()
    rates = {"pos": "pos_t", "vel": "vel_t", "S": "S_t", "rho": "rho_t", "T": "T_t"}
    start = {f: p[f] for f in rates}
    for f, r in rates.items():
        p[f] = p[f] + 0.5 * dt * p[r]
    _eos(c, p)
    pr = p["p"]
    a = _sums(c, geom, cases.default_rr2_min(c.dx), p)
    w = 0.5 * (a["xy"] - a["yx"])
    tr = (a["xx"] + a["yy"]) / 3
    G2, s = 2 * const.phys["G"], p["S"]
    p["S_t"] = torch.stack([G2 * (a["xx"] - tr) + 2 * w * s[:, 1],
                            G2 * 0.5 * (a["xy"] + a["yx"]) - w * s[:, 0] + w * s[:, 2],
                            G2 * (a["yy"] - tr) - 2 * w * s[:, 1], -G2 * tr], 1)
    p["rho_t"] = -p["rho"] * (a["xx"] + a["yy"])
    p["vel_t"] = (torch.stack([a["vx"] + a["sx"] + a["sy"], a["vy"] + a["sz"] + a["sw"]], 1)
                  + (p["fc"] + p["ft"]) / const.phys["mass"])
    p["pos_t"] = torch.stack([a["px"], a["py"]], 1) + p["vel"]
    if const.trml_wp["alpha"] != 0.0:
        p["T_t"] = const.trml_wp["alpha"] * a["T"]
    for f, r in rates.items():
        p[f] = start[f] + dt * p[r]
    if t is not None:
        _friction(c, t, p)
        t.end(dt)
    if const.joco is not None:
        _plastic(c, p, pr)
    if t is not None:
        _contact(c, t, p)
    held = p["fixed"] != 0
    for f in ("vel", "fc", "pos_t", "vel_t"):
        p[f][held] = 0.0
    if const.trml_wp["alpha"] != 0.0:        # the setups switch the thermal boundary on with the conduction
        p["T"][held] = const.trml_wp["T_init"]


def exact(case, seed):
    if case["kind"] in ("rigid", "batch"):
        return None
    c = _inputs(case, seed)
    dev = _device()
    p = {k: torch.tensor(v, device=dev) for k, v in cases.initial_particles(c).items()
         if k not in ("tool_particle", "R", "p", "S_der", "v_der")}
    if case["kind"] == "pass":
        geom = _grid(c, p)
        p["idx"] = _sort(geom, p, keep=("hash", "idx")).int()
        _eos(c, p)
        a = _sums(c, geom, cases.default_rr2_min(c.dx), p)
        f32c = case["f32c"]
        ax, ay = a["sx"] + a["sy"] + a["vx"], a["sz"] + a["sw"] + a["vy"]
        zero = torch.zeros_like(ax)
        return {"pos": p["pos"], "rho": p["rho"], "hash": p["hash"], "idx": p["idx"],
                "v_der": torch.stack([a["xx"], a["xy"], a["yx"], a["yy"]], 1),
                "S_der": torch.stack([ax, zero, ay, zero] if f32c else [a["sx"], a["sy"], a["sz"], a["sw"]], 1),
                "vel_t": torch.stack([zero, zero] if f32c else [a["vx"], a["vy"]], 1),
                "pos_t": torch.stack([a["px"], a["py"]], 1), "T_t": c.const.trml_wp["alpha"] * a["T"]}
    tool = _Tool(c, dev) if c.tool is not None else None
    for _ in range(2 if case["kind"] == "calls" else 3):
        _step(c, tool, p, case.get("grid") == "rothlin")
    out = {f: p[f] for f in PARTICLES}
    if tool is not None:
        out.update(tool_T=tool.T, tool_position=tool.pos, tool_left=tool.left, tool_heat_exchange=tool.exchange)
    return out
