"""The engine's work as a program that uses it gives it: IMC steps of the
problems that storm_amd.problems describes, through storm_amd.engine.

A case is one problem at one size in one precision:
  kind      which problem (below)
  n, n2     its size: cells along x, cells along y and z, cells of the
            tessellation, or instances of the batch
  scale     packets, as a multiple of the problem's own number
  fp64      the FP64 engine instead of the mixed one
  steps     IMC steps of a pass; a program that marches a problem reads the
            cells back every few steps (large problems: every step)
  warm      steps taken before, so that a pass starts with a census
  stepping  "resident": storm_gpu_step with the census kept in HBM;
            "noalloc": storm_gpu_step_noalloc;
            "exchange": what the C++ manager does by default for every step:
            material state and census in from the host, both back out

A pass returns the per-cell state after its last step (temperature, internal
energy, radiation energy, census energy, Fleck factor, opacity), the particle
and event counts of that step, and, where the case has them, the per-group
radiation energy and the census packets.
"""
from __future__ import annotations

import functools
import math

import numpy as np

from storm_amd import capi
from storm_amd import problems as P
from storm_amd.engine import GpuEngine

CELLS = ("T", "e", "erad", "census", "fleck", "sigma_p")
COUNTS = ("initial_particles", "prestep_particles", "start_particles", "end_particles", "emitted_particles",
          "boundary_particles", "census_before_comb", "leaving_particles", "segments", "random_walk_steps",
          "ddmc_steps", "energy_quantum_exp")

# Per kind: the ranges its drawn cases come from (n, n2, scale; the listed
# ones lie in them) and the segments a packet takes in a step, about.
RANGES = {
    "slab": dict(n=(10, 1000), n2=(1, 1), scale=(0.01, 8.0), segments=9),
    "marshak": dict(n=(64, 1024), n2=(1, 1), scale=(0.5, 20.0), segments=25),
    "densmore": dict(n=(64, 1024), n2=(1, 1), scale=(0.25, 8.0), segments=12),
    "cube": dict(n=(8, 64), n2=(1, 1), scale=(0.1, 1.0), segments=18),
    "step_slab": dict(n=(32, 256), n2=(4, 16), scale=(0.1, 1.0), segments=20),
    "voronoi_groups": dict(n=(500, 40000), n2=(8, 64), scale=(0.1, 1.0), segments=17),
    "voronoi_thick": dict(n=(200, 20000), n2=(1, 1), scale=(0.5, 8.0), segments=8),
    "batch": dict(n=(4, 48), n2=(1, 1), scale=(0.05, 0.5), segments=100),
}


def listed():
    def case(name, kind, n, n2=1, scale=1.0, fp64=False, steps=1, warm=3, stepping="resident"):
        return dict(name=name, kind=kind, n=n, n2=n2, scale=scale, fp64=fp64, steps=steps, warm=warm,
                    stepping=stepping)

    return [
        # A quick look at a coarse slab, the smallest calls: a step is all launches and waits.
        case("slab tiny", "slab", 20, scale=0.02, steps=8, stepping="noalloc"),
        # The gray 100-cell slab at its own 1e5 packets: a test problem that is run many times.
        case("slab", "slab", 100, steps=4),
        # An odd slab behind the drop-in C++ manager's default contract: the host hands in the
        # material and the particles and takes both back, every step.
        case("slab exchange", "slab", 333, scale=0.37, stepping="exchange"),
        # A Marshak wave as the examples run it: thousands of steps of few packets in opaque cells.
        case("marshak", "marshak", 256, steps=8),
        # The 30-group step-opacity slab with the partial-gray random walk and spectra per cell.
        case("densmore groups", "densmore", 512, n2=30, steps=4),
        # A small 3-D cube at an odd size.
        case("cube 21", "cube", 21, scale=0.5, steps=4),
        # The largest 3-D problem: a 64^3 cube, over 1e7 packets a step.
        case("cube 64", "cube", 64, steps=2),
        # The plain FP64 form, which users take to check the mixed one.
        case("cube 32 fp64", "cube", 32, scale=0.7, fp64=True, steps=2),
        # Two materials, the random walk and DDMC in the opaque half.
        case("step slab", "step_slab", 256, n2=16, scale=0.6, steps=2),
        # Multigroup on a Voronoi tessellation: 64 groups.
        case("voronoi groups", "voronoi_groups", 30000, n2=64, scale=0.8, warm=2),
        # Gray polyhedral cells with the random walk and DDMC.
        case("voronoi thick", "voronoi_thick", 5000, scale=2.0, steps=2),
        # Many independent slabs stepped as one engine.
        case("slab batch", "batch", 32, scale=0.4, warm=2),
    ]


def draw(rng):
    kind = rng.choice(sorted(RANGES))
    r = RANGES[kind]

    def log_uniform(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    n = int(round(log_uniform(*r["n"])))
    n2 = int(round(log_uniform(*r["n2"])))
    if kind == "densmore":
        n2 = rng.randint(4, 40)
    c = dict(kind=kind, n=n, n2=n2, scale=round(log_uniform(*r["scale"]), 3), fp64=rng.random() < 0.2,
             steps=rng.randint(1, 4), warm=2, stepping="resident")
    if kind == "batch":
        c["steps"] = 1
    if kind == "slab":
        c["stepping"] = rng.choice(["resident", "noalloc", "exchange"])
        if c["stepping"] == "exchange":
            c["steps"] = 1
        elif c["stepping"] == "noalloc":  # its fixed scratch holds about 1e5 packets in FP64
            c["scale"] = min(c["scale"], 0.5)
    return c


@functools.lru_cache(maxsize=3)
def _mesh(n, slab):
    """A tessellation (a program reads or builds its mesh once, whatever it then runs on it)."""
    if slab:
        return P.voronoi_slab(n=n).umesh
    return P.voronoi_mesh(P.voronoi_points(n, 0xC4))


@functools.lru_cache(maxsize=2)
def _batch(n, scale):
    return P.c5_batch(P.c5_instances(n, seed=1, packets_scale=scale, cells_range=(50, 600)))


def _spec(case, seed):
    kind, n, n2, s = case["kind"], case["n"], case["n2"], case["scale"]
    if kind == "slab":  # 1000 packets a cell at scale 1, whatever the cells
        return P.c1_slab(seed=seed, nx=n, packets_scale=s)
    if kind == "marshak":  # the wave's early nanoseconds, its bath at 0.2 ns
        spec = P.marshak(2, nx=n, seed=seed, new_photons=max(1, int(15 * s)), boundary_photons=int(100 * s), dt=2e-13)
        spec.source_T = P.marshak_bath_T(2, 2e-10)
        spec.comb_nmin = max(1, int(15 * s))
        return spec
    if kind == "densmore":
        spec = P.densmore(nx=n, seed=seed, groups=n2, new_photons=max(1, int(16 * s)),
                          boundary_photons=max(1, int(100 * s)), comb_nmin=max(1, int(200 * s)))
        spec.eg_time_avg = True
        return spec
    if kind == "cube":  # the packets of the 64^3 benchmark; smaller cubes keep them per cell
        return P.c2_cube(seed=seed, n=n, literal=True, packets_scale=s, source_per_face=2400, comb_nmin=8)
    if kind == "step_slab":
        return P.c3_step(seed=seed, nx=n, nyz=n2, packets_scale=s)
    if kind == "voronoi_groups":
        spec = P.c4_voronoi(seed=seed, n=n, groups=n2, mesh=_mesh(n, False), packets_scale=s)
        # the source's packets in proportion to the mesh (1e7 on 2e5 cells)
        spec.source_per_face = max(1, int(round(spec.source_per_face * n / 200000)))
        return spec
    if kind == "voronoi_thick":
        m = _mesh(n, True)
        x = m.mesh_point[:, 0]
        N = m.ncells
        spec = P.voronoi_slab(seed=seed, n=200, thick=True, packets_scale=s)
        spec.umesh = m
        spec.sigma_a0 = np.where(x < 0.5, 3.0, 2e3)
        spec.sigma_s0 = np.where(x < 0.5, 0.0, 2e3)
        spec.T0 = np.full(N, 0.05 * P.KEV_K)
        return spec
    return _batch(n, s).with_seed(seed)


def _material(spec):
    """What a host code with its own opacities and equation of state hands the engine (the gray slab)."""
    N = spec.ncells
    T = np.linspace(1.0, 0.05, N) * P.KEV_K
    return dict(T=T, sigma_a=spec.sigma_a0.copy(), sigma_s=np.zeros(N), cv=np.full(N, spec.eos_f),
                e=spec.eos_f * T * spec.volumes())


def prepare(case, seed):
    spec = _spec(case, seed)
    st = dict(case=case, spec=spec)
    exchange = case["stepping"] == "exchange"
    eng = GpuEngine(spec, capi.FP64 if case["fp64"] else capi.MIXED,
                    capi.MATERIAL_HOST if exchange else capi.MATERIAL_DEVICE)
    st["engine"] = eng
    if exchange:
        st["material"] = _material(spec)
        eng.set_cell_state(**st["material"])
    for _ in range(case["warm"]):
        eng.step()
    if exchange:
        st["particles"] = eng.export_census()
        # the host's particle arrays, sized once for what population control can leave
        room = 4 * spec.ncells * spec.comb_nmin
        st["rows"], st["row_cells"] = np.zeros((room, 8)), np.full(room, -1, dtype=np.int64)
    return st


def run(st):
    case, eng = st["case"], st["engine"]
    out = {}
    if case["stepping"] == "exchange":
        eng.set_cell_state(**st["material"])
        eng.import_census(st["particles"])
        eng.step()
        words = np.ascontiguousarray(eng.export_census()).view(np.float64).reshape(-1, 10)
        k = len(words)
        st["rows"][:k] = words[:, :8]  # position, velocity, weight, frequency
        st["rows"][k:] = 0.0
        st["row_cells"][:k] = words.view(np.int64)[:, 8]
        st["row_cells"][k:] = -1
        out["particles"], out["particle_cells"] = st["rows"], st["row_cells"]
    else:
        step = eng.step_noalloc if case["stepping"] == "noalloc" else eng.step
        for _ in range(case["steps"]):
            step()
    out["cells"] = eng.cells()
    counters = eng.counters()
    out["counts"] = {k: int(counters[k]) for k in COUNTS}
    if case["kind"] == "densmore":
        out["groups"] = eng.group_erad(case["n2"])
    return out


def _packets(case):
    """(cells, packets a step starts with, census after it), about, from the problem's own budgets."""
    n, n2, s, kind = case["n"], case["n2"], case["scale"], case["kind"]
    if kind == "slab":
        return n, 25000 * s + n * (250 + 500) * s, 500 * n * s
    if kind == "marshak":
        return n, 100 * s + n * 15 * s * (10 + 6), n * 15 * s * 6
    if kind == "densmore":
        return n, 100 * s + n * s * (160 + 1000), n * s * 1000
    if kind == "cube":
        face = 2400 * s * (64.0 / n)
        return n ** 3, n * n * face + n ** 3 * s * 28, n ** 3 * s * 10
    if kind == "step_slab":
        return n * n2 * n2, n2 * n2 * 4000 * s + n * n2 * n2 * 220 * s, n * n2 * n2 * 20 * s
    if kind == "voronoi_groups":
        return n, n * s * (50 + 100 + 120), n * s * 120
    if kind == "voronoi_thick":
        return n, s * (400 * n ** (2 / 3) + n * (80 + 24)), n * s * 24
    return 200 * n, 2.2e5 * n * s * 1.5, 2.2e5 * n * s * 0.75


def work(case):
    """A step reads its census and the cells' state and writes both; a packet
    takes some segments of about 150 operations each (a counter-based random
    block, three face distances, a logarithm, an exponential)."""
    cells, packets, census = _packets(case)
    size = 80 if case["fp64"] else 48
    per_step = 2 * size * census + 8 * 12 * cells
    flops = 150.0 * packets * RANGES[case["kind"]]["segments"]
    return dict(bytes=case["steps"] * per_step, flops=case["steps"] * flops)


def exact(case, seed):
    """The tallies of a Monte Carlo step have no exact value.  In the exchange
    the step's temperatures are the caller's own, so its Fleck factors and
    opacities follow from them."""
    if case["stepping"] != "exchange":
        return None
    spec = _spec(case, seed)
    m = _material(spec)
    beta = 4.0 * P.ARAD * m["T"] ** 3 * m["sigma_a"] * P.CLIGHT * spec.dt / m["cv"]
    cells = dict.fromkeys(CELLS)
    cells["fleck"] = 1.0 / (1.0 + beta)
    cells["sigma_p"] = m["sigma_a"]
    return dict(particles=None, particle_cells=None, cells=cells, counts=dict.fromkeys(COUNTS))
