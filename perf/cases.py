"""Performance cases of the coagulation library: what its users run.

A host model owns its particles between output times, so most cases are one
output interval of such a model: the particles of every box go to the device
(:meth:`CoagGPU.load_population`), a number of coagulation timesteps runs, and
the evolved particles come back.  The workloads are the package's own
(``partmc_amd.populations``), at sizes from a few thousand particles in one
box to millions over a batch of boxes.  The remaining cases are the in-situ
size distributions that a program takes of particles that stay on the device.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges,
``prepare`` makes inputs from a seed, ``run`` is one pass, ``work`` states the
bytes and operations a pass cannot do without and ``exact`` the value of the
outputs that have a closed form.  Monte Carlo outputs have none: they follow
from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import partmc_amd
from partmc_amd import populations as P

MODES = {"exact": partmc_amd.MODE_EXACT, "parallel": partmc_amd.MODE_PARALLEL}
PRECISIONS = {"fp64": partmc_amd.PREC_FP64, "fp32": partmc_amd.PREC_FP32_RECHECK}
# kernel and timestep of each family's configuration
KERNEL = {"golovin": P.KERNEL_ADDITIVE, "brown": P.KERNEL_BROWN, "classes": P.KERNEL_BROWN,
          "species": P.KERNEL_BROWN, "boxes": P.KERNEL_BROWN, "drops": P.KERNEL_SEDI,
          "scenario": P.KERNEL_BROWN}
DEL_T = {"golovin": 1.0, "brown": 60.0, "classes": 60.0, "species": 600.0, "boxes": 30.0,
         "drops": 1.0, "scenario": 60.0}
N_SPEC = {"golovin": 1, "brown": 4, "classes": 2, "species": 20, "boxes": 4, "drops": 1,
          "scenario": 4, "dist": 4}
# families whose evolved state comes back whole (every particle field and the
# removal log); the larger ones take identifiers and species volumes
WHOLE = ("golovin", "brown", "classes", "scenario")
D_MIN, D_MAX = 1e-9, 1e-4  # diameters of the size distributions


def listed():
    return [
        # the size distribution of a small resident box into the caller's
        # device memory: one output of an interactive or coupled run
        dict(name="dist small", family="dist", n_part=20000, n_bin=60, noalloc=True),
        # the same of a large box, the number, mass and volume distributions
        # that a run writes at each output time
        dict(name="dist large", family="dist", n_part=1500000, n_bin=160, noalloc=False),
        # the additive kernel against its analytic solution at the smallest
        # size in use: every step is bound by launches
        dict(name="golovin small", family="golovin", n_part=2001, steps=10, mode="parallel",
             precision="fp64"),
        # the same in the default mode, sequential-order replay: a parity or
        # regression run against the sequential algorithm
        dict(name="golovin exact", family="golovin", n_part=10000, steps=20, mode="exact",
             precision="fp64"),
        # the additive test at its usual size
        dict(name="golovin 1e5", family="golovin", n_part=100000, steps=20, mode="parallel",
             precision="fp32"),
        # Brownian coagulation under power weighting in the replay mode, with
        # bin pairs on the per-particle path
        dict(name="brown exact", family="brown", n_part=20000, steps=2, mode="exact",
             precision="fp64"),
        # one box of a Brownian aerosol, trimodal, power weights
        dict(name="brown 1e5", family="brown", n_part=100000, steps=30, mode="parallel",
             precision="fp32"),
        # two weight classes in plain FP64 at an odd size
        dict(name="brown classes", family="classes", n_part=9001, steps=8, mode="parallel",
             precision="fp64"),
        # many species a particle
        dict(name="brown 20 species", family="species", n_part=150000, steps=4, mode="parallel",
             precision="fp32"),
        # a batch of uneven boxes, as the columns of a regional model
        dict(name="brown boxes", family="boxes", n_box=28, n_min=10000, n_max=300000, steps=20,
             mode="parallel", precision="fp32"),
        # cloud and drizzle drops under sedimentation: chains on large drops
        dict(name="drops", family="drops", n_box=6, n_part=300000, steps=20, mode="parallel",
             precision="fp32"),
        # the whole particle timestep of a scenario: dilution, emissions,
        # coagulation and population control
        dict(name="scenario", family="scenario", n_box=6, n_part=20000, n_emit=150, steps=5,
             mode="parallel", precision="fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["dist", "golovin", "brown", "classes", "species", "boxes", "drops",
                         "scenario"])
    case = dict(family=family)
    if family == "dist":
        case.update(n_part=_log_int(rng, 2000, 1500000), n_bin=_log_int(rng, 30, 400),
                    noalloc=rng.random() < 0.5)
        return case
    exact = family in ("golovin", "brown") and rng.random() < 0.3
    case.update(mode="exact" if exact else "parallel",
                precision="fp64" if exact else rng.choice(["fp32", "fp32", "fp64"]))
    if family == "golovin":
        case.update(n_part=_log_int(rng, 2000, 20000 if exact else 150000),
                    steps=rng.randint(8, 20))
    elif family == "brown":
        case.update(n_part=_log_int(rng, 2000, 20000 if exact else 100000),
                    steps=2 if exact else rng.randint(6, 30))
    elif family == "classes":
        case.update(n_part=_log_int(rng, 2000, 20000), steps=rng.randint(4, 10))
    elif family == "species":
        case.update(n_part=_log_int(rng, 10000, 150000), steps=rng.randint(2, 8))
    elif family == "boxes":
        lo = _log_int(rng, 5000, 20000)
        case.update(n_box=rng.randint(3, 28), n_min=lo, n_max=_log_int(rng, 2 * lo, 300000),
                    steps=rng.randint(4, 20))
    elif family == "drops":
        case.update(n_box=rng.randint(1, 6), n_part=_log_int(rng, 20000, 300000),
                    steps=rng.randint(4, 20))
    else:
        case.update(n_box=rng.randint(1, 6), n_part=_log_int(rng, 3000, 20000),
                    n_emit=rng.randint(20, 300), steps=rng.randint(2, 5))
    return case


def _two_classes(seed, n):
    """Species volumes and weight classes of a box with two flat weight
    classes, nine tenths of the particles in the first."""
    rng = np.random.default_rng(seed)
    vol = 10 ** rng.uniform(-24, -21, size=(n, 1)) * rng.dirichlet([1, 1], size=n)
    klass = np.where(rng.uniform(size=n) < 0.9, 1, 2).astype(np.int32)
    return vol, klass


def _box_sizes(case):
    """Particles of each box of a batch: log-spaced from n_min to n_max."""
    sizes = np.geomspace(case["n_min"], case["n_max"], case["n_box"])
    return [int(round(n)) for n in sizes]


def _populations(case, seed):
    family = case["family"]
    if family == "golovin":
        pop = P.config_c1prime(seed=seed, n_part=case["n_part"])
        pop.grid = (160, 0.5e-8, 0.5e-3)
        return [pop]
    if family in ("brown", "dist"):
        return [P.config_c2(seed=seed, n_part=case["n_part"])]
    if family == "species":
        return [P.config_c3(seed=seed, n_part=case["n_part"])]
    if family == "boxes":
        return [P.config_c4(seed=1000 * seed + b, n_box=1, n_min=n, n_max=n)[0]
                for b, n in enumerate(_box_sizes(case))]
    if family == "drops":
        return P.config_c5(seed=seed, n_box=case["n_box"], n_part=case["n_part"])
    return [P.config_c2(seed=1000 * seed + b, n_part=case["n_part"])
            for b in range(case["n_box"])]


def prepare(case, seed):
    family = case["family"]
    state = dict(case=case, seed=seed)
    if family == "classes":
        n = case["n_part"]
        vol, klass = _two_classes(seed, n)
        # the concentrations of 6000 such particles at 9e7 and 3e7 m^-3 each
        state.update(vol=vol, klass=klass, ids=np.arange(1, n + 1), group=np.ones(n, np.int32),
                     magnitude=[[9e7 * 6000 / n, 3e7 * 6000 / n]])
        g = partmc_amd.CoagGPU(1, np.array([1800.0, 1000.0]))
        capacity = [3 * n]
    else:
        pops = _populations(case, seed)
        g = partmc_amd.CoagGPU(len(pops), pops[0].density)
        slack = 1.6 if family == "scenario" else 1.25
        capacity = [int(slack * p.n_part) + 4096 for p in pops]
        state["pops"] = pops
    g.reserve(capacity)
    if family == "scenario":
        # particles that emissions add to each box in each step
        state["emitted"] = [[P.config_c2(seed=100000 + 1000 * seed + 64 * s + b,
                                         n_part=case["n_emit"]).vol
                             for b in range(case["n_box"])] for s in range(case["steps"])]
    if family == "dist":
        # resident particles: the distributions are taken of them where they are
        g.load_population(0, state["pops"][0])
        if case["noalloc"]:
            state["hist"] = [torch.zeros(case["n_bin"], dtype=torch.float64, device="cuda")
                             for _ in range(2)]
    else:
        g.set_mode(MODES[case["mode"]], PRECISIONS[case["precision"]], 1e-5)
        state["buf"] = [_buffers(case, c, g.n_spec) for c in capacity]
        state["last"] = [[0, 0] for _ in capacity]
    state["g"] = g
    return state


def _buffers(case, capacity, n_spec):
    """The host model's arrays of one box, as large as its capacity."""
    i4, i8, f8 = np.int32, np.int64, np.float64
    fields = dict(vol=((capacity, n_spec), f8), id=((capacity,), i8))
    if case["family"] in WHOLE:
        fields.update(group=((capacity,), i4), klass=((capacity,), i4),
                      n_primary=((capacity,), i4), n_comp=((capacity,), i4))
        if case["family"] != "scenario":
            comp = (capacity, partmc_amd.MAX_COMP)
            fields.update(comp_source=(comp, i4), comp_time=(comp, f8), least=((capacity,), f8),
                          greatest=((capacity,), f8), removed_id=((capacity + 64,), i8),
                          removed_action=((capacity + 64,), i4),
                          removed_other=((capacity + 64,), i8))
    return {k: np.zeros(shape, dtype=t) for k, (shape, t) in fields.items()}


FIELDS = ("vol", "id", "group", "klass", "n_primary", "n_comp", "comp_source", "comp_time",
          "least", "greatest")
REMOVED = ("removed_id", "removed_action", "removed_other")


def _check(code):
    if code:
        raise RuntimeError(partmc_amd.load().pmc_gpu_last_error().decode())


def _download(g, box, buf, last):
    """The box's particles (and its removal log) into the host model's own
    arrays through the C ABI, as its Fortran binding calls it; rows past the
    particle count are zero.  last holds the counts of the download before."""
    lib = partmc_amd.load()
    n = np.zeros(1, dtype=np.int32)
    at = [buf[f].ctypes.data if f in buf else None for f in FIELDS]
    _check(lib.pmc_gpu_download(g._h, box, len(buf["id"]), n.ctypes.data, *at))
    for f in FIELDS:
        if f in buf:
            buf[f][n[0]:last[0]] = 0
    if REMOVED[0] in buf:
        m = np.zeros(1, dtype=np.int32)
        at = [buf[f].ctypes.data for f in REMOVED]
        _check(lib.pmc_gpu_get_removed(g._h, box, len(buf[REMOVED[0]]), m.ctypes.data, *at))
        for f in REMOVED:
            buf[f][m[0]:last[1]] = 0
        last[1] = m[0]
    last[0] = n[0]
    return n[0]


def _run_dist(state):
    g, case = state["g"], state["case"]
    n_bin = case["n_bin"]
    if case["noalloc"]:
        for h, quantity in zip(state["hist"], ("num", "mass")):
            g.size_dist_noalloc(0, n_bin, D_MIN, D_MAX, h.data_ptr(), quantity)
        g.sync()
        return state["hist"]
    return [g.size_dist(0, n_bin, D_MIN, D_MAX, q) for q in ("num", "mass", "vol")]


def run(state):
    case, g = state["case"], state["g"]
    family = case["family"]
    if family == "dist":
        return _run_dist(state)
    kernel, dt, steps = KERNEL[family], DEL_T[family], case["steps"]
    g.set_rng(state["seed"], 0)
    if family == "classes":
        g.set_env(0, 288.0, 1e5)
        g.set_weights(0, [[1, 1]], state["magnitude"], [[0.0, 0.0]])
        g.upload(0, state["vol"], state["ids"], state["group"], state["klass"])
        g.set_next_id(0, case["n_part"] + 1)
        g.set_bin_grid(0, 60, 1e-10, 1e-5)
    else:
        for b, pop in enumerate(state["pops"]):
            g.load_population(b, pop)
    n_box = g.n_box
    counts = []
    if family == "scenario":
        for b in range(n_box):
            g.set_n_part_ideal(b, 0.45 * case["n_part"])  # the first call halves each box
        for s in range(steps):
            g.dilute(np.full(n_box, 0.01))
            for b, vol in enumerate(state["emitted"][s]):
                one = np.ones(len(vol), np.int32)
                g.append(b, vol, one, one)
            counts.append(g.mc_coag(kernel, dt))
            g.rebalance()
    elif family in ("boxes", "drops"):
        # a batch steps without a host read of its counts each step
        g.reset_counters()
        for _ in range(steps):
            g.mc_coag_async(kernel, dt)
        g.sync()
        c = g.counters()
        counts.append((c["n_samp"], c["n_coag"]))
    else:
        for _ in range(steps):
            counts.append(g.mc_coag(kernel, dt))
    out = dict(n_samp=np.array([c[0] for c in counts]), n_coag=np.array([c[1] for c in counts]))
    out["n_part"] = np.array([_download(g, b, state["buf"][b], state["last"][b])
                              for b in range(n_box)])
    out["boxes"] = state["buf"]
    return out


def work(case):
    """Bytes in and out of a pass: particles as they are uploaded (volumes,
    identifier, group and class) and as they come back, or read once for each
    distribution; operations: the kernel terms of every particle once."""
    family = case["family"]
    ns = N_SPEC[family]
    if family == "dist":
        n = case["n_part"]
        k = 2 if case["noalloc"] else 3
        return {"bytes": k * (n * (8.0 * ns + 4) + 8 * case["n_bin"]), "flops": 60.0 * k * n}
    if family == "boxes":
        n = float(sum(_box_sizes(case)))
    else:
        n = float(case.get("n_box", 1) * case["n_part"])
    into = 8.0 * ns + 16
    # vol, id, group, class, primaries, component count, 20 components and
    # their times, two create times; or volumes and identifiers
    if family not in WHOLE:
        back = 8.0 * ns + 8
    elif family == "scenario":
        back = 8.0 * ns + 16
    else:
        back = 8.0 * ns + 8 + 4 * 4 + 20 * 12 + 16
    return {"bytes": n * (into + back), "flops": 100.0 * n}


def exact(case, seed):
    """The distributions of a resident box in plain numpy; Monte Carlo
    outputs have no value of their own."""
    if case["family"] != "dist":
        return None
    pop = _populations(case, seed)[0]
    v = pop.vol.sum(axis=1)
    mass = pop.vol @ pop.density
    d = 2.0 * (3.0 * v / (4.0 * np.pi)) ** (1.0 / 3.0)
    n_bin = case["n_bin"]
    width = (math.log(D_MAX) - math.log(D_MIN)) / n_bin
    b = np.floor((np.log(d) - math.log(D_MIN)) / width).astype(np.int64)
    b[d == D_MAX] = n_bin - 1
    inside = (b >= 0) & (b < n_bin)
    w = pop.weight_magnitude * (0.5 * d) ** pop.weight_exponent / width
    weights = {"num": w, "mass": w * mass, "vol": w * v}
    names = ("num", "mass") if case["noalloc"] else ("num", "mass", "vol")
    return [np.bincount(b[inside], weights=weights[q][inside], minlength=n_bin) for q in names]
