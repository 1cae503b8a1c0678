"""The work that a user of this framework has it do, as cases to be timed.

A case is a model on a lattice and a number of steps between two looks at it:
one pass advances the solver (or the ensemble) by that many steps through its
public calls and then takes what a simulation script takes there, the species
counts and a frame of the lattice on the device.  A pass goes on from where the last one
ended, as a trajectory does.

Models are the package's own builders (bimolecular, MinD/MinE capsule,
whole cell) and one constitutive expression model with a zero-order reaction.
The structure of a model (site types, reaction network, diffusion constants)
is fixed per case; the particles' places and species and the solver's seed
come from the seed.
"""
from __future__ import annotations

import dataclasses
import math

import numpy as np
import torch

import lattice_microbes_amd as lmx
from lattice_microbes_amd import models
from lattice_microbes_amd.solver import DeviceHookLattice


def listed():
    return [
        # The smallest lattice of the ensemble workload, one write interval.
        {"name": "bimolecular_32", "kind": "bimolecular", "X": 32, "Y": 32, "Z": 32, "P": 8, "n": 2000, "steps": 100},
        # The plain MPD benchmark model under a hook every 10 steps: the
        # shortest calls, where launches and synchronisation count.
        {"name": "bimolecular_64_hook", "kind": "bimolecular", "X": 64, "Y": 64, "Z": 64, "P": 8, "n": 2000, "steps": 10},
        # The same model between two writes of the species counts.
        {"name": "bimolecular_64", "kind": "bimolecular", "X": 64, "Y": 64, "Z": 64, "P": 8, "n": 2000, "steps": 200},
        # A bacterium with the membrane oscillator (2 um at 16 nm).
        {"name": "capsule", "kind": "capsule", "X": 128, "Y": 128, "Z": 256, "P": 8, "n": 15000, "steps": 50},
        # The same scheme on a lattice cut to the cell: odd extents.
        {"name": "capsule_odd", "kind": "capsule", "X": 63, "Y": 61, "Z": 151, "P": 8, "n": 9000, "steps": 50},
        # Constitutive expression: zero-order births, so that empty sites react.
        {"name": "expression", "kind": "expression", "X": 96, "Y": 96, "Z": 96, "P": 8, "n": 45000, "steps": 40},
        # Crowded: half a particle per site, 16 slots.
        {"name": "crowded_p16", "kind": "bimolecular", "X": 128, "Y": 64, "Z": 80, "P": 16, "n": 330000, "steps": 40},
        # The whole cell as it is served (a quarter of the full lattice).
        {"name": "cell_reduced", "kind": "cell", "X": 256, "Y": 256, "Z": 128, "P": 8, "nS": 30, "R": 90, "n": 250000, "steps": 20},
        # More than 255 species: the uint32 lattice.
        {"name": "cell_uint32", "kind": "cell", "X": 256, "Y": 256, "Z": 128, "P": 8, "nS": 300, "R": 900, "n": 250000,
         "words": True, "steps": 10},
        # The whole-cell benchmark model.
        {"name": "whole_cell", "kind": "cell", "X": 256, "Y": 256, "Z": 512, "P": 8, "nS": 100, "R": 300, "n": 1000000, "steps": 20},
        # Replicates of the bimolecular model on lattices of 32^3 to 128^3,
        # stepped as one ensemble.
        {"name": "ensemble", "kind": "ensemble", "n": 128, "P": 8, "steps": 100},
        # What a server holds at one time: bimolecular 64^3, capsules and
        # reduced whole cells, stepped as one ensemble.
        {"name": "serving", "kind": "serving", "n": 12, "P": 8, "steps": 20},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["bimolecular", "bimolecular", "capsule", "expression", "cell", "cell", "words", "ensemble", "serving"])
    P = rng.choice([8, 8, 8, 4, 16])
    if kind == "ensemble":
        return {"kind": kind, "n": int(_log(rng, 8, 64)), "P": P, "steps": int(_log(rng, 20, 100))}
    if kind == "serving":
        return {"kind": kind, "n": rng.randint(4, 14), "P": 8, "steps": rng.randint(10, 30)}
    words = kind == "words"
    if words:
        kind, P = "cell", 8
    # extents: mostly multiples of 4, as lattices are laid out, sometimes any
    step = rng.choice([4, 4, 8, 1])
    sites = _log(rng, 3e4, 4e6) if kind in ("bimolecular", "capsule", "expression") else _log(rng, 2.6e5, 8e6)
    edge = sites ** (1 / 3)
    aspect = rng.uniform(1.0, 2.5)
    ext = lambda v: max(16, int(v / step) * step)  # noqa: E731
    X, Y, Z = ext(edge / aspect ** (1 / 3)), ext(edge / aspect ** (1 / 3)), ext(edge * aspect ** (2 / 3))
    N = X * Y * Z
    case = {"kind": kind, "X": X, "Y": Y, "Z": Z, "P": P, "steps": int(_log(rng, 10, 100))}
    if kind == "bimolecular":
        case["n"] = int(N * _log(rng, 1e-3, 0.02 * P if P > 4 else 0.05))
    elif kind == "capsule":
        # the membrane, a thin shell, gathers most of the particles
        case["n"], case["P"] = int(N * _log(rng, 1e-3, 4e-3)), max(P, 8)
    elif kind == "expression":
        case["n"] = int(N * _log(rng, 3e-3, 0.06))
    else:
        case["n"] = int(N * _log(rng, 5e-3, 0.035))
        nS = rng.randint(256, 320) if words else rng.randint(20, 120)
        case["nS"], case["R"] = nS, 3 * nS
        if words:
            case["words"] = True
    return case


# ------------------------------------------------------------------ models
def _expression(shape, P, n):
    """A -> B -> nothing with constitutive production of A (steady state with
    n particles, half of each species): births happen at empty sites too."""
    N = shape[0] * shape[1] * shape[2]
    tau, spacing = 50e-6, 32e-9
    kd = 2.0                                    # 1/s, both A -> B and B -> nothing
    types = np.array([0, 1, 1], np.uint32)
    K = np.array([kd * n / 2.0, kd, kd])        # molecules/s over the lattice, 1/s
    S = np.array([[1, -1, 0], [0, 1, -1]], np.int32)
    D = np.array([[0, 1, 0], [0, 0, 1]], np.uint32)
    DF = np.zeros((2, 2, 2))
    DF[:, :, 0], DF[:, :, 1] = 1e-12, 5e-13
    RL = np.ones((3, 2), np.uint32)
    X, Y, Z = shape
    sites = np.zeros(shape, np.uint8)
    sites[X // 4:3 * X // 4, Y // 4:3 * Y // 4, Z // 4:3 * Z // 4] = 1  # a nucleoid block
    return models.ModelSpec("expression", shape, spacing, tau, P, 2, 2, types, K, S, D, DF, RL,
                            np.zeros(shape + (P,), np.uint8), sites, "periodic")


_structures = {}


def _structure(kind, shape, P, n, nS, R):
    """The seed-independent part of a model: a ModelSpec, the allowed sites of
    its particles (row-major indices) and their species' weights."""
    key = (kind, shape, P, n, nS, R)
    if key in _structures:
        return _structures[key]
    N = shape[0] * shape[1] * shape[2]
    weights = None
    if kind == "bimolecular":
        spec = models.bimolecular(shape=shape, P=P, nA=0, nB=0, seed=1)
        weights = (0.5, 0.5, 0.0)
    elif kind == "capsule":
        spec = models.capsule_minde(shape=shape, spacing=16e-9 * 128 / min(128, shape[0], shape[1], shape[2] // 2 + 1),
                                    P=P, counts=(0, 0, 0), seed=1)
        weights = (0.4, 0.4, 0.2, 0.0, 0.0)
    elif kind == "expression":
        spec = _expression(shape, P, n)
    else:
        spec = models.whole_cell(shape=shape, P=P, nS=nS, R=R, n_particles=0, seed=1)
    flat = spec.sites.reshape(-1)
    if kind == "capsule":
        allowed = np.flatnonzero(flat == 2)
    elif kind == "cell":
        allowed = np.flatnonzero((flat != 0) & (flat != 1) & (flat != 3))
    else:
        allowed = N
    spec.lattice = np.zeros(shape + (0,), np.uint8)  # made per seed
    _structures[key] = (spec, allowed, weights)
    return _structures[key]


def _model(case, seed):
    shape = (case["X"], case["Y"], case["Z"])
    spec, allowed, weights = _structure(case["kind"], shape, case["P"], case["n"], case.get("nS", 0), case.get("R", 0))
    rng = np.random.default_rng([seed, 7])
    n, P = case["n"], case["P"]
    at = rng.integers(0, allowed, n) if isinstance(allowed, int) else allowed[rng.integers(0, allowed.size, n)]
    sp = rng.integers(1, spec.nS + 1, n) if weights is None else rng.choice(spec.nS, n, p=weights) + 1
    lattice = np.zeros((shape[0] * shape[1] * shape[2], P), np.uint32 if case.get("words") else np.uint8)
    lattice[at, rng.integers(0, P, n)] = sp  # the solver packs each site's slots
    return dataclasses.replace(spec, lattice=lattice.reshape(shape + (P,)))


def _solver(spec, replicate, seed):
    s = (lmx.IntMpdRdmeSolver if spec.lattice.dtype == np.uint32 else lmx.MpdRdmeSolver)(0)
    spec.load_into(s, replicate=replicate, seed=1 + seed % 30000)
    return s


_EDGES = (32, 48, 64, 96, 128)


def _members(case):
    """The members of an ensemble: one single-solver case each."""
    if case["kind"] == "ensemble":
        # the lattice sizes in turn, so that any number of replicates has them all
        return [{"kind": "bimolecular", "X": e, "Y": e, "Z": e, "P": case["P"], "n": 2000}
                for e in (_EDGES[r % len(_EDGES)] for r in range(case["n"]))]
    mix = []
    for r in range(case["n"]):
        if r % 6 == 5:
            mix.append({"kind": "cell", "X": 256, "Y": 256, "Z": 128, "P": 8, "nS": 30, "R": 90, "n": 250000})
        elif r % 3 == 1:
            mix.append({"kind": "capsule", "X": 128, "Y": 128, "Z": 256, "P": 8, "n": 15000})
        else:
            mix.append({"kind": "bimolecular", "X": 64, "Y": 64, "Z": 64, "P": 8, "n": 2000})
    return mix


def prepare(case, seed):
    lmx.torch_interop()
    if case["kind"] in ("ensemble", "serving"):
        # replicates of one model start from the same particles, each with a
        # seed of its own
        specs, solvers = {}, []
        ens = lmx.Ensemble(0)
        for r, m in enumerate(_members(case)):
            key = tuple(sorted(m.items()))
            if key not in specs:
                specs[key] = _model(m, seed)
            solvers.append(_solver(specs[key], r, seed))
            ens.add(solvers[-1])
        shapes = {}
        for s in solvers:
            shapes.setdefault(s.shape, []).append(DeviceHookLattice(s))
        return {"ensemble": ens, "solvers": solvers, "views": list(shapes.values()), "steps": case["steps"]}
    s = _solver(_model(case, seed), 0, seed)
    return {"solver": s, "view": DeviceHookLattice(s), "steps": case["steps"]}


def run(state):
    if "ensemble" in state:
        state["ensemble"].run(state["steps"])
        counts = [s.getSpeciesCounts() for s in state["solvers"]]
        lattices = []
        for views in state["views"]:  # the replicates of one lattice size together
            for v in views:
                v.refresh()
            lattices.append(torch.stack([v.getParticleLatticeView() for v in views]))
        views[0].synchronize()  # the copies are done before the next step
        return {"counts": np.concatenate(counts), "lattices": lattices}
    s = state["solver"]
    s.runTimesteps(state["steps"])
    counts = s.getSpeciesCounts()
    view = state["view"]
    view.refresh()
    # A frame of its own: the view is the solver's buffer, which goes on to the
    # next step (and away with the solver).
    frame = view.getParticleLatticeView().clone()
    view.synchronize()
    return {"counts": counts, "lattice": frame}


def work(case):
    """A step reads every site's particles and type once and writes its
    particles once; a pass also writes the counts.  Integer operations: about
    60 per particle and axis for its random number and its move."""
    if case["kind"] in ("ensemble", "serving"):
        parts = [work(dict(m, steps=case["steps"])) for m in _members(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    N = case["X"] * case["Y"] * case["Z"]
    slot = 4 if case.get("words") else 1
    return {"bytes": float(case["steps"] * N * (2 * case["P"] * slot + 1)), "flops": float(case["steps"] * case["n"] * 180)}


def exact(case, seed):
    """Every output is whole numbers, which are compared bit for bit."""
    return None
