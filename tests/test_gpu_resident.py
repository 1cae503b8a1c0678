"""Resident runs: a solver of few particles steps inside one block for a whole
lmx_run_steps call (four steps or more), its particles as records in LDS.
Every case is compared word for word with the oracle.

Where it can go wrong: extents of one and two (a site is its own neighbour, or
both neighbours are one site), both boundaries, every slot count and the
uint32 lattice, sites of several particles and their reactions, overflow
entries with both handlers, more than one record per thread, particles that
multiply past the block's capacity, lattices filled on the device past it, and
runs enqueued behind one that stopped short."""
import numpy as np
import pytest

import lattice_microbes_amd as lmx
from lattice_microbes_amd import models
from lattice_microbes_amd.solver import DeviceHookLattice
import oracle

pytestmark = pytest.mark.gpu


class RelaxedInt(lmx.IntMpdRdmeSolver):
    _parses_overflow_handler = True


CASES = [
    # shape, P, boundary, particles per slot, overflow handler
    ((8, 8, 8), 8, "periodic", 0.1, "classic"),
    ((1, 9, 30), 8, "periodic", 0.1, "classic"),
    ((2, 1, 40), 8, "reflecting", 0.2, "classic"),
    ((7, 5, 3), 4, "periodic", 0.3, "classic"),
    ((13, 11, 9), 16, "reflecting", 0.1, "classic"),
    ((33, 20, 17), 8, "periodic", 0.03, "classic"),     # more records than threads
    ((10, 9, 8), 8, "periodic", 0.42, "classic"),       # overflow entries in every step
    ((10, 9, 8), 8, "reflecting", 0.42, "relaxed"),
    ((12, 8, 8), 4, "periodic", 0.5, "relaxed"),
    ((64, 64, 64), 8, "reflecting", 0.001, "classic"),
]


@pytest.mark.parametrize("words", [False, True], ids=["byte", "uint32"])
@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}-P{c[1]}-{c[2]}-{c[4]}" for c in CASES])
def test_resident_runs_match_oracle(gpu, case, words):
    shape, P, boundary, density, handler = case
    spec = models.random_model(shape=shape, P=P, nS=6, nST=3, R=9, density=density, seed=51, boundary=boundary,
                               include_zero_order=False)
    assert int(spec.initial_counts().sum()) <= 3000
    if words:
        spec.lattice = spec.lattice.astype(np.uint32)
    orc = oracle.Oracle(spec, seed_top=7, replicate=2, overflow=handler)
    s = (RelaxedInt if words else lmx.MpdRdmeSolver)(0)
    spec.load_into(s, replicate=2, seed=7, extra={"rdme.mpd.overflowhandler": handler})
    for chunk in (4, 1, 9):  # the middle one is no resident run
        s.runTimesteps(chunk)
        assert orc.run(chunk) == 0
        got = s.getLatticeNative()
        assert np.array_equal(got, orc.native()), f"{(got != orc.native()).sum()} words differ"
        assert s.timestep == orc.timestep
        assert s.getOverflowStats() == (orc.stats.overflow_entries, orc.stats.overflow_steps)
        assert s.getUnresolvedOverflows() == orc.unresolved
    s.close()


def _splitting(n, rate):
    """A -> A + A: the particles multiply."""
    spec = models.bimolecular(shape=(24, 20, 18), nA=n, nB=0, seed=5, boundary="periodic")
    spec.types, spec.K = np.array([1], np.uint32), np.array([rate])
    spec.S, spec.D = np.array([[1], [0], [0]], np.int32), np.array([[1], [0], [0]], np.uint32)
    spec.RL = np.ones((1, 1), np.uint32)
    return spec


@pytest.mark.parametrize("calls", [1, 4])
def test_particles_multiply_past_the_block(gpu, calls):
    """The run stops with the step in which the block is full and the missing
    steps run otherwise, also when further runs were enqueued behind it."""
    spec = _splitting(2900, 3000.0)  # about 14% more particles a step
    s = lmx.MpdRdmeSolver(0)
    spec.load_into(s, seed=3)
    orc = oracle.Oracle(spec, seed_top=3)
    for _ in range(calls):
        s.runTimesteps(8 // calls if calls == 1 else 4, synchronize=False)
    steps = 8 if calls == 1 else 16
    if calls == 4:
        orc_rc = orc.run(12)
        assert orc_rc == 0
        steps = 4
    assert orc.run(steps) == 0
    assert int(orc.species_counts().sum()) > 4096
    np.testing.assert_array_equal(s.getSpeciesCounts(), orc.species_counts())
    assert np.array_equal(s.getLatticeNative(), orc.native())
    assert s.timestep == orc.timestep
    s.runTimesteps(5)
    assert orc.run(5) == 0
    assert np.array_equal(s.getLatticeNative(), orc.native())
    s.close()


def test_lattice_filled_on_the_device_past_the_block(gpu):
    """More particles than a block holds, written through the device views:
    the run puts back what it listed and the steps run otherwise."""
    import torch
    shape = (20, 18, 16)
    spec = models.random_model(shape=shape, P=8, nS=5, nST=2, R=6, density=0.01, seed=9, include_zero_order=False)
    many = models.random_model(shape=shape, P=8, nS=5, nST=2, R=6, density=0.2, seed=10, include_zero_order=False)
    many.sites, many.DF, many.RL, many.K, many.S, many.D, many.types = (spec.sites, spec.DF, spec.RL, spec.K, spec.S,
                                                                        spec.D, spec.types)
    s = lmx.MpdRdmeSolver(0)
    spec.load_into(s, seed=6)
    orc = oracle.Oracle(many, seed_top=6)
    view = DeviceHookLattice(s)
    view.refresh()
    lat = view.getParticleLatticeView()
    lat.copy_(torch.from_numpy(np.ascontiguousarray(orc.native()).view(np.uint8).reshape(lat.shape)))
    view.synchronize()
    for chunk in (6, 4):
        s.runTimesteps(chunk)
        assert orc.run(chunk) == 0
        assert np.array_equal(s.getLatticeNative(), orc.native())
    s.close()


def test_ensemble_of_resident_and_batched_members(gpu):
    """Members of few particles run in blocks of their own beside the batched
    steps of the others; each equals its oracle run, also after a member
    changes sides."""
    ens = lmx.Ensemble(0)
    pairs = []
    for k, (shape, density) in enumerate([((16, 12, 10), 0.1), ((32, 24, 20), 0.2), ((12, 7, 9), 0.3),
                                          ((32, 32, 32), 0.005), ((64, 16, 16), 0.1)]):
        spec = models.random_model(shape=shape, P=8, nS=5, nST=3, R=7, density=density, seed=80 + k,
                                   boundary="reflecting" if k % 2 else "periodic", include_zero_order=False)
        s = lmx.MpdRdmeSolver(0)
        spec.load_into(s, replicate=k, seed=11 + k)
        ens.add(s)
        pairs.append((s, oracle.Oracle(spec, seed_top=11 + k, replicate=k)))
    grow = _splitting(2500, 3000.0)
    s = lmx.MpdRdmeSolver(0)
    grow.load_into(s, replicate=9, seed=4)
    ens.add(s)
    pairs.append((s, oracle.Oracle(grow, seed_top=4, replicate=9)))
    for chunk in (5, 2, 8):
        ens.run(chunk)
        for s, orc in pairs:
            assert orc.run(chunk) == 0
            assert np.array_equal(s.getLatticeNative(), orc.native()), f"{s.shape}"
            assert s.timestep == orc.timestep
    ens.close()
