"""What a resident run leaves to the calls after it, when it ended and when it
stopped short, on the device: every lattice is compared with the oracle."""
import ctypes
import time

import numpy as np
import pytest

import lattice_microbes_amd as lmx
from lattice_microbes_amd import _lib, models
from lattice_microbes_amd.solver import DeviceHookLattice
import oracle

pytestmark = pytest.mark.gpu


def _reversed_slots(native, P, words):
    """Every site's particles in its last slots: empty slots before occupied ones."""
    W = native.shape[0]
    if words:
        return np.ascontiguousarray(native[::-1])
    slots = np.ascontiguousarray(native).reshape(W, -1, 1).view(np.uint8)
    return np.ascontiguousarray(slots[::-1, :, ::-1]).view(np.uint32).reshape(native.shape)


@pytest.mark.parametrize("words", [False, True], ids=["byte", "uint32"])
def test_unpacked_lattice_past_the_block(gpu, words):
    """A lattice written on the device with more particles than a block holds,
    in the last slots of their sites: the run lists what fits, puts it back
    and ends, and the steps made up for it read every slot."""
    import torch
    shape = (20, 18, 16)
    spec = models.random_model(shape=shape, P=8, nS=5, nST=2, R=6, density=0.01, seed=9, include_zero_order=False)
    many = models.random_model(shape=shape, P=8, nS=5, nST=2, R=6, density=0.2, seed=10, include_zero_order=False)
    many.sites, many.DF, many.RL, many.K, many.S, many.D, many.types = (spec.sites, spec.DF, spec.RL, spec.K, spec.S,
                                                                        spec.D, spec.types)
    assert int(many.initial_counts().sum()) > 4096
    if words:
        spec.lattice, many.lattice = spec.lattice.astype(np.uint32), many.lattice.astype(np.uint32)
    s = (lmx.IntMpdRdmeSolver if words else lmx.MpdRdmeSolver)(0)
    spec.load_into(s, seed=6)
    orc = oracle.Oracle(many, seed_top=6)
    orc.lattice[:] = _reversed_slots(orc.native(), 8, words).reshape(-1)
    view = DeviceHookLattice(s)
    view.refresh()
    lat = view.getParticleLatticeView()
    ref = np.ascontiguousarray(orc.native())
    lat.copy_(torch.from_numpy(ref.view(np.int32 if words else np.uint8).reshape(lat.shape)))
    view.synchronize()
    for chunk in (6, 4):
        s.runTimesteps(chunk)
        assert orc.run(chunk) == 0
        got = s.getLatticeNative()
        assert np.array_equal(got, orc.native()), f"{(got != orc.native()).sum()} words differ"
    s.close()


def _splitting(n, rate):
    """A -> A + A: the particles multiply."""
    spec = models.bimolecular(shape=(24, 20, 18), nA=n, nB=0, seed=5, boundary="periodic")
    spec.types, spec.K = np.array([1], np.uint32), np.array([rate])
    spec.S, spec.D = np.array([[1], [0], [0]], np.int32), np.array([[1], [0], [0]], np.uint32)
    spec.RL = np.ones((1, 1), np.uint32)
    return spec


def _static(s, n):
    _lib.check(_lib.load().lmx_run_steps_static(s._h, ctypes.c_uint32(n)))


def test_short_calls_behind_a_run_that_stopped_short(gpu):
    """Calls of one and two steps, of either kind, enqueued behind runs whose
    block was full (about 14% more particles a step), and a new rate."""
    spec = _splitting(2040, 3000.0)
    s = lmx.MpdRdmeSolver(0)
    spec.load_into(s, seed=3)
    orc = oracle.Oracle(spec, seed_top=3)
    for n in (8, 1, 4, 2):
        s.runTimesteps(n, synchronize=False)
        _static(s, 1)
    assert orc.run(19) == 0
    assert int(orc.species_counts().sum()) > 4096
    assert np.array_equal(s.getLatticeNative(), orc.native())
    assert s.timestep == orc.timestep == 19
    s.close()


def test_steps_behind_a_resident_run_are_enqueued(gpu):
    """A run of 40000 steps takes half a second; calls behind it return before
    it has ended."""
    spec = models.bimolecular(shape=(64, 64, 64), seed=5)
    s = lmx.MpdRdmeSolver(0)
    spec.load_into(s, seed=3)
    s.runTimesteps(4)
    _static(s, 1)
    s.synchronize()
    t0 = time.perf_counter()
    s.runTimesteps(40000, synchronize=False)
    s.runTimesteps(2, synchronize=False)
    _static(s, 2)
    s.setReactionRate(0, float(spec.K[0]))
    enqueued = time.perf_counter() - t0
    s.synchronize()
    assert enqueued < 0.5 * (time.perf_counter() - t0)
    s.close()


def test_static_steps_while_a_graph_is_captured(gpu):
    """No wait and no blocking copy, which a capture elsewhere in the process
    would refuse."""
    import torch
    spec = models.bimolecular(shape=(32, 32, 32), seed=5)
    s = lmx.MpdRdmeSolver(0)
    spec.load_into(s, seed=3)
    orc = oracle.Oracle(spec, seed_top=3)
    _static(s, 1)
    s.synchronize()
    s.runTimesteps(6, synchronize=False)
    x = torch.zeros(8, device="cuda")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = x + 1
        _static(s, 2)
        _static(s, 5)
    g.replay()
    torch.cuda.synchronize()
    assert float(y.sum()) == 8.0
    assert orc.run(14) == 0
    assert np.array_equal(s.getLatticeNative(), orc.native())
    s.close()


def test_static_steps_of_the_uint32_lattice(gpu):
    """Two solvers' calls in turn, without a wait between them."""
    pairs = []
    for k, shape in enumerate([(40, 36, 28), (33, 30, 31)]):
        spec = models.random_model(shape=shape, P=8, nS=5, nST=2, R=6, density=0.03, seed=30 + k, include_zero_order=True)
        spec.lattice = spec.lattice.astype(np.uint32)
        s = lmx.IntMpdRdmeSolver(0)
        spec.load_into(s, replicate=k, seed=3)
        pairs.append((s, oracle.Oracle(spec, seed_top=3, replicate=k)))
    for turn in range(6):
        for s, _ in pairs:
            _static(s, 2)
    for s, orc in pairs:
        assert orc.run(12) == 0
        assert np.array_equal(s.getLatticeNative(), orc.native())
        s.close()


def test_autotune_of_a_resident_solver_keeps_the_state(gpu):
    """The tuner times the one-block run too (and one that outgrows its block);
    afterwards the state is as before."""
    for spec in (models.bimolecular(shape=(32, 32, 32), seed=5), _splitting(2040, 3000.0)):
        s = lmx.MpdRdmeSolver(0)
        spec.load_into(s, seed=3)
        orc = oracle.Oracle(spec, seed_top=3)
        s.runTimesteps(2)
        assert orc.run(2) == 0
        assert s.autotune(steps=8)["ms_per_step"] > 0
        assert np.array_equal(s.getLatticeNative(), orc.native()) and s.timestep == 2
        s.runTimesteps(9)
        assert orc.run(9) == 0
        assert np.array_equal(s.getLatticeNative(), orc.native()) and s.timestep == 11
        s.close()


MEMBERS = [
    # shape, particles per slot, boundary
    ((12, 10, 8), 0.15, "periodic"),
    ((4, 6, 5), 0.6, "reflecting"),     # sites of many particles, overflow entries
    ((16, 16, 24), 0.02, "periodic"),
    ((8, 3, 40), 0.1, "reflecting"),
    ((32, 20, 17), None, "periodic"),   # three records a thread
]


@pytest.mark.parametrize("P", [4, 8, 16])
def test_ensemble_of_resident_members(gpu, P):
    """Every slot count, in calls of four steps and more, from lattices of
    single particles to sites of all their slots."""
    ens = lmx.Ensemble(0)
    pairs = []
    for k, (shape, density, boundary) in enumerate(MEMBERS):
        if density is None:
            density = 2900 / (np.prod(shape) * P)
        spec = models.random_model(shape=shape, P=P, nS=5, nST=3, R=9, density=density, seed=90 + k, boundary=boundary,
                                   include_zero_order=False, rate_scale=0.1)
        assert 0 < int(spec.initial_counts().sum()) <= 3000
        s = lmx.MpdRdmeSolver(0)
        spec.load_into(s, replicate=k, seed=5)
        ens.add(s)
        pairs.append((s, oracle.Oracle(spec, seed_top=5, replicate=k)))
    for chunk in (4, 7, 12):
        ens.run(chunk)
        for s, orc in pairs:
            assert orc.run(chunk) == 0
            got = s.getLatticeNative()
            assert np.array_equal(got, orc.native()), f"{s.shape}: {(got != orc.native()).sum()} words differ"
            assert s.getOverflowStats() == (orc.stats.overflow_entries, orc.stats.overflow_steps)
    assert pairs[1][1].stats.overflow_entries > 0
    ens.close()


@pytest.mark.parametrize("words", [False, True], ids=["byte", "uint32"])
@pytest.mark.parametrize("P", [4, 8, 16])
def test_resident_reactions_of_full_sites(gpu, P, words):
    """Reactions of one to three products at sites of up to all their slots:
    records that are reused, that die and that are appended."""
    for shape, density in (((6, 5, 4), 0.5), ((20, 18, 16), 2400 / (20 * 18 * 16 * P))):
        spec = models.random_model(shape=shape, P=P, nS=6, nST=2, R=12, density=density, seed=7, include_zero_order=False,
                                   rate_scale=0.2)
        assert 0 < int(spec.initial_counts().sum()) <= 3000
        if words:
            spec.lattice = spec.lattice.astype(np.uint32)
        s = (lmx.IntMpdRdmeSolver if words else lmx.MpdRdmeSolver)(0)
        spec.load_into(s, seed=8)
        orc = oracle.Oracle(spec, seed_top=8)
        changed = orc.species_counts()
        for chunk in (4, 16):
            s.runTimesteps(chunk)
            assert orc.run(chunk) == 0
            got = s.getLatticeNative()
            assert np.array_equal(got, orc.native()), f"{shape}: {(got != orc.native()).sum()} words differ"
        assert not np.array_equal(changed, orc.species_counts())
        s.close()


class RelaxedInt(lmx.IntMpdRdmeSolver):
    _parses_overflow_handler = True


def _spot(shape, P, spot, density, seed, boundary):
    """A sparse lattice with a crowded corner, so that a run in one block has
    overflow entries in every step."""
    spec = models.random_model(shape=shape, P=P, nS=6, nST=2, R=9, density=0.002, seed=seed, boundary=boundary,
                               include_zero_order=False)
    corner = spec.lattice[tuple(slice(0, k) for k in spot)]
    rng = np.random.default_rng(seed)
    corner[...] = np.where(rng.random(corner.shape) < density, rng.integers(1, 7, corner.shape), 0)
    return spec


@pytest.mark.parametrize("words", [False, True], ids=["byte", "uint32"])
@pytest.mark.parametrize("handler", ["classic", "relaxed"])
@pytest.mark.parametrize("P,spot,density", [(4, (10, 9, 8), 0.6), (8, (7, 6, 6), 0.75), (16, (5, 4, 5), 0.85)])
def test_overflow_entries_of_resident_runs(gpu, P, spot, density, handler, words):
    spec = _spot((30, 28, 24), P, spot, density, 12, "periodic" if P == 8 else "reflecting")
    n = int((spec.lattice != 0).sum())
    assert 0 < n <= 2048
    if words:
        spec.lattice = spec.lattice.astype(np.uint32)
    orc = oracle.Oracle(spec, seed_top=7, replicate=2, overflow=handler)
    s = (RelaxedInt if words else lmx.MpdRdmeSolver)(0)
    spec.load_into(s, replicate=2, seed=7, extra={"rdme.mpd.overflowhandler": handler})
    for chunk in (10, 4, 11):
        s.runTimesteps(chunk)
        assert orc.run(chunk) == 0
        got = s.getLatticeNative()
        assert np.array_equal(got, orc.native()), f"{(got != orc.native()).sum()} words differ"
        assert s.getOverflowStats() == (orc.stats.overflow_entries, orc.stats.overflow_steps)
        assert s.getUnresolvedOverflows() == orc.unresolved
    assert orc.stats.overflow_entries > 20
    s.close()


def test_timed_runs_that_outgrow_the_block(gpu):
    """lmx_time_steps and the ensemble's, whose time includes the steps made up."""
    spec = _splitting(2040, 3000.0)
    pairs = []
    for k in range(2):
        s = lmx.MpdRdmeSolver(0)
        spec.load_into(s, replicate=k, seed=3)
        pairs.append((s, oracle.Oracle(spec, seed_top=3, replicate=k)))
    assert pairs[0][0].timeSteps(9)[0] > 0
    assert pairs[0][1].run(9) == 0
    ens = lmx.Ensemble(0)
    for s, _ in pairs:
        ens.add(s)
    assert ens.time_steps(8) > 0
    for s, orc in pairs:
        assert orc.run(8) == 0
        assert np.array_equal(s.getLatticeNative(), orc.native()) and s.timestep == orc.timestep
    ens.close()
