"""The boxed step (the default): one launch over boxes of 16 x TY x TZ sites
with a one-site shell, particles ranked on their sites through hash chains.
Every case is compared word for word with the oracle.

Where it can go wrong: lattice extents at, one below and one above a box or a
whole number of boxes; extents of one (both neighbours are the site itself);
odd x extents (no 16-byte loads); every slot count and the uint32 lattice;
births at empty sites; crowded boxes, which a block halves or cuts into small
ones; lattices that are not packed."""
import numpy as np
import pytest

import lattice_microbes_amd as lmx
from lattice_microbes_amd import models
from lattice_microbes_amd.solver import DeviceHookLattice
import oracle

pytestmark = pytest.mark.gpu

CASES = [
    # shape, P, boundary, density (particles per slot), zero-order reactions
    ((16, 14, 14), 8, "periodic", 0.02, False),      # one box, its own neighbour on every side
    ((16, 14, 14), 8, "reflecting", 0.02, True),
    ((17, 15, 15), 8, "periodic", 0.02, True),       # one site into the next box
    ((15, 13, 29), 8, "reflecting", 0.02, False),
    ((32, 28, 28), 4, "periodic", 0.03, False),
    ((36, 27, 29), 16, "periodic", 0.01, True),      # a partial last box, groups of four
    ((48, 1, 30), 8, "periodic", 0.05, False),
    ((1, 15, 1), 8, "periodic", 0.05, False),
    ((4, 43, 16), 16, "reflecting", 0.02, False),
    ((64, 30, 17), 8, "periodic", 0.004, False),     # boxes known to be empty
    ((33, 16, 31), 8, "periodic", 0.1, True),        # smaller boxes
    ((20, 18, 22), 4, "reflecting", 0.12, False),
    ((40, 12, 12), 16, "periodic", 0.05, False),
]


@pytest.mark.parametrize("words", [False, True], ids=["byte", "uint32"])
@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}-P{c[1]}-{c[2]}{'-births' if c[4] else ''}" for c in CASES])
def test_boxes_match_oracle(gpu, case, words):
    shape, P, boundary, density, births = case
    spec = models.random_model(shape=shape, P=P, nS=6, nST=3, R=9, density=density, seed=31, boundary=boundary,
                               include_zero_order=births, rate_scale=0.05 if births else 1.0)
    if words:
        spec.lattice = spec.lattice.astype(np.uint32)
    orc = oracle.Oracle(spec, seed_top=8, replicate=1)
    for boxes in (1, 0):
        s = (lmx.IntMpdRdmeSolver if words else lmx.MpdRdmeSolver)(0)
        spec.load_into(s, replicate=1, seed=8)
        s.setLaunchOption(lmx._lib.OPT_BOXES, boxes)
        if boxes:
            for chunk in (1, 4, 2):
                s.runTimesteps(chunk)
                assert orc.run(chunk) == 0
                got, ref = s.getLatticeNative(), orc.native()
                assert np.array_equal(got, ref), f"{(got != ref).sum()} words differ"
            assert s.getOverflowStats() == (orc.stats.overflow_entries, orc.stats.overflow_steps)
        else:  # the separate sweeps end on the same lattice
            s.runTimesteps(7)
            assert np.array_equal(s.getLatticeNative(), orc.native())
        s.close()


def _kernels(s, steps):
    return set(s.timeSteps(steps, per_kernel=True)[1])


def test_boxes_are_the_default_where_they_fit(gpu):
    """A sparse lattice steps in boxes, one fuller than the smallest box
    takes in sweeps, and setting a lattice decides again."""
    spec = models.bimolecular(shape=(32, 32, 32), nA=300, nB=300, seed=3)
    s = lmx.MpdRdmeSolver(0)
    spec.load_into(s, seed=2)
    assert _kernels(s, 1) == {"fused", "reaction"}
    rng = np.random.default_rng(1)
    full = rng.integers(1, 4, (32, 32, 32, 8)).astype(np.uint8)
    full[..., 4:] = 0  # four particles a site
    s.setLattice(full)
    assert "sweep_z" in _kernels(s, 1)
    s.setLattice(spec.lattice)
    assert _kernels(s, 1) == {"fused", "reaction"}
    s.setLaunchOption(lmx._lib.OPT_BOXES, 0)
    assert "sweep_z" in _kernels(s, 1)
    s.close()


@pytest.mark.parametrize("per_site,P,words", [(0.35, 8, False), (2.0, 8, False), (1.5, 16, False), (1.5, 8, True),
                                              (0.8, 4, False)])
def test_crowded_boxes_are_cut(gpu, per_site, P, words):
    """A lattice that becomes crowded on the device after the boxes were
    chosen: blocks halve their boxes, or cut them into ones that always fit,
    and the boxes are made smaller at the next synchronisation."""
    shape = (32, 28, 30)
    spec = models.random_model(shape=shape, P=P, nS=5, nST=2, R=6, density=0.01, seed=4, qmax=0.3,
                               include_zero_order=False)
    crowd = models.random_model(shape=shape, P=P, nS=5, nST=2, R=6, density=per_site / P, seed=5, qmax=0.3,
                                include_zero_order=False)
    crowd.sites, crowd.DF, crowd.RL, crowd.K, crowd.S, crowd.D, crowd.types = (
        spec.sites, spec.DF, spec.RL, spec.K, spec.S, spec.D, spec.types)
    if words:
        spec.lattice, crowd.lattice = spec.lattice.astype(np.uint32), crowd.lattice.astype(np.uint32)
    import torch
    s = (lmx.IntMpdRdmeSolver if words else lmx.MpdRdmeSolver)(0)
    spec.load_into(s, seed=6)
    s.runTimesteps(1)
    orc = oracle.Oracle(crowd, seed_top=6)
    orc.timestep = 1
    view = DeviceHookLattice(s)
    view.refresh()
    lat = view.getParticleLatticeView()
    ref = np.ascontiguousarray(orc.native())
    lat.copy_(torch.from_numpy(ref.view(np.int32 if words else np.uint8).reshape(lat.shape)))
    view.synchronize()
    for chunk in (2, 3, 1):
        s.runTimesteps(chunk)
        assert orc.run(chunk) == 0
        got = s.getLatticeNative()
        assert np.array_equal(got, orc.native()), f"{(got != orc.native()).sum()} words differ"
    assert s.getOverflowStats()[0] == orc.stats.overflow_entries
    s.close()


@pytest.mark.parametrize("P", [4, 8, 16])
def test_batch_of_boxed_members(gpu, P):
    """Members that step in boxes share two launches a step: lattices of one
    and of many boxes, births, no reactions, a reflecting edge, and one that
    an outside write left unpacked, beside one in sweeps (too crowded)."""
    ens = lmx.Ensemble(0)
    pairs = []
    for k, (shape, density, R) in enumerate([((16, 14, 14), 0.02, 6), ((36, 27, 29), 0.02, 6), ((64, 48, 40), 0.02, 0),
                                             ((20, 70, 17), 0.06, 9), ((16, 12, 12), 0.4, 6)]):
        spec = models.random_model(shape=shape, P=P, nS=5, nST=3, R=R, density=density, seed=50 + k, rate_scale=0.05,
                                   boundary="reflecting" if k % 2 else "periodic", include_zero_order=k in (0, 3))
        s = lmx.MpdRdmeSolver(0)
        spec.load_into(s, replicate=k, seed=3)
        ens.add(s)
        pairs.append((s, oracle.Oracle(spec, seed_top=3, replicate=k)))
    s, orc = pairs[2]  # its slots reversed: the first step reads sites with holes
    slots = np.ascontiguousarray(s.getLatticeNative()).reshape(P // 4, -1, 1).view(np.uint8)
    s.setLatticeNative(np.ascontiguousarray(slots[::-1, :, ::-1]).view(np.uint32).reshape(orc.native().shape))
    orc.lattice[:] = s.getLatticeNative().reshape(-1)
    for chunk in (1, 2, 3):
        ens.run(chunk)
        for s, orc in pairs:
            assert orc.run(chunk) == 0
            got, ref = s.getLatticeNative(), orc.native()
            assert np.array_equal(got, ref), f"{s.shape}: {(got != ref).sum()} words differ"
            assert s.getOverflowStats()[0] == orc.stats.overflow_entries
    ens.close()
