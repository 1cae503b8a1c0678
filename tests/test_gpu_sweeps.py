"""The separate x, y and z sweeps, which step every lattice too crowded for
boxes, with LMX_OPT_BOXES off (by default these lattices step in boxes or in one
block), and the batch maps that grow when members join: every lattice is
compared with the oracle."""
import numpy as np
import pytest

import lattice_microbes_amd as lmx
from lattice_microbes_amd import _lib, models
import oracle

pytestmark = pytest.mark.gpu


def _pair(spec, k, boxes):
    s = lmx.MpdRdmeSolver(0)
    s.setLaunchOption(_lib.OPT_BOXES, 1 if boxes else 0)
    spec.load_into(s, replicate=k, seed=5 + k)
    return s, oracle.Oracle(spec, seed_top=5 + k, replicate=k)


def _run_and_compare(run, pairs, steps):
    run(steps)
    for s, orc in pairs:
        assert orc.run(steps) == 0
        got = s.getLatticeNative()
        assert np.array_equal(got, orc.native()), f"{s.shape}: {(got != orc.native()).sum()} words differ"
        assert s.timestep == orc.timestep


@pytest.mark.parametrize("P", [4, 8, 16])
@pytest.mark.parametrize("density", [0.004, 0.1])
@pytest.mark.parametrize("zero_order", [False, True])
@pytest.mark.parametrize("shape", [(256, 12, 9), (64, 35, 34), (20, 17, 33)])
def test_default_sweeps_match_oracle(gpu, shape, P, density, zero_order):
    """Whole rows of a chunk, tiles with remainders and rows shorter than a
    tile: tile sweeps, the reaction list and the chunk flags, over calls
    between which the flags are kept."""
    spec = models.random_model(shape=shape, P=P, nS=5, nST=3, R=7, density=density, seed=31, rate_scale=0.1,
                               boundary="periodic" if zero_order else "reflecting", include_zero_order=zero_order)
    s, orc = _pair(spec, 1, False)
    for steps in (1, 5):
        _run_and_compare(s.runTimesteps, [(s, orc)], steps)
    s.close()


@pytest.mark.parametrize("boxes", [False, True], ids=["sweeps", "boxes"])
def test_members_joining_grow_the_block_maps(gpu, boxes):
    """Blocks past the 4096 that a batch first maps, after it has run: in the
    sweeps one lattice of 256x256x128 has 8192 (the captured step is captured
    again), in boxes two of 256x160x128 more than 4096."""
    ens, pairs = lmx.Ensemble(0), []

    def join(shape, density):
        k = len(pairs)
        spec = models.random_model(shape=shape, P=8, nS=5, nST=3, R=7, density=density, seed=70 + k)
        s, orc = _pair(spec, k, boxes)
        ens.add(s)
        pairs.append((s, orc))

    join((8, 12, 10), 0.2)
    join((32, 24, 20), 0.2)
    _run_and_compare(ens.run, pairs, 2)
    for shape in [(256, 160, 128)] * 2 if boxes else [(256, 256, 128)]:
        join(shape, 0.002)
        _run_and_compare(ens.run, pairs, 2)
    _run_and_compare(ens.run, pairs, 1)
    ens.close()
