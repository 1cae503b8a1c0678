"""What a resident run leaves to the calls after it, when it ended and when it
stopped short, on the device: every lattice is compared with the oracle."""
import numpy as np
import pytest

import lattice_microbes_amd as lmx
from lattice_microbes_amd import models
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
