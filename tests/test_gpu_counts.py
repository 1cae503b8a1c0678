"""Species counts: one launch that reads 16 bytes a thread and hands its sums to
the host.  Where it can go wrong: a lattice whose words are no multiple of
four, one thread's worth and many blocks, species past the kernel's bins
(uint32 lattice), a second count after the first, a lattice of holes."""
import numpy as np
import pytest

import lattice_microbes_amd as lmx
from lattice_microbes_amd import models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("words,nS", [(False, 3), (False, 255), (True, 3), (True, 1023), (True, 1500)])
@pytest.mark.parametrize("shape,P", [((1, 1, 1), 4), ((3, 5, 7), 4), ((5, 3, 9), 8), ((40, 36, 50), 8), ((64, 60, 21), 16)])
def test_counts_equal_the_lattice(gpu, shape, P, words, nS):
    spec = models.random_model(shape=shape, P=P, nS=nS, nST=2, R=0, density=0.0, seed=1)
    rng = np.random.default_rng(nS + P)
    lat = np.zeros(shape + (P,), np.uint32 if words else np.uint8)
    held = rng.integers(0, P + 1, shape)  # particles a site, in its first slots
    for j in range(P):
        lat[..., j] = np.where(held > j, rng.integers(1, nS + 1, shape), 0)
    spec.lattice = lat
    s = (lmx.IntMpdRdmeSolver if words else lmx.MpdRdmeSolver)(0)
    spec.load_into(s, seed=2)
    ref = np.bincount(lat.reshape(-1), minlength=nS + 1)[1:]
    for _ in range(3):
        assert np.array_equal(s.getSpeciesCounts(), ref)
    s.setLattice(np.zeros_like(lat))
    assert not s.getSpeciesCounts().any()
    s.close()
