"""Register budget of the boxed step's kernels, from the compiler's report of
the last build: 72 VGPRs are seven blocks of four waves per CU, and its 20 KB
of LDS leave room for as many, without a spill."""
import os

import pytest

from lattice_microbes_amd import build

pytestmark = pytest.mark.skipif(not os.path.exists(build.RESOURCES),
                                reason="no kernel resource report (build the library first)")


@pytest.mark.parametrize("W", [1, 2])
@pytest.mark.parametrize("vec", [0, 1])
def test_box_kernels_do_not_spill(W, vec):
    res = build.kernel_resources()
    names = [n for n in res if f"box_step_kernelINS_9ByteSitesILi{W}EE" in n and f"ELb{vec}E" in n]
    assert len(names) == 1, names
    r = res[names[0]]
    assert r["ScratchSize"] == 0 and r["Occupancy"] >= 7, r
    assert r["LDS Size"] <= 163840 // 7, r


@pytest.mark.parametrize("W", [1, 2])
@pytest.mark.parametrize("kernel", ["resident_run_kernel", "resident_run_jobs_kernel"])
def test_resident_kernels_do_not_spill(W, kernel):
    """A block of 16 waves has 128 VGPRs a lane."""
    res = build.kernel_resources()
    names = [n for n in res if f"{kernel}INS_9ByteSitesILi{W}EE" in n]
    assert len(names) == 1, names
    assert res[names[0]]["ScratchSize"] == 0 and res[names[0]]["Occupancy"] >= 4, res[names[0]]
