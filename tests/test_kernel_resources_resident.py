"""Register budget of the resident kernels and of the boxed step's in every
slot layout, from the compiler's report of the last build: a resident block of
16 waves has 128 VGPRs a lane, and its records fill the LDS of a CU."""
import os

import pytest

from lattice_microbes_amd import build

pytestmark = pytest.mark.skipif(not os.path.exists(build.RESOURCES),
                                reason="no kernel resource report (build the library first)")


@pytest.mark.parametrize("layout", ["ByteSitesILi1E", "ByteSitesILi2E", "ByteSitesILi4E", "WordSitesILi4E",
                                    "WordSitesILi8E", "WordSitesILi16E"])
@pytest.mark.parametrize("kernel", ["resident_run_kernel", "resident_run_jobs_kernel"])
def test_resident_kernels_of_every_layout_do_not_spill(kernel, layout):
    res = build.kernel_resources()
    names = [n for n in res if f"{kernel}INS_9{layout}E" in n]
    assert len(names) == 1, names
    r = res[names[0]]
    assert r["ScratchSize"] == 0 and r["VGPRs Spill"] == 0, r
    assert r["Occupancy"] >= 4 and r["LDS Size"] <= 163840, r


@pytest.mark.parametrize("layout,waves", [("ByteSitesILi1E", 7), ("ByteSitesILi2E", 7), ("ByteSitesILi4E", 6),
                                          ("WordSitesILi4E", 6), ("WordSitesILi8E", 6), ("WordSitesILi16E", 4)])
def test_boxed_kernels_of_every_layout(layout, waves):
    """They keep their waves.  The uint32 lattice's wide rows and a batch's
    kernels may spill a few registers, the reaction launches none."""
    res = build.kernel_resources()
    step = [n for n in res if f"box_step_kernelINS_9{layout}E" in n]
    assert len(step) == 2 and all(res[n]["Occupancy"] >= waves for n in step), step
    for n in step:
        assert res[n]["ScratchSize"] <= (28 if "WordSites" in layout and "ELb1E" in n else 0), (n, res[n])
    for n in [n for n in res if f"box_jobs_kernelINS_9{layout}E" in n]:
        assert res[n]["ScratchSize"] <= 16 and res[n]["Occupancy"] >= waves, (n, res[n])
    for n in [n for n in res if f"cand_react_kernelINS_9{layout}E" in n or f"cand_react_jobs_kernelINS_9{layout}E" in n]:
        assert res[n]["ScratchSize"] == 0, (n, res[n])
