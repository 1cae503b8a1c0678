"""Register budget of the resident kernels of every slot layout, from the
compiler's report of the last build: a block of 16 waves has 128 VGPRs a lane,
and its records fill the LDS of a CU."""
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
