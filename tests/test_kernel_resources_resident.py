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


@pytest.mark.parametrize("layout,waves", [("9ByteSitesILi1E", 7), ("9ByteSitesILi2E", 7), ("9ByteSitesILi4E", 6),
                                          ("9WordSitesILi4E", 6), ("9WordSitesILi8E", 5), ("9WordSitesILi16E", 3)])
def test_boxed_kernels_of_every_layout_do_not_spill(layout, waves):
    """Single solvers' kernels; a batch's (byte lattice) keep as many waves and
    may spill a register or two."""
    res = build.kernel_resources()
    for kernel in ("box_step_kernel", "cand_react_kernel", "cand_react_jobs_kernel"):
        for n in [n for n in res if f"{kernel}INS_{layout}E" in n]:
            assert res[n]["ScratchSize"] == 0, (n, res[n])
    step = [n for n in res if f"box_step_kernelINS_{layout}E" in n]
    assert len(step) == 2 and all(res[n]["Occupancy"] >= waves for n in step), step
    for n in [n for n in res if f"box_jobs_kernelINS_{layout}E" in n]:
        assert res[n]["ScratchSize"] <= 16 and res[n]["Occupancy"] >= waves, (n, res[n])
