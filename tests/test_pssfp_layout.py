"""The workgroup layout of the pSSFP kernels (compas/pssfp_layout.h), compiled
for the host: for every number of slice positions the groups cover the positions
without an empty one, and a workgroup holds at least one voxel and no more
isochromats than lanes."""

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "compas/pssfp_layout.h"
int main(int argc, char** argv) {
    const int lanes = atoi(argv[1]), most = atoi(argv[2]);
    const double cost = atof(argv[3]);
    for (int nz = 1; nz <= 20000; nz++) {
        const compas::PssfpWorkgroup w = compas::pssfp_workgroup(nz, lanes, most, cost);
        const bool covered = w.groups > 0 && w.nz_group > 0 && w.nz_group <= most &&
            (long long)(w.groups - 1) * w.nz_group < nz && (long long)w.groups * w.nz_group >= nz;
        const bool fits = w.nv_block >= lanes / most && w.nv_block * w.nz_group <= lanes;
        if (!covered || !fits) {
            printf("nz %d: %d voxels x %d positions, %d groups\n", nz, w.nv_block, w.nz_group, w.groups);
            return 1;
        }
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("layout")
    (d / "layout.cpp").write_text(PROGRAM)
    include = os.path.join(ROOT, "compas-toolkit_amd", "csrc", "include")
    subprocess.run(["g++", "-std=c++17", f"-I{include}", str(d / "layout.cpp"), "-o", str(d / "layout")], check=True)
    return str(d / "layout")


@pytest.mark.parametrize("lanes,most,cost", [(256, 128, 0.1), (128, 128, 0.04), (64, 64, 0.04)],
                         ids=["simulation", "one field", "two fields"])
def test_every_number_of_slice_positions(program, lanes, most, cost):
    run = subprocess.run([program, str(lanes), str(most), str(cost)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
