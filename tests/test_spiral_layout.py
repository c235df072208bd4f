"""The layout of the spiral J^H.y (compas/spiral_layout.h), compiled for the host:
the blocks hold every sample and coil, the chunks cover the readouts and none is
longer than 192 of them."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "compas/spiral_layout.h"
int main() {
    const int nvs[] = {1, 384, 385, 1000, 50176, 98304, 400000}, nrs[] = {1, 2, 191, 192, 193, 1120, 5000};
    const int nss[] = {1, 32, 33, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 2048};
    for (int nv : nvs) for (int nr : nrs) for (int ns : nss) for (int nc = 1; nc <= compas::SPIRAL_ADJOINT_COILS; nc++) {
        const auto l = compas::spiral_adjoint_layout(nv, nr, ns, nc, true, 256);
        const int s = 8 * l.ks * (l.t8 ? 8 : 4), coils = l.t8 ? 4 : 8;
        const bool samples = (l.blocks / l.groups) * s >= ns && l.groups * coils >= nc && l.blocks % l.groups == 0;
        const bool chunks = l.r_chunk >= 1 && l.r_chunk <= 192 && (long long)l.chunks * l.r_chunk >= nr &&
            (l.chunks - 1) * l.r_chunk < nr;
        const bool bytes = l.fragment_bytes(nr) == (long long)nr * l.blocks * l.ks * 8192;
        if (!samples || !chunks || !bytes) {
            printf("%d voxels, %d x %d, %d coils\n", nv, nr, ns, nc);
            return 1;
        }
    }
    return compas::spiral_adjoint_layout(64, 1, 1024, 8, true, 256).fragment_bytes(1) != 256 << 10;
}
"""


def test_layout(tmp_path):
    (tmp_path / "layout.cpp").write_text(PROGRAM)
    include = os.path.join(ROOT, "compas-toolkit_amd", "csrc", "include")
    subprocess.run(["g++", "-std=c++17", f"-I{include}", str(tmp_path / "layout.cpp"), "-o", str(tmp_path / "layout")], check=True)
    run = subprocess.run([str(tmp_path / "layout")], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
