"""The two-level spiral products against the FP64 oracle at the edges of their
tiles: sample counts around a column tile and a pass, one voxel to a step that
is not full, coil counts that take one row tile, two, and a padded one.

Tolerance: a BF16 hi + lo pair keeps a number to 2^-18 and the product of the two
lo parts, 2^-18 of the whole, is dropped: at most 3 x 3.8e-6 a term; 3e-5 with
the FP32 phasors and sums.  One BF16 product keeps 2^-9 of each operand: 2e-2.
"""

import numpy as np
import pytest

import compas_amd as ca
from compas_amd import workloads as W
from gpu_helpers import banner, context, rel

pytestmark = pytest.mark.gpu


def case(nv, nr, ns, nc):
    n = int(np.ceil(np.sqrt(nv)))
    rng = np.random.default_rng(nv * 7919 + ns)
    t = W.make_tissue(W.SplitMix64(8), n, 20.0, 40.0).slice(0, nv)
    traj = W.make_spiral(nr, ns, 20.0, max(n, 8), 5e-6)
    coils = W.make_coils(n, 20.0, nc)[:, :nv]
    c = lambda *shape: (rng.normal(size=shape) + 1j * rng.normal(size=shape)).astype(np.complex64)  # noqa: E731
    context()
    return (t, traj, coils, c(nr, nv), [c(nr, nv) for _ in range(4)], c(6, nv), c(nc, nr, ns),
            ca.TissueParameters.from_tissue(t), ca.SpiralTrajectory.from_trajectory(traj))


SHAPES = [(1, 1, 1, 1), (7, 2, 31, 1), (8, 2, 32, 3), (9, 3, 33, 4), (130, 2, 256, 4), (61, 3, 257, 2), (140, 2, 512, 4),
          (33, 2, 513, 1), (17, 2, 1024, 4), (5, 2, 1040, 3)]


@pytest.mark.parametrize("nv,nr,ns,nc", SHAPES + [(40, 2, 130, 5), (40, 2, 512, 8), (40, 2, 300, 9)])
@pytest.mark.parametrize("method,tol", [("matmul_fast", 3e-5), ("matmul_low", 2e-2)])
def test_signal(oracle, nv, nr, ns, nc, method, tol):
    banner(f"spiral signal {nv} voxels {nr} x {ns} {nc} coils {method}")
    t, traj, coils, m, _, _, _, p, tr = case(nv, nr, ns, nc)
    want = oracle.signal_spiral(t, traj, coils, m.astype(np.complex128), "f64")
    assert rel(ca.magnetization_to_signal(m, p, tr, coils, method=method).collect(), want) < tol


@pytest.mark.parametrize("nv,nr,ns,nc", SHAPES + [(40, 2, 130, 5), (40, 2, 300, 8)])
@pytest.mark.parametrize("method,tol", [("gemm_fast", 3e-5), ("gemm_low", 2e-2)])
def test_products(oracle, nv, nr, ns, nc, method, tol):
    banner(f"spiral products {nv} voxels {nr} x {ns} {nc} coils {method}")
    t, traj, coils, m, d, v, y, p, tr = case(nv, nr, ns, nc)
    wide = lambda a: a.astype(np.complex128)  # noqa: E731
    jv = oracle.jacobian_spiral(t, traj, coils, wide(m), *[wide(x) for x in d], wide(v), "f64")
    jh = oracle.jacobian_hermitian_spiral(t, traj, coils, wide(m), *[wide(x) for x in d], wide(y), "f64")
    assert rel(ca.compute_jacobian_spiral(m, d, p, tr, coils, v, method=method).collect(), jv) < tol
    assert rel(ca.compute_jacobian_hermitian_spiral(m, d, p, tr, coils, y, method=method).collect(), jh) < tol


@pytest.mark.parametrize("nv,nr,ns,nc", [(129, 1, 1, 1), (383, 1, 5, 2), (8191, 1, 3, 1), (8193, 2, 31, 4), (9000, 1, 33, 2)])
def test_many_voxel_ranges(oracle, nv, nr, ns, nc):
    """Few outputs of many voxel ranges each: several lanes add up one output, two
    ranges to one, a last lane with fewer or none."""
    banner(f"spiral sums over voxel ranges {nv} voxels {nr} x {ns} {nc} coils")
    t, traj, coils, m, d, v, _, p, tr = case(nv, nr, ns, nc)
    wide = lambda a: a.astype(np.complex128)  # noqa: E731
    want = oracle.signal_spiral(t, traj, coils, wide(m), "f64")
    assert rel(ca.magnetization_to_signal(m, p, tr, coils, method="matmul_fast").collect(), want) < 3e-5
    jv = oracle.jacobian_spiral(t, traj, coils, wide(m), *[wide(x) for x in d], wide(v), "f64")
    assert rel(ca.compute_jacobian_spiral(m, d, p, tr, coils, v, method="gemm_fast").collect(), jv) < 3e-5
