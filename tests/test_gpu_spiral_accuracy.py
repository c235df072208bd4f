"""Accuracy of the spiral products where one part of them stands alone: the
(s - ns/2) moment, and sums over many readouts."""

import numpy as np
import pytest

import compas_amd as ca
from compas_amd import workloads as W
from gpu_helpers import banner, context, rel

pytestmark = pytest.mark.gpu


def objects(nv, nr, ns, nc):
    n = int(np.ceil(np.sqrt(nv)))
    t = W.make_tissue(W.SplitMix64(8), n, 20.0, 40.0).slice(0, nv)
    traj = W.make_spiral(nr, ns, 20.0, max(n, 8), 5e-6)
    coils = W.make_coils(n, 20.0, nc)[:, :nv]
    context()
    return t, traj, coils, ca.TissueParameters.from_tissue(t), ca.SpiralTrajectory.from_trajectory(traj)


def noise(rng, *shape):
    return (rng.normal(size=shape) + 1j * rng.normal(size=shape)).astype(np.complex64)


# a BF16 hi + lo pair keeps a number to 2^-18 and the product of the two lo parts
# is dropped, 3 x 3.8e-6 of a term; one BF16 product keeps 2^-9 of each operand
METHODS = [("gemm_fast", 1.2e-5), ("gemm_low", 4e-3)]


@pytest.mark.parametrize("ns", [31, 64, 130, 250, 500, 512, 1040])
@pytest.mark.parametrize("width", [5.0, 20.0])
@pytest.mark.parametrize("method,tol", METHODS)
def test_adjoint_moment_of_a_peaked_readout(oracle, ns, width, method, tol):
    """Readouts that peak where they cross the centre of k-space, s = ns/2; with
    zero derivatives the T2 and B0 rows of J^H.y are the moment alone."""
    banner(f"spiral J^H.y moment {ns} samples, window {width}, {method}")
    nv, nr, nc = 130, 3, 4
    t, traj, coils, p, tr = objects(nv, nr, ns, nc)
    rng = np.random.default_rng(ns)
    m = noise(rng, nr, nv)
    zero = [np.zeros((nr, nv), np.complex64)] * 4
    y = noise(rng, nc, nr, ns) * np.exp(-0.5 * ((np.arange(ns) - ns / 2) / width) ** 2).astype(np.float32)
    wide = lambda a: a.astype(np.complex128)  # noqa: E731
    want = oracle.jacobian_hermitian_spiral(t, traj, coils, wide(m), *[wide(z) for z in zero], wide(y), "f64")
    got = ca.compute_jacobian_hermitian_spiral(m, zero, p, tr, coils, y, method=method).collect()
    for row in (1, 3):
        assert rel(got[row], want[row]) < tol


@pytest.mark.parametrize("ns", [31, 64, 130, 250, 500, 512, 1040])
@pytest.mark.parametrize("method,tol", METHODS)
def test_product_moment_at_the_centre(oracle, ns, method, tol):
    """With zero derivatives a step in T2 and B0 changes the signal by s - ns/2
    times a sum: the samples within four of ns/2, where that factor is small."""
    banner(f"spiral J.v moment {ns} samples, {method}")
    nv, nr, nc = 130, 3, 4
    t, traj, coils, p, tr = objects(nv, nr, ns, nc)
    rng = np.random.default_rng(ns + 1)
    m = noise(rng, nr, nv)
    zero = [np.zeros((nr, nv), np.complex64)] * 4
    v = noise(rng, 6, nv)
    v[[0, 2, 4, 5]] = 0
    wide = lambda a: a.astype(np.complex128)  # noqa: E731
    want = oracle.jacobian_spiral(t, traj, coils, wide(m), *[wide(z) for z in zero], wide(v), "f64")
    got = ca.compute_jacobian_spiral(m, zero, p, tr, coils, v, method=method).collect()
    at = slice(max(0, ns // 2 - 4), ns // 2 + 5)
    assert rel(got[..., at], want[..., at]) < tol


def test_adjoint_over_many_readouts():
    """1120 readouts of a constant field over as many voxels as the GPU takes in
    one round of workgroups: a voxel's sum over the readouts is FP32 within a
    chunk of readouts and FP64 over the chunks.  Every product is exact here, and a
    chain of L additions leaves 2.5e-8 L / sqrt(3 x 1120) of the sum: 8.3e-8 at
    192, and 2.5e-8 for the result."""
    import torch

    banner("spiral J^H.y over 1120 readouts")
    context()
    nv, nr, ns = 98304, 1120, 512
    one, nil = np.ones(nv, np.float32), np.zeros(nv, np.float32)
    p = ca.TissueParameters(nv, one, np.full(nv, 1e30, np.float32), one, nil, one, nil, nil, nil)
    tr = ca.SpiralTrajectory(nr, ns, 5e-6, np.zeros(nr, np.complex64), np.zeros(nr, np.complex64))
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(3)
    x = torch.rand(nr, nv, device="cuda:0", generator=gen) + 0.5
    m = ca.CompasArray.from_dlpack(torch.complex(x, torch.zeros_like(x)))
    coils = ca.CompasArray.from_numpy(np.ones((1, nv), np.complex64))
    y = ca.CompasArray.from_numpy(np.ones((1, nr, ns), np.complex64))
    got = ca.compute_jacobian_hermitian_spiral(m, [m] * 4, p, tr, coils, y, method="gemm_fast").collect()
    want = ns * x.double().sum(0).cpu().numpy()
    for row in (0, 4):
        assert rel(got[row], want) < 1.5e-7
