"""pSSFP by one affine map per isochromat and TR (pssfp_map.hip) against the
FP64 oracle, where its layout or its choice of form changes: workgroups of one
and of many voxels, a last voxel block and a last TR chunk that are not full,
several slice-position groups, trains with RF phases, trains too strong for the
maps, and trains too short for them.

Tolerance: the state is FP64 throughout and the maps leave at most 2e-12 per
TR, so what remains is one FP32 rounding of each echo and one of each partial
plane (at most 4 here): 5 x 6e-8 = 3e-7.
"""

import numpy as np
import pytest

import compas_amd as ca
from compas_amd import workloads as W
from gpu_helpers import banner, context, rel
from test_gpu_parity import central_difference

pytestmark = pytest.mark.gpu

TOL = 3e-7


def train(nTR, deg, nz, nRF, phase):
    seq = W.make_pssfp(nTR, deg, nz=nz, nRF=nRF)
    if phase:
        seq.RF = (seq.RF * np.exp(1j * phase * np.sin(np.arange(nTR)))).astype(np.complex64)
    if nz > 1:
        # a gradient that dephases the slice during the pulse as well
        seq.gamma_dt_GRz = (1.5 / nRF, 0.0, -0.75)
    return seq


@pytest.mark.parametrize("nv,nTR,nz,nRF,deg,phase", [
    (1, 65, 1, 12, 60.0, 0.0),       # one isochromat
    (257, 64, 1, 25, 70.0, 0.0),     # 256 voxels to a workgroup, then one
    (15, 71, 35, 25, 70.0, 0.0),     # 7 voxels to a workgroup; 71 = 8 x 8 + 7 TRs
    (15, 71, 35, 25, 70.0, 1.1),     # the same with RF phases
    (6, 72, 128, 9, 45.0, 0.7),      # the most slice positions of one group
    (5, 66, 131, 8, 45.0, 0.0),      # two groups
    (70, 64, 35, 25, 170.0, 0.4),    # too strong for the maps: sub-steps, by waves
    (3, 80, 10, 256, 60.0, 0.0),     # the longest waveform that is staged whole
    (3, 80, 10, 257, 60.0, 0.0),     # one more: sub-steps
    (40, 30, 35, 25, 70.0, 0.0),     # too few TRs: sub-steps
    (9, 100, 11, 25, 0.0, 0.0),      # no flip at all
])
def test_pssfp_map(oracle, nv, nTR, nz, nRF, deg, phase):
    banner(f"pssfp map {nv} voxels {nTR} TRs {nz} positions {nRF} sub-steps {deg} deg phase {phase}")
    context()
    n = int(np.ceil(np.sqrt(nv)))
    t = W.make_tissue(W.SplitMix64(77), n, 20.0, 40.0).slice(0, nv)
    seq = train(nTR, deg, nz, nRF, phase)
    got = ca.simulate_magnetization(ca.TissueParameters.from_tissue(t), ca.pSSFPSequence.from_sequence(seq)).collect()
    want = oracle.pssfp(t, seq, "f64")
    if deg == 0.0:
        assert np.array_equal(got, np.zeros_like(got))
    else:
        assert rel(got, want) < TOL


FIELDS = [(ca.T1, ca.T2, ca.B1, ca.B0), (ca.T1, ca.T2), (ca.T1,), (ca.T2,), (ca.B1,), (ca.B0,)]


@pytest.mark.parametrize("fields", FIELDS, ids=lambda f: "".join("T1 T2 B1 B0".split()[i] for i in f))
@pytest.mark.parametrize("nv,nTR,nz,nRF,deg,phase", [
    (1, 65, 1, 14, 60.0, 0.0),      # one isochromat
    (67, 64, 1, 25, 70.0, 0.0),     # 64 voxels to a workgroup, or half of 128
    (8, 71, 35, 25, 70.0, 0.0),     # several groups; a last chunk that is not full
    (8, 71, 35, 25, 70.0, 1.1),     # the same with RF phases
    (3, 66, 130, 12, 45.0, 0.6),    # more positions than a workgroup holds
    (20, 64, 7, 25, 170.0, 0.4),    # too strong for the maps
    (5, 20, 7, 8, 60.0, 0.0),       # too short for them
])
def test_pssfp_map_tangents(oracle, fields, nv, nTR, nz, nRF, deg, phase):
    """FP64 maps leave FP32 roundings of the outputs and of up to five partial
    planes, 3e-7, about 1e-10 per TR of interpolation, and the reference's
    central differences 1e-8: 1e-6."""
    banner(f"pssfp map tangents {fields} {nv} voxels {nTR} TRs {nz} positions {nRF} sub-steps {deg} deg phase {phase}")
    context()
    n = int(np.ceil(np.sqrt(nv)))
    t = W.make_tissue(W.SplitMix64(77), n, 20.0, 40.0).slice(0, nv)
    seq = train(nTR, deg, nz, nRF, phase)
    p, s = ca.TissueParameters.from_tissue(t), ca.pSSFPSequence.from_sequence(seq)
    out = [a.collect() for a in ca.simulate_magnetization_tangents(fields, p, s, echos=True)]
    assert rel(out[0], oracle.pssfp(t, seq, "f64")) < TOL
    for f, d in zip(fields, out[1:]):
        assert rel(d, central_difference(oracle.pssfp, t, seq, ["T1", "T2", "B1", "B0"][f])) < 1e-6


def test_many_slice_positions(oracle):
    """2500 slice positions, 20 groups of them to a voxel block: the echoes, the
    tangents and the request server.  Twenty FP32 partial planes and the echo's
    own rounding, each 6e-8 of a part of the sum, and up to 2500 positions that
    dephase by a radian: 1e-6; tangents as above with forty planes, 2e-6."""
    banner("pssfp map 2500 slice positions")
    context()
    t = W.make_tissue(W.SplitMix64(77), 2, 20.0, 40.0).slice(0, 3)
    seq = train(66, 45.0, 2500, 12, 0.6)
    p, s = ca.TissueParameters.from_tissue(t), ca.pSSFPSequence.from_sequence(seq)
    want = oracle.pssfp(t, seq, "f64")
    got = ca.simulate_magnetization(p, s).collect()
    assert rel(got, want) < 1e-6
    out = [a.collect() for a in ca.simulate_magnetization_tangents((ca.T1, ca.T2), p, s, echos=True)]
    assert rel(out[0], want) < 1e-6
    for name, d in zip(("T1", "T2"), out[1:]):
        assert rel(d, central_difference(oracle.pssfp, t, seq, name)) < 2e-6
    traj = ca.SpiralTrajectory.from_trajectory(W.make_spiral(66, 32, 20.0, 8, 5e-6))
    coils = ca.CompasArray.from_numpy(np.ones((1, 3), np.complex64))
    server = ca.Server(slots=1, memory_budget=1 << 30)
    ticket = server.submit_simulate_signal(p, s, traj, coils)
    assert server.wait(ticket, timeout=60) is not None
    assert np.array_equal(server.result(ticket, 0).collect(), got)
    server.release(ticket)
    server.close()


@pytest.mark.parametrize("nz,tangents", [(35, True), (200, False)], ids=["tangents", "simulation"])
def test_sums_of_groups_are_rounded_once(oracle, nz, tangents):
    """Slice positions in several groups: the sums are FP64 up to the echo, so the
    error is that of rounding the oracle's echoes to FP32.  FP32 planes of two or
    three groups would leave 1.15 times that or more; 1.03."""
    banner(f"pssfp map, rounding of {nz} positions")
    context()
    t = W.make_tissue(W.SplitMix64(77), 20, 20.0, 40.0)
    seq = train(80, 60.0, nz, 25, 0.0)
    p, s = ca.TissueParameters.from_tissue(t), ca.pSSFPSequence.from_sequence(seq)
    if tangents:
        got = ca.simulate_magnetization_tangents((ca.T1, ca.T2), p, s, echos=True)[0].collect()
    else:
        got = ca.simulate_magnetization(p, s).collect()
    want = oracle.pssfp(t, seq, "f64")
    once = rel(want.astype(np.complex64), want)
    print("error", rel(got, want), "of one rounding", once)
    assert rel(got, want) < 1.03 * once
