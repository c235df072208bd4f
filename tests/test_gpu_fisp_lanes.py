"""The complex FISP recursion in each of its layouts (one, two, four and eight
lanes per voxel) against the FP64 oracle, the top state in each of the last
places of its lane.  Tolerance: that of the other FISP parity tests, 1e-5."""

import numpy as np
import pytest

import compas_amd as ca
from compas_amd import workloads as W
from gpu_helpers import banner, context, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes,states", [(1, 1), (1, 2), (1, 32), (2, 2), (2, 3), (2, 31), (2, 63), (2, 64), (4, 4), (4, 5),
                                          (4, 13), (4, 14), (4, 62), (8, 9), (8, 16), (8, 17), (8, 23), (8, 121), (8, 128)])
def test_layout(oracle, monkeypatch, lanes, states):
    banner(f"fisp complex form, {states} states in {lanes} lanes")
    monkeypatch.setenv("COMPAS_FISP_LPV", str(lanes))
    context()
    t = W.make_tissue(W.SplitMix64(31), 9, 20.0, 40.0)
    seq = W.make_fisp(33, 60.0, states)
    n = np.arange(33)
    seq.RF = (seq.RF * np.exp(1j * np.deg2rad(117.0) * (n * (n + 1) // 2))).astype(np.complex64)
    got = ca.simulate_magnetization(ca.TissueParameters.from_tissue(t), ca.FispSequence.from_sequence(seq)).collect()
    assert rel(got, oracle.fisp(t, seq, "f64")) < 1e-5
