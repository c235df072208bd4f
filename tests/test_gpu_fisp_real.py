"""FISP trains of real pulses (fisp_real.h) against the FP64 oracle, where the
layout or the form changes: one lane per voxel and several, the options that
leave the plain loop, flip angles of either sign and beyond the polynomial's
range, and trains that are real but for one pulse (the complex form).

Tolerance: the recursion is the one the complex form runs, in FP32, with fewer
roundings; 1e-5 (echoes) and 1e-4 (tangents) relative to FP64 are the bounds of
the complex form over trains of this length.
"""

import numpy as np
import pytest

import compas_amd as ca
from compas_amd import workloads as W
from gpu_helpers import banner, context, rel
from test_gpu_parity import central_difference

pytestmark = pytest.mark.gpu

MAG_TOL = 1e-5
TANGENT_TOL = 1e-4


def case(nv, nTR, N, deg=60.0, b0=40.0):
    n = int(np.ceil(np.sqrt(nv)))
    t = W.make_tissue(W.SplitMix64(31), n, 20.0, b0).slice(0, nv)
    seq = W.make_fisp(nTR, deg, N)
    seq.RF = (seq.RF * np.where(np.arange(nTR) % 3 == 1, -1.0, 1.0)).astype(np.complex64)
    return t, seq


# (voxels, states) by the layout rule for 1024 SIMDs: 33 voxels take eight lanes
# from seven states on, 30000 one or two, 80000 one, and four for 40 states
LAYOUTS = [(33, 1), (33, 2), (33, 7), (33, 8), (33, 9), (33, 25), (33, 33), (33, 63), (33, 128), (30000, 3),
           (30000, 25), (30000, 32), (80000, 13), (80000, 32), (80000, 40)]


@pytest.mark.parametrize("nv,N", LAYOUTS)
def test_layouts(oracle, nv, N):
    banner(f"fisp real layouts {nv} voxels {N} states")
    context()
    t, seq = case(nv, 30, N)
    got = ca.simulate_magnetization(ca.TissueParameters.from_tissue(t), ca.FispSequence.from_sequence(seq)).collect()
    assert rel(got, oracle.fisp(t, seq, "f64")) < MAG_TOL


# every lane count with the top state in each of the last places of its lane
@pytest.mark.parametrize("lanes,N", [(1, 1), (1, 2), (1, 32), (2, 2), (2, 3), (2, 31), (2, 32), (4, 4), (4, 5), (4, 6), (4, 7),
                                     (4, 13), (4, 14), (4, 15), (4, 16), (4, 61), (4, 62), (4, 63), (4, 64), (8, 9), (8, 23),
                                     (8, 121), (8, 125), (8, 128)])
def test_lanes(oracle, monkeypatch, lanes, N):
    banner(f"fisp real, {N} states in {lanes} lanes")
    monkeypatch.setenv("COMPAS_FISP_LPV", str(lanes))
    context()
    t, seq = case(9, 33, N)
    got = ca.simulate_magnetization(ca.TissueParameters.from_tissue(t), ca.FispSequence.from_sequence(seq)).collect()
    assert rel(got, oracle.fisp(t, seq, "f64")) < MAG_TOL


@pytest.mark.parametrize("name,options", [
    ("slices", dict(profiles=np.stack([np.linspace(0.6, 1.1, 26), np.full(26, -0.9)]))),
    ("undersampled", dict(undersampling=3)),
    ("repetitions", dict(repetitions=3, TW=0.12)),
    ("no inversion", dict(repetitions=2, TW=0.12, inversion=False)),
    ("no spoiling", dict(repetitions=2, TW=0.12, wait_spoiling=False)),
    ("neither", dict(repetitions=2, TW=0.12, inversion=False, wait_spoiling=False)),
    ("neither once", dict(inversion=False, wait_spoiling=False)),
    ("wide angles", dict(deg=9000.0)),
    ("one pulse off axis", dict(off=1e-3)),
    ("imaginary", dict(off=None)),
])
@pytest.mark.parametrize("fields", [None, (ca.T1, ca.T2), (ca.T1, ca.T2, ca.B1, ca.B0), (ca.B0,), (ca.B1,)],
                         ids=["echoes", "T1T2", "all", "B0", "B1"])
def test_options(oracle, name, options, fields):
    banner(f"fisp real options {name} {fields}")
    context()
    options = dict(options)
    t, seq = case(70, 26, 11, deg=options.pop("deg", 60.0))
    if "off" in options:
        off = options.pop("off")
        seq.RF = (1j * seq.RF) if off is None else seq.RF * np.exp(1j * off * (np.arange(26) == 12))
        seq.RF = seq.RF.astype(np.complex64)
    for k, v in options.items():
        setattr(seq, k, np.asarray(v, np.complex64) if k == "profiles" else v)
    p, s = ca.TissueParameters.from_tissue(t), ca.FispSequence.from_sequence(seq)
    if name == "wide angles":
        # an angle of 157 rad is itself rounded to 1e-5 rad; 26 pulses of that
        # and their products leave 1e-3 (derivatives are not compared)
        tol_m, tol_t = 1e-3, None
    else:
        tol_m, tol_t = MAG_TOL, TANGENT_TOL
    if fields is None:
        assert rel(ca.simulate_magnetization(p, s).collect(), oracle.fisp(t, seq, "f64")) < tol_m
        return
    out = [a.collect() for a in ca.simulate_magnetization_tangents(fields, p, s, echos=True)]
    assert rel(out[0], oracle.fisp(t, seq, "f64")) < tol_m
    bare = [a.collect() for a in ca.simulate_magnetization_tangents(fields, p, s, echos=False)]
    for f, d, b in zip(fields, out[1:], bare):
        assert np.array_equal(d, b)
        if tol_t:
            assert rel(d, central_difference(oracle.fisp, t, seq, ["T1", "T2", "B1", "B0"][f])) < tol_t


@pytest.mark.parametrize("nv,N", [(33, 1), (33, 8), (33, 9), (33, 17), (33, 128), (40000, 2), (40000, 9), (40000, 32)])
def test_tangent_layouts(oracle, nv, N):
    banner(f"fisp real tangent layouts {nv} voxels {N} states")
    context()
    t, seq = case(nv, 14, N)
    p, s = ca.TissueParameters.from_tissue(t), ca.FispSequence.from_sequence(seq)
    for fields in ((ca.T1, ca.T2), (ca.T1, ca.T2, ca.B1, ca.B0)):
        out = [a.collect() for a in ca.simulate_magnetization_tangents(fields, p, s, echos=True)]
        assert rel(out[0], oracle.fisp(t, seq, "f64")) < MAG_TOL
        for f, d in zip(fields, out[1:]):
            assert rel(d, central_difference(oracle.fisp, t, seq, ["T1", "T2", "B1", "B0"][f])) < TANGENT_TOL
