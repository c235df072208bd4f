"""The workloads whose speed matters to a user of this framework.

A program of such a user simulates the magnetisation of a tissue map under a
FISP or pSSFP sequence, turns it into k-space signal on a Cartesian or spiral
trajectory, and in a reconstruction forms derivatives and the products J.v and
J^H.y; a serving program has a request server do the same for many clients.
Every case goes through compas_amd, arrays stay on the GPU between calls and
results come back as torch tensors over the library's own memory.

Sizes are those of the benchmark workloads (4096 voxels x 256 TRs; 50176
voxels x 1120 TRs with FISP, Cartesian, 4 coils x 224 samples; the same with
pSSFP of 35 slice positions x 25 RF steps, spiral, 512 samples), of the
Gauss-Newton fits, of the serving mix, and odd sizes between them.
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "compas-toolkit_amd"))
import compas_amd as ca  # noqa: E402

DEV = "cuda:0"
TAU = 2 * math.pi


def listed():
    return [
        # a small scan simulated whole: one coil, 64 x 64 voxels; launches and latency count
        dict(name="fisp-signal-4096", kind="fisp_signal", nv=4096, ntr=256, states=16, nc=1, ns=64, b0=0.0),
        # a full slice simulated whole: the benchmark's default step
        dict(name="fisp-signal-50176", kind="fisp_signal", nv=50176, ntr=1120, states=25, nc=4, ns=224, b0=50.0),
        # a train with RF spoiling phases, two slice profiles, an undersampled
        # dictionary and a second repetition, at odd sizes
        dict(name="fisp-phased-20011", kind="fisp", nv=20011, ntr=301, states=37, b0=50.0, phased=True, slices=2,
             undersampling=2, repetitions=2),
        # linearisation of a Cartesian fit: echoes with their T1 and T2 derivatives
        dict(name="fisp-tangents-50176", kind="fisp_tangents", nv=50176, ntr=1120, states=25, b0=50.0),
        # pSSFP simulation of a full slice
        dict(name="pssfp-50176", kind="pssfp", nv=50176, ntr=1120, nz=35, nrf=25, b0=50.0),
        # linearisation of a spiral fit at the size of the Gauss-Newton example: all four derivatives
        dict(name="pssfp-tangents-3136", kind="pssfp_tangents", nv=3136, ntr=280, nz=35, nrf=25, b0=50.0),
        # spiral k-space signal of a full slice
        dict(name="spiral-signal-50176", kind="spiral_signal", nv=50176, nr=1120, ns=512, nc=4),
        # one product of the normal operator of a spiral fit: J.v and J^H.y
        dict(name="spiral-normal-50176", kind="spiral_normal", nv=50176, nr=1120, ns=512, nc=4),
        # one product of the normal operator of a small Cartesian fit: the inner step of conjugate gradients
        dict(name="cartesian-normal-1024", kind="cartesian_normal", nv=1024, nr=128, ns=32, nc=1, method="default"),
        # the same for a full slice and four coils
        dict(name="cartesian-normal-50176", kind="cartesian_normal", nv=50176, nr=1120, ns=224, nc=4, method="default"),
        # signal of given echoes at odd sizes, eight coils, in the low-precision mode
        dict(name="cartesian-signal-30011", kind="cartesian_signal", nv=30011, nr=777, ns=130, nc=8, method="low"),
        # a burst of requests to the server: both sequences and both trajectories
        dict(name="serve-burst", kind="serve", requests=8, nv_low=1000, nv_high=12000, ntr_low=250, ntr_high=600),
    ]


def _between(rng, low, high):
    """A whole number, spread over the logarithm of the range."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["fisp_signal", "fisp", "fisp_tangents", "pssfp", "pssfp_tangents", "spiral_signal",
                       "spiral_normal", "cartesian_normal", "cartesian_signal", "serve"])
    while True:
        c = dict(kind=kind)
        if kind == "serve":
            c.update(requests=rng.randint(4, 10), nv_low=rng.randint(500, 2000), nv_high=rng.randint(4000, 12000),
                     ntr_low=rng.randint(200, 300), ntr_high=rng.randint(400, 700))
            return c
        c["nv"] = _between(rng, 1000, 60000)
        if kind.startswith("fisp"):
            c.update(ntr=_between(rng, 100, 1500), states=_between(rng, 5, 64), b0=rng.choice([0.0, 50.0, 50.0]))
            if c["nv"] * c["ntr"] * c["states"] > 50176 * 1120 * 25:
                continue
            if kind == "fisp_signal":
                c.update(nc=rng.randint(1, 8), ns=rng.choice([32, 64, 96, 100, 128, 131, 192, 224]))
                if c["nv"] * c["ntr"] * c["nc"] * c["ns"] > 50176 * 1120 * 4 * 224:
                    continue
            elif kind == "fisp":
                c.update(phased=rng.random() < 0.5, slices=rng.choice([1, 1, 2, 3]),
                         undersampling=rng.choice([1, 1, 2]), repetitions=rng.choice([1, 1, 2]))
        elif kind.startswith("pssfp"):
            c.update(ntr=_between(rng, 100, 1200), nz=rng.randint(1, 48), nrf=rng.randint(8, 40), b0=rng.choice([0.0, 50.0, 50.0]),
                     phased=rng.random() < 0.25)
            most = 50176 * 1120 * 35 * 25
            if c["nv"] * c["ntr"] * c["nz"] * c["nrf"] > (most if kind == "pssfp" else most // 12):
                continue
        else:
            c.update(nr=_between(rng, 60, 1200), nc=rng.randint(1, 8))
            if kind.startswith("spiral"):
                c.update(ns=_between(rng, 48, 1024))
                if kind == "spiral_normal":
                    c["nc"] = min(c["nc"], 4)
                most = 50176 * 1120 * 4 * 512
            else:
                c.update(ns=_between(rng, 32, 256), method=rng.choice(["default", "default", "low", "direct"]))
                most = 50176 * 1120 * 4 * 224 // (8 if c["method"] == "direct" else 1)
            if c["nv"] * c["nr"] * c["ns"] * c["nc"] > most:
                continue
        return c


# ------------------------------------------------------------------ inputs ---


class Inputs:
    """The numbers of a case, as numpy float32 / complex64 on the host and, for
    arrays of echo size, torch complex64 on the GPU."""


def _tissue(o, rng, nv, b0):
    n = math.isqrt(nv - 1) + 1
    T1 = np.exp(rng.uniform(math.log(0.1), math.log(4.0), nv))
    T2 = np.exp(rng.uniform(math.log(0.01), np.log(np.minimum(1.0, T1))))
    o.nv, o.T1, o.T2 = nv, T1.astype(np.float32), T2.astype(np.float32)
    o.B1 = rng.uniform(0.8, 1.2, nv).astype(np.float32)
    o.B0 = rng.uniform(-b0, b0, nv).astype(np.float32) if b0 else np.zeros(nv, np.float32)
    o.rho = (rng.uniform(0.5, 1.0, nv) * np.exp(1j * rng.uniform(0, TAU, nv))).astype(np.complex64)
    o.fov, o.n = 22.4, n
    c = (np.arange(n) - n // 2) * (o.fov / n)
    o.x = np.tile(c, n)[:nv].astype(np.float32)
    o.y = np.repeat(c, n)[:nv].astype(np.float32)


def _coils(o, rng, nc):
    centres = [(0.35, 0.0), (-0.35, 0.0), (0.0, 0.35), (0.0, -0.35)]
    maps = []
    for j in range(nc):
        cx, cy = centres[j % 4]
        d2 = (o.x / o.fov - cx) ** 2 + (o.y / o.fov - cy) ** 2
        maps.append(np.exp(-d2 / (2 * 0.35 ** 2)) * np.exp(1j * rng.uniform(0, TAU)))
    o.coils = np.array(maps).astype(np.complex64)


def _flips(rng, ntr, low, high):
    """A smooth train of positive flip angles in degrees."""
    return rng.uniform(low, high) * np.sin(np.pi * (np.arange(ntr) + 0.5) / ntr)


def _fisp(o, rng, case):
    ntr, slices = case["ntr"], case.get("slices", 1)
    rf = _flips(rng, ntr, 55, 70).astype(np.complex128)
    profiles = np.ones((slices, ntr), np.complex128)
    if slices > 1:
        profiles *= np.linspace(1.0, 0.5, slices)[:, None]
    if case.get("phased"):
        k = np.arange(ntr)
        rf *= np.exp(1j * np.deg2rad(117.0) * (k * (k + 1) // 2 % 360))  # RF spoiling
        profiles = profiles * np.exp(0.2j * np.arange(slices))[:, None]
    o.RF, o.profiles = rf.astype(np.complex64), profiles.astype(np.complex64)
    o.TR, o.TE, o.TI, o.TW = 8.7e-3, 4.35e-3, 20e-3, 0.5 if case.get("repetitions", 1) > 1 else 0.0
    o.states, o.undersampling, o.repetitions = case["states"], case.get("undersampling", 1), case.get("repetitions", 1)


def _pssfp(o, rng, case):
    ntr, nrf = case["ntr"], case["nrf"]
    t = -1.0 + 2.0 * (np.arange(nrf) + 0.5) / nrf
    w = np.sinc(3 * t) * np.exp(-t ** 2 / 0.5)
    o.grf = (np.pi / 180 * w / w.sum()).astype(np.complex64)
    phase = np.pi * (np.arange(ntr) % 2)
    if case.get("phased"):
        phase = phase + 1.5 * np.sin(TAU * np.arange(ntr) / 96)
    o.RF = (_flips(rng, ntr, 55, 70) * np.exp(1j * phase)).astype(np.complex64)
    if not case.get("phased"):
        o.RF.imag = 0
    o.TR, o.dt = 10e-3, (1e-3 / nrf, 20e-3, (10e-3 - 1e-3) / 2)
    o.grz = (0.002 / nrf, 0.0, -0.01)
    o.z = np.linspace(-1, 1, case["nz"]).astype(np.float32) if case["nz"] > 1 else np.zeros(1, np.float32)


def _cartesian(o, nr, ns):
    dk = TAU / o.fov
    ky = (np.arange(nr) % o.n) - o.n // 2
    o.nr, o.ns, o.dt_s = nr, ns, 5e-6
    o.k_start = (-ns / 2 * dk + 1j * ky * dk).astype(np.complex64)
    o.dk = np.float32(dk)


def _spiral(o, rng, nr, ns):
    dx = o.fov / o.n
    e = np.exp(1j * (np.deg2rad(111.246) * np.arange(nr) + rng.uniform(0, TAU)))
    o.nr, o.ns, o.dt_s = nr, ns, 5e-6
    o.k_start = (-(np.pi / dx) * e).astype(np.complex64)
    o.dk = (TAU / dx / ns * e).astype(np.complex64)


def _echo_like(gen, nr, nv, scale):
    """Smooth signal evolutions over the readouts, different in every voxel."""
    k = torch.arange(10, device=DEV, dtype=torch.float32)
    t = (torch.arange(nr, device=DEV, dtype=torch.float32) + 0.5) / nr
    basis = torch.cos(math.pi * t[:, None] * k[None, :]) / (1 + k[None, :])
    w = torch.view_as_complex(torch.randn(10, nv, 2, device=DEV, generator=gen))
    return (scale * basis.to(torch.complex64)) @ w


def _inputs(case, seed):
    rng = np.random.default_rng([seed, 20])
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    o, kind = Inputs(), case["kind"]
    _tissue(o, rng, case["nv"], case.get("b0", 50.0))
    if kind.startswith("fisp"):
        _fisp(o, rng, case)
    elif kind.startswith("pssfp"):
        _pssfp(o, rng, case)
    if "nc" in case:
        _coils(o, rng, case["nc"])
        if kind.startswith("spiral"):
            _spiral(o, rng, case["nr"], case["ns"])
        else:
            _cartesian(o, case.get("nr", case.get("ntr")), case["ns"])
    if kind in ("spiral_signal", "spiral_normal", "cartesian_normal", "cartesian_signal"):
        o.m = _echo_like(gen, o.nr, o.nv, 0.2)
    if kind in ("spiral_normal", "cartesian_normal"):
        fields = 4 if kind == "spiral_normal" else 2
        o.dm = [_echo_like(gen, o.nr, o.nv, s) for s in (0.05, 0.5, 0.2, 0.02)[:fields]]
        o.v = torch.view_as_complex(torch.randn(fields + 2, o.nv, 2, device=DEV, generator=gen))
        o.res = torch.view_as_complex(torch.randn(case["nc"], o.nr, o.ns, 2, device=DEV, generator=gen))
    return o


def _requests(case, seed):
    """The requests of a burst: FISP or pSSFP, Cartesian or spiral, in turn."""
    rng = np.random.default_rng([seed, 21])
    sizes = np.random.default_rng([case[k] for k in sorted(case) if k.startswith(("requests", "nv", "ntr"))])
    out = []
    for i in range(case["requests"]):
        o = Inputs()
        nv = int(math.exp(sizes.uniform(math.log(case["nv_low"]), math.log(case["nv_high"]))))
        nc = int(sizes.integers(1, 9))
        c = dict(ntr=int(sizes.integers(case["ntr_low"], case["ntr_high"] + 1)), states=25, nz=35, nrf=25)
        _tissue(o, rng, nv, 50.0)
        o.sequence = "pssfp" if i % 3 == 1 else "fisp"
        (_pssfp if o.sequence == "pssfp" else _fisp)(o, rng, c)
        _coils(o, rng, nc)
        o.trajectory = "spiral" if i % 4 in (1, 2) else "cartesian"
        if o.trajectory == "spiral":
            _spiral(o, rng, c["ntr"], 128)
        else:
            _cartesian(o, c["ntr"], 128)
        out.append(o)
    return out


# -------------------------------------------------------- the program's side ---

_SERVER = []


class State:
    """What a program keeps between calls: the library's objects and arrays."""


def _objects(s, o, sequence=None, trajectory=None):
    s.p = ca.TissueParameters(o.nv, o.T1, o.T2, o.B1, o.B0, o.rho.real, o.rho.imag, o.x, o.y)
    if sequence == "fisp":
        s.seq = ca.FispSequence(o.RF, o.profiles, o.TR, o.TE, o.states, o.TI, undersampling_factor=o.undersampling,
                                repetitions=o.repetitions, TW=o.TW)
    elif sequence == "pssfp":
        s.seq = ca.pSSFPSequence(o.RF, o.TR, o.grf, o.dt, o.grz, o.z)
    if trajectory:
        make = ca.SpiralTrajectory if trajectory == "spiral" else ca.CartesianTrajectory
        s.traj = make(o.nr, o.ns, o.dt_s, o.k_start, o.dk)
        s.coils = ca.CompasArray.from_numpy(o.coils)


def _start():
    try:
        ca.get_context()
    except ca.CompasError:
        ca.init_context(0)


def prepare(case, seed):
    _start()
    s, kind = State(), case["kind"]
    s.kind = kind
    if kind == "serve":
        if not _SERVER:
            _SERVER.append(ca.Server(slots=4, memory_budget=64 << 30))
        s.server, s.requests = _SERVER[0], []
        for o in _requests(case, seed):
            r = State()
            _objects(r, o, o.sequence, o.trajectory)
            s.requests.append(r)
        return s
    o = _inputs(case, seed)
    family = kind.split("_")[0]
    _objects(s, o, family if family in ("fisp", "pssfp") else None,
             "spiral" if family == "spiral" else "cartesian" if "nc" in case else None)
    if family in ("spiral", "cartesian"):
        s.m = ca.CompasArray.from_dlpack(o.m)
        if kind.endswith("normal"):
            s.dm = [ca.CompasArray.from_dlpack(d) for d in o.dm]
            s.v = ca.CompasArray.from_dlpack(o.v)
            s.res = ca.CompasArray.from_dlpack(o.res)
    s.method = case.get("method")
    return s


def run(s):
    if s.kind == "serve":
        tickets = [s.server.submit_simulate_signal(r.p, r.seq, r.traj, r.coils) for r in s.requests]
        out = []
        for t in tickets:
            s.server.wait(t)
            out.append(s.server.result(t, 1).to_torch())
            s.server.release(t)
        return out
    if s.kind in ("fisp", "pssfp"):
        return ca.simulate_magnetization(s.p, s.seq).to_torch()
    if s.kind == "fisp_signal":
        echos = ca.simulate_magnetization(s.p, s.seq)
        signal = ca.magnetization_to_signal(echos, s.p, s.traj, s.coils)
        return {"echos": echos.to_torch(), "signal": signal.to_torch()}
    if s.kind == "fisp_tangents":
        return [a.to_torch() for a in ca.simulate_magnetization_tangents((ca.T1, ca.T2), s.p, s.seq, echos=True)]
    if s.kind == "pssfp_tangents":
        fields = (ca.T1, ca.T2, ca.B1, ca.B0)
        return [a.to_torch() for a in ca.simulate_magnetization_tangents(fields, s.p, s.seq, echos=True)]
    if s.kind == "spiral_signal":
        return ca.magnetization_to_signal(s.m, s.p, s.traj, s.coils).to_torch()
    if s.kind == "spiral_normal":
        jv = ca.compute_jacobian_spiral(s.m, s.dm, s.p, s.traj, s.coils, s.v)
        jhy = ca.compute_jacobian_hermitian_spiral(s.m, s.dm, s.p, s.traj, s.coils, s.res)
        return {"jv": jv.to_torch(), "jhy": jhy.to_torch()}
    low = s.method == "low"
    direct = "direct" if s.method == "direct" else None
    if s.kind == "cartesian_signal":
        return ca.magnetization_to_signal(s.m, s.p, s.traj, s.coils, low_precision=low, method=direct).to_torch()
    jv = ca.compute_jacobian(s.m, s.dm, s.p, s.traj, s.coils, s.v, low_precision=low, method=direct)
    jhy = ca.compute_jacobian_hermitian(s.m, s.dm, s.p, s.traj, s.coils, s.res, low_precision=low, method=direct)
    return {"jv": jv.to_torch(), "jhy": jhy.to_torch()}


# -------------------------------------------------------------------- work ---


def work(case):
    """Inputs read once, outputs written once, and the operations of the
    mathematics: a real train moves each state by one real 3 x 3 matrix (18
    flop), a phased one by one on complex values (36); an isochromat's TR is
    at least one affine map of three components (24 flop) with its twelve
    entries found for that TR's flip angle (24); products take 8 flop for a
    complex multiply-add."""
    kind = case["kind"]
    if kind == "serve":
        nv, ntr = math.sqrt(case["nv_low"] * case["nv_high"]), (case["ntr_low"] + case["ntr_high"]) / 2
        n = case["requests"] * nv * ntr
        return {"bytes": case["requests"] * (nv * 80 + 4.5 * ntr * 128 * 8),
                "flops": n * (2 * 25 * 18 + 35 * 48) / 3 + n * 4.5 * 128 * 8}
    nv, nc, ns = case["nv"], case.get("nc", 0), case.get("ns", 0)
    nr = case.get("nr", case.get("ntr"))
    tissue, plane, kspace, coils = 32 * nv, 8 * nr * nv, 8 * nc * nr * ns, 8 * nc * nv
    mac = 8.0 * nc * nr * ns * nv
    if kind.startswith("fisp"):
        passes = case.get("slices", 1) * case.get("repetitions", 1)
        outs = 3 if kind == "fisp_tangents" else case.get("undersampling", 1)
        sets = 3 if kind == "fisp_tangents" else passes
        sim = (36.0 if case.get("phased") else 18.0) * case["states"] * nr * nv * sets
        return {"bytes": tissue + outs * plane + coils + kspace, "flops": sim + mac}
    if kind.startswith("pssfp"):
        sets = 5 if kind == "pssfp_tangents" else 1
        return {"bytes": tissue + sets * plane, "flops": 48.0 * case["nz"] * nr * nv * sets}
    if kind.endswith("signal"):
        return {"bytes": tissue + plane + coils + kspace, "flops": mac}
    planes = 5 if kind.startswith("spiral") else 3
    return {"bytes": 2 * (tissue + planes * plane + coils + kspace) + 16 * (planes + 1) * nv, "flops": 4 * mac}


# ------------------------------------------------------- the same in 64 bits ---


def _f64(a):
    return torch.from_numpy(np.ascontiguousarray(a).astype(np.complex128 if np.iscomplexobj(a) else np.float64)).to(DEV)


def _fields64(o):
    return {k: _f64(getattr(o, k)) for k in ("T1", "T2", "B1", "B0")}


def _f32(v):
    return float(np.float32(v))


def _exact_fisp(o, t):
    """Extended phase graph of F+, F- and Z, state by state of the textbook form."""
    T1, T2, B1, B0 = t["T1"], t["T2"], t["B1"], t["B0"]
    TR, TE, TI, TW = _f32(o.TR), _f32(o.TE), _f32(o.TI), _f32(o.TW)
    e1 = lambda dt: torch.exp(-dt / T1)  # noqa: E731
    f = lambda dt: torch.polar(torch.exp(-dt / T2), TAU * dt * B0)  # noqa: E731
    ntr, N = o.RF.shape[0], o.states
    rf64 = o.RF.astype(np.complex128)
    out = torch.zeros(ntr, o.nv, dtype=torch.complex128, device=DEV)
    E1a, E1b, Fa, Fb = e1(TE), e1(TR - TE), f(TE), f(TR - TE)
    Ca, Cb = Fa.conj().resolve_conj(), Fb.conj().resolve_conj()
    for prof in o.profiles.astype(np.complex128):
        rf = prof * rf64
        p, q, z = (torch.zeros(N, o.nv, dtype=torch.complex128, device=DEV) for _ in range(3))
        z[0] = 1
        for rep in range(o.repetitions):
            p.zero_(), q.zero_()
            z *= -e1(TI)
            z[0] += 1 - e1(TI)
            for n in range(ntr):
                a, ph = np.deg2rad(abs(rf[n])) * B1, complex(np.exp(1j * np.angle(rf[n])))
                c2, s2, sa = torch.cos(a / 2) ** 2, torch.sin(a / 2) ** 2, torch.sin(a)
                pn = c2 * p + (ph * ph * s2) * q + (-1j * ph * sa) * z
                qn = c2 * q + (s2 / (ph * ph)) * p + (1j / ph * sa) * z
                z = torch.cos(a) * z + (-0.5j / ph * sa) * p + (0.5j * ph * sa) * q
                pn *= Fa
                z *= E1a
                z[0] += 1 - E1a
                if rep == o.repetitions - 1:
                    out[n] += pn[0]
                qn *= Ca * Cb
                pn *= Fb
                z *= E1b
                z[0] += 1 - E1b
                p, q = torch.zeros_like(p), torch.zeros_like(q)
                p[1:], q[:-1] = pn[:-1], qn[1:]
                p[0] = q[0].conj()
            p.zero_(), q.zero_()
            z *= e1(TW)
            z[0] += 1 - e1(TW)
    return out.repeat_interleave(o.undersampling, 0)


def _exact_pssfp(o, t):
    """Isochromats: Rodrigues' rotation per RF step, summed over the slice positions.
    The tissue fields may be complex (a complex step gives the derivative)."""
    z = _f64(o.z)[:, None]
    T1, T2, B1, B0 = (t[k][None, :] for k in ("T1", "T2", "B1", "B0"))
    ex, inv, pr = (_f32(v) for v in o.dt)
    gex, _, gpr = (_f32(v) for v in o.grz)
    rf, grf = o.RF.astype(np.complex128), o.grf.astype(np.complex128)
    decay = lambda dt: (torch.exp(-dt / T1), torch.exp(-dt / T2))  # noqa: E731
    e1, e2 = decay(ex)
    p1, p2 = decay(pr)
    i1, _ = decay(inv)
    shape = (z.shape[0], T1.shape[1])
    kind = torch.result_type(T1, B0 + B1 + T2)
    mx, my = torch.zeros(shape, dtype=kind, device=DEV), torch.zeros(shape, dtype=kind, device=DEV)
    mz = (torch.cos(math.pi * B1) * i1 + 1 - i1).expand(shape).to(kind).clone()
    az = -(gex * z) - TAU * ex * B0
    az2 = az * az
    out = []

    def excite(theta, mx, my, mz):
        for g in grf:
            w = theta * g
            ax, ay = w.real * B1, -w.imag * B1
            u = az2 + (ax * ax + ay * ay)
            a = torch.sqrt(u)
            s1, s2 = torch.sin(a) / a, 0.5 * (torch.sin(0.5 * a) / (0.5 * a)) ** 2
            d = s2 * (ax * mx + ay * my + az * mz)
            c = 1 - u * s2
            nx = c * mx + s1 * (ay * mz - az * my) + d * ax
            ny = c * my + s1 * (az * mx - ax * mz) + d * ay
            nz = c * mz + s1 * (ax * my - ay * mx) + d * az
            mx, my, mz = nx * e2, ny * e2, nz * e1 + (1 - e1)
        return mx, my, mz

    def turn(k, mx, my, mz):
        a = -(k * gpr * z) - TAU * pr * B0
        c, s = torch.cos(a), torch.sin(a)
        return (c * mx - s * my) * p2, (c * my + s * mx) * p2, mz * p1 + (1 - p1)

    az = torch.where(az2 == 0, torch.full_like(az, 1e-30), az)
    az2 = torch.where(az2 == 0, torch.full_like(az2, 1e-30), az2)
    mx, my, mz = turn(2.0, *excite(-0.5 * rf[0], mx, my, mz))
    for n in range(rf.shape[0]):
        mx, my, mz = turn(1.0, *excite(rf[n], mx, my, mz))
        out.append((mx.sum(0), my.sum(0)))
        mx, my, mz = turn(1.0, mx, my, mz)
    return torch.stack([a for a, _ in out]), torch.stack([b for _, b in out])


def _sample_factors(o, r=None):
    """Phase and decay exponents: value at sample 0 and step per sample."""
    T2, B0, x, y = _f64(o.T2), _f64(o.B0), _f64(o.x), _f64(o.y)
    dt = _f32(o.dt_s)
    rate = torch.complex(-dt / T2, TAU * dt * B0)
    if r is None:
        step = float(o.dk) * x
        k0 = -0.5 * o.ns * step
    else:
        dk = o.dk.astype(np.complex128)[r]
        step = dk.real * x + dk.imag * y
        k0 = float(o.k_start.real[r]) * x
    return torch.complex(torch.zeros_like(x), k0) - 0.5 * o.ns * rate, torch.complex(torch.zeros_like(x), step) + rate


def _exact_signal(o, m):
    coils, rho = _f64(o.coils), _f64(o.rho)
    s = torch.arange(o.ns, device=DEV, dtype=torch.float64)
    if np.ndim(o.dk) == 0:
        first, step = _sample_factors(o)
        E = torch.exp(first[:, None] + step[:, None] * s) * rho[:, None]
        return torch.stack([m.to(torch.complex128) @ (E * c[:, None]) for c in coils])
    out = torch.empty(coils.shape[0], o.nr, o.ns, dtype=torch.complex128, device=DEV)
    for r in range(o.nr):
        first, step = _sample_factors(o, r)
        amp = m[r].to(torch.complex128) * rho * torch.exp(first)
        out[:, r] = (coils * amp) @ torch.exp(step[:, None] * s)
    return out


def _exact_normal(o):
    """J.v and J^H.y: T1 and T2 rows scaled by T1 and T2, then B1, B0 (spiral), then the density."""
    coils, rho, T1, T2 = _f64(o.coils), _f64(o.rho), _f64(o.T1), _f64(o.T2)
    spiral = np.ndim(o.dk) > 0
    dt, v = _f32(o.dt_s), o.v.to(torch.complex128)
    scale = [T1, T2, torch.ones_like(T1), torch.ones_like(T1)][: len(o.dm)]
    s = torch.arange(o.ns, device=DEV, dtype=torch.float64)
    sp = s - 0.5 * o.ns
    rate = [None, dt / T2 ** 2, None, 1j * TAU * dt * torch.ones_like(T1)][: len(o.dm)]
    k, nc = len(o.dm), coils.shape[0]
    jv = torch.empty(nc, o.nr, o.ns, dtype=torch.complex128, device=DEV)
    jhy = torch.zeros(k + 2, o.nv, dtype=torch.complex128, device=DEV)
    step = 1 if spiral else 64
    for r0 in range(0, o.nr, step):
        rows = slice(r0, min(o.nr, r0 + step))
        if spiral or r0 == 0:
            first, inc = _sample_factors(o, r0 if spiral else None)
            E = torch.exp(first[:, None] + inc[:, None] * s)
        m = o.m[rows].to(torch.complex128)
        dm = [d[rows].to(torch.complex128) for d in o.dm]
        a = rho * sum(v[i] * scale[i] * dm[i] for i in range(k)) + (v[k] + 1j * v[k + 1]) * m
        b = rho * m * sum(v[i] * scale[i] * rate[i] for i in range(k) if rate[i] is not None)
        Ec = E.conj().resolve_conj().T
        ab = torch.cat([(coils[:, None] * x).reshape(-1, o.nv) for x in (a, b)]) @ E
        ab = ab.reshape(2, nc, -1, o.ns)
        jv[:, rows] = ab[0] + ab[1] * sp
        y = o.res[:, rows].to(torch.complex128)
        uw = (torch.cat([y.reshape(-1, o.ns), (y * sp).reshape(-1, o.ns)]) @ Ec).reshape(2, nc, -1, o.nv)
        U, W = (torch.conj(coils) * x for x in [(uw[i].transpose(0, 1)) for i in (0, 1)])
        U, W = U.sum(1), W.sum(1)
        for i in range(k):
            g = (dm[i].conj() * U).sum(0)
            if rate[i] is not None:
                g = g + (m.conj() * W).sum(0) * torch.conj(rate[i] * torch.ones_like(rho))
            jhy[i] += torch.conj(rho * scale[i]) * g
        u = (m.conj() * U).sum(0)
        jhy[k] += u
        jhy[k + 1] += -1j * u
    return {"jv": jv, "jhy": jhy}


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve":
        out = []
        for o in _requests(case, seed):
            t = _fields64(o)
            m = _exact_fisp(o, t) if o.sequence == "fisp" else torch.complex(*_exact_pssfp(o, t))
            out.append(_exact_signal(o, m))
        return out
    o = _inputs(case, seed)
    if kind in ("spiral_normal", "cartesian_normal"):
        return _exact_normal(o)
    if kind in ("spiral_signal", "cartesian_signal"):
        return _exact_signal(o, o.m)
    t = _fields64(o)
    if kind == "fisp":
        return _exact_fisp(o, t)
    if kind == "fisp_signal":
        m = _exact_fisp(o, t)
        return {"echos": m, "signal": _exact_signal(o, m)}
    if kind == "fisp_tangents":
        out = [_exact_fisp(o, t)]
        for k in ("T1", "T2"):  # fourth-order central differences
            h = 2e-4 * t[k]
            f = [_exact_fisp(o, dict(t, **{k: t[k] + i * h})) for i in (-2, -1, 1, 2)]
            out.append((8 * (f[2] - f[1]) - (f[3] - f[0])) / (12 * h))
        return out
    if kind == "pssfp":
        return torch.complex(*_exact_pssfp(o, t))
    out = [torch.complex(*_exact_pssfp(o, t))]
    for k in ("T1", "T2", "B1", "B0"):  # complex step
        x, y = _exact_pssfp(o, dict(t, **{k: torch.complex(t[k], torch.full_like(t[k], 1e-30))}))
        out.append(torch.complex(x.imag, y.imag) / 1e-30)
    return out
