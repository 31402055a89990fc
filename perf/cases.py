"""The engine's timed workloads: what programs that use it have it do, through
its public Python entry points.

listed() names twelve of them, draw() gives more of the same ranges.  Kinds:

  job      a circuit through the job / circuit API, from gate list to shots,
           probabilities, amplitudes or <Z> on the host ("scheduler": the
           drop-in moonlab_scheduler_run; "qgtl": moonlab_qgtl_execute;
           "ex": moonlab_mi355x_execute_ex)
  state    a gate list on a resident state, then <Z> of every qubit: one
           kernel per gate ("gates"), fused blocks on the matrix cores
           ("fused") or cache-blocked passes ("blocked")
  hea      energies of many hardware-efficient-ansatz instances of the
           transverse-field Ising chain, packed once (a parameter loop)
  heagrad  energies and parameter-shift gradients of such instances
  qng      one natural-gradient step of a Pauli-sum Hamiltonian: gradients,
           then the regularized metric solve
  vqe      Pauli-sum energies of several parameter sets
  readout  observables, shots and a collapsing measurement of a resident state
  serve    a burst of requests of mixed sizes through the serving loop

Values that a complex64 state yields are single precision whatever type they
come back in, so they are returned as float32, <Z> as P(1) = (1 - <Z>) / 2
(<Z> of a deep circuit is a small difference of two halves of the norm);
complex64 cases ask for no shots (an outcome is the side of a rounded boundary
a draw falls on).
"""
import math

import numpy as np
import torch

import moonlab_amd as m
from moonlab_amd import workloads
from moonlab_amd import GateType as G

C128, C64 = m.C128, m.C64


def listed():
    return [
        # the smallest job a scheduler client submits: latency of the drop-in API
        {"name": "job_10q", "kind": "job", "api": "scheduler", "n": 10, "depth": 10, "shots": 1024,
         "prec": C128, "amps": False},
        # a control-plane circuit: probabilities and shots of a mid-sized register
        {"name": "circuit_14q", "kind": "job", "api": "qgtl", "n": 14, "depth": 12, "shots": 4096,
         "prec": C128, "amps": True},
        # the 20-qubit, depth-20 circuit with amplitudes, <Z> and shots read back
        {"name": "job_20q", "kind": "job", "api": "ex", "n": 20, "depth": 20, "shots": 1024,
         "prec": C128, "amps": True},
        # the 30-qubit bandwidth sweep (two layers of it): one kernel per gate on 16 GiB
        {"name": "sweep_30q", "kind": "state", "path": "gates", "n": 30, "depth": 2, "prec": C128, "fuse": 0},
        # a large single-precision state, SU(2) + CZ layers as fused blocks
        {"name": "fused_31q_c64", "kind": "state", "path": "fused", "n": 31, "depth": 12, "prec": C64, "fuse": 5},
        # the largest complex128 register most users run, cache-blocked
        {"name": "blocked_30q", "kind": "state", "path": "blocked", "n": 30, "depth": 10, "prec": C128, "fuse": 0},
        # an odd-sized single-precision register, a deeper circuit
        {"name": "blocked_27q_c64", "kind": "state", "path": "blocked", "n": 27, "depth": 25, "prec": C64,
         "fuse": 0},
        # a parameter sweep: thousands of small uneven circuits in one launch
        {"name": "hea_4096", "kind": "hea", "count": 4096, "n_lo": 8, "n_hi": 18, "l_lo": 4, "l_hi": 12,
         "prec": C128},
        # one optimizer step of one mid-sized ansatz: 193 shifted circuits
        {"name": "heagrad_12q", "kind": "heagrad", "count": 1, "n_lo": 12, "n_hi": 12, "l_lo": 4, "l_hi": 4,
         "prec": C128},
        # a quantum-natural-gradient step of a molecule-sized Hamiltonian
        {"name": "qng_8q", "kind": "qng", "count": 1, "n": 8, "layers": 3, "terms": 40, "prec": C128},
        # reading a prepared 24-qubit state out
        {"name": "readout_24q", "kind": "readout", "n": 24, "shots": 2048, "strings": 8, "prec": C128},
        # 48 requests that arrived together, small ones among large ones
        {"name": "serve_48", "kind": "serve", "count": 48, "n_lo": 10, "n_hi": 24, "d_lo": 10, "d_hi": 50},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["job", "job", "state", "state", "state", "hea", "heagrad", "qng", "vqe", "readout", "serve"])
    if kind == "job":
        api = rng.choice(["scheduler", "qgtl", "ex"])
        prec = rng.choice([C128, C64]) if api == "ex" else C128
        return {"kind": kind, "api": api, "n": rng.randint(3, 21), "depth": _log_int(rng, 2, 40),
                "shots": 0 if prec == C64 else _log_int(rng, 1, 4096), "prec": prec, "amps": rng.random() < 0.5}
    if kind == "state":
        path = rng.choice(["gates", "fused", "blocked", "blocked"])
        n = rng.randint(11, 28)
        return {"kind": kind, "path": path, "n": n, "depth": rng.randint(1, 6) if path == "gates" else
                _log_int(rng, 2, 30), "prec": rng.choice([C128, C64]),
                "fuse": rng.randint(3, 5) if path == "fused" else 0}
    if kind in ("hea", "heagrad"):
        lo = rng.randint(3, 14)
        hi = rng.randint(lo, 18 if kind == "hea" else 15)
        llo = rng.randint(1, 6)
        count = _log_int(rng, 1, 1024) if kind == "hea" else rng.randint(1, 4)
        return {"kind": kind, "count": count, "n_lo": lo, "n_hi": hi, "l_lo": llo, "l_hi": rng.randint(llo, 8),
                "prec": C128}
    if kind == "qng":
        return {"kind": kind, "count": rng.randint(1, 3), "n": rng.randint(2, 11), "layers": rng.randint(1, 4),
                "terms": _log_int(rng, 4, 100), "prec": C128}
    if kind == "vqe":
        return {"kind": kind, "count": _log_int(rng, 1, 64), "n": rng.randint(3, 15), "layers": rng.randint(1, 6),
                "terms": _log_int(rng, 4, 100), "prec": C128}
    if kind == "readout":
        return {"kind": kind, "n": rng.randint(6, 28), "shots": _log_int(rng, 16, 8192),
                "strings": rng.randint(1, 12), "prec": C128}
    lo = rng.randint(4, 14)
    dlo = rng.randint(5, 20)
    return {"kind": "serve", "count": _log_int(rng, 4, 96), "n_lo": lo, "n_hi": rng.randint(lo + 2, 24),
            "d_lo": dlo, "d_hi": dlo + rng.randint(0, 30)}


# ---- inputs -------------------------------------------------------------------


class _Amplitudes:
    """A state's device amplitudes for torch (no copy); keeps the state alive."""

    def __init__(self, sv):
        self.sv = sv
        ptr = m.lib().moonlab_hip_state_device_ptr(sv.handle)
        self.__cuda_array_interface__ = {"shape": (1 << sv.n,), "typestr": "<c8" if sv.precision == C64 else "<c16",
                                         "data": (ptr, False), "strides": None, "version": 2}


def _view(sv):
    return torch.as_tensor(_Amplitudes(sv), device="cuda")


def _circuit(case, seed):
    if case.get("path") == "fused":
        return workloads.su2_cz_circuit(case["n"], case["depth"], seed)
    return workloads.random_layer_circuit(case["n"], case["depth"], seed, h_layer=True)


def _hea_instances(case, seed):
    # which sizes a case mixes is part of the case; the angles and fields are the seed's
    sizes, rng = np.random.default_rng(2026), np.random.default_rng(seed)
    out = []
    for _ in range(case["count"]):
        n = int(sizes.integers(case["n_lo"], case["n_hi"] + 1))
        L = int(sizes.integers(case["l_lo"], case["l_hi"] + 1))
        out.append((n, L, rng.uniform(0.0, 2.0 * math.pi, (L, n, 2)), float(rng.uniform(0.5, 1.5))))
    return out


def _pauli_string(rng, n, weight):
    s = ["I"] * n
    for q in rng.choice(n, size=min(n, weight), replace=False):
        s[int(q)] = "XYZ"[int(rng.integers(3))]
    return "".join(s)


def _vqe_instances(case, seed):
    rng = np.random.default_rng(seed)
    n, L = case["n"], case["layers"]
    terms = [(float(rng.normal()), _pauli_string(rng, n, int(rng.integers(1, 5)))) for _ in range(case["terms"])]
    return [{"n": n, "layers": L, "angles": rng.uniform(0.0, 2.0 * math.pi, (L, n, 2)), "terms": terms,
             "hf": (1 << (n // 2)) - 1, "constant": 0.5} for _ in range(case["count"])]


def _readout_ops(case, seed):
    rng = np.random.default_rng(seed)
    n = case["n"]
    return {"strings": [_pauli_string(rng, n, int(rng.integers(1, 7))) for _ in range(case["strings"])],
            "pairs": [tuple(int(q) for q in rng.choice(n, size=2, replace=False)) for _ in range(2)],
            "u": rng.random(case["shots"]), "measured": [int(q) for q in rng.choice(n, size=3, replace=False)],
            "u_measure": float(rng.random())}


def _requests(case, seed):
    sizes, rng = np.random.default_rng(2026), np.random.default_rng(seed)   # as _hea_instances
    ns = np.arange(case["n_lo"], case["n_hi"] + 1)
    w = 2.0 ** (-(ns - ns[0]) / 4.0)
    out = []
    for _ in range(case["count"]):
        n = int(sizes.choice(ns, p=w / w.sum()))
        prec = int(sizes.integers(2))
        depth = int(sizes.integers(case["d_lo"], case["d_hi"] + 1))
        out.append({"n": n, "gates": workloads.random_layer_circuit(n, depth, int(rng.integers(1 << 62))),
                    "shots": 0 if prec == C64 else 1024, "seed": int(rng.integers(1, 1 << 62)), "precision": prec})
    return out


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "job":
        g = _circuit(case, seed)
        h = m.Circuit(case["n"]) if case["api"] == "qgtl" else m.Job(case["n"])
        for row in g:
            t = int(row["type"])
            h.add_gate(t, int(row["target"]), int(row["control"]), float(row["theta"]) if t in (7, 8, 9) else None)
        s["handle"], s["seed"] = h, 2 * seed + 1
        if case["api"] != "qgtl":
            h.set_num_shots(max(case["shots"], 1)).set_num_workers(4).set_rng_seed(s["seed"])
    elif kind == "state":
        s["sv"] = m.StateVector(case["n"], case["prec"])
        s["gates"], s["view"] = _circuit(case, seed), _view(s["sv"])
    elif kind in ("hea", "heagrad"):
        s["batch"], s["pack"] = m.Batch(), m.HeaPack(_hea_instances(case, seed))
    elif kind in ("qng", "vqe"):
        s["batch"], s["inst"] = m.Batch(), _vqe_instances(case, seed)
    elif kind == "readout":
        s["sv"], s["work"] = m.StateVector(case["n"], case["prec"]), m.StateVector(case["n"], case["prec"])
        s["sv"].apply(workloads.random_layer_circuit(case["n"], 6, seed, h_layer=True), blocked=True).synchronize()
        s["view"] = _view(s["work"])
        s.update(_readout_ops(case, seed))
    else:
        s["server"], s["requests"] = m.Server(), _requests(case, seed)
    return s


# ---- one pass -------------------------------------------------------------------


def _z(z, prec):
    return (0.5 - 0.5 * np.asarray(z)).astype(np.float32) if prec == C64 else z


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "job":
        h = s["handle"]
        if case["api"] == "scheduler":
            return np.asarray(h.execute().outcomes, np.uint64)
        if case["api"] == "qgtl":
            r = h.execute(num_shots=case["shots"], rng_seed=s["seed"], return_probabilities=case["amps"])
            return [r.outcomes, r.probabilities]
        r = h.execute_ex(precision=case["prec"], amplitudes=case["amps"], expect_z=True,
                         skip_shots=case["shots"] == 0)
        amps = r.amplitudes
        if amps is not None and case["prec"] == C64:
            amps = amps.astype(np.complex64)
        return [r.outcomes, amps, _z(r.expect_z, case["prec"])]
    if kind == "state":
        sv = s["sv"].reset().apply(s["gates"], fuse=case["fuse"], blocked=case["path"] == "blocked")
        z, norm = sv.expect_z_all()
        return [s["view"], _z(z, case["prec"]), np.float32(norm) if case["prec"] == C64 else norm]
    if kind == "hea":
        return s["batch"].hea_tfim(s["pack"], case["prec"])
    if kind == "heagrad":
        e, g = s["batch"].hea_tfim_gradients(s["pack"], case["prec"])
        return [e, g]
    if kind == "vqe":
        return s["batch"].vqe_energies(s["inst"], case["prec"])
    if kind == "qng":
        e, g = s["batch"].vqe_gradients(s["inst"])
        d = s["batch"].vqe_natural_gradient(s["inst"], g)
        return [e, np.concatenate(g), np.concatenate([x[0] for x in d]), np.asarray([x[1] for x in d])]
    if kind == "readout":
        sv, w = s["sv"], s["work"]
        z, norm = sv.expect_z_all()
        zz = [sv.correlation_zz(a, b) for a, b in s["pairs"]]
        p = [sv.expect_pauli(t) for t in s["strings"]]
        shots = sv.sample(s["u"])
        r = w.copy_from(sv).measure_partial(s["measured"], s["u_measure"])
        ov = w.inner(sv)
        return [z, norm, np.asarray(zz + p), shots, r, np.asarray([ov.real, ov.imag]), s["view"]]
    srv = s["server"]
    tickets = [srv.submit(q["n"], q["gates"], shots=q["shots"], seed=q["seed"], precision=q["precision"])
               for q in s["requests"]]
    rs = [srv.wait(t) for t in tickets]
    by = [[r for r, q in zip(rs, s["requests"]) if q["precision"] == p] for p in (C128, C64)]
    cat = lambda xs: np.concatenate(xs) if xs else np.zeros(0)  # noqa: E731
    return [cat([r.expect_z for r in by[0]]), cat([r.outcomes for r in by[0]]),
            _z(cat([r.expect_z for r in by[1]]), C64)]


# ---- what one pass cannot do without ----------------------------------------------

#: real operations per amplitude of a gate: a full 2x2, a real or RX-form one, a phase on every amplitude
_FLOPS = {int(G.U3): 14, int(G.RX): 6, int(G.RY): 6, int(G.H): 6, int(G.RZ): 6}


def _gate_flops(gates, n):
    return float(sum(_FLOPS.get(int(t), 0) for t in gates["type"])) * 2.0 ** n


def work(case):
    kind = case["kind"]
    b = 8.0 if case.get("prec") == C64 else 16.0
    if kind in ("job", "state"):
        n, g = case["n"], _circuit(case, 1)
        flops, dim = _gate_flops(g, n) + 3.0 * 2.0 ** n, 2.0 ** n
        if kind == "state":   # the state written and read for <Z>; one kernel per gate moves it for every gate
            by = 2.0 * dim * b
            if case["path"] == "gates":
                by += float(workloads.algorithmic_bytes(g, n, int(b)))
            return {"bytes": by, "flops": flops}
        out = 8.0 * case["shots"] + (dim * (8.0 if case["api"] == "qgtl" else 16.0) if case["amps"] else 0.0)
        return {"bytes": 2.0 * dim * b + 40.0 * len(g) + out, "flops": flops}
    if kind in ("hea", "heagrad"):
        # every circuit's state lives and dies in the call: angles in, values out
        n, L = (case["n_lo"] + case["n_hi"]) / 2.0, (case["l_lo"] + case["l_hi"]) / 2.0
        sizes = range(case["n_lo"], case["n_hi"] + 1)
        amps = sum(2.0 ** k for k in sizes) / len(sizes)
        c = case["count"] * (1.0 + (4.0 * n * L if kind == "heagrad" else 0.0))
        return {"bytes": case["count"] * (16.0 * n * L + 8.0), "flops": c * amps * (L * 14.0 * n + 6.0 * n)}
    if kind in ("qng", "vqe"):
        n, P, dim = case["n"], 2.0 * case["n"] * case["layers"], 2.0 ** case["n"]
        one = dim * (7.0 * P + 4.0 * case["terms"])
        c = case["count"]
        if kind == "vqe":
            return {"bytes": c * (8.0 * P + 8.0) + 16.0 * case["terms"], "flops": c * one}
        return {"bytes": c * (24.0 * P + 8.0), "flops": c * ((1 + 2 * P) * one + (P + 1) * dim * 7.0 * P +
                                                            4.0 * (P + 1) ** 2 * dim)}
    if kind == "readout":   # the state read once for all observables; the copy written, collapsed and read
        dim = 2.0 ** case["n"]
        return {"bytes": 4.0 * dim * b, "flops": dim * (3.0 + 8.0 * case["strings"])}
    rs = _requests(case, 1)
    return {"bytes": sum(40.0 * len(q["gates"]) + 8.0 * (q["shots"] + q["n"]) for q in rs),
            "flops": sum(_gate_flops(q["gates"], q["n"]) for q in rs)}


# ---- the same values in 64 bits, by plain torch -------------------------------------

#: amplitudes times gates that plain torch applies in well under 20 seconds
_EXACT_MOST = 180.0 * 2.0 ** 30


def _mat(t, th=0.0, phi=0.0, lam=0.0):
    c, s = math.cos(th / 2), math.sin(th / 2)
    r = math.sqrt(0.5)
    return {int(G.H): [[r, r], [r, -r]], int(G.RX): [[c, -1j * s], [-1j * s, c]], int(G.RY): [[c, -s], [s, c]],
            int(G.RZ): [[complex(c, -s), 0], [0, complex(c, s)]], int(G.X): [[0, 1], [1, 0]],
            int(G.Y): [[0, -1j], [1j, 0]], int(G.Z): [[1, 0], [0, -1]],
            int(G.U3): [[c, -np.exp(1j * lam) * s], [np.exp(1j * phi) * s, np.exp(1j * (phi + lam)) * c]]}[int(t)]


def _apply_1q(a, q, u):
    """u (2 x 2 numbers, or 2 x 2 of [B, 1, 1] tensors) on qubit q of a [B, 2^n]."""
    v = a.view(a.shape[0], -1, 2, 1 << q)
    x, y = v[:, :, 0].clone(), v[:, :, 1].clone()
    v[:, :, 0] = u[0][0] * x + u[0][1] * y
    v[:, :, 1] = u[1][0] * x + u[1][1] * y


def _apply_2q(a, c, t, kind):
    lo, hi = min(c, t), max(c, t)
    v = a.view(a.shape[0], -1, 2, 1 << (hi - lo - 1), 2, 1 << lo)   # [.., hi, .., lo, ..]
    pick = lambda bc, bt: v[:, :, bc, :, bt] if c > t else v[:, :, bt, :, bc]  # noqa: E731
    if kind == int(G.CZ):
        pick(1, 1).neg_()
    else:   # CNOT
        x = pick(1, 0).clone()
        pick(1, 0).copy_(pick(1, 1))
        pick(1, 1).copy_(x)


def _zero(n, count=1):
    a = torch.zeros((count, 1 << n), dtype=torch.complex128, device="cuda")
    a[:, 0] = 1.0
    return a


def _simulate(gates, n):
    a = _zero(n)
    for row in gates:
        t = int(row["type"])
        if t in (int(G.CNOT), int(G.CZ)):
            _apply_2q(a, int(row["control"]), int(row["target"]), t)
        else:
            _apply_1q(a, int(row["target"]), _mat(t, float(row["theta"]), float(row["phi"]), float(row["lam"])))
    return a[0]


def _z_of(p, n):
    out = []
    for q in range(n):
        v = p.view(-1, 2, 1 << q)
        out.append((v[:, 0].sum() - v[:, 1].sum()).item())
    return np.asarray(out)


def _exact_z(z, prec):
    return 0.5 - 0.5 * z if prec == C64 else z


def _ansatz(n, L, angles, ladder, hf=0, insert=None):
    """[B, 2^n] states of angle sets [B, L, n, 2]: RY, RZ on every qubit, then the ladder; insert: [B] parameter
    index whose generator (Y after RY, Z after RZ) follows its rotation, or -1."""
    th = torch.as_tensor(angles, dtype=torch.float64, device="cuda")
    a = _zero(n, th.shape[0])
    if hf:
        a[:, 0], a[:, hf] = 0.0, 1.0
    for l in range(L):
        for q in range(n):
            for k in (0, 1):
                x = th[:, l, q, k].view(-1, 1, 1) / 2
                c, s = torch.cos(x), torch.sin(x)
                u = [[c, -s], [s, c]] if k == 0 else [[torch.complex(c, -s), 0.0], [0.0, torch.complex(c, s)]]
                _apply_1q(a, q, u)
                if insert is not None:
                    for i in np.nonzero(insert == (l * n + q) * 2 + k)[0]:
                        _apply_1q(a[int(i):int(i) + 1], q, _mat(int(G.Y) if k == 0 else int(G.Z)))
        for q in range(n - 1):
            _apply_2q(a, q, q + 1, ladder)
    return a


def _hea_energies(n, L, angles, h):
    out = []
    most = max(1, (1 << 27) >> n)
    for i in range(0, len(angles), most):
        a = _ansatz(n, L, angles[i:i + most], int(G.CZ))
        p = a.real ** 2 + a.imag ** 2
        e = torch.zeros(len(a), dtype=torch.float64, device="cuda")
        idx = torch.arange(1 << n, device="cuda")
        for q in range(n - 1):
            e -= (p * (1.0 - 2.0 * (((idx >> q) ^ (idx >> (q + 1))) & 1))).sum(1)
        hh = torch.as_tensor(h[i:i + most], dtype=torch.float64, device="cuda")
        for q in range(n):
            v = a.view(len(a), -1, 2, 1 << q)
            e -= hh * 2.0 * (v[:, :, 0].conj() * v[:, :, 1]).real.sum((1, 2))
        out.append(e.cpu().numpy())
    return np.concatenate(out)


def _pauli(a, s):
    """<s> of every state of a [B, 2^n]."""
    n = len(s)
    x = sum(1 << q for q in range(n) if s[q] in "XY")
    z = sum(1 << q for q in range(n) if s[q] in "YZ")
    idx = torch.arange(1 << n, device="cuda")
    sign = torch.zeros_like(idx)
    for q in range(n):
        if (z >> q) & 1:
            sign ^= (idx >> q) & 1
    v = (a[:, idx ^ x].conj() * a * (1.0 - 2.0 * sign)).sum(1) * 1j ** s.count("Y")
    return v.real


def _vqe_energies(inst, angles, insert=None):
    a = _ansatz(inst["n"], inst["layers"], angles, int(G.CNOT), inst["hf"], insert)
    e = torch.full((len(a),), inst["constant"], dtype=torch.float64, device="cuda")
    for c, s in inst["terms"]:
        e += c * _pauli(a, s)
    return e.cpu().numpy()


def _shifted(ang):
    """The base point and theta +- pi/2 of every angle, as [1 + 2 P, L, n, 2]."""
    out = np.repeat(ang[None], 1 + 2 * ang.size, 0).reshape(1 + 2 * ang.size, -1)
    for k in range(ang.size):
        out[1 + 2 * k, k] += math.pi / 2
        out[2 + 2 * k, k] -= math.pi / 2
    return out.reshape((-1,) + ang.shape)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("job", "state"):
        n, g = case["n"], _circuit(case, seed)
        if kind == "job" and case["api"] == "scheduler" or len(g) * 2.0 ** n > _EXACT_MOST:
            return None
        a = _simulate(g, n)
        if kind == "job":
            p = a.real ** 2 + a.imag ** 2
            if case["api"] == "qgtl":
                return [None, p.cpu().numpy() if case["amps"] else None]
            return [None, a.cpu().numpy() if case["amps"] else None, _exact_z(_z_of(p, n), case["prec"])]
        p = a.real ** 2
        p += a.imag ** 2
        return [a, _exact_z(_z_of(p, n), case["prec"]), p.sum().item()]
    if kind == "hea":
        inst = _hea_instances(case, seed)
        if sum(2.0 ** n * L * (2 * n + 4) for n, L, _, _ in inst) > _EXACT_MOST:
            return None
        out = np.zeros(len(inst))
        for shape in sorted({(n, L) for n, L, _, _ in inst}):
            at = [i for i, (n, L, _, _) in enumerate(inst) if (n, L) == shape]
            out[at] = _hea_energies(*shape, np.stack([inst[i][2] for i in at]), np.asarray([inst[i][3] for i in at]))
        return out
    if kind == "heagrad":
        es, gs = [], []
        for n, L, ang, h in _hea_instances(case, seed):
            e = _hea_energies(n, L, _shifted(ang), np.full(1 + 2 * ang.size, h))
            es.append(e[0])
            gs.append((0.5 * (e[1::2] - e[2::2])).reshape(L, n, 2))
        return [np.asarray(es), gs]
    if kind == "vqe":
        return np.asarray([_vqe_energies(v, v["angles"][None])[0] for v in _vqe_instances(case, seed)])
    if kind == "qng":
        es, gs, ds = [], [], []
        for v in _vqe_instances(case, seed):
            e = _vqe_energies(v, _shifted(v["angles"]))
            g = 0.5 * (e[1::2] - e[2::2])
            P = g.size
            a = _ansatz(v["n"], v["layers"], np.repeat(v["angles"][None], P + 1, 0), int(G.CNOT), v["hf"],
                        np.arange(-1, P))
            gram = (a.conj() @ a.T).cpu().numpy()
            Q = 0.25 * (gram[1:, 1:] - np.outer(gram[1:, 0], gram[0, 1:]))
            es.append(e[0])
            gs.append(g)
            ds.append(np.linalg.solve(Q.real + 1e-3 * np.eye(P), g))
        return [np.asarray(es), np.concatenate(gs), np.concatenate(ds), None]
    if kind == "readout":
        n, ops = case["n"], _readout_ops(case, seed)
        a = _simulate(workloads.random_layer_circuit(n, 6, seed, h_layer=True), n)
        p = a.real ** 2 + a.imag ** 2
        pair = lambda x, y: "".join("Z" if q in (x, y) else "I" for q in range(n))  # noqa: E731
        vals = [_pauli(a[None], s).item() for s in [pair(x, y) for x, y in ops["pairs"]] + ops["strings"]]
        return [_z_of(p, n), p.sum().item(), np.asarray(vals), None, None, None, None]
    zs = [[], []]
    for q in _requests(case, seed):
        a = _simulate(q["gates"], q["n"])
        zs[q["precision"]].append(_z_of(a.real ** 2 + a.imag ** 2, q["n"]))
    cat = lambda xs: np.concatenate(xs) if xs else np.zeros(0)  # noqa: E731
    return [cat(zs[0]), None, _exact_z(cat(zs[1]), C64)]
