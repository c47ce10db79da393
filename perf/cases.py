"""Workloads of the state-vector engine for timing and comparison, each a call a program makes through
the ctypes binding (riken-braket_amd/py/brk.py).

Paths and what they stand for:
  run       brk.Circuit.run: gate by gate, the plain form.  Small states are simulation of few-qubit
            circuits (launch-bound), 20 qubits is the reference's CPU case, the largest the headline
            circuit on a state far above the caches.
  blocked   brk.Circuit.run_blocked: how the front end runs every stretch of gates -- planned for this
            call, run, waited for.
  blocks    brk.BlockPlan.run: gate blocks of a circuit that is run again and again.
  fused     brk.FusedPlan.apply: the precision form, blocks of 4..6 qubits on a complex64 state.
  batch     brk.Batch.run: energies of many small ansatz circuits (a population or a parameter scan),
            or of a few (one optimiser step).
  gradient  brk.adjoint_ising_gradient of the layered ansatz from |0...0>, one optimiser step.
  readout   the Ising energy and the spin components of every qubit (DO MEASUREMENT).
  events    sampled basis states from given draws (GENERATE EVENTS).
"""
from __future__ import annotations

import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "riken-braket_amd", "py"))

import brk  # noqa: E402
import circuits as W  # noqa: E402

DTYPES = {"c128": (brk.C128, torch.complex128, 16), "c64": (brk.C64, torch.complex64, 8)}


def listed():
    return [
        # a few-qubit circuit on a state of 64 KiB: launches and their latency
        {"name": "run_12q", "path": "run", "qubits": 12, "dtype": "c128", "circuit": "layered", "layers": 10},
        # the reference's CPU case: H wall, then RZ and CNOT bricks, 315 gates on 16 MiB
        {"name": "run_20q", "path": "run", "qubits": 20, "dtype": "c128", "circuit": "layered", "layers": 10},
        # the headline circuit's mix of gates and local swaps on 8 GiB, streamed from HBM gate by gate
        {"name": "run_29q", "path": "run", "qubits": 29, "dtype": "c128", "circuit": "random", "gates": 100, "swaps": 4},
        # a program of the front end at an ordinary size, planned and run in one call
        {"name": "blocked_18q", "path": "blocked", "qubits": 18, "dtype": "c128", "circuit": "random", "gates": 120,
         "swaps": 0},
        # the headline circuit in gate blocks
        {"name": "blocks_29q", "path": "blocks", "qubits": 29, "dtype": "c128", "circuit": "random", "gates": 200,
         "swaps": 8},
        # the headline circuit in the precision form
        {"name": "fused_w4_30q", "path": "fused", "qubits": 30, "circuit": "random", "gates": 150, "swaps": 6,
         "width": 4},
        # a population of circuits of every size of the batching workload
        {"name": "batch_1024", "path": "batch", "circuits": 1024, "min_qubits": 10, "max_qubits": 20, "layers": 8},
        # one optimiser step's handful of circuits
        {"name": "batch_24", "path": "batch", "circuits": 24, "min_qubits": 13, "max_qubits": 19, "layers": 8},
        # the differentiation workload: 576 parameters on 24 qubits
        {"name": "gradient_24q", "path": "gradient", "qubits": 24, "dtype": "c128", "layers": 12},
        # a small ansatz, where the host's planning and the launches count
        {"name": "gradient_15q", "path": "gradient", "qubits": 15, "dtype": "c128", "layers": 6},
        # energy and every qubit's spin of a 4 GiB state
        {"name": "readout_28q", "path": "readout", "qubits": 28, "dtype": "c128"},
        # a sample of 100 000 events from a 2 GiB state
        {"name": "events_27q", "path": "events", "qubits": 27, "dtype": "c128", "events": 100000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["run", "blocked", "blocks", "fused", "batch", "gradient", "readout", "events"])
    dtype = rng.choice(["c128", "c128", "c64"])
    if path in ("run", "blocked", "blocks"):
        # (states are sized by qubits, the logarithm of their length)
        n = rng.randint(8, {"run": 28, "blocked": 24, "blocks": 28}[path])
        case = {"path": path, "qubits": n, "dtype": dtype, "circuit": rng.choice(["random", "random", "layered"])}
        if case["circuit"] == "random":
            case |= {"gates": rng.randint(30, 100), "swaps": rng.randint(0, 4)}
        else:
            case["layers"] = rng.randint(1, 3 if n > 24 else 8)
        return case
    if path == "fused":
        return {"path": path, "qubits": rng.randint(12, 29), "circuit": "random", "gates": rng.randint(40, 150),
                "swaps": rng.randint(0, 6), "width": rng.choice([4, 4, 5, 6])}
    if path == "batch":
        lo = rng.randint(3, 14)
        hi = rng.randint(lo, 19)
        return {"path": path, "circuits": _log_int(rng, 1, 600), "min_qubits": lo, "max_qubits": hi,
                "layers": rng.randint(1, 8)}
    if path == "gradient":
        return {"path": path, "qubits": rng.randint(6, 23), "dtype": dtype, "layers": rng.randint(1, 10)}
    if path == "readout":
        return {"path": path, "qubits": rng.randint(6, 27), "dtype": dtype}
    return {"path": path, "qubits": rng.randint(6, 27), "dtype": dtype, "events": _log_int(rng, 1, 100000)}


def _ops(case, seed):
    n = case["qubits"]
    if case["circuit"] == "layered":
        return W.layered_rz_cnot(n, case["layers"], seed)
    return W.random_circuit(n, case["gates"], case["swaps"], seed)


def _random_state(n, dtype, seed):
    """A normalised state with independent Gaussian amplitudes (the amplitudes of a deep random circuit)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    real = torch.float64 if dtype == "c128" else torch.float32
    s = torch.randn(1 << n, 2, dtype=real, device="cuda", generator=g)
    s *= 2.0 ** (-0.5 * (n + 1))  # |amplitude|^2 averages 2^-n
    if n <= 20:
        s /= s.square().sum().sqrt()
    return torch.view_as_complex(s)


def _polarised_state(n, dtype, seed):
    """A product state of random directions with a Gaussian part over it, as an ansatz leaves it: energies and
    spins of order one, all amplitudes different."""
    g = torch.Generator(device="cpu").manual_seed(seed + 2000)
    psi = torch.ones(1, dtype=torch.complex128, device="cuda")
    for _ in range(n):
        a = torch.view_as_complex(torch.randn(2, 2, dtype=torch.float64, generator=g)).tolist()
        r = math.sqrt(abs(a[0]) ** 2 + abs(a[1]) ** 2)
        psi = torch.cat([psi * (0.9 * a[0] / r + 0.1), psi * (0.9 * a[1] / r)])
    psi *= 0.9 / math.sqrt(float(torch.view_as_real(psi).square().sum()))
    psi = psi.to(DTYPES[dtype][1])
    psi += 0.4 * _random_state(n, dtype, seed)
    return psi


def _chain(n, seed):
    rng = np.random.default_rng(seed + 1000)
    return rng.uniform(-1.0, 1.0, max(0, n - 1)), rng.uniform(-1.0, 1.0, n)


def _batch_items(case, seed):
    return W.batch_ansatz(case["circuits"], case["min_qubits"], case["max_qubits"], case["layers"], seed)


def prepare(case, seed):
    path = case["path"]
    st = {"path": path}
    if path == "batch":
        st["batch"] = brk.Batch(_batch_items(case, seed))
        return st
    n = case["qubits"]
    st["n"], st["size"] = n, 1 << n
    dtype = case.get("dtype", "c64")
    st["dtype"] = DTYPES[dtype][0]
    if path == "gradient":
        ops, _ = W.adjoint_ansatz(n, case["layers"], seed)
        st["circuit"] = brk.Circuit(n, ops)
        st["J"], st["h"] = _chain(n, seed)
        st["psi"] = torch.empty(1 << n, dtype=DTYPES[dtype][1], device="cuda")
        st["work"] = torch.empty_like(st["psi"])
        return st
    st["psi"] = (_polarised_state if path == "readout" else _random_state)(n, dtype, seed)
    st["ptr"] = st["psi"].data_ptr()
    if path == "readout":
        st["J"], st["h"] = _chain(n, seed)
    elif path == "events":
        st["draws"] = np.random.default_rng(seed).random(case["events"])
    else:
        st["circuit"] = brk.Circuit(n, _ops(case, seed))
        if path == "blocks":
            st["plan"] = brk.BlockPlan(st["circuit"], st["dtype"])
        elif path == "fused":
            st["plan"] = brk.FusedPlan(st["circuit"], case["width"])
    return st


def run(st):
    path = st["path"]
    if path == "run":
        st["circuit"].run(st["ptr"], st["dtype"])
        return st["psi"]
    if path == "blocked":
        st["circuit"].run_blocked(st["ptr"], st["dtype"])
        return st["psi"]
    if path == "blocks":
        st["plan"].run(st["ptr"])
        return st["psi"]
    if path == "fused":
        st["plan"].apply(st["ptr"])
        return st["psi"]
    if path == "batch":
        # energies of complex64 states: kept in their precision, as an optimiser keeps its losses
        return st["batch"].run().astype(np.float32)
    if path == "gradient":
        brk.set_basis_state(st["psi"].data_ptr(), st["size"], st["dtype"], 0)
        e, g = brk.adjoint_ising_gradient(st["circuit"], st["psi"].data_ptr(), st["work"].data_ptr(), st["dtype"],
                                          st["J"], st["h"])
        if st["dtype"] == brk.C64:  # (as for the batch: values of complex64 states)
            return np.float32(e), g.astype(np.float32)
        return e, g
    if path == "readout":
        e = brk.expectation_ising(st["ptr"], st["size"], st["dtype"], st["J"], st["h"])
        spins = [brk.spin_expectation_value(st["ptr"], st["size"], st["dtype"], q) for q in range(st["n"])]
        return e, np.array(spins)
    draws = st["draws"]
    events = np.empty(draws.size, dtype=np.uint64)
    brk.call("brk_generate_events", st["ptr"], st["size"], st["dtype"], draws.ctypes.data_as(C.POINTER(C.c_double)),
             int(draws.size), events.ctypes.data_as(C.POINTER(C.c_uint64)), 0)
    return events.view(np.int64)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def _gate_flops(op, n):
    name, t, c, _ = op
    amps = 2.0 ** (n - len(c))
    if name in ("H", "RY"):
        return 6 * amps
    if name == "U3":
        return 14 * amps
    if name == "RZ":
        return 6 * amps
    return 0.0


def work(case):
    path = case["path"]
    if path == "batch":
        flops = 0.0
        for i in range(case["circuits"]):
            n = case["min_qubits"] + i % (case["max_qubits"] - case["min_qubits"] + 1)
            flops += case["layers"] * n * 12 * 2.0 ** n
        return {"bytes": 8.0 * case["circuits"], "flops": flops}
    n = case["qubits"]
    amp = DTYPES[case.get("dtype", "c64")][2]
    state = amp * 2.0 ** n
    if path == "gradient":
        # three sweeps of the circuit's gates (psi forward, psi and lambda back) and two sums per parameter
        return {"bytes": 2 * state, "flops": case["layers"] * n * 2.0 ** n * (3 * 12 + 8)}
    if path == "readout":
        return {"bytes": state, "flops": n * 2.0 ** n * 6}
    if path == "events":
        return {"bytes": state, "flops": 4 * 2.0 ** n}
    return {"bytes": 2 * state, "flops": sum(_gate_flops(o, n) for o in _ops(case, 1))}


# ---------------------------------------------------------------------------
# The same results in 64 bits by plain torch
# ---------------------------------------------------------------------------

def _one_qubit(psi, q, m):
    v = psi.view(-1, 2, 1 << q)
    a0, a1 = v[:, 0], v[:, 1]
    n0 = a0 * m[0] + a1 * m[1]
    n1 = a0 * m[2] + a1 * m[3]
    v[:, 0], v[:, 1] = n0, n1


def _pair_view(psi, a, b):
    """psi with qubits a and b as axes 1 and 3 (the higher one first) and whether a is axis 1."""
    hi, lo = max(a, b), min(a, b)
    return psi.view(-1, 2, 1 << (hi - lo - 1), 2, 1 << lo), a == hi


def _swap_parts(x, y):
    t = x.clone()
    x.copy_(y)
    y.copy_(t)


def _matrix(name, p):
    e = lambda x: complex(math.cos(x), math.sin(x))  # noqa: E731
    if name == "H":
        r = math.sqrt(0.5)
        return (r, r, r, -r)
    if name == "RY":
        c, s = math.cos(p[0] / 2), math.sin(p[0] / 2)
        return (c, -s, s, c)
    c, s = math.cos(p[0] / 2), math.sin(p[0] / 2)
    return (c, -s * e(p[2]), s * e(p[1]), c * e(p[1] + p[2]))  # U3


def _apply(psi, op, place):
    name, t, c, p = op
    t, c = [place[q] for q in t], [place[q] for q in c]
    if name == "RZ":
        v = psi.view(-1, 2, 1 << t[0])
        v[:, 0] *= complex(math.cos(p[0] / 2), -math.sin(p[0] / 2))
        v[:, 1] *= complex(math.cos(p[0] / 2), math.sin(p[0] / 2))
    elif name == "X" and not c:
        v = psi.view(-1, 2, 1 << t[0])
        _swap_parts(v[:, 0], v[:, 1])
    elif name == "X":
        v, first = _pair_view(psi, c[0], t[0])
        if first:
            _swap_parts(v[:, 1, :, 0], v[:, 1, :, 1])
        else:
            _swap_parts(v[:, 0, :, 1], v[:, 1, :, 1])
    elif name == "Z":
        a, b = t + c
        v, _ = _pair_view(psi, a, b)
        v[:, 1, :, 1] *= -1
    else:
        _one_qubit(psi, t[0], _matrix(name, p))


def _simulate(psi, n, ops):
    place = list(range(n))  # logical qubit -> bit of the state
    for op in ops:
        if op[0] == "LOCAL_SWAP":
            a, b = op[1]
            v, _ = _pair_view(psi, a, b)
            _swap_parts(v[:, 0, :, 1], v[:, 1, :, 0])
            i, j = place.index(a), place.index(b)
            place[i], place[j] = place[j], place[i]
        else:
            _apply(psi, op, place)


def _zero(n):
    psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
    psi[0] = 1.0
    return psi


def _zz_diagonal(n, J):
    """sum_i J_i Z_i Z_(i+1) of every basis state, and its parts' doubling from the low qubits up."""
    e = torch.zeros(2, dtype=torch.float64, device="cuda")
    for q in range(1, n):
        lo = e.clone()
        half = 1 << (q - 1)
        s = torch.ones(1 << q, dtype=torch.float64, device="cuda")
        s[half:] = -1.0
        e = torch.cat([lo + J[q - 1] * s, lo - J[q - 1] * s])
    return e


def _energy(psi, n, J, h):
    p = torch.view_as_real(psi).square().sum(1)
    e = float((p * _zz_diagonal(n, J)).sum()) if n > 1 else 0.0
    for q in range(n):
        v = psi.view(-1, 2, 1 << q)
        e += 2.0 * h[q] * float((v[:, 0].conj() * v[:, 1]).real.sum())
    return e


def _cz_signs(n):
    """The diagonal of the CZ ladder."""
    s = torch.ones(2, dtype=torch.float64, device="cuda")
    for q in range(1, n):
        up = s.clone()
        up[1 << (q - 1):] *= -1.0
        s = torch.cat([s, up])
    return s


def _layers(ops, n):
    """The ansatz's angles as [(RY angle, RZ angle) per qubit] per layer."""
    angles = [o[3][0] for o in ops if o[0] in ("RY", "RZ")]
    return np.array(angles).reshape(-1, n, 2)


def _ansatz_matrix(ry, rz):
    c, s = math.cos(ry / 2), math.sin(ry / 2)
    e0, e1 = complex(math.cos(rz / 2), -math.sin(rz / 2)), complex(math.cos(rz / 2), math.sin(rz / 2))
    return (c * e0, -s * e0, s * e1, c * e1)


def _ansatz_state(n, layers, signs):
    psi = _zero(n)
    for layer in layers:
        for q in range(n):
            _one_qubit(psi, q, _ansatz_matrix(*layer[q]))
        psi *= signs
    return psi


def _exact_gradient(n, ops, J, h):
    layers, signs = _layers(ops, n), _cz_signs(n)
    psi = _ansatz_state(n, layers, signs)
    lam = psi * _zz_diagonal(n, J) if n > 1 else torch.zeros_like(psi)
    for q in range(n):
        v, w = psi.view(-1, 2, 1 << q), lam.view(-1, 2, 1 << q)
        w[:, 0] += h[q] * v[:, 1]
        w[:, 1] += h[q] * v[:, 0]
    energy = torch.view_as_real(psi).mul(torch.view_as_real(lam)).sum()
    grads = torch.zeros(layers.shape, dtype=torch.float64, device="cuda")
    for k in range(len(layers) - 1, -1, -1):
        psi *= signs
        lam *= signs
        for q in range(n - 1, -1, -1):
            v, w = psi.view(-1, 2, 1 << q), lam.view(-1, 2, 1 << q)
            # 2 Re <lam| -(i/2) Z |psi> = Im <lam|Z|psi>; the RZ is undone with the RY below
            grads[k, q, 1] = (w[:, 0].conj() * v[:, 0]).imag.sum() - (w[:, 1].conj() * v[:, 1]).imag.sum()
            ry, rz = layers[k, q]
            back = _matrix_dagger(_ansatz_matrix(0.0, rz))
            _one_qubit(psi, q, back)
            _one_qubit(lam, q, back)
            # 2 Re <lam| -(i/2) Y |psi>, -iY = [[0, -1], [1, 0]]
            v, w = psi.view(-1, 2, 1 << q), lam.view(-1, 2, 1 << q)
            grads[k, q, 0] = (w[:, 1].conj() * v[:, 0]).real.sum() - (w[:, 0].conj() * v[:, 1]).real.sum()
            back = _matrix_dagger(_ansatz_matrix(ry, 0.0))
            _one_qubit(psi, q, back)
            _one_qubit(lam, q, back)
    return float(energy), grads.reshape(-1).cpu().numpy()


def _matrix_dagger(m):
    return tuple(complex(x).conjugate() for x in (m[0], m[2], m[1], m[3]))


def exact(case, seed):
    path = case["path"]
    if path == "batch":
        signs = {n: _cz_signs(n) for n in range(1, case["max_qubits"] + 1)}
        return np.array([_energy(_ansatz_state(n, _layers(ops, n), signs[n]), n, J, h)
                         for n, ops, J, h in _batch_items(case, seed)])
    n = case["qubits"]
    if path == "gradient":
        ops, _ = W.adjoint_ansatz(n, case["layers"], seed)
        return _exact_gradient(n, ops, *_chain(n, seed))
    if path == "events":
        return None  # whole numbers: the same draws give the same events
    dtype = case.get("dtype", "c64")
    if path == "readout":
        psi = _polarised_state(n, dtype, seed).to(torch.complex128)
        J, h = _chain(n, seed)
        spins = []
        for q in range(n):
            v = psi.view(-1, 2, 1 << q)
            x = (v[:, 0].conj() * v[:, 1]).sum()
            z = torch.view_as_real(v[:, 0]).square().sum() - torch.view_as_real(v[:, 1]).square().sum()
            spins.append((float(x.real), float(x.imag), 0.5 * float(z)))
        return _energy(psi, n, J, h), np.array(spins)
    psi = _random_state(n, dtype, seed).to(torch.complex128)
    _simulate(psi, n, _ops(case, seed))
    return psi
