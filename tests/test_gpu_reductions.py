"""GPU parity of the FP64 reductions against the CPU oracle (through the C ABI)."""
import sys

import numpy as np
import pytest

import brk
import dense as D
from devstate import DeviceState

pytestmark = pytest.mark.gpu

TOL = 1e-12


def note(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def test_reference_observable_fixtures(oracle):
    note("gpu reductions: reference fixtures")
    p1, p2 = D.observable_state1(4), D.observable_state2(4)
    a, b = DeviceState.from_host(p1), DeviceState.from_host(p2)
    assert abs(brk.inner_product(a.ptr, brk.C128, b.ptr, brk.C128, 16) - oracle.inner_product(p1, p2)) < TOL
    assert abs(brk.norm2(a.ptr, 16, brk.C128) - oracle.norm2(p1)) < TOL
    ip = oracle.inner_product(p1, p2)
    out = (brk.C.c_double * 1)()
    brk.call("brk_fidelity", a.ptr, brk.C128, b.ptr, brk.C128, 16, out, None)
    assert abs(out[0] - abs(ip) ** 2) < 1e-10
    a.free()
    b.free()


@pytest.mark.parametrize("n", [3, 11, 20])
def test_spin_and_pauli(oracle, n):
    rng = np.random.default_rng(n)
    s = D.random_state(n, rng)
    st = DeviceState.from_host(s)
    for q in sorted({0, 1, n // 2, n - 1}):
        note(f"gpu spin n={n} q={q}")
        g = brk.spin_expectation_value(st.ptr, st.size, brk.C128, q)
        o = oracle.spin_expectation_value(s, q)
        assert np.max(np.abs(np.array(g) - np.array(o))) < TOL
    for pauli, qs in (("X", [0]), ("ZZ", [0, n - 1]), ("XYZ", [n - 1, 0, 1]), ("YY", [1, 2])):
        if max(qs) >= n:
            continue
        note(f"gpu pauli n={n} {pauli}{qs}")
        g = brk.expectation_pauli_string(st.ptr, st.size, brk.C128, pauli, qs)
        o = oracle.expectation_pauli_string(s, pauli, qs)
        assert abs(g - o) < TOL
    st.free()


@pytest.mark.parametrize("n,dtype", [(10, brk.C128), (16, brk.C128), (12, brk.C64)])
def test_ising(oracle, n, dtype):
    note(f"gpu ising n={n} dtype={dtype}")
    rng = np.random.default_rng(50 + n)
    s = D.random_state(n, rng)
    J = rng.uniform(-1, 1, n - 1)
    h = rng.uniform(-1, 1, n)
    tol = TOL if dtype == brk.C128 else 1e-6
    host = s if dtype == brk.C128 else s.astype(np.complex64)
    ref = host.astype(np.complex128)
    st = DeviceState.from_host(host, dtype)
    e = brk.expectation_ising(st.ptr, st.size, dtype, J, h)
    assert abs(e - oracle.expectation_ising(ref, J, h)) < tol
    out = DeviceState(n, dtype)
    brk.apply_ising(out.ptr, st.ptr, st.size, dtype, J, h)
    got = out.download().astype(np.complex128)
    assert np.max(np.abs(got - oracle.apply_ising(ref, J, h))) < (tol * 10)
    st.free()
    out.free()


@pytest.mark.parametrize("dtype", [brk.C128, brk.C64])
@pytest.mark.parametrize("n", [1, 2, 5, 9, 11, 12, 13, 14, 21, 22])
def test_ising_chunk_edges(oracle, n, dtype):
    """Sizes around a chunk (2^12 or 2^13 amplitudes) and around the 9 further qubits of each pass, with terms
    left out (h = 0); both sides sum 2^n terms of a unit state in FP64, each rounding at most eps of a partial
    sum bounded by the sum of the coefficients."""
    note(f"gpu ising chunk edges n={n} dtype={dtype}")
    rng = np.random.default_rng(70 + n)
    host = D.random_state(n, rng).astype(np.complex128 if dtype == brk.C128 else np.complex64)
    J, h = rng.uniform(-1, 1, max(0, n - 1)), rng.uniform(-1, 1, n)
    h[1::3] = 0.0
    st = DeviceState.from_host(host, dtype)
    e = brk.expectation_ising(st.ptr, st.size, dtype, J, h)
    ref = oracle.expectation_ising(host.astype(np.complex128), J, h)
    assert abs(e - ref) < 2 * (2.0 ** n + 16) * np.finfo(float).eps * (np.sum(np.abs(J)) + np.sum(np.abs(h)) + 1)
    for q in {0, n // 2, n - 1}:  # one X term alone
        one = np.zeros(n)
        one[q] = 1.0
        e = brk.expectation_ising(st.ptr, st.size, dtype, np.zeros(max(0, n - 1)), one)
        assert abs(e - oracle.expectation_ising(host.astype(np.complex128), np.zeros(max(0, n - 1)), one)) < (
            2 * (2.0 ** n + 16) * np.finfo(float).eps)
    st.free()


def test_mixed_precision_inner_product(oracle):
    note("gpu mixed inner product")
    rng = np.random.default_rng(9)
    s = D.random_state(15, rng)
    a = DeviceState.from_host(s)
    b = DeviceState.from_host(s.astype(np.complex64), brk.C64)
    ip = brk.inner_product(b.ptr, brk.C64, a.ptr, brk.C128, a.size)
    ref = oracle.inner_product(s.astype(np.complex64).astype(np.complex128), s)
    assert abs(ip - ref) < 1e-12
    a.free()
    b.free()


def test_reductions_are_deterministic():
    note("gpu reduction determinism")
    st = DeviceState(22)
    brk.fill_hash(st.ptr, st.size, brk.C128, 123, 1e-3)
    vals = {brk.norm2(st.ptr, st.size, brk.C128) for _ in range(3)}
    assert len(vals) == 1
    st.free()


def test_fill_hash_matches_numpy_twin():
    note("gpu fill_hash twin")
    st = DeviceState(12)
    brk.fill_hash(st.ptr, st.size, brk.C128, 99, 0.5)
    got = st.download()
    st.free()
    assert np.array_equal(got, D.hash_state_values(99, np.arange(4096), 0.5))


@pytest.mark.parametrize("n,dtype", [(1, brk.C128), (9, brk.C64), (10, brk.C128), (11, brk.C128), (12, brk.C64),
                                     (20, brk.C128), (21, brk.C128)])
def test_reduction_tiles(oracle, n, dtype):
    """Tiles of 1024 items on 1024 blocks: a part of one tile, one tile, some of the blocks, a tile each
    (2^20 items) and two; against FP64 numpy sums.  At most 2^21 products of at most 1 / 2^n each."""
    note(f"gpu reduction tiles n={n} dtype={dtype}")
    rng = np.random.default_rng(n)
    s, r = D.random_state(n, rng), D.random_state(n, rng)
    if dtype == brk.C64:
        s, r = (x.astype(np.complex64).astype(np.complex128) for x in (s, r))
    a, b = DeviceState.from_host(s, dtype), DeviceState.from_host(r, dtype)
    assert abs(brk.norm2(a.ptr, a.size, dtype) - np.vdot(s, s).real) < 1e-12
    assert abs(brk.inner_product(a.ptr, dtype, b.ptr, dtype, a.size) - oracle.inner_product(s, r)) < 1e-12
    for q in sorted({0, n // 2, n - 1}):
        p = s.reshape(-1, 2, 1 << q)
        up, down = p[:, 0], p[:, 1]
        zero, one = np.sum(np.abs(up) ** 2), np.sum(np.abs(down) ** 2)
        x = np.sum(np.conj(up) * down)
        spin = brk.spin_expectation_value(a.ptr, a.size, dtype, q)
        assert np.max(np.abs(np.array(spin) - [x.real, x.imag, 0.5 * (zero - one)])) < 1e-12
        assert np.max(np.abs(np.array(brk.zero_one_probabilities(a.ptr, a.size, dtype, q)) - [zero, one])) < 1e-12
        assert abs(brk.expectation_pauli_string(a.ptr, a.size, dtype, "X", [q]) - 2 * x.real) < 1e-12
    a.free()
    b.free()


@pytest.mark.parametrize("n,dtype", [(3, brk.C128), (9, brk.C64), (14, brk.C128), (16, brk.C64)])
def test_ising_fields_that_are_not_finite(n, dtype):
    """A field multiplies its qubit's whole <X>: an infinite one gives the infinity of that sign beside finite
    terms (also where the state is smaller than a chunk, and where parts of the sum differ in sign), two of
    opposite results give no number, and so does one that is no number."""
    note(f"gpu ising with infinite fields n={n} dtype={dtype}")
    rng = np.random.default_rng(90 + n)
    host = D.random_state(n, rng).astype(np.complex128 if dtype == brk.C128 else np.complex64)
    st = DeviceState.from_host(host, dtype)
    J, h = rng.uniform(-1, 1, n - 1), rng.uniform(-1, 1, n)
    signs = []
    for q in (0, n // 2, n - 1):
        x = brk.spin_expectation_value(st.ptr, st.size, dtype, q)[0]
        assert x != 0.0
        signs.append((q, np.sign(x)))
        for value in (np.inf, -np.inf, 1.7e308):  # (the last: finite, its double is not)
            g = h.copy()
            g[q] = value
            assert brk.expectation_ising(st.ptr, st.size, dtype, J, g) == np.copysign(np.inf, value) * np.sign(x)
        g = h.copy()
        g[q] = np.nan
        assert np.isnan(brk.expectation_ising(st.ptr, st.size, dtype, J, g))
    g = h.copy()
    (a, sa), (b, sb) = signs[:2]
    g[a], g[b] = np.inf * sa, -np.inf * sb
    assert np.isnan(brk.expectation_ising(st.ptr, st.size, dtype, J, g))
    st.free()
