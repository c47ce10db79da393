"""GPU parity of gate blocks (brk_circuit_run_blocked / brk_block_plan_run).

Bar: bit-identical amplitudes to the per-gate path (brk_circuit_run) -- a
block applies each gate with the same IEEE operation sequence -- and, for
complex<double>, within 1e-12 of the CPU oracle.  Circuits mix every op kind
with controls, multi-target strings, local swaps and a non-identity starting
permutation."""
import ctypes as C
import sys

import numpy as np
import pytest

import brk
import dense as D
import hip
from devstate import DeviceState
from oracle_circuits import run_ops
from randops import random_ops

pytestmark = pytest.mark.gpu


def note(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def run_both(n, ops, dtype, perm0=None, seed=0):
    rng = np.random.default_rng(seed)
    s = D.random_state(n, rng)
    if dtype == brk.C64:
        s = s.astype(np.complex64).astype(np.complex128)
    c = brk.Circuit(n, ops)
    a, b = DeviceState.from_host(s, dtype), DeviceState.from_host(s, dtype)
    pa = c.run(a.ptr, dtype, perm0)
    pb = c.run_blocked(b.ptr, dtype, perm0)
    out_a, out_b = a.download(), b.download()
    a.free()
    b.free()
    return s, out_a, out_b, pa, pb


def same_bits(x, y):
    w = np.uint64 if x.dtype == np.complex128 else np.uint32
    return np.array_equal(x.view(w), y.view(w))


@pytest.fixture(params=["temporal", "nontemporal"])
def access(request):
    """Default access policy, then the non-temporal instantiations large states take."""
    if request.param == "temporal":
        yield request.param
        return
    old = brk.get_tune("nt_min_bytes")
    brk.tune("nt_min_bytes", 0)
    try:
        yield request.param
    finally:
        brk.tune("nt_min_bytes", old)


@pytest.mark.parametrize("n,dtype,seed", [(3, brk.C128, 1), (9, brk.C128, 2), (12, brk.C128, 3), (13, brk.C128, 4),
                                          (16, brk.C128, 5), (20, brk.C128, 6), (12, brk.C64, 7), (14, brk.C64, 8),
                                          (20, brk.C64, 9)])
def test_blocked_equals_plain_bitwise(oracle, n, dtype, seed, access):
    note(f"gpu blocks n={n} dtype={dtype} seed={seed} ({access})")
    ops = random_ops(n, 160, seed, local_swaps=3 if n >= 4 else 0)
    perm0 = list(np.random.default_rng(seed).permutation(n))
    s, plain, blocked, pa, pb = run_both(n, ops, dtype, perm0, seed)
    assert pa == pb
    assert same_bits(plain, blocked)
    if dtype == brk.C128:
        ref = s.copy()
        run_ops(oracle, ref, ops, perm0)
        assert np.max(np.abs(blocked - ref)) < 1e-12


@pytest.mark.parametrize("n,dtype,seed", [(2, brk.C128, 31), (8, brk.C64, 32), (9, brk.C128, 33), (10, brk.C64, 34),
                                          (11, brk.C128, 35), (12, brk.C128, 36), (13, brk.C64, 37),
                                          (13, brk.C128, 38), (16, brk.C64, 39), (19, brk.C128, 40),
                                          (21, brk.C64, 41)])
def test_run_equals_gate_by_gate_bitwise(n, dtype, seed, access):
    """brk_circuit_run and a block plan (launches of many gates, controls and diagonal gates on any qubit,
    moves deferred) against brk_circuit_run_timed, which launches the plain kernel of every op: the same
    bits, zeros' signs included (a state with zeros), for every op kind."""
    note(f"gpu run vs gate by gate n={n} dtype={dtype} seed={seed} ({access})")
    rng = np.random.default_rng(seed)
    ops = random_ops(n, 220, seed, local_swaps=6 if n >= 4 else 0)
    ops += [("X", (0,), (), ()), ("X", (n - 1,), (0,), ()), ("SWAP", (0, n - 1), (), ())] * (n > 1)
    perm0 = [int(q) for q in rng.permutation(n)]
    s = D.random_state(n, rng)
    s[rng.random(s.size) < 0.3] = 0.0
    c = brk.Circuit(n, ops)
    plan = brk.BlockPlan(c, dtype, perm0)
    states = [DeviceState.from_host(s, dtype) for _ in range(3)]
    final, _ = c.run_timed(states[0].ptr, dtype, perm0)
    assert c.run(states[1].ptr, dtype, perm0) == final
    plan.run(states[2].ptr)
    assert plan.final_permutation == final
    want, *got = [st.download() for st in states]
    for st in states:
        st.free()
    for x in got:
        assert same_bits(want, x)


@pytest.mark.parametrize("n,dtype,moves", [(14, brk.C128, 0.5), (15, brk.C64, 0.8), (18, brk.C128, 0.8),
                                           (20, brk.C64, 0.97), (22, brk.C128, 0.97)])
def test_moves_out_of_order_bitwise(n, dtype, moves):
    """Moves that pass, or are passed by, gates that a launch leaves for later (and long runs of moves that
    no launch takes together): the bits of the op-by-op run, and the same final permutation."""
    note(f"gpu moves out of order n={n} dtype={dtype} moves={moves}")
    rng = np.random.default_rng(n)
    ops = []
    for _ in range(500):
        q = [int(x) for x in rng.permutation(n)[:4]]
        if rng.random() < moves:
            ops.append([("X", (q[0],), (), ()), ("X", (q[0],), (q[1],), ()), ("X", (q[0],), (q[1], q[2]), ()),
                        ("SWAP", (q[0], q[1]), (), ()), ("LOCAL_SWAP", (q[0], q[1]), (), ())][rng.integers(5)])
        else:
            ops.append([("H", (q[0],), (), ()), ("RX", (q[0],), (q[1],), (0.3,)), ("RZ", (q[0],), (), (0.7,)),
                        ("Z", (q[0],), (q[1],), ())][rng.integers(4)])
    s = D.random_state(n, rng)
    s[rng.random(s.size) < 0.3] = 0.0
    c = brk.Circuit(n, ops)
    a, b = DeviceState.from_host(s, dtype), DeviceState.from_host(s, dtype)
    final, _ = c.run_timed(a.ptr, dtype)
    assert c.run(b.ptr, dtype) == final
    want, got = a.download(), b.download()
    a.free()
    b.free()
    assert same_bits(want, got)


def test_dense_low_qubit_blocks(oracle):
    """Many gates on the line qubits and their neighbours: long blocks, every pair mode."""
    n = 18
    note("gpu blocks: low-qubit circuit")
    ops = random_ops(n, 400, 11, qubit_pool=range(10))
    plan = brk.BlockPlan(brk.Circuit(n, ops))
    assert max(k for _, k, _ in plan.steps) == 64
    s, plain, blocked, _, _ = run_both(n, ops, brk.C128, None, 11)
    assert same_bits(plain, blocked)


def test_plan_reuse_and_large_state(oracle):
    """A 26-qubit random circuit (1 GiB), the plan run twice: each run equals the plain path."""
    n = 26
    note(f"gpu blocks: n={n} plan reuse")
    ops = random_ops(n, 60, 12, max_controls=1)
    c = brk.Circuit(n, ops)
    plan = brk.BlockPlan(c)
    st = DeviceState(n)
    ref = DeviceState(n)
    for dev in (st, ref):
        brk.fill_modular(dev.ptr, dev.size, brk.C128, (1e-4, 3e-4), (7, 3, 101, 11, 5, 97))
    plan.run(st.ptr)
    plan.run(st.ptr)
    c.run(ref.ptr)
    c.run(ref.ptr)
    brk.call("brk_stream_synchronize", None)
    x, y = st.download(), ref.download()
    assert same_bits(x, y)
    st.free()
    ref.free()


@pytest.mark.parametrize("n,dtype,seed", [(14, brk.C128, 21), (20, brk.C128, 22), (16, brk.C64, 23)])
def test_block_order_run_matches_plain(oracle, n, dtype, seed):
    """The circuit in block order (brk_circuit_block_order) run as gate blocks: fewer blocks,
    the same final permutation, amplitudes within rounding of the per-gate run of the given
    order (1e-12 complex128, 1e-5 complex64) and, for complex128, of the oracle."""
    note(f"gpu blocks: block order n={n} dtype={dtype} seed={seed}")
    ops = random_ops(n, 200, seed, local_swaps=4)
    c = brk.Circuit(n, ops)
    L = 12 if dtype == brk.C128 else 13
    ordered = c.reordered(c.block_order(L, 3 if dtype == brk.C128 else 4))
    nb = lambda p: sum(1 for _, _, local in p.steps if local)
    assert nb(brk.BlockPlan(ordered, dtype)) <= nb(brk.BlockPlan(c, dtype))
    rng = np.random.default_rng(seed)
    s = D.random_state(n, rng)
    if dtype == brk.C64:
        s = s.astype(np.complex64).astype(np.complex128)
    a, b = DeviceState.from_host(s, dtype), DeviceState.from_host(s, dtype)
    pa = c.run(a.ptr, dtype)
    pb = ordered.run_blocked(b.ptr, dtype)
    plain, blocked = a.download(), b.download()
    a.free()
    b.free()
    assert pa == pb
    tol = 1e-12 if dtype == brk.C128 else 1e-5
    assert np.max(np.abs(plain - blocked)) < tol
    if dtype == brk.C128:
        ref = s.copy()
        run_ops(oracle, ref, ops)
        assert np.max(np.abs(blocked - ref)) < 1e-12


@pytest.mark.parametrize("n,dtype,seed", [(22, brk.C128, 61), (23, brk.C64, 62), (24, brk.C128, 63)])
def test_many_controls_gate_by_gate_bitwise(n, dtype, seed):
    """Gates with up to 9 controls among others, on states where two or three of them are cheaper as plain
    kernels than as a launch: the bits of brk_circuit_run_timed (a plain kernel per op)."""
    note(f"gpu blocks: many controls n={n} dtype={dtype} seed={seed}")
    rng = np.random.default_rng(seed)
    ops = []
    for _ in range(12):
        ops += random_ops(n, int(rng.integers(1, 4)), int(rng.integers(1 << 30)), max_controls=9, local_swaps=1)
        q = [int(x) for x in rng.permutation(n)[:7]]
        ops += [("Z", (q[0],), tuple(q[1:]), ()), ("X", (q[0],), tuple(q[1:5]), ()),
                ("X", (q[1],), (q[0], q[2], q[3]), ())]
    s = D.random_state(n, rng)
    s[rng.random(s.size) < 0.3] = 0.0
    c = brk.Circuit(n, ops)
    a, b = DeviceState.from_host(s, dtype), DeviceState.from_host(s, dtype)
    final, _ = c.run_timed(a.ptr, dtype)
    assert c.run(b.ptr, dtype) == final
    want, got = a.download(), b.download()
    a.free()
    b.free()
    assert same_bits(want, got)


# brk_circuit_run itself runs in gate blocks: what follows compares with brk_circuit_run_timed, which launches
# a plain kernel for every op.
def gate_by_gate(n, ops, dtype, runs, perm0=None, seed=0):
    """The final state of the ops on plain kernels, and of every run (circuit, pointer) -> permutation."""
    rng = np.random.default_rng(seed)
    s = D.random_state(n, rng)
    c = brk.Circuit(n, ops)
    a = DeviceState.from_host(s, dtype)
    final, _ = c.run_timed(a.ptr, dtype, perm0)
    want = a.download()
    for run in runs:
        a.upload(s)
        assert run(c, a.ptr) == final
        yield want, a.download()
    a.free()


@pytest.mark.parametrize("n,dtype,seed", [(3, brk.C128, 1), (9, brk.C128, 2), (12, brk.C128, 3), (13, brk.C128, 4),
                                          (16, brk.C128, 5), (20, brk.C128, 6), (9, brk.C64, 10), (12, brk.C64, 7),
                                          (14, brk.C64, 8), (20, brk.C64, 9), (23, brk.C64, 11)])
def test_blocked_equals_gate_by_gate_bitwise(n, dtype, seed, access):
    note(f"gpu blocked vs gate by gate n={n} dtype={dtype} seed={seed} ({access})")
    ops = random_ops(n, 160, seed, local_swaps=3 if n >= 4 else 0)
    perm0 = [int(q) for q in np.random.default_rng(seed).permutation(n)]
    for want, got in gate_by_gate(n, ops, dtype, [lambda c, p: c.run_blocked(p, dtype, perm0)], perm0, seed):
        assert same_bits(want, got)


@pytest.mark.parametrize("dtype", [brk.C128, brk.C64])
def test_dense_low_qubits_gate_by_gate_bitwise(dtype):
    """Many gates on the line qubits and their neighbours: long blocks, every pair mode."""
    n = 18
    note(f"gpu blocks vs gate by gate: low-qubit circuit dtype={dtype}")
    ops = random_ops(n, 400, 11, qubit_pool=range(10))
    runs = [lambda c, p: c.run(p, dtype), lambda c, p: c.run_blocked(p, dtype)]
    for want, got in gate_by_gate(n, ops, dtype, runs, None, 11):
        assert same_bits(want, got)


@pytest.mark.parametrize("dtype", [brk.C128, brk.C64])
def test_large_state_gate_by_gate_bitwise(dtype):
    """26 qubits, a plan run twice and the circuit run twice against two runs of plain kernels."""
    n = 26
    note(f"gpu blocks vs gate by gate: n={n} dtype={dtype}")
    c = brk.Circuit(n, random_ops(n, 60, 12, max_controls=1))
    plan = brk.BlockPlan(c, dtype)
    got = []
    for run in (lambda p: c.run_timed(p, dtype), plan.run, lambda p: c.run(p, dtype)):
        st = DeviceState(n, dtype)
        brk.fill_modular(st.ptr, st.size, dtype, (1e-4, 3e-4), (7, 3, 101, 11, 5, 97))
        run(st.ptr)
        run(st.ptr)
        brk.call("brk_stream_synchronize", None)
        got.append(st.download())
        st.free()
    assert same_bits(got[0], got[1]) and same_bits(got[0], got[2])


@pytest.mark.parametrize("n,dtype", [(12, brk.C128), (14, brk.C64), (23, brk.C128)])
def test_captured_runs_replay(n, dtype):
    """A plan's run and a circuit's run captured in a graph: nothing of them lies in memory that a replay
    could find changed.  Several replays, each from a new state after other runs, bit for bit the plain
    kernels' result (23 qubits: launches and plain kernels)."""
    note(f"gpu blocks captured n={n} dtype={dtype}")

    def call(name, *args):  # the HIP runtime that the engine is linked against (its C ABI wraps no graphs)
        assert getattr(brk.load(), name)(*args) == 0, name

    rng = np.random.default_rng(n)
    ops = random_ops(n, 80, 70 + n, max_controls=4, local_swaps=2)
    ops += [("Z", (n - 1,), tuple(range(n - 8, n - 1)), ()), ("X", (n - 2,), tuple(range(n - 9, n - 2)), ())]
    c = brk.Circuit(n, ops)
    plan = brk.BlockPlan(c, dtype)
    st, other = DeviceState(n, dtype), DeviceState(n, dtype)
    stream = C.c_void_p(hip.create_stream())
    graphs = []
    for run in (plan.run, lambda p, s: c.run(p, dtype, None, s)):
        graph, executable = C.c_void_p(), C.c_void_p()
        call("hipStreamBeginCapture", stream, 0)
        run(st.ptr, stream.value)
        call("hipStreamEndCapture", stream, C.byref(graph))
        call("hipGraphInstantiate", C.byref(executable), graph, None, None, C.c_size_t(0))
        call("hipGraphDestroy", graph)
        graphs.append(executable)
    del plan
    for k in range(4):
        s = D.random_state(n, rng)
        other.upload(s)
        c.run_timed(other.ptr, dtype)
        want = other.download()
        for executable in graphs:
            st.upload(s)
            brk.call("brk_stream_synchronize", None)
            call("hipGraphLaunch", executable, stream)
            hip.synchronize(stream.value)
            assert same_bits(want, st.download()), k
            c.run(other.ptr, dtype)  # other runs between the replays
            brk.call("brk_stream_synchronize", None)
    for executable in graphs:
        call("hipGraphExecDestroy", executable)
    call("hipStreamDestroy", stream)
    st.free()
    other.free()


@pytest.mark.slow
def test_33_qubits_gate_by_gate_bitwise():
    """More than 2^32 amplitudes (64-bit indices in the blocks): gates, controls, moves and a local swap on the
    highest qubits, in gate blocks against plain kernels, every amplitude."""
    n = 33
    if hip.mem_info()[0] < 140 << 30:
        pytest.skip("needs 140 GiB of free device memory")
    note(f"gpu blocks: n={n} complex64")
    ops = [("H", (32,), (), ()), ("X", (0,), (32,), ()), ("RZ", (32,), (), (0.7,)), ("X", (32,), (5,), ()),
           ("U3", (31,), (), (0.3, 0.9, -0.4)), ("H", (4,), (32,), ()), ("Z", (32,), (31,), ()),
           ("SWAP", (32, 3), (), ()), ("RX", (3,), (32,), (1.1,)), ("LOCAL_SWAP", (32, 2), (), ()),
           ("RY", (32,), (), (0.2,)), ("ESWAP", (32, 30), (), (0.6,)), ("X", (32,), (30, 31), ()),
           ("EZ", (32, 7), (), (0.5,)), ("H", (20,), (), ()), ("X", (20,), (32,), ()), ("U1", (32,), (20,), (0.8,)),
           ("EX", (32, 8), (), (0.4,)), ("Y", (32,), (), ()), ("H", (32,), (), ())]
    c = brk.Circuit(n, ops)
    a, b = DeviceState(n, brk.C64), DeviceState(n, brk.C64)
    try:
        for st in (a, b):
            brk.fill_hash(st.ptr, st.size, brk.C64, 33, 2.0 ** -16)
        final, _ = c.run_timed(a.ptr, brk.C64)
        assert c.run(b.ptr, brk.C64) == final
        brk.call("brk_stream_synchronize", None)
        part = 1 << 30  # bytes a time
        x, y = np.empty(part // 8, dtype=np.uint64), np.empty(part // 8, dtype=np.uint64)
        for at in range(0, a.nbytes, part):
            if at % (8 * part) == 0:
                note(f"gpu blocks: n={n}, GiB {at // part} of {a.nbytes // part}")
            brk.call("brk_memcpy_dtoh", x.ctypes.data, a.ptr + at, part, None)
            brk.call("brk_memcpy_dtoh", y.ctypes.data, b.ptr + at, part, None)
            assert np.array_equal(x, y), at
    finally:
        a.free()
        b.free()
