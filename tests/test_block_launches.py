"""CPU checks of which kernels a circuit launches (tests/cpp/block_launch_check.cpp, compiled here against the
library): a launch of a gate block moves the whole state, so gates that act on a small part of a large
state keep their plain kernels."""
import os
import shutil
import subprocess

import pytest

import brk

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "riken-braket_amd")


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("launches") / "block_launch_check")
    subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(PKG, "host"), "-I" + os.path.join(PKG, "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "block_launch_check.cpp"), "-L" + PKG, "-lbraket_hip",
                    "-L/opt/rocm/lib", "-Wl,-rpath-link,/opt/rocm/lib", "-Wl,-rpath," + PKG], check=True)

    def run(n, dtype, ops):
        text = "".join(" ".join(str(x) for x in [brk.OP[name], len(t), *t, len(c), *c, len(p), *p]) + "\n"
                       for name, t, c, p in ops)
        r = subprocess.run([exe, str(n), str(dtype)], input=text, capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stdout + r.stderr
        run, plan = r.stdout.split("plan\n")
        assert run == plan  # a circuit's run and its plan's launch the same
        code = {v: k for k, v in brk.OP.items()}
        return [("block", int(x)) if kind == "block" else ("plain", code[int(x)])
                for kind, x in (line.split() for line in run.splitlines())]

    return run


def controlled(name, target, num_controls):
    return (name, (target,), tuple(range(target - num_controls, target)), ())


def test_gates_with_many_controls_stay_plain(launches):
    """Two gates on 2^-11 or 2^-4 of 28 qubits: a launch would move 2^28 amplitudes for them."""
    z = [controlled("Z", 27, 10), controlled("Z", 26, 10)]
    x = [controlled("X", 27, 4), controlled("H", 26, 4), controlled("X", 25, 4)]
    for dtype in (brk.C128, brk.C64):
        assert launches(28, dtype, z) == [("plain", "Z"), ("plain", "Z")]
        assert launches(28, dtype, x) == [("plain", "X"), ("plain", "H"), ("plain", "X")]
        # enough of them, or one that acts on every amplitude and one on a quarter: a launch
        assert launches(28, dtype, x * 8) == [("block", 24)]
        assert launches(28, dtype, [("H", (27,), (), ()), ("Z", (26,), (25,), ())]) == [("block", 2)]
        # small states: what counts is the number of launches
        assert launches(13, dtype, [controlled("Z", 12, 10), controlled("Z", 11, 8)]) == [("block", 2)]


def test_line_between_launch_and_plain_kernels(launches):
    """Two CNOT act on half the state each: 1.36 against 1.42 ms at 28 qubits complex128, 0.73 against 0.70
    complex64.  A condition within a line of memory saves nothing."""
    cnots = [("X", (27,), (20,), ()), ("X", (26,), (21,), ())]
    assert launches(28, brk.C128, cnots) == [("plain", "X"), ("plain", "X")]
    assert launches(28, brk.C64, cnots) == [("block", 2)]
    for dtype in (brk.C128, brk.C64):
        assert launches(28, dtype, [("Z", (0,), (1,), ()), ("Z", (0,), (1,), ())]) == [("block", 2)]
        assert launches(28, dtype, [("X", (27,), (0,), ()), ("X", (26,), (1,), ())]) == [("block", 2)]
        # a SWAP moves half the amplitudes; of a lane and a high qubit, every line of the state
        assert launches(28, dtype, [("SWAP", (26, 27), (), ()), controlled("Z", 25, 10)]) == [("plain", "SWAP"),
                                                                                             ("plain", "Z")]
        assert launches(28, dtype, [("SWAP", (0, 27), (), ()), ("SWAP", (1, 26), (), ())]) == [("block", 2)]


def test_lone_gate_stays_plain(launches):
    assert launches(20, brk.C128, [("H", (3,), (), ())]) == [("plain", "H")]
