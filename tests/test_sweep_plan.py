"""CPU checks of the planner of the adjoint gradient's sweeps (riken-braket_amd/host/sweep.cpp): the program
tests/cpp/sweep_plan_check.cpp, compiled here with the planner, plans a circuit and reads its programs back."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "riken-braket_amd")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("sweep") / "sweep_plan_check")
    subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", "-I" + os.path.join(PKG, "host"),
                    "-I" + os.path.join(PKG, "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "sweep_plan_check.cpp"),
                    os.path.join(PKG, "host", "sweep.cpp")], check=True)

    def run(kind, gates, n, num_local):
        r = subprocess.run([exe, kind, str(gates), str(n), str(num_local)], capture_output=True, text=True, timeout=300)
        print(r.stdout, flush=True)
        values = dict(re.findall(r"(\w+) ([\d.]+)", r.stdout))
        return r.returncode, {k: float(v) for k, v in values.items()}

    return run


@pytest.mark.parametrize("kind,gates,n,num_local", [("chain", 66000, 12, 12), ("chain", 66000, 20, 11),
                                                    ("layers", 300000, 12, 12), ("layers", 576, 24, 11),
                                                    ("phases", 3000, 14, 11)])
def test_every_gate_runs_once(check, kind, gates, n, num_local):
    """Also in circuits of more than 2^16 macros, and in blocks of a bounded size."""
    code, got = check(kind, gates, n, num_local)
    assert got["status"] == 0 and got["blocks"] >= 1
    assert (got["wrong"], got["missed"], got["twice"]) == (0, 0, 0)
    assert code == 0


@pytest.mark.parametrize("kind,gates,n,num_local", [("chain", 100000, 12, 12), ("phases", 60000, 20, 11),
                                                    ("layers", 300000, 12, 12)])
def test_planning_time_grows_with_the_circuit(check, kind, gates, n, num_local):
    """About 2 us a gate (0.1-0.2 s here), however long the circuit: planning that looks at all gates left for
    every macro or segment takes 8 s or more for the first and the second."""
    code, got = check(kind, gates, n, num_local)
    assert code == 0
    assert got["seconds"] < 1.5
