"""The expectation planner (expect_plan.cpp), checked on the CPU: the model in
tests/cpp/expect_emu.cpp evaluates its tables the way k_expect_tiles does and
compares with the direct sum over terms, for chains and random strings of 4 to
16 qubits in both tile shapes (wide masks, masks no tile holds, complex
coefficients, repeated masks), under the address and undefined-behaviour
sanitizers."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    exe = tmp_path_factory.mktemp("expect_emu") / "expect_emu"
    cmd = ["g++", "-O1", "-std=c++17", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
           str(ROOT / "tests" / "cpp" / "expect_emu.cpp"), str(ROOT / "quant-iron_amd" / "csrc" / "expect_plan.cpp"),
           "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return exe


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_planned_tables_equal_the_direct_sum(emu, seed):
    r = subprocess.run([str(emu), str(seed)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr[-3000:]
