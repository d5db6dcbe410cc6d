"""Long SumOps on the CPU: tests/cpp/expect_long.cpp plans more distinct x
masks than the greedy search looks through and thousands of terms on one mask,
compares with the direct sums under the address and undefined-behaviour
sanitizers, and bounds the planning time of 65536 terms on one mask (quadratic
planning took about a minute here)."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_long_term_lists_are_planned_right_and_in_linear_time(tmp_path):
    exe = tmp_path / "expect_long"
    cmd = ["g++", "-O1", "-std=c++17", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
           str(ROOT / "tests" / "cpp" / "expect_long.cpp"), str(ROOT / "quant-iron_amd" / "csrc" / "expect_plan.cpp"),
           "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr[-3000:]
