"""Which SumOps the planner sends to tile passes and which it streams, on both
sides of each limit (tests/cpp/expect_routes.cpp, on the CPU)."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_lists_on_both_sides_of_each_limit(tmp_path):
    exe = tmp_path / "expect_routes"
    cmd = ["g++", "-O1", "-std=c++17", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
           str(ROOT / "tests" / "cpp" / "expect_routes.cpp"), str(ROOT / "quant-iron_amd" / "csrc" / "expect_plan.cpp"),
           "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr[-3000:]
