"""Staging and planning memory (stage.cpp) on the CPU with the HIP calls
replaced (tests/cpp/stage_host.cpp), under the address and undefined-behaviour
sanitizers: a failed growth loses nothing, large tables are not kept."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_staging_memory(tmp_path):
    exe, csrc = tmp_path / "stage_host", ROOT / "quant-iron_amd" / "csrc"
    cmd = ["g++", "-O1", "-std=c++17", "-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-D__HIP_PLATFORM_AMD__",
           "-I/opt/rocm/include", str(ROOT / "tests" / "cpp" / "stage_host.cpp"), str(csrc / "stage.cpp"),
           str(csrc / "host_common.cpp"), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr[-3000:]
