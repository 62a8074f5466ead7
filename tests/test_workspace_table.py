"""The library's scratch table (csrc/km_runtime.cpp) in a CPU program that
stands in for the HIP calls it makes: what a failed allocation, a full table
and a race for its last place leave behind."""
import os
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_optional_scratch_disturbs_nothing(tmp_path):
    exe = tmp_path / "workspace_check"
    csrc = ROOT / "k-mamba_amd" / "csrc"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-fsanitize=address",
                    f"-I{rocm}/include", f"-I{ROOT}/include", f"-I{csrc}", "-o", str(exe),
                    str(ROOT / "tests" / "c" / "workspace_check.cpp"), str(csrc / "km_runtime.cpp"),
                    "-lpthread", "-Wl,--unresolved-symbols=ignore-all"], check=True, timeout=120,
                   stderr=subprocess.DEVNULL)
    env = {k: v for k, v in os.environ.items() if k != "LD_PRELOAD"}
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60, env=env)
    assert r.returncode == 0, r.stdout + r.stderr[-3000:]
