"""Host bookkeeping of the ScanND forward's tiles (csrc/kernels/scannd_tiles.hpp)
in a CPU program under the address and undefined-behaviour sanitizers."""
import os
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_band_tables_hold_every_tiling(tmp_path):
    exe = tmp_path / "scannd_tiles_check"
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-Werror", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=undefined", f"-I{ROOT}/k-mamba_amd/csrc/kernels", "-o", str(exe),
                    str(ROOT / "tests" / "c" / "scannd_tiles_check.cpp")], check=True, timeout=120)
    env = {k: v for k, v in os.environ.items() if k != "LD_PRELOAD"}
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0, r.stdout + r.stderr[-3000:]
