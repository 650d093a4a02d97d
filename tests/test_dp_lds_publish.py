"""A single solve returns when its kernel publishes "done": by then every wave
has to have written its part of the tables (gisbdw_amd/csrc/dplds.hpp, run on
the CPU thread by thread)."""
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


# one wave, two, four and sixteen
@pytest.mark.parametrize("n", [13, 14, 15, 18])
def test_done_follows_every_wave(tmp_path, n):
    exe = tmp_path / "lds_publish_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", str(HERE / "lds_publish_check.cpp"), "-o",
                    str(exe)], check=True)
    out = subprocess.run([str(exe), str(n)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout == f"ok {3 << (n - 5)}\n", out.stdout + out.stderr
