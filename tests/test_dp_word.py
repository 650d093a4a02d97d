"""The bitwise word solver of the subset DP (gisbdw_amd/csrc/dpword.hpp),
compiled for the CPU, against the textbook recurrence on every subset."""
import subprocess
from pathlib import Path

HERE = Path(__file__).resolve().parent


def test_word_solver_equals_recurrence(tmp_path):
    exe = tmp_path / "word_check"
    subprocess.run(["g++", "-O2", "-std=c++17", str(HERE / "word_check.cpp"), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout
