"""The account of the two vectors of the single-launch solves (senk_amd/csrc/sweep_vec.hpp),
built with g++: whatever solves ran, were refused or failed before, a solve finds its vector
holding the sentinel.  The same program with refused solves counted as solved must report a
vector that does not."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_every_solve_finds_a_clean_vector(tmp_path):
    exe = tmp_path / "sweep_vec"
    r = subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-fsanitize=address,undefined", f"-I{ROOT / 'senk_amd' / 'csrc'}",
                        str(ROOT / "tests" / "sanitize" / "sweep_vec_main.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    env = {"PATH": "/usr/bin:/bin"}
    ok = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60, env=env)
    assert ok.returncode == 0 and ok.stderr == "", ok.stdout + ok.stderr
    assert subprocess.run([str(exe), "refused"], capture_output=True, timeout=60, env=env).returncode == 1
