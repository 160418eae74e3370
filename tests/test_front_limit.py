"""The limit of the direct solve's symbolic analysis on the CPU: it refuses exactly the
patterns with a larger front, and a mesh far past it at its first cuts (the analysis of one
that the direct solve does not take is thrown away)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_front_limit(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no C++ compiler")
    out = str(tmp_path / "front_limit_check")
    r = subprocess.run([cxx, "-O2", "-std=c++17", os.path.join(HERE, "native", "front_limit_check.cpp"), "-o", out],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([out], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    # one cut of the whole mesh where the analysis has 14 levels of them
    assert float(r.stdout.split()[-1]) < 0.5, r.stdout
