"""The direct solve's symbolic analysis (nested dissection and fronts,
jaxsso_amd/csrc/direct_symbolic.hpp) on the CPU: a multifrontal Cholesky over its
fronts against a dense Cholesky, on grids, chains, a star, a clique, random graphs,
several components and single nodes, with leaves of 1 and 12 nodes."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check_exe(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no C++ compiler")
    out = str(tmp_path_factory.mktemp("fronts") / "front_check")
    r = subprocess.run([cxx, "-O2", "-std=c++17", os.path.join(HERE, "native", "front_check.cpp"), "-o", out],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    return out


def _run(exe, plant):
    r = subprocess.run([exe, str(plant)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-500:]
    return {ln.split()[0]: [float(v) for v in ln.split()[1:]] for ln in r.stdout.strip().splitlines()}


def test_fronts_factor_like_dense(check_exe):
    # diagonally dominant matrices of up to 418 rows: both factorisations are exact to a
    # few hundred roundings
    got = _run(check_exe, 0)
    assert len(got) == 26
    assert max(v[-1] for v in got.values()) < 1e-13, got
    # a 31 x 8 mesh is cut across: the largest front stays near two separators
    assert got["quad_31x8_leaf12"][3] <= 30 and got["quad_2x200_leaf12"][3] <= 24


@pytest.mark.parametrize("plant", [1, 2])
def test_fronts_check_catches_planted_mistakes(check_exe, plant):
    assert max(v[-1] for v in _run(check_exe, plant).values()) > 1e-3
