"""The quad adjoint's reverse mode (jaxsso_amd/csrc/quad_adjoint.hpp) against forward mode
through the same element routines, on the CPU: 600 random elements (warped, square with
ties in the drilling minimum, orthotropic, thin, up to 40 m, nu = 0), lambda = u/2 and a
general lambda.  Both are exact derivatives, so they differ by rounding: some hundred
operations on an element of aspect ratio up to 6 and thickness 1e-3 leave well under 1e-11."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "jaxsso_amd", "csrc")
INCLUDE = os.path.join(HERE, "..", "include")


@pytest.fixture(scope="module")
def check_exe(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("adj") / "adjoint_reverse_check")
    r = subprocess.run([hipcc, "-O2", "-std=c++17", "-I", CSRC, "-I", INCLUDE,
                        os.path.join(HERE, "native", "adjoint_reverse_check.cpp"), "-o", out],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    return out


@pytest.mark.parametrize("plant", [0, 1, 2, 3])   # 1..3: planted mistakes, which it has to find
def test_reverse_mode_matches_forward_mode(check_exe, plant):
    r = subprocess.run([check_exe, str(plant)], capture_output=True, text=True, timeout=300)
    worst = float(r.stdout.strip().splitlines()[-1].split()[-1])
    if plant:
        assert r.returncode != 0 and worst > 1e-8, worst
    else:
        assert r.returncode == 0 and worst < 1e-11, r.stdout
