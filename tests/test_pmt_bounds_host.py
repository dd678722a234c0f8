"""The error bound of the PMT detection's approximate weights, compiled for the host:
directions that are admitted as antipodes without being quite opposite."""
import os
import subprocess

import pytest

from conftest import ROOT

SRC = os.path.join(ROOT, "tests", "hostcheck", "pmt_bounds_check.cpp")


@pytest.fixture(scope="module")
def bounds_check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("pmt") / "pmt_bounds_check")
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "-O1", "-I",
                        os.path.join(ROOT, "include"), "-o", exe, SRC],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return exe


# shifts of each component: none, a rounding, and up to what is admitted (1e-6)
@pytest.mark.parametrize("shift", [0.0, 6e-8, 5e-7, 8e-7])
@pytest.mark.parametrize("sigma", [(0.217, 0.290), (0.3, 0.05), (0.4, 0.4)])
def test_bound_covers_directions(bounds_check, sigma, shift):
    r = subprocess.run([bounds_check, str(sigma[0]), str(sigma[1]), str(shift)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    tried, admitted, worst = r.stdout.split()
    print(tried, admitted, worst)
    assert int(admitted) > 0 or sigma != (0.217, 0.290)  # the POM's own widths are served
    assert float(worst) <= 1.0


def test_shifts_beyond_the_limit_are_refused(bounds_check):
    r = subprocess.run([bounds_check, "0.217", "0.29", "2e-6"], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.split()[1] == "0"
