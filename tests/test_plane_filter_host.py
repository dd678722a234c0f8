"""The plane filter of the mixed every-target scan, compiled for the host: it may
let misses through, never pass over a hit."""
import os
import subprocess

import pytest

from conftest import ROOT

SRC = os.path.join(ROOT, "tests", "hostcheck", "plane_check.cpp")


@pytest.fixture(scope="module")
def plane_check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plane") / "plane_check")
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "-O1", "-I",
                        os.path.join(ROOT, "include"), "-o", exe, SRC],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return exe


@pytest.mark.parametrize("scale", [1e-3, 1.0, 30.0, 1e4])
def test_no_hit_is_passed_over(plane_check, scale):
    r = subprocess.run([plane_check, str(scale), "3", "2000000"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    hits, over, through = map(int, r.stdout.split())
    print(hits, over, through)
    assert hits > 200_000 and over == 0
