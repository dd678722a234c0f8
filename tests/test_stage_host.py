"""Copies through pinned halves (pp_stage.h), compiled for the host over stand-ins of
the runtime's calls: also where no pinned memory is left."""
import os
import subprocess

import pytest

from conftest import ROOT

SRC = os.path.join(ROOT, "tests", "hostcheck", "stage_check.cpp")


@pytest.fixture(scope="module")
def stage_check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("stage") / "stage_check")
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "-O1", "-I",
                        os.path.join(ROOT, "include"), "-o", exe, SRC],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return exe


def test_every_byte_arrives(stage_check):
    r = subprocess.run([stage_check], capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stderr[-2000:])
    checked, without = map(int, r.stdout.split())
    assert checked == 52 and without > 12
