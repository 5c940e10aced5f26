"""The host's wait for a number that a kernel publishes (gip_amd/csrc/gip_wait.h),
on the CPU: a later number counts as arrived (another thread on the context
asked after this one), a finished stream without the number and a failed one
end the wait.
"""
import shutil
import subprocess

import pytest

from .conftest import ROOT


def test_wait_ends_as_it_should(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    exe = tmp_path / "wait_check"
    subprocess.run([gxx, "-O2", "-std=c++17", "-o", str(exe), str(ROOT / "tests" / "wait_check.cpp")], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout
    got = {n: (int(rc), int(q)) for n, rc, q in (line.split() for line in out.splitlines())}
    assert got == {"there": (0, 0), "newer": (0, 0), "wrapped": (0, 0), "missing": (1, 1), "arrives": (0, 2),
                   "last": (0, 1), "failed": (42, 1)}
