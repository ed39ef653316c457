"""A call that fails after it has forked work to other streams waits for all of
them before it returns (tests/c_caller/failing_caller.c)."""
import os
import subprocess

import pytest

from cm_halofinder_amd import _lib as L

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_failed_call_waits_for_its_streams(tmp_path):
    exe = str(tmp_path / "failing_caller")
    libdir = os.path.dirname(L.LIB_PATH)
    subprocess.run(["gcc", "-O2", "-std=c99", "-Wall", "-rdynamic", "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "c_caller", "failing_caller.c"), "-o", exe, "-L", libdir, "-lcmfof",
                    "-L", "/opt/rocm/lib", "-lamdhip64", "-ldl", f"-Wl,-rpath,{libdir}", "-Wl,-rpath,/opt/rocm/lib"],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    waited = [int(line.split()[1]) for line in r.stdout.splitlines()]
    # the fork of the pipelines, and each one's fork, join and its own join:
    # two pipelines with a side stream each
    assert len(waited) >= 6 and min(waited) == 4, waited
