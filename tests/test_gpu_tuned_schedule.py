"""The autotuner's trials overlap the link kernels where the tuned call does:
an eager call forks them to a side stream, a captured or timed one runs them
one after the other (tests/c_caller/schedule_caller.c counts the forks)."""
import os
import subprocess

import pytest

from cm_halofinder_amd import _lib as L

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_trials_run_the_schedule_of_the_call(tmp_path):
    exe = str(tmp_path / "schedule_caller")
    libdir = os.path.dirname(L.LIB_PATH)
    subprocess.run(["gcc", "-O2", "-std=c99", "-Wall", "-rdynamic", "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "c_caller", "schedule_caller.c"), "-o", exe, "-L", libdir, "-lcmfof",
                    "-L", "/opt/rocm/lib", "-lamdhip64", "-ldl", f"-Wl,-rpath,{libdir}", "-Wl,-rpath,/opt/rocm/lib"],
                   check=True)
    env = {k: v for k, v in os.environ.items() if k != "FOF_TUNE_CACHE"}
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0, r.stdout + r.stderr
    forks = {line.split()[0]: int(line.split()[1]) for line in r.stdout.splitlines()}
    assert forks["eager"] == 2 and forks["tuned"] > 2
    assert [forks[k] for k in ("timed", "graph", "tuned+graph", "tuned+timed")] == [0] * 4, forks
