"""fof_link_gpu_noalloc as the first call of a context makes nothing through the
HIP runtime: no device or page-locked memory, stream, event or graph
(tests/c_caller/noalloc_caller.c counts the library's calls)."""
import os
import subprocess

import pytest

from cm_halofinder_amd import _lib as L

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_first_noalloc_call_makes_nothing(tmp_path):
    exe = str(tmp_path / "noalloc_caller")
    libdir = os.path.dirname(L.LIB_PATH)
    subprocess.run(["gcc", "-O2", "-std=c99", "-Wall", "-rdynamic", "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "c_caller", "noalloc_caller.c"), "-o", exe, "-L", libdir, "-lcmfof",
                    "-L", "/opt/rocm/lib", "-lamdhip64", "-ldl", f"-Wl,-rpath,{libdir}", "-Wl,-rpath,/opt/rocm/lib"],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    count = {line.split()[0]: line.split()[1:] for line in r.stdout.splitlines() if line}
    assert count["noalloc"] == ["0"], r.stdout
    assert "hipMalloc" in count["ex"], r.stdout
