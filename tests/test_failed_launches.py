"""A launch that fails inside the density network's entry points: nothing they queued
is left behind (tests/host_runtime/failed_launches.cpp, on the CPU: a stand-in for
the HIP runtime makes each launch in turn fail)."""
import os
import shutil
import subprocess

import pytest

from conftest import MG1, REPO

import sqminiapp_amd as sq

ROCM = "/opt/rocm/include"
pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(ROCM), reason="needs g++ and HIP's headers")


def test_no_entry_point_returns_with_work_queued(tmp_path):
    sq.lib()
    libdir = os.path.join(REPO, "sqminiapp_amd")
    exe = str(tmp_path / "failed_launches")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I" + ROCM, "-rdynamic", "-o", exe,
                    os.path.join(REPO, "tests", "host_runtime", "failed_launches.cpp"), "-L" + libdir, "-lsqamd",
                    "-Wl,--allow-shlib-undefined", "-Wl,-rpath," + libdir], check=True)
    r = subprocess.run([exe, MG1, "Mg1"], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0 and "all queues empty" in r.stdout, r.stdout + r.stderr
