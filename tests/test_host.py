"""The library's host code on the CPU, over a HIP runtime that records (tests/fake_hip.cpp): which kernels a call takes,
who may use which workspace on which stream, and what happens where memory runs out."""
import os
import subprocess
import sys

import pytest

import host_cases
from smq_pkg import ROOT

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(ROOT, "smolmoe-c99_amd", "libsmq_gfx950.so")


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if not os.path.exists(LIB):
        pytest.skip("libsmq_gfx950.so is not built")
    out = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-fPIC", "-shared", "-I/opt/rocm/include", "-o", out,
                    os.path.join(HERE, "fake_hip.cpp")], check=True)
    return out


@pytest.mark.parametrize("case", [f.__name__ for f in host_cases.CASES])
def test_host(fake, case):
    r = subprocess.run([sys.executable, os.path.join(HERE, "host_cases.py"), fake, case], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout[-2000:] + r.stderr[-4000:]
