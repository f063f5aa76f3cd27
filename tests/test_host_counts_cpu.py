"""csrc/host_counts.h (the counts per expert that moe_dispatch_prefill watches arrive) without a GPU: a C++ program with
stand-ins for the HIP calls.  Which device and flags the buffer is allocated with, several threads, streams that end or fail
without the counts, calls that fail while their kernels are still queued."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_counts") / "check")
    subprocess.check_call([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-Wall", "-pthread", "-D__HIP_PLATFORM_AMD__=1",
                           "-I", "/opt/rocm/include", os.path.join(HERE, "host_counts_check.cpp"), "-o", out])
    return out


@pytest.mark.parametrize("check", ["device", "arrive", "threads", "errors", "late"])
def test_host_counts(program, check):
    p = subprocess.run([program, check], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert p.returncode == 0, p.stdout
