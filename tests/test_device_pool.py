"""The device memory pool's rules on the CPU: csrc/runtime.cpp linked against
a counting stand-in for the HIP calls it makes (tests/cpp/pool_check.cpp),
under AddressSanitizer and UndefinedBehaviorSanitizer."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "btc-tc-artifact_amd")
HIP_INC = "/opt/rocm/include"

pytestmark = pytest.mark.skipif(not shutil.which("g++") or not os.path.isdir(HIP_INC),
                                reason="needs g++ and the HIP headers")


@pytest.fixture(scope="module")
def pool_check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("pool") / "pool_check")
    cmd = ["g++", "-std=c++17", "-g", "-O1", "-fopenmp", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
           "-I", os.path.join(ROOT, "include"), "-I", os.path.join(PKG, "csrc"), "-I", HIP_INC,
           "-D__HIP_PLATFORM_AMD__", os.path.join(PKG, "csrc", "runtime.cpp"),
           os.path.join(ROOT, "tests", "cpp", "pool_check.cpp"), "-o", exe]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout
    return exe


@pytest.mark.parametrize("check", ["per_thread_stream", "no_waits", "handles", "waited_streams", "bounded",
                                   "sizes", "trim", "count_sums"])
def test_pool(pool_check, check):
    r = subprocess.run([pool_check, check], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0 and "pool ok" in r.stdout, r.stdout[-4000:]
