"""The host side of reads (rhip_ring.h: pinned rings, pieces, helper threads) on a stream of one thread, without a GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def ring_host(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("ring") / "ring_host")
    cmd = ["g++", "-std=c++17", "-O2", "-Wall", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
           "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "softglrender_amd", "csrc"), "-o", exe,
           os.path.join(ROOT, "tests", "ring_host.cpp"), "-ldl"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return exe


@pytest.mark.parametrize("check", ["bytes", "events", "idle", "refused", "helpers"])
def test_ring(ring_host, check):
    r = subprocess.run([ring_host, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr
