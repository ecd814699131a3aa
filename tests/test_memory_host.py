"""Result blocks and read-backs around several devices (CPU): compiles
csrc/ckf/handles.hpp and csrc/common/readback.hip with g++ for a runtime that
keeps devices, allocations and launches on the host (tests/cpp/host_runtime)."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    out = tmp_path_factory.mktemp("memory") / "libmemory.so"
    cmd = ["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-Wall", "-Wno-class-memaccess", "-Itests/cpp/host_runtime",
           "-Iinclude", "-Itraccc_amd/csrc", "-x", "c++", "tests/cpp/memory_check.cpp",
           "traccc_amd/csrc/common/readback.hip", "-o", str(out), "-lpthread"]
    b = subprocess.run(cmd, cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-3000:]
    return C.CDLL(str(out))


def test_cached_blocks_stay_on_their_device(lib):
    assert lib.cache_keeps_devices_apart() == 0


# one chunk, two, and more than are on their way at once (copied by threads)
@pytest.mark.parametrize("n", [1, 777, 15000, 120000])
@pytest.mark.parametrize("device", [0, 1, 2])
def test_read_back_runs_where_the_result_is(lib, device, n):
    assert lib.read_back_from(device, n) == 0
