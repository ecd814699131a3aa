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


def test_large_results_take_what_they_need(lib):
    """A fit's columns for 3.8 million tracks of 37 million states, and a small one's."""
    lib.bytes_over.restype = C.c_uint64
    for tracks, states in ((3840000, 37300000), (20000, 106000)):
        need = [2 * tracks, 4 * tracks, 24 * tracks, 84 * tracks, 4 * tracks, 4 * states, 128 * states, 128 * states, states]
        over = lib.bytes_over((C.c_uint64 * len(need))(*need), len(need))
        # an eighth up to 256 MiB, a sixteenth up to 1 GiB, and a step of a sixteenth; 2 MiB beyond
        assert over < sum(n // 5 if n <= 256 << 20 else n // 7 if n <= 1 << 30 else 2 << 20
                          for n in need) + len(need) * (2 << 20)
    small = [1, 255, 256, 257, 4000, 100000]
    assert lib.bytes_over((C.c_uint64 * len(small))(*small), len(small)) <= sum(small) + 256 * len(small)


@pytest.mark.parametrize("size", [1000, 300000, 5000000, 90000000])
def test_events_of_different_sizes_reuse_blocks(lib, size):
    lib.allocations_of.restype = C.c_uint64
    lib.allocations_of.argtypes = [C.c_uint64, C.c_uint32]
    # sizes spread over 0.8 to 1.2: one that is an eighth larger than any before needs a new block
    assert lib.allocations_of(size, 200) <= 8


def test_blocks_of_a_larger_call_before_do_not_keep_later_ones_out(lib):
    lib.allocations_after.restype = C.c_uint64
    lib.allocations_after.argtypes = [C.c_uint64, C.c_uint64, C.c_uint32]
    gb = 1 << 30
    for stale in (gb, int(3.9 * gb), 9 * gb):
        assert lib.allocations_after(stale, gb, 50) <= 2


def test_a_full_device_gets_the_cached_blocks_back(lib):
    lib.room_from_the_cache.argtypes = [C.c_uint64] * 3
    assert lib.room_from_the_cache(100 << 20, 70 << 20, 34 << 20) == 0
    assert lib.room_from_the_cache(100 << 20, 70 << 20, 80 << 20) == 0


def test_a_buffer_whose_growth_failed_is_empty(lib):
    """A call that runs out of memory leaves an object that the next, smaller call can use."""
    assert lib.buffer_after_a_failed_growth() == 0


# one chunk, two, and more than are on their way at once (copied by threads)
@pytest.mark.parametrize("n", [1, 777, 15000, 120000])
@pytest.mark.parametrize("device", [0, 1, 2])
def test_read_back_runs_where_the_result_is(lib, device, n):
    assert lib.read_back_from(device, n) == 0


@pytest.mark.parametrize("n", [1, 777, 15000, 120000])
def test_read_back_without_pinned_memory(lib, n):
    assert lib.read_back_without_pinned_memory(n) == 0


def test_large_transfers_pin_no_block_of_their_own(lib):
    lib.staging.restype, lib.staging.argtypes = C.c_uint64, [C.c_uint64] * 2
    mb = 1 << 20
    assert lib.staging(5000, 100 * mb) == 8192
    assert lib.staging(32 * mb, 100 * mb) == 32 * mb
    assert lib.staging(32 * mb + 1, 100 * mb) == 0
    assert lib.staging(5000, 0) == 0
