"""How many lanes take a chain of work together (CPU): the rules of
traccc_amd/csrc/ckf/teams.hpp, compiled for the host."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ALL = 0xffffffff


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    out = tmp_path_factory.mktemp("teams") / "libteams.so"
    cmd = ["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-Wall", "-Itraccc_amd/csrc", "tests/cpp/teams_check.cpp",
           "-o", str(out)]
    b = subprocess.run(cmd, cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-3000:]
    lib = C.CDLL(str(out))
    lib.propagate_launches.argtypes = [C.c_uint32, C.c_uint64, C.c_uint32, C.POINTER(C.c_uint32)]
    lib.step_bound.restype = C.c_uint64
    lib.chain_team.argtypes = [C.c_uint64, C.c_uint32]
    return lib


def _launches(lib, n_cu, bound, fixed=0):
    out = (C.c_uint32 * 8)()
    lib.propagate_launches(n_cu, bound, fixed, out)
    return [tuple(out[4 * k:4 * k + 3]) for k in range(2) if out[4 * k]], [out[3], out[7]]


@pytest.mark.parametrize("bound,want", [
    (1, [(16, 0, ALL)]), (5120, [(16, 0, ALL)]), (5121, [(8, 0, ALL)]), (16384, [(8, 0, ALL)]),
    (16385, [(4, 8192, ALL), (16, 0, 8192)]), (32768, [(4, 8192, ALL), (16, 0, 8192)]),
    (32769, [(2, 27648, ALL), (8, 0, 27648)]), (57344, [(2, 27648, ALL), (8, 0, 27648)]),
    (57345, [(1, 27648, ALL), (8, 0, 27648)]), (1 << 30, [(1, 27648, ALL), (8, 0, 27648)])])
def test_propagation_launches(lib, bound, want):
    got, blocks = _launches(lib, 256, bound)
    assert got == want
    # every step has a launch, and its grid the waves that the chip holds at most
    assert sorted((f, b) for _, f, b in got)[0][0] == 0 and max(b for _, _, b in got) == ALL
    assert all(b <= 512 for b in blocks)
    # a part of the chip: the lines move with its CUs
    part, _ = _launches(lib, 32, -(-bound // 8))
    assert [t for t, _, _ in part] == [t for t, _, _ in want]
    assert _launches(lib, 256, bound, 4)[0] == [(4, 0, ALL)]


@pytest.mark.parametrize("seeds,surface,seed", [(30, 3, 100), (1000, 2, 100), (1000, 5, 10), (1, 3, 1)])
def test_a_large_call_before_changes_nothing(lib, seeds, surface, seed):
    """Buffers as large as a call of 60,000 seeds left them, and those of the call by itself."""
    own = seeds * min(seed, surface ** 2) * surface
    fresh = lib.step_bound(seeds, surface, seed, own, 0)
    assert fresh == own == lib.step_bound(seeds, surface, seed, 27 * 60000 * 3, 0)
    # a call that has outgrown its first buffers goes by what they are now
    assert lib.step_bound(seeds, surface, seed, 4 * own, 1) == 4 * own
    assert lib.step_bound(seeds, 1, seed, 4 * own, 1) == seeds


@pytest.mark.parametrize("n,want", [(0, 16), (1, 16), (5120, 16), (5121, 8), (28672, 8), (28673, 1), (1 << 32, 1)])
def test_chain_teams_follow_the_cus(lib, n, want):
    """The fit's and the progressive filter's teams: on an eighth of the chip an
    eighth of the chains fill it."""
    assert lib.chain_team(n, 256) == want
    assert lib.chain_team(-(-n // 8), 32) == want
