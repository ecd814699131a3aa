"""The end of a step (CPU): k_prop_emit's last partition advances the control
block while other blocks of the launch may only be starting.  Whatever mixture of
old and new words such a block reads, it goes by the same partitions as the
others, finds their queue spent and does nothing.  Compiles
traccc_amd/csrc/ckf/step_ctl.hpp for the host."""
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
    out = tmp_path_factory.mktemp("step") / "libstepctl.so"
    cmd = ["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-Wall", "-Iinclude", "-Itraccc_amd/csrc",
           "tests/cpp/step_ctl_check.cpp", "-o", str(out)]
    b = subprocess.run(cmd, cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-3000:]
    return C.CDLL(str(out))


def test_fewer_links_may_be_more_partitions(lib):
    """Why a late block must not go by fewer links than the others."""
    assert lib.emit_parts(32768) == 64 and lib.emit_parts(32767) == 128


# links on both sides of where partitions grow; link buffers that hold the step with
# room for the next one's base, just so, and far more; tips and inputs overflowing
@pytest.mark.parametrize("n_links", [1, 255, 256, 32767, 32768, 65535, 65536, 300000])
@pytest.mark.parametrize("room", [0, 1, 1000, 32767, 65535, 10000000])
@pytest.mark.parametrize("n_live,raised", [(0, 0), (77, 0), (77, 8 | 16)])
def test_torn_control_block(lib, n_links, room, n_live, raised):
    n = C.c_uint32()
    wrong = lib.torn_extents(n_links, 50000, 50000 + n_links + room, n_live, 5, 20, raised, C.byref(n))
    assert n.value >= 64 and wrong == 0
