"""Deferred propagations (GPU): with one lane per link and steps of many links, a
propagation that needs a second layer search is saved (48 words) and continued by
a kernel of its own, past the buffer in place.  Only calls of hundreds of
thousands of seeds do so by themselves; here the line is set to 0, so that the
oracle-checked sizes take the same path.  The tracks are the ones of a team that
never defers: the same measurements, chi2 and parameters to 1e-5 relative (the
kernels' compiled arithmetic may fuse multiply-adds differently)."""
import ctypes as C

import numpy as np
import pytest

from traccc_amd import _ffi as F
from traccc_amd import ckf
from traccc_amd import simulation as S

pytestmark = pytest.mark.gpu

RULE = 0xffffffff


@pytest.fixture(scope="module", autouse=True)
def _gpu(gpu_available):
    return gpu_available


def _lib():
    lib = F.load_library(ckf.LIB)
    lib.ckf_debug_set_schedule.argtypes = [C.c_void_p, C.c_uint32]
    lib.ckf_debug_set_deferral.argtypes = [C.c_void_p, C.c_uint32, C.c_uint32]
    lib.ckf_debug_get_deferred.argtypes = [C.c_void_p, C.POINTER(C.c_uint64)]
    return lib


def _run(cfg, ddet, dev, lanes, from_links, capacity):
    lib = _lib()
    alg = ckf.combinatorial_kalman_filter_algorithm(cfg)
    assert lib.ckf_debug_set_schedule(alg._h, lanes) == 0
    assert lib.ckf_debug_set_deferral(alg._h, from_links, capacity) == 0
    tracks = alg.run_device(ddet, dev).download()
    n = C.c_uint64()
    assert lib.ckf_debug_get_deferred(alg._h, C.byref(n)) == 0
    return tracks, n.value, alg.last_stats()


@pytest.mark.parametrize("workload,n", [("C2", 3000), ("C4", 2000), ("C5", 2500)])
# the whole buffer, one that most propagations find full, one entry, and none
@pytest.mark.parametrize("capacity", [RULE, 8, 1, 0])
def test_deferred_propagations_give_the_same_tracks(workload, n, capacity):
    det, fld, gun = S.workload(workload, n_particles=n, seed=17)
    ev = S.generate_event(det, fld, gun)
    cfg = S.finding_config_for(workload)
    cfg.max_num_branches_per_surface = 2
    ddet = ckf.DeviceDetector(det, fld)
    dev = ckf.DeviceEvents(ddet, ev)
    want, none, _ = _run(cfg, ddet, dev, 4, RULE, RULE)
    got, asked, stats = _run(cfg, ddet, dev, 1, 0, capacity)
    assert none == 0
    if capacity == 0:
        assert asked == 0
    else:
        # a few percent of the propagations; more than the small buffers hold
        assert 0.001 * stats.n_propagations < asked < stats.n_propagations
        assert asked > 16 * stats.n_steps
    assert np.array_equal(got.offsets, want.offsets)
    assert np.array_equal(got.constituents, want.constituents)
    assert np.allclose(got.chi2, want.chi2, rtol=1e-5, atol=1e-6)
    assert np.allclose(got.params_vector, want.params_vector, rtol=1e-5, atol=1e-6)


def test_large_calls_defer_by_themselves():
    """The rule's own line: a step of 700,000 links needs 350,000 seeds."""
    det, fld, gun = S.workload("C2", n_particles=1000, seed=3)
    one = S.generate_event(det, fld, gun)
    cfg = S.finding_config_for("C2")
    cfg.max_num_branches_per_surface = 1
    ddet = ckf.DeviceDetector(det, fld)
    for events, defers in ((699, False), (701, True)):
        tracks, asked, stats = _run(cfg, ddet, ckf.DeviceEvents(ddet, [one] * events), 0, RULE, RULE)
        assert (one.n_seeds * events >= 700000) == defers
        assert (asked > 0) == defers
        first, last = tracks.event(0), tracks.event(events - 1)
        assert np.array_equal(first.offsets, last.offsets)
        assert np.array_equal(first.constituents, last.constituents)
        assert np.allclose(first.chi2, last.chi2, rtol=1e-5, atol=1e-6)
