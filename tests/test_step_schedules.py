"""Which kernels a step runs is chosen by how much of it there is; the tracks
do not depend on it (GPU).

The sizes lie on both sides of every line of the choice: one branch per
surface bounds a step's links by the seeds, so 5,000 muons take one launch of
16-lane teams, 16,000 one of 8-lane teams, 30,000 a 4 / 16 pair, 50,000 a 2 / 8
pair and 60,000 a 1 / 8 pair; their later steps, with ever fewer links, cross
from the first launch of a pair to the second.
"""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from traccc_amd import _ffi as F
from traccc_amd import ckf
from traccc_amd import simulation as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu(gpu_available):
    return gpu_available


def _columns(tracks):
    return [tracks.offsets, tracks.constituents, tracks.chi2, tracks.ndf, tracks.pval, tracks.nholes]


@pytest.mark.parametrize("n,branches", [(1, 1), (5120, 1), (5121, 1), (16384, 1), (16385, 1), (32769, 1),
                                        (57345, 1), (3000, 3)])
def test_propagation_launches_by_size(n, branches):
    """The chosen launches and a fixed team give the same tracks, bit for bit."""
    det, fld, gun = S.workload("C2", n_particles=n, seed=29)
    ev = S.generate_event(det, fld, gun)
    cfg = S.finding_config_for("C2")
    cfg.max_num_branches_per_surface = branches
    lib = F.load_library(ckf.LIB)
    lib.ckf_debug_set_schedule.argtypes = [C.c_void_p, C.c_uint32]
    ddet = ckf.DeviceDetector(det, fld)
    dev = ckf.DeviceEvents(ddet, ev)
    alg = ckf.combinatorial_kalman_filter_algorithm(cfg)
    got = _columns(alg.run_device(ddet, dev).download())
    assert lib.ckf_debug_set_schedule(alg._h, 4) == 0
    want = _columns(alg.run_device(ddet, dev).download())
    assert len(want[2]) > 0.9 * ev.n_seeds
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [255, 256, 257, 1024, 1025, 32768, 65537])
def test_compaction_partition_edges(n):
    """Compaction works on partitions of 256 items, of 512 from 32,768 items on
    and so up to 1,024 from 65,536 on: a batch of small events with that many
    seeds in all gives each event the tracks the CPU oracle finds in it."""
    import oracle
    from concurrent.futures import ThreadPoolExecutor
    det, fld, gun = S.workload("C1", n_particles=512, seed=31)
    sizes = [512] * (n // 512) + ([n % 512] if n % 512 else [])
    guns = [dataclasses.replace(gun, n_particles=k, seed=700 + e) for e, k in enumerate(sizes)]
    events = S.generate_events(det, fld, guns)
    cfg = S.finding_config_for("C1")
    ddet = ckf.DeviceDetector(det, fld)
    got = ckf.combinatorial_kalman_filter_algorithm(cfg).run_device(ddet, ckf.DeviceEvents(ddet, events)).download()
    with ThreadPoolExecutor(8) as pool:
        want = list(pool.map(lambda ev: oracle.run(cfg, det, fld, ev, 64), events))
    assert sum(e.n_seeds for e in events) == n
    for e, w in enumerate(want):
        g = got.event(e)
        assert np.array_equal(g.offsets, w.offsets), e
        assert np.array_equal(g.constituents, w.constituents), e


@pytest.mark.parametrize("minimum", [0, 1, 2, 3, 4, 7])
def test_duplicate_removal_lengths(minimum):
    """Links are compared by the hash of the measurements that duplicates must
    share, which are fewer than four for a small minimum length: the tracks are
    the oracle's for every minimum (dense enough that some links are dropped)."""
    import oracle
    det, fld, gun = S.workload("C4", n_particles=2500, seed=37)
    ev = S.generate_event(det, fld, gun)
    # every second seed again: identical histories from different seeds
    again = np.concatenate([np.arange(ev.n_seeds), np.arange(0, ev.n_seeds, 2)])
    ev = S.with_seeds(ev, ev.seed_surface_link[again], ev.seed_vector[again], ev.seed_covariance[again],
                      ev.seed_particle[again])
    cfg = S.finding_config_for("C4")
    cfg.max_num_branches_per_surface = 3
    cfg.duplicate_removal_minimum_length = minimum
    got = ckf.combinatorial_kalman_filter_algorithm(cfg)(det, fld, ev)
    want = oracle.run(cfg, det, fld, ev, 64)
    assert len(want) < 1.5 * len(again)
    assert np.array_equal(got.offsets, want.offsets)
    assert np.array_equal(got.constituents, want.constituents)


@pytest.mark.parametrize("events", [2, 10])  # 6,000 and 30,000 seeds
def test_progressive_teams_and_window(events):
    """The progressive filter walks a seed with 16, 8 or one lane by how many
    seeds there are: an event's tracks are the same alone and in a batch, and with
    its surfaces' measurements in reverse order (no loc0 window then)."""
    det, fld, gun = S.workload("C4", n_particles=3000, seed=41)
    evs = S.generate_events(det, fld, [dataclasses.replace(gun, seed=90 + e) for e in range(events)])
    cfg = S.finding_config_for("C4")
    cfg.run_pkf = 1
    ddet = ckf.DeviceDetector(det, fld)
    alg = ckf.combinatorial_kalman_filter_algorithm(cfg)
    one = alg.run_device(ddet, ckf.DeviceEvents(ddet, evs[:1])).download()
    many = alg.run_device(ddet, ckf.DeviceEvents(ddet, evs)).download()
    assert len(one) <= 5120 < len(many) and (len(many) > 28672) == (events == 10)
    assert np.diff(one.offsets.astype(np.int64)).max() > 3
    for a, b in zip(_columns(one), _columns(many.event(0))):
        assert np.array_equal(a, b)
    sl = evs[0].surface_link
    order = np.lexsort((-np.arange(len(sl)), sl))
    rev = dataclasses.replace(evs[0], **{f: np.ascontiguousarray(getattr(evs[0], f)[order]) for f in (
        "local_position", "local_variance", "dimensions", "time", "diameter", "identifier", "surface_link", "subspace",
        "cluster_index", "meas_particle")}, _keep=[])
    back = alg.run_device(ddet, ckf.DeviceEvents(ddet, rev)).download()
    assert np.array_equal(one.offsets, back.offsets) and np.array_equal(one.constituents, order[back.constituents])
    assert np.array_equal(one.chi2, back.chi2)


def test_small_event_after_a_large_one():
    """The launches of a call go by its own seeds, not by the buffers that an
    earlier, larger call of the same object left."""
    det, fld, gun = S.workload("C4", n_particles=9000, seed=43)
    large, small = S.generate_events(det, fld, [gun, dataclasses.replace(gun, n_particles=40, seed=44)])
    cfg = S.finding_config_for("C4")
    cfg.max_num_branches_per_surface = 3
    lib = F.load_library(ckf.LIB)
    lib.ckf_debug_get_launches.argtypes = [C.c_void_p, C.POINTER(C.c_uint32), C.POINTER(C.c_uint32)]
    ddet = ckf.DeviceDetector(det, fld)

    def run(alg, ev):
        tracks = alg.run_device(ddet, ckf.DeviceEvents(ddet, ev)).download()
        lanes, since = (C.c_uint32 * 2)(), (C.c_uint32 * 2)()
        assert lib.ckf_debug_get_launches(alg._h, lanes, since) == 0
        return tracks, list(lanes), list(since)

    want, lanes, since = run(ckf.combinatorial_kalman_filter_algorithm(cfg), small)
    assert lanes == [16, 0] and since[0] == 0
    alg = ckf.combinatorial_kalman_filter_algorithm(cfg)
    assert run(alg, large)[1] == [1, 8]
    got, again, _ = run(alg, small)
    assert again == lanes
    for a, b in zip(_columns(got), _columns(want)):
        assert np.array_equal(a, b)
