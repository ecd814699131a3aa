"""Triplet seeding at the sizes where its path changes (GPU): middles whose tops
or triplets fit in LDS, those that do not, 64-lane and 64-top remainders, empty
and rejected spacepoints around the grid's bounds.  Seeds and weights are the
single-precision oracle's, bit for bit."""
import numpy as np
import pytest

import oracle
from traccc_amd import seeding as SD

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu(gpu_available):
    return gpu_available


def _fan(n_bottom, n_middle, n_top, seed=0, spread=2e-3):
    """Straight tracks from the origin, nearly on one line: every bottom and
    every top of a middle belong together."""
    r = np.random.default_rng(seed)
    out = []
    for n, lo, hi in ((n_bottom, 50.0, 60.0), (n_middle, 100.0, 101.0), (n_top, 140.0, 155.0)):
        rad = r.uniform(lo, hi, n)
        phi = 0.3 + spread * r.standard_normal(n) / rad
        out.append(np.stack([rad * np.cos(phi), rad * np.sin(phi), 0.4 * rad + spread * r.standard_normal(n)], 1))
    xyz = np.concatenate(out).astype(np.float32)
    return xyz[r.permutation(len(xyz))]


def _same(xyz, **kw):
    finder = SD.seedfinder_config(bFieldInZ=2.0 * SD.TESLA, **kw)
    grid, filt = SD.spacepoint_grid_config(finder), SD.seedfilter_config()
    got = SD.seeding_algorithm(finder, grid, filt)(xyz)
    b, m, t, w, _ = oracle.seeding(finder, grid, filt, xyz)
    assert np.array_equal(got.bottom, b) and np.array_equal(got.middle, m) and np.array_equal(got.top, t)
    assert np.array_equal(got.weight.view(np.uint32), w.view(np.uint32))
    return len(got)


@pytest.mark.parametrize("bottoms,middles,tops", [(1, 1, 1), (64, 3, 1), (65, 2, 4), (3, 2, 64), (3, 2, 65),
                                                 (16, 1, 16), (17, 2, 16), (2, 1, 256), (2, 1, 257), (300, 2, 300)])
def test_middles_of_every_size(bottoms, middles, tops):
    assert _same(_fan(bottoms, middles, tops)) >= 1


@pytest.mark.parametrize("bottoms,middles,tops", [
    (3, 40, 300), (64, 9, 300), (65, 9, 300), (300, 9, 65),  # counted with lanes on tops or on bottoms
    (3, 40, 200), (16, 5, 17), (130, 5, 3), (70, 5, 256)])   # more triplets than fit: the first bottoms, or later ones
def test_middles_that_do_not_fit(bottoms, middles, tops):
    assert _same(_fan(bottoms, middles, tops)) >= 1
    assert _same(_fan(bottoms, middles, tops, spread=2.0)) >= 1


def test_small_and_large_middles_together():
    """Some middles through LDS, some through HBM, one run: the seeds keep the
    middles' order."""
    r = np.random.default_rng(4)
    turn = 1.2
    c, s = np.cos(turn), np.sin(turn)
    few = _fan(5, 4, 6, seed=2) @ np.array([[c, s, 0], [-s, c, 0], [0, 0, 1]], np.float32)
    far = _fan(40, 3, 40, seed=3)
    xyz = np.concatenate([few, far])[r.permutation(len(few) + len(far))].astype(np.float32)
    assert _same(xyz) > 5
    assert _same(xyz, maxSeedsPerSpM=2) > 5


def test_rejected_spacepoints():
    xyz = _fan(10, 5, 10)
    outside = xyz.copy()
    outside[:, 2] += 5000.0
    assert _same(np.concatenate([outside, xyz, outside])) >= 1
    assert _same(outside) == 0
    assert _same(xyz[:1]) == 0
    assert _same(np.zeros((0, 3), np.float32)) == 0


def test_parameters_of_more_seeds_than_a_pinned_block_holds():
    """Past 32 MiB of indices and spacepoints the arrays are copied one by one: the
    parameters are those of the same seeds in smaller calls."""
    import ctypes as C
    from traccc_amd import simulation as S
    lib = SD._lib()
    r = np.random.default_rng(8)
    det, fld, gun = S.workload("C2", n_particles=500, seed=3)
    ev = S.generate_event(det, fld, gun)
    meas, cfg, field = ev.measurements_struct(), SD.track_params_estimation_config(), (C.c_float * 3)(0, 0, 2 * SD.TESLA)
    points, seeds = 50000, 1680000
    xyz = r.normal(0, 100, (points, 3)).astype(np.float32)
    index = r.integers(0, ev.n_meas, points).astype(np.uint32)
    b, m, t = (r.integers(0, points, seeds).astype(np.uint32) for _ in range(3))
    w = np.zeros(seeds, np.float32)
    sp = SD.Spacepoints(points, xyz.ctypes.data, None, None, index.ctypes.data)

    def estimate(lo, hi):
        part = [v[lo:hi] for v in (b, m, t, w)]
        struct = SD.Seeds(hi - lo, *[v.ctypes.data for v in part])
        out = np.zeros(hi - lo, np.uint64), np.zeros((hi - lo, 6), np.float32), np.zeros((hi - lo, 36), np.float32)
        assert lib.ckf_estimate_track_params(C.byref(cfg), C.byref(sp), C.byref(struct), C.byref(meas), C.byref(field),
                                             *[v.ctypes.data for v in out]) == 0
        return out

    assert 20 * seeds + 12 * points > 32 << 20 > 20 * (seeds // 2) + 12 * points
    whole = estimate(0, seeds)
    for lo, hi in ((0, seeds // 2), (seeds // 2, seeds)):
        for a, part in zip(whole, estimate(lo, hi)):
            assert np.array_equal(a[lo:hi].view(np.uint32), part.view(np.uint32))
    assert np.isfinite(whole[1]).mean() > 0.9
