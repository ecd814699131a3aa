"""Downloads leave the device in one pass: in one chunk (small results), in chunks,
and in more chunks than are on their way at once, copied by several threads (GPU).
An event's columns are the same whichever way they came, and with only some of the
host arrays given."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from traccc_amd import _ffi as F
from traccc_amd import ckf
from traccc_amd import fitting as FT
from traccc_amd import simulation as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu(gpu_available):
    return gpu_available


def _run(det, fld, events):
    cfg = S.finding_config_for("C4")
    ddet = ckf.DeviceDetector(det, fld)
    dev = ckf.DeviceEvents(ddet, events)
    cand = ckf.combinatorial_kalman_filter_algorithm(cfg).run_device(ddet, dev)
    fitted = FT.kalman_fitting_algorithm(FT.fitting_config(cfg)).run_device(ddet, dev, cand)
    return cand, fitted


# bytes of the fit's download: 10 KB (one chunk), 3 MB (two), 10 MB (five, threads)
@pytest.mark.parametrize("particles", [3, 800, 2900])
def test_one_pass_and_chunks_agree(particles):
    det, fld, gun = S.workload("C4", n_particles=particles, seed=11)
    first = S.generate_events(det, fld, [dataclasses.replace(gun, seed=70)])
    det, fld, gun = S.workload("C4", n_particles=3000, seed=11)
    rest = S.generate_events(det, fld, [dataclasses.replace(gun, seed=71 + e) for e in range(4)])
    cand, fitted = _run(det, fld, first)
    cand_all, fitted_all = _run(det, fld, [*first, *rest])  # 50 MB: the chunks' slots are used again
    one, many = cand.download(), cand_all.download().event(0)
    for f in dataclasses.fields(one):
        assert np.array_equal(getattr(one, f.name), getattr(many, f.name)), f.name
    a, b = fitted.download(), fitted_all.download()
    n, ns = len(a), len(a.state_flags)
    for f in dataclasses.fields(a):
        x, y = getattr(a, f.name), getattr(b, f.name)
        assert np.array_equal(x, y[:len(x)], equal_nan=x.dtype.kind == "f"), f.name
    for cov in (a.params_covariance, a.filtered_covariance, a.smoothed_covariance):
        assert np.array_equal(cov, cov.transpose(0, 2, 1)) and cov.any()
    # some of the arrays only; the identifiers then don't know the outcomes
    part = F.FittedTracks()
    chi2, links, flags = np.zeros(n, np.float32), np.zeros(n, np.uint64), np.zeros(ns, np.uint8)
    part.n_tracks, part.n_states = n, ns
    part.chi2, part.params_surface_link = F.ptr(chi2, C.c_float), F.ptr(links, C.c_uint64)
    part.state_flags = F.ptr(flags, C.c_uint8)
    assert FT._lib().ckf_fitted_download(fitted._h, C.byref(part)) == 0
    good = a.fit_outcome == FT.OUTCOME_SUCCESS
    assert np.array_equal(chi2, a.chi2) and np.array_equal(flags, a.state_flags)
    assert np.array_equal(links[good], a.params_surface_link[good]) and np.all(a.params_surface_link[~good] == 2**64 - 1)


def test_downloads_from_threads():
    """Several threads read their own results at once."""
    import threading
    det, fld, gun = S.workload("C4", n_particles=3000, seed=12)
    evs = S.generate_events(det, fld, [dataclasses.replace(gun, seed=80 + e) for e in range(2)])
    results = [_run(det, fld, evs[:e + 1])[1] for e in (0, 1, 0)]
    want = [r.download() for r in results]
    got = [[] for _ in results]

    def work(i):
        for _ in range(3):
            got[i].append(results[i].download())

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(results))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, w in enumerate(want):
        assert len(got[i]) == 3
        for g in got[i]:
            for f in dataclasses.fields(w):
                assert np.array_equal(getattr(w, f.name), getattr(g, f.name),
                                      equal_nan=getattr(w, f.name).dtype.kind == "f"), f.name
