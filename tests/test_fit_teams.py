"""The fit's forward pass runs 16, 8 or one lane per candidate by how many there
are (GPU): an event's fit is the same alone (16 lanes), among few others (8) and
among many (1), bit for bit; every word of a result is written, also where the
fit ends early (results reuse the device blocks of earlier ones)."""
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


def _fit(det, fld, events, fcfg=None):
    cfg = S.finding_config_for("C4")
    ddet = ckf.DeviceDetector(det, fld)
    dev = ckf.DeviceEvents(ddet, events)
    cand = ckf.combinatorial_kalman_filter_algorithm(cfg).run_device(ddet, dev)
    fitter = FT.kalman_fitting_algorithm(fcfg or FT.fitting_config(cfg))
    return cand.event_offsets(), fitter.run_device(ddet, dev, cand).download()


def _columns(fitted, tracks):
    a, b = fitted.state_offsets[0], fitted.state_offsets[tracks]
    out = {}
    for f in dataclasses.fields(fitted):
        v = getattr(fitted, f.name)
        if f.name == "state_offsets":
            continue
        per_state = len(v) == len(fitted.state_flags) and len(v) != len(fitted.chi2)
        out[f.name] = v[a:b] if per_state else v[:tracks]
    return out


@pytest.mark.parametrize("events", [2, 12])  # 6,000 and 36,000 candidates
def test_teams_agree(events):
    det, fld, gun = S.workload("C4", n_particles=3000, seed=5)
    evs = S.generate_events(det, fld, [dataclasses.replace(gun, seed=50 + e) for e in range(events)])
    off, one = _fit(det, fld, evs[:1])
    off_all, many = _fit(det, fld, evs)
    assert off[1] == off_all[1] <= 5120 < off_all[2]
    assert (off_all[-1] > 28672) == (events == 12)
    a, b = _columns(one, int(off[1])), _columns(many, int(off[1]))
    for name in a:
        assert np.array_equal(a[name], b[name], equal_nan=a[name].dtype.kind == "f"), name
    _early_ends(many)


def _early_ends(many):
    """Fits that end early are among them, and what they did not reach is zero."""
    failed = many.fit_outcome != FT.OUTCOME_SUCCESS
    assert 0 < failed.sum() < 0.2 * len(failed)
    assert np.all(many.params_vector[failed] == 0) and np.all(many.params_covariance[failed] == 0)
    track_of = np.repeat(np.arange(len(many)), np.diff(many.state_offsets.astype(np.int64)))
    unsmoothed = (many.state_flags & FT.STATE_SMOOTHED) == 0
    first = unsmoothed & failed[track_of] & (np.arange(len(track_of)) == many.state_offsets[track_of])
    assert first.any()
    for column in (many.smoothed_vector, many.smoothed_covariance, many.smoothed_chi2, many.backward_chi2):
        assert np.all(column[first] == 0)
    # a forward pass that stops leaves the states behind it without a record: of a
    # track's filtered records the first ones are there (their variances are
    # positive) and all words of the others are zero
    there = many.filtered_covariance[:, 0, 0] > 0
    assert np.any(~there & failed[track_of]) and not np.any(~there & ~failed[track_of])
    for column in (many.filtered_vector, many.filtered_covariance, many.filtered_chi2):
        assert np.all(column[~there] == 0)
    start = many.state_offsets[track_of].astype(np.int64) == np.arange(len(track_of))
    assert not np.any(there & ~start & ~np.concatenate([[False], there[:-1]]))


@pytest.mark.parametrize("events", [1, 2, 12])  # teams of 16, 8 and one lane
def test_every_word_is_written_over_an_earlier_result(events):
    """A fit into the device blocks of another events' fit, full of its records, is
    the same as one into new blocks."""
    import torch
    lib = F.load_library(ckf.LIB)
    det, fld, gun = S.workload("C4", n_particles=3000, seed=5)
    cfg = S.finding_config_for("C4")
    ddet = ckf.DeviceDetector(det, fld)
    finder = ckf.combinatorial_kalman_filter_algorithm(cfg)
    fitter = FT.kalman_fitting_algorithm(FT.fitting_config(cfg))

    def candidates(seed):
        evs = S.generate_events(det, fld, [dataclasses.replace(gun, seed=seed + e) for e in range(events)])
        dev = ckf.DeviceEvents(ddet, evs)
        return dev, finder.run_device(ddet, dev)

    mine, others = candidates(50), candidates(170)
    fitter.run_device(ddet, *others)  # the fitter's own buffers
    lib.ckf_release_cached_memory()
    want = fitter.run_device(ddet, *mine).download()
    lib.ckf_release_cached_memory()
    old = fitter.run_device(ddet, *others)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    del old  # its blocks go to the cache, nothing of them cleared
    again = fitter.run_device(ddet, *mine)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == before  # and are where this result is
    got = again.download()
    for f in dataclasses.fields(got):
        a, b = getattr(want, f.name), getattr(got, f.name)
        assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f"), f.name
    _early_ends(got)
