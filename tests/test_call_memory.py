"""Device memory that an algorithm object holds after a call (GPU): the step buffers
are what bounds the events of a call, so their size for a seed has a limit."""
import pytest

from traccc_amd import _ffi as F
from traccc_amd import ckf
from traccc_amd import simulation as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu(gpu_available):
    return gpu_available


def _held(make):
    """Device bytes that what `make` returns holds, cached result blocks left out."""
    import torch
    lib = F.load_library(ckf.LIB)
    torch.cuda.synchronize()
    lib.ckf_release_cached_memory()
    before = torch.cuda.mem_get_info()[0]
    made = make()
    torch.cuda.synchronize()
    lib.ckf_release_cached_memory()
    return before - torch.cuda.mem_get_info()[0], made


# a seed's inputs of a step: the square of the branches; its slots: the cube.  A slot
# takes 376 B (two propagated states of 112 B, a filtered one, two histories of 20 B,
# 12 B more), an input 40 B, a link of the 100 a seed has at first 32 B, its tips 20 B
# each; the rest (tables by events and surfaces) is below 2 %.
@pytest.mark.parametrize("branches", [1, 2, 3])
def test_step_buffers(branches):
    det, fld, gun = S.workload("C2", n_particles=1000, seed=3)
    one = S.generate_event(det, fld, gun)
    ddet = ckf.DeviceDetector(det, fld)
    cfg = S.finding_config_for("C2")
    ckf.combinatorial_kalman_filter_algorithm(cfg).run_device(ddet, ckf.DeviceEvents(ddet, one))
    cfg.max_num_branches_per_surface = branches
    dev = ckf.DeviceEvents(ddet, [one] * 360)

    def call():
        alg = ckf.combinatorial_kalman_filter_algorithm(cfg)
        alg.run_device(ddet, dev)
        return alg

    held, alg = _held(call)
    assert alg.last_stats().n_regrows == 0
    inputs = branches ** 2
    want = 376 * inputs * branches + 40 * inputs + 32 * 100 + 20 * 25 + 8 * one.n_meas / one.n_seeds
    assert held / dev.n_seeds < 1.02 * want


def test_fit_results():
    """A fit's columns: 134 B a track, 267 B a state at most, and at most an eighth and a sixteenth for their blocks."""
    from traccc_amd import fitting as FT
    det, fld, gun = S.workload("C2", n_particles=1000, seed=3)
    one = S.generate_event(det, fld, gun)
    ddet = ckf.DeviceDetector(det, fld)
    cfg = S.finding_config_for("C2")
    dev = ckf.DeviceEvents(ddet, [one] * 360)
    tracks = ckf.combinatorial_kalman_filter_algorithm(cfg).run_device(ddet, dev)
    fitter = FT.kalman_fitting_algorithm(FT.fitting_config(cfg))
    first = fitter.run_device(ddet, dev, tracks)  # the fitter's own buffers
    held, fitted = _held(lambda: fitter.run_device(ddet, dev, tracks))
    n, states = fitted.sizes()
    assert first.sizes() == (n, states) and states > 1500000
    assert held < (134 * n + 267 * states) * 19 / 16 + 14 * (2 << 20)
