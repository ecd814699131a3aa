"""Ambiguity resolution at the edges of its kernels' blocks, identifier chunks
and list batches (GPU): blocks of 256 threads up to 131,072 tracks or identifiers,
then of 1,024, up to 512 of them; a track's identifiers eight at a time; a shared
identifier's tracks four at a time.  The kept tracks are the oracle's."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu(gpu_available):
    return gpu_available


def _tracks(seed, n, longest, n_ids, repeat):
    r = np.random.default_rng(seed)
    length = r.integers(1, longest + 1, n)
    off = np.concatenate([[0], np.cumsum(length)]).astype(np.uint32)
    ids = r.integers(0, n_ids, off[-1]).astype(np.uint32)
    if repeat:  # a track's first identifier again at its end: in another chunk for the long ones
        ids[off[1:] - 1] = ids[off[:-1]]
    return off, ids, r.random(n).astype(np.float32)


@pytest.mark.parametrize("n,longest,n_ids,repeat", [
    (1023, 8, 900, False), (1024, 9, 5000, True), (1025, 17, 3000, True), (700, 40, 60, True),
    (3000, 7, 20, False), (524289, 6, 2000000, True),
    (255, 8, 300, False), (256, 8, 300, True), (257, 8, 300, False),
    (131072, 5, 131073, True), (131073, 5, 131072, False)])
def test_blocks_chunks_and_lists(n, longest, n_ids, repeat):
    from traccc_amd import ambiguity as AMB
    off, ids, pv = _tracks(n, n, longest, n_ids, repeat)
    resolver = AMB.greedy_ambiguity_resolution_algorithm()
    kept = resolver(off, ids, pv, n_ids)
    want, removed = oracle.greedy_resolve(off, ids, pv)
    assert np.array_equal(kept, np.nonzero(want)[0])
    assert resolver.last_stats().n_removed == removed
    assert resolver.last_stats().n_accepted == len(kept)
