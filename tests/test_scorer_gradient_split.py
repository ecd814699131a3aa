"""The gradient's partial sums: blocks of 64 rows, from 20,480 rows on of
256 (up to 256 blocks, then they loop), against the oracle at the edges, with
feature rows that start on 16 bytes and that do not (GPU)."""

import numpy as np
import pytest

from test_scorer import M, _random_data, _random_params, _scorer_with, _torch_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 17, 65, 20479, 20480, 20481, 65536 + 257])
def test_gradient_at_split_edges(n, gpu_available):
    torch, dev = _torch_dev()
    p = _random_params(0.25, np.random.default_rng(7))
    X, y = _random_data(n, np.random.default_rng(n))
    mean, std = X.mean(axis=0), X.std(axis=0) + (n == 1)
    s = _scorer_with(p, mean, std)
    Xd = torch.tensor(X, dtype=torch.float32, device=dev)
    yd = torch.tensor(y, dtype=torch.uint8, device=dev)
    loss, g = s.gradient(Xd, yd, pos_weight=1.5)
    lq, gq = M.loss_and_grad(p.astype(np.float32).astype(np.float64), X.astype(np.float32), y, mean.astype(np.float32),
                             std.astype(np.float32), pos_weight=1.5, bf16_points=True)
    # the bounds of test_scorer's gradient test; 2^-8 is BF16's rounding of one
    # activation, which one row's gradient shows in full
    assert loss == pytest.approx(lq, rel=2e-3 if n > 64 else 2.0**-7)
    assert np.linalg.norm(g - gq) <= (1e-2 if n > 64 else 2.0**-6) * np.linalg.norm(gq)
    again = s.gradient(Xd, yd, pos_weight=1.5)
    assert again[0] == loss and np.array_equal(again[1], g)
    # the same rows one word further on: read in words, not pieces
    flat = torch.empty(n * M.N_IN + 1, dtype=torch.float32, device=dev)
    flat[1:] = Xd.reshape(-1)
    odd = s.gradient(flat[1:].view(n, M.N_IN), yd, pos_weight=1.5)
    assert odd[0] == loss and np.array_equal(odd[1], g)


@pytest.mark.parametrize("batch", [4096, 20480])
def test_training_ragged_last_batch(batch, gpu_available):
    """A last batch of few rows takes fewer partial sums than the launch has blocks."""
    torch, dev = _torch_dev()
    from traccc_amd import scorer
    n = 2 * batch + 70
    X, y = _random_data(n, np.random.default_rng(n))
    Xd = torch.tensor(X, dtype=torch.float32, device=dev)
    yd = torch.tensor(y, dtype=torch.uint8, device=dev)
    out = []
    for _ in range(2):
        s = scorer.Scorer(seed=3)
        s.fit_normalisation(Xd)
        st = s.train(Xd, yd, scorer.train_config(epochs=2, batch=batch, learning_rate=3e-3))
        assert st.steps == 6 and np.isfinite(st.last_loss) and st.last_loss < st.first_loss
        out.append(s.params()[0])
    assert np.array_equal(out[0], out[1]) and np.all(np.isfinite(out[0]))
