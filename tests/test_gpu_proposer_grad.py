"""The proposer's gradient (FP32 matrix tiles over chunks of samples) against
the float64 oracle at batch sizes around the edges of its chunks: one sample,
a chunk of 32 less and more one, odd remainders, more than 256 chunks' worth.

Tolerance: every gradient entry is a sum over samples of products a_b c_b; an
FP32 product of activations from up to 64-term dot products is within
80 * 2^-23 of its size, and so is the sum of the chunk sums, so an entry is
within 2e-5 of sum |a_b c_b| (units of the batch mean)."""
import numpy as np
import pytest

import proposer_oracle as po
import pyadg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 31, 33, 255, 8191, 8193, 20011])
def test_gradient_sizes(n):
    print(f"[case] proposer gradient n={n}", flush=True)
    r = np.random.default_rng(n)
    x = r.normal(0, 1, (n, po.F)).astype(np.float32)
    y = (r.random(n) < 0.3).astype(np.uint8)
    w = r.uniform(0.5, 2.0, n).astype(np.float32)
    s = pyadg.Solution(2, 1, 2, 3)
    s.proposer_init(7)
    p = s.proposer_params().astype(np.float64)
    g, loss = s.proposer_gradient(x, y, w)
    ref_loss, ref = po.loss_and_grad(p, x, y, w)
    W1, b1, W2, b2, W3, b3 = po.unpack(p)
    z, prob, h1, h2 = po.forward(p, x)
    dz = np.abs(w * (prob - y)) / w.sum()
    dh2 = np.outer(dz, np.abs(W3)) * (h2 > 0)
    dh1 = (dh2 @ np.abs(W2)) * (h1 > 0)
    size = np.concatenate([(dh1.T @ np.abs(x)).ravel(), dh1.sum(0), (dh2.T @ h1).ravel(), dh2.sum(0), h2.T @ dz,
                           [dz.sum()]])
    # (a unit whose pre-activation is within rounding of zero may switch: its terms are allowed in full)
    a1, a2 = x @ W1.T + b1, h1 @ W2.T + b2
    edge = (np.abs(a1) < 1e-5).any(axis=1) | (np.abs(a2) < 1e-5).any(axis=1)
    assert edge.mean() < 0.05 or n < 40
    slack = dz[edge].sum() * 50.0
    assert np.all(np.abs(g - ref) <= 2e-5 * size + slack + 1e-9), np.max(np.abs(g - ref) / (size + 1e-12))
    assert abs(loss - ref_loss) <= 1e-5 * max(1.0, abs(ref_loss))
