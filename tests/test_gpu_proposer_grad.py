"""The proposer's gradient (FP32 matrix tiles over chunks of samples) against
the float64 oracle at batch sizes around the edges of its chunks: one sample,
a chunk of 32 less and more one, odd remainders, more than 256 chunks' worth.

Tolerance: rounding of FP32 (u = 2^-24 an operation) carried through the
network entry by entry.  A sum of n products and a bias is within (n + 2) u of
the sum of their sizes, an entry's sum over a chunk of c samples and N chunks
within (c + N / 8 + 16) u, the logistic function within 8 u; the errors of the
factors come in by their products' sizes; all of it doubled.  Samples with a
unit whose pre-activation is within its own bound of zero (the unit may switch)
are drawn again.  That a missing chunk or sample is seen within this tolerance is
checked on the CPU."""
import numpy as np
import pytest

import proposer_oracle as po
import pyadg

SIZES = [1, 2, 31, 33, 255, 8191, 8193, 20011]
U = 2.0 ** -24


def _chunk(n):
    return max(32, ((n + 255) // 256 + 7) // 8 * 8)


def _errors(p, x):
    """Activations, and bounds of the FP32 errors of pre-activations and logits."""
    W1, b1, W2, b2, W3, b3 = po.unpack(p)
    z, prob, h1, h2 = po.forward(p, x)
    e1 = (po.F + 2) * U * (np.abs(x) @ np.abs(W1).T + np.abs(b1))
    e2 = (po.H + 2) * U * ((h1 + e1) @ np.abs(W2).T + np.abs(b2)) + e1 @ np.abs(W2).T
    ez = (po.H + 2) * U * ((h2 + e2) @ np.abs(W3) + abs(b3)) + e2 @ np.abs(W3)
    return h1, h2, z, prob, e1, e2, ez


def _case(n):
    """Parameters, samples, labels and weights; the last sample weighs a fiftieth of the batch."""
    r = np.random.default_rng(n)
    F, H = po.F, po.H
    p = np.concatenate([r.normal(0, (2 / F) ** 0.5, H * F), r.normal(0, 0.1, H), r.normal(0, (2 / H) ** 0.5, H * H),
                        r.normal(0, 0.1, H), r.normal(0, (1 / H) ** 0.5, H), [0.1]]).astype(np.float32)
    W1, b1, W2, b2, _, _ = po.unpack(p)
    x = r.normal(0, 1, (n, F)).astype(np.float32)
    while True:
        h1, _, _, _, e1, e2, _ = _errors(p, x)
        again = (np.abs(x @ W1.T + b1) <= 2 * e1).any(axis=1) | (np.abs(h1 @ W2.T + b2) <= 2 * e2).any(axis=1)
        if not again.any():
            break
        x[again] = r.normal(0, 1, (int(again.sum()), F)).astype(np.float32)
    y = (r.random(n) < 0.3).astype(np.uint8)
    w = r.uniform(0.5, 2.0, n).astype(np.float32)
    w[-1] = max(1.0, n / 50)
    return p, x, y, w


def _tolerance(p, x, y, w):
    n = len(y)
    W1, b1, W2, b2, W3, b3 = po.unpack(p)
    w = w.astype(np.float64) / w.astype(np.float64).sum()
    h1, h2, z, prob, e1, e2, ez = _errors(p, x)
    dz = w * np.abs(prob - y)
    edz = w * (ez / 4 + 8 * U) + 2 * U * dz
    on1, on2 = h1 > 0, h2 > 0
    dh2, edh2 = np.outer(dz, np.abs(W3)) * on2, np.outer(edz + U * dz, np.abs(W3)) * on2
    dh1 = (dh2 @ np.abs(W2)) * on1
    edh1 = ((edh2 + (po.H + 2) * U * dh2) @ np.abs(W2)) * on1
    x = np.abs(x.astype(np.float64))
    c = _chunk(n)
    a = (c + -(-n // c) / 8 + 16) * U

    def entry(f, ef, g, eg):  # sum over samples of products f g
        return a * (f.T @ g) + ef.T @ (g + eg) + f.T @ eg
    one = np.ones((n, 1))
    none = np.zeros((n, 1))
    col = [dz[:, None], edz[:, None]]
    return 2 * np.concatenate([entry(dh1, edh1, x, 0 * x).ravel(), entry(dh1, edh1, one, none).ravel(),
                               entry(dh2, edh2, h1, e1 * on1).ravel(), entry(dh2, edh2, one, none).ravel(),
                               entry(h2, e2 * on2, *col).ravel(), entry(*col, one, none).ravel()]) + 1e-30


def _gradient_without(p, x, y, w, drop):
    """The oracle's gradient with samples left out of the sums but not of the batch's weight."""
    w0 = w.copy()
    w0[drop] = 0.0
    if not w0.any():
        return np.zeros(p.size)
    return po.loss_and_grad(p, x, y, w0)[1] * (w0.astype(np.float64).sum() / w.astype(np.float64).sum())


@pytest.mark.parametrize("n", SIZES)
def test_tolerance_sees_missing_samples(n):
    case = _case(n)
    tol, c = _tolerance(*case), _chunk(n)
    ref = po.loss_and_grad(*case)[1]
    last = (n - 1) // c * c
    for drop in (slice(n - 1, n), slice(last, n), slice(last // 2 // c * c, last // 2 // c * c + c)):
        moved = np.abs(_gradient_without(*case, drop) - ref)
        seen = (moved > tol)[moved > 1e-12 * np.abs(ref)]  # of the entries that these samples have a part in
        assert seen.size > 100 and seen.mean() > 0.5, (drop, seen.size, seen.mean())


@pytest.mark.gpu
@pytest.mark.parametrize("n", SIZES)
def test_gradient_sizes(n):
    print(f"[case] proposer gradient n={n}", flush=True)
    p, x, y, w = _case(n)
    s = pyadg.Solution(2, 1, 2, 3)
    s.set_proposer_params(p)
    g, loss = s.proposer_gradient(x, y, w)
    ref_loss, ref = po.loss_and_grad(p, x, y, w)
    tol = _tolerance(p, x, y, w)
    assert np.all(np.abs(g - ref) <= tol), np.max(np.abs(g - ref) / tol)
    assert abs(loss - ref_loss) <= 1e-5 * max(1.0, abs(ref_loss))
