"""The guess network's gradient where its workgroups' last pass is not full."""

import numpy as np
import pytest

from oracle import mlp
from ccq_amd import guess as GS

pytestmark = pytest.mark.gpu


def _samples(n, seed):
    r = np.random.default_rng(seed)
    x = np.stack([np.abs(r.normal(0, 1, n)), r.uniform(-3.0, -0.8, n), r.uniform(0.4, 5.0, n), r.normal(0, 0.05, n),
                  r.normal(0, 0.05, n)], 1).astype(np.float32)
    return x, r.normal(1.0, 0.2, n).astype(np.float32), r.normal(0.0, 0.2, n).astype(np.float32)


@pytest.mark.parametrize("n", [1, 17, 31])
def test_infinite_weight_of_a_partial_pass(n):
    """Rows past the batch take no part: a first-layer weight at infinity
    saturates its unit on every sample (no input is zero) and the gradient
    stays finite.  Tolerance: 2^-6, a few BF16 roundings to the other neighbour."""
    print(f"case infinite weight, {n} samples", flush=True)
    X, M, Y = _samples(n, 31)
    p = GS.init_params(_samples(400, 32)[0], seed=33)
    p[mlp.OFF["W1"][0] + 3] = np.inf
    loss, g = GS.grad(X, M, Y, p)
    lw, gw = mlp.loss_grad(p.astype(np.float64), X, M, Y, rounding=True)
    assert np.isfinite(lw) and np.isfinite(gw).all()
    assert abs(loss - lw) <= 2.0 ** -6 * lw
    assert np.abs(g - gw).max() <= 2.0 ** -6 * np.abs(gw).max()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 4095, 4096, 4097, 4113])
def test_each_edge_sample_counts(n):
    """One sample alone has a loss (M = Y = 0 elsewhere): the first and last of the
    batch and the first of its last sixteen, so leaving that sample out, or
    counting it twice, changes loss and gradient by their whole size.  Tolerance
    as above."""
    X, M, Y = _samples(n, 41)
    p = GS.init_params(_samples(400, 42)[0], seed=43)
    for k in sorted({0, n - 1, (n - 1) // 16 * 16}):
        print(f"case edge sample {k} of {n}", flush=True)
        m, y = np.zeros_like(M), np.zeros_like(Y)
        m[k], y[k] = M[k], M[k] + 1.0
        loss, g = GS.grad(X, m, y, p)
        lw, gw = mlp.loss_grad(p.astype(np.float64), X, m, y, rounding=True)
        assert lw > 0 and abs(loss - lw) <= 2.0 ** -6 * lw
        assert np.abs(g - gw).max() <= 2.0 ** -6 * np.abs(gw).max()
