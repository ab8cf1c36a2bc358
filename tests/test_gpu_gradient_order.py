"""The order of summation of the network's gradient, bit for bit: weight
gradients by 256 rows at a time, these partial sums in order; bias gradients
as the sums over the rows equal modulo 256, in order, and a tree over these.
A training run is as reproducible as this order.

M is a power of two, so the factor 2 / M of the loss is exact and partial
sums of fewer rows scale without rounding.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
CHUNK = 256
B1, W2, B2, W3, B3 = 48 * 128, 48 * 128 + 128, 48 * 128 + 128 + 128 * 128, 48 * 128 + 256 + 128 * 128, \
    48 * 128 + 256 + 128 * 128 + 384


def _data(rows, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((rows, 48)).astype(np.float32), rng.standard_normal((rows, 3)).astype(np.float32)


@pytest.mark.parametrize("rows", [512, 2048])
def test_weight_gradient_sums_chunks_in_order(rows):
    from akmc_amd import learn as LN
    X, T = _data(rows, rows)
    m = LN.MLP(max_rows=rows, seed=2)
    _, g = m.loss_grad(X, T)
    s = np.zeros_like(g)
    for c in range(0, rows, CHUNK):
        s += m.loss_grad(X[c:c + CHUNK], T[c:c + CHUNK])[1] * np.float32(CHUNK / rows)
    for lo, hi in ((0, B1), (W2, B2), (W3, B3)):
        assert np.array_equal(g[lo:hi], s[lo:hi])


@pytest.mark.parametrize("rows", [64, 256, 1024])
def test_output_bias_gradient_is_a_tree_over_residues(rows):
    from akmc_amd import learn as LN
    X, T = _data(rows, rows + 1)
    m = LN.MLP(max_rows=rows, seed=2)
    _, g = m.loss_grad(X, T)
    dy = np.float32(2) * (m.forward(X) - T) / np.float32(rows)
    t = np.zeros((CHUNK, 3), np.float32)
    for c in range(0, rows, CHUNK):
        t[:len(dy[c:c + CHUNK])] += dy[c:c + CHUNK]
    o = CHUNK // 2
    while o:
        t[:o] += t[o:2 * o]
        o //= 2
    assert np.array_equal(g[B3:], t[0])
