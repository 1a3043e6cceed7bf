"""MLP gradients at the end of the number range: they are infinite, or NaN, where the same sums in
single precision are, and finite values up to the largest one stay so."""
import numpy as np
import pytest
import torch

from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("row,sign", [(0, 1), (37, -1), (69, 1)])
def test_infinite_target(sw, gpu, row, sign):
    rng = np.random.default_rng(row)
    p = mo.init_params(5)
    x, t = (rng.standard_normal((70, 32)).astype(np.float32) for _ in range(2))
    t[row, 9] = sign * np.inf
    m = sw.mlp.ColumnMLP(p, max_batch=70, device=gpu)
    loss, g = m.gradient(torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda())
    m.close()
    with np.errstate(invalid="ignore"):
        _, ref = mo.loss_and_gradient(p, x, t, rounding=True)
    assert np.isposinf(loss.item())
    g, ref = mo.unpack(g.cpu().numpy().astype(np.float64)), mo.unpack(ref)
    for k in ref:
        assert np.array_equal(np.isposinf(g[k]), np.isposinf(ref[k])), k
        assert np.array_equal(np.isneginf(g[k]), np.isneginf(ref[k])), k
        assert np.array_equal(np.isnan(g[k]), np.isnan(ref[k])), k
        ok = np.isfinite(ref[k])
        assert np.linalg.norm(g[k][ok] - ref[k][ok]) <= 5e-3 * np.linalg.norm(ref[k][ok]), k


def test_largest_finite_gradient(sw, gpu):
    """W3 = 16 at one output, z2 = 10 (derivative 1): dL/dz2 = 3.4e38, which BF16 rounds to
    infinity; the other gradients are products with zeros."""
    n = sw.mlp.nparams()
    W1, b1, W2, b2 = 128 * 32, 128, 128 * 128, 128
    p = np.zeros(n, np.float32)
    o2 = W1 + b1 + W2
    p[o2:o2 + b2] = 10.0
    p[o2 + b2:o2 + b2 + 128] = 16.0  # output 0
    m = sw.mlp.ColumnMLP(p, max_batch=1, device=gpu)
    x, t = torch.zeros(1, 32), torch.full((1, 32), 0.0)
    t[0, 0] = -3.4e38
    _, g = m.gradient(x.cuda(), t.cuda())
    m.close()
    g = g.cpu().numpy().astype(np.float64)
    assert np.all(np.abs(g[o2:o2 + b2] / 3.4e38 - 1) < 2.0 ** -21)
    assert not g[:o2].any()
    assert np.all(np.abs(g[o2 + b2:o2 + b2 + 128] / (10 * 3.4e38 / 16) - 1) < 2.0 ** -21)
