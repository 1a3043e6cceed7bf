"""GPU parity of the MLP kernels at the edges of their row tiles: 16 rows per wave in forward;
in the gradient 32 rows per tile, one tile per workgroup up to 256 workgroups, then two."""
import numpy as np
import pytest
import torch

from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu

# As for the kernels' other tests: a value within one FP32 ulp of a BF16 rounding boundary may
# round the other way than in the oracle's FP64 sums, moving that activation by 2^-8.
TOL_Y = 2e-3
TOL_G = 5e-3
MAX_BATCH = 8225


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


@pytest.fixture(scope="module")
def net(sw, gpu):
    p = mo.init_params(11)
    m = sw.mlp.ColumnMLP(p, max_batch=MAX_BATCH, device=gpu)
    yield m, p
    m.close()


def data(B):
    rng = np.random.default_rng(B)
    return rng.standard_normal((B, 32)).astype(np.float32), rng.standard_normal((B, 32)).astype(np.float32)


@pytest.mark.parametrize("B", [15, 16, 17, 65])
def test_forward_tile_edges(net, B):
    m, p = net
    x, _ = data(B)
    # rows past the last one stay untouched
    out = torch.full((B + 64, 32), float("nan"), device="cuda")
    m.forward(torch.from_numpy(x).cuda(), out=out[:B])
    ref, _ = mo.forward(p, x, rounding=True)
    assert rel(out[:B].cpu().numpy(), ref) < TOL_Y
    assert torch.isnan(out[B:]).all()


@pytest.mark.parametrize("B", [1, 31, 32, 33, 8192, 8193, MAX_BATCH])
def test_gradient_tile_edges(net, B):
    m, p = net
    x, t = data(B)
    loss, g = m.gradient(torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda())
    lref, gref = mo.loss_and_gradient(p, x, t, rounding=True)
    assert abs(float(loss.item()) - lref) <= 1e-4 * lref
    blocks, rblocks = mo.unpack(g.cpu().numpy().astype(np.float64)), mo.unpack(gref)
    for name in blocks:
        assert rel(blocks[name], rblocks[name]) < TOL_G, name
