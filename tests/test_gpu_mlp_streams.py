"""Gradients of one network on several streams, or from several threads, at once give what they
give one after another."""
from concurrent.futures import ThreadPoolExecutor

import pytest
import torch

from oracle import mlp_oracle as mo


@pytest.mark.gpu
def test_gradients_overlap(sw, gpu):
    B, n = 16384, 4
    gen = torch.Generator(device="cuda").manual_seed(3)
    x, t = (torch.randn(n, B, 32, device="cuda", generator=gen) for _ in range(2))
    m = sw.mlp.ColumnMLP(mo.init_params(3), max_batch=B, device=gpu)
    alone = [m.gradient(x[i], t[i]) for i in range(n)]
    streams = [torch.cuda.Stream() for _ in range(n)]
    torch.cuda.synchronize()
    got = []
    for _ in range(8):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got.append((i, m.gradient(x[i], t[i])))
    with ThreadPoolExecutor(n) as threads:  # on the default stream
        runs = [threads.submit(lambda i: [m.gradient(x[i], t[i]) for _ in range(16)], i) for i in range(n)]
        got += [(i, r) for i in range(n) for r in runs[i].result()]
    torch.cuda.synchronize()
    for i, (loss, g) in got:
        assert torch.equal(loss, alone[i][0]) and torch.equal(g, alone[i][1]), i
    m.close()


def test_scratch_size(sw):
    """Partial gradients (24 864 parameters and a loss) of at most 256 workgroups, one per 32 rows."""
    f = sw.lib().sht_mlp_scratch_bytes
    one = 4 * (24864 + 1)
    assert [f(B) for B in (-1, 0, 1, 32, 33, 8192, 8193, 16384)] == [0, 0, one, one, 2 * one, 256 * one, 129 * one, 256 * one]
