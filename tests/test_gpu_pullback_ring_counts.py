"""GPU parity of the spectral->grid pullback on octahedral grids whose ring count is not a multiple
of the XCD count: the padding blocks of the FFT analysis launch must leave before they scale and
store rows (they carry no ring whose solid angle could be read)."""
import numpy as np
import pytest
import torch

from sht_cases import oracle, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,trunc", [(9, 8), (23, 25), (30, 34), (97, 63)])
@pytest.mark.parametrize("K", [2, 7])
@pytest.mark.parametrize("unscale", [False, True])
def test_spec2grid_pullback(sw, gpu, n, trunc, K, unscale):
    lmax, mmax = trunc + 2, trunc + 1
    print(f"n={n} K={K} unscale={unscale}", flush=True)
    o = oracle("octahedral", n, lmax, mmax)
    S = sw.SpectralTransform(sw.Spectrum(lmax, mmax), sw.OctahedralGaussianGrid(n), nlayers=K)
    gbar = np.random.default_rng(n + K).standard_normal((K, S.grid.npoints)).astype(np.float32)
    ref = o.spec2grid_pullback(gbar.astype(np.float64), unscale_coslat=unscale)
    for _ in range(2):
        c = sw.LowerTriangularArray.zeros(S.spectrum, K, device="cuda")
        sw.spec2grid_pullback_(c, sw.Field(torch.from_numpy(gbar).cuda(), S.grid), S, unscale_coslat=unscale)
        torch.cuda.synchronize()
        assert rel(c.data.cpu().numpy(), ref) < 1e-5
    S.close()
