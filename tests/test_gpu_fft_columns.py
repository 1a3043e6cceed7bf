"""GPU parity of the ring FFT at the edges of its column choices: a pass takes one column per
work item up to 64 butterflies per column and two beyond (11 and 13: two sub-passes), on full
Gaussian grids whose single ring length puts chosen radices on either side, and on octahedral
grids whose ring count is not a multiple of the XCD count (padding blocks)."""
import numpy as np
import pytest
import torch

from sht_cases import oracle, rel
from test_gpu_transform import to_dev

pytestmark = pytest.mark.gpu

# full Gaussian: N = 4 nlat_half = 64 (8 butterflies of 8), 256 and 260 (64 and 65 butterflies of
# 4), 704 and 792 (64 and 72 of 11), 832 and 936 (64 and 72 of 13), 972 (324 of 3), 980 (140 of
# 7), 1000 (200 of 5), 1024 (128 of 8)
FULL = [16, 64, 65, 176, 198, 208, 234, 243, 245, 250, 256]


@pytest.mark.parametrize("n", FULL)
@pytest.mark.parametrize("eights", [0, 1, 2])
def test_full_gaussian_ring_lengths(sw, gpu, n, eights):
    lmax, mmax, K = 13, 12, 5  # a full and a partial column group
    o = oracle("full", n, lmax, mmax)
    S = sw.SpectralTransform(sw.Spectrum(lmax, mmax), sw.FullGaussianGrid(n), nlayers=K)
    S.set_tuning(eights=eights)
    check(sw, S, o, K, n)
    S.close()


@pytest.mark.parametrize("n", [9, 23, 97])
def test_ring_counts_off_the_xcd_count(sw, gpu, n):
    lmax, mmax, K = 22, 21, 7
    o = oracle("octahedral", n, lmax, mmax)
    S = sw.SpectralTransform(sw.Spectrum(lmax, mmax), sw.OctahedralGaussianGrid(n), nlayers=K)
    check(sw, S, o, K, n)
    S.close()


def check(sw, S, o, K, n):
    print(f"{S.grid} K={K}", flush=True)
    a = sw.seeded_spectrum(S.spectrum, K, seed=n)
    f_ref = o.synthesis(a)
    # rows past the last column stay untouched, every point of the others is written
    wide = torch.full((K + 3, S.grid.npoints), float("nan"), device="cuda")
    f = sw.transform_(sw.Field(wide[:K], S.grid), to_dev(sw, a, S.spectrum), S)
    b = sw.transform(sw.Field(torch.from_numpy(f_ref.astype(np.float32)).cuda(), S.grid), S)
    g = sw.Field(torch.zeros((K, S.grid.npoints), device="cuda"), S.grid)
    sw.grid2spec_pullback_(g, to_dev(sw, a, S.spectrum), S)  # the accumulating synthesis
    torch.cuda.synchronize()
    assert rel(f.data.cpu().numpy(), f_ref) < 1e-5
    assert rel(b.data.cpu().numpy(), o.analysis(f_ref)) < 1e-5
    assert rel(g.data.cpu().numpy(), o.grid2spec_pullback(a)) < 1e-5
    assert torch.isnan(wide[K:]).all()
