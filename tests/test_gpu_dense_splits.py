"""GPU parity of the dense transform's GEMM at the edges of its chunks, splits and column tiles:
contractions shorter than one chunk of 64 rows, one split stored directly, several splits
whose last chunk is partial, and column counts around the 16-column tiles and the 64-column
groups."""
import numpy as np
import pytest
import torch

from sht_cases import oracle, rel
from test_gpu_transform import to_dev

pytestmark = pytest.mark.gpu

# (nlat_half, lmax, mmax): 40 spectral rows (less than a chunk) and 208 points (one split);
# 550 rows (35 groups: two splits of 18) and 1600 points (100 groups: six splits of 17)
SIZES = {"tiny": (4, 6, 5), "T21": (16, 23, 22)}


@pytest.mark.parametrize("name,K", [("tiny", 1), ("tiny", 17), ("tiny", 65), ("T21", 1), ("T21", 16), ("T21", 33),
                                    ("T21", 48), ("T21", 64), ("T21", 65)])
def test_dense_gemm_edges(sw, gpu, name, K):
    n, lmax, mmax = SIZES[name]
    o = oracle("octahedral", n, lmax, mmax)
    M = sw.MatrixSpectralTransform(sw.Spectrum(lmax, mmax), sw.OctahedralGaussianGrid(n), nlayers=K)
    print(f"dense transform {name} K={K}", flush=True)
    a = sw.seeded_spectrum(M.spectrum, K, seed=31)
    f_ref = o.synthesis(a)
    f = sw.transform(to_dev(sw, a, M.spectrum), M)
    fu = sw.transform(to_dev(sw, a, M.spectrum), M, unscale_coslat=True)
    b = sw.transform(sw.Field(torch.from_numpy(f_ref.astype(np.float32)).cuda(), M.grid), M)
    torch.cuda.synchronize()
    # FP32 sums over at most 1600 terms: the transforms' tolerance
    assert rel(f.data.cpu().numpy(), f_ref) < 1e-5
    assert rel(fu.data.cpu().numpy(), o.synthesis(a, unscale_coslat=True)) < 1e-5
    assert rel(b.data.cpu().numpy(), o.analysis(f_ref)) < 1e-5
    M.close()
