"""GPU parity of the Legendre kernels where parts of a workgroup's products are skipped: column
counts around half a column group (16 of 32) and around whole groups, last chunks of up to half
and of more than half of their 32 rings, and degree tiles of an order's last block that hold no
degree."""
import pytest

from sht_cases import oracle
from test_gpu_fft_columns import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp32", "fp16x3", "bf16x3"])
@pytest.mark.parametrize("n,trunc", [(16, 31), (33, 32), (48, 63), (49, 66)])
@pytest.mark.parametrize("K", [1, 8, 16, 17, 33, 48, 49])
def test_column_and_chunk_edges(sw, gpu, precision, n, trunc, K):
    lmax, mmax = trunc + 2, trunc + 1
    o = oracle("octahedral", n, lmax, mmax)
    S = sw.SpectralTransform(sw.Spectrum(lmax, mmax), sw.OctahedralGaussianGrid(n), nlayers=K, precision=precision)
    check(sw, S, o, K, n)
    S.close()
