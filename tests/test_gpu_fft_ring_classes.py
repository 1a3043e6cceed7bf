"""GPU parity of the ring FFT at the edges of its ring classes: the kernels are compiled for rings
of up to 256, 512 and 1024 points, and a plan takes the smallest class that holds its longest ring
and the row tiles of its prime passes.  Octahedral grids of n rings per hemisphere end at
4n + 16 points; full Gaussian grids have rings of 4n, here also four times a prime."""
import pytest
import torch

from sht_cases import oracle, rel
from test_gpu_fft_columns import check
from test_gpu_transform import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n", [("octahedral", 60), ("octahedral", 61), ("octahedral", 124),
                                    ("octahedral", 125), ("full", 61), ("full", 127), ("full", 128),
                                    ("full", 129), ("full", 251)])
def test_class_edges(sw, gpu, kind, n):
    lmax, mmax, K = 18, 17, 5
    o = oracle(kind, n, lmax, mmax)
    grid = (sw.OctahedralGaussianGrid if kind == "octahedral" else sw.FullGaussianGrid)(n)
    S = sw.SpectralTransform(sw.Spectrum(lmax, mmax), grid, nlayers=K)
    check(sw, S, o, K, n)
    S.close()


def test_batch_over_all_classes(sw, gpu):
    lmax, mmax = 18, 17
    plans, ins, outs, want = [], [], [], []
    for n, K in ((24, 5), (60, 3), (96, 6), (125, 4)):
        o, s = oracle("octahedral", n, lmax, mmax), sw.Spectrum(lmax, mmax)
        S = sw.SpectralTransform(s, sw.OctahedralGaussianGrid(n), nlayers=K)
        a = sw.seeded_spectrum(s, K, seed=n)
        plans.append(S)
        ins.append(to_dev(sw, a, s))
        outs.append(sw.Field(torch.empty((K, S.grid.npoints), device="cuda"), S.grid))
        want.append(o.synthesis(a))
    batch = sw.SpectralBatch([(S, c, f) for S, c, f in zip(plans, ins, outs)])
    batch.launch()
    torch.cuda.synchronize()
    for f, w in zip(outs, want):
        assert rel(f.data.cpu().numpy(), w) < 1e-5
