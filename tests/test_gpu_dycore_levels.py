"""Level counts and radii whose single-precision reciprocals are not the rounded exact ones:
the dry core's kernels give bit for bit what the array operations give, which multiply by the
rounded exact reciprocal."""
import pytest
import torch

from test_gpu_dycore_kernels import reference, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,radius", [(7, 6.371e6), (13, 6.371e6), (8, 6.4e6 / 3), (5, 3389.5e3 / 7)])
def test_tendencies(sw, gpu, L, radius):
    m = sw.dycore.DryPrimitiveModel(21, L, nmembers=2, radius=radius)
    st = state(sw, m, L)
    ref, bound, grid_ref = reference(m, st)
    tend, grid = m.tendencies(st, with_grid=True)
    for k in grid_ref:
        assert torch.equal(grid[k], grid_ref[k]), k
    for k in ref:
        assert bool(((tend[k] - ref[k]).abs() <= (bound if k == "div" else 0)).all()), k
    m.close()
