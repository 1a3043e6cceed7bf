"""The dry core's one synthesis of columns with and without 1/cos(lat) in every precision:
against the two syntheses that it stands for.  2 E L + 2 E columns are unscaled: 36 and 70 end
inside a group of 32 columns, 64 at its edge."""
import pytest
import torch

from test_gpu_dycore_kernels import reference, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp32", "fp16x3", "bf16x3"])
@pytest.mark.parametrize("L,E,trunc", [(8, 2, 31), (4, 7, 21), (7, 4, 30), (1, 2, 22)])
def test_tendencies(sw, gpu, precision, L, E, trunc):
    m = sw.dycore.DryPrimitiveModel(trunc, L, nmembers=E, precision=precision)
    st = state(sw, m, trunc + L)
    ref, bound, grid_ref = reference(m, st)
    tend, grid = m.tendencies(st, with_grid=True)
    for k in grid_ref:
        assert torch.equal(grid[k], grid_ref[k]), k
    for k in ref:
        assert bool(((tend[k] - ref[k]).abs() <= (bound if k == "div" else 0)).all()), k
    m.set_state(st)
    m.step()
    first = {k: v.clone() for k, v in m.state.items()}
    m.set_state(st)
    m.step(correction=lambda model, tend, grid: None)
    for k in st:
        assert torch.equal(m.state[k], first[k]), k
    m.close()
