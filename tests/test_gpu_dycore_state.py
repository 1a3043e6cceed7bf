"""What a step does with the tensors and dictionaries that a program holds of the dry model."""
import pytest
import torch

from test_gpu_dycore_kernels import state

pytestmark = pytest.mark.gpu


def test_tendencies_are_changed_in_place_one_by_one(sw, gpu):
    """A correction may add what carries a gradient to one field in place; the others stay
    without one, and with their own count of writes."""
    w = torch.ones((), device="cuda", requires_grad=True)
    m = sw.dycore.DryPrimitiveModel(21, 3, nmembers=2)
    m.set_state(state(sw, m, 9))

    def correction(model, tend, grid):
        versions = {k: t._version for k, t in tend.items()}
        tend["temp"] += w
        grid["T"] += w
        for k in ("vor", "div", "lnps"):
            assert not tend[k].requires_grad and tend[k]._version == versions[k], k
        assert not grid["u"].requires_grad
    for _ in range(2):
        m.step(correction)
        assert m.state["temp"].requires_grad and not m.state["vor"].requires_grad
        m.state["temp"] = m.state["temp"].detach()
        m.state["vor"] *= 1.0 + 0j
    m.close()


def test_a_held_state_becomes_the_filtered_one(sw, gpu):
    """The filter writes the present state's dictionary, which then is the previous one."""
    m = sw.dycore.DryPrimitiveModel(21, 8)
    m.set_state(state(sw, m, 10))
    m.step()
    held, before = m.state, dict(m.state)
    m.step()
    assert m.state_prev is held
    assert not torch.equal(held["vor"], before["vor"])
    m.close()
