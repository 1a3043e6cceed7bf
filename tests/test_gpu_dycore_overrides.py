"""What a program may change of the dry model - methods, operators, levels, tables, the form of
states and tendencies - takes effect in its steps, as it does in the equations as array
operations."""
import math

import pytest
import torch

from test_gpu_dycore_kernels import reference, state

pytestmark = pytest.mark.gpu


def same(m, st):
    """The model's tendencies are those of the array operations on its own methods and tables."""
    ref, bound, _ = reference(m, st)
    tend = m.tendencies(st)
    for k in ref:
        assert bool(((tend[k] - ref[k]).abs() <= (bound if k == "div" else 0)).all()), k
    return tend


def half(f):
    return lambda *a, **kw: 0.5 * f(*a, **kw)


def halves(f):
    return lambda *a: tuple(0.5 * x for x in f(*a))


CHANGES = {
    "synth": lambda m: setattr(m, "synth", half(m.synth)),
    "analyse": lambda m: setattr(m, "analyse", half(m.analyse)),
    "uv": lambda m: setattr(m, "uv", halves(m.uv)),
    "operator": lambda m: setattr(m.ops, "curl", half(m.ops.curl)),
    "operator table": lambda m: m.ops.keep.mul_(0.5),
    "levels": lambda m: setattr(m, "sigma_half", m.sigma_half ** 2),
    "full levels in place": lambda m: m.sigma_full.add_(0.01),
    "geopotential": lambda m: m.G.add_(5.0),  # below the diagonal too
    "no rotation": lambda m: setattr(m, "f", 0.0),
    "rotation of rows": lambda m: setattr(m, "f", 2 * m.f[None, None].expand(m.E, m.L, -1)),
}


@pytest.mark.parametrize("change", CHANGES)
def test_changes_take_effect(sw, gpu, change):
    m = sw.dycore.DryPrimitiveModel(21, 3, nmembers=2)
    st = state(sw, m, 2)
    before = same(m, st)
    CHANGES[change](m)
    after = same(m, st)
    assert any(not torch.equal(before[k], after[k]) for k in before)
    m.close()


def test_subclass_methods_and_class_changes(sw, gpu, monkeypatch):
    class Half(sw.dycore.DryPrimitiveModel):
        def synth(self, coeffs, unscale=False):
            return 0.5 * super().synth(coeffs, unscale)
    m = Half(21, 3)
    same(m, state(sw, m, 3))
    m.close()
    m = sw.dycore.DryPrimitiveModel(21, 3)
    monkeypatch.setattr(sw.dycore.SpectralOps, "laplace", lambda self, q: 0.5 * self.eig * q)
    st = state(sw, m, 3)
    ref = reference(m, st)[0]["div"]
    assert float((m.tendencies(st)["div"] - ref).abs().max()) <= 1e-4 * float(ref.abs().max())
    m.close()


def test_layer_thickness(sw, gpu):
    m = sw.dycore.DryPrimitiveModel(21, 3, nmembers=2)
    st = state(sw, m, 4)
    q = m.tendencies(st)["lnps"]
    for ds in (2.0 / 3, torch.full((1, 3, 1), 2.0 / 3, device="cuda")):
        m.dsigma = ds
        assert torch.equal(m.tendencies(st)["lnps"], 2 * q)  # linear in it, a power of two
    m.close()


def steps(sw, change, correction, nsteps=2, **kw):
    m = sw.dycore.DryPrimitiveModel(21, 3, nmembers=2)
    m.set_state(state(sw, m, 6))
    change(m)
    for _ in range(nsteps):
        m.step(correction)
    return m


def test_no_diffusion(sw, gpu):
    """Its coefficient as a number, as one element, as a method."""
    def zero(m):
        m.nu, m.nu_div = torch.zeros_like(m.nu), torch.zeros_like(m.nu_div)

    def number(m):
        m.nu = m.nu_div = 0.0

    def element(m):
        m.nu, m.nu_div = torch.zeros((), device="cuda"), torch.zeros(1, device="cuda")

    def method(m):
        m._diffuse = lambda name, x, dt2: x
    ref = steps(sw, zero, None)
    for change in (number, element, method):
        m = steps(sw, change, None)
        for k in ref.state:
            assert torch.equal(m.state[k], ref.state[k]) and torch.equal(m.state_prev[k], ref.state_prev[k]), (change, k)


def test_tendencies_of_other_shapes_and_types(sw, gpu):
    """A correction may put in whatever broadcasts to the field."""
    def full(m, tend, grid):
        tend["temp"] = torch.zeros_like(tend["temp"])
        tend["lnps"] = torch.zeros_like(tend["lnps"])

    def other(m, tend, grid):
        tend["temp"] = torch.zeros((1, m.spectrum.nharm), device="cuda")  # real
        tend["lnps"] = 0.0
        tend["remark"] = None
    ref, m = steps(sw, lambda m: None, full), steps(sw, lambda m: None, other)
    for k in ref.state:
        assert torch.equal(m.state[k], ref.state[k]), k


def test_state_of_other_types_and_fields(sw, gpu):
    """ln ps in 64 bits stays so, and a field of the program's own is stepped with the others."""
    m = sw.dycore.DryPrimitiveModel(21, 3, nmembers=2)
    st = state(sw, m, 7)
    q = st["lnps"].to(torch.complex128) * (1 + 2.0 ** -40)
    tracer = torch.ones((6, m.spectrum.nharm), dtype=torch.complex64, device="cuda")
    m.set_state({**st, "lnps": q, "tracer": tracer})

    def correction(model, tend, grid):
        tend["tracer"] = torch.zeros_like(tracer)
    t = m.tendencies(m.state)["lnps"]
    m.step(correction)
    assert m.state["lnps"].dtype == torch.complex128
    assert torch.equal(m.state["lnps"], q + m.dt * t)
    assert torch.equal(m.state["tracer"], tracer / (1 + m.dt * m.nu))
    m.close()


def test_gradient_of_a_correction(sw, gpu):
    """A step carries the gradient of what a correction put in."""
    w = torch.ones((), device="cuda", requires_grad=True)

    def correction(model, tend, grid):
        tend["temp"] = tend["temp"] + w
    m = steps(sw, lambda m: None, correction, nsteps=1)
    n = m.spectrum.nharm
    m.state["temp"].real.sum().backward()
    ref = 6 * float((m.dt / (1 + m.dt * m.nu.double())).sum())
    assert math.isclose(float(w.grad), ref, rel_tol=1e-5) and n > 0
    assert not m.state["vor"].requires_grad


def test_missing_tendencies_raise(sw, gpu):
    class Nothing(sw.dycore.DryPrimitiveModel):
        def tendencies(self, st, with_grid=False):
            pass
    m = Nothing(21, 3)
    m.set_state(state(sw, m, 9))
    with pytest.raises(TypeError):
        m.step()
    m.close()

    def drop(model, tend, grid):
        del tend["div"]
    with pytest.raises(KeyError):
        steps(sw, lambda m: None, drop)


def test_unchanged_models_run_on_the_kernels(sw, gpu):
    with torch.inference_mode():
        a = sw.dycore.DryPrimitiveModel(21, 3)
    b = sw.dycore.DryPrimitiveModel(21, 8, nmembers=2, precision="fp16x3")
    c = sw.dycore.DryPrimitiveModel(21, 1, nmembers=2)
    for m in (a, b, c):
        m.set_state(state(sw, m, 8))
        for _ in range(3):
            assert m._kernels() and m._step_kernels(None) is not None
            m.step()
        assert m._kernels() and m._step_kernels(m.tendencies(m.state)) is not None
        m.close()
