"""The dry core's tendency and time-step kernels against the same equations written as array
operations on the engine's transforms: the unrolled 8-level grid kernel and the one for any
number of levels, one and several members, the grid outputs, and the leapfrog step with its
filter.  The kernels keep the array operations' rounding, so everything but the geopotential
sum (a matrix product there) is bitwise the same."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def reference(m, st):
    """Tendencies and grid fields in FP32 array operations, and a bound on the rounding of the
    divergence tendency's geopotential sum."""
    E, L, a, ops = m.E, m.L, m.a, m.ops
    EL, R, kappa = E * L, 287.05, 287.05 / 1004.0
    U, V = m.uv(st["vor"], st["div"])
    g1 = m.synth(torch.cat([U, V, ops.dlambda(st["lnps"]), ops.coslat_dlat(st["lnps"])]), unscale=True)
    g2 = m.synth(torch.cat([st["temp"], st["div"], st["vor"], st["lnps"]]))
    u, v = g1[:EL].view(E, L, -1), g1[EL:2 * EL].view(E, L, -1)
    qx, qy = (g1[2 * EL:2 * EL + E] / a).view(E, 1, -1), (g1[2 * EL + E:] / a).view(E, 1, -1)
    T, D, Z = (g2[i * EL:(i + 1) * EL].view(E, L, -1) for i in range(3))
    ds = 1.0 / L
    uq = u * qx + v * qy
    dsum = ds * (D + uq)
    csum = torch.cumsum(dsum, dim=1)
    lt = -csum[:, -1:]
    sh, sf = m.sigma_half.view(1, -1, 1), m.sigma_full.view(1, -1, 1)
    sdot = torch.zeros((E, L + 1, u.shape[-1]), device=u.device)
    sdot[:, 1:L] = -csum[:, :L - 1] - sh[:, 1:L] * lt

    def vadv(X):
        dX = X[:, 1:] - X[:, :-1]
        out = torch.zeros_like(X)
        out[:, :-1] += sdot[:, 1:L] * dX
        out[:, 1:] += sdot[:, 1:L] * dX
        return out / (2 * ds)
    omp = uq - (csum - 0.5 * dsum) / sf
    absvor = Z + m.f
    Au = absvor * v - vadv(u) - R * T * qx
    Av = -absvor * u - vadv(v) - R * T * qy
    Tt = T * D - vadv(T) + kappa * T * omp
    ci = m.coslat_inv
    s = m.analyse(torch.cat([(Au * ci).view(EL, -1), (Av * ci).view(EL, -1), (u * T * ci).view(EL, -1),
                             (v * T * ci).view(EL, -1), (0.5 * (u * u + v * v)).view(EL, -1), Tt.view(EL, -1),
                             lt.view(E, -1)]))
    Aus, Avs, uTs, vTs, kes, Tts = (s[i * EL:(i + 1) * EL] for i in range(6))
    lts = s[6 * EL:].clone()
    lts[:, 0] = 0
    temp = st["temp"].view(E, L, -1)
    phi = torch.einsum("kj,ejn->ekn", m.G.to(torch.complex64), temp).reshape(EL, -1)
    tend = {"vor": ops.curl(Aus, Avs) / a * ops.keep,
            "div": (ops.divergence(Aus, Avs) / a - ops.laplace(phi + kes) / (a * a)) * ops.keep,
            "temp": (-ops.divergence(uTs, vTs) / a + Tts) * ops.keep, "lnps": lts * ops.keep}
    # L-term FP32 sums in either order, then a few roundings of the terms and the result
    terms = torch.einsum("kj,ejn->ekn", m.G.abs(), temp.abs()).reshape(EL, -1) + kes.abs()
    bound = 2 * (L + 4) * 2.0 ** -24 * terms * ops.eig.abs() / (a * a) + 2.0 ** -22 * tend["div"].abs()
    grid = {"u": u, "v": v, "T": T, "lnps": g2[3 * EL:].view(E, 1, -1)}
    return tend, bound, grid


def state(sw, m, seed):
    a = sw.seeded_spectrum(m.spectrum, 3 * m.E * m.L + m.E, seed)
    ls, _ = m.spectrum.degrees_orders()
    a *= (ls < m.spectrum.lmax - 1) & (ls > 0)
    EL, norm = m.E * m.L, 2 * math.sqrt(math.pi)
    st = {"vor": 5e-5 * a[:EL], "div": 2e-6 * a[EL:2 * EL], "temp": 2.0 * a[2 * EL:3 * EL], "lnps": 2e-3 * a[3 * EL:]}
    st["temp"][:, 0] = 260.0 * norm
    st["lnps"][:, 0] = math.log(1e5) * norm
    return {k: torch.from_numpy(v).to(torch.complex64).cuda() for k, v in st.items()}


@pytest.mark.parametrize("L,E,trunc", [(8, 2, 21), (8, 1, 31), (3, 3, 21), (1, 2, 30)])
def test_tendencies_and_step(sw, gpu, L, E, trunc):
    m = sw.dycore.DryPrimitiveModel(trunc, L, nmembers=E)
    st = state(sw, m, trunc + L)
    host = {k: v.cpu().numpy() for k, v in st.items()}
    ref, bound, grid_ref = reference(m, st)
    tend, grid = m.tendencies(st, with_grid=True)
    plain = m.tendencies(st)
    for k in ref:
        assert torch.equal(tend[k], plain[k]), k
        if k != "div":
            assert torch.equal(tend[k], ref[k]), k
    assert bool(((tend["div"] - ref["div"]).abs() <= bound).all())
    for k in grid_ref:
        assert torch.equal(grid[k], grid_ref[k]), k
    # time steps: Euler, then leapfrog with the filter, from the engine's own tendencies
    m.set_state(st)
    m.step()
    shape = (m.ops.l.cpu().numpy() * (m.ops.l.cpu().numpy() + 1) / (trunc * (trunc + 1.0))) ** 4 * (trunc + 1) / 32.0
    nu = {"vor": shape / 14400, "temp": shape / 14400, "div": shape / 3600, "lnps": 0 * shape}
    t0 = {k: v.cpu().numpy().astype(np.complex128) for k, v in plain.items()}
    first = {k: (host[k] + m.dt * t0[k]) / (1 + m.dt * nu[k]) for k in host}
    got = {k: v.cpu().numpy().astype(np.complex128) for k, v in m.state.items()}
    for k in host:
        assert np.abs(got[k] - first[k]).max() <= 1e-6 * np.abs(first[k]).max(), k
    t1 = {k: v.cpu().numpy().astype(np.complex128) for k, v in m.tendencies(m.state).items()}
    held = {k: v.clone() for k, v in m.state.items()}
    kept = dict(m.state)
    m.step()
    for k in host:
        new = (host[k] + 2 * m.dt * t1[k]) / (1 + 2 * m.dt * nu[k])
        d = host[k] - 2 * got[k] + new
        # FP32 sums of terms as large as the field
        tol = 1e-6 * np.abs(host[k]).max()
        assert np.abs(m.state_prev[k].cpu().numpy() - (got[k] + 0.1 * 0.53 / 2 * d)).max() <= tol, k
        assert np.abs(m.state[k].cpu().numpy() - (new - 0.1 * 0.47 / 2 * d)).max() <= tol, k
        assert torch.equal(kept[k], held[k]), k  # earlier states stay as they were
    m.close()


def test_bad_states_raise(sw, gpu):
    m = sw.dycore.DryPrimitiveModel(21, 8, nmembers=2)
    st = state(sw, m, 1)
    with pytest.raises(sw.DimensionMismatch):
        m.tendencies({**st, "temp": st["temp"][:-1]})
    with pytest.raises(TypeError):
        m.tendencies({**st, "vor": st["vor"].to(torch.complex128)})
    with pytest.raises(ValueError):
        m.tendencies({**st, "div": st["div"].cpu()})
    m.close()


@pytest.mark.parametrize("L,E,trunc", [(8, 2, 31), (3, 3, 21), (1, 1, 30)])
def test_fused_step_is_the_step_of_the_tendencies(sw, gpu, L, E, trunc):
    """A step without a correction (tendencies applied where they are computed) gives bit for
    bit what a step with a correction that changes nothing gives."""
    m, w = (sw.dycore.DryPrimitiveModel(trunc, L, nmembers=E) for _ in range(2))
    st = state(sw, m, 3 * trunc + L)
    m.set_state(st)
    w.set_state(st)
    for _ in range(3):  # Euler, then two leapfrog steps with the filter
        m.step()
        w.step(correction=lambda model, tend, grid: None)
        for k in st:
            assert torch.equal(m.state[k], w.state[k]), k
            assert torch.equal(m.state_prev[k], w.state_prev[k]), k
    m.close()
    w.close()


def test_own_tendencies_are_used(sw, gpu):
    class Still(sw.dycore.DryPrimitiveModel):
        def tendencies(self, st, with_grid=False):
            return {k: torch.zeros_like(v) for k, v in st.items()}
    m = Still(21, 3, nmembers=1)
    st = state(sw, m, 5)
    m.set_state(st)
    m.step()
    assert torch.equal(m.state["lnps"], st["lnps"])
    m.close()
