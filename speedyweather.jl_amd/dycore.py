"""Minimal dry primitive-equation dynamical core on the MI355X transform engine.

A dynamics-only restatement of the reference's PrimitiveDryModel time step, used to
generate training data for the learned column correction and to run it: no physics, no
orography (NoOrography), dry, sigma coordinates with equally spaced levels, explicit
leapfrog with the Robert-Asselin-Williams filter and implicit hyperdiffusion.

Reference formulation (SpeedyWeather.jl):
  tendency pipeline          SpeedyWeather/src/dynamics/tendencies.jl:119-177
  pressure gradient flux     tendencies.jl:182-213
  vertical integration,
  vertical velocity          tendencies.jl:231-473
  vertical advection         SpeedyWeather/src/dynamics/vertical_advection.jl:23-185 (centred)
  geopotential               SpeedyWeather/src/dynamics/geopotential.jl:42-209
  vorticity / divergence
  flux form                  tendencies.jl:513-768, 897-998, 1123-1212
  mass conservation          SpeedyWeather/src/dynamics/horizontal_diffusion.jl:345 (l = 0 of ln ps)
  hyperdiffusion             horizontal_diffusion.jl:29-250 (power 4, 4 h / 1 h at T32)
  leapfrog + RAW filter      SpeedyWeather/src/time_stepping/steppers/leapfrog.jl:175-286
  sigma levels               SpeedyWeather/src/dynamics/vertical_coordinates.jl:83-87
  constants                  SpeedyWeather/src/dynamics/atmosphere.jl:14-74, planet.jl:4-28
  spectral truncation        LowerTriangularArrays/src/truncation.jl:67-89
The reference integrates the linear gravity-wave terms semi-implicitly
(implicit/implicit_primitive_equations.jl:69-352); this restatement is fully explicit with
a correspondingly shorter time step.

Spectral operators follow SpeedyTransforms/src/spectral_gradients.jl:30-125 (curl and
divergence of a vector whose grid components carry a 1/cos(lat) factor), :386-421
(Laplacian) and :483-527 (gradient), with the factors of gradient_arrays.jl:4-145.
Every spectral <-> grid transform runs on the engine, and so do the tendencies and the time
step (sht_dry_tendencies, sht_dry_leapfrog: one kernel per pass over the data between the
transforms); setup and initial states use torch.
"""
from __future__ import annotations

import ctypes as C
import math
import operator

import numpy as np
import torch

from ._lib import DimensionMismatch, ShtDryModel, check, lib
from .grids import OctahedralGaussianGrid, get_nlat_half
from .spectrum import LowerTriangularArray, Spectrum
from .transform import SpectralTransform, UV_from_vordiv_, transform_

RADIUS = 6.371e6        # m
ROTATION = 7.29e-5      # 1/s
GRAVITY = 9.81          # m/s^2
R_DRY = 287.05          # J/kg/K
CP = 1004.0             # J/kg/K
KAPPA = R_DRY / CP


_version, _requires_grad = operator.attrgetter("_version"), operator.attrgetter("requires_grad")
_TENSORS = (torch.Tensor, torch.nn.Parameter)


def _plain(t, shape) -> bool:
    """t is memory: a tensor of that shape with nothing to differentiate (nor to map through:
    _untraced)."""
    return type(t) in _TENSORS and t.shape == shape and not (t.requires_grad and torch.is_grad_enabled())


def _real(t, shape) -> bool:
    return _plain(t, shape) and not t.is_complex()


def _untraced() -> bool:
    """No transform of functions (vmap, jvp, ...) and no forward differentiation is on."""
    return torch._C._functorch.peek_interpreter_stack() is None and torch.autograd.forward_ad._current_level < 0


def _eps(l, m):
    l = np.asarray(l, np.float64)
    m = np.asarray(m, np.float64)
    with np.errstate(invalid="ignore", divide="ignore"):
        e = np.sqrt(np.maximum(l * l - m * m, 0.0) / (4.0 * l * l - 1.0))
    return np.where(l > 0, e, 0.0)


class SpectralOps:
    """Linear operators on packed coefficients, tensors (K, nharm) complex64."""

    def __init__(self, spectrum: Spectrum, device):
        l, m = spectrum.degrees_orders()  # 0-based
        last = l == spectrum.lmax - 1
        n = spectrum.nharm
        idx = np.arange(n)
        self.prev = torch.as_tensor(np.maximum(idx - 1, 0), device=device)
        self.next = torch.as_tensor(np.minimum(idx + 1, n - 1), device=device)
        e_l, e_l1 = _eps(l, m), _eps(l + 1, m)
        f = lambda a: torch.as_tensor(np.asarray(a, np.float32), device=device)
        # cos(lat) d/dlat of a scalar: -(l-1) eps_l q_{l-1} + (l+2) eps_{l+1} q_{l+1}
        self.dy1 = f(-(l - 1) * e_l)
        self.dy2 = f(np.where(last, 0.0, (l + 2) * e_l1))
        # divergence / curl of (u, v) / cos(lat): (l+1) eps_l and l eps_{l+1}, last row 0
        self.vd1 = f(np.where(last, 0.0, (l + 1) * e_l))
        self.vd2 = f(np.where(last, 0.0, l * e_l1))
        self.m = f(m)
        self.keep = f(np.where(last, 0.0, 1.0))
        self.eig = f(-l * (l + 1.0))
        self.l = torch.as_tensor(l, device=device)

    def dlambda(self, q):
        """d/dlon: i m q."""
        return torch.complex(-self.m * q.imag, self.m * q.real)

    def coslat_dlat(self, q):
        return self.dy1 * q[:, self.prev] + self.dy2 * q[:, self.next]

    def divergence(self, u, v):
        """div of the vector whose grid components, times 1/cos(lat), have coefficients u, v."""
        return (self.dlambda(u) - self.vd1 * v[:, self.prev] + self.vd2 * v[:, self.next]) * self.keep

    def curl(self, u, v):
        return (self.dlambda(v) + self.vd1 * u[:, self.prev] - self.vd2 * u[:, self.next]) * self.keep

    def laplace(self, q):
        return self.eig * q


def truncate(x: torch.Tensor, src: Spectrum, dst: Spectrum) -> torch.Tensor:
    """Coefficients of the smaller spectrum dst copied from src (truncation.jl:67-89)."""
    ls, ms = dst.degrees_orders()
    idx = torch.as_tensor([src.offset(int(m)) + int(l) - int(m) for l, m in zip(ls, ms)], device=x.device)
    return x[:, idx].contiguous()


def grid_latitudes(grid) -> np.ndarray:
    """Latitude (radians) of every grid point, rings north to south."""
    nlat = 2 * grid.nlat_half
    x = np.zeros(nlat)
    w = np.zeros(nlat)
    lib().sht_gauss_legendre(nlat, x.ctypes.data_as(C.c_void_p), w.ctypes.data_as(C.c_void_p))
    lat_ring = np.arcsin(x[::-1])  # ascending nodes -> north to south
    return np.repeat(lat_ring, grid.nlons)


class DryPrimitiveModel:
    """Dry primitive equations at spectral truncation `trunc` (0-based, e.g. 31 or 127) on
    the octahedral Gaussian grid with quadratic dealiasing, `nlayers` sigma levels, for
    `nmembers` independent states side by side (columns of every transform).

    A subclass may override `tendencies`, `uv`, `synth`, `analyse` and `_diffuse`, and the
    tables (sigma levels, G, f, nu, ops, ...) may be replaced or written to: the step follows
    them, as array operations instead of the library's kernels where these have the original
    built in."""

    @torch.inference_mode(False)  # its tables count writes, whatever mode it is built in
    def __init__(self, trunc: int, nlayers: int = 8, nmembers: int = 1, dt: float | None = None,
                 precision: str = "fp32", device="cuda:0", radius: float = RADIUS):
        self.device = torch.device(device)
        self.trunc, self.L, self.E = trunc, nlayers, nmembers
        self.spectrum = Spectrum(trunc + 2, trunc + 1)  # one more degree for the vector path
        self.grid = OctahedralGaussianGrid(get_nlat_half(trunc + 1))
        self.a = radius
        L, E = nlayers, nmembers
        # columns of a tendency's transforms: 5 L + 3 fields to the grid, 6 L + 1 back
        self.S = SpectralTransform(self.spectrum, self.grid, nlayers=E * max(6 * L + 1, 5 * L + 3), precision=precision,
                                   device=self.device.index or 0)
        self.ops = SpectralOps(self.spectrum, self.device)
        lat = grid_latitudes(self.grid)
        self.coslat = torch.as_tensor(np.cos(lat), dtype=torch.float32, device=self.device)
        self.coslat_inv = 1.0 / self.coslat
        self.f = torch.as_tensor(2 * ROTATION * np.sin(lat), dtype=torch.float32, device=self.device)
        self.lat = lat
        # sigma: half levels k/L, full levels (k - 1/2)/L, top to bottom
        sh = np.arange(L + 1) / L
        sf = (np.arange(L) + 0.5) / L
        self.dsigma = 1.0 / L
        self.sigma_half = torch.as_tensor(sh, dtype=torch.float32, device=self.device)
        self.sigma_full = torch.as_tensor(sf, dtype=torch.float32, device=self.device)
        # hydrostatic geopotential, linear in T: Phi_k = sum_j G[k, j] T_j (no orography)
        G = np.zeros((L, L))
        for k in range(L):
            G[k, k] = R_DRY * math.log(sh[k + 1] / sf[k])
            for j in range(k + 1, L):
                G[k, j] = R_DRY * math.log(sh[j + 1] / sh[j])
        self.G = torch.as_tensor(G, dtype=torch.float32, device=self.device)
        # time step: explicit leapfrog, gravity-wave limited
        self.dt = float(dt) if dt else 300.0 * 32.0 / (trunc + 1)
        # hyperdiffusion (l(l+1)/(T(T+1)))^4 with 4 h (1 h for divergence) at T32, scaled
        T1 = trunc + 1
        scale = 32.0 / T1
        ll = self.ops.l.to(torch.float64)
        shape = (ll * (ll + 1) / (trunc * (trunc + 1.0))) ** 4
        self.nu = (shape / (4 * 3600.0 * scale)).to(torch.float32)
        self.nu_div = (shape / (3600.0 * scale)).to(torch.float32)
        self.robert, self.williams = 0.1, 0.53
        self.state_prev = None
        self.state = None
        self.nsteps = 0
        self._dev = self.coslat.device
        # what the kernels have built in, to see that it is unchanged: each table and its count
        # of in-place writes
        self._levels = (L, self.dsigma)
        self._built = self._tables()
        self._writes = list(map(_version, self._built))

    # ------------------------------------------------------------------ transforms
    def _lta(self, t):
        return LowerTriangularArray(t.contiguous(), self.spectrum)

    def synth(self, coeffs: torch.Tensor, unscale=False) -> torch.Tensor:
        from .grids import Field
        out = torch.empty((coeffs.shape[0], self.grid.npoints), device=self.device)
        transform_(Field(out, self.grid), self._lta(coeffs), self.S, unscale_coslat=unscale)
        return out

    def analyse(self, field: torch.Tensor) -> torch.Tensor:
        from .grids import Field
        out = torch.empty((field.shape[0], self.spectrum.nharm), dtype=torch.complex64, device=self.device)
        transform_(self._lta(out), Field(field.contiguous(), self.grid), self.S)
        return out

    def uv(self, vor: torch.Tensor, div: torch.Tensor):
        """Spectral u cos(lat), v cos(lat) from vorticity and divergence (radius scaled)."""
        U = torch.empty_like(vor)
        V = torch.empty_like(div)
        UV_from_vordiv_(self._lta(U), self._lta(V), self._lta(vor), self._lta(div), self.S, radius=self.a)
        return U, V

    # ------------------------------------------------------------------ dynamics
    # The equations are written twice: as array operations (_tendencies_arrays, _diffuse, the
    # last part of step), which take whatever torch takes, and as the library's kernels, 6 to 24
    # times faster (8 members and levels: T127 1.2 -> 0.19 ms per step, T31 1.1 -> 0.05), which
    # read raw memory of one form.  The kernels run where the model is as it was built
    # (_kernels) and the tensors have that form (_real, _columns); both give the same values.
    # A step spends its host time on these checks, so each looks at a thing once.
    def _tables(self) -> tuple:
        return (self.sigma_half, self.sigma_full, self.G, *vars(self.ops).values())

    def _kernels(self) -> bool:
        """The library's kernels state this model: nothing that they have built in was replaced
        or written to (sigma levels, geopotential matrix, operators, transforms, methods), and
        the tables that they read hold one real value per grid point."""
        S, grid, tables, E, L = self.S, (self.grid.npoints,), self._tables(), self.E, self.L
        return (_untraced()
                and _methods(type(self)) == _METHODS_AS_BUILT and _METHODS.isdisjoint(vars(self))
                and type(self.ops) is SpectralOps and _operators(SpectralOps) == _OPERATORS_AS_BUILT
                and isinstance(self.dsigma, float) and (L, self.dsigma) == self._levels
                and len(tables) == len(self._built) and all(map(operator.is_, tables, self._built))
                and list(map(_version, tables)) == self._writes
                and not (torch.is_grad_enabled() and any(map(_requires_grad, tables)))
                and type(S) is SpectralTransform and S.device == self._dev.index
                and (S.spectrum is self.spectrum or S.spectrum == self.spectrum)
                and (S.grid is self.grid or S.grid == self.grid)
                and S.nlayers >= E * (6 * L + 1) and (L > 1 or S.nlayers >= 8 * E)
                and isinstance(self.a, (int, float)) and self.a > 0
                and _real(self.f, grid) and _real(self.coslat_inv, grid))

    def _columns(self, st: dict):
        """Device pointers of a state's vor, div, temp (E*L, nharm) and lnps (E, nharm), and the
        tensors that hold them; None where a tensor has another form."""
        E, EL, n = self.E, self.E * self.L, self.spectrum.nharm
        keep, ptr = [], []
        for name, rows in (("vor", EL), ("div", EL), ("temp", EL), ("lnps", E)):
            t = st[name] if name in st else None
            if not _plain(t, (rows, n)) or t.dtype is not torch.complex64 or t.device != self._dev:
                return None
            if not t.is_contiguous() or t.is_conj() or t.is_neg():
                t = t.resolve_conj().resolve_neg().contiguous()
            keep.append(t)
            ptr.append(t.data_ptr())
        return ptr, keep

    def _check_state(self, st: dict):
        """Raises for a state that neither form of the equations takes (the transforms convert
        ln ps from any complex type)."""
        E, EL, n = self.E, self.E * self.L, self.spectrum.nharm
        for name, rows in (("vor", EL), ("div", EL), ("temp", EL), ("lnps", E)):
            t = st[name]
            if t.dtype != torch.complex64 and name != "lnps":
                raise TypeError(f"state {name} has dtype {t.dtype}, the model needs {torch.complex64}")
            if tuple(t.shape) != (rows, n):
                raise DimensionMismatch(f"state {name} is {tuple(t.shape)}, the model needs {(rows, n)}")
            if t.device != self._dev:
                raise ValueError(f"state {name} is on {t.device}, the model on {self._dev}")

    def _split(self, x: torch.Tensor) -> dict:
        """The columns vor, div, temp (E*L each) and lnps (E) of one tensor, each a tensor of
        its own to autograd (no view of the others)."""
        EL = self.E * self.L
        vor, div, temp, lnps = x.unsafe_split_with_sizes((EL, EL, EL, self.E))
        return {"vor": vor, "div": div, "temp": temp, "lnps": lnps}

    def _vector(self, x: torch.Tensor) -> torch.Tensor:
        if x.dtype is torch.float32 and x.device == self._dev and x.is_contiguous() and not x.is_neg():
            return x
        return x.to(device=self._dev, dtype=torch.float32).resolve_neg().contiguous()

    def _model(self):
        """The model's descriptor and the tensors it points to."""
        tables = [self._vector(t) for t in (self.coslat_inv, self.f, self.G)]
        return ShtDryModel(self.L, self.E, self.a, R_DRY, KAPPA, *(t.data_ptr() for t in tables)), tables

    def _work(self, with_grid: bool):
        """The arrays between the kernels of a tendency, as pointers to spectral columns, grid and
        grid tendencies, and the tensors that hold them: one, or with_grid the grid (as columns)
        on its own, which then stays."""
        E, EL, n, npts = self.E, self.E * self.L, self.spectrum.nharm, self.grid.npoints
        down, up = 5 * EL + (3 if with_grid else 2) * E, 6 * EL + E
        spec, fields, g = 2 * n * max(5 * EL + 3 * E, up), npts * up, npts * down
        spec, fields = (x + -x % 64 for x in (spec, fields))  # 256-byte steps
        work = torch.empty(spec + fields + (0 if with_grid else g), dtype=torch.float32, device=self._dev)
        grid = torch.empty((down, npts), dtype=torch.float32, device=self._dev) if with_grid else None
        p = work.data_ptr()
        return (p, grid.data_ptr() if with_grid else p + 4 * (spec + fields), p + 4 * spec), (work, grid)

    def tendencies(self, st: dict, with_grid: bool = False):
        """Spectral tendencies of vor, div, temp (E*L, nharm) and lnps (E, nharm); with_grid
        also u, v, T (E, L, npoints) and lnps (E, 1, npoints)."""
        L, E = self.L, self.E
        EL, n, dev = E * L, self.spectrum.nharm, self._dev
        kernels = self._kernels()
        columns = self._columns(st) if kernels else None
        if columns is None:
            if kernels:
                self._check_state(st)
            return self._tendencies_arrays(st, with_grid)
        ptr, keep = columns
        model, tables = self._model()
        tend = torch.empty((3 * EL + E, n), dtype=torch.complex64, device=dev)
        work, (held, g) = self._work(with_grid)
        check(lib().sht_dry_tendencies(self.S._plan, C.byref(model), *ptr, tend.data_ptr(), *work,
                                       int(bool(with_grid)), self.S._stream()), "sht_dry_tendencies")
        out = self._split(tend)
        if with_grid:
            u, v, _, T, _, q = g.unsafe_split_with_sizes((EL, EL, 2 * E, EL, 2 * EL, E))
            return out, {"u": u.view(E, L, -1), "v": v.view(E, L, -1), "T": T.view(E, L, -1), "lnps": q.view(E, 1, -1)}
        return out

    def _tendencies_arrays(self, st: dict, with_grid: bool):
        """The same as array operations around the engine's transforms."""
        L, E, a = self.L, self.E, self.a
        ops = self.ops
        EL = E * L
        vor, div, temp, lnps = st["vor"], st["div"], st["temp"], st["lnps"]
        U, V = self.uv(vor, div)
        g1 = self.synth(torch.cat([U, V, ops.dlambda(lnps), ops.coslat_dlat(lnps)]), unscale=True)
        g2 = self.synth(torch.cat([temp, div, vor, lnps]))
        u, v = g1[:EL].view(E, L, -1), g1[EL:2 * EL].view(E, L, -1)
        dqdx, dqdy = (g1[2 * EL:2 * EL + E] / a).view(E, 1, -1), (g1[2 * EL + E:] / a).view(E, 1, -1)
        T, D, Z = (g2[i * EL:(i + 1) * EL].view(E, L, -1) for i in range(3))
        ds, half, full = self.dsigma, self.sigma_half.view(1, -1, 1), self.sigma_full.view(1, -1, 1)
        uq = u * dqdx + v * dqdy                      # (u, v) . grad ln ps
        dsum = ds * (D + uq)                          # layer mass-flux divergence
        csum = torch.cumsum(dsum, dim=1)
        lnps_t = -csum[:, -1:, :]                     # d ln ps / dt
        sdot = torch.zeros((E, L + 1, u.shape[-1]), device=self.device)
        sdot[:, 1:L] = -csum[:, :L - 1] - half[:, 1:L] * lnps_t

        def vadv(X):
            flux = sdot[:, 1:L] * (X[:, 1:] - X[:, :-1])
            out = torch.zeros_like(X)
            out[:, :-1] += flux
            out[:, 1:] += flux
            return out / (2 * ds)
        omp = uq - (csum - 0.5 * dsum) / full         # omega / p on full levels
        absvor, ci = Z + self.f, self.coslat_inv
        Au = absvor * v - vadv(u) - R_DRY * T * dqdx
        Av = -absvor * u - vadv(v) - R_DRY * T * dqdy
        Tt = T * D - vadv(T) + KAPPA * T * omp
        flds = ((Au * ci), (Av * ci), (u * T * ci), (v * T * ci), 0.5 * (u * u + v * v), Tt)
        s = self.analyse(torch.cat([*(x.view(EL, -1) for x in flds), lnps_t.view(E, -1)]))
        Aus, Avs, uTs, vTs, kes, Tts = (s[i * EL:(i + 1) * EL] for i in range(6))
        lnps_ts = s[6 * EL:].clone()
        phi = torch.einsum("kj,ejn->ekn", self.G.to(torch.complex64), temp.view(E, L, -1)).reshape(EL, -1)
        lnps_ts[:, 0] = 0                              # global mass conservation
        # the extra degree only serves the vector path: no prognostic tendency there
        tend = {"vor": ops.curl(Aus, Avs) / a * ops.keep,
                "div": (ops.divergence(Aus, Avs) / a - ops.laplace(phi + kes) / (a * a)) * ops.keep,
                "temp": (-ops.divergence(uTs, vTs) / a + Tts) * ops.keep, "lnps": lnps_ts * ops.keep}
        if with_grid:
            return tend, {"u": u, "v": v, "T": T, "lnps": g2[3 * EL:].view(E, 1, -1)}
        return tend

    # ------------------------------------------------------------------ time stepping
    def _diffuse(self, name, x, dt2):
        nu = self.nu_div if name == "div" else self.nu
        if name == "lnps":
            return x
        return x / (1.0 + dt2 * nu)

    def _step_kernels(self, tend):
        """_columns of the state, of the previous one and of the tendencies (None: none) where
        the time-step kernels state the step; otherwise None."""
        n, now, prev = (self.spectrum.nharm,), self.state, self.state_prev
        if not (_untraced() and type(self)._diffuse is _DIFFUSE and "_diffuse" not in vars(self)
                and isinstance(self.dt, (int, float)) and isinstance(self.robert, (int, float))
                and isinstance(self.williams, (int, float)) and _real(self.nu, n) and _real(self.nu_div, n)
                and len(now) == 4):
            return None
        columns = []
        for st in (now, prev, tend):
            columns.append(None if st is None else self._columns(st))
            if columns[-1] is None and st is not None:
                return None
        return columns

    def step(self, correction=None):
        """One leapfrog step (Euler forward for the first); `correction(model, tend, grid)`
        may add to the spectral tendencies."""
        # without a correction the tendencies go straight into the step, unless a subclass or an
        # instance has its own, or the class was given another
        fused = (correction is None and "tendencies" not in vars(self) and type(self).tendencies is _TENDENCIES
                 and self._kernels())
        columns = self._step_kernels(None) if fused else None
        if columns is None:
            need_grid = correction is not None
            out = self.tendencies(self.state, with_grid=need_grid)
            tend, grid = (out if need_grid else (out, None))
            if correction is not None:
                correction(self, tend, grid)
            columns = None if tend is None else self._step_kernels(tend)
        dt2 = self.dt if self.state_prev is None else 2.0 * self.dt
        w1 = self.robert * self.williams / 2
        w2 = self.robert * (1 - self.williams) / 2
        if columns is not None:
            filtered, new = self._leapfrog(*columns, dt2, w1, w2)
        else:
            base = self.state if self.state_prev is None else self.state_prev
            new = {k: self._diffuse(k, base[k] + dt2 * tend[k], dt2) for k in self.state}
            filtered = {}
            if self.state_prev is not None:
                for k in self.state:
                    d = self.state_prev[k] - 2 * self.state[k] + new[k]
                    filtered[k] = self.state[k] + w1 * d
                    new[k] = new[k] - w2 * d
        for k in filtered:
            self.state[k] = filtered[k]
        self.state_prev, self.state = self.state, new
        self.nsteps += 1

    def _leapfrog(self, now, prev, tend, dt2, w1, w2):
        """The filtered present state and the next one from _columns of the present state, of the
        previous one (None: the first step) and of the tendencies (None: the state's own)."""
        L, E, n, dev = self.L, self.E, self.spectrum.nharm, self._dev
        nu, nu_div = self._vector(self.nu), self._vector(self.nu_div)
        arr = C.c_void_p * 4
        new = torch.empty((3 * E * L + E, n), dtype=torch.complex64, device=dev)
        state, filtered = arr(*now[0]), None
        if prev is not None:
            filtered, prev = torch.empty_like(new), arr(*prev[0])
        out = (None if filtered is None else filtered.data_ptr(), new.data_ptr())
        if tend is None:
            model, tables = self._model()
            work, held = self._work(False)
            check(lib().sht_dry_step(self.S._plan, C.byref(model), state, prev, nu.data_ptr(), nu_div.data_ptr(),
                                     dt2, w1, w2, *out, *work, self.S._stream()), "sht_dry_step")
        else:
            tptr, tkeep = tend
            if any(p != tptr[0] + 8 * n * E * L * i for i, p in enumerate(tptr)):  # a correction put its own tensors there
                tkeep = torch.cat(tkeep)
                tptr = [tkeep.data_ptr()]
            check(lib().sht_dry_leapfrog(self.S._plan, L, E, state, prev, tptr[0], nu.data_ptr(),
                                         nu_div.data_ptr(), dt2, w1, w2, *out, self.S._stream()), "sht_dry_leapfrog")
        return {} if filtered is None else self._split(filtered), self._split(new)

    # ------------------------------------------------------------------ initial conditions
    def jet_state(self, seeds, u0=35.0, lat0=30.0, width=10.0, T0=288.0, lapse=0.0065,
                  noise_K=1.0, noise_trunc=None) -> dict:
        """Zonal jets at +-lat0 (peak u0 m/s, Gaussian in latitude) over an atmosphere at
        rest in the vertical mean, T0 at the surface with a constant lapse rate, plus
        N(0, noise_K) temperature noise per grid point from each member's seed.  With
        noise_trunc, the noise keeps only degrees l <= noise_trunc and is rescaled to
        noise_K root mean square per level."""
        L, E = self.L, self.E
        assert len(seeds) == E
        latd = np.degrees(self.lat)
        ujet = u0 * (np.exp(-((latd - lat0) / width) ** 2) + np.exp(-((latd + lat0) / width) ** 2))
        sig = self.sigma_full.cpu().numpy()
        u = np.tile(ujet, (E * L, 1)).astype(np.float32)
        Tprof = T0 * sig ** (R_DRY * lapse / GRAVITY)
        T = np.empty((E * L, self.grid.npoints), np.float32)
        for e, seed in enumerate(seeds):
            rng = np.random.default_rng(int(seed))
            T[e * L:(e + 1) * L] = Tprof[:, None] + noise_K * rng.standard_normal((L, self.grid.npoints))
        u_t = torch.as_tensor(u, device=self.device)
        us = self.analyse(u_t * self.coslat_inv)
        zero = torch.zeros_like(us)
        vor = self.ops.curl(us, zero) / self.a
        div = torch.zeros_like(vor)
        if noise_trunc is not None:
            Tn = torch.as_tensor(T - Tprof.astype(np.float32)[None, :, None].repeat(E, 0).reshape(E * L, 1),
                                 device=self.device)
            ns = self.analyse(Tn) * (self.ops.l <= noise_trunc).to(torch.float32)
            Tn = self.synth(ns)
            Tn = Tn * (noise_K / Tn.pow(2).mean(dim=1, keepdim=True).sqrt().clamp_min(1e-30))
            T = Tn.cpu().numpy() + Tprof.astype(np.float32)[None, :, None].repeat(E, 0).reshape(E * L, 1)
        temp = self.analyse(torch.as_tensor(T, device=self.device))
        lnps = self.analyse(torch.full((E, self.grid.npoints), math.log(1e5), device=self.device))
        keep = self.ops.keep
        return {"vor": vor * keep, "div": div * keep, "temp": temp * keep, "lnps": lnps * keep}

    def set_state(self, st: dict):
        self.state = {k: v.clone() for k, v in st.items()}
        self.state_prev = None
        self.nsteps = 0

    def run(self, nsteps: int, correction=None):
        for _ in range(nsteps):
            self.step(correction)

    def close(self):
        self.S.close()


# The methods and operators that the kernels stand for.
_TENDENCIES, _DIFFUSE = DryPrimitiveModel.tendencies, DryPrimitiveModel._diffuse
_METHODS = {"_lta", "synth", "analyse", "uv", "_tendencies_arrays"}
_methods = operator.attrgetter(*_METHODS)
_operators = operator.attrgetter("dlambda", "coslat_dlat", "divergence", "curl", "laplace")
_METHODS_AS_BUILT, _OPERATORS_AS_BUILT = _methods(DryPrimitiveModel), _operators(SpectralOps)
