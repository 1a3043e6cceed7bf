"""Performance cases: the work that users of the transform engine have it do.

Every case goes through the package's public entry points.  Sizes are those of the
repository's own configurations (T31, T63, T127 and T255 with 8 or 16 layers of up to four
fields, 64 uneven transforms in one batch, the dry model's ensembles, the column network)
plus one odd grid; `draw` spreads truncation, columns, grid, precision and shortcut over the
same ranges.  Truncations are 0-based ("T255": 256 orders and one more degree for vectors).

`exact` restates every case in 64 bits with torch on the CPU, from the definitions alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from __graft_entry__ import load_package

sw = load_package()

RADIUS, ROTATION, R_DRY, CP = 6.371e6, 7.29e-5, 287.05, 1004.0
LAYERS = 8  # sigma levels of the dry model


def listed():
    return [
        # one field of the coarse model on its 8 layers: the smallest call, bound by launches
        {"name": "t31_k8_fp32", "kind": "round_trip", "trunc": 31, "nlat_half": 24, "grid": "octahedral",
         "columns": 8, "precision": "fp32", "shortcut": "linear"},
        # an odd size on the full Gaussian grid: prime ring length factor, ragged columns, the
        # three-term BF16 mode and a quadratic shortcut
        {"name": "t62_full47_k13_bf16x3", "kind": "round_trip", "trunc": 62, "nlat_half": 47, "grid": "full",
         "columns": 13, "precision": "bf16x3", "shortcut": "quadratic"},
        # the transforms of a medium-resolution model step: four fields round trip, u and v
        # from vorticity and divergence
        {"name": "t127_vector_l8_fp32", "kind": "vector", "trunc": 127, "layers": 8, "precision": "fp32"},
        # the headline size, in plain FP32 and in the split mode
        {"name": "t255_k64_fp32", "kind": "round_trip", "trunc": 255, "nlat_half": 192, "grid": "octahedral",
         "columns": 64, "precision": "fp32", "shortcut": "linear"},
        {"name": "t255_k64_fp16x3", "kind": "round_trip", "trunc": 255, "nlat_half": 192, "grid": "octahedral",
         "columns": 64, "precision": "fp16x3", "shortcut": "linear"},
        # a backward pass through both directions, into cotangents zeroed for the pass
        {"name": "t127_pullbacks_k16_fp16x3", "kind": "pullbacks", "trunc": 127, "columns": 16,
         "precision": "fp16x3"},
        # the dense transform, which the reference takes by default at small truncations
        {"name": "t63_dense_k32", "kind": "dense", "trunc": 63, "columns": 32},
        # 64 independent round trips of four truncations as one launch per stage
        {"name": "batch_64_uneven_fp32", "kind": "batch", "items": 64, "choice": 1234},
        # the learned correction on every grid column of eight coarse members
        {"name": "mlp_forward_25344", "kind": "mlp_forward", "rows": 25344},
        # one training batch: loss and parameter gradient
        {"name": "mlp_gradient_4096", "kind": "mlp_gradient", "rows": 4096},
        # one hour of the coarse model for eight members
        {"name": "forecast_t31_e8", "kind": "forecast", "trunc": 31, "members": 8, "steps": 12},
        # a few steps of the fine model's ensemble, as it generates training data
        {"name": "forecast_t127_e8", "kind": "forecast", "trunc": 127, "members": 8, "steps": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["round_trip", "round_trip", "round_trip", "vector", "pullbacks", "dense", "batch",
                       "mlp_forward", "mlp_gradient", "forecast"])
    precision = rng.choice(["fp32", "fp16x3", "bf16x3"])
    trunc = _log_int(rng, 21, 255)
    if kind == "round_trip":
        # the grid that dealiases the truncation, or a ring or two more
        nlat_half = sw.get_nlat_half(trunc + 1) + rng.choice([0, 0, 0, 1, 2])
        grid = rng.choice(["octahedral", "octahedral", "octahedral", "full"])
        # octahedral rings have up to 16 + 4 nlat_half points; both grids stay within 1024
        return {"kind": kind, "trunc": trunc, "nlat_half": nlat_half, "grid": grid, "columns": _log_int(rng, 1, 64),
                "precision": precision,
                "shortcut": rng.choice(["linear", "linear", "linear", "quadratic", "cubic"])}
    if kind == "vector":
        return {"kind": kind, "trunc": trunc, "layers": _log_int(rng, 1, 16), "precision": precision}
    if kind == "pullbacks":
        return {"kind": kind, "trunc": trunc, "columns": _log_int(rng, 1, 64), "precision": precision}
    if kind == "dense":
        return {"kind": kind, "trunc": _log_int(rng, 21, 63), "columns": _log_int(rng, 1, 32)}
    if kind == "batch":
        return {"kind": kind, "items": _log_int(rng, 4, 40), "choice": rng.randrange(1 << 30)}
    if kind == "mlp_forward":
        return {"kind": kind, "rows": _log_int(rng, 3168, 65536)}
    if kind == "mlp_gradient":
        return {"kind": kind, "rows": _log_int(rng, 256, 16384)}
    trunc = _log_int(rng, 21, 85)
    return {"kind": kind, "trunc": trunc, "members": rng.randint(1, 8), "steps": rng.randint(2, 8)}


# ------------------------------------------------------------------------- inputs


def _generator(seed):
    return torch.Generator().manual_seed(int(seed) % (1 << 62))


def _spectra(spectrum, columns, gen):
    """Real and imaginary parts N(0, 1) (l+1)^-1.5, the imaginary part zero at m = 0."""
    ls, ms = spectrum.degrees_orders()
    a = torch.randn(columns, spectrum.nharm, 2, generator=gen, dtype=torch.float64)
    a *= torch.from_numpy((ls + 1.0) ** -1.5)[None, :, None]
    a[:, torch.from_numpy(ms == 0), 1] = 0.0
    return torch.view_as_complex(a).to(torch.complex64)


def _grid(kind, nlat_half):
    return sw.FullGaussianGrid(nlat_half) if kind == "full" else sw.OctahedralGaussianGrid(nlat_half)


def _setup(case):
    """(spectrum, grid, columns) of a transform case."""
    trunc = case["trunc"]
    spectrum = sw.Spectrum(trunc + 2, trunc + 1)
    grid = _grid(case.get("grid", "octahedral"), case.get("nlat_half") or sw.get_nlat_half(trunc + 1))
    return spectrum, grid, case.get("columns") or 4 * case["layers"]


def _batch_items(case):
    """(truncation, columns) of every item: truncations of four classes, 1-16 layers of 1-4 fields."""
    rng = np.random.default_rng(case["choice"])
    return [(int(rng.choice([31, 63, 127, 255])), int(rng.integers(1, 17)) * int(rng.integers(1, 5)))
            for _ in range(case["items"])]


def _mlp_inputs(case, seed):
    """Normalised columns and targets, He-normal weights with small biases."""
    gen = _generator(seed)
    x = torch.randn(case["rows"], 32, generator=gen)
    t = torch.randn(case["rows"], 32, generator=gen)
    parts = []
    for o, i in ((128, 32), (128, 128), (32, 128)):
        parts.append((torch.randn(o, i, generator=gen) * math.sqrt(2.0 / i)).ravel())
        parts.append(0.1 * torch.randn(o, generator=gen))
    return x, t, torch.cat(parts)


def _model_state(case, seed):
    """Vorticity and divergence of a turbulent atmosphere (winds of about 20 m/s), temperature
    with the standard lapse rate and 1 K perturbations, ln ps around 1000 hPa."""
    gen = _generator(seed)
    spectrum, E = sw.Spectrum(case["trunc"] + 2, case["trunc"] + 1), case["members"]
    ls, _ = spectrum.degrees_orders()
    EL = E * LAYERS
    # the extra degree serves vectors only; the largest scales carry no vorticity
    shape = torch.from_numpy(((ls > 0) & (ls < spectrum.lmax - 1)).astype(np.float32))
    vor = _spectra(spectrum, EL, gen) * (5e-5 * shape)
    div = _spectra(spectrum, EL, gen) * (2e-6 * shape)
    temp = _spectra(spectrum, EL, gen) * (2.0 * shape)
    lnps = _spectra(spectrum, E, gen) * (2e-3 * shape)
    sigma = (torch.arange(LAYERS, dtype=torch.float64) + 0.5) / LAYERS
    norm = 2.0 * math.sqrt(math.pi)
    temp[:, 0] = (288.0 * sigma ** (R_DRY * 0.0065 / 9.81) * norm).to(torch.float32).repeat(E)
    lnps[:, 0] = math.log(1e5) * norm
    return {"vor": vor, "div": div, "temp": temp, "lnps": lnps}


def prepare(case, seed):
    kind = case["kind"]
    dev = torch.device("cuda", torch.cuda.current_device())
    st = {"kind": kind}
    if kind in ("round_trip", "vector", "pullbacks", "dense"):
        spectrum, grid, K = _setup(case)
        if kind == "dense":
            S = sw.MatrixSpectralTransform(spectrum, grid, nlayers=K)
        else:
            S = sw.SpectralTransform(spectrum, grid, nlayers=K, LegendreShortcut=case.get("shortcut", "linear"),
                                     precision=case["precision"])
        lta = lambda t: sw.LowerTriangularArray(t, spectrum)
        field = lambda k: sw.Field(torch.empty((k, grid.npoints), device=dev), grid)
        coeffs = lta(_spectra(spectrum, K, _generator(seed)).to(dev))
        st.update(S=S, coeffs=coeffs, field=field(K), back=lta(torch.empty_like(coeffs.data)))
        if kind == "vector":
            L = case["layers"]
            uv = torch.empty((2 * L, spectrum.nharm), dtype=torch.complex64, device=dev)
            st.update(vor=lta(coeffs.data[:L]), div=lta(coeffs.data[L:2 * L]), U=lta(uv[:L]), V=lta(uv[L:]),
                      uv=lta(uv), uv_field=field(2 * L))
        if kind == "pullbacks":
            gen = _generator(seed + 1)
            st["field"].data.copy_(torch.randn(K, grid.npoints, generator=gen))
            st["field_bar"] = field(K)
    elif kind == "batch":
        gen = _generator(seed)
        sizes = _batch_items(case)
        plans = {t: sw.SpectralTransform(sw.Spectrum(t + 2, t + 1), sw.OctahedralGaussianGrid(sw.get_nlat_half(t + 1)),
                                         nlayers=64) for t in sorted({t for t, _ in sizes})}
        # every item's grid and coefficients are slices of two arrays
        points = [K * plans[t].grid.npoints for t, K in sizes]
        modes = [K * plans[t].spectrum.nharm for t, K in sizes]
        grids = torch.empty(sum(points), device=dev)
        spectra = torch.empty(sum(modes), dtype=torch.complex64, device=dev)
        items = []
        for (t, K), g, b in zip(sizes, grids.split(points), spectra.split(modes)):
            S = plans[t]
            c = sw.LowerTriangularArray(_spectra(S.spectrum, K, gen).to(dev), S.spectrum)
            items.append((S, c, sw.LowerTriangularArray(b.view(K, -1), S.spectrum), sw.Field(g.view(K, -1), S.grid)))
        st.update(batch=sw.SpectralBatch(items), grids=grids, spectra=spectra)
    elif kind in ("mlp_forward", "mlp_gradient"):
        x, t, params = _mlp_inputs(case, seed)
        st.update(net=sw.ColumnMLP(params, max_batch=case["rows"], device=dev), x=x.to(dev), t=t.to(dev))
    else:
        model = sw.dycore.DryPrimitiveModel(case["trunc"], LAYERS, nmembers=case["members"], device=dev)
        st.update(model=model, start={k: v.to(dev) for k, v in _model_state(case, seed).items()}, steps=case["steps"])
    return st


# ------------------------------------------------------------------------- one pass


def run(st):
    kind = st["kind"]
    if kind in ("round_trip", "dense"):
        sw.transform_(st["field"], st["coeffs"], st["S"])
        sw.transform_(st["back"], st["field"], st["S"])
        return {"field": st["field"].data, "back": st["back"].data}
    if kind == "vector":
        sw.transform_(st["field"], st["coeffs"], st["S"])
        sw.transform_(st["back"], st["field"], st["S"])
        sw.UV_from_vordiv_(st["U"], st["V"], st["vor"], st["div"], st["S"])
        sw.transform_(st["uv_field"], st["uv"], st["S"], unscale_coslat=True)
        return {"field": st["field"].data, "back": st["back"].data, "uv": st["uv"].data, "uv_field": st["uv_field"].data}
    if kind == "pullbacks":
        st["back"].data.zero_()
        sw.spec2grid_pullback_(st["back"], st["field"], st["S"])
        st["field_bar"].data.zero_()
        sw.grid2spec_pullback_(st["field_bar"], st["coeffs"], st["S"])
        return {"coeffs_bar": st["back"].data, "field_bar": st["field_bar"].data}
    if kind == "batch":
        st["batch"].launch()
        return {"fields": st["grids"], "back": st["spectra"]}
    if kind == "mlp_forward":
        return st["net"].forward(st["x"])
    if kind == "mlp_gradient":
        loss, grad = st["net"].gradient(st["x"], st["t"])
        return {"loss": loss, "grad": grad}
    model = st["model"]
    model.set_state(st["start"])
    model.run(st["steps"])
    return dict(model.state)


# ------------------------------------------------------------------- necessary work


def _transform_work(spectrum, grid, K, shortcut="linear"):
    """Bytes and flops of one direction: spectra, grid and the polynomials once each; the
    order-by-order contraction (real polynomial x complex column) and the ring transforms."""
    nlons = grid.nlons[:grid.nlat_half].astype(np.int64)
    mt = np.minimum(nlons // {"linear": 2, "quadratic": 3, "cubic": 4}[shortcut], spectrum.mmax - 1)
    macs = sum(int(((spectrum.lmax - np.arange(t + 1))).sum()) for t in mt)
    fft = float((5.0 * nlons * np.log2(nlons)).sum()) * K  # both hemispheres, real input
    return (8 * spectrum.nharm * K + 4 * grid.npoints * K + 4 * spectrum.nharm * grid.nlat_half, 4.0 * K * macs + fft)


def work(case):
    kind = case["kind"]
    if kind in ("round_trip", "vector", "pullbacks"):
        spectrum, grid, K = _setup(case)
        b, f = _transform_work(spectrum, grid, K, case.get("shortcut", "linear"))
        b, f = 2 * b, 2 * f
        if kind == "vector":
            L = case["layers"]
            b2, f2 = _transform_work(spectrum, grid, 2 * L)
            b, f = b + b2 + 8 * spectrum.nharm * 4 * L, f + f2 + 20.0 * spectrum.nharm * L
        return {"bytes": b, "flops": f}
    if kind == "dense":
        spectrum, grid, K = _setup(case)
        elements = 2 * spectrum.nharm * grid.npoints
        return {"bytes": 2 * (4 * elements + 8 * spectrum.nharm * K + 4 * grid.npoints * K),
                "flops": 4.0 * elements * K}
    if kind == "batch":
        b = f = 0
        for trunc, K in _batch_items(case):
            w = _transform_work(sw.Spectrum(trunc + 2, trunc + 1),
                                sw.OctahedralGaussianGrid(sw.get_nlat_half(trunc + 1)), K)
            b, f = b + 2 * w[0], f + 2 * w[1]
        return {"bytes": b, "flops": f}
    if kind in ("mlp_forward", "mlp_gradient"):
        n, weights = case["rows"], 128 * 32 + 128 * 128 + 32 * 128
        passes = 3 if kind == "mlp_gradient" else 1  # forward, input gradients, weight gradients
        return {"bytes": 256 * n + 4 * passes * (weights + 288), "flops": 2.0 * passes * n * weights}
    # per step: the state in and out, the grids between the transforms and the grid-point work
    trunc, E = case["trunc"], case["members"]
    spectrum, grid = sw.Spectrum(trunc + 2, trunc + 1), sw.OctahedralGaussianGrid(sw.get_nlat_half(trunc + 1))
    EL = E * LAYERS
    down, up = 5 * EL + 3 * E, 6 * EL + E  # columns to the grid (u, v, T, D, vor, ln ps and its gradient) and back
    bd, fd = _transform_work(spectrum, grid, down)
    bu, fu = _transform_work(spectrum, grid, up)
    point = 4 * grid.npoints * (down + up)
    state = 3 * 8 * spectrum.nharm * (3 * EL + E)
    return {"bytes": case["steps"] * (bd + bu + point + state),
            "flops": case["steps"] * (fd + fu + 100.0 * grid.npoints * EL)}


# ------------------------------------------------- the same in 64 bits, without the package


class _Exact:
    """The transform in 64 bits: Legendre polynomials by the three-term recursion in degree,
    ring sums by FFT, Gaussian latitudes by Newton's method."""

    def __init__(self, lmax, mmax, grid, nlat_half, shortcut="linear"):
        self.lmax, self.mmax, self.n = lmax, mmax, nlat_half
        n = nlat_half
        self.nlon = [4 * n] * n if grid == "full" else [16 + 4 * (j + 1) for j in range(n)]
        self.npoints = 2 * sum(self.nlon)
        self.start = np.concatenate([[0], np.cumsum(self.nlon + self.nlon[::-1])])
        part = {"linear": 2, "quadratic": 3, "cubic": 4}[shortcut]
        self.mt = [min(N // part, mmax - 1) for N in self.nlon]
        x, w = self._gauss(2 * n)
        self.x = x[::-1][:n].copy()  # north to equator
        self.lat = np.arcsin(x[::-1])
        self.coslat = np.sqrt(1.0 - self.x ** 2)
        self.area = w[::-1][:n] * 2 * np.pi / np.array(self.nlon)
        self.offset = [m * lmax - m * (m - 1) // 2 for m in range(mmax)]
        self.nharm = lmax * mmax - mmax * (mmax - 1) // 2
        self.l = np.concatenate([np.arange(m, lmax) for m in range(mmax)])
        self.m = np.concatenate([np.full(lmax - m, m) for m in range(mmax)])
        self.lam = torch.from_numpy(self._polynomials())

    @staticmethod
    def _gauss(N):
        x = -np.cos(np.pi * (np.arange(1, N + 1) - 0.25) / (N + 0.5))
        for _ in range(8):
            p0, p1 = np.ones_like(x), x.copy()
            for k in range(2, N + 1):
                p0, p1 = p1, ((2 * k - 1) * x * p1 - (k - 1) * p0) / k
            dp = N * (x * p1 - p0) / (x * x - 1)
            x = x - p1 / dp
        return x, 2.0 / ((1 - x * x) * dp * dp)

    def _polynomials(self):
        lam = np.zeros((self.nharm, self.n))
        m = np.arange(self.mmax)[:, None].astype(np.float64)
        offset = np.array(self.offset)
        p1 = np.zeros((self.mmax, self.n))
        p2 = np.zeros_like(p1)
        diagonal = np.full(self.n, 1.0 / math.sqrt(4 * math.pi))
        for l in range(self.lmax):
            k = min(l, self.mmax)  # orders below the degree
            p = np.zeros_like(p1)
            mm = m[:k]
            a = np.sqrt((4.0 * l * l - 1) / (l * l - mm * mm))
            b = np.sqrt(np.maximum((l - 1.0) ** 2 - mm * mm, 0.0) / (4.0 * (l - 1.0) ** 2 - 1)) if l > 1 else 0.0
            p[:k] = a * (self.x * p1[:k] - b * p2[:k])
            if l < self.mmax:
                if l:
                    diagonal = -math.sqrt((2 * l + 1) / (2.0 * l)) * self.coslat * diagonal
                p[l] = diagonal
                k += 1
            lam[offset[:k] + l - np.arange(k)] = p[:k]
            p1, p2 = p, p1
        return lam

    def _rings(self, m):
        return [j for j in range(self.n) if self.mt[j] >= m]

    def legendre_synthesis(self, a):
        """(K, nharm) -> per ring northern and southern sums (mt + 1, K)."""
        at = a.T.contiguous()
        K = a.shape[0]
        north = [torch.zeros(t + 1, K, dtype=torch.complex128) for t in self.mt]
        south = [torch.zeros(t + 1, K, dtype=torch.complex128) for t in self.mt]
        for m in range(self.mmax):
            rings = self._rings(m)
            if not rings:
                continue
            rows = slice(self.offset[m], self.offset[m] + self.lmax - m)
            lam, c = self.lam[rows][:, rings], torch.view_as_real(at[rows]).reshape(self.lmax - m, 2 * K)
            even, odd = lam[0::2].T @ c[0::2], lam[1::2].T @ c[1::2]
            gn = torch.view_as_complex((even + odd).reshape(len(rings), K, 2))
            gs = torch.view_as_complex((even - odd).reshape(len(rings), K, 2))
            for i, j in enumerate(rings):
                north[j][m], south[j][m] = gn[i], gs[i]
        return north, south

    def fourier_synthesis(self, north, south):
        K = north[0].shape[1]
        out = torch.empty(K, self.npoints, dtype=torch.float64)
        for j, N in enumerate(self.nlon):
            for rows, ring in ((north[j], j), (south[j], 2 * self.n - 1 - j)):
                z = torch.zeros(N // 2 + 1, K, dtype=torch.complex128)
                z[:self.mt[j] + 1] = rows
                z[0].imag.zero_()
                z[-1].imag.zero_()
                out[:, self.start[ring]:self.start[ring] + N] = torch.fft.irfft(z.T, n=N, norm="forward")
        return out

    def fourier_analysis(self, f):
        north, south = [], []
        for j, N in enumerate(self.nlon):
            for rows, ring in ((north, j), (south, 2 * self.n - 1 - j)):
                rows.append(torch.fft.rfft(f[:, self.start[ring]:self.start[ring] + N]).T[:self.mt[j] + 1].contiguous())
        return north, south

    def legendre_analysis(self, north, south, weights):
        K = north[0].shape[1]
        out = torch.zeros(self.nharm, K, dtype=torch.complex128)
        for m in range(self.mmax):
            rings = self._rings(m)
            if not rings:
                continue
            rows = slice(self.offset[m], self.offset[m] + self.lmax - m)
            w = torch.tensor([weights(j, m) for j in rings], dtype=torch.float64)[:, None]
            fn, fs = torch.stack([north[j][m] for j in rings]), torch.stack([south[j][m] for j in rings])
            lam = self.lam[rows][:, rings]
            res = torch.empty(self.lmax - m, 2 * K, dtype=torch.float64)
            res[0::2] = lam[0::2] @ torch.view_as_real(w * (fn + fs)).reshape(len(rings), 2 * K)
            res[1::2] = lam[1::2] @ torch.view_as_real(w * (fn - fs)).reshape(len(rings), 2 * K)
            out[rows] = torch.view_as_complex(res.reshape(self.lmax - m, K, 2))
        return out.T.contiguous()

    def synthesis(self, a, unscale=False):
        north, south = self.legendre_synthesis(a)
        if unscale:
            for j in range(self.n):
                north[j], south[j] = north[j] / self.coslat[j], south[j] / self.coslat[j]
        return self.fourier_synthesis(north, south)

    def analysis(self, f):
        return self.legendre_analysis(*self.fourier_analysis(f), lambda j, m: self.area[j])

    def _bin(self, j, m):
        """Bins counted twice by a real transform: all but the mean and the Nyquist one."""
        return 1.0 if m == 0 or 2 * m == self.nlon[j] else 2.0

    def synthesis_adjoint(self, f):
        return self.legendre_analysis(*self.fourier_analysis(f), self._bin)

    def analysis_adjoint(self, a):
        north, south = self.legendre_synthesis(a)
        for j in range(self.n):
            w = torch.tensor([self.area[j] / self._bin(j, m) for m in range(self.mt[j] + 1)], dtype=torch.float64)
            north[j], south[j] = north[j] * w[:, None], south[j] * w[:, None]
        return self.fourier_synthesis(north, south)

    # operators on packed coefficients
    def eps(self, shift):
        l, m = self.l + shift, self.m
        return np.where(l > 0, np.sqrt(np.maximum(l * l - m * m, 0.0) / (4.0 * l * l - 1.0)), 0.0)

    @staticmethod
    def shifted(q, d):
        out = torch.zeros_like(q)
        if d > 0:
            out[:, :-1] = q[:, 1:]
        else:
            out[:, 1:] = q[:, :-1]
        return out

    def uv(self, vor, div, radius=1.0):
        l, top = self.l, self.lmax - 1
        with np.errstate(invalid="ignore", divide="ignore"):
            x = np.where(l > 0, -self.m / (l * (l + 1.0)), 0.0) * (l < top)
            lower = np.where(l > 0, self.eps(0) / l, 0.0)
        # degrees above the truncation feed nothing down, the l = m = 0 mode apart
        upper = self.eps(1) / (l + 1.0) * ((l < top - 1) | ((np.arange(self.nharm) == 0) & (l < top)))
        x, lower, upper = (torch.from_numpy(v) for v in (x, lower, upper))
        U = 1j * x * div + upper * self.shifted(vor, 1) - lower * self.shifted(vor, -1)
        V = 1j * x * vor - upper * self.shifted(div, 1) + lower * self.shifted(div, -1)
        return U * radius, V * radius


def _exact_forecast(case, seed):
    """The dry primitive equations as the model's documentation states them: sigma levels,
    centred vertical advection, explicit leapfrog with the Robert-Asselin-Williams filter,
    power-4 hyperdiffusion."""
    trunc, E, L = case["trunc"], case["members"], LAYERS
    T = _Exact(trunc + 2, trunc + 1, "octahedral", sw.get_nlat_half(trunc + 1))
    state = {k: v.to(torch.complex128) for k, v in _model_state(case, seed).items()}
    a, EL, ds, kappa = RADIUS, E * L, 1.0 / L, R_DRY / CP
    real = lambda v: torch.from_numpy(np.asarray(v, np.float64))
    last = T.l == T.lmax - 1
    keep, m, lap = real(np.where(last, 0.0, 1.0)), real(T.m), real(-T.l * (T.l + 1.0))
    e0, e1 = T.eps(0), T.eps(1)
    dy1, dy2 = real(-(T.l - 1) * e0), real(np.where(last, 0.0, (T.l + 2) * e1))
    vd1, vd2 = real(np.where(last, 0.0, (T.l + 1) * e0)), real(np.where(last, 0.0, T.l * e1))
    divergence = lambda u, v: (1j * m * u - vd1 * T.shifted(v, -1) + vd2 * T.shifted(v, 1)) * keep
    curl = lambda u, v: (1j * m * v + vd1 * T.shifted(u, -1) - vd2 * T.shifted(u, 1)) * keep
    lat = np.repeat(T.lat, T.nlon + T.nlon[::-1])
    coslat, f = real(np.cos(lat)), real(2 * ROTATION * np.sin(lat))
    half, full = np.arange(L + 1) / L, (np.arange(L) + 0.5) / L
    G = np.zeros((L, L))
    for k in range(L):
        G[k, k] = R_DRY * math.log(half[k + 1] / full[k])
        G[k, k + 1:] = R_DRY * np.log(half[k + 2:] / half[k + 1:-1])
    G = real(G).to(torch.complex128)
    sf, sh = real(full).view(1, L, 1), real(half).view(1, L + 1, 1)

    def tendencies(st):
        vor, div, temp, lnps = st["vor"], st["div"], st["temp"], st["lnps"]
        U, V = T.uv(vor, div, a)
        dlat = dy1 * T.shifted(lnps, -1) + dy2 * T.shifted(lnps, 1)
        g = T.synthesis(torch.cat([U, V, 1j * m * lnps, dlat]), unscale=True)
        u, v = g[:EL].view(E, L, -1), g[EL:2 * EL].view(E, L, -1)
        qx, qy = g[2 * EL:2 * EL + E].view(E, 1, -1) / a, g[2 * EL + E:].view(E, 1, -1) / a
        g = T.synthesis(torch.cat([temp, div, vor]))
        Tg, D, Z = (g[i * EL:(i + 1) * EL].view(E, L, -1) for i in range(3))
        uq = u * qx + v * qy
        dsum = ds * (D + uq)
        csum = torch.cumsum(dsum, 1)
        lnps_t = -csum[:, -1:]
        sdot = torch.zeros(E, L + 1, u.shape[-1], dtype=torch.float64)
        sdot[:, 1:L] = -csum[:, :L - 1] - sh[:, 1:L] * lnps_t

        def vadv(X):
            flux = sdot[:, 1:L] * (X[:, 1:] - X[:, :-1])
            out = torch.zeros_like(X)
            out[:, :-1] += flux
            out[:, 1:] += flux
            return out / (2 * ds)
        omp = uq - (csum - 0.5 * dsum) / sf
        Au = (Z + f) * v - vadv(u) - R_DRY * Tg * qx
        Av = -(Z + f) * u - vadv(v) - R_DRY * Tg * qy
        Tt = Tg * D - vadv(Tg) + kappa * Tg * omp
        s = T.analysis(torch.cat([(Au / coslat).view(EL, -1), (Av / coslat).view(EL, -1),
                                  (u * Tg / coslat).view(EL, -1), (v * Tg / coslat).view(EL, -1),
                                  (0.5 * (u * u + v * v)).view(EL, -1), Tt.view(EL, -1), lnps_t.view(E, -1)]))
        Aus, Avs, uTs, vTs, kes, Tts = (s[i * EL:(i + 1) * EL] for i in range(6))
        lnps_ts = s[6 * EL:].clone()
        lnps_ts[:, 0] = 0
        phi = (G @ temp.view(E, L, -1)).reshape(EL, -1)
        return {"vor": curl(Aus, Avs) / a * keep,
                "div": (divergence(Aus, Avs) / a - lap * (phi + kes) / (a * a)) * keep,
                "temp": (-divergence(uTs, vTs) / a + Tts) * keep, "lnps": lnps_ts * keep}

    dt, previous = 300.0 * 32.0 / (trunc + 1), None
    shape = (T.l * (T.l + 1.0) / (trunc * (trunc + 1.0))) ** 4 * (trunc + 1) / 32.0
    damping = {"vor": real(shape / 14400.0), "temp": real(shape / 14400.0), "div": real(shape / 3600.0), "lnps": 0.0}
    robert, williams = 0.1, 0.53
    for _ in range(case["steps"]):
        tend = tendencies(state)
        step, base = (dt, state) if previous is None else (2 * dt, previous)
        new = {k: (base[k] + step * tend[k]) / (1.0 + step * damping[k]) for k in state}
        if previous is not None:
            for k in state:
                d = previous[k] - 2 * state[k] + new[k]
                state[k] = state[k] + robert * williams / 2 * d
                new[k] = new[k] - robert * (1 - williams) / 2 * d
        previous, state = state, new
    return state


def _exact_mlp(case, seed):
    x, t, params = (v.to(torch.float64) for v in _mlp_inputs(case, seed))
    params.requires_grad_(True)
    sizes = ((128, 32), (128,), (128, 128), (128,), (32, 128), (32,))
    w1, b1, w2, b2, w3, b3 = (p.view(s) for p, s in zip(params.split([math.prod(s) for s in sizes]), sizes))
    gelu = torch.nn.functional.gelu
    y = gelu(gelu(x @ w1.T + b1) @ w2.T + b2) @ w3.T + b3
    if case["kind"] == "mlp_forward":
        return y.detach()
    loss = ((y - t) ** 2).mean()
    return {"loss": loss.detach().view(1), "grad": torch.autograd.grad(loss, params)[0]}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("mlp_forward", "mlp_gradient"):
        return _exact_mlp(case, seed)
    if kind == "forecast":
        return _exact_forecast(case, seed)
    if kind == "batch":
        gen, items = _generator(seed), _batch_items(case)
        fields, back = [None] * len(items), [None] * len(items)
        spectra = [_spectra(sw.Spectrum(trunc + 2, trunc + 1), K, gen).to(torch.complex128) for trunc, K in items]
        for trunc in sorted({t for t, _ in items}):  # the columns of one truncation together
            T = _Exact(trunc + 2, trunc + 1, "octahedral", sw.get_nlat_half(trunc + 1))
            mine = [i for i, (t, _) in enumerate(items) if t == trunc]
            f = T.synthesis(torch.cat([spectra[i] for i in mine]))
            b = T.analysis(f)
            sizes = [items[i][1] for i in mine]
            for i, fi, bi in zip(mine, f.split(sizes), b.split(sizes)):
                fields[i], back[i] = fi.reshape(-1), bi.reshape(-1)
        return {"fields": torch.cat(fields), "back": torch.cat(back)}
    spectrum, grid, K = _setup(case)
    T = _Exact(spectrum.lmax, spectrum.mmax, case.get("grid", "octahedral"), grid.nlat_half,
               case.get("shortcut", "linear"))
    a = _spectra(spectrum, K, _generator(seed)).to(torch.complex128)
    if kind == "pullbacks":
        f = torch.randn(K, grid.npoints, generator=_generator(seed + 1)).to(torch.float64)
        return {"coeffs_bar": T.synthesis_adjoint(f), "field_bar": T.analysis_adjoint(a)}
    f = T.synthesis(a)
    out = {"field": f, "back": T.analysis(f)}
    if kind == "vector":
        L = case["layers"]
        U, V = T.uv(a[:L], a[L:2 * L])
        uv = torch.cat([U, V])
        out.update(uv=uv, uv_field=T.synthesis(uv, unscale=True))
    return out
