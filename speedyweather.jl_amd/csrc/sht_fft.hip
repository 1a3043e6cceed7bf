// gfx950 ring FFT of the spherical harmonic transform (Fourier stage).
//
// One complex FFT of length nlon per ring and column carries the northern ring in the
// real part and the mirrored southern ring in the imaginary part: the per-ring
// rfft / brfft pairs of SpeedyTransforms/src/fourier.jl:27-77,129-250 for both hemispheres
// at once.  Mixed-radix Stockham autosort in LDS, decimation in time.  With
// N = r_1 r_2 ... r_s, pass p of radix r (l = r_1...r_{p-1}, M = N/(l r)) maps, for
// b in [0,M), u in [0,l):
//   in[b + M(q + r u)], q < r   ->   out[b + M(u + l s)], s < r
//   out = sum_q (w_N^{q u M} in_q) w_r^{q s},   w_N = exp(-/+ 2 pi i / N).
// Every pass runs in place in one LDS buffer.  A first-pass prime >= 17 (the octahedral
// rings nlon = 16 + 4j have prime factors up to 193 at T255) runs across the workgroup as
// two small GEMMs on MFMA; all other passes (radices 2..16, register butterflies) run
// across the workgroup with one thread per butterfly and group of columns.
//
// Bound by the chain of load, passes with a barrier each, and store, at 5 or 6 workgroups per CU:
// T255 K=64 takes 26.2 (synthesis) and 27.1 us (analysis), 15 of them what a copy of its traffic
// takes, about 6 each the prime and the register passes.  All global loads of a workgroup are one
// phase, and the synthesis's last pass stores the grid (before: 30.6 and 30.0 us).
#include "sht_device.h"

namespace sht {

// multiply by -i (forward) or +i (inverse)
template <bool INV>
__device__ inline float2 mul_mi(float2 a) {
    return INV ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}

template <bool INV>
__device__ inline float2 twid(const float2 *tw, int idx) {
    const float2 t = tw[idx];
    return INV ? make_float2(t.x, -t.y) : t;
}

__device__ inline float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
__device__ inline float2 cfma(float2 a, float s, float2 c) { return make_float2(fmaf(a.x, s, c.x), fmaf(a.y, s, c.y)); }

// DFT of R values in place (R = 2, 3, 4, 5, 7)
template <int R, bool INV>
__device__ inline void bfly(float2 *a) {
    if constexpr (R == 2) {
        const float2 t = a[0];
        a[0] = cadd(t, a[1]);
        a[1] = csub(t, a[1]);
    } else if constexpr (R == 4) {
        const float2 s02 = cadd(a[0], a[2]), d02 = csub(a[0], a[2]);
        const float2 s13 = cadd(a[1], a[3]), d13 = mul_mi<INV>(csub(a[1], a[3]));
        a[0] = cadd(s02, s13);
        a[1] = cadd(d02, d13);
        a[2] = csub(s02, s13);
        a[3] = csub(d02, d13);
    } else if constexpr (R == 3) {
        const float s3 = 0.86602540378443864676f;
        const float2 s = cadd(a[1], a[2]);
        const float2 d = mul_mi<INV>(csub(a[1], a[2]));
        const float2 base = cfma(s, -0.5f, a[0]);
        a[0] = cadd(a[0], s);
        a[1] = cfma(d, s3, base);
        a[2] = cfma(d, -s3, base);
    } else if constexpr (R == 5) {
        const float c1 = 0.30901699437494742410f, c2 = -0.80901699437494742410f;
        const float s1 = 0.95105651629515357212f, s2 = 0.58778525229247312917f;
        const float2 s14 = cadd(a[1], a[4]), d14 = mul_mi<INV>(csub(a[1], a[4]));
        const float2 s23 = cadd(a[2], a[3]), d23 = mul_mi<INV>(csub(a[2], a[3]));
        const float2 a0 = a[0];
        const float2 b1 = cfma(s23, c2, cfma(s14, c1, a0));
        const float2 b2 = cfma(s23, c1, cfma(s14, c2, a0));
        const float2 e1 = cfma(d23, s2, cscale(d14, s1));
        const float2 e2 = cfma(d23, -s1, cscale(d14, s2));
        a[0] = cadd(a0, cadd(s14, s23));
        a[1] = cadd(b1, e1);
        a[4] = csub(b1, e1);
        a[2] = cadd(b2, e2);
        a[3] = csub(b2, e2);
    } else {  // R == 7
        const float c1 = 0.62348980185873353053f, c2 = -0.22252093395631440429f, c3 = -0.90096886790241912624f;
        const float s1 = 0.78183148246802980871f, s2 = 0.97492791218182360702f, s3 = 0.43388373911755812048f;
        const float2 a0 = a[0];
        const float2 p1 = cadd(a[1], a[6]), q1 = mul_mi<INV>(csub(a[1], a[6]));
        const float2 p2 = cadd(a[2], a[5]), q2 = mul_mi<INV>(csub(a[2], a[5]));
        const float2 p3 = cadd(a[3], a[4]), q3 = mul_mi<INV>(csub(a[3], a[4]));
        const float2 b1 = cfma(p3, c3, cfma(p2, c2, cfma(p1, c1, a0)));
        const float2 b2 = cfma(p3, c1, cfma(p2, c3, cfma(p1, c2, a0)));
        const float2 b3 = cfma(p3, c2, cfma(p2, c1, cfma(p1, c3, a0)));
        const float2 e1 = cfma(q3, s3, cfma(q2, s2, cscale(q1, s1)));
        const float2 e2 = cfma(q3, -s1, cfma(q2, -s3, cscale(q1, s2)));
        const float2 e3 = cfma(q3, s2, cfma(q2, -s1, cscale(q1, s3)));
        a[0] = cadd(a0, cadd(p1, cadd(p2, p3)));
        a[1] = cadd(b1, e1);
        a[6] = csub(b1, e1);
        a[2] = cadd(b2, e2);
        a[5] = csub(b2, e2);
        a[3] = cadd(b3, e3);
        a[4] = csub(b3, e3);
    }
}

// DFT of an odd prime number R of values in place (R = 11, 13), by the symmetric
// pairs a_t +- a_{R-t}; cos / sin of 2 pi k / R come from the ring's table tw at k N/R.
template <int R, bool INV>
__device__ inline void bfly_odd(float2 *a, const float2 *tw, int stepR) {
    constexpr int H = (R - 1) / 2;
    float cs[H + 1], sn[H + 1];
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        const float2 w = tw[k * stepR];
        cs[k] = w.x;
        sn[k] = -w.y;
    }
    float2 p[H], q[H];
    float2 y0 = a[0];
#pragma unroll
    for (int t = 1; t <= H; ++t) {
        p[t - 1] = cadd(a[t], a[R - t]);
        q[t - 1] = mul_mi<INV>(csub(a[t], a[R - t]));
        y0 = cadd(y0, p[t - 1]);
    }
#pragma unroll
    for (int s = 1; s <= H; ++s) {
        float2 b = a[0], e = make_float2(0.f, 0.f);
#pragma unroll
        for (int t = 1; t <= H; ++t) {
            const int k = (s * t) % R;
            const float c = k <= H ? cs[k] : cs[R - k];
            const float sg = k <= H ? sn[k] : -sn[R - k];
            b = cfma(p[t - 1], c, b);
            e = cfma(q[t - 1], sg, e);
        }
        a[s] = cadd(b, e);
        a[R - s] = csub(b, e);
    }
    a[0] = y0;
}

// multiply by w8^k = exp(-+ i pi k / 4), k = 1, 2, 3
template <int K, bool INV>
__device__ inline float2 mul_w8(float2 a) {
    constexpr float h = 0.70710678118654752440f;
    if constexpr (K == 2) return mul_mi<INV>(a);
    // forward: w8 = (1 - i) h, w8^3 = (-1 - i) h; inverse: conjugates
    const float2 m = mul_mi<INV>(a);  // a * w8^2
    if constexpr (K == 1) return make_float2(h * (a.x + m.x), h * (a.y + m.y));
    return make_float2(h * (m.x - a.x), h * (m.y - a.y));
}

// radix 8: two radix-4 halves (even / odd inputs) joined by w8^k
template <bool INV>
__device__ inline void bfly8(float2 *a) {
    float2 e[4] = {a[0], a[2], a[4], a[6]}, o[4] = {a[1], a[3], a[5], a[7]};
    bfly<4, INV>(e);
    bfly<4, INV>(o);
    o[1] = mul_w8<1, INV>(o[1]);
    o[2] = mul_w8<2, INV>(o[2]);
    o[3] = mul_w8<3, INV>(o[3]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        a[k] = cadd(e[k], o[k]);
        a[k + 4] = csub(e[k], o[k]);
    }
}

// radix 16: four radix-4 DFTs over q = t mod 4, twiddles w16^{q k1}, radix-4 across q
template <bool INV>
__device__ inline void bfly16(float2 *a) {
    // cos / sin of 2 pi k / 16, k = 0..9 (only q k1 <= 9 occurs)
    const float C[10] = {1.f, 0.92387953251128675613f, 0.70710678118654752440f, 0.38268343236508977173f, 0.f,
                         -0.38268343236508977173f, -0.70710678118654752440f, -0.92387953251128675613f, -1.f,
                         -0.92387953251128675613f};
    const float S[10] = {0.f, 0.38268343236508977173f, 0.70710678118654752440f, 0.92387953251128675613f, 1.f,
                         0.92387953251128675613f, 0.70710678118654752440f, 0.38268343236508977173f, 0.f,
                         -0.38268343236508977173f};
    float2 b[4][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        b[q][0] = a[q];
        b[q][1] = a[q + 4];
        b[q][2] = a[q + 8];
        b[q][3] = a[q + 12];
        bfly<4, INV>(b[q]);
    }
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        float2 c[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = q * k1;
            const float2 v = b[q][k1];
            if (e == 0) {
                c[q] = v;
            } else {
                const float sn = INV ? S[e] : -S[e];  // w16^e = cos - i sin (forward)
                c[q] = make_float2(v.x * C[e] - v.y * sn, v.x * sn + v.y * C[e]);
            }
        }
        bfly<4, INV>(c);
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) a[k1 + 4 * k2] = c[k2];
    }
}

template <int R, bool INV>
__device__ inline void bfly_any(float2 *a, const float2 *tw, int stepR) {
    if constexpr (R == 8)
        bfly8<INV>(a);
    else if constexpr (R == 16)
        bfly16<INV>(a);
    else if constexpr (R <= 7)
        bfly<R, INV>(a);
    else
        bfly_odd<R, INV>(a, tw, stepR);
}

// A pass of radix R over all columns of N <= MAXN points, run by the workgroup.
// Work item = (column group of CB columns, butterfly t); items go to threads in order, so
// neighbouring lanes take neighbouring butterflies of one column group.  The index
// arithmetic and the twiddles of a butterfly serve all CB columns of its item.  Every
// thread reads all its items into registers, the workgroup synchronises, then the results
// are written in place.  Columns past the call's last column hold scratch values that are
// transformed along and never stored.
// CB by the number of butterflies per column (pass_columns): the fewest columns per item whose
// items still fit the workgroup's threads at once, so that short rings use all four waves
// instead of a few lanes with all columns each (T31 K=8: 5.7 -> 4.6 us synthesis, 5.8 -> 5.0
// analysis; T127 K=32: 9.2 -> 8.8, 9.4 -> 9.2).
// Radices 11 and 13 (one column per item) run as two sub-passes of two columns each where the
// items of four columns exceed the threads.
template <int R, int MAXN, int CBv, int SUBv = 1>
struct PassCols {
    static constexpr int CB = CBv;                   // columns per work item
    static constexpr int SUB = SUBv;                 // column sub-passes
    static constexpr int NCG = kFFTCols / CB / SUB;  // column groups per sub-pass
    static constexpr int kMaxB = MAXN / R;           // butterflies per column
    // the largest butterfly count this choice serves (pass_columns)
    static constexpr int kMaxNb = CB == 1 && SUB == 1 ? 64 : kMaxB;
    static constexpr int MAXI = ((kMaxNb < kMaxB ? kMaxNb : kMaxB) * NCG + kFFTThreads - 1) / kFFTThreads;
};
// Calls f with the column choice for nb butterflies per column.
template <int R, int MAXN, class F>
__device__ __forceinline__ void pass_columns(int nb, F &&f) {
    if constexpr (MAXN / R <= 64) {
        f(PassCols<R, MAXN, 1>{});
    } else {
        if (nb <= 64)
            f(PassCols<R, MAXN, 1>{});
        else if constexpr (R > 8)
            f(PassCols<R, MAXN, 1, 2>{});
        else
            f(PassCols<R, MAXN, 2>{});
    }
}

// The rings of a workgroup's columns in the grid: northern ring fn, southern ring fs of the
// first column, columns ld apart, ncol of them.
struct GridRings {
    SHT_GLOBAL float *fn, *fs;
    long long ld;
    int ncol;
};

// Twiddles of a ring on their way to LDS: loaded together with the ring's data (one memory
// latency for both), stored after every load of the thread is in flight.
template <int MAXN>
struct Twiddles {
    static constexpr int U = MAXN / kFFTThreads;
    float2 v[U];
    __device__ __forceinline__ void load(const float *twiddle, long long tw_off, int N, int tid) {
        const SHT_GLOBAL float2 *g = as_global(reinterpret_cast<const float2 *>(twiddle)) + tw_off;
#pragma unroll
        for (int q = 0; q < U; ++q) v[q] = gload(g + (unsigned)min(q * kFFTThreads + tid, N - 1));
    }
    __device__ __forceinline__ void store(float2 *tw, int N, int tid) const {
#pragma unroll
        for (int q = 0; q < U; ++q) {
            const int i = q * kFFTThreads + tid;
            if (i < N) tw[i] = v[q];
        }
    }
};

// The work items of a (sub-)pass: item it = tid + kFFTThreads i is butterfly t of column group
// cg; butterfly t = (b, u) reads points b + M (q + R u), q < R, of its columns.
template <class PC>
struct PassItem {
    int cg, u, b;
    __device__ __forceinline__ PassItem(int it, int nb, const FastDiv &divM) {
        cg = 0;
#pragma unroll
        for (int k = 1; k < PC::NCG; ++k) cg += it >= k * nb ? 1 : 0;  // NCG <= 4
        const int t = it - cg * nb;
        u = divM.div(t);
        b = t - u * divM.d;
    }
};

// Butterflies of one thread's items in registers.
template <int R, bool INV, class PC>
struct PassRegs {
    static constexpr int CB = PC::CB, NCG = PC::NCG, MAXI = PC::MAXI;
    float2 a[MAXI][CB][R];
    __device__ __forceinline__ void read(const float2 *buf, int N, const FFTPass &pd, int tid) {
        const int M = pd.M, nb = N / R, items = nb * NCG;
        const FastDiv divM(M, pd.mulM);
#pragma unroll
        for (int i = 0; i < MAXI; ++i) {
            const int it = tid + kFFTThreads * i;
            if (it >= items) continue;
            const PassItem<PC> p(it, nb, divM);
            const float2 *src = buf + p.cg * CB * N + p.b + M * R * p.u;
#pragma unroll
            for (int cc = 0; cc < CB; ++cc)
#pragma unroll
                for (int q = 0; q < R; ++q) a[i][cc][q] = src[cc * N + M * q];
        }
    }
    __device__ __forceinline__ void butterflies(int i, int u, const float2 *tw, int stepR, int M) {
        if (u > 0) {
#pragma unroll
            for (int q = 1; q < R; ++q) {
                const float2 w = twid<INV>(tw, q * u * M);
#pragma unroll
                for (int cc = 0; cc < CB; ++cc) a[i][cc][q] = cmul(a[i][cc][q], w);
            }
        }
#pragma unroll
        for (int cc = 0; cc < CB; ++cc) bfly_any<R, INV>(a[i][cc], tw, stepR);
    }
};

template <int R, bool INV, class PC>
__device__ __forceinline__ void fft_subpass_wg(float2 *buf, const float2 *tw, int N, const FFTPass &pd, int tid) {
    typedef PassRegs<R, INV, PC> Regs;
    constexpr int CB = Regs::CB;
    const int M = pd.M, nb = N / R, items = nb * Regs::NCG;
    const FastDiv divM(M, pd.mulM);
    Regs x;
    x.read(buf, N, pd, tid);
    __syncthreads();
    const int ls = nb;  // output stride between s: M l = N / R
#pragma unroll
    for (int i = 0; i < Regs::MAXI; ++i) {
        const int it = tid + kFFTThreads * i;
        if (it >= items) continue;
        const PassItem<PC> p(it, nb, divM);
        x.butterflies(i, p.u, tw, N / R, pd.M);
        float2 *dst = buf + p.cg * CB * N + p.b + M * p.u;
#pragma unroll
        for (int cc = 0; cc < CB; ++cc)
#pragma unroll
            for (int s = 0; s < R; ++s) dst[cc * N + ls * s] = x.a[i][cc][s];
    }
    __syncthreads();
}

template <int R, bool INV, int MAXN>
__device__ void fft_pass_wg(float2 *buf, const float2 *tw, int N, const FFTPass &pd, int tid) {
    pass_columns<R, MAXN>(N / R, [&](auto pc) {
        typedef decltype(pc) PC;
#pragma unroll
        for (int sp = 0; sp < PC::SUB; ++sp)
            fft_subpass_wg<R, INV, PC>(buf + sp * (kFFTCols / PC::SUB) * N, tw, N, pd, tid);
    });
}

// Last pass (M = 1, u = t) with its results stored straight to the grid: point u + l s of a
// butterfly's column, so neighbouring lanes store neighbouring points.  Nothing is written to
// LDS, so the items (one column each) run in a loop.  Even radices read their consecutive
// inputs in pairs (16-byte aligned: rings have a multiple of 4 points).
template <int R, bool INV>
__device__ void fft_last_pass(const float2 *buf, const float2 *tw, int N, const GridRings &out, int tid) {
    const int nb = N / R, items = nb * out.ncol;
#pragma unroll 1
    for (int it = tid; it < items; it += kFFTThreads) {
        int c = 0;
#pragma unroll
        for (int k = 1; k < kFFTCols; ++k) c += it >= k * nb ? 1 : 0;
        const int u = it - c * nb;
        const float2 *src = buf + c * N + R * u;
        float2 a[R];
        if constexpr (R % 2 == 0) {
#pragma unroll
            for (int q = 0; q < R; q += 2) {
                const float4 v = *reinterpret_cast<const float4 *>(src + q);
                a[q] = make_float2(v.x, v.y);
                a[q + 1] = make_float2(v.z, v.w);
            }
        } else {
#pragma unroll
            for (int q = 0; q < R; ++q) a[q] = src[q];
        }
        if (u > 0) {
#pragma unroll
            for (int q = 1; q < R; ++q) a[q] = cmul(a[q], twid<INV>(tw, q * u));
        }
        bfly_any<R, INV>(a, tw, nb);
        SHT_GLOBAL float *fn = out.fn + c * out.ld + u, *fs = out.fs + c * out.ld + u;
#pragma unroll
        for (int s = 0; s < R; ++s) {
            fn[(unsigned)(nb * s)] = a[s].x;
            fs[(unsigned)(nb * s)] = a[s].y;
        }
    }
}

// First pass (l = 1) of an odd prime radix r >= 11 as two small GEMMs on MFMA, in place.
// With the inputs x_q = buf[b + M q] of butterfly b, a_t = x_t + x_{r-t},
// b_t = x_t - x_{r-t} (t = 1..h, h = (r-1)/2):
//   T1[s] = sum_t cos(2 pi s t / r) a_t   (s = 0..h),   T2[s] = sum_t sin(2 pi s t / r) b_t
//   y_0 = x_0 + T1[0],  y_s = x_0 + T1[s] -+ i T2[s],  y_{r-s} = x_0 + T1[s] +- i T2[s]
// (upper signs forward), y_s -> buf[b + M s].  GEMM rows = s (row tiles of 16), columns =
// (butterfly, re/im) (column tiles of 16), K = t in chunks of 32.
//
// Products in three-part BF16 (v_mfma_f32_16x16x32_bf16, 16 cycles per 32-wide K chunk,
// against 8 FP32 MFMAs 16x16x4 of 32 cycles): cos / sin come from the plan's table for r
// (hi + mid + lo of the FP64 values, sht_plan.cpp: prime_tables); a_t and b_t are split the
// same way once per chunk and wave (x = hi + mid + lo exactly: BF16 keeps FP32's exponent
// range, so no scaling); the six products whose parts sum to at most 2 accumulate in FP32,
// smallest first, so the pass keeps FP32-level accuracy in every precision mode.
//
// Column tiles go to the waves in rounds of four; with fewer column tiles left, the waves of
// one column tile split its row tiles (at most prime_row_tiles(MAXN) per wave: rings of N = 4p
// points have M = N / r >= 4, see sht_plan.cpp: factorize).  All row tiles of a round's
// column tiles are computed before the workgroup synchronises and any output is written
// (a butterfly's outputs overwrite its inputs, which the other row tiles still read).
// tmax: the last pair t with nonzero inputs (a synthesis reads only the orders m <= mt and
// their mirrors N - m: x_t, x_{r-t} vanish for t > (mt + M - 1) / M); h otherwise.
//
// Pairs of values are rounded by one instruction per part (v_cvt_pk_bf16_f32) and widened
// again by a shift or a mask.
__device__ inline void split3_bf16(const float (&x)[8], b8 &hi, b8 &mid, b8 &lo) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    u4 part[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float a = x[2 * e], b = x[2 * e + 1];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const unsigned v = __builtin_bit_cast(unsigned, b2{(__bf16)a, (__bf16)b});
            part[q][e] = v;
            a -= __uint_as_float(v << 16);  // exact
            b -= __uint_as_float(v & 0xFFFF0000u);
        }
    }
    hi = __builtin_bit_cast(b8, part[0]);
    mid = __builtin_bit_cast(b8, part[1]);
    lo = __builtin_bit_cast(b8, part[2]);
}

// c += a b over the parts (i, j) with i + j <= 2, smallest first
__device__ inline f4 mma_bf16x3(const b8 &ah, const b8 &am, const b8 &al, const b8 &bh, const b8 &bm, const b8 &bl,
                                f4 c) {
    c = Split<kBF16x3>::mma(al, bh, c);
    c = Split<kBF16x3>::mma(ah, bl, c);
    c = Split<kBF16x3>::mma(am, bm, c);
    c = Split<kBF16x3>::mma(am, bh, c);
    c = Split<kBF16x3>::mma(ah, bm, c);
    return Split<kBF16x3>::mma(ah, bh, c);
}

template <bool INV, int MAXN>
__device__ void fft_pass_mfma_first(float2 *buf, const SHT_GLOBAL b8 *tab, int N, const FFTPass &pd, int ncol,
                                    int tmax, int tid) {
    const int r = pd.R, M = pd.M;
    const int h = (r - 1) >> 1;
    const int nseq = ncol * M;  // butterflies over all columns
    constexpr int NW = kFFTThreads / 64, kRows = prime_row_tiles(MAXN);
    // the wave index is uniform per wave: keep it (and all tile ownership) scalar
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = lane & 15, grp = lane >> 4, ri = row & 1;
    const int Mt = (h + 16) >> 4;         // row tiles (rows 0..h)
    const int Nt = (2 * nseq + 15) >> 4;  // column tiles over (butterfly, re/im)
    const int KC = (h + 31) >> 5;         // K chunks of the table
    const int KU = (tmax + 31) >> 5;      // K chunks with nonzero inputs
    const FastDiv divM(M, pd.mulM);
    const float *bf = reinterpret_cast<const float *>(buf);
    for (int n0 = 0; n0 < Nt; n0 += NW) {  // uniform: every wave takes part in every round's barriers
        const int nc = min(NW, Nt - n0);   // column tiles this round
        const int G = NW / nc;             // waves per column tile
        const int nt = n0 + wave % nc, r0 = wave / nc;
        const int nrt = wave < nc * G ? min((Mt - r0 + G - 1) / G, kRows) : 0;  // uniform per wave
        f4 t1[kRows], t2[kRows];
#pragma unroll
        for (int i = 0; i < kRows; ++i) t1[i] = t2[i] = f4{0.f, 0.f, 0.f, 0.f};
        int ob = -1;
        float2 z0 = make_float2(0.f, 0.f);
        if (nrt > 0) {
            const int c = nt * 16 + row, sq = c >> 1;
            int base = 0;  // columns past the data read column 0; their outputs are dropped
            if (sq < nseq) {
                const int col = divM.div(sq);
                base = col * N + (sq - col * M);
                ob = base;
                z0 = buf[base];  // x_0, read before any output of the round is written
            }
            // t past h re-reads the pair h, for which the table holds zeros; pairs between tmax and
            // h are zero themselves
            const float *pa = bf + 2 * base + ri, *pb = pa + 2 * M * r;
            for (int kc = 0; kc < KU; ++kc) {
                float xs[8], xd[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int o = __mul24(min(32 * kc + 8 * grp + e + 1, h), 2 * M);
                    const float xa = pa[o], xb = pb[-o];
                    xs[e] = xa + xb;
                    xd[e] = xa - xb;
                }
                b8 sh, sm, sl, dh, dm, dl;
                split3_bf16(xs, sh, sm, sl);
                split3_bf16(xd, dh, dm, dl);
#pragma unroll
                for (int i = 0; i < kRows; ++i) {
                    if (i >= nrt) break;  // uniform per wave
                    const SHT_GLOBAL b8 *a = tab + ((r0 + i * G) * KC + kc) * 384 + lane;
                    const b8 ch = a[0], cm = a[64], cl = a[128];
                    t1[i] = mma_bf16x3(ch, cm, cl, sh, sm, sl, t1[i]);
                    const b8 nh = a[192], nm = a[256], nl = a[320];
                    t2[i] = mma_bf16x3(nh, nm, nl, dh, dm, dl, t2[i]);
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            if (i >= nrt) break;  // uniform per wave
            const int mt = r0 + i * G;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // the partner lane (c ^ 1) holds the other part of the same butterfly
                const float a1 = t1[i][e], a2 = t2[i][e];
                const float p1 = lane_xor1(a1), p2 = lane_xor1(a2);
                const int s = mt * 16 + 4 * grp + e;
                if (ob < 0 || s > h) continue;
                const float T1re = ri ? p1 : a1, T1im = ri ? a1 : p1;
                const float T2re = ri ? p2 : a2, T2im = ri ? a2 : p2;
                const float sg = INV ? -1.f : 1.f;
                if (s == 0) {
                    if (ri == 0) buf[ob] = make_float2(z0.x + T1re, z0.y + T1im);
                } else if (ri == 0) {
                    buf[ob + M * s] = make_float2(z0.x + T1re + sg * T2im, z0.y + T1im - sg * T2re);
                } else {
                    buf[ob + M * (r - s)] = make_float2(z0.x + T1re - sg * T2im, z0.y + T1im + sg * T2re);
                }
            }
        }
        __syncthreads();
    }
}

// A pass descriptor read field by field (structures do not copy through global pointers).
__device__ __forceinline__ FFTPass load_pass(const SHT_GLOBAL FFTPass *p) {
    const SHT_GLOBAL int *q = reinterpret_cast<const SHT_GLOBAL int *>(p);
    FFTPass d;
    d.R = q[0];
    d.l = q[1];
    d.M = q[2];
    d.mulM = (unsigned)q[3];
    return d;
}

// The plan tables the FFT kernels read, fetched with the ring record (one level of scalar loads).
struct FFTPlanTables {
    const float *twiddle;
    const FFTPass *passes;
    const unsigned short *prime_tab;
};

// Runs all passes in place on buf (kFFTCols columns of N points, the first ncol of them data):
// a first-pass MFMA radix, then the register passes, all across the workgroup.  pd: the first
// register pass's descriptor, fetched before the ring's data.  Every pass ends with a barrier,
// but LAST's, which stores the grid.

template <bool INV, bool LAST, int MAXN>
__device__ __attribute__((always_inline)) void fft_run(const FFTPlanTables &P, const FFTRing &R, float2 *buf,
                                                        const float2 *tw, int N, int mt, int ncol, FFTPass pd,
                                                        const GridRings &out, int tid) {
    const SHT_GLOBAL FFTPass *passes = as_global(P.passes) + R.passes;
    const int nf = R.nf;
    int f = 0;
    if (R.prime) {  // the MFMA first pass (its descriptor and table offset come with the ring)
        FFTPass p0;
        p0.R = R.prime;
        p0.l = 1;
        p0.M = R.M0;
        p0.mulM = R.mulM0;
        const SHT_GLOBAL b8 *tab = reinterpret_cast<const SHT_GLOBAL b8 *>(as_global(P.prime_tab)) + R.prime_off;
        const int h = (p0.R - 1) >> 1;
        const int tmax = INV ? min(h, (mt + p0.M - 1) / p0.M) : h;
        int t = tid;
        asm volatile("" : "+v"(t));
        fft_pass_mfma_first<INV, MAXN>(buf, tab, N, p0, ncol, max(tmax, 1), t);
        f = 1;
    }
    for (int g = f; g < nf - (LAST ? 1 : 0); ++g) {
        // the next pass's descriptor loads while this one runs (past the last: its own again)
        const FFTPass nx = load_pass(passes + min(g + 1, nf - 1));
        int t = tid;  // keeps every pass's index arithmetic inside the loop (hoisted, it spills)
        asm volatile("" : "+v"(t));
        switch (pd.R) {
            case 16: fft_pass_wg<16, INV, MAXN>(buf, tw, N, pd, t); break;
            case 8: fft_pass_wg<8, INV, MAXN>(buf, tw, N, pd, t); break;
            case 2: fft_pass_wg<2, INV, MAXN>(buf, tw, N, pd, t); break;
            case 3: fft_pass_wg<3, INV, MAXN>(buf, tw, N, pd, t); break;
            case 4: fft_pass_wg<4, INV, MAXN>(buf, tw, N, pd, t); break;
            case 5: fft_pass_wg<5, INV, MAXN>(buf, tw, N, pd, t); break;
            case 7: fft_pass_wg<7, INV, MAXN>(buf, tw, N, pd, t); break;
            case 11: fft_pass_wg<11, INV, MAXN>(buf, tw, N, pd, t); break;
            default: fft_pass_wg<13, INV, MAXN>(buf, tw, N, pd, t); break;  // the plan admits no other radix
        }
        pd = nx;
    }
    if constexpr (LAST) {
        int t = tid;
        asm volatile("" : "+v"(t));
        switch (pd.R) {
            case 16: fft_last_pass<16, INV>(buf, tw, N, out, t); break;
            case 8: fft_last_pass<8, INV>(buf, tw, N, out, t); break;
            case 2: fft_last_pass<2, INV>(buf, tw, N, out, t); break;
            case 3: fft_last_pass<3, INV>(buf, tw, N, out, t); break;
            case 4: fft_last_pass<4, INV>(buf, tw, N, out, t); break;
            case 5: fft_last_pass<5, INV>(buf, tw, N, out, t); break;
            case 7: fft_last_pass<7, INV>(buf, tw, N, out, t); break;
            case 11: fft_last_pass<11, INV>(buf, tw, N, out, t); break;
            default: fft_last_pass<13, INV>(buf, tw, N, out, t); break;
        }
    }
}

// The ring record of a rank, read field by field (structures do not copy through global
// pointers): one level of loads after the rank is known.
__device__ __forceinline__ FFTRing load_ring(const SHT_GLOBAL FFTRing *p) {
    const SHT_GLOBAL int *q = reinterpret_cast<const SHT_GLOBAL int *>(p);
    const SHT_GLOBAL long long *w = reinterpret_cast<const SHT_GLOBAL long long *>(p);
    FFTRing r;
    r.j = q[0];
    r.N = q[1];
    r.mt = q[2];
    r.mte = q[3];
    r.nf = q[4];
    r.prime = q[5];
    r.M0 = q[6];
    r.mulM0 = (unsigned)q[7];
    r.tw_off = w[6];
    r.fboff = w[7];
    r.ring_n = w[8];
    r.ring_s = w[9];
    r.prime_off = w[10];
    r.passes = w[11];
    return r;
}

// Per-workgroup launch geometry of the FFT kernels: the ring's record, first column k0,
// columns ncol.
struct FFTTile {
    FFTRing R;
    int k0, ncol;
};

// Single-call launch orders, rings heaviest first.  Grouped: every column group of ring rank r
// on XCD r % 8 (blocks go round-robin over the XCDs), so the ring's twiddles and tables are
// fetched into one L2, and the two column groups that share the 128-byte lines of the Fourier
// rows (64 bytes each) meet in it: T255 K=64 with buffers that are not cache-resident, the
// analysis, which writes those rows, takes 34.1 us with its column groups spread over the
// XCDs and 30.3 us grouped.  Otherwise (a tuning choice of the synthesis): block b -> ring
// rank b / kgs, column group b % kgs.  Batch tiles carry the rank (m) and column group.
// rings: the plan's ring records (single calls pass them in place of a tile list), followed by
// copies of the first marked j < 0 up to a multiple of the XCD count: blocks past the last ring
// issue a valid ring's loads and then exit, so that no branch stands between the kernel's
// arguments and the loads that depend on them.
template <bool BATCH>
__device__ inline void fft_tile(const SHT_GLOBAL FFTRing *rings, const Tile &T, int K, bool paired, FFTTile &t) {
    const int kgs = (K + kFFTCols - 1) / kFFTCols;
    int cg, r;
    if (BATCH) {
        r = T.m;
        cg = T.blk;
    } else {
        const int b = blockIdx.x;
        if (paired) {
            const int s = b / kXCDs;
            r = (s / kgs) * kXCDs + b % kXCDs;
            cg = s - (s / kgs) * kgs;
        } else {
            r = b / kgs;
            cg = b - r * kgs;
        }
    }
    t.R = load_ring(rings + r);
    t.k0 = cg * kFFTCols;
    t.ncol = min(kFFTCols, K - t.k0);
}

// Fourier rows are read and written with thread -> (order mm = tid/4 + 64 u, column tid%4).
constexpr int kFFTRowsPerPass = kFFTThreads / kFFTCols;
constexpr int fft_row_passes(int max_ring) { return (max_ring / 2 + kFFTRowsPerPass) / kFFTRowsPerPass; }
// Workgroups (4 waves) per CU that a class is compiled for.  The passes wait on LDS more than they
// compute, so what bounds short rings is workgroups in flight, and registers (512 per SIMD lane)
// limit these before LDS does: 80 registers for rings of up to 512 points against 96 of the general
// kernel, with no loads past the ring's length.  T127 K=392 synthesis + analysis 46.7 + 49.2 ->
// 40.7 + 42.3 us, K=32 9.0 + 9.1 -> 8.6 + 8.4, T31 K=8 4.8 + 4.9 -> 4.2 + 4.2; a 7th workgroup
// spills (T127 K=392 49.4 + 41.3).
constexpr int fft_waves(int max_ring) { return max_ring <= 512 ? 6 : 5; }

// spectral -> grid, Fourier stage (fourier.jl:215-250): per ring, brfft of g_N and g_S as
// one complex inverse FFT of Z = g_N + i g_S (Hermitian-extended; Im of the DC and
// Nyquist bins ignored as FFTW's c2r does; orders above mt are zero).  ACC: the pullback
// that adds into the caller's grid (its own instantiation, so the plain transform keeps
// its registers).
template <int MAXN, bool BATCH, bool ACC = false>
__global__ __launch_bounds__(kFFTThreads, fft_waves(MAXN))
void fft_synthesis_kernel(const DevPlan *__restrict__ plans, CallArgs single, const CallArgs *__restrict__ calls,
                          const Tile *__restrict__ tiles) {
    extern __shared__ float4 smem4[];
    float2 *smem = reinterpret_cast<float2 *>(smem4);
    const int tid = threadIdx.x;
    const Tile T = BATCH ? tiles[blockIdx.x] : Tile{0, 0, 0, 0};
    if (BATCH && T.m < 0) return;  // padding of the launch order
    const CallArgs C = BATCH ? calls[T.call] : single;
    const DevPlan &P = plans[BATCH ? C.plan : 0];
    const int K = C.K;
    const SHT_GLOBAL FFTRing *rings =
        BATCH ? as_global(P.rings) : as_global(reinterpret_cast<const FFTRing *>(tiles));
    const FFTPlanTables tables{P.twiddle, P.passes, P.prime_tab};
    FFTTile G;
    fft_tile<BATCH>(rings, T, K, C.paired != 0, G);
    const FFTRing &R = G.R;
    const int N = R.N, mt = R.mt, ncol = G.ncol;
    __builtin_assume(N >= 1 && N <= MAXN);  // offsets within a ring fit scalar-base loads
    float2 *tw = smem;
    float2 *b0 = smem + N;
    const FFTPass pass0 = load_pass(as_global(tables.passes) + R.passes + (R.prime ? min(1, R.nf - 1) : 0));
    Twiddles<MAXN> twr;
    twr.load(tables.twiddle, R.tw_off, N, tid);
    constexpr int kRowPasses = fft_row_passes(MAXN);
    {
        const SHT_GLOBAL float4 *fb =
            as_global(static_cast<const float4 *>(C.fbuf)) + R.fboff * (long long)K + G.k0;
        const int half = N / 2;
        const int col = tid % kFFTCols, m0 = tid / kFFTCols;
        float4 v[kRowPasses];
#pragma unroll
        for (int u = 0; u < kRowPasses; ++u) {
            const int mm = m0 + kFFTRowsPerPass * u;
            v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (col < ncol && mm <= mt) v[u] = gload(fb + (unsigned)(mm * K + col));
        }
        if (!BATCH && R.j < 0) return;
        __builtin_amdgcn_sched_barrier(0);  // every load in flight before the first LDS store
        twr.store(tw, N, tid);
        if (C.adj) {  // adjoint of the analysis (grid2spec pullback): rows times ΔΩ_j / s_m
            const float wj = as_global(P.domega)[R.j];
#pragma unroll
            for (int u = 0; u < kRowPasses; ++u) {
                const int mm = m0 + kFFTRowsPerPass * u;
                const float sw = mm == 0 || 2 * mm == N ? wj : 0.5f * wj;
                v[u] = make_float4(v[u].x * sw, v[u].y * sw, v[u].z * sw, v[u].w * sw);
            }
        }
        float2 *z = b0 + col * N;
#pragma unroll
        for (int u = 0; u < kRowPasses; ++u) {
            const int mm = m0 + kFFTRowsPerPass * u;
            if (col >= ncol || mm > half) continue;
            const float4 w = v[u];
            if (mm == 0) {
                z[0] = make_float2(w.x, w.z);
            } else if (mm < half) {
                z[mm] = make_float2(w.x - w.w, w.y + w.z);
                z[N - mm] = make_float2(w.x + w.w, w.z - w.y);
            } else {
                z[half] = make_float2(w.x, w.z);
            }
        }
    }
    __syncthreads();
    SHT_GLOBAL float *field = as_global(static_cast<float *>(C.out)) + (long long)G.k0 * C.ld_out;
    const GridRings out{field + R.ring_n, field + R.ring_s, C.ld_out, ncol};
    fft_run<true, !ACC, MAXN>(tables, R, b0, tw, N, mt, ncol, pass0, out, tid);
    if constexpr (ACC) {
        // pullback: add into the caller's cotangent; a column's old values are all read before
        // its first store, so the reads are in flight together
        constexpr int U = MAXN / kFFTThreads;
#pragma unroll
        for (int c = 0; c < kFFTCols; ++c) {
            if (c >= ncol) break;  // uniform
            SHT_GLOBAL float *fn = out.fn + c * out.ld, *fs = out.fs + c * out.ld;
            const float2 *z = b0 + c * N;
            float on[U], os[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = min(u * kFFTThreads + tid, N - 1);
                on[u] = fn[(unsigned)i];
                os[u] = fs[(unsigned)i];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = u * kFFTThreads + tid;
                if (i < N) {
                    const float2 v = z[i];
                    fn[(unsigned)i] = on[u] + v.x;
                    fs[(unsigned)i] = os[u] + v.y;
                }
            }
        }
    }
}

// grid -> spectral, Fourier stage (fourier.jl:129-166): per ring, rfft of the northern and
// southern ring as one complex FFT of z = f_N + i f_S, separated by symmetry into f_N, f_S
// and stored as (f_N + f_S, f_N - f_S) for orders 0..mt.
template <int MAXN, bool BATCH>
__global__ __launch_bounds__(kFFTThreads, fft_waves(MAXN))
void fft_analysis_kernel(const DevPlan *__restrict__ plans, CallArgs single, const CallArgs *__restrict__ calls,
                         const Tile *__restrict__ tiles) {
    extern __shared__ float4 smem4[];
    float2 *smem = reinterpret_cast<float2 *>(smem4);
    const int tid = threadIdx.x;
    const Tile T = BATCH ? tiles[blockIdx.x] : Tile{0, 0, 0, 0};
    if (BATCH && T.m < 0) return;  // padding of the launch order
    const CallArgs C = BATCH ? calls[T.call] : single;
    const DevPlan &P = plans[BATCH ? C.plan : 0];
    const int K = C.K;
    const SHT_GLOBAL FFTRing *rings =
        BATCH ? as_global(P.rings) : as_global(reinterpret_cast<const FFTRing *>(tiles));
    const FFTPlanTables tables{P.twiddle, P.passes, P.prime_tab};
    FFTTile G;
    fft_tile<BATCH>(rings, T, K, true, G);
    const FFTRing &R = G.R;
    const int N = R.N, mt = R.mt, ncol = G.ncol;
    __builtin_assume(N >= 1 && N <= MAXN);  // offsets within a ring fit scalar-base loads
    float2 *tw = smem;
    float2 *b0 = smem + N;
    const FFTPass pass0 = load_pass(as_global(tables.passes) + R.passes + (R.prime ? min(1, R.nf - 1) : 0));
    Twiddles<MAXN> twr;
    twr.load(tables.twiddle, R.tw_off, N, tid);
    const SHT_GLOBAL float *field = as_global(static_cast<const float *>(C.in)) + (long long)G.k0 * C.ld_in;
    const GridRings in{const_cast<SHT_GLOBAL float *>(field + R.ring_n), const_cast<SHT_GLOBAL float *>(field + R.ring_s),
                       C.ld_in, ncol};
    {
        constexpr int U = MAXN / kFFTThreads;
        // all loads of the thread in flight before the first LDS store (columns past ncol
        // re-read column 0 and are not stored)
        float vn[kFFTCols][U], vs[kFFTCols][U];
#pragma unroll
        for (int c = 0; c < kFFTCols; ++c) {
            const long long o = (long long)(c < ncol ? c : 0) * in.ld;
            const SHT_GLOBAL float *fn = in.fn + o, *fs = in.fs + o;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const unsigned i = min(u * kFFTThreads + tid, N - 1);
                vn[c][u] = fn[i];
                vs[c][u] = fs[i];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        twr.store(tw, N, tid);
#pragma unroll
        for (int c = 0; c < kFFTCols; ++c) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = u * kFFTThreads + tid;
                if (c < ncol && i < N) b0[c * N + i] = make_float2(vn[c][u], vs[c][u]);
            }
        }
        __syncthreads();
    }
    // padding of the launch order leaves here, the whole workgroup (ahead of the LDS stores the exit
    // costs the other workgroups' schedule: T255 K=64 28.8 us instead of 28.1)
    if (!BATCH && R.j < 0) return;
    fft_run<false, false, MAXN>(tables, R, b0, tw, N, mt, ncol, pass0, GridRings{}, tid);
    {
        SHT_GLOBAL float4 *fb = as_global(static_cast<float4 *>(C.fbuf)) + R.fboff * (long long)K + G.k0;
        int t = tid;
        asm volatile("" : "+v"(t));
        const int col = t % kFFTCols, m0 = t / kFFTCols;
        const float2 *z = b0 + col * N;
        // adjoint of the synthesis (spec2grid pullback): rows times s_m (1/cos lat) / ΔΩ_j
        const float wj = C.adj ? (C.unscale ? as_global(P.coslat_inv)[R.j] : 1.f) / as_global(P.domega)[R.j] : 1.f;
        // rows mt < m <= mte (orders that rings nearer the pole keep under a non-monotonic
        // shortcut) are written as zeros: the Legendre analysis sums every ring from the
        // first one of an order on
        const int mte = R.mte;
#pragma unroll
        for (int u = 0; u < fft_row_passes(MAXN); ++u) {
            const int mm = m0 + kFFTRowsPerPass * u;
            if (col >= ncol || mm > mte) continue;
            if (mm > mt) {
                gstore(fb + (unsigned)(mm * K + col), make_float4(0.f, 0.f, 0.f, 0.f));
                continue;
            }
            const float2 p = z[mm];
            const float2 q = z[mm == 0 ? 0 : N - mm];
            // f_N = (Z_m + conj Z_{N-m})/2, f_S = (Z_m - conj Z_{N-m})/(2i)
            const float h = C.adj ? (mm == 0 || 2 * mm == N ? 0.5f * wj : wj) : 0.5f;
            const float nre = h * (p.x + q.x), nim = h * (p.y - q.y);
            const float sre = h * (p.y + q.y), sim = h * (q.x - p.x);
            gstore(fb + (unsigned)(mm * K + col), make_float4(nre + sre, nim + sim, nre - sre, nim - sim));
        }
    }
}

// ================================================================== entry points

template <int MAXN>
static const void *fft_entry(int stage, bool batch, bool accumulate) {
    if (stage == kFFTSynthesis) {
        if (accumulate && !batch) return reinterpret_cast<const void *>(&fft_synthesis_kernel<MAXN, false, true>);
        return batch ? reinterpret_cast<const void *>(&fft_synthesis_kernel<MAXN, true>)
                     : reinterpret_cast<const void *>(&fft_synthesis_kernel<MAXN, false>);
    }
    return batch ? reinterpret_cast<const void *>(&fft_analysis_kernel<MAXN, true>)
                 : reinterpret_cast<const void *>(&fft_analysis_kernel<MAXN, false>);
}

const void *fft_kernel(int stage, bool batch, int cls, bool accumulate) {
    if (cls == 0) return fft_entry<fft_class_ring(0)>(stage, batch, accumulate);
    if (cls == 1) return fft_entry<fft_class_ring(1)>(stage, batch, accumulate);
    return fft_entry<fft_class_ring(2)>(stage, batch, accumulate);
}

}  // namespace sht
