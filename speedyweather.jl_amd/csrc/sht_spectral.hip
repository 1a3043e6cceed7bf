// Spectral-space operators that feed the transform (vector path of the model step), and
// the dense transform's GEMM.
#include <algorithm>

#include "sht_device.h"

namespace sht {

// ============================================================ UV from vor, div
__global__ void uv_from_vordiv_kernel(const DevPlan *__restrict__ PP, const float2 *__restrict__ vor_,
                                      const float2 *__restrict__ dv_, float2 *__restrict__ U_,
                                      float2 *__restrict__ V_, long long ld, float radius) {
    const DevPlan &P = *PP;
    const int lm = blockIdx.x * blockDim.x + threadIdx.x;
    if (lm >= P.nharm) return;
    const long long base = (long long)blockIdx.y * ld;  // column k = blockIdx.y
    float2 uu, vv;
    uv_stencil(P, as_global(vor_) + base, as_global(dv_) + base, lm, uu, vv);
    gstore(as_global(U_) + base + lm, make_float2(uu.x * radius, uu.y * radius));
    gstore(as_global(V_) + base + lm, make_float2(vv.x * radius, vv.y * radius));
}

// ======================================================= spectral gradient operators
// Per packed (l, m) and column, stencils in l with the reference's factor arrays
// (gradient_arrays.jl:4-21,27-76,80-100,150-170), in float:
//   divergence (spectral_gradients.jl:105-125): i m_x u - gyvd1 v[lm-1] + gyvd2 v[lm+1]
//   curl (:30-41, the divergence kernel on (v, u) with the signs of b, c swapped)
//   Laplacian (:385-420): a * (-l(l+1)) or a / (-l(l+1)) (0 at l = 0)
//   gradient (:483-527): dpdx = i m p, dpdy = gy1 p[lm-1] + gy2 p[lm+1]
// Factors crossing an order boundary (l = m below, l = lmax-1 above) are zero by construction.
// The last packed element of the divergence / curl is 0; flipsign, add and the radius
// scaling follow the reference's order (scaling after adding).
__global__ void spectral_op_kernel(const DevPlan *__restrict__ PP, int op, const float2 *__restrict__ a_,
                                   const float2 *__restrict__ b_, float2 *__restrict__ o1_, float2 *__restrict__ o2_,
                                   long long ld, int flags, float rscale) {
    const DevPlan &P = *PP;
    const int lm = blockIdx.x * blockDim.x + threadIdx.x;
    const int last = P.nharm - 1;
    if (lm > last) return;
    const long long base = (long long)blockIdx.y * ld;
    const SHT_GLOBAL float2 *a = as_global(a_) + base;
    SHT_GLOBAL float2 *o1 = as_global(o1_) + base;
    const bool flip = flags & kOpFlip, add = flags & kOpAdd;
    float2 val;
    if (op == kOpDivergence || op == kOpCurl) {
        if (lm == last) {
            val = make_float2(0.f, 0.f);
        } else {
            const SHT_GLOBAL float2 *b = as_global(b_) + base;
            const SHT_GLOBAL float2 *X = op == kOpCurl ? b : a;  // zonal operand
            const SHT_GLOBAL float2 *Y = op == kOpCurl ? a : b;  // meridional operand
            const float4 gy = gload(as_global(P.gy) + lm);       // (gyvd1, gyvd2, gy1, gy2)
            const float mx = gload(as_global(P.gx) + lm).x;
            const float2 z = gload(X + lm);
            const float2 ym = lm > 0 ? gload(Y + lm - 1) : make_float2(0.f, 0.f);
            const float2 yp = gload(Y + lm + 1);
            const float sg = op == kOpCurl ? 1.f : -1.f;
            val = make_float2(-mx * z.y + sg * (gy.x * ym.x - gy.y * yp.x), mx * z.x + sg * (gy.x * ym.y - gy.y * yp.y));
            if (flip) val = make_float2(-val.x, -val.y);
            if (add) {
                const float2 o = gload(o1 + lm);
                val = make_float2(o.x + val.x, o.y + val.y);
            }
        }
    } else if (op == kOpLaplace) {
        const int l = as_global(P.l_of)[lm];
        float e = -(float)(l * (l + 1));
        if (flags & kOpInverse) e = l == 0 ? 0.f : 1.f / e;
        const float2 z = gload(a + lm);
        val = make_float2(z.x * e, z.y * e);
        if (flip) val = make_float2(-val.x, -val.y);
        if (add) {
            const float2 o = gload(o1 + lm);
            val = make_float2(o.x + val.x, o.y + val.y);
        }
    } else {  // gradient: o1 = dpdx, o2 = dpdy
        const float m = gload(as_global(P.gx) + lm).y;
        const float4 gy = gload(as_global(P.gy) + lm);
        const float2 z = gload(a + lm);
        const float2 pm = lm > 0 ? gload(a + lm - 1) : make_float2(0.f, 0.f);
        const float2 pp = lm < last ? gload(a + lm + 1) : make_float2(0.f, 0.f);
        gstore(o1 + lm, make_float2(-m * z.y * rscale, m * z.x * rscale));
        val = make_float2(gy.z * pm.x + gy.w * pp.x, gy.z * pm.y + gy.w * pp.y);
        gstore(as_global(o2_) + base + lm, make_float2(val.x * rscale, val.y * rscale));
        return;
    }
    gstore(o1 + lm, make_float2(val.x * rscale, val.y * rscale));
}

int launch_spectral_op(const DevPlan *P, int nharm, int op, const void *a, const void *b, void *o1, void *o2,
                       long long ld, int K, int flags, float rscale, void *stream) {
    if (nharm < 1 || K < 1 || K > 65535) return (int)hipErrorInvalidValue;
    const dim3 grid((nharm + 255) / 256, K);
    spectral_op_kernel<<<grid, 256, 0, as_stream(stream)>>>(P, op, static_cast<const float2 *>(a),
                                                            static_cast<const float2 *>(b), static_cast<float2 *>(o1),
                                                            static_cast<float2 *>(o2), ld, flags, rscale);
    return (int)hipGetLastError();
}

// =========================================================== per-point scaling
__global__ void scale_points_kernel(const float *__restrict__ scale, float *__restrict__ field, long long npoints,
                                    long long ld) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npoints) return;
    SHT_GLOBAL float *f = as_global(field) + (long long)blockIdx.y * ld + p;
    *f = *f * as_global(scale)[p];
}

int launch_scale_points(const float *scale, void *field, long long npoints, long long ld, int K, void *stream) {
    if (npoints < 1 || K < 1 || K > 65535) return (int)hipErrorInvalidValue;
    const dim3 grid((unsigned)((npoints + 255) / 256), K);
    scale_points_kernel<<<grid, 256, 0, as_stream(stream)>>>(scale, static_cast<float *>(field), npoints, ld);
    return (int)hipGetLastError();
}

// ============================================================ dense transform GEMM
// C (M x K, column stride ldc) = A (M x N) B (N x K, column stride ldb), then optionally
// C[r, k] *= row_scale[r].  The dense transform's products have few columns (K layers) and
// a large A that must be read once, so the GEMM runs on v_mfma_f32_16x16x4_f32 with A in
// fragment order (dense_fragment_index: each wave's load of four K-steps is 1 KiB
// contiguous) and is bound by reading A.  Workgroup = four waves, each one 16-row tile, times a
// split of the contraction; the split's rows of B (all K columns, up to 64 per column group)
// are staged in LDS 64 at a time, double-buffered (one barrier per chunk), and shared by the
// four row tiles.  A step issues the next chunk's B loads before its A loads, so storing B
// waits for no A, and A stays in flight through the step's products.  T63 K=32 (188 MB of A
// per direction), round trip: 144 us with one buffer, B loaded after A and 16-way bank
// conflicts of the stores; 106 us so (3.6 TB/s; K=2: 94.5 -> 78.8 us, 4.8 TB/s).  With one
// split the result is stored directly; otherwise partial sums go to W[s][k][r] and a second
// kernel adds them in a fixed order (no atomics, deterministic).

constexpr int kDenseChunk = 4;  // fragment groups (16 contraction values each) staged at once
constexpr int kDenseMinGroups = 16;  // shortest split of the contraction, in fragment groups
constexpr int kDenseCols = 64;  // columns of B per column group (four column tiles)

template <int NCT>
__global__ __launch_bounds__(256) void dense_mfma_kernel(const float4 *__restrict__ Af_, long long RT, long long S4,
                                                         long long M, long long N, const float *__restrict__ B_,
                                                         long long ldb, int K, int s4_split, float *__restrict__ out_,
                                                         long long ldo, int direct,
                                                         const float *__restrict__ row_scale) {
    // LDS row stride (17 modulo 32): a wave stores 64 rows of one column to distinct banks, and
    // the four lane groups read their rows of 16 columns from nearly disjoint ones
    constexpr int BST = 16 * NCT + (NCT % 2 ? 1 : 17);
    constexpr int CR = kDenseChunk * 16;  // rows of B staged per chunk
    __shared__ float Bs[2][CR][BST];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = lane & 15, kg = lane >> 4;
    const long long rt = (long long)blockIdx.x * 4 + w;  // idle waves (rt >= RT) still stage and synchronise
    const int sp = blockIdx.y;
    const int k0 = blockIdx.z * kDenseCols, Kg = min(kDenseCols, K - k0);
    const long long s4a = (long long)sp * s4_split, s4b = min(S4, s4a + s4_split);
    const SHT_GLOBAL float *B = as_global(B_) + (long long)k0 * ldb;
    const SHT_GLOBAL fv4 *Aw = reinterpret_cast<const SHT_GLOBAL fv4 *>(as_global(Af_)) +
                               (min(rt, RT - 1) * S4) * 64 + lane;
    f4 acc[NCT], sum[NCT];
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) acc[ct] = sum[ct] = f4{0.f, 0.f, 0.f, 0.f};
    // every 256 contraction values the running sum moves on (blocked summation: the longer
    // splits of fewer workgroups would otherwise lose accuracy)
    auto fold = [&]() {
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) {
            sum[ct] += acc[ct];
            acc[ct] = f4{0.f, 0.f, 0.f, 0.f};
        }
    };
    // Chunks of kDenseChunk fragment groups.  Step c stores the staged rows of B into LDS
    // buffer c % 2, issues the loads of B and A of chunk c + 1 (B first: the next step waits
    // for it while A is still in flight), synchronises once and multiplies.  Loads past the
    // split re-read its last group (of A) or row 0 (of B, stored as zero).
    constexpr int PER = CR * 16 * NCT / 256;  // B values per thread and chunk
    const int nch = (int)((s4b - s4a + kDenseChunk - 1) / kDenseChunk);
    const long long nmax = min(16 * s4b, N);
    static_assert(CR == 64, "a lane stages one row of a chunk");
    struct Ops {
        fv4 a[kDenseChunk];
        float b[PER];
    };
    auto load = [&](Ops &S, int c) {
        c = min(c, nch - 1);
        const long long c0 = s4a + (long long)c * kDenseChunk;
#pragma unroll
        for (int u = 0; u < PER; ++u) {  // row lane of the chunk, column w + 4 u (uniform per wave)
            const SHT_GLOBAL float *col = B + (long long)min(w + 4 * u, Kg - 1) * ldb;
            S.b[u] = col[(unsigned)(16 * c0 + lane < nmax ? (int)(16 * c0) + lane : 0)];
        }
#pragma unroll
        for (int v = 0; v < kDenseChunk; ++v) S.a[v] = Aw[(unsigned)min((int)c0 + v, (int)s4b - 1) * 64u];
    };
    auto step = [&](Ops &cur, Ops &nxt, int c) {
        const long long c0 = s4a + (long long)c * kDenseChunk;
        float (*bs)[BST] = Bs[c & 1];
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int j = w + 4 * u;
            bs[lane][j] = 16 * c0 + lane < nmax && j < Kg ? cur.b[u] : 0.f;
        }
        load(nxt, c + 1);
        __syncthreads();
#pragma unroll
        for (int v = 0; v < kDenseChunk; ++v) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int q = 16 * v + 4 * k + kg;
#pragma unroll
                for (int ct = 0; ct < NCT; ++ct) acc[ct] = mfma_f32(cur.a[v][k], bs[q][ct * 16 + row], acc[ct]);
            }
        }
    };
    Ops S0, S1;
    load(S0, 0);
    int c = 0;
    for (; c + 1 < nch; c += 2) {  // straight-line body: each set waits for its own loads
        step(S0, S1, c);
        step(S1, S0, c + 1);
        if (c & 2) fold();
    }
    if (c < nch) step(S0, S1, c);
    fold();
    if (rt >= RT) return;
    SHT_GLOBAL float *out = as_global(out_);
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
        const int k = ct * 16 + row;
        if (k >= Kg) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const long long r = rt * 16 + 4 * kg + i;
            if (r >= M) continue;
            if (direct)
                out[r + (long long)(k0 + k) * ldo] = sum[ct][i] * (row_scale ? as_global(row_scale)[r] : 1.f);
            else
                out[((long long)sp * K + k0 + k) * M + r] = sum[ct][i];
        }
    }
}

// Sum of the S partials of 32 rows of one column k: 8 thread groups each add every 8th
// split (independent loads in flight), then group 0 adds the 8 group sums in order.
constexpr int kReduceRows = 32, kReduceGroups = 8;
__global__ __launch_bounds__(256) void dense_reduce_kernel(const float *__restrict__ W_, long long M, int K, int S,
                                                           const float *__restrict__ row_scale,
                                                           float *__restrict__ C_, long long ldc) {
    __shared__ float part[kReduceGroups][kReduceRows];
    const int row = threadIdx.x % kReduceRows, grp = threadIdx.x / kReduceRows;
    const long long r = (long long)blockIdx.x * kReduceRows + row;
    const int k = blockIdx.y;
    const long long rc = r < M ? r : M - 1;  // rows past M read row M - 1 and are not stored
    const SHT_GLOBAL float *W = as_global(W_) + (long long)k * M + rc;
    const long long step = (long long)K * M;
    float sum = 0.f;
#pragma unroll 4
    for (int sp = grp; sp < S; sp += kReduceGroups) sum += W[(long long)sp * step];
    part[grp][row] = sum;
    __syncthreads();
    if (grp != 0 || r >= M) return;
    float t = part[0][row];
#pragma unroll
    for (int g = 1; g < kReduceGroups; ++g) t += part[g][row];
    if (row_scale) t *= as_global(row_scale)[r];
    as_global(C_)[r + (long long)k * ldc] = t;
}

DenseSplit dense_split(long long M, long long N, int K) {
    DenseSplit d;
    d.rt = (M + 15) / 16;
    d.s4 = (N + 15) / 16;
    d.cg = (K + kDenseCols - 1) / kDenseCols;
    const long long wgs = (d.rt + 3) / 4 * d.cg;
    // About 1024 workgroups (four per CU resident), but at least kDenseMinGroups groups per
    // split: shorter ones spend their time on partial sums (T31 K=32, round trip: 21.7 us with
    // 16 groups, 43.8 with 2; T63 K=32: 106.7 us with 1024 workgroups, 110.5 with 2048, 118.1
    // with 3072).
    auto splits = [&](long long want, int &per) {  // of at most `want` equal parts, none empty
        want = std::max(1LL, std::min(want, d.s4));
        per = (int)((d.s4 + want - 1) / want);
        return (int)((d.s4 + per - 1) / per);
    };
    d.s = splits(std::min((1024 + wgs - 1) / wgs, d.s4 / kDenseMinGroups), d.s4_split);
    int per;
    d.s_work = splits((2048 + wgs - 1) / wgs, per);  // plans are accepted and refused by this size
    return d;
}

long long dense_fragment_index(long long r, long long n, long long S4) {
    const long long rt = r / 16, s4 = n / 16, q = n % 16;
    const long long lane = (r % 16) + 16 * (q % 4), v = q / 4;
    return ((rt * S4 + s4) * 64 + lane) * 4 + v;
}

int launch_dense_gemm(const float *Af, long long M, long long N, const float *B, long long ldb, int K, float *C,
                      long long ldc, const float *row_scale, float *work, void *stream) {
    if (M < 1 || N < 1 || K < 1 || K > 65535 || ldb < N || ldc < M) return (int)hipErrorInvalidValue;
    const DenseSplit d = dense_split(M, N, K);
    if ((d.rt + 3) / 4 > 0x7fffffffLL || d.s > 65535 || d.cg > 65535) return (int)hipErrorInvalidValue;
    const hipStream_t st = as_stream(stream);
    const dim3 grid((unsigned)((d.rt + 3) / 4), d.s, d.cg);
    const bool direct = d.s == 1;
    float *out = direct ? C : work;
    const long long ldo = direct ? ldc : M;
    const float4 *A4 = reinterpret_cast<const float4 *>(Af);
    const int nct = std::min(4, (std::min(K, kDenseCols) + 15) / 16);
    switch (nct) {
        case 1: dense_mfma_kernel<1><<<grid, 256, 0, st>>>(A4, d.rt, d.s4, M, N, B, ldb, K, d.s4_split, out, ldo, direct, row_scale); break;
        case 2: dense_mfma_kernel<2><<<grid, 256, 0, st>>>(A4, d.rt, d.s4, M, N, B, ldb, K, d.s4_split, out, ldo, direct, row_scale); break;
        case 3: dense_mfma_kernel<3><<<grid, 256, 0, st>>>(A4, d.rt, d.s4, M, N, B, ldb, K, d.s4_split, out, ldo, direct, row_scale); break;
        default: dense_mfma_kernel<4><<<grid, 256, 0, st>>>(A4, d.rt, d.s4, M, N, B, ldb, K, d.s4_split, out, ldo, direct, row_scale); break;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || direct) return (int)e;
    dense_reduce_kernel<<<dim3((unsigned)((M + kReduceRows - 1) / kReduceRows), K), 256, 0, st>>>(work, M, K, d.s,
                                                                                                row_scale, C, ldc);
    return (int)hipGetLastError();
}

int launch_uv_from_vordiv(const DevPlan *P, int nharm, const void *vor, const void *div, void *U,
                          void *V, long long ld, int K, float radius, void *stream) {
    if (nharm < 1 || K < 1 || K > 65535) return (int)hipErrorInvalidValue;
    const dim3 grid((nharm + 255) / 256, K);
    uv_from_vordiv_kernel<<<grid, 256, 0, as_stream(stream)>>>(
        P, static_cast<const float2 *>(vor), static_cast<const float2 *>(div),
        static_cast<float2 *>(U), static_cast<float2 *>(V), ld, radius);
    return (int)hipGetLastError();
}

}  // namespace sht
