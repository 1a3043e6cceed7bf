// Per-column MLP of the learned tendency correction: 32 -> 128 -> 128 -> 32 with GELU,
// BF16 weights (FP32 master copy), FP32 accumulation.  Inputs are the 32 values of one
// grid column (8 levels x {u, v, T, ln ps}); outputs the 32 tendency corrections.
//
// Everything runs on MFMA (v_mfma_f32_16x16x32_bf16).  Forward: activations are rounded to
// BF16 at each layer input, products accumulate in FP32, bias and GELU in FP32.  Backward
// differentiates exactly that function: one operand of each of its products is a BF16-rounded
// weight or activation, the other an FP32 gradient split into BF16 hi + mid + lo (its value
// exactly), so three MFMAs give the FP32 product.  Weight gradients are summed over row tiles
// in the accumulators and over workgroups in a fixed order (deterministic), then Adam updates
// the FP32 master weights and refreshes their BF16 copies.
//
// Parameter vector (float, kMlpParams): W1[128][32] b1[128] W2[128][128] b2[128]
// W3[32][128] b3[32], W[o][i] maps input i to output o.
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/sht.h"
#include "sht_device.h"

namespace sht {

constexpr int kIn = 32, kHid = 128, kOut = 32;
constexpr int kOffW1 = 0, kOffB1 = kOffW1 + kHid * kIn, kOffW2 = kOffB1 + kHid, kOffB2 = kOffW2 + kHid * kHid,
              kOffW3 = kOffB2 + kHid, kOffB3 = kOffW3 + kOut * kHid, kMlpParams = kOffB3 + kOut;

// BF16 weights in MFMA fragment order: fragments of 16 outputs x 32 contraction values, 8
// values per lane (512 values, 1 KiB).  Activations stay where the accumulators have them:
// lane (batch row n, group g) holds rows 4 g + i of output tile t, and needs contraction values
// 32 c + 8 g + e of chunk c in the next layer.  The hidden layers' output rows are therefore
// dealt to the tiles 2 c, 2 c + 1 so that these are the same features (feature 32 c + 8 g + 4 (t
// & 1) + i, out_feature), and no activation moves between lanes from one layer to the next.
// T2, T3: the transposes, for backward (inputs dealt to the tiles the same way).
constexpr int kF1 = 0, kF2 = kF1 + 8, kF3 = kF2 + 32, kT3 = kF3 + 8, kT2 = kT3 + 8, kFrags = kT2 + 32;
__host__ __device__ inline int frag_index(int frag, int row, int k) {
    return (frag * 64 + (k >> 3) * 16 + row) * 8 + (k & 7);
}
// First of the four consecutive features that lane group g holds of tile t.
__host__ __device__ constexpr int out_feature(int t, int g) { return 32 * (t >> 1) + 8 * g + 4 * (t & 1); }
// Tile and row of feature f under that dealing.
__host__ __device__ inline void feature_tile(int f, int &t, int &row) {
    t = 2 * (f >> 5) + ((f >> 2) & 1);
    row = 4 * ((f >> 3) & 3) + (f & 3);
}

typedef __bf16 bf16;
typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

__device__ inline float gelu(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752f)); }
// GELU and its derivative
__device__ inline float gelu(float x, float &d) {
    const float c = 1.f + erff(x * 0.70710678118654752f);
    d = 0.5f * c + x * 0.39894228040143268f * expf(-0.5f * x * x);
    return 0.5f * x * c;
}

__device__ inline f4 mfma_bf16(bf16x8 a, bf16x8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ bf16x8 load_frag(const SHT_GLOBAL bf16x8 *W, int frag, int lane) {
    return W[frag * 64 + lane];
}
__device__ __forceinline__ f4 load_f4(const SHT_GLOBAL float *p) {
    return *reinterpret_cast<const SHT_GLOBAL f4 *>(p);
}
// Inputs 8 g .. 8 g + 7 of one row, rounded to BF16 (zeros past the last row).  The pointer is
// read float by float: callers pass rows of any float alignment.
__device__ __forceinline__ bf16x8 load_inputs(const SHT_GLOBAL float *X, long long r, int g, bool ok) {
    const SHT_GLOBAL float *x = X + r * kIn + 8 * g;
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (bf16)(ok ? x[e] : 0.f);
    return v;
}

// Forward: y = W3 g(W2 g(W1 x + b1) + b2) + b3.  One wave per 16 rows, which it takes through
// all three layers in registers (z^T = W act^T: a lane's accumulators of two tiles are its
// contraction values of the next layer), so no LDS and no barrier; the layers' weight
// fragments come from L2.  Bound by the GELUs (256 error functions per row: 7.8 us without
// them in a timing copy).  25 344 rows:
// 25.0 us with the layers through LDS and a barrier around each, 15.4 us so (results bitwise
// the same).
__global__ __launch_bounds__(256) void mlp_forward_kernel(const bf16 *__restrict__ Wf, const float *__restrict__ P_,
                                                          const float *__restrict__ X, float *__restrict__ Y, int B) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n = lane & 15, g = lane >> 4;
    const long long r = ((long long)blockIdx.x * 4 + wave) * 16 + n;
    const bool ok = r < B;
    const SHT_GLOBAL bf16x8 *W = reinterpret_cast<const SHT_GLOBAL bf16x8 *>(as_global(Wf));
    const SHT_GLOBAL float *P = as_global(P_);
    const f4 zero{0.f, 0.f, 0.f, 0.f};
    const bf16x8 xb = load_inputs(as_global(X), ok ? r : 0, g, ok);
    bf16x8 h[4];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const f4 z = mfma_bf16(load_frag(W, kF1 + t, lane), xb, zero) + load_f4(P + kOffB1 + out_feature(t, g));
#pragma unroll
        for (int i = 0; i < 4; ++i) h[t >> 1][4 * (t & 1) + i] = (bf16)gelu(z[i]);
    }
    f4 z2[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        z2[t] = zero;
#pragma unroll
        for (int c = 0; c < 4; ++c) z2[t] = mfma_bf16(load_frag(W, kF2 + 4 * t + c, lane), h[c], z2[t]);
        z2[t] += load_f4(P + kOffB2 + out_feature(t, g));
    }
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) h[t >> 1][4 * (t & 1) + i] = (bf16)gelu(z2[t][i]);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        f4 y = zero;
#pragma unroll
        for (int c = 0; c < 4; ++c) y = mfma_bf16(load_frag(W, kF3 + 4 * t + c, lane), h[c], y);
        y += load_f4(P + kOffB3 + out_feature(t, g));
        SHT_GLOBAL float *out = as_global(Y) + r * kOut + out_feature(t, g);
        if (ok)
#pragma unroll
            for (int i = 0; i < 4; ++i) out[i] = y[i];
    }
}

// ------------------------------------------------------------------ loss and gradient
//
// L = mean((y - t)^2) over B x 32 values: forward, backward and the weight gradients of a
// range of 32-row tiles in one workgroup of 8 waves.  In the chain of layers wave (rg, fg)
// takes row group rg (16 rows) and the 32 features fg of every hidden layer; activations and
// gradients pass between the waves of a row group through LDS, row-major (N tiles).  For the
// weight gradients, whose contraction runs over the 32 rows, they are also kept feature-major
// (F tiles): wave w owns output tile w of W2 and W1
// and input tile w of W3, accumulated over all tiles of the workgroup; the bias gradients are
// products with ones.  Each workgroup writes one partial parameter gradient (97 KiB): one
// 32-row tile per workgroup up to 256 workgroups (one per CU), then more tiles each.  Bound by
// the chain of five barriers and the weights' latency at one workgroup per CU, then by the
// partials' traffic (4096 rows: 12.7 MB written and read).  4096 rows, loss and gradient:
// 273 us with scalar FP32 products, 64 rows per workgroup and the activations through HBM;
// 20.9 us so.
constexpr int kGradRows = 32, kGradThreads = 512, kMaxGradBlocks = 256;
constexpr int kSN = kHid + 8, kSF = kGradRows + 8;  // row strides (16-bit): 16-byte aligned, bank-spread
constexpr int kNTile = kGradRows * kSN, kFTile = kHid * kSF, kFSmall = 32 * kSF;
constexpr int kLdsH1N = 0, kLdsH2N = kLdsH1N + kNTile, kLdsD2N = kLdsH2N + kNTile, kLdsH1F = kLdsD2N + 3 * kNTile,
              kLdsH2F = kLdsH1F + kFTile, kLdsD2F = kLdsH2F + kFTile, kLdsD1F = kLdsD2F + 3 * kFTile,
              kLdsDyF = kLdsD1F + 3 * kFTile, kLdsXF = kLdsDyF + 3 * kFSmall, kLdsEnd = kLdsXF + kFSmall;
constexpr int kGradLds = kLdsEnd * 2;  // bytes
static_assert(kGradLds <= 160 * 1024, "one workgroup per CU");

__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
    typedef bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(unsigned, bf16x2{(bf16)a, (bf16)b});
}
__device__ __forceinline__ unsigned dpp_xor1(unsigned x) {
    return (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, false);  // quad_perm [1,0,3,2]
}
// Four features f .. f+3 (packed pairs) of row n, row-major.
__device__ __forceinline__ void put_n(u16 *lds, int n, int f, unsigned a, unsigned b) {
    *reinterpret_cast<u32x2 *>(lds + n * kSN + f) = u32x2{a, b};
}
// The same feature-major: lanes n, n ^ 1 exchange halves, the even one writes feature f of
// both rows, the odd one feature f + 1, as one 32-bit store each.
__device__ __forceinline__ void put_f(u16 *lds, int f, int n, unsigned a, unsigned b) {
    const bool odd = n & 1;
    const unsigned sel = odd ? 0x03020706u : 0x05040100u;
    const int o = (f + (odd ? 1 : 0)) * kSF + (n & ~1);
    // v_perm: bytes 0-3 from the second operand, 4-7 from the first
    *reinterpret_cast<unsigned *>(lds + o) = __builtin_amdgcn_perm(dpp_xor1(a), a, sel);
    *reinterpret_cast<unsigned *>(lds + o + 2 * kSF) = __builtin_amdgcn_perm(dpp_xor1(b), b, sel);
}
// BF16 parts of four FP32 values as packed pairs: part[q][0..1], hi + mid + lo = v exactly.  hi
// is truncated, not rounded, and the rest of an infinity is 0, so that products of the parts
// overflow only where those of v do (rounded up, hi may exceed the range that v is in; inf - inf
// would make the rest NaN).
__device__ __forceinline__ float nan_to_zero(float r) {
    float z;  // the median of r, r, 0; with a NaN among them the least number
    asm("v_med3_f32 %0, %1, %1, 0" : "=v"(z) : "v"(r));
    return z;
}
__device__ __forceinline__ void split4(const float (&v)[4], unsigned (&part)[3][2]) {
    float r[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = nan_to_zero(v[e] - __uint_as_float(__float_as_uint(v[e]) & 0xFFFF0000u));
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        part[0][k] = __builtin_amdgcn_perm(__float_as_uint(v[2 * k + 1]), __float_as_uint(v[2 * k]), 0x07060302u);
        part[1][k] = pack_bf16(r[2 * k], r[2 * k + 1]);
        part[2][k] = pack_bf16(r[2 * k] - __uint_as_float(part[1][k] << 16),
                               r[2 * k + 1] - __uint_as_float(part[1][k] & 0xFFFF0000u));
    }
}
__device__ __forceinline__ bf16x8 frag_n(const u16 *lds, int n, int pos) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8 *>(lds + n * kSN + pos));
}
__device__ __forceinline__ bf16x8 frag_f(const u16 *lds, int f, int g) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8 *>(lds + f * kSF + 8 * g));
}

__global__ __launch_bounds__(kGradThreads, 2) void mlp_gradient_kernel(const bf16 *__restrict__ Wf,
                                                                       const float *__restrict__ P_,
                                                                       const float *__restrict__ X_,
                                                                       const float *__restrict__ T_,
                                                                       float *__restrict__ G, float *__restrict__ Lp,
                                                                       int B, int tiles) {
    extern __shared__ float4 mlp_lds[];
    u16 *lds = reinterpret_cast<u16 *>(mlp_lds);
    __shared__ float red[kGradThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15, g = lane >> 4;
    const int rg = wave & 1, fg = wave >> 1;
    const int n = 16 * rg + c16;  // row within the tile
    const SHT_GLOBAL float *P = as_global(P_);
    const SHT_GLOBAL float *X = as_global(X_);
    const SHT_GLOBAL float *T = as_global(T_);
    const f4 zero{0.f, 0.f, 0.f, 0.f};
    const float scale = 2.f / ((float)B * kOut);
    f4 a2[8], a1[2], a3[2], b1 = zero, b2 = zero, b3[2] = {zero, zero};
#pragma unroll
    for (int j = 0; j < 8; ++j) a2[j] = zero;
#pragma unroll
    for (int j = 0; j < 2; ++j) a1[j] = a3[j] = zero;
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = (bf16)1.f;
    float lsum = 0.f;
    for (int tile = blockIdx.x * tiles; tile < (blockIdx.x + 1) * tiles; ++tile) {  // uniform
        // the weights are read anew for every tile (kept across tiles they would spill)
        int w0 = 0;
        asm volatile("" : "+s"(w0));
        const SHT_GLOBAL bf16x8 *W = reinterpret_cast<const SHT_GLOBAL bf16x8 *>(as_global(Wf)) + w0;
        const long long r = (long long)tile * kGradRows + n;
        const bool ok = r < B;
        const long long rr = ok ? r : 0;
        const bf16x8 xb = load_inputs(X, rr, g, ok);
        if (fg == 0)
#pragma unroll
            for (int e = 0; e < 8; ++e) lds[kLdsXF + (8 * g + e) * kSF + n] = __builtin_bit_cast(u16, (bf16)xb[e]);
        // layer 1
        float g1[2][4], g2[2][4];  // GELU derivatives
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int f = out_feature(2 * fg + t, g);
            const f4 z = mfma_bf16(load_frag(W, kF1 + 2 * fg + t, lane), xb, zero) + load_f4(P + kOffB1 + f);
            float h[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = gelu(z[i], g1[t][i]);
            const unsigned pa = pack_bf16(h[0], h[1]), pb = pack_bf16(h[2], h[3]);
            put_n(lds + kLdsH1N, n, out_feature(2 * fg + t, g), pa, pb);
            put_f(lds + kLdsH1F, f, n, pa, pb);
        }
        __syncthreads();
        // layer 2
        {
            f4 z[2] = {zero, zero};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const bf16x8 b = frag_n(lds + kLdsH1N, n, 32 * c + 8 * g);
#pragma unroll
                for (int t = 0; t < 2; ++t) z[t] = mfma_bf16(load_frag(W, kF2 + 4 * (2 * fg + t) + c, lane), b, z[t]);
            }
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int f = out_feature(2 * fg + t, g);
                z[t] += load_f4(P + kOffB2 + f);
                float h[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) h[i] = gelu(z[t][i], g2[t][i]);
                const unsigned pa = pack_bf16(h[0], h[1]), pb = pack_bf16(h[2], h[3]);
                put_n(lds + kLdsH2N, n, out_feature(2 * fg + t, g), pa, pb);
                put_f(lds + kLdsH2F, f, n, pa, pb);
            }
        }
        __syncthreads();
        // output layer and loss, in every wave of the row group (two tiles); dL/dy as BF16 parts
        unsigned dy[2][3][2];
        {
            f4 y[2] = {zero, zero};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const bf16x8 b = frag_n(lds + kLdsH2N, n, 32 * c + 8 * g);
#pragma unroll
                for (int t = 0; t < 2; ++t) y[t] = mfma_bf16(load_frag(W, kF3 + 4 * t + c, lane), b, y[t]);
            }
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int o = out_feature(t, g);
                y[t] += load_f4(P + kOffB3 + o);
                float d[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    d[i] = ok ? y[t][i] - T[rr * kOut + o + i] : 0.f;
                    if (fg == 0) lsum = fmaf(d[i], d[i], lsum);
                    d[i] *= scale;
                }
                split4(d, dy[t]);
                if (fg == 0)
#pragma unroll
                    for (int q = 0; q < 3; ++q) put_f(lds + kLdsDyF + q * kFSmall, o, n, dy[t][q][0], dy[t][q][1]);
            }
        }
        // dz2 = (W3^T dy) gelu'(z2): the 32 outputs are one chunk, straight from the registers
        {
            bf16x8 b[3];
            typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
            for (int q = 0; q < 3; ++q)
                b[q] = __builtin_bit_cast(bf16x8, u32x4{dy[0][q][0], dy[0][q][1], dy[1][q][0], dy[1][q][1]});
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const bf16x8 a = load_frag(W, kT3 + 2 * fg + t, lane);
                f4 d = mfma_bf16(a, b[2], zero);
                d = mfma_bf16(a, b[1], d);
                d = mfma_bf16(a, b[0], d);
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = d[i] * g2[t][i];
                unsigned part[3][2];
                split4(v, part);
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    put_n(lds + kLdsD2N + q * kNTile, n, out_feature(2 * fg + t, g), part[q][0], part[q][1]);
                    put_f(lds + kLdsD2F + q * kFTile, out_feature(2 * fg + t, g), n, part[q][0], part[q][1]);
                }
            }
        }
        __syncthreads();
        // dz1 = (W2^T dz2) gelu'(z1)
        {
            f4 d[2] = {zero, zero};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                bf16x8 b[3];
#pragma unroll
                for (int q = 0; q < 3; ++q) b[q] = frag_n(lds + kLdsD2N + q * kNTile, n, 32 * c + 8 * g);
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const bf16x8 a = load_frag(W, kT2 + 4 * (2 * fg + t) + c, lane);
                    d[t] = mfma_bf16(a, b[2], d[t]);
                    d[t] = mfma_bf16(a, b[1], d[t]);
                    d[t] = mfma_bf16(a, b[0], d[t]);
                }
            }
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = d[t][i] * g1[t][i];
                unsigned part[3][2];
                split4(v, part);
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    put_f(lds + kLdsD1F + q * kFTile, out_feature(2 * fg + t, g), n, part[q][0], part[q][1]);
            }
        }
        __syncthreads();
        // weight gradients: contraction over the tile's 32 rows, smallest part first
#pragma unroll
        for (int q = 2; q >= 0; --q) {
            const bf16x8 d2 = frag_f(lds + kLdsD2F + q * kFTile, 16 * wave + c16, g);
            const bf16x8 d1 = frag_f(lds + kLdsD1F + q * kFTile, 16 * wave + c16, g);
            b2 = mfma_bf16(d2, ones, b2);
            b1 = mfma_bf16(d1, ones, b1);
#pragma unroll
            for (int j = 0; j < 8; ++j) a2[j] = mfma_bf16(d2, frag_f(lds + kLdsH1F, 16 * j + c16, g), a2[j]);
            const bf16x8 h2 = frag_f(lds + kLdsH2F, 16 * wave + c16, g);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                a1[t] = mfma_bf16(d1, frag_f(lds + kLdsXF, 16 * t + c16, g), a1[t]);
                const bf16x8 d3 = frag_f(lds + kLdsDyF + q * kFSmall, 16 * t + c16, g);
                a3[t] = mfma_bf16(d3, h2, a3[t]);
                b3[t] = mfma_bf16(d3, ones, b3[t]);
            }
        }
        __syncthreads();
    }
    SHT_GLOBAL float *out = as_global(G) + (long long)blockIdx.x * kMlpParams;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int o = 16 * wave + 4 * g + i;
#pragma unroll
        for (int j = 0; j < 8; ++j) out[kOffW2 + o * kHid + 16 * j + c16] = a2[j][i];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            out[kOffW1 + o * kIn + 16 * t + c16] = a1[t][i];
            out[kOffW3 + (16 * t + 4 * g + i) * kHid + 16 * wave + c16] = a3[t][i];
        }
        if (c16 == 0) {
            out[kOffB1 + o] = b1[i];
            out[kOffB2 + o] = b2[i];
            if (wave == 0)
#pragma unroll
                for (int t = 0; t < 2; ++t) out[kOffB3 + 16 * t + 4 * g + i] = b3[t][i];
        }
    }
    for (int s = 32; s > 0; s >>= 1) lsum += __shfl_xor(lsum, s);
    if (lane == 0) red[wave] = lsum;
    __syncthreads();
    if (tid == 0) Lp[blockIdx.x] = red[0] + red[1];  // fg = 0: the waves of both row groups
}

// Writes one BF16 weight (parameter p) to its fragments.
__device__ inline void store_weight(bf16 *Wf, int p, float w) {
    const bf16 v = (bf16)w;
    int t, row;
    if (p < kOffB1) {
        const int o = p / kIn, i = p % kIn;
        feature_tile(o, t, row);
        Wf[frag_index(kF1 + t, row, i)] = v;
    } else if (p >= kOffW2 && p < kOffB2) {
        const int o = (p - kOffW2) / kHid, i = (p - kOffW2) % kHid;
        feature_tile(o, t, row);
        Wf[frag_index(kF2 + 4 * t + i / 32, row, i % 32)] = v;
        feature_tile(i, t, row);
        Wf[frag_index(kT2 + 4 * t + o / 32, row, o % 32)] = v;
    } else if (p >= kOffW3 && p < kOffB3) {
        const int o = (p - kOffW3) / kHid, i = (p - kOffW3) % kHid;
        feature_tile(o, t, row);
        Wf[frag_index(kF3 + 4 * t + i / 32, row, i % 32)] = v;
        feature_tile(i, t, row);
        Wf[frag_index(kT3 + t, row, o)] = v;
    }
}

// Sums the workgroups' partial gradients (64 parameters per workgroup; four thread groups
// take every fourth partial and are added in order: deterministic) and the loss, then either
// stores the gradient or, with ADAM, takes an Adam step on the FP32 master weights and
// refreshes their BF16 fragments.
struct AdamArgs {
    float *P;
    bf16 *Wf;
    float *M, *V;
    float lr, b1, b2, eps, c1, c2;
};
template <bool ADAM>
__global__ __launch_bounds__(256) void mlp_reduce_kernel(const float *__restrict__ Gp_, float *__restrict__ G,
                                                         const float *__restrict__ Lp, float *__restrict__ loss,
                                                         int nblk, int B, AdamArgs A) {
    __shared__ float part[4][64];
    const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + lane;
    const SHT_GLOBAL float *Gp = as_global(Gp_) + min(p, kMlpParams - 1);
    float s = 0.f;
#pragma unroll 8
    for (int b = grp; b < nblk; b += 4) s += Gp[(long long)b * kMlpParams];
    part[grp][lane] = s;
    __syncthreads();
    if (grp == 1 && blockIdx.x == 0) {
        float l = 0.f;
        for (int b = lane; b < nblk; b += 64) l += Lp[b];
        for (int k = 32; k > 0; k >>= 1) l += __shfl_xor(l, k);
        if (lane == 0) loss[0] = l / ((float)B * kOut);
    }
    if (grp != 0 || p >= kMlpParams) return;
    const float gv = ((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane];
    if constexpr (!ADAM) {
        G[p] = gv;
    } else {
        const float m = A.b1 * A.M[p] + (1.f - A.b1) * gv;
        const float v = A.b2 * A.V[p] + (1.f - A.b2) * gv * gv;
        A.M[p] = m;
        A.V[p] = v;
        const float w = A.P[p] - A.lr * (m / A.c1) / (sqrtf(v / A.c2) + A.eps);
        A.P[p] = w;
        store_weight(A.Wf, p, w);
    }
}

__global__ void mlp_cast_kernel(const float *__restrict__ P, bf16 *__restrict__ Wf) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < kMlpParams) store_weight(Wf, p, P[p]);
}

// Workgroups of a gradient over B rows and their tiles each: one tile per workgroup while
// the device's 256 CUs have room, then evenly more.
inline int grad_blocks(int B, int &tiles) {
    const int nt = (B + kGradRows - 1) / kGradRows;
    tiles = (nt + kMaxGradBlocks - 1) / kMaxGradBlocks;
    return (nt + tiles - 1) / tiles;
}

}  // namespace sht

using namespace sht;

struct sht_mlp {
    int device = 0;
    int max_batch = 0;
    float *P = nullptr, *M = nullptr, *V = nullptr, *Gp = nullptr, *Lp = nullptr, *loss = nullptr;
    bf16 *Wf = nullptr;  // BF16 weights in fragment order
    long long step = 0;
    std::mutex launch;
};

namespace {
int mlp_fail(int code, const std::string &m) {
    sht::set_last_error(m);
    return code;
}
struct Dev {
    int prev = -1;
    bool ch = false;
    explicit Dev(int d) {
        if (hipGetDevice(&prev) == hipSuccess && prev != d) ch = hipSetDevice(d) == hipSuccess;
    }
    ~Dev() {
        if (ch) (void)hipSetDevice(prev);
    }
};
void mlp_free(sht_mlp *m) {
    if (!m) return;
    for (void *p : {(void *)m->P, (void *)m->M, (void *)m->V, (void *)m->Gp, (void *)m->Lp, (void *)m->loss,
                    (void *)m->Wf})
        if (p) (void)hipFree(p);
    delete m;
}
hipStream_t st(void *s) { return reinterpret_cast<hipStream_t>(s); }
}  // namespace

extern "C" {

int sht_mlp_nparams(void) { return kMlpParams; }

int sht_mlp_create(int32_t device, int32_t max_batch, sht_mlp **out) {
    if (!out || max_batch < 1) return mlp_fail(SHT_ERR_ARG, "bad arguments");
    *out = nullptr;
    sht_mlp *m = new (std::nothrow) sht_mlp();
    if (!m) return mlp_fail(SHT_ERR_ALLOC, "host allocation failed");
    m->device = device;
    m->max_batch = max_batch;
    Dev g(device);
    // partial gradients of the largest batch: at most kMaxGradBlocks workgroups, and never
    // more than one per row tile
    const int nblk = std::min(kMaxGradBlocks, (max_batch + kGradRows - 1) / kGradRows);
    struct A {
        void **p;
        size_t bytes;
    } allocs[] = {{(void **)&m->P, kMlpParams * 4},
                  {(void **)&m->M, kMlpParams * 4},
                  {(void **)&m->V, kMlpParams * 4},
                  {(void **)&m->Gp, (size_t)nblk * kMlpParams * 4},
                  {(void **)&m->Lp, (size_t)nblk * 4},
                  {(void **)&m->loss, 4},
                  {(void **)&m->Wf, (size_t)kFrags * 512 * 2}};
    for (auto &a : allocs) {
        if (hipMalloc(a.p, a.bytes) != hipSuccess) {
            mlp_free(m);
            return mlp_fail(SHT_ERR_ALLOC, "hipMalloc failed");
        }
    }
    if (hipMemset(m->M, 0, kMlpParams * 4) != hipSuccess || hipMemset(m->V, 0, kMlpParams * 4) != hipSuccess) {
        mlp_free(m);
        return mlp_fail(SHT_ERR_HIP, "hipMemset failed");
    }
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(&mlp_gradient_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kGradLds) != hipSuccess) {
        mlp_free(m);
        return mlp_fail(SHT_ERR_HIP, "hipFuncSetAttribute failed");
    }
    *out = m;
    return SHT_OK;
}

int sht_mlp_set_params(sht_mlp *m, const float *host_params) {
    if (!m || !host_params) return mlp_fail(SHT_ERR_ARG, "bad arguments");
    Dev g(m->device);
    if (hipMemcpy(m->P, host_params, kMlpParams * 4, hipMemcpyHostToDevice) != hipSuccess)
        return mlp_fail(SHT_ERR_HIP, "hipMemcpy failed");
    mlp_cast_kernel<<<(kMlpParams + 255) / 256, 256>>>(m->P, m->Wf);
    (void)hipMemset(m->M, 0, kMlpParams * 4);
    (void)hipMemset(m->V, 0, kMlpParams * 4);
    m->step = 0;
    return hipDeviceSynchronize() == hipSuccess ? SHT_OK : mlp_fail(SHT_ERR_HIP, "kernel failed");
}

int sht_mlp_get_params(sht_mlp *m, float *host_params) {
    if (!m || !host_params) return mlp_fail(SHT_ERR_ARG, "bad arguments");
    Dev g(m->device);
    return hipMemcpy(host_params, m->P, kMlpParams * 4, hipMemcpyDeviceToHost) == hipSuccess
               ? SHT_OK
               : mlp_fail(SHT_ERR_HIP, "hipMemcpy failed");
}

int sht_mlp_forward(sht_mlp *m, const float *x, float *y, int32_t B, void *stream) {
    if (!m || !x || !y || B < 1) return mlp_fail(SHT_ERR_ARG, "bad arguments");
    Dev g(m->device);
    const int nblk = (B + 63) / 64;  // four waves of 16 rows
    mlp_forward_kernel<<<nblk, 256, 0, st(stream)>>>(m->Wf, m->P, x, y, B);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? SHT_OK : mlp_fail(SHT_ERR_HIP, hipGetErrorString(e));
}

// Partial gradients and losses (into Gp, Lp), then their sum into grad (adam null) or an Adam step.
static int mlp_grad(sht_mlp *m, const float *x, const float *t, int B, float *grad, float *loss,
                    const AdamArgs *adam, float *Gp, float *Lp, void *stream) {
    int tiles = 0;
    const int nblk = grad_blocks(B, tiles);
    std::lock_guard<std::mutex> lock(m->launch);  // another thread's pair may use the same partials
    mlp_gradient_kernel<<<nblk, kGradThreads, kGradLds, st(stream)>>>(m->Wf, m->P, x, t, Gp, Lp, B, tiles);
    const int rblk = (kMlpParams + 63) / 64;
    if (adam)
        mlp_reduce_kernel<true><<<rblk, 256, 0, st(stream)>>>(Gp, nullptr, Lp, loss, nblk, B, *adam);
    else
        mlp_reduce_kernel<false><<<rblk, 256, 0, st(stream)>>>(Gp, grad, Lp, loss, nblk, B, AdamArgs{});
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? SHT_OK : mlp_fail(SHT_ERR_HIP, hipGetErrorString(e));
}

int sht_mlp_gradient(sht_mlp *m, const float *x, const float *t, int32_t B, float *grad, float *loss, void *stream) {
    if (!m || !x || !t || !grad || !loss || B < 1 || B > m->max_batch) return mlp_fail(SHT_ERR_ARG, "bad arguments");
    Dev g(m->device);
    return mlp_grad(m, x, t, B, grad, loss, nullptr, m->Gp, m->Lp, stream);
}

int64_t sht_mlp_scratch_bytes(int32_t B) {
    int tiles = 0;
    return B < 1 ? 0 : (int64_t)grad_blocks(B, tiles) * (kMlpParams + 1) * 4;
}

int sht_mlp_gradient_scratch(sht_mlp *m, const float *x, const float *t, int32_t B, float *grad, float *loss,
                             void *scratch, void *stream) {
    if (!m || !x || !t || !grad || !loss || !scratch || B < 1 || B > m->max_batch)
        return mlp_fail(SHT_ERR_ARG, "bad arguments");
    Dev g(m->device);
    int tiles = 0;
    float *Gp = static_cast<float *>(scratch);
    return mlp_grad(m, x, t, B, grad, loss, nullptr, Gp, Gp + (size_t)grad_blocks(B, tiles) * kMlpParams, stream);
}

int sht_mlp_train_step(sht_mlp *m, const float *x, const float *t, int32_t B, float lr, float *loss, void *stream) {
    if (!m || !x || !t || B < 1 || B > m->max_batch) return mlp_fail(SHT_ERR_ARG, "bad arguments");
    Dev g(m->device);
    m->step += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - powf(b1, (float)m->step), c2 = 1.f - powf(b2, (float)m->step);
    const AdamArgs adam{m->P, m->Wf, m->M, m->V, lr, b1, b2, 1e-8f, c1, c2};
    const int rc = mlp_grad(m, x, t, B, nullptr, loss ? loss : m->loss, &adam, m->Gp, m->Lp, stream);
    if (rc) m->step -= 1;
    return rc;
}

int sht_mlp_destroy(sht_mlp *m) {
    if (!m) return SHT_OK;
    Dev g(m->device);
    (void)hipDeviceSynchronize();
    mlp_free(m);
    return SHT_OK;
}

}  // extern "C"
