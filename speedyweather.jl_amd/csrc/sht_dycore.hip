// Kernels of the minimal dry primitive-equation core around its transforms: one pass each for
// the columns of the spectral -> grid transform, the grid-point tendencies, the spectral
// tendencies and the time step.  Formulation and citations: dycore.py.
//
// Every kernel is a single pass bound by memory (large ensembles) or by its launch (T31).
// Written as array operations, a step was about 190 kernels of 2-7 us with the host issuing
// them, 1.1 ms per step at T31 with 8 members; with these kernels around the four of the
// two transforms it is 47 us (T127, 8 members: 1.2 ms -> 0.19 ms).  The kernels keep the array
// operations' rounding (no contraction to FMA) and give bit for bit what they give, but for the
// geopotential: a sum of products by FMA here, a matrix product there, which moves the last
// digits of the divergence tendency.
#include <algorithm>

#include "sht_device.h"
#include "sht_dycore.h"

namespace sht {

namespace {

constexpr int kMaxGridY = 65535;  // columns past it: the kernels loop over columns

__device__ __forceinline__ float2 cneg_i(float m, float2 q) { return make_float2(-m * q.y, m * q.x); }  // i m q

// Columns of the spectral -> grid transform of a state (EL = E L): U, V (EL each), the
// longitudinal derivative and cos(lat) times the latitudinal derivative of ln ps (E each),
// temperature, divergence, vorticity (EL each), ln ps (E).
__global__ __launch_bounds__(256) void dry_columns_kernel(const DevPlan *__restrict__ PP, const float2 *__restrict__ vor_,
                                                          const float2 *__restrict__ div_,
                                                          const float2 *__restrict__ temp_,
                                                          const float2 *__restrict__ lnps_, float2 *__restrict__ out_,
                                                          int EL, int E, float radius) {
#pragma clang fp contract(off)
    const DevPlan &P = *PP;
    const int nharm = P.nharm, lm = blockIdx.x * blockDim.x + threadIdx.x;
    if (lm >= nharm) return;
    SHT_GLOBAL float2 *out = as_global(out_) + lm;
    auto at = [&](int r) { return out + (long long)r * nharm; };
    for (int row = blockIdx.y; row < EL + E; row += gridDim.y) {
        if (row < EL) {
            const long long o = (long long)row * nharm;
            const SHT_GLOBAL float2 *vor = as_global(vor_) + o, *div = as_global(div_) + o;
            const float2 T = gload(as_global(temp_) + o + lm), D = gload(div + lm), Z = gload(vor + lm);
            float2 U, V;
            uv_stencil(P, vor, div, lm, U, V);
            gstore(at(row), make_float2(U.x * radius, U.y * radius));
            gstore(at(EL + row), make_float2(V.x * radius, V.y * radius));
            gstore(at(2 * EL + 2 * E + row), T);
            gstore(at(3 * EL + 2 * E + row), D);
            gstore(at(4 * EL + 2 * E + row), Z);
        } else {
            const int e = row - EL;
            const SHT_GLOBAL float2 *q = as_global(lnps_) + (long long)e * nharm;
            const float2 z = gload(q + lm), lo = gload(q + max(lm - 1, 0)), hi = gload(q + min(lm + 1, nharm - 1));
            const float4 gy = gload(as_global(P.gy) + lm);  // zero factors across orders
            gstore(at(2 * EL + e), cneg_i(gload(as_global(P.gx) + lm).y, z));
            gstore(at(2 * EL + E + e), make_float2(gy.z * lo.x + gy.w * hi.x, gy.z * lo.y + gy.w * hi.y));
            gstore(at(5 * EL + 2 * E + e), z);
        }
    }
}

// Grid-point tendencies, one thread per (point, member): g holds the columns above on the grid
// (u, v and the ln ps gradient divided by cos(lat); ln ps not needed), fields takes Au, Av, u T,
// v T (each over cos(lat)), kinetic energy, temperature tendency (EL columns each) and the ln ps
// tendency (E).  The vertical sums run over the levels in registers; LT levels known at compile
// time (LT = 0: L levels, the second sweep reads its values again).
template <int LT>
__global__ __launch_bounds__(256) void dry_grid_kernel(const float *__restrict__ g_, float *__restrict__ fields_,
                                                       const float *__restrict__ coslat_inv_,
                                                       const float *__restrict__ coriolis_, int npoints, int Lrt, int E,
                                                       float rinv, float r_dry, float kappa) {
#pragma clang fp contract(off)
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npoints) return;
    const int L = LT ? LT : Lrt;
    const long long np = npoints, EL = (long long)E * L;
    const float ci = as_global(coslat_inv_)[p], f = as_global(coriolis_)[p];
    const float ds = 1.f / (float)L, h = 0.5f * (float)L;  // layer thickness; 1 / (2 ds), exactly
    for (int e = blockIdx.y; e < E; e += gridDim.y) {
        const SHT_GLOBAL float *g = as_global(g_) + p;
        const SHT_GLOBAL float *gq = g + 2 * EL * np;
        const float qx = gq[e * np] * rinv, qy = gq[(E + e) * np] * rinv;
        const SHT_GLOBAL float *gu = g + (long long)e * L * np, *gv = gu + EL * np;
        const SHT_GLOBAL float *gT = gv + (EL + 2 * E) * np, *gD = gT + EL * np, *gZ = gD + EL * np;
        constexpr int N = LT ? LT : 1;
        float u_[N], v_[N], T_[N], D_[N], Z_[N];
        if constexpr (LT > 0) {
#pragma unroll
            for (int k = 0; k < LT; ++k) {
                u_[k] = gu[k * np];
                v_[k] = gv[k * np];
                T_[k] = gT[k * np];
                D_[k] = gD[k * np];
                Z_[k] = gZ[k * np];
            }
        }
        auto U = [&](int k) { if constexpr (LT > 0) return u_[k]; else return gu[k * np]; };
        auto V = [&](int k) { if constexpr (LT > 0) return v_[k]; else return gv[k * np]; };
        auto T = [&](int k) { if constexpr (LT > 0) return T_[k]; else return gT[k * np]; };
        auto D = [&](int k) { if constexpr (LT > 0) return D_[k]; else return gD[k * np]; };
        auto Z = [&](int k) { if constexpr (LT > 0) return Z_[k]; else return gZ[k * np]; };
        float total = 0.f;  // vertically integrated mass-flux divergence
        auto integrate = [&](int k) { total += ds * (D(k) + (U(k) * qx + V(k) * qy)); };
        SHT_GLOBAL float *o = as_global(fields_) + p + (long long)e * L * np;
        const long long gs = EL * np;  // one group of EL columns
        float lnps_t = 0.f, csum = 0.f;
        float fu = 0.f, fv = 0.f, fT = 0.f;  // vertical fluxes through the level's upper face
        float u = U(0), v = V(0), t = T(0);
        auto level = [&](int k) {
            const float d = D(k), uq = u * qx + v * qy, dsum = ds * (d + uq);
            csum += dsum;
            float fu1 = 0.f, fv1 = 0.f, fT1 = 0.f, un = 0.f, vn = 0.f, tn = 0.f;
            if (k + 1 < L) {
                un = U(k + 1);
                vn = V(k + 1);
                tn = T(k + 1);
                const float sdot = -csum - ((float)(k + 1) / (float)L) * lnps_t;
                fu1 = sdot * (un - u);
                fv1 = sdot * (vn - v);
                fT1 = sdot * (tn - t);
            }
            const float omp = uq - (csum - 0.5f * dsum) / (((float)k + 0.5f) / (float)L);  // omega / p
            const float av = Z(k) + f, rt = r_dry * t;
            o[0] = (av * v - (fu1 + fu) * h - rt * qx) * ci;
            o[gs] = (-av * u - (fv1 + fv) * h - rt * qy) * ci;
            o[2 * gs] = u * t * ci;
            o[3 * gs] = v * t * ci;
            o[4 * gs] = 0.5f * (u * u + v * v);
            o[5 * gs] = t * d - (fT1 + fT) * h + kappa * t * omp;
            o += np;
            fu = fu1, fv = fv1, fT = fT1;
            u = un, v = vn, t = tn;
        };
        if constexpr (LT > 0) {
#pragma unroll
            for (int k = 0; k < LT; ++k) integrate(k);
            lnps_t = -total;
#pragma unroll
            for (int k = 0; k < LT; ++k) level(k);
        } else {
            for (int k = 0; k < L; ++k) integrate(k);
            lnps_t = -total;
            for (int k = 0; k < L; ++k) level(k);
        }
        (as_global(fields_) + p + 6 * gs)[e * np] = lnps_t;
    }
}

// Time step of one coefficient: new = (base + dt2 tend) / (1 + dt2 nu), and with a previous
// state (base = b, else base = x) the Robert-Asselin-Williams filter of the present one, x.
__device__ __forceinline__ void dry_step(float2 x, float2 b, float2 t, float damp, float dt2, float w1, float w2,
                                         int filter, SHT_GLOBAL float2 *now1, SHT_GLOBAL float2 *next) {
#pragma clang fp contract(off)
    const float rd = 1.f / damp;
    float2 y = make_float2((b.x + dt2 * t.x) * rd, (b.y + dt2 * t.y) * rd);
    if (filter) {
        const float2 d = make_float2(b.x - 2.f * x.x + y.x, b.y - 2.f * x.y + y.y);
        gstore(now1, make_float2(x.x + w1 * d.x, x.y + w1 * d.y));
        y = make_float2(y.x - w2 * d.x, y.y - w2 * d.y);
    }
    gstore(next, y);
}

// Spectral tendencies (columns: vorticity, divergence, temperature EL each, ln ps E) from the
// analysed fields s (columns of dry_grid_kernel) and the temperature (geopotential, G L x L
// with zeros below the diagonal); ri, rr: the radius's reciprocal and its square's, rounded from
// 64 bits as the array operations round them.  One thread per coefficient and level.  LT levels known at
// compile time: the temperatures of the levels below are all in flight at once (8 members and
// levels: T31 5.2 -> 3.8 us, T127 13.6 -> 12.7); LT = 0: L levels, one load after another.
// STEP: the tendencies are not stored but applied (dry_step), one pass over the state instead of
// two (8 members and levels: T31 3.8 + 3.4 -> 4.8 us, T127 12.7 + 12.4 -> 19.6).
template <int LT, bool STEP>
__global__ __launch_bounds__(256) void dry_tendency_kernel(const DevPlan *__restrict__ PP, const float2 *__restrict__ s_,
                                                           const float2 *__restrict__ temp_,
                                                           const float *__restrict__ G_, float2 *__restrict__ tend_,
                                                           int Lrt, int E, float ri, float rr, DryStep S) {
#pragma clang fp contract(off)
    const int L = LT > 0 ? LT : Lrt;
    const DevPlan &P = *PP;
    const int nharm = P.nharm, lm = blockIdx.x * blockDim.x + threadIdx.x;
    if (lm >= nharm) return;
    const long long nh = nharm, EL = (long long)E * L;
    const SHT_GLOBAL float2 *s = as_global(s_) + lm;
    SHT_GLOBAL float2 *tend = as_global(tend_) + lm;
    const int l = as_global(P.l_of)[lm];
    const float keep = l == P.lmax - 1 ? 0.f : 1.f;  // the extra degree has no prognostic tendency
    // tendency t of prognostic field f, column `row` of all
    auto put = [&](int f, long long row, float2 t, float2 x, float2 b) {
        if constexpr (STEP) {
            const float damp = f == 3 ? 1.f : 1.f + S.dt2 * (f == 1 ? as_global(S.nu_div) : as_global(S.nu))[lm];
            dry_step(x, b, t, damp, S.dt2, S.w1, S.w2, S.filter, as_global(S.now1) + lm + row * nh,
                     as_global(S.next) + lm + row * nh);
        } else {
            gstore(tend + row * nh, t);
        }
    };
    auto state = [&](const float2 *now, const float2 *prev, long long col, float2 &x, float2 &b) {
        if constexpr (STEP) {
            x = b = gload(as_global(now) + lm + col * nh);
            if (S.filter) b = gload(as_global(prev) + lm + col * nh);  // uniform
        }
    };
    for (int row = blockIdx.y; row < EL + E; row += gridDim.y) {
        if (row >= EL) {
            const int e = row - (int)EL;
            const float2 q = gload(s + (6 * EL + e) * nh);
            const float w = lm == 0 ? 0.f : keep;  // mass conservation: the mean of ln ps stays
            float2 x = q, b = q;
            state(S.now.lnps, S.prev.lnps, e, x, b);
            put(3, 3 * EL + e, make_float2(q.x * w, q.y * w), x, b);
            continue;
        }
        const int e = row / L, k = row - e * L;
        const int dm = lm > 0 ? -1 : 0, dp = lm + 1 < nharm ? 1 : 0;
        const SHT_GLOBAL float2 *a = s + row * nh;
        const float2 u = gload(a), um = gload(a + dm), up = gload(a + dp);
        a += EL * nh;
        const float2 v = gload(a), vm = gload(a + dm), vp = gload(a + dp);
        a += EL * nh;
        const float2 uT = gload(a);
        a += EL * nh;
        const float2 vTm = gload(a + dm), vTp = gload(a + dp);
        const float2 ke = gload(a + EL * nh), Tt = gload(a + 2 * EL * nh);
        const float4 gy = gload(as_global(P.gy) + lm);  // gy.x, gy.y, gx.x are zero at the last degree
        const float mx = gload(as_global(P.gx) + lm).x;
        float2 xz = u, bz = u, xd = u, bd = u, xt = u, bt = u;
        state(S.now.vor, S.prev.vor, row, xz, bz);
        state(S.now.div, S.prev.div, row, xd, bd);
        state(S.now.temp, S.prev.temp, row, xt, bt);
        float2 phi = make_float2(0.f, 0.f);
        const SHT_GLOBAL float2 *T = as_global(temp_) + (long long)e * L * nh + lm;
        const SHT_GLOBAL float *G = as_global(G_) + k * L;
        if constexpr (LT > 0) {
            float2 t[LT];
#pragma unroll
            for (int j = 0; j < LT; ++j)
                if (j >= k) t[j] = gload(T + j * nh);  // uniform
#pragma unroll
            for (int j = 0; j < LT; ++j)
                if (j >= k) {
                    phi.x = fmaf(G[j], t[j].x, phi.x);
                    phi.y = fmaf(G[j], t[j].y, phi.y);
                }
        } else {
            for (int j = k; j < L; ++j) {
                const float c = G[j];
                const float2 t = gload(T + j * nh);
                phi.x = fmaf(c, t.x, phi.x);
                phi.y = fmaf(c, t.y, phi.y);
            }
        }
        const float2 iu = cneg_i(mx, u), iv = cneg_i(mx, v), iuT = cneg_i(mx, uT);
        const float2 curl = make_float2(iv.x + gy.x * um.x - gy.y * up.x, iv.y + gy.x * um.y - gy.y * up.y);
        const float2 div = make_float2(iu.x - gy.x * vm.x + gy.y * vp.x, iu.y - gy.x * vm.y + gy.y * vp.y);
        const float2 divT = make_float2(iuT.x - gy.x * vTm.x + gy.y * vTp.x, iuT.y - gy.x * vTm.y + gy.y * vTp.y);
        const float eig = -(float)l * (float)(l + 1);
        const float2 lap = make_float2(eig * (phi.x + ke.x), eig * (phi.y + ke.y));
        put(0, row, make_float2(curl.x * ri * keep, curl.y * ri * keep), xz, bz);
        put(1, EL + row, make_float2((div.x * ri - lap.x * rr) * keep, (div.y * ri - lap.y * rr) * keep), xd, bd);
        put(2, 2 * EL + row, make_float2((-divT.x * ri + Tt.x) * keep, (-divT.y * ri + Tt.y) * keep), xt, bt);
    }
}

// Time step of every prognostic column from stored tendencies (a correction may have changed
// them).  Outputs: columns as the tendencies'.
__global__ __launch_bounds__(256) void dry_leapfrog_kernel(DryState now, DryState prev, const float2 *__restrict__ tend_,
                                                           const float *__restrict__ nu_,
                                                           const float *__restrict__ nu_div_, float2 *__restrict__ now1_,
                                                           float2 *__restrict__ next_, int nharm, int EL, int rows,
                                                           float dt2, float w1, float w2, int filter) {
#pragma clang fp contract(off)
    const int lm = blockIdx.x * blockDim.x + threadIdx.x;
    if (lm >= nharm) return;
    for (int row = blockIdx.y; row < rows; row += gridDim.y) {
        const int f = min(row / EL, 3);
        const long long in = (long long)(row - f * EL) * nharm + lm, out = (long long)row * nharm + lm;
        const float2 x = gload(as_global(f == 0 ? now.vor : f == 1 ? now.div : f == 2 ? now.temp : now.lnps) + in);
        const float2 t = gload(as_global(tend_) + out);
        float2 b = x;
        if (filter) b = gload(as_global(f == 0 ? prev.vor : f == 1 ? prev.div : f == 2 ? prev.temp : prev.lnps) + in);
        const float damp = f == 3 ? 1.f : 1.f + dt2 * (f == 1 ? as_global(nu_div_) : as_global(nu_))[lm];
        dry_step(x, b, t, damp, dt2, w1, w2, filter, as_global(now1_) + out, as_global(next_) + out);
    }
}

}  // namespace

int launch_dry_columns(const DevPlan *P, int nharm, const DryState &s, void *out, int L, int E, float radius,
                       void *stream) {
    const dim3 grid((nharm + 255) / 256, std::min(E * L + E, kMaxGridY));
    dry_columns_kernel<<<grid, 256, 0, as_stream(stream)>>>(P, s.vor, s.div, s.temp, s.lnps, static_cast<float2 *>(out),
                                                            E * L, E, radius);
    return (int)hipGetLastError();
}

int launch_dry_grid(const float *g, float *fields, const float *coslat_inv, const float *coriolis, int npoints, int L, int E,
                    float rinv, float r_dry, float kappa, void *stream) {
    const dim3 grid((npoints + 255) / 256, std::min(E, kMaxGridY));
    // the level count of the column network has its own instantiation: a step of 8 members and
    // levels takes 183 us at T127 and 51 at T31 with it (here and in launch_tendency), 192 and 57 on
    // the general one, which the other counts take (7 levels 166 us, 10 levels 233)
    if (L == 8)
        dry_grid_kernel<8><<<grid, 256, 0, as_stream(stream)>>>(g, fields, coslat_inv, coriolis, npoints, L, E, rinv,
                                                                r_dry, kappa);
    else
        dry_grid_kernel<0><<<grid, 256, 0, as_stream(stream)>>>(g, fields, coslat_inv, coriolis, npoints, L, E, rinv,
                                                                r_dry, kappa);
    return (int)hipGetLastError();
}

template <bool STEP>
static int launch_tendency(const DevPlan *P, int nharm, const void *s, const float2 *temp, const float *G, void *tend,
                           int L, int E, double radius, const DryStep &S, void *stream) {
    const dim3 grid((nharm + 255) / 256, std::min(E * L + E, kMaxGridY));
    auto *f = L == 8 ? &dry_tendency_kernel<8, STEP> : &dry_tendency_kernel<0, STEP>;
    f<<<grid, 256, 0, as_stream(stream)>>>(P, static_cast<const float2 *>(s), temp, G, static_cast<float2 *>(tend), L, E,
                                           (float)(1.0 / radius), (float)(1.0 / (radius * radius)), S);
    return (int)hipGetLastError();
}

int launch_dry_tendency(const DevPlan *P, int nharm, const void *s, const float2 *temp, const float *G, void *tend, int L,
                        int E, double radius, void *stream) {
    return launch_tendency<false>(P, nharm, s, temp, G, tend, L, E, radius, DryStep{}, stream);
}

int launch_dry_step(const DevPlan *P, int nharm, const void *s, const float *G, const DryStep &S, int L, int E,
                    double radius, void *stream) {
    return launch_tendency<true>(P, nharm, s, S.now.temp, G, nullptr, L, E, radius, S, stream);
}

int launch_dry_leapfrog(int nharm, const DryState &now, const DryState &prev, const void *tend, const float *nu,
                        const float *nu_div, void *now1, void *next, int L, int E, float dt2, float w1, float w2,
                        int filter, void *stream) {
    const dim3 grid((nharm + 255) / 256, std::min(3 * E * L + E, kMaxGridY));
    dry_leapfrog_kernel<<<grid, 256, 0, as_stream(stream)>>>(now, prev, static_cast<const float2 *>(tend), nu, nu_div,
                                                             static_cast<float2 *>(now1), static_cast<float2 *>(next),
                                                             nharm, E * L, 3 * E * L + E, dt2, w1, w2, filter);
    return (int)hipGetLastError();
}

}  // namespace sht
