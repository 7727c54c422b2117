// Linear-field features of the learned second-order surrogate and the
// assembly of its output (no counterpart in the reference).
//
// Per column (x, y) at time t, in two passes over the components:
//   pass 1: eta1, its slopes d eta1/dx, d eta1/dy and the first-order Taylor
//           gradients at z = 0 (Irregular.cpp:178-293 terms: A, -A k cos(theta_dir),
//           phi1_d*dz);
//   pass 2: u1, v1, w1 and the first-order dynamic pressure p1 at the nlev
//           levels z_l = eta1 + sigma_l (h + eta1), profiles at min(0, z_l)
//           and the Taylor term times max(0, z_l) (the s-grid's first-order
//           column semantics with the linear elevation).
// Outputs per column: features X = [eta1, eta1_x, eta1_y, (u1, v1, w1) at
// every fstride-th level, h, kp] and the linear fields
// Lin = [eta1, (u1, v1, w1, p1) at every level].
#include <hip/hip_runtime.h>

#include <cstring>
#include <memory>
#include <type_traits>

#include "engine.hpp"
#include "../../include/cfdwm.h"

namespace cfdwm {

namespace {

constexpr double kInv2PiS = 0.15915494309189533577;

__device__ __forceinline__ double s_ramp(double t, double rt, double ts, double du) {
    const double a = 1. - ((t - ts - du + rt) / (rt + 1e-12));
    const double b = (t - ts) / (rt + 1e-12);
    const double down = a < 1. ? (a < 0. ? 0. : a) : 1.;
    const double up = b < 1. ? (b < 0. ? 0. : b) : 1.;
    return up * down;
}
__device__ __forceinline__ void s_cs(double ph, double& c, double& s) { sincos(ph, &s, &c); }
__device__ __forceinline__ void s_cs(double ph, float& c, float& s) {
    double r = ph * kInv2PiS;
    r -= rint(r);
    const float f = (float)r;
    s = __builtin_amdgcn_sinf(f);
    c = __builtin_amdgcn_cosf(f);
}
__device__ __forceinline__ double s_exp(double a) { return exp(a); }
__device__ __forceinline__ float s_exp(float a) { return __builtin_amdgcn_exp2f(a); }
__device__ __forceinline__ void s_prof(double pk, double pg, double z, double& E, double& G) {
    E = exp(pk * z);
    G = exp(fma(-pk, z, pg));
}
__device__ __forceinline__ void s_prof(float pk, float pg, float z, float& E, float& G) {
    E = __builtin_amdgcn_exp2f(pk * z);
    G = __builtin_amdgcn_exp2f(fmaf(-pk, z, pg));
}

// read-only records through scalar loads (the component index is wave-uniform)
template <typename T>
__device__ __forceinline__ T s_const(const T* p, int i) {
#if defined(__HIP_DEVICE_COMPILE__)
    return ((const __attribute__((address_space(4))) T*)p)[i];
#else
    return p[i];                              // host pass: never executed
#endif
}

// Vector-issue bound (16 levels x up to two exponentials and four products per
// component and column).  What is the same for every column -- a component's
// ramp (two FP64 divisions), its products with cos and sin of the direction --
// is computed once a block, kSurrCh components at a time through LDS; one
// phase serves all levels of the second pass; and e^{-k(z+2h)} is left out of
// four levels of a block of components where it lies below half a unit in the
// last place of e^{kz} at every column of the wave for the block's smallest k,
// so that sum and difference with it are e^{kz} itself: results are bit for
// bit those of the plain sums.  (Tested per block: a test per component splits
// the level loop into short pieces, 3060 us.)  512 x 512
// columns of 1,024 components: 3985 -> 2118 us.
constexpr int kSurrCh = 256;
template <typename R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void k_surr_linear(SeaDev<R> S, SurrJob J) {
    // levels a thread carries at once; components whose terms meet in R before
    // a fold into the FP64 totals (FP32: 8, the outputs are FP32; FP64: none)
    constexpr int LC = sizeof(R) == 4 ? 16 : 8;
    constexpr int BLK = sizeof(R) == 4 ? 8 : 1;
    // exponent (base 2, base e) of a G that leaves E + G and E - G at E
    constexpr R kNone = sizeof(R) == 4 ? (R)-28 : (R)-39.6;
    __shared__ __align__(16) R rec[kSurrCh][8];
    __shared__ R cs[BLK][2][256];
    const int tid = threadIdx.x;
    const int64_t q0 = (int64_t)blockIdx.x * blockDim.x + tid;
    const bool live = q0 < J.n;
    const int64_t q = live ? q0 : J.n - 1;
    const double dx = J.x[q] - S.x0, dy = J.y[q] - S.y0, t = J.t;
    double e1 = 0, sx = 0, sy = 0, gx = 0, gy = 0, gz = 0, gp = 0;
    double eh = 0, hx = 0, hy = 0;                 // quadrature (Hilbert pair) of eta1 and its slopes
    for (int c0 = 0; c0 < S.n; c0 += kSurrCh) {
        const int cn = S.n - c0 < kSurrCh ? S.n - c0 : kSurrCh;
        __syncthreads();
        if (tid < cn) {
            const PhaseRec ph = S.ph[c0 + tid];
            const CompRec<R>& c = S.cr[c0 + tid];
            const R ak = c.A * (R)ph.k;
            R* o = rec[tid];
            o[0] = (R)s_ramp(t, ph.rt, ph.ts, ph.du);
            o[1] = c.A;
            o[2] = ak * (R)ph.cth;
            o[3] = ak * (R)ph.sth;
            o[4] = c.gxz; o[5] = c.gyz; o[6] = c.gzz; o[7] = c.gpz;
        }
        __syncthreads();
        // four components' records on their way together
#pragma unroll 4
        for (int i = 0; i < cn; ++i) {
            const PhaseRec ph = s_const(S.ph, c0 + i);
            const R* c = rec[i];
            R ci, si;
            s_cs(ph.k * (ph.cth * dx + ph.sth * dy) - ph.omega * t + ph.ph0, ci, si);
            const R cr = ci * c[0], sr = si * c[0];
            e1 += (double)(c[1] * cr);
            sx -= (double)(c[2] * sr);
            sy -= (double)(c[3] * sr);
            gx += (double)(c[4] * cr);
            gy += (double)(c[5] * cr);
            gz += (double)(c[6] * sr);
            gp += (double)(c[7] * cr);
            eh += (double)(c[1] * sr);
            hx += (double)(c[2] * cr);
            hy += (double)(c[3] * cr);
        }
    }
    float* X = J.X + q * J.xstride;
    float* L = J.Lin + q * (1 + 4 * J.nlev);
    if (live) {
        if (J.quad) {
            X[J.nx] = (float)eh; X[J.nx + 1] = (float)hx; X[J.nx + 2] = (float)hy;
        }
        X[0] = (float)e1; X[1] = (float)sx; X[2] = (float)sy;
        X[J.nx - 2] = (float)J.h;
        X[J.nx - 1] = (float)J.kp;
        L[0] = (float)e1;
    }
    for (int l0 = 0; l0 < J.nlev; l0 += LC) {
        double U[LC], V[LC], W[LC], P[LC];
        R zp[LC], zl[LC / 4];                      // levels, and the lowest of each four
#pragma unroll
        for (int l = 0; l < LC; ++l) {
            const int lv = l0 + l < J.nlev ? l0 + l : J.nlev - 1;
            const double z = e1 + J.sigma[lv] * (J.h + e1);
            zp[l] = (R)(z < 0. ? z : 0.);
            zl[l / 4] = l % 4 == 0 || zp[l] < zl[l / 4] ? zp[l] : zl[l / 4];
            U[l] = V[l] = W[l] = P[l] = 0.;
        }
        for (int c0 = 0; c0 < S.n; c0 += kSurrCh) {
            const int cn = S.n - c0 < kSurrCh ? S.n - c0 : kSurrCh;
            __syncthreads();
            if (tid < cn) {
                const PhaseRec ph = S.ph[c0 + tid];
                const CompRec<R>& c = S.cr[c0 + tid];
                R* o = rec[tid];
                o[0] = (R)s_ramp(t, ph.rt, ph.ts, ph.du);
                o[1] = c.lu; o[2] = c.lv; o[3] = c.lw; o[4] = c.lp; o[5] = c.pk; o[6] = c.pg;
            }
            // the smallest k of each BLK components beside them
            R km = tid < cn ? rec[tid][5] : (R)1e30;
#pragma unroll
            for (int d = 1; d < BLK; d *= 2) {
                const R o = __shfl_xor(km, d);
                km = o < km ? o : km;
            }
            if (tid < cn) rec[tid][7] = km;
            __syncthreads();
            for (int i0 = 0; i0 < cn; i0 += BLK) {
                const int bn = cn - i0 < BLK ? cn - i0 : BLK;
                auto phase = [&](int i) {
                    const PhaseRec ph = s_const(S.ph, c0 + i0 + i);
                    R ci, si;
                    s_cs(ph.k * (ph.cth * dx + ph.sth * dy) - ph.omega * t + ph.ph0, ci, si);
                    cs[i][0][tid] = ci * rec[i0 + i][0];
                    cs[i][1][tid] = si * rec[i0 + i][0];
                };
                if (bn == BLK) {
#pragma unroll
                    for (int i = 0; i < BLK; ++i) phase(i);
                } else {
                    for (int i = 0; i < bn; ++i) phase(i);
                }
                // a component's record and phase, read one ahead
                auto get = [&](R(&c)[8], int i) {
#pragma unroll
                    for (int k = 1; k < 7; ++k) c[k] = rec[i0 + i][k];
                    c[0] = cs[i][0][tid];
                    c[7] = cs[i][1][tid];
                };
#pragma unroll
                for (int h = 0; h < LC; h += 8) {
                    R Ub[8], Vb[8], Wb[8], Pb[8];
#pragma unroll
                    for (int l = 0; l < 8; ++l) Ub[l] = Vb[l] = Wb[l] = Pb[l] = 0;
                    // the block's components, G at the first ng levels
                    auto comps = [&](auto ng) {
                        R c[8], cx[8];
                        get(c, 0);
#pragma unroll 1
                        for (int i = 0; i < bn; ++i) {
                            get(cx, i + 1 < bn ? i + 1 : i);
                            const R cr = c[0], sr = c[7], pk = c[5], pg = c[6];
                            const R lu = c[1] * cr, lv = c[2] * cr, lw = c[3] * sr, lp = c[4] * cr;
#pragma unroll
                            for (int l = 0; l < 8; ++l) {
                                R ch, sh;
                                if (l < ng.value) {
                                    R E, G;
                                    s_prof(pk, pg, zp[h + l], E, G);
                                    ch = E + G;
                                    sh = E - G;
                                } else {
                                    ch = sh = s_exp(pk * zp[h + l]);
                                }
                                Ub[l] += lu * ch;
                                Vb[l] += lv * ch;
                                Wb[l] += lw * sh;
                                Pb[l] += lp * ch;
                            }
#pragma unroll
                            for (int k = 0; k < 8; ++k) c[k] = cx[k];
                        }
                    };
                    // (the exponent of G / E is largest for the block's smallest k)
                    const R kl = (R)-2 * rec[i0][7], hz = (R)S.h;
                    const bool lo = __any(!(kl * (hz + zl[h / 4]) < kNone));
                    const bool hi = __any(!(kl * (hz + zl[h / 4 + 1]) < kNone));
                    if (hi) comps(std::integral_constant<int, 8>{});
                    else if (lo) comps(std::integral_constant<int, 4>{});
                    else comps(std::integral_constant<int, 0>{});
#pragma unroll
                    for (int l = 0; l < 8; ++l) {
                        U[h + l] += (double)Ub[l];
                        V[h + l] += (double)Vb[l];
                        W[h + l] += (double)Wb[l];
                        P[h + l] += (double)Pb[l];
                    }
                }
            }
        }
        if (!live) continue;
#pragma unroll
        for (int l = 0; l < LC; ++l) {
            const int lv = l0 + l;
            if (lv >= J.nlev) break;
            const double z = e1 + J.sigma[lv] * (J.h + e1), zt = z > 0. ? z : 0.;
            const float u = (float)(U[l] + gx * zt), v = (float)(V[l] + gy * zt);
            const float w = (float)(W[l] + gz * zt), p = (float)(P[l] + gp * zt);
            L[1 + 4 * lv] = u; L[2 + 4 * lv] = v; L[3 + 4 * lv] = w; L[4 + 4 * lv] = p;
            if (lv % J.fstride == 0) {
                const int f = 3 + 3 * (lv / J.fstride);
                X[f] = u; X[f + 1] = v; X[f + 2] = w;
            }
        }
    }
}

// X[q][col] = src[q] (row stride `stride`): a column of FP64 values into an FP32 matrix
__global__ void k_surr_set_column(int64_t n, const double* __restrict__ src, float* __restrict__ X, int stride,
                                  int col) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) X[q * stride + col] = (float)src[q];
}

// out = lin + pred elementwise (the surrogate's total fields)
__global__ void k_surr_add(int64_t n, const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ o) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) o[i] = a[i] + b[i];
}

}  // namespace

int surrogate_linear(Sea& s, const SurrJob& J) {
    hipStream_t st = Engine::get().stream();
    const unsigned nb = (unsigned)((J.n + 255) / 256);
    if (J.n <= 0) return 0;
    if (s.prec == kFP32)
        hipLaunchKernelGGL((k_surr_linear<float>), dim3(nb), dim3(256), 0, st, s.dev<float>(), J);
    else
        hipLaunchKernelGGL((k_surr_linear<double>), dim3(nb), dim3(256), 0, st, s.dev<double>(), J);
    CFDWM_HIP(hipGetLastError());
    return 0;
}

int surrogate_set_column(int64_t n, const double* src, float* X, int stride, int col) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_surr_set_column, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, Engine::get().stream(),
                       n, src, X, stride, col);
    CFDWM_HIP(hipGetLastError());
    return 0;
}

int surrogate_add(int64_t n, const float* a, const float* b, float* o) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_surr_add, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, Engine::get().stream(), n, a, b, o);
    CFDWM_HIP(hipGetLastError());
    return 0;
}

}  // namespace cfdwm
