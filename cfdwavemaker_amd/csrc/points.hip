// Unfiltered second-order kinematics (u2, v2, w2, dp2 with the first-order,
// Taylor and filtered eta2 terms of the same points; Irregular.cpp:178-293,
// 394-812, 1107-1192) at points of long-crested seas.
//
// Where every component runs in one direction and the components ascend in k,
// the combined wavenumbers of a pair i < m are k_m + k_i and k_m - k_i, so its
// depth profiles split:
//   e^{(k_m + k_i) z}        = E_i E_m,   e^{-(k_m + k_i)(z + 2h)} = g_i g_m
//   e^{(k_m - k_i) z}        = F_i X_m,   e^{-(k_m - k_i)(z + 2h)} = f_i x_m
// with E = e^{kz}, g = e^{-k(z+2h)}, X_m = e^{(k_m - kr) z}, F_i = e^{(kr - k_i) z}
// and so on, kr a wavenumber of the row's own block (neither factor leaves the
// number range, and their exponents are no larger than the pair's own near the
// diagonal, where the difference terms live).  The pair sums of a block of 16
// rows then are products of constant matrices (16 rows x components) with the
// per-point vectors cos(phi_m) E_m, sin(phi_m) E_m, ... : 18 matrix products
// on v_mfma_f32_16x16x4_f32 / v_mfma_f64_16x16x4_f64 serve u, v, w, p and
// eta2.  u, v and w share theirs: along the crest the u coefficient is the w
// coefficient times cos(theta) (sum) or -cos(theta) (difference).
//
// A wave owns 16 points x one run of (row block, 4 components) steps.  The
// lane (k = lane / 16, point = lane % 16) computes the sine, cosine and
// profiles of component 4 j + k at its point straight into the B operand's
// register: no LDS and no barrier; the operands of the next step load while
// this one runs (without that the loads cost a third of the time in FP64).
// What bounds it: the matrix instructions and the vector work of sines and
// exponentials together, which this chip's SIMDs do not overlap for FP32 and
// FP64 products (measured: 72 FP64 fused multiply-adds beside 18 products add
// their whole time, FP32 ones half of it).  16 rows a wave: their 18
// accumulators leave three waves a SIMD in FP32 and two in FP64; 32 would
// halve the sines per row and leave FP64 one wave.
//
// Measured against one thread a point walking the pairs (a sine, a cosine and
// four exponentials per pair): 131,072 points, 512 components, FP32 30.8 ->
// 6.9 ms (92 TFLOP/s on the matrix cores); 4,096 points, 256 components, FP64
// 1.4 ms -> 0.17 ms.  Error against 64 bits at the FP32 size 4.4e-6 -> 4.9e-7.
#include <hip/hip_runtime.h>

#include "device_math.hpp"
#include "engine.hpp"
#include "kernels.hpp"

namespace cfdwm {
namespace {

using dm::freq_ramp;

typedef float f4v __attribute__((ext_vector_type(4)));
typedef double d4v __attribute__((ext_vector_type(4)));

template <typename R> struct Acc;
template <> struct Acc<float> {
    using V = f4v;
    static __device__ __forceinline__ V mul(float a, float b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    // row of accumulator element r in a lane of group g
    static __device__ __forceinline__ int row(int g, int r) { return 4 * g + r; }
    static constexpr double kLim = 40.;       // exponents of one factor
};
template <> struct Acc<double> {
    using V = d4v;
    static __device__ __forceinline__ V mul(double a, double b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int g, int r) { return g + 4 * r; }
    static constexpr double kLim = 300.;
};

// A wavenumber or a depth as the exponentials take it: FP64 plain, FP32 as a
// pair of floats (wavenumbers times log2 e).  e^{k z} then is right to the
// working precision's last places: the rounding of the exponent is put back.
template <typename R> struct Hl;
template <> struct Hl<double> {
    double v;
    static __device__ __forceinline__ Hl k(double a) { return {a}; }
    static __device__ __forceinline__ Hl of(const PointRec& m) { return {m.k}; }
    static __device__ __forceinline__ Hl z(double a) { return {a}; }
};
template <> struct Hl<float> {
    float hi, lo;
    static __device__ __forceinline__ Hl z(double a) {
        const float h = (float)a;
        return {h, (float)(a - (double)h)};
    }
    static __device__ __forceinline__ Hl k(double a) { return z(a * 1.4426950408889634074); }
    static __device__ __forceinline__ Hl of(const PointRec& m) { return {m.khi, m.klo}; }
};
__device__ __forceinline__ double pe(Hl<double> k, Hl<double> z) {
    const double a = k.v * z.v, e = exp(a);
    return fma(e, fma(k.v, z.v, -a), e);
}
__device__ __forceinline__ float pe(Hl<float> k, Hl<float> z) {
    const float a = k.hi * z.hi;
    const float lo = fmaf(k.lo, z.hi, fmaf(k.hi, z.lo, fmaf(k.hi, z.hi, -a)));
    const float e = __builtin_amdgcn_exp2f(a);
    return fmaf(e, lo * 0.69314718f, e);
}

// sine and cosine of a component's phase
__device__ __forceinline__ void cs_at(const PointRec& m, double xa, double t, double& c, double& s) {
    // the phase itself as everywhere, brought to a revolution by 1 / 2 pi in two parts
    const double ph = m.k * xa - m.omega * t + m.ph0;
    const double n = rint(ph * 0.15915494309189535);
    const double r = fma(ph, -9.839338337591243e-18, fma(ph, 0.15915494309189535, -n));
    sincospi(r + r, &s, &c);
}
__device__ __forceinline__ void cs_at(const PointRec& m, double xa, double t, float& c, float& s) {
    const double r = fma(m.kr, xa, fma(-m.wr, t, m.pr));
    const float f = (float)(r - rint(r));
    s = __builtin_amdgcn_sinf(f);
    c = __builtin_amdgcn_cosf(f);
}

// the pair's own profile, for points outside the split's range
__device__ __forceinline__ void prof(double k, double z, double h, double& E, double& G) {
    E = exp(k * z);
    G = exp(-k * (z + 2. * h));
}
__device__ __forceinline__ void prof(double k, double z, double h, float& E, float& G) {
    const double s = 1.4426950408889634074;
    E = __builtin_amdgcn_exp2f((float)(k * s * z));
    G = __builtin_amdgcn_exp2f((float)(-k * s * (z + 2. * h)));
}

__device__ __forceinline__ double over_groups(double v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
}

// A row block's steps [a, b) pair by pair, each with its own exponentials:
// for waves with a point whose split exponents leave the number range.  Beside
// points far below the bed or far above the surface that is deep water, for
// points near the surface (z + 2h about 2h): in FP64 where kmax (z + 2h) > 600
// (components to 2.5 rad/s: from 470 m on, all row blocks), in FP32 where half
// a row block's spread of k times (z + 2h) exceeds 40 (evenly spaced
// frequencies from 0.3 to 2.5 rad/s: 48 components from 130 m on in the topmost
// of three row blocks, in all from 430 m; 128 from 320 m; 512 from 1200 m).
// What it costs there, 65,536 points at 500 m, against the pair loop with a
// thread a point (matrix path at 150 m): 48 components FP32 283 us, 248 (137),
// FP64 550, 597 (161); 128 FP32 676, 1030 (361), FP64 3.38 ms, 3.64 (0.57);
// 4,096 points 48 components FP32 58, 98 (52).  A lane takes
// its point's rows of group g.  Kept out of line: it would cost the matrix
// path its registers.
template <typename R>
struct PairSum {
    double U, W, P2, e2, K1, K2;
};
template <typename R>
__device__ __attribute__((noinline)) PairSum<R> pairs_one_by_one(const PhaseRec* ph, const PointRec* mr, const R* coef,
                                                                 int N, double h, int i0, int a, int b, double xa,
                                                                 double t, double z, int g, bool wp) {
    PairSum<R> o{0, 0, 0, 0, 0, 0};
    for (int r = 0; r < 4; ++r) {
        const int i = i0 + Acc<R>::row(g, r);
        if (i >= N) break;
        const PhaseRec p = ph[i];
        const PointRec q = mr[i];
        R c, s;
        cs_at(q, xa, t, c, s);
        const R ri = (R)freq_ramp(t, p.rt, p.ts, p.du), cr = c * ri, sr = s * ri;
        for (int mi = max(i0 + 4 * a, i + 1); mi < min(i0 + 4 * b, N); ++mi) {
            const PointRec m = mr[mi];
            R cm, sm, E, G;
            cs_at(m, xa, t, cm, sm);
            const R* cf = coef + ((mi - i0) >> 2) * 6 * 64 + ((mi - i0) & 3) * 16 + (i - i0);
            const R cP = cr * cm - sr * sm, cM = cr * cm + sr * sm;
            const R sP = sr * cm + cr * sm, sM = sr * cm - cr * sm;
            prof(m.k + p.k, z, h, E, G);
            o.U += (double)(cf[0] * cP * (E + G));
            o.W += (double)(cf[0] * sP * (E - G));
            o.P2 += (double)(cf[64] * cP * (E + G));
            prof(m.k - p.k, z, h, E, G);
            o.U -= (double)(cf[128] * cM * (E + G));
            o.W += (double)(cf[128] * sM * (E - G));
            o.P2 += (double)(cf[192] * cM * (E + G));
            o.e2 += (double)(cr * cm * cf[256] + sr * sm * cf[320]);
        }
    }
    if (wp)
        for (int mi = i0 + max(4 * a, 16) + g; mi < min(i0 + 4 * b, N); mi += 4) {
            const PointRec m = mr[mi];
            R E, G;
            prof(m.k, z, h, E, G);
            o.K1 += m.X * ((double)E + (double)G);
            o.K2 += m.X * ((double)E - (double)G);
        }
    return o;
}

// the point's outputs from its totals
__device__ __forceinline__ void point_store(const PointJob& J, int64_t q, const double* a) {
    const double z = J.z[q];
    const double z1 = z - J.swl > 0. ? z - J.swl : 0.;
    // (without the Taylor terms their gradients, which deep water may leave
    // without a value, stay out)
    const bool tay = (J.flags & EV_TAYLOR) != 0;
    if (J.o_eta1) J.o_eta1[q] = a[0];
    if (J.o_eta2) J.o_eta2[q] = J.want_eta2 ? a[1] : 0.;
    for (int k = 0; k < 4; ++k)
        if (J.o_g[k]) J.o_g[k][q] = a[2 + k];
    if (J.o_u) J.o_u[q] = a[6] + (tay ? a[2] * z1 : 0.);
    if (J.o_v) J.o_v[q] = a[7] + (tay ? a[3] * z1 : 0.);
    if (J.o_w) J.o_w[q] = a[8] + (tay ? a[4] * z1 : 0.);
    if (J.o_p) J.o_p[q] = a[9] + J.rho * a[10] + (tay ? a[5] * z1 : 0.);
}

template <typename R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 3 : 2)))
void k_point_forms(SeaDev<R> S, PointJob J) {
    using V = typename Acc<R>::V;
    const int lane = threadIdx.x & 63, g = lane >> 4, pt = lane & 15;
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int64_t q = ((int64_t)blockIdx.x * 4 + wv) * 16 + pt;
    const bool live = q < J.n;
    const int64_t qc = live ? q : J.n - 1;
    const int N = S.n, nrb = (N + 15) / 16;
    const double x = J.x[qc] - S.x0, y = J.y[qc] - S.y0, t = J.t[qc];
    const double xa = J.cth * x + J.sth * y;
    double z = J.z[qc];
    if (J.flags & EV_ZCLAMP) z = (z - J.swl) < 0. ? (z - J.swl) : 0.;
    else if (J.flags & EV_ZSHIFT) z = z - J.swl;
    if (sizeof(R) == 4) z = (double)(R)z;
    const double zb = -(z + 2. * S.h);
    const Hl<R> zh = Hl<R>::z(z), zbh = Hl<R>::z(zb);
    const bool lin = (J.flags & EV_LIN) != 0, wp = (J.flags & EV_P) != 0;
    const double L = fmax(fabs(z), fabs(zb)), up = J.kmax * fmax(z, zb);
    const int ns = J.nseg, sg = blockIdx.y;
    const int s0 = (int)((int64_t)J.steps * sg / ns), s1 = (int)((int64_t)J.steps * (sg + 1) / ns);
    // totals: e1 e2 gx gy gz gp U (along the crest) W P P2
    double e1 = 0, e2 = 0, gx = 0, gy = 0, gz = 0, gp = 0, U = 0, U1 = 0, V1 = 0, W = 0, P = 0, P2 = 0;
    int off = 0;
    for (int rb = 0; rb < nrb; ++rb) {
        const int cnt = (N - 16 * rb + 3) / 4;
        const int a = s0 - off > 0 ? s0 - off : 0, b = s1 - off < cnt ? s1 - off : cnt;
        const int base = off;
        off += cnt;
        if (a >= b) continue;
        const int i0 = 16 * rb, il = i0 + 15 < N ? i0 + 15 : N - 1;
        const double k0 = J.mr[i0].k, k1 = J.mr[il].k, kr = 0.5 * (k0 + k1);
        bool far = !(0.5 * (k1 - k0) * L <= Acc<R>::kLim && up <= Acc<R>::kLim);
        if (sizeof(R) == 8) far = far || !(J.kmax * L <= 600.);
        const bool slow = __any(far);
        V T[18];
#pragma unroll
        for (int v = 0; v < 18; ++v)
#pragma unroll
            for (int r = 0; r < 4; ++r) T[v][r] = 0;
        double K1 = 0, K2 = 0;
        double Ekr = 1, Gkr = 1;              // FP64: X_m = E_m e^{-kr z}, x_m = g_m e^{kr (z + 2h)}
        if (!slow) {
            if constexpr (sizeof(R) == 8) {
                Ekr = pe(Hl<R>::k(-kr), zh);
                Gkr = pe(Hl<R>::k(-kr), zbh);
            }
            // the components of the block itself first, then those past it,
            // which alone enter K1 and K2
            double KE = 0, KG = 0;
#pragma unroll 1
            for (int j0 = a; j0 < b;) {
                const int j1 = j0 < 4 && b > 4 ? 4 : b;
                const R* cf = (const R*)J.coef + (int64_t)base * 6 * 64 + lane;
                const PointRec* mp = J.mr + i0 + g;
                KE = KG = 0;
                // operands a step ahead, in two register sets
                auto load = [&](R(&A)[6], PointRec& m, int j) {
                    const R* p = cf + (int64_t)j * 6 * 64;
#pragma unroll
                    for (int v = 0; v < 6; ++v) A[v] = p[v * 64];
                    m = mp[4 * j];
                    __builtin_amdgcn_sched_barrier(0);
                };
                auto step = [&](const R(&A)[6], const PointRec& m) {
                    R c, s, X, Y;
                    cs_at(m, xa, t, c, s);
                    const Hl<R> km = Hl<R>::of(m);
                    const R E = pe(km, zh), G = pe(km, zbh);
                    if constexpr (sizeof(R) == 8) {
                        X = E * Ekr;
                        Y = G * Gkr;
                    } else {
                        const Hl<R> kd = Hl<R>::k(m.k - kr);
                        X = pe(kd, zh);
                        Y = pe(kd, zbh);
                    }
                    KE = fma(m.X, (double)E, KE);
                    KG = fma(m.X, (double)G, KG);
                    const R bP[4] = {c * E, c * G, s * E, s * G};
                    const R bM[4] = {c * X, c * Y, s * X, s * Y};
                    T[16] = Acc<R>::mul(A[4], c, T[16]);
                    T[17] = Acc<R>::mul(A[5], s, T[17]);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        T[v] = Acc<R>::mul(A[0], bP[v], T[v]);
                        T[4 + v] = Acc<R>::mul(A[1], bP[v], T[4 + v]);
                        T[8 + v] = Acc<R>::mul(A[2], bM[v], T[8 + v]);
                        T[12 + v] = Acc<R>::mul(A[3], bM[v], T[12 + v]);
                    }
                };
                R A0[6], A1[6];
                PointRec m0, m1;
                load(A0, m0, j0);
                int j = j0;
#pragma unroll 1
                for (; j + 1 < j1; j += 2) {
                    load(A1, m1, j + 1);
                    step(A0, m0);
                    load(A0, m0, j + 2 < j1 ? j + 2 : j + 1);
                    step(A1, m1);
                }
                if (j < j1) step(A0, m0);
                j0 = j1;
            }
            if (b > 4) {
                K1 = KE + KG;
                K2 = KE - KG;
            }
        }
        // ---- the block's 16 rows: contraction, and their own terms once
        const bool own = a == 0;
        double Bx = 0, Bz = 0, fx[4], fz[4], rr[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = i0 + Acc<R>::row(g, r);
            const bool val = i < N;
            const int ic = val ? i : N - 1;
            const PhaseRec p = S.ph[ic];
            R c, s, E, G;
            const PointRec pr = J.mr[ic];
            cs_at(pr, xa, t, c, s);
            const Hl<R> ki = Hl<R>::of(pr);
            E = pe(ki, zh);
            G = pe(ki, zbh);
            const double rid = val ? freq_ramp(t, p.rt, p.ts, p.du) : 0.;
            const R ri = (R)rid, cr = c * ri, sr = s * ri;
            const double X = pr.X;
            rr[r] = rid;
            fx[r] = val ? X * ((double)E + (double)G) : 0.;
            fz[r] = val ? X * ((double)E - (double)G) : 0.;
            Bx += rid * fx[r];
            Bz += rid * fz[r];
            if (!slow) {
                R F, f;
                if constexpr (sizeof(R) == 8) {
                    F = dm::rcp_nr(E * Ekr);
                    f = dm::rcp_nr(G * Gkr);
                } else {
                    const Hl<R> kd = Hl<R>::k(kr - pr.k);
                    F = pe(kd, zh);
                    f = pe(kd, zbh);
                }
                const R uc = E * T[0][r] + G * T[1][r], us = E * T[2][r] + G * T[3][r];
                const R wc = E * T[0][r] - G * T[1][r], ws = E * T[2][r] - G * T[3][r];
                const R pc = E * T[4][r] + G * T[5][r], ps = E * T[6][r] + G * T[7][r];
                const R vc = F * T[8][r] + f * T[9][r], vs = F * T[10][r] + f * T[11][r];
                const R xc = F * T[8][r] - f * T[9][r], xs = F * T[10][r] - f * T[11][r];
                const R qc_ = F * T[12][r] + f * T[13][r], qs = F * T[14][r] + f * T[15][r];
                U += (double)(cr * (uc - vc) - sr * (us + vs));
                W += (double)(sr * (wc + xc) + cr * (ws - xs));
                P2 += (double)(cr * (pc + qc_) + sr * (qs - ps));
                e2 += (double)(cr * T[16][r] + sr * T[17][r]);
            }
            if (own && val) {
                const CompRec<R>& cc = S.cr[i];
                const R ch = E + G, sh = E - G;
                e1 += (double)(cc.A * cr);
                gx += (double)(cc.gxz * cr);
                gy += (double)(cc.gyz * cr);
                gz += (double)(cc.gzz * sr);
                gp += (double)(cc.gpz * cr);
                const R c2 = (c * c - s * s) * ri, s2 = (R)2 * s * c * ri;
                e2 += (double)(cc.e2d * c2);
                if (lin) {
                    U1 += (double)(cc.lu * cr * ch);
                    V1 += (double)(cc.lv * cr * ch);
                    W += (double)(cc.lw * sr * sh);
                    P += (double)(cc.lp * cr * ch);
                }
                const R ch2 = E * E + G * G, sh2 = E * E - G * G;       // profile of 2k
                U1 += (double)(cc.ddu * c2 * ch2);
                V1 += (double)(cc.ddv * c2 * ch2);
                W += (double)(cc.ddw * s2 * sh2);
                P2 += (double)(cc.ddp * c2 * ch2);
                P2 += rid * (-(double)cc.kd1 * (double)ch + (double)cc.kd2 * (double)sh);
            }
        }
        if (slow) {
            const PairSum<R> v = pairs_one_by_one<R>(S.ph, J.mr, (const R*)J.coef + (int64_t)base * 6 * 64, N, S.h, i0, a, b,
                                                     xa, t, z, g, wp);
            U += v.U; W += v.W; P2 += v.P2; e2 += v.e2;
            K1 = v.K1; K2 = v.K2;
        }
        if (wp) {
            // kinetic terms of dp2 (Irregular.cpp:755-756, 786-787): phase-free
            // and separable over the pair; rows against the components past the
            // block, and (once) against the later rows of the block itself
            P2 += Bz * over_groups(K2) - Bx * over_groups(K1);
            if (own) {
                double Sx[4] = {0, 0, 0, 0}, Sz[4] = {0, 0, 0, 0};
                for (int gg = 0; gg < 4; ++gg) {
#pragma unroll
                    for (int rq = 0; rq < 4; ++rq) {
                        const double ox = __shfl(fx[rq], gg * 16 + pt), oz = __shfl(fz[rq], gg * 16 + pt);
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (Acc<R>::row(gg, rq) > Acc<R>::row(g, r)) {
                                Sx[r] += ox;
                                Sz[r] += oz;
                            }
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) P2 += rr[r] * (fz[r] * Sz[r] - fx[r] * Sx[r]);
            }
        }
    }
    double o[11] = {e1, e2, gx, gy, gz, gp, U1 + J.cth * U, V1 + J.sth * U, W, P, P2};
#pragma unroll
    for (int k = 0; k < 11; ++k) o[k] = over_groups(o[k]);
    if (!live || g != 0) return;
    if (J.partial) {
#pragma unroll
        for (int k = 0; k < 11; ++k) J.partial[((int64_t)sg * 11 + k) * J.n + q] = o[k];
    } else {
        point_store(J, q, o);
    }
}

__global__ __launch_bounds__(64) void k_point_reduce(PointJob J) {
    const int64_t q = (int64_t)blockIdx.x * 64 + threadIdx.x;
    if (q >= J.n) return;
    double o[11] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int s = 0; s < J.nseg; ++s)
#pragma unroll
        for (int k = 0; k < 11; ++k) o[k] += J.partial[((int64_t)s * 11 + k) * J.n + q];
    point_store(J, q, o);
}

}  // namespace

template <typename R>
hipError_t launch_point_forms(const SeaDev<R>& S, const PointJob& J, hipStream_t st) {
    hipLaunchKernelGGL((k_point_forms<R>), dim3((unsigned)((J.n + 63) / 64), J.nseg), dim3(256), 0, st, S, J);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || !J.partial) return e;
    hipLaunchKernelGGL(k_point_reduce, dim3((unsigned)((J.n + 63) / 64)), dim3(64), 0, st, J);
    return hipGetLastError();
}
template hipError_t launch_point_forms<float>(const SeaDev<float>&, const PointJob&, hipStream_t);
template hipError_t launch_point_forms<double>(const SeaDev<double>&, const PointJob&, hipStream_t);

}  // namespace cfdwm
