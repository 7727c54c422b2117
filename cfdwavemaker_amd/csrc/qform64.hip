// FP64 s-grid fills: the filtered second-order pair sums as quadratic forms
// on the FP64 matrix cores.
//
// A column needs, at every level z, the pair sums of src/Irregular.cpp:975-1102
// (u, v, w) and, once, those of eta2 (:223-293).  The depth enters a pair term
// only through its profile P_kappa(z) = e^{kappa z} +- e^{-kappa (z + 2h)}, an
// entire function of z.  The sums are therefore evaluated at the S nodes of a
// mapped Chebyshev grid on [-h, 0] and carried to the column's levels by
// barycentric interpolation, which is exact to rounding for every kappa of the
// sea (DepthNodes, depth_basis.hpp: S = 28 to 44 for kmax h = 32 to 200,
// measured error <= 4e-15 of the profile).  At a fixed node the sum over pairs
// is a quadratic form in the column's cosines and sines,
//
//   Q(p) = sum_i c_pi sum_{m>i} B1_im c_pm + s_pi sum_{m>i} B2_im s_pm   (u, v, eta2)
//   Q(p) = sum_i s_pi sum_{m>i} B1_im c_pm + c_pi sum_{m>i} B2_im s_pm   (w)
//
// B1, B2 = the pair's sum and difference coefficients times their profiles at
// the node, added and subtracted.  The inner sums are products on
// v_mfma_f64_16x16x4_f64, the outer sum a fused epilogue.  Everything is FP64.
//
// Against the pair loop (one FP64 sincos per pair and column, up to four FP64
// exponentials per pair, column and level) the work per pair and column drops
// to 3 S + 1 pairs of multiply-adds on the matrix cores, whatever the number
// of levels.
//
// Operand layout: 16 x 8 tiles of 64 lanes x 2 values; lane l holds row l % 16
// at k = l / 16 and k = 4 + l / 16, the operands of two matrix instructions in
// one 16-byte load (1 KiB per tile, contiguous).
#include <hip/hip_runtime.h>

#include "device_math.hpp"
#include "engine.hpp"

namespace cfdwm {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------- Z operands
// cos and sin of every (point, component): one thread per lane of a tile.
// Points past P and components past n are zero.
__global__ __launch_bounds__(256) void k_qd_zgen(QdJob J) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int nkb = J.npad >> 3;
    const int64_t tile = tid >> 6;
    if (tile >= (J.ppad >> 4) * nkb) return;
    const int lane = (int)(tid & 63);
    const int64_t rb = tile / nkb;
    const int kb = (int)(tile - rb * nkb);
    const int64_t p = rb * 16 + (lane & 15);
    double c[2] = {0, 0}, s[2] = {0, 0};
    if (p < J.P) {
        const int64_t q = J.p0 + p;
        const int slot = (int)(q / J.ncol);
        const int64_t cq = q - (int64_t)slot * J.ncol;
        const int64_t col = J.cols ? J.cols[cq] : cq;
        const double dx = J.g.x0 + J.g.dx * (double)(col / J.g.ny) - J.x0;
        const double dy = J.g.y0 + J.g.dy * (double)(col % J.g.ny) - J.y0;
        const double t = J.slot_t[slot];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int m = kb * 8 + 4 * e + (lane >> 4);
            if (m < J.n) dm::cs_of(dm::phase_of(J.ph[m], dx, dy, t), c[e], s[e]);
        }
    }
    reinterpret_cast<double2*>(J.zc)[tile * 64 + lane] = make_double2(c[0], c[1]);
    reinterpret_cast<double2*>(J.zs)[tile * 64 + lane] = make_double2(s[0], s[1]);
}

// ------------------------------------------------------------- form tables
// One thread per lane of a table tile (row i, m at 8 kb + l / 16 and + 4) for
// every form of the group: eta2 (with the first group), then u, v, w (nf 3) or
// u, w (nf 2: every v coefficient of the sea is zero) at nn nodes.  Tiles
// wholly below the diagonal 64-row block are never read and not written.
__global__ __launch_bounds__(256) void k_qd_build(QdBuild B) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int nkb = B.npad >> 3;
    const int64_t tile = tid >> 6;
    if (tile >= (int64_t)(B.npad >> 4) * nkb) return;
    const int lane = (int)(tid & 63);
    const int ib = (int)(tile / nkb), kb = (int)(tile - (int64_t)ib * nkb);
    if (kb * 8 < (ib * 16) / 64 * 64) return;         // wave-uniform
    const int i = ib * 16 + (lane & 15);
    const int64_t nn = (int64_t)B.npad * B.npad / 2;  // double2 per array
    double2* out = reinterpret_cast<double2*>(B.b) + tile * 64 + lane;
    int64_t e[2];
    bool on[2];
    UvwRec<double> r[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int m = kb * 8 + 4 * h + (lane >> 4);
        on[h] = i < B.n && m > i && m < B.fmhi[i];
        e[h] = on[h] ? B.frow[i] - (i + 1) + m : 0;
        if (on[h]) r[h] = B.uvw[e[h]];
    }
    if (B.eta) {
        double b1[2] = {0, 0}, b2[2] = {0, 0};
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (on[h]) {
                const XRec<double> x = B.x[e[h]];
                b1[h] = x.xM + x.xP;
                b2[h] = x.xM - x.xP;
            }
        out[0] = make_double2(b1[0], b1[1]);
        out[nn] = make_double2(b2[0], b2[1]);
        out += 2 * nn;
    }
    for (int q = 0; q < B.nn; ++q) {
        const double z = B.zs[B.node0 + q];
        double b[6][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int k = 0; k < 6; ++k) b[k][h] = 0.;
            if (!on[h]) continue;
            const double eP = exp(r[h].pkP * z), gP = exp(fma(-r[h].pkP, z, r[h].pgP));
            const double eM = exp(r[h].pkM * z), gM = exp(fma(-r[h].pkM, z, r[h].pgM));
            const double cP = eP + gP, sP = eP - gP, cM = eM + gM, sM = eM - gM;
            const double uP = r[h].cuP * cP, uM = r[h].cuM * cM, vP = r[h].cvP * cP, vM = r[h].cvM * cM;
            const double wP = r[h].cwP * sP, wM = r[h].cwM * sM;
            b[0][h] = uM + uP; b[1][h] = uM - uP;
            b[2][h] = vM + vP; b[3][h] = vM - vP;
            b[4][h] = wP + wM; b[5][h] = wP - wM;
        }
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            if (B.nf == 2 && (k == 2 || k == 3)) continue;
            *out = make_double2(b[k][0], b[k][1]);
            out += nn;
        }
    }
}

// ------------------------------------------------------------------- forms
// One wave evaluates one form for 16 NP points, walking 64-row tiles of i and,
// per tile, the cosine and the sine product: 4 x NP accumulators of 16 x 16
// (128 registers at NP = 4), operands straight from L2, the next 8 values of k
// in flight while these 8 NP instructions (64 cycles each) run.  No LDS and no
// barrier: a 64 x 64 tile takes 8 KiB of operands per 2048 matrix cycles.
// The table is the row operand, so a lane's results are one point and rows
// l / 16 + 4 r of each 16: exactly the rows its own lane holds in the Z tiles,
// which the epilogue therefore reads as ordinary operand loads.
// Tile order: 8 blocks of points run side by side, one per XCD under the
// round-robin dispatch, each for all forms in turn: a block's Z operands stay
// in its XCD's L2 while the tables stream through the last-level cache.  The
// last group takes the blocks that are left, spread over all XCDs.
// Measured: 66.8 TFLOP/s executed (16,384 points, 256 components, 121 forms;
// rocBLAS reaches 72.8 on an 8192^3 product of this card), the fill
// 31.0 -> 5.3 ms against the pair loop.
template <int NP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_qd_forms(QdJob J, int npt) {
    const int per = 8 * J.nform, npb = (npt + 3) >> 2;
    const int pg = blockIdx.x / per, in = blockIdx.x - pg * per;
    const int gsz = min(8, npb - pg * 8);
    const int form = in / gsz;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int ptile = __builtin_amdgcn_readfirstlane((pg * 8 + in - form * gsz) * 4 + w);
    if (ptile >= npt) return;                          // whole wave, no barriers below
    const int nkb = J.npad >> 3;
    const int64_t nn = (int64_t)J.npad * J.npad / 2;
    const bool sint = J.form0 + form >= 1 && (J.form0 + form - 1) % J.nf == J.nf - 1;   // w
    // wave-uniform bases; every load adds the lane's 16 bytes
    const double2* zc = reinterpret_cast<const double2*>(J.zc) + (int64_t)ptile * NP * nkb * 64;
    const double2* zs = reinterpret_cast<const double2*>(J.zs) + (int64_t)ptile * NP * nkb * 64;
    double tp[NP];
#pragma unroll
    for (int b = 0; b < NP; ++b) tp[b] = 0.;
    for (int it = 0; it < J.npad; it += 64) {
        const int k0 = it >> 3, k1 = __builtin_amdgcn_readfirstlane(J.kend[it >> 6] >> 3);
        if (k1 <= k0) continue;
#pragma unroll 1
        for (int cs = 0; cs < 2; ++cs) {
            const double2* ta = reinterpret_cast<const double2*>(J.b) + (int64_t)(2 * form + cs) * nn +
                                (int64_t)(it >> 4) * nkb * 64;
            const double2* zb = cs ? zs : zc;
            f64x4 acc[4][NP];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < NP; ++b) acc[a][b] = f64x4{0., 0., 0., 0.};
            double2 xa[4], xb[NP], ya[4], yb[NP];
            auto load = [&](double2 (&la)[4], double2 (&lb)[NP], int kb) {
#pragma unroll
                for (int a = 0; a < 4; ++a) la[a] = (ta + (a * nkb + kb) * 64)[lane];
#pragma unroll
                for (int b = 0; b < NP; ++b) lb[b] = (zb + (b * nkb + kb) * 64)[lane];
            };
            auto mul = [&](const double2 (&la)[4], const double2 (&lb)[NP]) {
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int b = 0; b < NP; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(la[a].x, lb[b].x, acc[a][b], 0, 0, 0);
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int b = 0; b < NP; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(la[a].y, lb[b].y, acc[a][b], 0, 0, 0);
            };
            load(xa, xb, k0);
#pragma unroll 1
            for (int kb = k0; kb < k1; kb += 2) {      // an even number of steps (kend)
                load(ya, yb, kb + 1);
                mul(xa, xb);
                load(xa, xb, min(kb + 2, k1 - 1));     // the last repeats a step (unused)
                mul(ya, yb);
            }
            // rows of the tile: 16 a + l / 16 + 4 r, weighted with c or s of the same (point, i)
            const double2* ze = (cs != 0) != sint ? zs : zc;
#pragma unroll
            for (int b = 0; b < NP; ++b) {
                const double2* zr = ze + (b * nkb + (it >> 3)) * 64;
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const double2 e0 = (zr + 128 * a)[lane], e1 = (zr + 128 * a + 64)[lane];
                    tp[b] += (acc[a][b][0] * e0.x + acc[a][b][1] * e0.y) + (acc[a][b][2] * e1.x + acc[a][b][3] * e1.y);
                }
                // one group of points at a time: all loads at once would not fit the registers
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // a point's four row groups sit in lanes l, l ^ 16, l ^ 32, l ^ 48
#pragma unroll
    for (int b = 0; b < NP; ++b) {
        tp[b] += __shfl_xor(tp[b], 16);
        tp[b] += __shfl_xor(tp[b], 32);
        const int64_t p = ((int64_t)ptile * NP + b) * 16 + lane;
        if (lane < 16 && p < J.P) J.out[(int64_t)(J.form0 + form) * J.ostride + J.p0 + p] = tp[b];
    }
}

bool qd_shape_ok(const QdJob& J) {
    return J.npad > 0 && (J.npad & 63) == 0 && J.npad >= J.n && (J.ppad & 63) == 0 && J.ppad >= J.P && J.ncol > 0 &&
           (J.nf == 2 || J.nf == 3) && J.p0 + J.P <= J.ostride;
}

}  // namespace

hipError_t launch_qd_zgen(const QdJob& J, hipStream_t st) {
    if (J.P <= 0) return hipSuccess;
    if (!qd_shape_ok(J)) return hipErrorInvalidValue;
    const int64_t thr = (J.ppad >> 4) * (J.npad >> 3) * 64;
    hipLaunchKernelGGL(k_qd_zgen, dim3((unsigned)((thr + 255) / 256)), dim3(256), 0, st, J);
    return hipGetLastError();
}

hipError_t launch_qd_build(const QdBuild& B, hipStream_t st) {
    if (B.n <= 0 || (B.npad & 63) || B.npad < B.n || B.nn < 0 || (B.nf != 2 && B.nf != 3)) return hipErrorInvalidValue;
    const int64_t thr = (int64_t)(B.npad >> 4) * (B.npad >> 3) * 64;
    hipLaunchKernelGGL(k_qd_build, dim3((unsigned)((thr + 255) / 256)), dim3(256), 0, st, B);
    return hipGetLastError();
}

hipError_t launch_qd_forms(const QdJob& J, hipStream_t st) {
    if (J.P <= 0 || J.nform <= 0) return hipSuccess;
    if (!qd_shape_ok(J)) return hipErrorInvalidValue;
    // 64 points per wave where that leaves two waves per SIMD (2048) or more,
    // else 32 (more waves, more table loads per product)
    const int64_t t4 = (J.P + 63) / 64;
    const bool wide = t4 * J.nform >= 2048;
    const int npt = (int)(wide ? t4 : (J.P + 31) / 32);
    const unsigned nb = (unsigned)((npt + 3) / 4 * J.nform);
    if (wide) hipLaunchKernelGGL(k_qd_forms<4>, dim3(nb), dim3(256), 0, st, J, npt);
    else hipLaunchKernelGGL(k_qd_forms<2>, dim3(nb), dim3(256), 0, st, J, npt);
    return hipGetLastError();
}

}  // namespace cfdwm
