// Filtered second-order elevation eta2 as a quadratic form on the matrix cores.
//
// The pair sum of Irregular::eta2 (src/Irregular.cpp:223-293, pair-cache
// semantics of lsGridSpline's column update) is, per point p,
//
//   eta2_p = sum_i r_i [ c_pi sum_{m>i} Bcc_im c_pm + s_pi sum_{m>i} Bss_im s_pm ]
//
// with c_pi = cos(theta_i(p)), s_pi = sin(theta_i(p)), r_i the frequency ramp
// of component i at the point's time, Bcc = xP + xM and Bss = xM - xP built
// from the filtered pair coefficients (the real form of Re(Z^T B+ Z + Z^H B- Z)
// with Z_i = e^{i theta_i}).  The inner sums are GEMMs (points x components
// times components x components) on v_mfma_f32_32x32x16_bf16.  In the
// three-product mode every operand is split into bf16 hi + lo parts and the
// products hi*hi + hi*lo + lo*hi are accumulated in FP32, which keeps about 16
// significant bits per product; the one-product mode takes hi*hi alone (about
// 8 bits per product, a third of the matrix work and half the staged bytes).
// The outer sum over i is a fused epilogue (accumulator times c or s, summed
// in the lane, two exchanges at the end); the column kernel folds the result into
// its FP64 total.  The same kernel evaluates the z-independent forms of the
// velocity pair sums under the two profile depth bases (depth_basis.hpp): per
// skeleton wavenumber mu_q of the cosh-type basis one cos-type form each for
// u and v, per skeleton wavenumber of the sinh-type basis one sin-type form
// for w, with B entries cuP c_q(kP) +- cuM c_q(kM) (and cv, cw).
//
// The per-row ramp r_i must be the same for every i at a given time (the
// usual case: all ramps finished, or all components ramped alike); the host
// checks this and passes one factor per time slot.
#include <hip/hip_runtime.h>

#include "device_math.hpp"
#include "engine.hpp"
#include "kernels.hpp"

namespace cfdwm {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr double kInv2PiQ = 0.15915494309189533577;

// float -> bf16 bits, round to nearest even (finite inputs)
__device__ __forceinline__ uint32_t bf16_bits(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ float bf16_val(uint32_t b) { return __uint_as_float(b << 16); }
// bf16 element e (< 4) of four packed in a uint2, as float
__device__ __forceinline__ float bf16_half(uint2 v, int e) {
    const uint32_t w = e < 2 ? v.x : v.y;
    return __uint_as_float((e & 1) ? (w & 0xFFFF0000u) : (w << 16));
}

// ------------------------------------------------------------------ Z operands
// One thread per (point, 8 consecutive components): FP64 phase and range
// reduction, hardware sin/cos, bf16 hi/lo split, 16-byte stores.  A chunk
// holds at most 2^28 (point, component) entries (its Z arrays stay under
// 2 GiB), so thread, tile and s-grid column indices fit 32-bit arithmetic.
__global__ __launch_bounds__(256) void k_qf_zgen(QfJob J) {
    const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t nkb = (uint32_t)J.npad >> 4;
    const uint32_t ntile = (uint32_t)(J.ppad >> 5) * nkb;
    const uint32_t tile = tid >> 6;
    if (tile >= ntile) return;
    const int h = (int)((tid >> 5) & 1), r = (int)(tid & 31);
    const uint32_t rb = tile / nkb;
    const int kb = (int)(tile - rb * nkb);
    const int64_t p = (int64_t)rb * 32 + r;     // point within the chunk
    const int m0 = kb * 16 + h * 8;
    uint32_t ch[8], cl[8], sh[8], sl[8];
    const bool live = p < J.P;
    double x = 0, y = 0, t = 0;
    if (live) {
        const int64_t q = J.p0 + p;
        if (J.grid) {
            // q < 4 ncol and col < nx ny: 32-bit
            const uint32_t ncol = (uint32_t)J.ncol, ny = (uint32_t)J.g.ny;
            const uint32_t slot = (uint32_t)q / ncol;
            const uint32_t cq = (uint32_t)q - slot * ncol;
            const uint32_t col = J.cols ? (uint32_t)J.cols[cq] : cq;
            const uint32_t ci = col / ny;
            x = J.g.x0 + J.g.dx * (double)ci;
            y = J.g.y0 + J.g.dy * (double)(col - ci * ny);
            t = J.slot_t[slot];
        } else {
            x = J.x[q]; y = J.y[q]; t = J.t[q];
        }
    }
    const double dx = x - J.x0, dy = y - J.y0;
    // no branch around a component: its record's loads would wait one by one
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int m = m0 + j;
        const bool in = live && m < J.n;
        const PhaseRec ph = J.ph[m < J.n ? m : J.n - 1];
        double a = ph.k * (ph.cth * dx + ph.sth * dy) - ph.omega * t + ph.ph0;
        a *= kInv2PiQ;
        a -= rint(a);
        const float f = (float)a;
        const float s = in ? __builtin_amdgcn_sinf(f) : 0.f, c = in ? __builtin_amdgcn_cosf(f) : 0.f;
        ch[j] = bf16_bits(c); cl[j] = bf16_bits(c - bf16_val(ch[j]));
        sh[j] = bf16_bits(s); sl[j] = bf16_bits(s - bf16_val(sh[j]));
    }
    auto pack = [](const uint32_t* v) {
        return make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
    };
    const int64_t o = (int64_t)tile * 512 + h * 256 + r * 8;
    *reinterpret_cast<uint4*>(J.zc_hi + o) = pack(ch);
    *reinterpret_cast<uint4*>(J.zc_lo + o) = pack(cl);
    *reinterpret_cast<uint4*>(J.zs_hi + o) = pack(sh);
    *reinterpret_cast<uint4*>(J.zs_lo + o) = pack(sl);
}

// ----------------------------------------------------------- quadratic forms
// Form f of a launch:  Q_f(p) = sum_i e1_pi sum_m B1_f[i][m] c_pm + e2_pi sum_m B2_f[i][m] s_pm
// with (e1, e2) = (c, s) for cos-type forms and (s, c) for sin-type forms.
// One tile of work is (64 NP points, form): 4 waves, one per SIMD, walk the i
// range in tiles of 128 and, per i tile, the cosine and then the sine product;
// wave (w & 1, w >> 1) takes 32 NP points x 64 i as NP x 2 MFMA 32 x 32 blocks,
// computed with the table operand first, so that each lane's accumulator holds
// one point and 16 values of i.  The k (= m) range of an i tile runs from its
// first row (pairs have m > i) to the end of its filtered rows; the waves of
// the tile's second 64 rows leave out its first 64 values of k (m <= i there).
// The epilogue of a product multiplies the accumulators by c or s of the same
// (point, i) and sums over i in the lane; one exchange between the two
// half-waves and one between the two waves of a point range at the end write
// Q_f(p).  Single-job launches swizzle blocks in groups of 8 forms x 32 point
// tiles so that the Z and B tables a group reads stay in the last-level cache.
constexpr int kQfGF = 8, kQfGP = 32;

__device__ __forceinline__ bf16x8 lds8(const char* base, int off) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(base + off));
}

// A wave-uniform global pointer as scalar registers: the address arithmetic
// before it stays scalar and is not re-associated with per-lane offsets
// added after it, so loads take the scalar-base + vector-offset form.
typedef const uint16_t __attribute__((address_space(1)))* gu16p;
__device__ __forceinline__ gu16p uni_ptr(const uint16_t* p) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    return reinterpret_cast<gu16p>(((uint64_t)hi << 32) | lo);
}

// 16 bytes per lane from a wave-uniform base
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4 uni_load4(const uint16_t* base, int off) {
    return *reinterpret_cast<const u32x4 __attribute__((address_space(1)))*>(uni_ptr(base) + off);
}

// Operands move global -> LDS directly (global_load_lds_dwordx4, no
// registers) through three LDS stages.  NLV is the number of bf16 products per
// term: 3 (hi*hi + lo*hi + hi*lo of table and Z operands, about 16 significant
// bits) or 1 (hi*hi, about 8 significant bits; only the hi arrays are staged).
// A stage holds two operand sets of the block's 64 NP points and 128 i: with
// NLV 1 two consecutive k steps (16 values of m each), with NLV 3 the hi and
// the lo arrays of one k step; 24 KiB at NP = 4, so that two blocks share a
// CU's LDS and its registers (the accumulators take 128 of 256) and one block
// computes while the other waits.  Stage j is worked off in phases of 2 NP
// products whose operands were read from LDS one phase earlier:
//   NLV 1   A: set 0, reading set 1     | sync | B: set 1, reading set 0 of stage j + 1
//   NLV 3   A: hi x hi, reading lo      | sync | B: lo x hi | C: hi x lo, reading hi of stage j + 1
// The sync (s_waitcnt, then s_barrier as asm with a memory clobber:
// __syncthreads() would wait for every request) says that stage j + 1 has
// landed for all waves and that all waves have read stage j, whose buffer the
// requests of stage j + 3 then fill; they have two stages' time to land.
// NP = 4 serves three products; NP = 2 three products in launches of few rounds
// of the wide tile, and one product in launches too small for
// a form pair (below) per CU.
//
// What bounds three products: the matrix pipe at the clock that random bf16
// operands leave it (near 1.9 GHz; hipBLASLt reaches 1.21 PFLOP/s on an 8192^3
// product of this card).  43 forms, 30,300 points, 320 components: 0.94 ms,
// 1.15 PFLOP/s executed, against 1.21 ms with one block of 128-point tiles per
// CU, whose waits nothing covered.
//
// The table rows of a 32-row block are read from LDS in the order that puts
// the 16 rows of a lane's accumulator (8 q + 4 h + e, q < 4, h the half-wave)
// on the i values 16 (q / 2) + 8 h + 4 (q % 2) + e: the 8-value runs that the
// same lane holds in the Z tiles, so the epilogue reads whole 1 KiB tiles.
template <int NLV, int NP>
__device__ __forceinline__ void qf_tile_il(const QfJob& J, int ptile, int form) {
    static_assert(NLV == 1 || NLV == 3, "one or three bf16 products per term");
    constexpr int NB = 3;                         // stages
    constexpr int G = NP / 2 + 1;                 // groups of four 1 KiB tiles per operand set: points, then table rows
    constexpr int ND = 2 * G;                     // requests per wave and stage
    constexpr int SB = ND * 4096;                 // stage bytes
    constexpr int NF = NP + 2;                    // operand fragments of a set
    __shared__ __attribute__((aligned(16))) char lds[NB][SB];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int wv = __builtin_amdgcn_readfirstlane(w);
    const int wp = wv & 1, wi = wv >> 1;
    const int nkb = J.npad >> 4;
    const size_t nn = (size_t)J.npad * J.npad;
    // tables: 4 arrays per form (B1 hi, B1 lo, B2 hi, B2 lo) or 2 (B1 hi, B2 hi)
    const uint16_t* __restrict__ Bf = J.b + (size_t)form * J.nbarr * nn;
    const int bhs = J.nbarr == 4 ? 2 : 1;         // arrays between B1 hi and B2 hi
    const bool sint = J.ftype[form] != 0;
    const int64_t PB = (int64_t)ptile * (64 * NP);
    const int64_t rbB = PB >> 5;
    const int64_t P0 = PB + wp * (32 * NP);
    const int hl = lane >> 5, cl32 = lane & 31;
    const int loff = (hl * 256 + cl32 * 8) * 2;
    const int irow = (cl32 & 16) | ((cl32 & 4) << 1) | ((cl32 & 8) >> 1) | (cl32 & 3);
    const int loffB = (hl * 256 + irow * 8) * 2;
    float tp[NP];                                 // per lane: points P0 + 32 a + cl32
#pragma unroll
    for (int a = 0; a < NP; ++a) tp[a] = 0.f;
    const int lo8 = lane * 8;
    typedef __attribute__((address_space(3))) void* lds_vp;
    typedef const __attribute__((address_space(1))) void* glb_vp;
#define QF_WAIT(VM) __builtin_amdgcn_s_waitcnt(((VM) & 15) | (7 << 4) | (((VM) >> 4) << 14))
#define QF_BARRIER() __asm__ volatile("s_barrier" ::: "memory")
    const uint16_t* gp[ND];                       // request r of a stage at k step 0 (wave-uniform)
    auto dma = [&](int r, int kb, int st) {
        __builtin_amdgcn_global_load_lds((glb_vp)(uni_ptr(gp[r] + kb * 512) + lo8),
                                         (lds_vp)(lds[0] + st * SB + (r * 4 + wv) * 1024), 16, 0, 0);
    };
    // fragment f of operand set u of a stage: f < NP the point block f, else table block f - NP
    auto frag = [&](int st, int u, int f) {
        const char* L = lds[0] + st * SB + u * (G * 4096);
        return f < NP ? lds8(L, (wp * NP + f) * 1024 + loff)
                      : lds8(L, ((G - 1) * 4 + wi * 2 + (f - NP)) * 1024 + loffB);
    };
    constexpr int KS = NLV == 1 ? 2 : 1;          // k steps per stage
    for (int it = 0; it < J.npad; it += 128) {
        const int t0 = it >> 6;
        const int kb_lo = it >> 4;
        const int kb_hi = __builtin_amdgcn_readfirstlane(max(J.kend[t0], J.kend[t0 + 1]) >> 4);
        if (kb_hi <= kb_lo) continue;                 // block-uniform
        const int ns = (kb_hi - kb_lo + KS - 1) / KS; // stages (a last odd k step reads zero table entries)
        const int skip = wi ? 4 / KS : 0;             // stages this wave leaves out
        const int ib0 = it >> 5;
        // rows of this wave that have pairs at all
        const bool rows = __builtin_amdgcn_readfirstlane(J.kend[t0 + wi]) > it + wi * 64;
#pragma unroll 1
        for (int cs = 0; cs < 2; ++cs) {
            f32x16 acc[NP * 2];
#pragma unroll
            for (int q = 0; q < NP * 2; ++q)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[q][r] = 0.f;
#pragma unroll
            for (int r = 0; r < ND; ++r) {
                const int u = r / G, g = r % G;
                // NLV 1: set u is k step u of the hi arrays; NLV 3: u = 0 hi, 1 lo
                const int arr = NLV == 1 ? 0 : u, k = NLV == 1 ? u : 0;
                gp[r] = g < G - 1 ? J.zc_hi + (int64_t)(2 * cs + arr) * J.zn + ((rbB + 4 * g + wv) * nkb + k) * 512
                                  : Bf + (size_t)(cs * bhs + arr) * nn + ((int64_t)(ib0 + wv) * nkb + k) * 512;
            }
            auto request = [&](int j, int st, int r0, int r1) {
                if (j >= ns) return;                  // block-uniform
#pragma unroll
                for (int r = 0; r < ND; ++r)
                    if (r >= r0 && r < r1) dma(r, kb_lo + j * KS, st);
            };
            bf16x8 X[NF], Y[NF];
            auto mma = [&](const bf16x8& t, const bf16x8& z, int q) {
                acc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(t, z, acc[q], 0, 0, 0);
            };
            // waits until at most the last VM requests are outstanding; near the
            // end fewer were issued: wait for all
            auto sync = [&](bool last) {
                __builtin_amdgcn_sched_barrier(0);    // this phase's LDS reads are issued before the wait
                if (last) QF_WAIT(0);
                else QF_WAIT(ND);
                QF_BARRIER();
            };
            int s0 = 0, s1 = 1, s2 = 2;               // buffers of stages j, j + 1, j + 2
            request(0, 0, 0, ND);
            request(1, 1, 0, ND);
            request(2, 2, 0, NLV == 1 ? ND / 2 : ND);
            if (ns > 2) QF_WAIT(NLV == 1 ? ND + ND / 2 : 2 * ND);
            else QF_WAIT(0);
            QF_BARRIER();
            auto rotate = [&]() {
                const int t = s0;
                s0 = s1; s1 = s2; s2 = t;
            };
            int j = 0;
            // the stages whose table entries are zero for this wave's rows: requests and syncs only
            for (; j < min(skip, ns); ++j) {
                if constexpr (NLV == 1) request(j + 2, s2, ND / 2, ND);
                sync(j + 2 >= ns);
                request(j + 3, s0, 0, NLV == 1 ? ND / 2 : ND);
                rotate();
            }
            if (j < ns) {
#pragma unroll
                for (int f = 0; f < NF; ++f) X[f] = frag(s0, 0, f);
            }
            // products of set z (table fragments z[NP], z[NP + 1]) with the reads
            // of fragments into y from operand set u of stage buffer st between them
            auto phase = [&](const bf16x8 (&x)[NF], bf16x8 (&y)[NF], int st, int u) {
#pragma unroll
                for (int q = 0; q < 2 * NP; ++q) {
                    mma(x[NP + (q & 1)], x[q >> 1], q);
                    if (q < NF) y[q] = frag(st, u, q);
                    if (q & 1) __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int f = 2 * NP; f < NF; ++f) y[f] = frag(st, u, f);
            };
#pragma unroll 1
            for (; j < ns; ++j) {
                if constexpr (NLV == 1) {
                    phase(X, Y, s0, 1);
                    request(j + 2, s2, ND / 2, ND);
                    sync(j + 2 >= ns);
                    request(j + 3, s0, 0, ND / 2);
                    phase(Y, X, s1, 0);
                } else {
                    phase(X, Y, s0, 1);
                    sync(j + 2 >= ns);
                    request(j + 3, s0, 0, ND);
#pragma unroll
                    for (int q = 0; q < 2 * NP; ++q) mma(Y[NP + (q & 1)], X[q >> 1], q);
                    __builtin_amdgcn_sched_barrier(0);
                    Y[NP] = X[NP];
                    Y[NP + 1] = X[NP + 1];
                    phase(Y, X, s1, 0);
                }
                rotate();
            }
            // every wave is past its reads before the next product's requests
            QF_WAIT(0);
            QF_BARRIER();
            if (rows) {                               // wave-uniform
                // element r of block (a, b): point P0 + 32 a + cl32,
                // i = it + 64 wi + 32 b + 16 (r / 8) + 8 hl + r % 8
                const uint16_t* zrow = J.zc_hi + ((cs != 0) != sint ? 2 * J.zn : 0) +
                                       ((P0 >> 5) * nkb + (it >> 4) + wi * 4) * 512;
#pragma unroll
                for (int a = 0; a < NP; ++a) {
                    float s = 0.f, sl = 0.f;
#pragma unroll
                    for (int b = 0; b < 2; ++b)
#pragma unroll
                        for (int t = 0; t < 2; ++t) {
                            const uint16_t* z = zrow + ((int64_t)a * nkb + 2 * b + t) * 512;
                            const u32x4 hv = uni_load4(z, lo8), lv = uni_load4(z + J.zn, lo8);
#pragma unroll
                            for (int e = 0; e < 8; ++e) {
                                const uint32_t hw = hv[e >> 1], lw = lv[e >> 1];
                                const float vh = __uint_as_float((e & 1) ? hw & 0xFFFF0000u : hw << 16);
                                const float vl = __uint_as_float((e & 1) ? lw & 0xFFFF0000u : lw << 16);
                                if (NLV == 1) {       // the order of qf_pair_tile
                                    s += acc[a * 2 + b][8 * t + e] * vh;
                                    sl += acc[a * 2 + b][8 * t + e] * vl;
                                } else {
                                    s += acc[a * 2 + b][8 * t + e] * (vh + vl);
                                }
                            }
                        }
                    tp[a] += s;
                    if (NLV == 1) tp[a] += sl;
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    }
#undef QF_WAIT
#undef QF_BARRIER
    // lane l ends with points P0 + 64 c + l: its own half's i sums plus the other half's
    float* red = reinterpret_cast<float*>(lds[0]);
    float tot[NP / 2];
#pragma unroll
    for (int c = 0; c < NP / 2; ++c) {
        const float t0 = tp[2 * c] + __shfl_xor(tp[2 * c], 32);
        const float t1 = tp[2 * c + 1] + __shfl_xor(tp[2 * c + 1], 32);
        tot[c] = hl ? t1 : t0;
    }
    __syncthreads();
    if (wi)
#pragma unroll
        for (int c = 0; c < NP / 2; ++c) red[wp * 32 * NP + 64 * c + lane] = tot[c];
    __syncthreads();
    if (!wi)
#pragma unroll
        for (int c = 0; c < NP / 2; ++c) {
            const int64_t p = P0 + 64 * c + lane;
            if (p < J.P) J.out[(int64_t)form * J.ostride + J.p0 + p] = tot[c] + red[wp * 32 * NP + 64 * c + lane];
        }
}

// Velocity forms of the bf16 mode (one product per term): one block of 8 waves
// per CU evaluates two forms of one type for 256 points, 128 i at a time.
//
// What bounds these launches is the operands' way: with one form per block the
// requests for tables and Z operands took 14.8 ms of a 16.7 ms launch (262,144
// points, 1024 components, 26 forms) when only an eighth of the matrix
// products were left in it, and the epilogue's c and s another 3.5 ms; past L2
// they moved 92 GB.  Two forms share the staged Z operands and the epilogue's
// c and s, and two blocks' worth of rows share each table row: 512 rows per
// 2^16 products where 768 passed before, and half the epilogue's loads.
// The wave tile is 64 points x 64 i x 2 forms (128 accumulator registers).
//
// The block's work is one stream of stages (32 values of k: two operand sets),
// pass after pass ((i tile, cosine or sine product)), four LDS stages of 32
// KiB, requests three and a half stages ahead and running on across pass ends,
// so that the next pass's operands land during the epilogue.  Stage j:
//   A: products of set 0, reading set 1 | sync | B: products of set 1, reading set 0 of the stage after
// and the sync says that the stage after j has landed for all waves and that
// all waves have read stage j, whose buffer then takes the fourth stage after.
// The c or s of the epilogue are read as 16-byte runs of 8 i per lane (see
// qf_tile_il): the hi parts a stage ahead, the lo parts while the hi parts'
// products run.
//
// Measured on the launch above: 17.5 ms with one form, 128 points and both
// products per block (two blocks per CU), 16.7 with 256 points, 14.8 now, 1.03
// PFLOP/s executed.  Of these, the matrix products and barriers alone take
// 10.2, the LDS reads 1.0, the epilogue 1.4, the requests 2.3 (0.8 of them
// because the operands come from past L2).
constexpr int kPairStage = 32768;
__device__ __forceinline__ void qf_pair_tile(const QfJob& J, int ptile, int form, bool two) {
    constexpr int NB = 4;
    __shared__ __attribute__((aligned(16))) char lds[NB][kPairStage];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wp = wv & 3, wi = wv >> 2;
    const int nkb = J.npad >> 4;
    const size_t nn = (size_t)J.npad * J.npad;
    const int bhs = J.nbarr == 4 ? 2 : 1;
    const uint16_t* __restrict__ Bf = J.b + (size_t)form * J.nbarr * nn;
    // the block's second form; without one the first again, its values unused
    const size_t f2 = two ? (size_t)J.nbarr * nn : 0;
    const bool sint = J.ftype[form] != 0;
    const int64_t P0 = (int64_t)ptile * 256 + wp * 64;
    const int hl = lane >> 5, cl32 = lane & 31;
    const int loff = lane * 16;
    const int irow = (cl32 & 16) | ((cl32 & 4) << 1) | ((cl32 & 8) >> 1) | (cl32 & 3);
    const int loffB = (hl * 256 + irow * 8) * 2;
    const int lo8 = lane * 8;
    typedef __attribute__((address_space(3))) void* lds_vp;
    typedef const __attribute__((address_space(1))) void* glb_vp;
#define QF_WAIT(VM) __builtin_amdgcn_s_waitcnt(((VM) & 15) | (7 << 4) | (((VM) >> 4) << 14))
    // k steps of the i tile it, in stages (a last odd k step reads zero table entries)
    auto stages = [&](int it) {
        const int t0 = it >> 6;
        const int kb_hi = __builtin_amdgcn_readfirstlane(max(J.kend[t0], J.kend[t0 + 1]) >> 4);
        return max(0, (kb_hi - (it >> 4) + 1) >> 1);
    };
    int left = 0;                                     // stages of the stream not yet worked off
    for (int it = 0; it < J.npad; it += 128) left += 2 * stages(it);
    if (left > 0) {
        // request cursor: pass (rit, rcs), stage rj of rns; bases of this wave's tiles at the pass's first k step
        int rit = -128, rcs = 1, rj = 0, rns = 0;
        const uint16_t *ga = nullptr, *gb = nullptr;
        auto next_pass = [&](int& it, int& cs, int& ns) {
            if (cs == 0) { cs = 1; return; }
            cs = 0;
            do { it += 128; ns = stages(it); } while (ns == 0);
        };
        auto dma = [&](const uint16_t* g, int r, int st) {
            __builtin_amdgcn_global_load_lds((glb_vp)(uni_ptr(g) + lo8),
                                             (lds_vp)(lds[0] + st * kPairStage + (r * 8 + wv) * 1024), 16, 0, 0);
        };
        int toreq = left;                             // stages not yet requested
        // first half of a request: the point operands of both sets; second half: the table rows
        auto req_a = [&](int st) {
            if (toreq <= 0) return;
            if (rj == rns) {
                next_pass(rit, rcs, rns);
                rj = 0;
                ga = J.zc_hi + (int64_t)(2 * rcs) * J.zn + (((int64_t)ptile * 8 + wv) * nkb + (rit >> 4)) * 512;
                gb = Bf + (wv >> 2) * f2 + (size_t)(rcs * bhs) * nn +
                     ((int64_t)((rit >> 5) + (wv & 3)) * nkb + (rit >> 4)) * 512;
            }
            dma(ga + rj * 1024, 0, st);
            dma(ga + rj * 1024 + 512, 1, st);
        };
        auto req_b = [&](int st) {
            if (toreq <= 0) return;
            dma(gb + rj * 1024, 2, st);
            dma(gb + rj * 1024 + 512, 3, st);
            ++rj;
            --toreq;
        };
        // fragments of set u: 0, 1 the points, 2 .. 5 the table rows of (form, i block)
        auto frag = [&](int st, int u, int f) {
            const char* L = lds[0] + st * kPairStage + u * 8192;
            return f < 2 ? lds8(L, (wp * 2 + f) * 1024 + loff)
                         : lds8(L + 16384, (((f - 2) >> 1) * 4 + wi * 2 + ((f - 2) & 1)) * 1024 + loffB);
        };
        bf16x8 X[6], Y[6];
        f32x16 acc[8];                                // [(form * 2 + i block) * 2 + point block]
        auto clear = [&]() {
#pragma unroll
            for (int q = 0; q < 8; ++q)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[q][r] = 0.f;
        };
        auto phase = [&](const bf16x8 (&x)[6], bf16x8 (&y)[6], int st, int u) {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                acc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[2 + (q >> 1)], x[q & 1], acc[q], 0, 0, 0);
                if (q < 6) y[q] = frag(st, u, q);
                if (q & 1) __builtin_amdgcn_sched_barrier(0);
            }
        };
        float tp[2][2] = {{0.f, 0.f}, {0.f, 0.f}};    // [form][point block]
        req_a(0); req_b(0); req_a(1); req_b(1); req_a(2); req_b(2); req_a(3);
        QF_WAIT(0);
        __asm__ volatile("s_barrier" ::: "memory");
        int it = -128, cs = 1, ns = 0, buf = 0;
        while (left > 0) {                            // one pass; block-uniform
            next_pass(it, cs, ns);
            // the waves of the tile's second 64 rows leave out its first 64 k: m <= i there
            const int skip = min(wi ? 2 : 0, ns);
            const uint16_t* zrow = J.zc_hi + ((cs != 0) != sint ? 2 * J.zn : 0) +
                                   ((P0 >> 5) * nkb + (it >> 4) + wi * 4) * 512;
            u32x4 eh[8];
            auto load_hi = [&]() {
#pragma unroll
                for (int q = 0; q < 8; ++q) eh[q] = uni_load4(zrow + ((int64_t)(q >> 2) * nkb + (q & 3)) * 512, lo8);
            };
            // the next stage has landed once only the newest two stages' requests
            // (and, in a pass's last stage, the epilogue's 8 loads) are outstanding;
            // fewer were issued near the stream's end
            auto sync = [&](bool end) {
                __builtin_amdgcn_sched_barrier(0);
                if (left < 4) QF_WAIT(0);
                else if (end) QF_WAIT(16);
                else QF_WAIT(8);
                __asm__ volatile("s_barrier" ::: "memory");
            };
            clear();
            int j = 0;
            for (; j < skip; ++j) {
                const bool end = j == ns - 1;
                if (end) load_hi();
                req_b((buf + 3) & 3);
                sync(end);
                req_a(buf);
                --left;
                buf = (buf + 1) & 3;
            }
#pragma unroll
            for (int f = 0; f < 6; ++f) X[f] = frag(buf, 0, f);
#pragma unroll 1
            for (; j < ns; ++j) {
                const bool end = j == ns - 1;
                if (end) load_hi();
                phase(X, Y, buf, 1);
                req_b((buf + 3) & 3);
                sync(end);
                req_a(buf);
                const int nb = (buf + 1) & 3;
                phase(Y, X, nb, 0);
                --left;
                buf = nb;
            }
            // element r of block (f, b, a): point P0 + 32 a + cl32, i = it + 64 wi + 32 b + 16 (r / 8) + 8 hl + r % 8
            u32x4 el[8];
#pragma unroll
            for (int q = 0; q < 8; ++q)
                el[q] = uni_load4(zrow + J.zn + ((int64_t)(q >> 2) * nkb + (q & 3)) * 512, lo8);
            auto weigh = [&](const u32x4 (&e)[8]) {
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    float s0 = 0.f, s1 = 0.f;
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int k = 0; k < 8; ++k) {
                            const uint32_t hw = e[4 * a + t][k >> 1];
                            const float v = __uint_as_float((k & 1) ? hw & 0xFFFF0000u : hw << 16);
                            s0 += acc[(t >> 1) * 2 + a][8 * (t & 1) + k] * v;
                            s1 += acc[4 + (t >> 1) * 2 + a][8 * (t & 1) + k] * v;
                        }
                    tp[0][a] += s0;
                    tp[1][a] += s1;
                }
            };
            weigh(eh);
            weigh(el);
        }
#undef QF_WAIT
        // lane l: point P0 + l, its own half's i sums plus the other half's; then the two i halves
        float* red = reinterpret_cast<float*>(lds[0]);
        float tot[2];
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            const float t0 = tp[f][0] + __shfl_xor(tp[f][0], 32);
            const float t1 = tp[f][1] + __shfl_xor(tp[f][1], 32);
            tot[f] = hl ? t1 : t0;
        }
        __syncthreads();
        if (wi) {
            red[wp * 64 + lane] = tot[0];
            red[256 + wp * 64 + lane] = tot[1];
        }
        __syncthreads();
        if (!wi) {
            const int64_t p = P0 + lane;
            if (p < J.P) {
                float* o = J.out + (int64_t)form * J.ostride + J.p0 + p;
                o[0] = tot[0] + red[wp * 64 + lane];
                if (two) o[J.ostride] = tot[1] + red[256 + wp * 64 + lane];
            }
        }
    } else if (!wi) {
        const int64_t p = P0 + lane;
        if (p < J.P) {
            float* o = J.out + (int64_t)form * J.ostride + J.p0 + p;
            o[0] = 0.f;
            if (two) o[J.ostride] = 0.f;
        }
    }
}

// Blocks of an XCD (round-robin dispatch) walk the form pairs of two point
// tiles together: the two tiles' Z operands stay in its L2 (1 MiB of hi parts
// each at 1024 components), the tables stream through the last-level cache and
// serve both tiles.  Past L2 a launch of one-form blocks read 92 GB in groups of
// 8 forms x 32 point tiles, 89 GB one point tile at a time, 73 GB two at a time.
// Tile counts that 16 does not divide leave blocks that exit at once.  A
// numbering without them was compiled to a kernel 4 % slower at 256 tiles
// (65,536 points, 1024 components, step 4.73 -> 4.93 ms), where both give every
// block the same work; why is not known, nor how they compare at other counts.
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_qf_pairs(QfJob J, int npt) {
    const int np = qf_pairs(J.nform, J.ncos), sq = blockIdx.x >> 3;
    const int in = sq % (2 * np);
    const int ptile = (sq / (2 * np) * 2 + (in & 1)) * 8 + (blockIdx.x & 7);
    if (ptile >= npt) return;                         // whole block, before any barrier
    int form;
    bool two;
    qf_pair(J.nform, J.ncos, in >> 1, &form, &two);
    if (!J.clk) {
        qf_pair_tile(J, ptile, form, two);
        return;
    }
    const unsigned long long c0 = clock64(), w0 = wall_clock64();
    qf_pair_tile(J, ptile, form, two);
    if (threadIdx.x == 0) {
        atomicAdd(J.clk, clock64() - c0);
        atomicAdd(J.clk + 1, wall_clock64() - w0);
    }
}

// The eta2 form: one form, three products per term.  A block of 4 waves, one
// per SIMD, takes 128 points and 128 i at a time with the cosine and the sine
// products together (64 x 64 per wave, 128 accumulator and 203 other
// registers), four 32 KiB stages of one k step, requests three steps ahead.
// Step j of an i tile:
//   1. s_waitcnt vmcnt(8) lgkmcnt(0) + s_barrier: the requests of step j + 1
//      (issued during step j - 2) have landed for all waves, and all waves'
//      LDS reads of step j - 1 are done;
//   2. the 24 products of step j (operand set X) are issued interleaved with
//      the 16 LDS reads of step j + 1's operands (set Y, stage (j + 1) % 4)
//      and the 8 requests of step j + 3 (stage (j + 3) % 4 = (j - 1) % 4, last
//      read during step j - 2, before step j - 1's barrier).
// The sums run in one fixed order, the cosine and sine terms of an i together:
// whoever rounds functions of eta2 to bf16, as the surrogate's network does
// with its inputs, sees any other order.  Measured: 2.0 ms for 262,144 points
// and 1024 components (1.77e12 FLOP executed); qf_tile_il takes the same, and
// 8 waves on 128 points x 256 i, which read the points' operands 3.5 instead
// of 5.5 times, 2.1 ms.
__device__ __forceinline__ void qf_eta_tile(const QfJob& J, int ptile) {
    constexpr int NB = 4;                         // stages
    constexpr int NA = 4;                         // operand arrays per side in a stage
    constexpr int SB = 8192 * NA;                 // stage bytes
    constexpr int NF = 4 * NA;                    // operand fragments per set
    constexpr int NG = 2 * NA;                    // request chunks per step = issue groups
    constexpr int PG = 24 / NG;                   // products per issue group
    __shared__ __attribute__((aligned(16))) char lds[NB][SB];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int wp = w & 1, wi = w >> 1;
    const int nkb = J.npad >> 4;
    const size_t nn = (size_t)J.npad * J.npad;
    const uint16_t* __restrict__ Bf = J.b;       // B1 hi, B1 lo, B2 hi, B2 lo
    const bool sint = J.ftype[0] != 0;
    const int64_t PB = (int64_t)ptile * 128;
    const int64_t rbB = PB >> 5;
    const int64_t P0 = PB + wp * 64;
    const int hl = lane >> 5, cl32 = lane & 31;
    const int loff = ((lane >> 5) * 256 + (lane & 31) * 8) * 2;
    float tp[2] = {0.f, 0.f};                     // per lane: points P0 + cl32 and P0 + 32 + cl32
    const int wv = __builtin_amdgcn_readfirstlane(w);
    const int lo8 = lane * 8;
    typedef __attribute__((address_space(3))) void* lds_vp;
    typedef const __attribute__((address_space(1))) void* glb_vp;
#define QF4_SYNC(VM)                                                                 \
    __builtin_amdgcn_s_waitcnt(((VM) & 15) | (7 << 4) | (((VM) >> 4) << 14));        \
    __asm__ volatile("s_barrier" ::: "memory")
    // chunk r (< 2 NA) of a stage: A (array r, row block rbB + wv) for r < NA,
    // B (array r - NA, i row block ib0 + wv) for r >= NA; gp[r] is its address
    // at k step 0 of the current i tile (wave-uniform)
    const uint16_t* gp[NG];
    auto dma = [&](int r, int kb, int st) {
        __builtin_amdgcn_global_load_lds((glb_vp)(uni_ptr(gp[r] + kb * 512) + lo8),
                                         (lds_vp)(lds[0] + st * SB + (r * 4 + wv) * 1024), 16, 0, 0);
    };
    // operand fragment f of a stage: f < 2 NA A (a2 = f / NA, array f % NA),
    // else B (b = (f - 2 NA) / NA, array f % NA)
    auto frag = [&](int st, int f) {
        const char* L = lds[0] + st * SB;
        return f < 2 * NA ? lds8(L, ((f % NA) * 4 + wp * 2 + f / NA) * 1024 + loff)
                          : lds8(L, NA * 4096 + ((f % NA) * 4 + wi * 2 + (f - 2 * NA) / NA) * 1024 + loff);
    };
    bf16x8 opA[NF], opB[NF];
    for (int it = 0; it < J.npad; it += 128) {
        const int t0 = it >> 6;
        const int kb_lo = it >> 4;
        const int kb_hi = __builtin_amdgcn_readfirstlane(max(J.kend[t0], J.kend[t0 + 1]) >> 4);
        if (kb_hi <= kb_lo) continue;                 // block-uniform
        const int I0 = it + wi * 64;
        const int wk0 = I0 >> 4, wk1 = J.kend[t0 + wi] >> 4;
        const int ib0 = it >> 5;
        f32x16 acc[8];                                // [(a2 * 2 + b) * 2 + (0 cos part, 1 sin part)]
#pragma unroll
        for (int q = 0; q < 8; ++q)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[q][r] = 0.f;
        // product s (< 24) of a step: level s / 8 (hi x hi, lo x hi, hi x
        // lo of table x Z), accumulator s % 8; an accumulator's products are
        // 8 issues apart
        auto mma = [&](const bf16x8 (&op)[NF], int s) {
            const int lv = s >> 3, q = s & 7, cs = q & 1, a2 = q >> 2, b = (q >> 1) & 1;
            const int fa = a2 * 4 + 2 * cs + (lv == 2 ? 1 : 0);
            const int fb = 8 + b * 4 + 2 * cs + (lv == 1 ? 1 : 0);
            acc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op[fb], op[fa], acc[q], 0, 0, 0);
        };
        // one step: products of operand set x, reads of step j + 1 into set y
        // from stage s1, requests of step kbd into stage s3; NG chunks of PG
        // products, 2 reads and 1 request in a fixed issue order
        auto step = [&](const bf16x8 (&x)[NF], bf16x8 (&y)[NF], int s1, int s3, int kbd) {
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                mma(x, PG * g);
                y[2 * g] = frag(s1, 2 * g);
                mma(x, PG * g + 1);
                y[2 * g + 1] = frag(s1, 2 * g + 1);
                dma(g, kbd, s3);
                if (PG > 2) mma(x, PG * g + 2);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // global array of chunk r: A arrays c_hi, c_lo, s_hi, s_lo; B arrays likewise
#pragma unroll
        for (int r = 0; r < NG; ++r) {
            const int a = r % NA;
            gp[r] = r < NA ? J.zc_hi + (int64_t)a * J.zn + (rbB + wv) * nkb * 512
                           : Bf + (size_t)a * nn + (int64_t)(ib0 + wv) * nkb * 512;
        }
        // requests past the last step re-read step kb_hi - 1 (in bounds, unused)
        const int kl = kb_hi - 1;
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int r = 0; r < NG; ++r) dma(r, min(kb_lo + d, kl), d);
        QF4_SYNC(2 * NG);
#pragma unroll
        for (int f = 0; f < NF; ++f) opA[f] = frag(0, f);
        int s3 = 3, s1 = 1;                           // stages of steps j + 3 and j + 1
        for (int kb = kb_lo; kb < kb_hi; kb += 2) {
            QF4_SYNC(NG);
            step(opA, opB, s1, s3, min(kb + 3, kl));
            if (kb + 1 >= kb_hi) break;               // block-uniform
            s3 = (s3 + 1) & 3;
            s1 = (s1 + 1) & 3;
            QF4_SYNC(NG);
            step(opB, opA, s1, s3, min(kb + 4, kl));
            s3 = (s3 + 1) & 3;
            s1 = (s1 + 1) & 3;
        }
        // every request has landed and every wave is past its reads before
        // the next i tile's requests reuse stages 0 .. 2
        QF4_SYNC(0);
        if (wk1 > wk0) {                              // wave-uniform
            // accumulator element r of block (a2, b): point P0 + a2 * 32 + cl32,
            // i = I0 + b * 32 + 8 j + 4 hl + e (j = r / 4, e = r % 4); the four
            // i of one j are consecutive k of one half-tile row (8 bytes)
#pragma unroll
            for (int a2 = 0; a2 < 2; ++a2) {
                const uint16_t* zrow = J.zc_hi + ((P0 >> 5) + a2) * nkb * 512 + cl32 * 8 + 4 * hl;
                float s = 0.f;
#pragma unroll
                for (int b = 0; b < 2; ++b) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint16_t* zp = zrow + ((I0 >> 4) + 2 * b + (j >> 1)) * 512 + (j & 1) * 256;
                        const uint2 ch = *reinterpret_cast<const uint2*>(zp);
                        const uint2 cl = *reinterpret_cast<const uint2*>(zp + J.zn);
                        const uint2 sh = *reinterpret_cast<const uint2*>(zp + 2 * J.zn);
                        const uint2 sl = *reinterpret_cast<const uint2*>(zp + 3 * J.zn);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int r = 4 * j + e;
                            const float c = bf16_half(ch, e) + bf16_half(cl, e);
                            const float sv = bf16_half(sh, e) + bf16_half(sl, e);
                            s += acc[(a2 * 2 + b) * 2][r] * (sint ? sv : c) + acc[(a2 * 2 + b) * 2 + 1][r] * (sint ? c : sv);
                        }
                    }
                }
                tp[a2] += s;
            }
        }
    }
#undef QF4_SYNC
    // lane l ends with point P0 + l: its own half's i sums plus the other half's
    const float t0 = tp[0] + __shfl_xor(tp[0], 32);
    const float t1 = tp[1] + __shfl_xor(tp[1], 32);
    const float tot = hl ? t1 : t0;
    float* red = reinterpret_cast<float*>(lds[0]);
    __syncthreads();
    if (wi) red[wp * 64 + lane] = tot;
    __syncthreads();
    if (!wi) {
        const int64_t p = P0 + lane;
        if (p < J.P) J.out[J.p0 + p] = tot + red[wp * 64 + lane];
    }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2)))
void k_qf_eta(QfJob J) {
    if (!J.clk) {
        qf_eta_tile(J, blockIdx.x);
        return;
    }
    const unsigned long long c0 = clock64(), w0 = wall_clock64();
    qf_eta_tile(J, blockIdx.x);
    if (threadIdx.x == 0) {
        atomicAdd(J.clk, clock64() - c0);
        atomicAdd(J.clk + 1, wall_clock64() - w0);
    }
}

// Single-job launch: block -> (point tile, form) through the swizzle, without
// idle blocks between live ones.  Blocks go round-robin to the XCDs and there to
// the shader engines, so that groups filled up with blocks that exit at once
// leave the live ones on some of the engines only: 40 forms, 1008 components,
// three products, 640 points 732 -> 231 us (NP 2), 3040 points 1330 -> 668 us
// (NP 4), where 7680 points took 1630 us.
template <int NLV, int NP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_qf_forms_il(QfJob J, int npt, int by_xcd) {
    // the tiles this block's index runs over: all, or its XCD's (xcd, xcd + 8, ...)
    const int x = by_xcd ? blockIdx.x & 7 : 0, st = by_xcd ? 8 : 1;
    const int id = (int)blockIdx.x / st, nt = (npt - x + st - 1) / st, full = kQfGP / st;
    const int pg = id / (J.nform * full);
    const int rem = id - pg * J.nform * full;
    const int gp = min(full, nt - pg * full);         // point tiles of this group, fewer in the last
    if (gp <= 0 || rem >= gp * J.nform) return;       // whole block, before any barrier
    const int fg = rem / (kQfGF * gp), in = rem - fg * kQfGF * gp;
    const int ptile = (pg * full + in % gp) * st + x;
    const int form = fg * kQfGF + in / gp;
    if (!J.clk) {
        qf_tile_il<NLV, NP>(J, ptile, form);
        return;
    }
    const unsigned long long c0 = clock64(), w0 = wall_clock64();
    qf_tile_il<NLV, NP>(J, ptile, form);
    if (threadIdx.x == 0) {
        atomicAdd(J.clk, clock64() - c0);
        atomicAdd(J.clk + 1, wall_clock64() - w0);
    }
}

// Persistent launches over the tiles of many jobs (sea states): block b takes
// tiles b, b + gridDim.x, ... of the ordered tile list; every block exits
// after its last tile.  KIND 0: (256 points, form) tiles at three products,
// two blocks per CU; 1: (256 points, form pair) tiles at one product, one block
// of 8 waves per CU; 2: (128 points) tiles of the eta2 forms, one block per CU.
template <int KIND>
__global__ __launch_bounds__(KIND == 1 ? 512 : 256) __attribute__((amdgpu_waves_per_eu(KIND == 2 ? 1 : 2, 2)))
void k_qf_forms_persist(const QfJob* __restrict__ jobs, const QfTile* __restrict__ tiles, int ntiles) {
    for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const QfTile tl = tiles[t];
        const QfJob J = jobs[tl.job];
        __syncthreads();                              // the previous tile's LDS readers are done
        if constexpr (KIND == 0) qf_tile_il<3, 4>(J, tl.ptile, tl.form);
        else if constexpr (KIND == 1) qf_pair_tile(J, tl.ptile, tl.form, tl.two != 0);
        else qf_eta_tile(J, tl.ptile);
    }
}

// a wave-uniform element of a table no launch writes: a scalar load
__device__ __forceinline__ double ro_load(const double* p, int i) {
#if defined(__HIP_DEVICE_COMPILE__)
    return ((const __attribute__((address_space(4))) double*)p)[i];
#else
    return p[i];
#endif
}

// Form tables: one thread per (i, m).  Profile-basis coefficients c_q(kappa) =
// sum_s finv[q][s] P_kappa(z_s) in FP64 (finv is ill-conditioned: its entries
// are large while |c| stays O(1)), entries written as bf16 hi + lo into the
// tiled layout, zeros where there is no pair, over all the forms kernels read:
// m from the first row of i's 128-row tile on.  The exponentials bound it, so
// the second one of a profile is e^{-2 kappa h} over the first while both stay
// normal numbers; a wave takes 4 rows x 16 m, so that its 2-byte stores fill
// 64 bytes.  Loads and exponentials go in fours and eights without a branch
// between them, and ranks to 16 (the one-product mode's) take half the
// registers.  2048 components, 38 forms: 465 us and 140 for zeroing the tables
// before, 366 now.
template <int RM>
__global__ __launch_bounds__(256) void k_qf_build(QfBuild B) {
    const int lane = threadIdx.x & 63;
    if ((int)blockIdx.x * 64 < (((int)blockIdx.y * 4) & ~127)) return;
    const int i = blockIdx.y * 4 + ((lane >> 3) & 3);
    const int m = blockIdx.x * 64 + (threadIdx.x >> 6) * 16 + (lane & 7) + (lane >> 5) * 8;
    const bool pair = i < B.n && m > i && m < B.fmhi[i];
    UvwRec<float> r{};
    XRec<float> xr{};
    if (pair) {
        const int64_t e = B.frow[i] - (i + 1) + m;
        r = B.uvw[e];
        xr = B.x[e];
    }
    constexpr double kL2eInv = 0.69314718055994530942;   // ln 2: kappa = pk / log2 e
    const double kp = (double)r.pkP * kL2eInv, km = (double)r.pkM * kL2eInv;
    const int nkb = B.npad >> 4;
    const size_t nn = (size_t)B.npad * B.npad;
    const size_t o = ((size_t)(i >> 5) * nkb + (m >> 4)) * 512 + ((m >> 3) & 1) * 256 + (i & 31) * 8 + (m & 7);
    auto put = [&](int f, int k, double v) {
        const bool sep = B.beta && f == 0;            // the eta2 form in its own hi/lo table
        const bool lo = sep || B.nbarr == 4;
        const int fi = B.beta ? f - 1 : f;
        uint16_t* d = sep ? B.beta + (size_t)(2 * k) * nn : B.b + ((size_t)fi * B.nbarr + (lo ? 2 * k : k)) * nn;
        // (opaque: else the two roundings become one from FP64)
        float x = (float)v;
        __asm__ volatile("" : "+v"(x));
        const uint32_t hi = bf16_bits(x);
        d[o] = (uint16_t)hi;
        if (lo) d[o + nn] = (uint16_t)bf16_bits(x - bf16_val(hi));
    };
    put(0, 0, (double)xr.xP + (double)xr.xM);
    put(0, 1, (double)xr.xM - (double)xr.xP);
    if (!__any(pair)) {
        for (int f = 1; f < B.nform; ++f) {
            put(f, 0, 0.0);
            put(f, 1, 0.0);
        }
        return;
    }
    // profile P_kappa(z) = e^{kappa z} + sg e^{-kappa (z + 2h)} at the
    // skeleton depths, then its basis coefficients c = finv P (one family at a time)
    double eP[RM], eM[RM];
    const double gP = exp(-2.0 * kp * B.h), gM = exp(-2.0 * km * B.h);
    auto family = [&](int R, const double* zs, const double* finv, double sg, int f0, int nf) {
        // four depths at a time: their exponentials' chains run side by side
#pragma unroll
        for (int c = 0; c < RM; c += 4) {
            if (c < R) {
#pragma unroll
                for (int q = c; q < c + 4; ++q) {
                    const double z = ro_load(zs, q);
                    const double E = exp(kp * z), F = exp(km * z);
                    if (B.normal) {
                        eP[q] = E + sg * (gP * dm::rcp_nr(E));
                        eM[q] = F + sg * (gM * dm::rcp_nr(F));
                    } else {
                        eP[q] = E + sg * exp(-kp * (z + 2.0 * B.h));
                        eM[q] = F + sg * exp(-km * (z + 2.0 * B.h));
                    }
                }
            } else {
#pragma unroll
                for (int q = c; q < c + 4; ++q) eP[q] = eM[q] = 0.0;
            }
        }
        for (int q = 0; q < R; ++q) {
            double cp = 0, cm = 0;
// (rows of 32, zeros past R: eight at a time come with one scalar load)
#pragma unroll
            for (int c = 0; c < RM; c += 8) {
                if (c < R) {
#pragma unroll
                    for (int s2 = c; s2 < c + 8; ++s2) {
                        const double w = ro_load(finv, q * 32 + s2);
                        cp += w * eP[s2];
                        cm += w * eM[s2];
                    }
                }
            }
            if (nf == 2) {                            // u, v (cos-type)
                put(f0 + q, 0, r.cuP * cp + r.cuM * cm);
                put(f0 + q, 1, r.cuM * cm - r.cuP * cp);
                if (B.Rv) {
                    put(f0 + R + q, 0, r.cvP * cp + r.cvM * cm);
                    put(f0 + R + q, 1, r.cvM * cm - r.cvP * cp);
                }
            } else {                                  // w (sin-type)
                put(f0 + q, 0, r.cwP * cp + r.cwM * cm);
                put(f0 + q, 1, r.cwP * cp - r.cwM * cm);
            }
        }
    };
    family(B.R, B.zs, B.finv, 1.0, 1, 2);
    family(B.Rw, B.zsw, B.finvw, -1.0, 1 + B.R + B.Rv, 1);
}

}  // namespace

hipError_t launch_qf_build(const QfBuild& B, hipStream_t st) {
    if (B.n <= 0 || B.R < 0 || B.R > 32 || B.Rw < 0 || B.Rw > 32 || (B.Rv && B.Rv != B.R) || B.nform != 1 + B.R + B.Rv + B.Rw ||
        (B.npad & 127) || B.npad < B.n || (B.nbarr != 2 && B.nbarr != 4))
        return hipErrorInvalidValue;
    // ranks to 16 leave twice the waves: 578 us with 32 where 16 takes 366
    const dim3 grid((unsigned)(B.npad / 64), (unsigned)(B.npad / 4));
    if (B.R <= 16 && B.Rw <= 16) hipLaunchKernelGGL(k_qf_build<16>, grid, dim3(256), 0, st, B);
    else hipLaunchKernelGGL(k_qf_build<32>, grid, dim3(256), 0, st, B);
    return hipGetLastError();
}

static bool qf_shape_ok(const QfJob& J) {
    if ((J.nlv != 1 && J.nlv != 3) || (J.nbarr != 2 && J.nbarr != 4) || (J.nlv == 3 && J.nbarr != 4)) return false;
    if (J.ncos < 0 || J.ncos > J.nform) return false;
    return !((J.ppad & (kQfTile - 1)) || (J.npad & 127) || J.ppad < J.P || J.npad < J.n);
}

hipError_t launch_qf_zgen(const QfJob& J, hipStream_t st) {
    if (J.P <= 0) return hipSuccess;
    if (!qf_shape_ok(J)) return hipErrorInvalidValue;
    const int64_t nthr = (J.ppad >> 5) * (J.npad >> 4) * 64;
    // the kernel's 32-bit indices: at most 2^28 Z entries per chunk, and an
    // s-grid chunk's points within 4 slots of ncol columns
    if ((int64_t)J.ppad * J.npad > ((int64_t)1 << 28) || (J.grid && J.p0 + J.P > ((int64_t)1 << 31))) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_qf_zgen, dim3((unsigned)((nthr + 255) / 256)), dim3(256), 0, st, J);
    return hipGetLastError();
}

hipError_t launch_qf_persist(const QfJob* jobs, const QfTile* tiles, int ntiles, int blocks, int kind, hipStream_t st) {
    if (ntiles <= 0) return hipSuccess;
    if (blocks <= 0) return hipErrorInvalidValue;
    const dim3 g((unsigned)blocks);
    if (kind == kQfTileForm) hipLaunchKernelGGL(k_qf_forms_persist<0>, g, dim3(256), 0, st, jobs, tiles, ntiles);
    else if (kind == kQfTilePair) hipLaunchKernelGGL(k_qf_forms_persist<1>, g, dim3(512), 0, st, jobs, tiles, ntiles);
    else if (kind == kQfTileEta) hipLaunchKernelGGL(k_qf_forms_persist<2>, g, dim3(256), 0, st, jobs, tiles, ntiles);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_qf_forms(const QfJob& J, hipStream_t st) {
    if (J.P <= 0 || J.nform <= 0) return hipSuccess;
    if (!qf_shape_ok(J)) return hipErrorInvalidValue;
    // eta2 alone
    if (J.nlv == 3 && J.nform == 1) {
        hipLaunchKernelGGL(k_qf_eta, dim3((unsigned)((J.P + 127) / 128)), dim3(256), 0, st, J);
        return hipGetLastError();
    }
    // one product per term: form pairs where they give every CU a block
    if (J.nlv == 1 && J.ppad / 256 * qf_pairs(J.nform, J.ncos) >= 256) {
        const int np = (int)(J.ppad / 256);
        hipLaunchKernelGGL(k_qf_pairs, dim3((unsigned)((np + 15) / 16 * 16 * qf_pairs(J.nform, J.ncos))), dim3(512), 0, st,
                           J, np);
        return hipGetLastError();
    }
    // 256-point tiles where they come to two and a half rounds of two blocks per
    // CU, else 128-point ones, whose last round is shorter (40 forms, 1008
    // components: 600 wide tiles 1001 us against 899, 1000 1680 against 1456,
    // 1280 1628 against 1658; 320 components, 2560 458 against 478)
    const bool wide = J.nlv == 3 && J.ppad / 256 * J.nform >= 1280;
    const int npt = (int)(wide ? J.ppad / 256 : (J.P + 127) / 128);
    // An XCD that keeps its point tiles reads their Z operands through its own L2,
    // but where 8 does not divide the tiles some XCDs have one fewer, else the
    // tiles go block after block.  The lines are drawn through measurements; that
    // three products lose at 70 tiles, with 3 % of padding, has no explanation
    // here.  One product waits for the operands most: kept
    // from 16 tiles on, if that adds under 30 % (23 forms, 1024 components, 25
    // tiles 276 us against 329).  Three: kept up to 64 tiles, if it adds under
    // 5 % (40 forms, 752 components, 61 tiles 1177 us against 1271; 1008
    // components, 55 tiles 1552 against 1688, but 43 tiles 1320 against 1205, 70
    // tiles 2061 against 1832).
    const int npt8 = (npt + 7) / 8 * 8;
    const int by_xcd = npt >= 16 && (J.nlv == 1 ? npt8 * 10 <= npt * 13 : npt <= 64 && npt8 * 20 <= npt * 21);
    const unsigned nblk = (unsigned)((int64_t)(by_xcd ? npt8 : npt) * J.nform);
    if (J.nlv == 1)
        hipLaunchKernelGGL((k_qf_forms_il<1, 2>), dim3(nblk), dim3(256), 0, st, J, npt, by_xcd);
    else if (wide)
        hipLaunchKernelGGL((k_qf_forms_il<3, 4>), dim3(nblk), dim3(256), 0, st, J, npt, by_xcd);
    else
        hipLaunchKernelGGL((k_qf_forms_il<3, 2>), dim3(nblk), dim3(256), 0, st, J, npt, by_xcd);
    return hipGetLastError();
}

}  // namespace cfdwm
