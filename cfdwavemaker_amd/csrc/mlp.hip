// Per-column MLP of the learned second-order surrogate: hand-written HIP
// kernels for inference and training (no counterpart in the reference; the
// surrogate predicts the second-order correction that src/Irregular.cpp's
// pair sums produce, and the exact kernels stay the fallback).
//
// Network: L linear layers, GELU (erf form) after every layer but the last.
// Master parameters are FP32 (Adam state too); every product runs on the
// matrix cores with both operands rounded to bf16 (round to nearest even)
// and FP32 accumulation, i.e. bf16 weights and activations, FP32 sums.
// Inputs and outputs are standardised inside (per-feature mean / std).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "engine.hpp"
#include "../../include/cfdwm.h"

namespace cfdwm {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint16_t to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// C[M x N] = A[M x K] . B[K x N] with A(m, k) = A[m sam + k sak],
// B(k, n) = B[k sbk + n sbn]; bf16 operands, FP32 accumulation.
// epi 0: C = acc;  1: Z = acc + bias, C = gelu(Z);  2: C = acc + bias;
// 3: C = acc * gelu'(Z).
struct MmArgs {
    int M, N, K;
    const float* A;
    int64_t sam, sak;
    const float* B;
    int64_t sbk, sbn;
    float* C;
    int64_t scm;
    const float* bias;
    float* Z;
    int epi;
    int kchunk;                           // values of k per blockIdx.z (K: no split)
    int64_t cz;                           // elements between the outputs of two chunks
    float* colsum;                        // when set (ak false): sums of A's columns, per chunk
    bool ak, bk;                          // the operand is contiguous in k, else in m (n)
};

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_d(float x) {
    return 0.5f * (1.f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}

// Epilogue of a block's 64 x 64 tile through LDS (64 x 68 floats, the block's
// threads past a barrier): a thread takes four consecutive columns of a row,
// four times in a rolled loop.  Straight from the accumulators the 16 unrolled
// copies of erf and exp ran from cold instruction memory and the stores were
// single floats (4096 x 256 x 256: 15.2 -> 11.4 us with bias and gelu, 18.2 ->
// 12.9 with gelu', the longer k steps of mm_tile included).
constexpr int kMmT = 68;
__device__ __forceinline__ void mm_store(const MmArgs& a, const f32x16& acc, float* T, int m0, int n0) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
#pragma unroll
    for (int r = 0; r < 16; ++r)
        T[((w & 1) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * kMmT + (w >> 1) * 32 + (lane & 31)] = acc[r];
    __syncthreads();
    const int c0 = (t & 15) * 4;
    const bool hasb = a.epi == 1 || a.epi == 2;
    float bias[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) bias[k] = hasb ? a.bias[min(n0 + c0 + k, a.N - 1)] : 0.f;
    const bool v4 = n0 + 64 <= a.N && (a.scm & 3) == 0 && (a.cz & 3) == 0 &&
                    ((reinterpret_cast<uintptr_t>(a.C) | reinterpret_cast<uintptr_t>(a.Z)) & 15) == 0;
#pragma unroll 1
    for (int j = 0; j < 4; ++j) {
        const int r = j * 16 + (t >> 4), m = m0 + r;
        if (m >= a.M) break;
        const int64_t o = (int64_t)m * a.scm + n0 + c0;
        const float4 q = *reinterpret_cast<const float4*>(T + r * kMmT + c0);
        float v[4] = {q.x + bias[0], q.y + bias[1], q.z + bias[2], q.w + bias[3]};
        if (v4) {
            float4 z = make_float4(v[0], v[1], v[2], v[3]);
            if (a.epi == 1) *reinterpret_cast<float4*>(a.Z + o) = z;
            if (a.epi == 3) z = *reinterpret_cast<const float4*>(a.Z + o);
            const float zz[4] = {z.x, z.y, z.z, z.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (a.epi == 1) v[k] = gelu(v[k]);
                if (a.epi == 3) v[k] *= gelu_d(zz[k]);
            }
            *reinterpret_cast<float4*>(a.C + o) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll 1
            for (int k = 0; k < 4; ++k) {
                if (n0 + c0 + k >= a.N) break;
                const float x = k == 0 ? v[0] : k == 1 ? v[1] : k == 2 ? v[2] : v[3];
                if (a.epi == 1) a.Z[o + k] = x;
                a.C[o + k] = a.epi == 1 ? gelu(x) : a.epi == 3 ? x * gelu_d(a.Z[o + k]) : x;
            }
        }
    }
}

// Block 256 threads = 4 waves, 64 x 64 outputs; wave (w & 1, w >> 1) takes a
// 32 x 32 tile (one v_mfma_f32_32x32x16_bf16 accumulator).  Operands are
// staged through LDS 64 values of k at a time, rounded to bf16 on the way:
// [row][k], so that a lane's operand (row l % 32, 8 values of k) is one
// 16-byte LDS read.  AK, BK: the operand is contiguous in k in memory (a
// thread stages 8 values of k of one row, two 16-byte loads where the rows
// are aligned), else contiguous in m or n (a thread stages 8 values of k of
// one m or n, the 64 lanes of a load reading 64 consecutive floats).  The
// next step's loads are in flight while this step's products run; k runs in
// ascending order, out-of-range elements are zero.
//
// blockIdx.z splits k into chunks of kchunk (weight gradients: k is the row
// of the minibatch): chunk z writes its own C + z cz.  colsum: the chunk's
// sums over k of A's columns in FP32 (the bias gradient), by the blocks of
// the first n tile.
//
// What bounds it: latency (a 4096-row step is 0.3 to 0.5 GFLOP per product).
// Before, the gradient products read strided scalars per lane (22 us each,
// 207 us for the 33-wide input) and one thread summed a whole column (851 us
// for 4096 rows, four times): 4.0 ms per loss and gradient of 4096 rows of the
// 33-256-256-256-65 network, 0.21 ms now (products 11 to 13 us each).
template <bool AK, bool BK>
__device__ __forceinline__ void mm_tile(const MmArgs& a, int bx, int by, int bz) {
    constexpr int KS = 64, LS = KS + 8;                        // LDS row stride in bf16 (144 bytes: rows start 4 banks apart, no conflicts at 16 bytes)
    __shared__ __attribute__((aligned(16))) uint16_t lds[2][2][64 * LS];
    uint16_t(*As)[64 * LS] = lds[0], (*Bs)[64 * LS] = lds[1];
    float* T = reinterpret_cast<float*>(lds);     // 64 x 68 floats in the end
    static_assert(sizeof(lds) >= 64 * kMmT * sizeof(float), "the output tile takes the operands' place");
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int m0 = by * 64, n0 = bx * 64;
    const int kb = bz * a.kchunk, ke = min(a.K, kb + a.kchunk);
    // one operand's 8 values of this thread: row (m or n) r0 + r, k0 + 8 q ..
    const int ra = AK ? t >> 2 : lane, qa = AK ? t & 3 : w;
    const int rb = BK ? t >> 2 : lane, qb = BK ? t & 3 : w;
    auto fetch = [&](const float* P, int64_t sr, int64_t sk, int row, int rows, int k, bool kc, bool v4, float (&f)[8]) {
#pragma unroll
        for (int j = 0; j < 8; ++j) f[j] = 0.f;
        if (row >= rows) return;
        const float* p = P + (int64_t)row * sr + (int64_t)k * sk;
        if (kc && v4 && k + 8 <= ke) {
            const float4 u = *reinterpret_cast<const float4*>(p), v = *reinterpret_cast<const float4*>(p + 4);
            f[0] = u.x; f[1] = u.y; f[2] = u.z; f[3] = u.w;
            f[4] = v.x; f[5] = v.y; f[6] = v.z; f[7] = v.w;
            return;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (k + j < ke) f[j] = p[(int64_t)j * sk];
    };
    const bool av4 = AK && (a.sam & 3) == 0 && (reinterpret_cast<uintptr_t>(a.A) & 15) == 0 && (kb & 3) == 0;
    const bool bv4 = BK && (a.sbn & 3) == 0 && (reinterpret_cast<uintptr_t>(a.B) & 15) == 0 && (kb & 3) == 0;
    auto stash = [&](uint16_t* L, int r, int q, const float (&f)[8]) {
        uint4 o;
        o.x = to_bf16(f[0]) | ((uint32_t)to_bf16(f[1]) << 16);
        o.y = to_bf16(f[2]) | ((uint32_t)to_bf16(f[3]) << 16);
        o.z = to_bf16(f[4]) | ((uint32_t)to_bf16(f[5]) << 16);
        o.w = to_bf16(f[6]) | ((uint32_t)to_bf16(f[7]) << 16);
        *reinterpret_cast<uint4*>(L + r * LS + q * 8) = o;
    };
    float cs = 0.f;
    const bool sums = a.colsum && bx == 0;
    float fa[KS / 32][8], fb[KS / 32][8];
    auto fetch2 = [&](int k0) {
#pragma unroll
        for (int s = 0; s < KS / 32; ++s) {
            fetch(a.A, a.sam, a.sak, m0 + ra, a.M, k0 + 32 * s + 8 * qa, AK, av4, fa[s]);
            fetch(a.B, a.sbn, a.sbk, n0 + rb, a.N, k0 + 32 * s + 8 * qb, BK, bv4, fb[s]);
        }
    };
    auto stash2 = [&](int b) {
#pragma unroll
        for (int s = 0; s < KS / 32; ++s) {
            stash(As[b], ra, 4 * s + qa, fa[s]);
            stash(Bs[b], rb, 4 * s + qb, fb[s]);
            if (!AK && sums) {
#pragma unroll
                for (int j = 0; j < 8; ++j) cs += fa[s][j];
            }
        }
    };
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    fetch2(kb);
    stash2(0);
    __syncthreads();
    const int oa = ((w & 1) * 32 + (lane & 31)) * LS + (lane >> 5) * 8;
    const int ob = ((w >> 1) * 32 + (lane & 31)) * LS + (lane >> 5) * 8;
    int b = 0;
    for (int k0 = kb; k0 < ke; k0 += KS) {        // block-uniform
        if (k0 + KS < ke) fetch2(k0 + KS);
#pragma unroll
        for (int h = 0; h < KS / 16; ++h) {
            const bf16x8 A8 = *reinterpret_cast<const bf16x8*>(As[b] + oa + 16 * h);
            const bf16x8 B8 = *reinterpret_cast<const bf16x8*>(Bs[b] + ob + 16 * h);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A8, B8, acc, 0, 0, 0);
        }
        if (k0 + KS < ke) stash2(b ^ 1);          // its readers passed the last barrier
        __syncthreads();
        b ^= 1;
    }
    MmArgs o = a;
    o.C = a.C + (int64_t)bz * a.cz;
    __syncthreads();                              // the operands have been read
    mm_store(o, acc, T, m0, n0);
    if (!AK && sums) {                            // block-uniform: the four threads of a column, in order
        float* red = T;
        __syncthreads();
        red[t] = cs;
        __syncthreads();
        if (w == 0 && m0 + lane < a.M)
            a.colsum[(int64_t)bz * a.cz + m0 + lane] =
                ((red[lane] + red[64 + lane]) + red[128 + lane]) + red[192 + lane];
    }
}

template <bool AK, bool BK>
__global__ __launch_bounds__(256) void k_mm(MmArgs a) {
    mm_tile<AK, BK>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

// The weight gradients of up to kMmBatch layers in one launch: block x is an
// output tile of the layer whose range holds it.  One after the other they
// cost 11 us each; all four of the network above 20.
constexpr int kMmBatch = 8;
struct MmBatch {
    int n;
    int tile0[kMmBatch + 1];
    MmArgs g[kMmBatch];
};
__global__ __launch_bounds__(256) void k_mm_grads(MmBatch b) {
    int l = 0;
    while (l + 1 < b.n && (int)blockIdx.x >= b.tile0[l + 1]) ++l;      // block-uniform
    const MmArgs& a = b.g[l];
    const int q = (int)blockIdx.x - b.tile0[l], nx = (a.N + 63) / 64;
    mm_tile<false, false>(a, q % nx, q / nx, blockIdx.z);
}

// g[i] = sum over the chunks z, in order, of part[z np + i]
__global__ __launch_bounds__(256) void k_sum_chunks(int64_t np, int nz, const float* __restrict__ part,
                                                    float* __restrict__ g) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    float s = 0.f;
    for (int z = 0; z < nz; ++z) s += part[(int64_t)z * np + i];
    g[i] = s;
}

// ------------------------------------------------------------ fused inference
// The whole network for 64 rows per block: the standardised input and each
// hidden layer's output stay in LDS as bf16 (the operand rounding the
// layer-wise kernels apply when they load them), weights come from the FP32
// master parameters, and only the unstandardised outputs reach HBM.  Each
// wave takes 32-column blocks of a layer in turn, both 32-row halves at once
// (k order, products and epilogue as k_mm), so the outputs equal
// the layer-wise path's bit for bit.  Weights come as bf16 operands laid out
// once a call (k_mlp_pack, 5 us): read as FP32 rows and rounded in every block
// they took a third of the time (262,144 rows of the 33-256-256-256-65 network
// 665 us, 490 now; the erf of 768 values a row bounds it at about 300).
// Limits: at most kFiL layers, widths up to kFiW.
constexpr int kFiR = 64, kFiW = 256, kFiS = kFiW + 8, kFiL = 8;   // rows, max width, LDS row stride

struct MlpFused {
    int64_t n = 0;
    int L = 0, nin = 0, nout = 0;
    int din[kFiL] = {}, dout[kFiL] = {};
    const float* W[kFiL] = {};            // W_l[j][k], dout x din
    uint16_t* Wp = nullptr;               // their bf16 operands (k_mlp_pack), layer l from woff[l]
    int woff[kFiL + 1] = {};
    const float* b[kFiL] = {};
    const float *mu_in = nullptr, *sd_in = nullptr, *mu_out = nullptr, *sd_out = nullptr;
    const float* X = nullptr;             // n x nin
    float* Y = nullptr;                   // n x nout
};

// Weights as the products take them: layer by layer, a lane's 8 bf16 values of
// each (32-column block, 16 values of k) consecutive, zero past N and K.
__global__ __launch_bounds__(256) void k_mlp_pack(MlpFused a) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    int l = 0;
    while (l < a.L && i * 8 >= a.woff[l + 1]) ++l;
    if (l >= a.L) return;
    const int K = a.din[l], N = a.dout[l], ks = (K + 15) / 16;
    const int e = i - a.woff[l] / 8, lane = e & 63, s = (e >> 6) % ks, ct = (e >> 6) / ks;
    const int col = ct * 32 + (lane & 31), k0 = s * 16 + (lane >> 5) * 8;
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j)
        v[j] = __builtin_bit_cast(__bf16, to_bf16(col < N && k0 + j < K ? a.W[l][(int64_t)col * K + k0 + j] : 0.f));
    *reinterpret_cast<bf16x8*>(a.Wp + (int64_t)i * 8) = v;
}

__global__ __launch_bounds__(256) void k_mlp_fused(MlpFused a) {
    __shared__ __attribute__((aligned(16))) uint16_t H[2][kFiR * kFiS];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t r0 = (int64_t)blockIdx.x * kFiR;
    // layer 0 input, standardised (as k_standardise), zero past nin up to a multiple of 16
    const int k0p = (a.nin + 15) & ~15;
    for (int idx = threadIdx.x; idx < kFiR * k0p; idx += 256) {
        const int r = idx / k0p, c = idx - r * k0p;
        float v = 0.f;
        if (c < a.nin && r0 + r < a.n) v = (a.X[(r0 + r) * a.nin + c] - a.mu_in[c]) / a.sd_in[c];
        H[0][r * kFiS + c] = to_bf16(v);
    }
    __syncthreads();
    const int kh = (lane >> 5) * 8, hl = lane >> 5;
    int cur = 0;
    for (int l = 0; l < a.L; ++l) {
        const int K = a.din[l], N = a.dout[l];
        const int Kp = (K + 15) & ~15;
        const bool last = l == a.L - 1;
        const uint16_t* __restrict__ W = a.Wp + a.woff[l];
        const float* __restrict__ bias = a.b[l];
        const int nct = (N + 31) / 32;
        // column block ct of both 32-row halves: two accumulators sharing each B operand
        for (int ct = w; ct < nct; ct += 4) {
            const int col = ct * 32 + (lane & 31);
            const uint16_t* h0 = &H[cur][(lane & 31) * kFiS + kh];
            const uint16_t* h1 = h0 + 32 * kFiS;
            f32x16 acc0, acc1;
#pragma unroll
            for (int r = 0; r < 16; ++r) acc0[r] = acc1[r] = 0.f;
            // the next k step's weights requested before this step's products
            const uint4* q = reinterpret_cast<const uint4*>(W) + (int64_t)ct * (Kp / 16) * 64 + lane;
            uint4 u = *q;
            for (int k0 = 0; k0 < Kp; k0 += 16) {
                q += k0 + 16 < Kp ? 64 : 0;
                const uint4 un = *q;
                const bf16x8 B8 = __builtin_bit_cast(bf16x8, u);
                const bf16x8 A0 = *reinterpret_cast<const bf16x8*>(h0 + k0);
                const bf16x8 A1 = *reinterpret_cast<const bf16x8*>(h1 + k0);
                acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A0, B8, acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A1, B8, acc1, 0, 0, 0);
                u = un;
            }
            if (col >= N) continue;
            const float bc = bias[col];
            const float so = last ? a.sd_out[col] : 0.f, mo = last ? a.mu_out[col] : 0.f;
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = rt * 32 + 8 * (r >> 2) + 4 * hl + (r & 3);
                    const float v = (rt ? acc1[r] : acc0[r]) + bc;
                    if (!last) {
                        H[cur ^ 1][row * kFiS + col] = to_bf16(gelu(v));
                    } else if (r0 + row < a.n) {
                        a.Y[(r0 + row) * a.nout + col] = v * so + mo;
                    }
                }
            }
        }
        if (!last) {
            // columns past N read as zeros by the next layer's last k step
            const int Np = (N + 15) & ~15;
            for (int idx = threadIdx.x; idx < kFiR * (Np - N); idx += 256) {
                const int r = idx / (Np - N), c = N + idx - r * (Np - N);
                H[cur ^ 1][r * kFiS + c] = 0;
            }
        }
        __syncthreads();
        cur ^= 1;
    }
}

// X_hat = (X - mean) / std over n rows of d features (row-major)
__global__ void k_standardise(int64_t n, int d, const float* __restrict__ X, const float* __restrict__ mu,
                              const float* __restrict__ sd, float* __restrict__ Y) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * d) return;
    const int j = (int)(i % d);
    Y[i] = (X[i] - mu[j]) / sd[j];
}
// Y = Y_hat * std + mean
__global__ void k_unstandardise(int64_t n, int d, float* __restrict__ Y, const float* __restrict__ mu,
                                const float* __restrict__ sd) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * d) return;
    const int j = (int)(i % d);
    Y[i] = Y[i] * sd[j] + mu[j];
}
// rows of X (and Y) picked by idx (null: in order) into Xb (Yb), standardised
__global__ void k_gather_std(int64_t nb, int d, const int64_t* __restrict__ idx, const float* __restrict__ X,
                             const float* __restrict__ mu, const float* __restrict__ sd, float* __restrict__ Xb) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nb * d) return;
    const int64_t r = i / d;
    const int j = (int)(i - r * d);
    Xb[i] = (X[(idx ? idx[r] : r) * d + j] - mu[j]) / sd[j];
}
// dY = 2 (Yp - Y) / (n d) and per-block partial sums of (Yp - Y)^2
__global__ __launch_bounds__(256) void k_mse(int64_t n, int d, const float* __restrict__ Yp, const float* __restrict__ Y,
                                             float* __restrict__ dY, float* __restrict__ part) {
    __shared__ float red[256];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    float e2 = 0.f;
    if (i < n * d) {
        const float e = Yp[i] - Y[i];
        dY[i] = 2.f * e / (float)(n * d);
        e2 = e * e;
    }
    red[threadIdx.x] = e2;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}
__global__ void k_adam(int64_t n, float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

inline unsigned nb256(int64_t n) { return (unsigned)((n + 255) / 256); }

// Row chunks of a weight gradient, at most: 4096 rows in 32 cost 22 us and 11 for
// the chunks' sum, in 16 20 and 6.
constexpr int kGradChunks = 16;

}  // namespace

struct Mlp {
    int nin = 0, width = 0, nhid = 0, nout = 0;
    std::vector<int> din, dout;           // per layer
    std::vector<int64_t> woff, boff;      // parameter offsets
    int64_t np = 0;
    DevBuf par, grad, am, av;             // FP32 master parameters, gradients, Adam moments
    DevBuf norm;                          // in_mean, in_std, out_mean, out_std
    DevBuf act;                           // H_0..H_L and Z_0..Z_{L-1} for a batch
    DevBuf tmp, part, idx;
    DevBuf wpk;                          // bf16 weights of the fused kernel
    bool fused() const {
        bool f = layers() <= kFiL && nin <= kFiW;
        for (int l = 0; l < layers(); ++l) f = f && dout[l] <= kFiW;
        return f;
    }
    // bf16 values of layer l in wpk
    int packed(int l) const { return (dout[l] + 31) / 32 * ((din[l] + 15) / 16) * 512; }
    DevBuf gpart;                         // [chunk][np]: the row chunks' gradients
    int64_t cap = 0;                      // rows the activation buffers hold
    int64_t adam_t = 0;
    int layers() const { return (int)din.size(); }
    float* P() const { return (float*)par.get(); }
    float* G() const { return (float*)grad.get(); }
    float* nin_mu() const { return (float*)norm.get(); }
    float* nin_sd() const { return nin_mu() + nin; }
    float* nout_mu() const { return nin_sd() + nin; }
    float* nout_sd() const { return nout_mu() + nout; }
    // activation layout for a batch of cap rows
    int64_t hoff(int l) const {          // H_l, l = 0..L
        int64_t o = 0;
        for (int q = 0; q < l; ++q) o += cap * din[q];
        return o;
    }
    int64_t zoff(int l) const {          // Z_l after all H
        int64_t o = hoff(layers()) + cap * nout;
        for (int q = 0; q < l; ++q) o += cap * dout[q];
        return o;
    }
    int reserve(int64_t rows);
    int forward(int64_t n, hipStream_t st);   // H_0 filled; runs all layers
    int backward(int64_t n, const float* dY, hipStream_t st);
};

int Mlp::reserve(int64_t rows) {
    if (rows <= cap) return 0;
    cap = rows;
    int64_t tot = 0;
    for (int l = 0; l < layers(); ++l) tot += cap * (din[l] + dout[l]);
    tot += cap * nout;
    if (act.alloc((size_t)tot * sizeof(float))) return -3;
    if (tmp.alloc((size_t)cap * nout * 2 * sizeof(float))) return -3;     // dY and the targets
    if (part.alloc((size_t)(nb256(cap * nout) + 1) * sizeof(float))) return -3;
    if (idx.alloc((size_t)cap * sizeof(int64_t))) return -3;
    return 0;
}

static hipError_t mm(MmArgs a, hipStream_t st) {
    if (a.M <= 0 || a.N <= 0) return hipSuccess;
    if (a.kchunk <= 0 || a.kchunk > a.K) a.kchunk = a.K;
    if ((a.ak ? a.sak : a.sam) != 1 || (a.bk ? a.sbk : a.sbn) != 1 || (a.colsum && a.ak)) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((a.N + 63) / 64), (unsigned)((a.M + 63) / 64), (unsigned)((a.K + a.kchunk - 1) / a.kchunk));
    if (a.ak && a.bk) hipLaunchKernelGGL((k_mm<true, true>), grid, dim3(256), 0, st, a);
    else if (a.ak) hipLaunchKernelGGL((k_mm<true, false>), grid, dim3(256), 0, st, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

int Mlp::forward(int64_t n, hipStream_t st) {
    float* A = (float*)act.get();
    for (int l = 0; l < layers(); ++l) {
        MmArgs a{};
        a.M = (int)n; a.N = dout[l]; a.K = din[l];
        a.A = A + hoff(l); a.sam = din[l]; a.sak = 1;
        a.B = P() + woff[l]; a.sbk = 1; a.sbn = din[l];          // B(k, j) = W[j][k]
        a.ak = a.bk = true;
        a.bias = P() + boff[l];
        a.scm = dout[l];
        if (l + 1 < layers()) {
            a.C = A + hoff(l + 1);
            a.Z = A + zoff(l);
            a.epi = 1;
        } else {
            a.C = A + hoff(l + 1);
            a.epi = 2;
        }
        CFDWM_HIP(mm(a, st));
    }
    return 0;
}

// dY sits in tmp; dZ_l takes the place of Z_l.
int Mlp::backward(int64_t n, const float* dY, hipStream_t st) {
    float* A = (float*)act.get();
    // weight gradients sum over the rows: split into at most kGradChunks chunks
    // of 128 rows or more, so that a minibatch's few 64 x 64 output tiles
    // fill the chip; the chunks' gradients (parameter layout) meet at the end
    // (the chunks' gradients take at most 256 MiB, or one chunk's)
    const int64_t most = std::max<int64_t>(1, std::min<int64_t>(kGradChunks, (int64_t(64) << 20) / np));
    const int chunk = (int)(((n + most - 1) / most + 127) / 128 * 128);
    const int nz = (int)((n + chunk - 1) / chunk);
    if (gpart.alloc((size_t)nz * np * sizeof(float))) return -3;
    float* GP = (float*)gpart.get();
    auto dZ = [&](int l) { return l + 1 < layers() ? (const float*)(A + zoff(l)) : dY; };
    // dZ_{l-1} = (dZ_l W_l) * gelu'(Z_{l-1}) : (n x dout) . (dout x din)
    for (int l = layers() - 1; l > 0; --l) {
        MmArgs h{};
        h.M = (int)n; h.N = din[l]; h.K = dout[l];
        h.A = dZ(l); h.sam = dout[l]; h.sak = 1;
        h.B = P() + woff[l]; h.sbk = din[l]; h.sbn = 1;
        h.C = h.Z = A + zoff(l - 1); h.scm = din[l]; h.epi = 3;
        h.ak = true;
        CFDWM_HIP(mm(h, st));
    }
    // dW_l = dZ_l^T H_l : (dout x n) . (n x din), db_l = column sums of dZ_l
    for (int l0 = 0; l0 < layers(); l0 += kMmBatch) {
        MmBatch b{};
        b.n = std::min(kMmBatch, layers() - l0);
        for (int q = 0; q < b.n; ++q) {
            const int l = l0 + q;
            MmArgs& g = b.g[q];
            g.M = dout[l]; g.N = din[l]; g.K = (int)n;
            g.A = dZ(l); g.sam = 1; g.sak = dout[l];
            g.B = A + hoff(l); g.sbk = din[l]; g.sbn = 1;
            g.C = GP + woff[l]; g.scm = din[l]; g.epi = 0;
            g.kchunk = chunk; g.cz = np; g.colsum = GP + boff[l];
            b.tile0[q + 1] = b.tile0[q] + (g.M + 63) / 64 * ((g.N + 63) / 64);
        }
        hipLaunchKernelGGL(k_mm_grads, dim3((unsigned)b.tile0[b.n], 1, (unsigned)nz), dim3(256), 0, st, b);
        CFDWM_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_sum_chunks, dim3(nb256(np)), dim3(256), 0, st, np, nz, (const float*)GP, G());
    CFDWM_HIP(hipGetLastError());
    return 0;
}

}  // namespace cfdwm

using namespace cfdwm;

struct cfdwm_mlp {
    Mlp m;
};

extern "C" {

int cfdwm_mlp_create(cfdwm_mlp** out, int nin, int width, int nhidden, int nout, uint64_t seed) {
    if (!out || nin < 1 || width < 1 || nhidden < 0 || nout < 1) return -1;
    if (int e = Engine::get().init()) return e;
    auto* h = new cfdwm_mlp();
    Mlp& M = h->m;
    M.nin = nin; M.width = width; M.nhid = nhidden; M.nout = nout;
    int d = nin;
    for (int l = 0; l <= nhidden; ++l) {
        const int o = l < nhidden ? width : nout;
        M.din.push_back(d);
        M.dout.push_back(o);
        d = o;
    }
    for (int l = 0; l < M.layers(); ++l) {
        M.woff.push_back(M.np);
        M.np += (int64_t)M.din[l] * M.dout[l];
        M.boff.push_back(M.np);
        M.np += M.dout[l];
    }
    if (M.fused()) {
        size_t wp = 0;
        for (int l = 0; l < M.layers(); ++l) wp += M.packed(l);
        if (M.wpk.alloc(wp * sizeof(uint16_t))) { delete h; return -3; }
    }
    // He-style uniform initialisation (limit sqrt(6 / fan_in)), zero biases
    std::vector<float> p(M.np, 0.f);
    std::mt19937_64 rng(seed);
    for (int l = 0; l < M.layers(); ++l) {
        const double lim = std::sqrt(6.0 / M.din[l]);
        std::uniform_real_distribution<double> U(-lim, lim);
        for (int64_t q = 0; q < (int64_t)M.din[l] * M.dout[l]; ++q) p[M.woff[l] + q] = (float)U(rng);
    }
    std::vector<float> nrm(2 * nin + 2 * nout, 0.f);
    for (int j = 0; j < nin; ++j) nrm[nin + j] = 1.f;
    for (int j = 0; j < nout; ++j) nrm[2 * nin + nout + j] = 1.f;
    hipStream_t st = Engine::get().stream();
    std::vector<float> z(M.np, 0.f);
    if (M.par.upload(p.data(), p.size() * 4, st) || M.grad.upload(z.data(), z.size() * 4, st) ||
        M.am.upload(z.data(), z.size() * 4, st) || M.av.upload(z.data(), z.size() * 4, st) ||
        M.norm.upload(nrm.data(), nrm.size() * 4, st) || hipStreamSynchronize(st) != hipSuccess) {
        delete h;
        return -3;
    }
    *out = h;
    return 0;
}

void cfdwm_mlp_destroy(cfdwm_mlp* h) {
    if (h) {
        (void)hipStreamSynchronize(Engine::get().stream());
        delete h;
    }
}

int64_t cfdwm_mlp_nparams(cfdwm_mlp* h) { return h ? h->m.np : -1; }

int cfdwm_mlp_get_params(cfdwm_mlp* h, float* out) {
    if (!h || !out) return -1;
    hipStream_t st = Engine::get().stream();
    CFDWM_HIP(hipMemcpyAsync(out, h->m.P(), h->m.np * 4, hipMemcpyDeviceToHost, st));
    CFDWM_HIP(hipStreamSynchronize(st));
    return 0;
}

int cfdwm_mlp_set_params(cfdwm_mlp* h, const float* in) {
    if (!h || !in) return -1;
    hipStream_t st = Engine::get().stream();
    CFDWM_HIP(hipMemcpyAsync(h->m.P(), in, h->m.np * 4, hipMemcpyHostToDevice, st));
    CFDWM_HIP(hipStreamSynchronize(st));
    h->m.adam_t = 0;
    return 0;
}

int cfdwm_mlp_set_norm(cfdwm_mlp* h, const float* in_mean, const float* in_std, const float* out_mean,
                       const float* out_std) {
    if (!h || !in_mean || !in_std || !out_mean || !out_std) return -1;
    const Mlp& M = h->m;
    for (int j = 0; j < M.nin; ++j) if (!(in_std[j] > 0)) return -1;
    for (int j = 0; j < M.nout; ++j) if (!(out_std[j] > 0)) return -1;
    std::vector<float> n(2 * M.nin + 2 * M.nout);
    std::memcpy(n.data(), in_mean, M.nin * 4);
    std::memcpy(n.data() + M.nin, in_std, M.nin * 4);
    std::memcpy(n.data() + 2 * M.nin, out_mean, M.nout * 4);
    std::memcpy(n.data() + 2 * M.nin + M.nout, out_std, M.nout * 4);
    hipStream_t st = Engine::get().stream();
    if (h->m.norm.upload(n.data(), n.size() * 4, st)) return -3;
    CFDWM_HIP(hipStreamSynchronize(st));
    return 0;
}

int cfdwm_mlp_get_norm(cfdwm_mlp* h, float* out) {
    if (!h || !out) return -1;
    hipStream_t st = Engine::get().stream();
    CFDWM_HIP(hipMemcpyAsync(out, h->m.norm.get(), (2 * h->m.nin + 2 * h->m.nout) * 4, hipMemcpyDeviceToHost, st));
    CFDWM_HIP(hipStreamSynchronize(st));
    return 0;
}

// Y = net(X) for n rows (device pointers, raw units), in chunks of at most 65536 rows.
int cfdwm_mlp_forward_device(cfdwm_mlp* h, int64_t n, const float* X, float* Y) {
    if (!h || n < 0 || (n && (!X || !Y))) return -1;
    Mlp& M = h->m;
    hipStream_t st = Engine::get().stream();
    // large batches: the fused kernel (256 blocks of 64 rows fill the GPU);
    // smaller ones run layer by layer, whose 64 x 64 output tiles give more blocks
    if (M.fused() && n >= 256 * kFiR) {
        MlpFused F;
        F.n = n; F.L = M.layers(); F.nin = M.nin; F.nout = M.nout;
        for (int l = 0; l < F.L; ++l) {
            F.din[l] = M.din[l]; F.dout[l] = M.dout[l];
            F.W[l] = M.P() + M.woff[l]; F.b[l] = M.P() + M.boff[l];
            F.woff[l + 1] = F.woff[l] + M.packed(l);
        }
        F.Wp = (uint16_t*)M.wpk.get();
        F.mu_in = M.nin_mu(); F.sd_in = M.nin_sd(); F.mu_out = M.nout_mu(); F.sd_out = M.nout_sd();
        F.X = X; F.Y = Y;
        hipLaunchKernelGGL(k_mlp_pack, dim3(nb256(F.woff[F.L] / 8)), dim3(256), 0, st, F);
        CFDWM_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_mlp_fused, dim3((unsigned)((n + kFiR - 1) / kFiR)), dim3(256), 0, st, F);
        CFDWM_HIP(hipGetLastError());
        return 0;
    }
    const int64_t chunk = 65536;
    if (M.reserve(std::min(n, chunk))) return -3;
    float* A = (float*)M.act.get();
    for (int64_t r0 = 0; r0 < n; r0 += chunk) {
        const int64_t nr = std::min(chunk, n - r0);
        hipLaunchKernelGGL(k_standardise, dim3(nb256(nr * M.nin)), dim3(256), 0, st, nr, M.nin, X + r0 * M.nin,
                           (const float*)M.nin_mu(), (const float*)M.nin_sd(), A + M.hoff(0));
        CFDWM_HIP(hipGetLastError());
        if (int e = M.forward(nr, st)) return e;
        float* out = A + M.hoff(M.layers());
        hipLaunchKernelGGL(k_unstandardise, dim3(nb256(nr * M.nout)), dim3(256), 0, st, nr, M.nout, out,
                           (const float*)M.nout_mu(), (const float*)M.nout_sd());
        CFDWM_HIP(hipGetLastError());
        CFDWM_HIP(hipMemcpyAsync(Y + r0 * M.nout, out, nr * M.nout * 4, hipMemcpyDeviceToDevice, st));
    }
    return 0;
}

// Loss (mean squared error of the standardised outputs) and its gradient over
// the first n rows (n <= 65536), gradient copied to grad_host when given.
int cfdwm_mlp_loss_grad_device(cfdwm_mlp* h, int64_t n, const float* X, const float* Y, float* loss,
                               float* grad_host) {
    if (!h || n <= 0 || n > 65536 || !X || !Y) return -1;
    Mlp& M = h->m;
    hipStream_t st = Engine::get().stream();
    if (M.reserve(n)) return -3;
    float* A = (float*)M.act.get();
    hipLaunchKernelGGL(k_gather_std, dim3(nb256(n * M.nin)), dim3(256), 0, st, n, M.nin, (const int64_t*)nullptr, X,
                       (const float*)M.nin_mu(), (const float*)M.nin_sd(), A + M.hoff(0));
    CFDWM_HIP(hipGetLastError());
    if (int e = M.forward(n, st)) return e;
    // targets standardised into the dY buffer's slot, then MSE in place
    float* Yb = (float*)M.tmp.get() + (M.tmp.size() / sizeof(float)) / 2;
    hipLaunchKernelGGL(k_gather_std, dim3(nb256(n * M.nout)), dim3(256), 0, st, n, M.nout, (const int64_t*)nullptr, Y,
                       (const float*)M.nout_mu(), (const float*)M.nout_sd(), Yb);
    CFDWM_HIP(hipGetLastError());
    const unsigned nbk = nb256(n * M.nout);
    float* dY = (float*)M.tmp.get();
    hipLaunchKernelGGL(k_mse, dim3(nbk), dim3(256), 0, st, n, M.nout, (const float*)(A + M.hoff(M.layers())),
                       (const float*)Yb, dY, (float*)M.part.get());
    CFDWM_HIP(hipGetLastError());
    if (int e = M.backward(n, dY, st)) return e;
    std::vector<float> pt(nbk);
    CFDWM_HIP(hipMemcpyAsync(pt.data(), M.part.get(), nbk * 4, hipMemcpyDeviceToHost, st));
    if (grad_host) CFDWM_HIP(hipMemcpyAsync(grad_host, M.G(), M.np * 4, hipMemcpyDeviceToHost, st));
    CFDWM_HIP(hipStreamSynchronize(st));
    double s = 0;
    for (float v : pt) s += v;
    if (loss) *loss = (float)(s / (double)(n * M.nout));
    return 0;
}

// Adam on minibatches of `batch` rows drawn (with a seeded generator) from the
// n rows of X / Y (device pointers, raw units); learning rate lr with cosine
// decay to lr / 20 over `steps`.  loss_curve[s] (optional, host) receives the
// minibatch loss every `report` steps (others 0).
int cfdwm_mlp_train_device(cfdwm_mlp* h, int64_t n, const float* X, const float* Y, int steps, int batch, float lr,
                           uint64_t seed, int report, float* loss_curve) {
    if (!h || n <= 0 || !X || !Y || steps < 0 || batch <= 0 || batch > 65536) return -1;
    Mlp& M = h->m;
    hipStream_t st = Engine::get().stream();
    const int64_t nbt = std::min<int64_t>(batch, n);
    if (M.reserve(nbt)) return -3;
    std::mt19937_64 rng(seed);
    std::uniform_int_distribution<int64_t> U(0, n - 1);
    std::vector<int64_t> id(nbt);
    float* A = (float*)M.act.get();
    float* dY = (float*)M.tmp.get();
    float* Yb = dY + (M.tmp.size() / sizeof(float)) / 2;
    const unsigned nbk = nb256(nbt * M.nout);
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (int s = 0; s < steps; ++s) {
        for (auto& v : id) v = U(rng);
        if (M.idx.upload(id.data(), nbt * sizeof(int64_t), st)) return -3;
        hipLaunchKernelGGL(k_gather_std, dim3(nb256(nbt * M.nin)), dim3(256), 0, st, nbt, M.nin,
                           (const int64_t*)M.idx.get(), X, (const float*)M.nin_mu(), (const float*)M.nin_sd(),
                           A + M.hoff(0));
        hipLaunchKernelGGL(k_gather_std, dim3(nb256(nbt * M.nout)), dim3(256), 0, st, nbt, M.nout,
                           (const int64_t*)M.idx.get(), Y, (const float*)M.nout_mu(), (const float*)M.nout_sd(), Yb);
        CFDWM_HIP(hipGetLastError());
        if (int e = M.forward(nbt, st)) return e;
        hipLaunchKernelGGL(k_mse, dim3(nbk), dim3(256), 0, st, nbt, M.nout, (const float*)(A + M.hoff(M.layers())),
                           (const float*)Yb, dY, (float*)M.part.get());
        CFDWM_HIP(hipGetLastError());
        if (int e = M.backward(nbt, dY, st)) return e;
        ++M.adam_t;
        const double frac = steps > 1 ? (double)s / (steps - 1) : 1.0;
        const float lrs = (float)(lr * (0.05 + 0.95 * 0.5 * (1.0 + std::cos(3.14159265358979323846 * frac))));
        const float c1 = (float)(1.0 - std::pow(b1, (double)M.adam_t)), c2 = (float)(1.0 - std::pow(b2, (double)M.adam_t));
        hipLaunchKernelGGL(k_adam, dim3(nb256(M.np)), dim3(256), 0, st, M.np, M.P(), (const float*)M.G(),
                           (float*)M.am.get(), (float*)M.av.get(), lrs, b1, b2, eps, c1, c2);
        CFDWM_HIP(hipGetLastError());
        if (loss_curve) {
            loss_curve[s] = 0.f;
            if (report > 0 && (s % report == 0 || s == steps - 1)) {
                std::vector<float> pt(nbk);
                CFDWM_HIP(hipMemcpyAsync(pt.data(), M.part.get(), nbk * 4, hipMemcpyDeviceToHost, st));
                CFDWM_HIP(hipStreamSynchronize(st));
                double q = 0;
                for (float v : pt) q += v;
                loss_curve[s] = (float)(q / (double)(nbt * M.nout));
            }
        }
    }
    CFDWM_HIP(hipStreamSynchronize(st));
    return 0;
}

}  // extern "C"
