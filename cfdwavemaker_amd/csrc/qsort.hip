// Cell order for large spline-query batches.
//
// Queries in the caller's order (a random point cloud) make the blocks of
// every XCD read all of the packed grid; grouped by tiles of neighbouring
// columns the node records around them are read about once per batch.  The
// order inside a tile does not matter (four lanes load a query's records
// together, k_query), so one counting pass over at most 16384 tiles replaces a
// sort: blocks count their queries per tile, the counts are scanned per tile
// over the blocks and then over the tiles, and each block writes its queries'
// records (coordinates and index in the caller's arrays) into its ranges.  No
// global atomics; the query kernel then reads its inputs contiguously and only
// its outputs are scattered (to the caller's order).
//
// Measured (256 x 256 x 16 FP32 grid, ordering / query kernel, us): 1e6 queries
// 37 / 73 with 4096 tiles of 4 x 4 columns (a radix sort by column and a record
// per lane took 230 / 104), 1e7 queries 308 / 607 with 16384 tiles of 2 x 2
// columns (with the query kernel of that time, 642: 4096 tiles 250 / 748, radix
// sort 380 / 806).  At 1e7 the scattered records and results, 16 bytes to a line
// each, take about 250 of these.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "engine.hpp"
#include "kernels.hpp"

namespace cfdwm {

namespace {

constexpr int kBinThreads = 1024, kMaxBins = kQueryBins, kMaxBinBlocks = kQueryBinBlocks;

// Tiles of 2^shift x 2^shift columns, and the blocks' share of the queries.
struct BinPlan {
    int shift = 0, ty = 1, bins = 1, blocks = 1;
    int64_t chunk = 0;
};
BinPlan bin_plan(int64_t n, int nx, int ny) {
    BinPlan b;
    // about 64 queries per tile or more: a wavefront's queries share a tile
    const int64_t most = std::min<int64_t>(kMaxBins, std::max<int64_t>(64, n / 64));
    auto tiles = [&](int s) { return (((int64_t)nx + (1 << s) - 1) >> s) * (((int64_t)ny + (1 << s) - 1) >> s); };
    while (tiles(b.shift) > most) ++b.shift;
    b.ty = (ny + (1 << b.shift) - 1) >> b.shift;
    b.bins = (int)tiles(b.shift);
    b.chunk = std::max<int64_t>(kBinThreads, (n + kMaxBinBlocks - 1) / kMaxBinBlocks);
    b.blocks = (int)((n + b.chunk - 1) / b.chunk);
    return b;
}

// tile of the cell holding (x, y), with the edge clamps of the query kernel
// (the order only affects locality, not results)
template <typename TQ>
__device__ __forceinline__ int bin_of(const GridGeom& g, double inv_dx, double inv_dy, TQ x, TQ y, int shift, int ty) {
    double cx = ((double)x - g.x0) * inv_dx;
    cx = cx < (g.nx - 1.) ? cx : (g.nx - 1.);
    cx = cx > 0. ? cx : 0.;
    double cy = ((double)y - g.y0) * inv_dy;
    cy = cy < (g.ny - 1.) ? cy : (g.ny - 1.);
    cy = cy > 0. ? cy : 0.;
    return ((int)cx >> shift) * ty + ((int)cy >> shift);
}

// counts[block][bin]
template <typename TQ>
__global__ __launch_bounds__(kBinThreads) void k_bin_count(int64_t n, GridGeom g, double inv_dx, double inv_dy,
                                                           const TQ* __restrict__ x, const TQ* __restrict__ y, int shift,
                                                           int ty, int bins, int64_t chunk, uint32_t* __restrict__ counts) {
    __shared__ uint32_t h[kMaxBins];
    for (int b = threadIdx.x; b < bins; b += kBinThreads) h[b] = 0;
    __syncthreads();
    const int64_t p1 = min(n, ((int64_t)blockIdx.x + 1) * chunk);
    for (int64_t p = (int64_t)blockIdx.x * chunk + threadIdx.x; p < p1; p += kBinThreads)
        atomicAdd(&h[bin_of(g, inv_dx, inv_dy, x[p], y[p], shift, ty)], 1u);
    __syncthreads();
    for (int b = threadIdx.x; b < bins; b += kBinThreads) counts[(int64_t)blockIdx.x * bins + b] = h[b];
}

// Per bin, counts become the exclusive sums over the blocks; total[bin] their
// sum.  A block takes 64 bins, four threads per bin a quarter of the blocks each.
__global__ __launch_bounds__(256) void k_bin_columns(int bins, int blocks, uint32_t* __restrict__ counts,
                                                     uint32_t* __restrict__ total) {
    __shared__ uint32_t part[4][64];
    const int b = blockIdx.x * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6;
    const int per = (blocks + 3) / 4, k0 = q * per, k1 = min(blocks, k0 + per);
    uint32_t s = 0;
    if (b < bins) {
#pragma unroll 8
        for (int k = k0; k < k1; ++k) s += counts[(int64_t)k * bins + b];
    }
    part[q][threadIdx.x & 63] = s;
    __syncthreads();
    uint32_t run = 0;
    for (int k = 0; k < q; ++k) run += part[k][threadIdx.x & 63];
    if (b >= bins) return;
    if (q == 3) total[b] = run + s;
#pragma unroll 8
    for (int k = k0; k < k1; ++k) {
        const uint32_t c = counts[(int64_t)k * bins + b];
        counts[(int64_t)k * bins + b] = run;
        run += c;
    }
}

// exclusive scan of total (one block; at most 16 bins per thread)
__global__ __launch_bounds__(kBinThreads) void k_bin_scan(int bins, uint32_t* __restrict__ total) {
    __shared__ uint32_t w[kBinThreads];
    const int t = threadIdx.x;
    uint32_t v[16], s = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int b = 16 * t + k;
        v[k] = b < bins ? total[b] : 0u;
        s += v[k];
    }
    w[t] = s;
    __syncthreads();
    for (int d = 1; d < kBinThreads; d <<= 1) {
        const uint32_t o = t >= d ? w[t - d] : 0u;
        __syncthreads();
        w[t] += o;
        __syncthreads();
    }
    uint32_t run = w[t] - s;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const int b = 16 * t + k;
        if (b < bins) total[b] = run;
        run += v[k];
    }
}

template <typename TQ>
__global__ __launch_bounds__(kBinThreads) void k_bin_place(int64_t n, GridGeom g, double inv_dx, double inv_dy,
                                                           const TQ* __restrict__ x, const TQ* __restrict__ y,
                                                           const TQ* __restrict__ z, int shift, int ty, int bins,
                                                           int64_t chunk, const uint32_t* __restrict__ counts,
                                                           const uint32_t* __restrict__ total, QRec<TQ>* __restrict__ rec) {
    __shared__ uint32_t h[kMaxBins];
    for (int b = threadIdx.x; b < bins; b += kBinThreads) h[b] = total[b] + counts[(int64_t)blockIdx.x * bins + b];
    __syncthreads();
    const int64_t p1 = min(n, ((int64_t)blockIdx.x + 1) * chunk);
    for (int64_t p = (int64_t)blockIdx.x * chunk + threadIdx.x; p < p1; p += kBinThreads) {
        QRec<TQ> r;
        r.x = x[p]; r.y = y[p]; r.z = z[p];
        r.p = (decltype(r.p))p;
        const uint32_t at = atomicAdd(&h[bin_of(g, inv_dx, inv_dy, r.x, r.y, shift, ty)], 1u);
        rec[at] = r;
    }
}

}  // namespace

size_t query_bins_bytes(int64_t n, int nx, int ny) {
    const BinPlan b = bin_plan(n, nx, ny);
    return ((size_t)b.blocks * b.bins + b.bins) * sizeof(uint32_t);
}

template <typename TQ>
hipError_t launch_query_bins(int64_t n, const GridGeom& g, const TQ* x, const TQ* y, const TQ* z, uint32_t* counts,
                             QRec<TQ>* recs, hipStream_t st) {
    if (n <= 0 || n > INT32_MAX || g.nx < 1 || g.ny < 1) return hipErrorInvalidValue;
    const BinPlan b = bin_plan(n, g.nx, g.ny);
    uint32_t* total = counts + (size_t)b.blocks * b.bins;
    // (a grid one column wide has dx or dy 0: its cell index is then 0 by the clamps)
    const double ix = 1.0 / g.dx, iy = 1.0 / g.dy;
    hipLaunchKernelGGL(k_bin_count<TQ>, dim3(b.blocks), dim3(kBinThreads), 0, st, n, g, ix, iy, x, y, b.shift, b.ty,
                       b.bins, b.chunk, counts);
    hipLaunchKernelGGL(k_bin_columns, dim3((b.bins + 63) / 64), dim3(256), 0, st, b.bins, b.blocks, counts, total);
    hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(kBinThreads), 0, st, b.bins, total);
    hipLaunchKernelGGL(k_bin_place<TQ>, dim3(b.blocks), dim3(kBinThreads), 0, st, n, g, ix, iy, x, y, z, b.shift, b.ty,
                       b.bins, b.chunk, (const uint32_t*)counts, (const uint32_t*)total, recs);
    return hipGetLastError();
}

template hipError_t launch_query_bins<float>(int64_t, const GridGeom&, const float*, const float*, const float*,
                                             uint32_t*, QRec<float>*, hipStream_t);
template hipError_t launch_query_bins<double>(int64_t, const GridGeom&, const double*, const double*, const double*,
                                              uint32_t*, QRec<double>*, hipStream_t);

}  // namespace cfdwm
