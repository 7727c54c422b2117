// Allocation-free device spline query: the variant of
// cfdwm_grid_query_device_f32 for callers that cannot allocate device memory
// (code under HIP graph capture, tight serving loops, harnesses that forbid
// hipMalloc).  Batches of 65,536 queries or more are evaluated in cell order;
// the tile counts and query records of that ordering live here in a file-scope
// device array instead of the grid's own buffers.  Each GPU holds
// its own copy of the array until the process ends.  Calls are enqueued on
// the library stream, one after another, so they never overlap; a caller that
// enqueued a query on another stream while one of these runs would race for
// the array.  Nothing in the array needs clearing: the counting pass writes
// every count, the placing pass every record.
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>

#include "engine.hpp"

namespace cfdwm {

namespace {
// the entry's limit, and what its ordering buffers take on the grid of most
// tiles: counts and totals, then records (33.1 MiB)
constexpr int64_t kMaxQueries = 1115336;
constexpr size_t kScratchBytes = (size_t)(kQueryBinBlocks + 1) * kQueryBins * sizeof(uint32_t) +
                                 ((size_t)kMaxQueries * sizeof(QRec<float>) + 255) / 256 * 256;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of this GPU's scratch array, looked up once per device with
// that device current.  In host code the array's name is only a stand-in:
// kernels and copies take this address, never the name.
int scratch_address(void** out) {
    *out = nullptr;
    int dev = 0;
    CFDWM_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) {
        set_error("allocation-free query: device index out of range");
        return -1;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        CFDWM_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) {
            set_error("allocation-free query: no device address for the scratch array");
            return -3;
        }
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}
}  // namespace

int query_device_f32_noalloc(Grid& grid, int64_t n, double t, const float* x, const float* y, const float* z,
                             float* eta, float* u, float* v, float* w) {
    if (n <= 0) return 0;
    if (int e = Engine::get().init()) return e;
    if (n > kMaxQueries) {
        set_error("allocation-free query: " + std::to_string(n) + " queries exceed the maximum of " +
                  std::to_string(kMaxQueries));
        return -1;
    }
    void* ws = nullptr;
    if (query_ws_bytes<float>(n, grid.g.nx, grid.g.ny) > 0)
        if (int e = scratch_address(&ws)) return e;
    return grid.query_device_f32(n, t, x, y, z, eta, u, v, w, nullptr, ws, kScratchBytes);
}

}  // namespace cfdwm
