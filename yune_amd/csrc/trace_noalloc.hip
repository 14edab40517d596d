// trace_noalloc.hip — traceRay on caller rays without allocating device
// memory: the variant of yn_trace for callers that cannot call hipMalloc
// (code under HIP graph capture, tight serving loops).
//
// What the call needs beyond the caller's inputs and outputs (the traversal
// stack's overflow area, the work counters and, where results are to be
// written over the rays, the rays) lives in `scratch`, one static device array
// per GPU.  Its device address is taken once per device with
// hipGetSymbolAddress at context creation; host code only ever uses that
// address, never the array's name (a host-side stand-in).  Every call on one
// GPU shares the array: calls that overlap on one GPU race.
#include <algorithm>
#include <mutex>

#include "yn_internal_dev.h"

namespace {

using namespace yune;

constexpr size_t kScratchBytes = 35663104;
// traversal stack overflow entries, 6 B each (a reference and a distance)
constexpr size_t kWorkBytes = sizeof(uint32_t) * kMaxXcd * kWorkStride;
constexpr size_t kOffWork = kScratchBytes - kWorkBytes;
static_assert(kOffWork % 256 == 0, "the scratch array's parts");

// Overflow entries in `bytes` of the array.
constexpr size_t ovf_entries(size_t bytes) { return bytes / 6 / 256 * 256; }

// Whether two arrays share memory.
bool overlap(const void* a, size_t na, const void* b, size_t nb)
{
    return (uintptr_t)a < (uintptr_t)b + nb && (uintptr_t)b < (uintptr_t)a + na;
}

}  // namespace

static __device__ __align__(256) uint8_t scratch[kScratchBytes];

namespace yune {

namespace {

// Clears the work counters.
__global__ __launch_bounds__(64) void k_na_clear(uint32_t* work)
{
    if (threadIdx.x < (unsigned)kMaxXcd) work[threadIdx.x * kWorkStride] = 0u;
}

std::mutex g_na_mu;
void* g_na_ptr[64] = {};

}  // namespace

int trace_noalloc_init(int device, void** ptr)
{
    if (device < 0 || device >= 64) return -1;
    std::lock_guard<std::mutex> lk(g_na_mu);
    if (!g_na_ptr[device]) {
        // the device is current (the caller set it); each GPU has its own copy
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return -1;
        g_na_ptr[device] = p;
    }
    *ptr = g_na_ptr[device];
    return 0;
}

// `max_depth`: traversal stack entries the scene can need; `max_grid`: the
// blocks that fit at once.
int trace_noalloc_enqueue(void* base, const RaysArgs& rays, int width, int lds, int max_depth, int max_grid,
                          hipStream_t s)
{
    if (!base || rays.n < 0 || rays.n > kTraceNoAllocMaxRays) return -1;
    if (rays.n == 0) return 0;
    uint8_t* b = static_cast<uint8_t*>(base);
    RaysArgs a = rays;
    // Results over the rays: the kernel writes a ray's while others are still
    // to be read, so it reads a copy (8 MB at most).
    const size_t n = (size_t)a.n;
    size_t used = 0;
    if (overlap(a.tri, 4 * n, a.rays, 32 * n) || overlap(a.light, 4 * n, a.rays, 32 * n) ||
        overlap(a.t, 4 * n, a.rays, 32 * n)) {
        used = (32 * n + 255) / 256 * 256;
        if (hipMemcpyAsync(b, a.rays, 32 * n, hipMemcpyDeviceToDevice, s) != hipSuccess) return -1;
        a.rays = reinterpret_cast<const float*>(b);
        a.aligned = 1;
    }
    const size_t ovf = ovf_entries(kOffWork - used);
    a.ovf_ref = reinterpret_cast<uint32_t*>(b + used);
    a.ovf_t = reinterpret_cast<uint16_t*>(b + used + 4 * ovf);
    a.work = reinterpret_cast<uint32_t*>(b + kOffWork);
    // as many entries per thread as the scene needs, kTraceNoAllocOvfDepth
    // beyond the configured LDS part at most (a deeper traversal stops there
    // and raises the overflow flag), and as many threads as then have room
    const int entries = std::min(max_depth, trace_lds_stack(lds) + kTraceNoAllocOvfDepth);
    a.ovf_depth = std::max(entries - rays_lds_stack(lds), 0);
    const size_t threads = ovf / (size_t)std::max(a.ovf_depth, 1);
    const int grid = (int)std::min<size_t>((size_t)max_grid, threads / kRaysBlock);
    if ((int64_t)a.n > (int64_t)(grid / a.n_slices) * a.n_slices * kRaysBlock)
        hipLaunchKernelGGL(k_na_clear, dim3(1), dim3(64), 0, s, a.work);
    launch_rays(a, width, lds, grid, s);
    return 0;
}

}  // namespace yune
