// noalloc.hip — drp_reduce_noalloc: the diagnostics reductions of drp_reduce
// without any device allocation, for callers that cannot allocate (code under
// HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).
//
// drp_reduce keeps its partial sums in a buffer the lattice allocates on first
// use.  Here they, the total sums and the phi-range words live in one file-scope
// device array, `scratch`, which every GPU the library runs on holds until the
// process ends (REDUCE_WORK_DOUBLES doubles, 160 KiB + 128 B).  Both entry points run the
// same kernels over the same work items and return identical statistics.  Calls
// that overlap on one GPU share the array and race.
#include <hip/hip_runtime.h>

#include <mutex>

#include "../../include/droplet.h"
#include "d3q15.h"
#include "kernels.h"
#include "lattice_impl.h"

using namespace drp;

namespace {

constexpr int64_t REDUCE_NOALLOC_MAX_NODES = DRP_REDUCE_NOALLOC_MAX_NODES;  // 2^25, e.g. 512 x 256 x 256

// partial sums | total sums [NPART] | phi range slot (2 words) | pad
__device__ __align__(256) double scratch[REDUCE_WORK_DOUBLES];

// device address of `scratch` per device, looked up once per device with that
// device current (the host-side name is not a device address)
std::mutex g_mu;
double* g_scratch[64] = {};

int scratch_for(int dev, double** out) {
    std::lock_guard<std::mutex> lock(g_mu);
    if (dev < 0 || dev >= 64) return drp_fail(DRP_ERR_ARG, "device %d out of range", dev);
    if (!g_scratch[dev]) {
        int prev = -1;
        if (hipGetDevice(&prev) != hipSuccess) return drp_fail(DRP_ERR_HIP, "hipGetDevice failed");
        if (prev != dev && hipSetDevice(dev) != hipSuccess) return drp_fail(DRP_ERR_HIP, "hipSetDevice(%d) failed", dev);
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (prev != dev) (void)hipSetDevice(prev);
        if (e != hipSuccess || !p)
            return drp_fail(DRP_ERR_HIP, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
        g_scratch[dev] = (double*)p;
    }
    *out = g_scratch[dev];
    return DRP_OK;
}

}  // namespace

extern "C" int drp_reduce_noalloc(drp_lattice* L, drp_stats* st) {
    if (!L || !st) return drp_fail(DRP_ERR_ARG, "null argument");
    if (L->n > REDUCE_NOALLOC_MAX_NODES)
        return drp_fail(DRP_ERR_ARG, "drp_reduce_noalloc: %lld nodes exceed its maximum of %lld",
                        (long long)L->n, (long long)REDUCE_NOALLOC_MAX_NODES);
    if (!L->initialized) return drp_fail(DRP_ERR_STATE, "lattice not initialised");
    if (L->cfg.precision != DRP_FP64)
        return drp_fail(DRP_ERR_UNSUPPORTED, "drp_reduce_noalloc: FP64 lattices only (the FP32 FP64 view allocates)");
    double* ptr = nullptr;
    int rc = scratch_for(L->dev, &ptr);
    if (rc) return rc;
    hipError_t e = launch_reduce_fp64(L->G, L->phys, (const double*)L->mac[L->cur],
                                      L->range, (int)(L->step % 3), ptr, L->stream);
    if (e != hipSuccess) return drp_fail(DRP_ERR_HIP, "reduce launch failed: %s", hipGetErrorString(e));
    double host[NPART + 2];
    if ((e = hipMemcpyAsync(host, ptr + REDUCE_OUT, sizeof host, hipMemcpyDeviceToHost, L->stream)) != hipSuccess ||
        (e = hipStreamSynchronize(L->stream)) != hipSuccess)
        return drp_fail(DRP_ERR_HIP, "drp_reduce_noalloc copy failed: %s", hipGetErrorString(e));
    uint64_t rg[2];
    static_assert(sizeof(double) == sizeof(uint64_t), "range words");
    __builtin_memcpy(rg, host + NPART, sizeof rg);
    stats_from_sums(L, host, rg, st);
    return DRP_OK;
}
