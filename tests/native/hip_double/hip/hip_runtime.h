// A host-only double of the part of the HIP runtime that the library's host code calls,
// so that its copies, its devices and its failure paths can be tested without a GPU (and
// with more than one device).  Two devices; device memory is host memory; kernels run on
// the calling thread when they are launched, one thread after the other, so only kernels
// without barriers can run.  What the runtime's documentation asks of a caller is counted
// in `violations` when it is not met.
#pragma once

#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

enum hipError_t {
    hipSuccess = 0,
    hipErrorInvalidValue = 1,
    hipErrorOutOfMemory = 2,
    hipErrorInvalidConfiguration = 9,
    hipErrorInvalidHandle = 400
};
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice };
constexpr unsigned hipHostMallocPortable = 0x1, hipHostMallocMapped = 0x2, hipHostMallocCoherent = 0x40000000;
constexpr unsigned hipEventDisableTiming = 0x2, hipEventReleaseToSystem = 0x80000000;
constexpr unsigned hipStreamNonBlocking = 0x1;

struct dim3 {
    unsigned x, y, z;
    constexpr dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
struct double2 {
    double x, y;
};
inline double2 make_double2(double x, double y) { return {x, y}; }
inline int min(int a, int b) { return a < b ? a : b; }

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __shared__ static
#define __launch_bounds__(...)
#define __align__(n) alignas(n)

namespace hip_double {

struct Stream {
    int dev = 0;
    std::mutex m;
    std::condition_variable cv;
    bool stalled = false;  // its work does not end until this is taken back
    void wait() {
        std::unique_lock<std::mutex> lock(m);
        cv.wait(lock, [&] { return !stalled; });
    }
    void stall(bool on) {
        {
            std::lock_guard<std::mutex> lock(m);
            stalled = on;
        }
        cv.notify_all();
    }
};
struct Event {
    int dev = 0;
    unsigned flags = 0;
    Stream* stream = nullptr;
};
struct Block {
    size_t bytes;
    int dev;
    bool host;
    unsigned flags;
};

struct Runtime {
    std::mutex m;
    std::map<void*, Block> live;
    size_t device_limit = SIZE_MAX, device_bytes = 0;  // hipMalloc fails beyond the limit
    size_t largest = 0;                                // largest device allocation asked for since it was cleared
    std::atomic<int> copies{0}, launches{0};           // asked for since they were cleared
    int pinned_limit = 1 << 30;                        // blocks of pinned memory that can be had
    std::vector<std::string> violations;
    void violation(const std::string& s) {
        std::lock_guard<std::mutex> lock(m);
        violations.push_back(s);
    }
    int pinned_blocks() {
        int k = 0;
        for (auto& b : live) k += b.second.host;
        return k;
    }
};
inline Runtime rt;
inline thread_local int current = 0;
inline thread_local hipError_t last = hipSuccess;
inline thread_local dim3 block_idx, thread_idx, block_dim, grid_dim;
inline hipError_t fail(hipError_t e) { return last = e; }

template <typename... P, typename... A>
void launch(void (*kernel)(P...), dim3 grid, dim3 block, Stream* s, A&&... args) {
    if (s && s->dev != current) {
        rt.violation("kernel launched to a stream of another device");
        fail(hipErrorInvalidHandle);
        return;
    }
    rt.launches++;
    grid_dim = grid;
    block_dim = block;
    for (block_idx.x = 0; block_idx.x < grid.x; block_idx.x++)
        for (thread_idx.x = 0; thread_idx.x < block.x; thread_idx.x++) kernel(args...);
}

}  // namespace hip_double

using hipStream_t = hip_double::Stream*;
using hipEvent_t = hip_double::Event*;
using hipGraph_t = void*;
using hipGraphExec_t = void*;

#define blockIdx hip_double::block_idx
#define threadIdx hip_double::thread_idx
#define blockDim hip_double::block_dim
#define gridDim hip_double::grid_dim
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) \
    hip_double::launch(kernel, grid, block, stream, __VA_ARGS__)

// device functions that kernels on the double never reach
[[noreturn]] inline void hip_double_unsupported() { std::abort(); }
inline void __syncthreads() { hip_double_unsupported(); }
template <typename T> T __shfl_xor(T, int, int) { hip_double_unsupported(); }
inline void atomicMax(unsigned long long*, unsigned long long) { hip_double_unsupported(); }
inline void atomicMin(unsigned long long*, unsigned long long) { hip_double_unsupported(); }
inline double __builtin_amdgcn_rcp(double x) { return 1.0 / x; }
inline bool __builtin_amdgcn_class(double, int) { hip_double_unsupported(); }

inline const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
inline hipError_t hipGetLastError() {
    const hipError_t e = hip_double::last;
    hip_double::last = hipSuccess;
    return e;
}
inline hipError_t hipGetDeviceCount(int* n) { return *n = 2, hipSuccess; }
inline hipError_t hipGetDevice(int* d) { return *d = hip_double::current, hipSuccess; }
inline hipError_t hipSetDevice(int d) {
    if (d < 0 || d > 1) return hip_double::fail(hipErrorInvalidValue);
    hip_double::current = d;
    return hipSuccess;
}
inline hipError_t hipMalloc(void** p, size_t bytes) {
    std::lock_guard<std::mutex> lock(hip_double::rt.m);
    auto& rt = hip_double::rt;
    rt.largest = bytes > rt.largest ? bytes : rt.largest;
    if (bytes > rt.device_limit || rt.device_bytes > rt.device_limit - bytes) return hip_double::fail(hipErrorOutOfMemory);
    *p = std::malloc(bytes ? bytes : 1);
    rt.device_bytes += bytes;
    rt.live[*p] = {bytes, hip_double::current, false, 0};
    return hipSuccess;
}
inline hipError_t hipFree(void* p) {
    std::lock_guard<std::mutex> lock(hip_double::rt.m);
    auto it = hip_double::rt.live.find(p);
    if (it == hip_double::rt.live.end()) std::abort();
    hip_double::rt.device_bytes -= it->second.bytes;
    hip_double::rt.live.erase(it);
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t bytes, unsigned flags) {
    std::lock_guard<std::mutex> lock(hip_double::rt.m);
    if (hip_double::rt.pinned_blocks() >= hip_double::rt.pinned_limit) return hip_double::fail(hipErrorOutOfMemory);
    *p = std::malloc(bytes);
    hip_double::rt.live[*p] = {bytes, hip_double::current, true, flags};
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    std::lock_guard<std::mutex> lock(hip_double::rt.m);
    hip_double::rt.live.erase(p);
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = new hip_double::Stream;
    (*s)->dev = hip_double::current;
    return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s) { return delete s, hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s) { return s->wait(), hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags) {
    *e = new hip_double::Event{hip_double::current, flags, nullptr};
    return hipSuccess;
}
inline hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
inline hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (e->dev != s->dev) {
        hip_double::rt.violation("event recorded on a stream of another device");
        return hip_double::fail(hipErrorInvalidHandle);
    }
    e->stream = s;
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    if (e->stream) e->stream->wait();
    // an event without a system-scope release makes coherent host memory visible, no other
    bool coherent = true;
    {
        std::lock_guard<std::mutex> lock(hip_double::rt.m);
        for (auto& b : hip_double::rt.live) coherent &= !b.second.host || (b.second.flags & hipHostMallocCoherent);
    }
    if (!coherent && !(e->flags & hipEventReleaseToSystem))
        hip_double::rt.violation("event of device scope waited for before reading non-coherent host memory");
    return hipSuccess;
}
inline hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    hip_double::rt.copies++;
    return std::memcpy(d, s, n), hipSuccess;
}
inline hipError_t hipMemcpy2DAsync(void* d, size_t dpitch, const void* s, size_t spitch, size_t width, size_t height,
                                   hipMemcpyKind, hipStream_t) {
    hip_double::rt.copies++;
    for (size_t r = 0; r < height; r++) std::memcpy((char*)d + r * dpitch, (const char*)s + r * spitch, width);
    return hipSuccess;
}
inline hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
