// host_io.hip — node arrays to the caller's host memory, and from there.
//
// The caller's arrays are pageable, and usually fresh: the runtime's own copy moves
// them through one staging buffer with one host thread, which also takes the page
// faults, at 8..10 GB/s (66 ms for the five fields of a 256^3 lattice, as long as 30 of
// its steps).  Here a kernel drops the row padding (and widens FP32 deviations)
// straight into pinned host memory, chunk by chunk, and several host threads copy the
// chunks out (one thread, for short arrays), so that the link, the copies and the page
// faults overlap: 19 ms.  Arrays from the host go the same way back, except where the
// runtime's copies are the faster ones.
//
// The pinned chunks belong to the process: at most POOL_SLOTS of CHUNK_BYTES (64 MiB),
// made on demand, shared by all lattices and threads, and freed with the last lattice.  A
// transfer takes what is free and never waits for another one, whose stream may stand
// still for as long as its owner likes: one that finds none goes by the runtime's copies.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "../../include/droplet.h"
#include "kernels.h"
#include "lattice_impl.h"

using namespace drp;

namespace {

constexpr size_t CHUNK_BYTES = (size_t)4 << 20;
constexpr int64_t CHUNK = (int64_t)(CHUNK_BYTES / sizeof(double));
constexpr int MAX_SLOTS = 8;               // chunks of one transfer
constexpr int POOL_SLOTS = 2 * MAX_SLOTS;  // chunks of the process
// Doubles (16 MiB) that are worth a host thread.  Shorter transfers use the caller's
// thread alone, two chunks deep: in a program whose other threads are busy (spinning
// OpenMP workers on every core) eight threads took 38 ms for the 60 fields of twelve
// FP32 members of 48..128^3, one thread 18 ms; the fields of 256^3 take 86 ms with
// one and 35 ms with eight threads there, 63 and 17 ms on idle cores.
constexpr int64_t PER_THREAD = (int64_t)1 << 21;
// Host arrays of DIRECT_MIN doubles (512 KiB) or more go in by the runtime's copies as long as
// they are DIRECT_TOTAL (16 MiB) together, which it reads where they lie faster than one
// thread fills chunks: three force fields of 64^3 190 us, by chunks 234.  Shorter ones it may
// write through the bus at 3 GB/s (24^3 44 or 150 us, by chunks 35), longer ones it moves
// one after the other (populations of 128^3 8.4 ms, by chunks 5.2; of 64^3 880 us and 790).
constexpr int64_t DIRECT_MIN = (int64_t)1 << 16, DIRECT_TOTAL = (int64_t)1 << 21;
constexpr int64_t SHORT_CHUNK = (int64_t)1 << 17;  // doubles (1 MiB): smallest chunk of a transfer in parts

// values [first, first + len) of the contiguous sequence of node arrays (nx ny nz
// each), G.ns apart in memory, FP32 ones added to ref[array]
template <typename T>
__global__ __launch_bounds__(256) void pack_out(Grid G, const T* __restrict__ nodes, HostRef ref, int64_t first,
                                                int64_t len, double* __restrict__ out) {
    const int64_t n = (int64_t)G.nx * G.ny * G.nz;
    for (int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; j < len; j += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = first + j, a = i / n, s = i - a * n, row = s / G.nx;
        const T v = nodes[a * G.ns + G.px * row + (s - row * G.nx)];
        double d = (double)v;
        if (sizeof(T) == 4 && ref.r[a] != 0.0) d = ref.r[a] + d;
        out[j] = d;
    }
}

class Slots {
  public:
    void retain() {
        std::lock_guard<std::mutex> lock(mu_);
        users_++;
    }
    void release() {
        std::lock_guard<std::mutex> lock(mu_);
        if (--users_ > 0) return;
        for (void* p : free_) (void)hipHostFree(p);  // no lattice, so no transfer: all are here
        made_ -= (int)free_.size();
        free_.clear();
    }
    // up to `want` chunks: fewer, or none, where other transfers hold them or pinned
    // memory cannot be had
    std::vector<void*> take(int want) {
        std::vector<void*> got;
        got.reserve(want);
        int make = 0;
        {
            std::lock_guard<std::mutex> lock(mu_);
            free_.reserve(POOL_SLOTS);  // so that giving back cannot fail
            while ((int)got.size() < want && !free_.empty()) {
                got.push_back(free_.back());
                free_.pop_back();
            }
            make = std::min(want - (int)got.size(), POOL_SLOTS - made_);
            made_ += make;
        }
        for (; make > 0; make--) {
            void* p = nullptr;
            // coherent, whatever the environment's default: an event's wait makes only such memory visible
            if (hipHostMalloc(&p, CHUNK_BYTES, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) !=
                hipSuccess) {
                (void)hipGetLastError();
                std::lock_guard<std::mutex> lock(mu_);
                made_ -= make;
                break;
            }
            got.push_back(p);
        }
        return got;
    }
    void give(const std::vector<void*>& v) {
        std::lock_guard<std::mutex> lock(mu_);
        free_.insert(free_.end(), v.begin(), v.end());
    }

  private:
    std::mutex mu_;
    std::vector<void*> free_;
    int made_ = 0, users_ = 0;
};

Slots& slots() {
    static Slots* s = new Slots;  // outlives every static of the caller
    return *s;
}

template <typename T>
hipError_t launch_pack(const Grid& G, const T* nodes, const HostRef& ref, int64_t first, int64_t len, double* out,
                       hipStream_t st) {
    const unsigned nb = (unsigned)std::min<int64_t>((len + 255) / 256, 1024);
    hipLaunchKernelGGL(pack_out<T>, dim3(nb), dim3(256), 0, st, G, nodes, ref, first, len, out);
    return hipGetLastError();
}

// One array after the other by the runtime's own copies, for a transfer that gets no
// pinned chunk: packed on the device, or row by row where that has no memory for it.
template <typename T>
int to_host_unpinned(drp_lattice* L, const Grid& G, const T* nodes, int count, const HostRef& ref, double* host) {
    const bool doubles = sizeof(T) == sizeof(double);
    const int64_t n = (int64_t)G.nx * G.ny * G.nz;
    const size_t row = G.nx * sizeof(double);
    double* const pack = doubles && G.px == G.nx ? nullptr : pack_buffer(L, n);
    if (!doubles && !pack) return drp_fail(DRP_ERR_ALLOC, "no device memory to widen an array");
    hipError_t e = hipSuccess;
    for (int a = 0; a < count && e == hipSuccess; a++) {
        const T* src = nodes + a * G.ns;
        double* const dst = host + a * n;
        if (pack) {
            e = launch_pack(G, nodes, ref, a * n, n, pack, L->stream);
            if (e == hipSuccess) e = hipMemcpyAsync(dst, pack, n * sizeof(double), hipMemcpyDeviceToHost, L->stream);
        } else if (G.px == G.nx) {
            e = hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyDeviceToHost, L->stream);
        } else {
            e = hipMemcpy2DAsync(dst, row, src, G.px * sizeof(double), row, (size_t)G.ny * G.nz, hipMemcpyDeviceToHost,
                                 L->stream);
        }
    }
    const hipError_t s = hipStreamSynchronize(L->stream);
    if (e == hipSuccess) e = s;
    if (e != hipSuccess) return drp_fail(DRP_ERR_HIP, "copy to the host failed: %s", hipGetErrorString(e));
    return DRP_OK;
}

// Moves `total` values in chunks, each by launch(first, len, chunk), a kernel between the
// node arrays and the pinned chunk, and copy(first, len, chunk), the host's part: after the
// kernel to the host (OUT), before it from there.  `found` is false where there is no chunk.
template <bool OUT, typename Launch, typename Copy>
int transfer(drp_lattice* L, int64_t total, Launch&& launch, Copy&& copy, bool* found) {
    const int cores = std::max(1, (int)std::thread::hardware_concurrency());
    const int want = (int)std::max<int64_t>(1, std::min<int64_t>({MAX_SLOTS, cores, total / PER_THREAD}));
    std::vector<void*> slot;
    try {
        slot = slots().take(want == 1 && total > SHORT_CHUNK ? 2 : want);
    } catch (...) {
        return drp_fail(DRP_ERR_ALLOC, "host allocation failed");
    }
    *found = !slot.empty();
    if (slot.empty()) return DRP_OK;
    const int nt = std::min<int>(want, (int)slot.size()), deep = want == 1 ? (int)slot.size() : 1;
    const int64_t chunk = std::min(CHUNK, nt > 1 ? (total + nt - 1) / nt : std::max(SHORT_CHUNK, (total + 3) / 4));
    const int64_t chunks = (total + chunk - 1) / chunk;
    std::atomic<int64_t> next{0};
    std::atomic<int> failed{(int)hipSuccess};
    // each thread takes the next chunk and moves it through its slot (with two slots the other
    // one meanwhile)
    auto work = [&](int t, bool own_thread) {
        hipError_t e = own_thread ? hipSetDevice(L->dev) : hipSuccess;
        hipEvent_t ev[2] = {nullptr, nullptr};
        int64_t chunk_of[2] = {chunks, chunks};
        for (int k = 0; k < deep && e == hipSuccess && chunks > 1; k++)
            e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
        auto len_of = [&](int k) { return std::min(chunk, total - chunk_of[k] * chunk); };
        auto fill = [&](int k) {
            chunk_of[k] = next.fetch_add(1);
            if (chunk_of[k] >= chunks || e != hipSuccess) return;
            if (!OUT) copy(chunk_of[k] * chunk, len_of(k), (double*)slot[t + k]);
            e = launch(chunk_of[k] * chunk, len_of(k), (double*)slot[t + k]);
            if (e == hipSuccess && ev[k]) e = hipEventRecord(ev[k], L->stream);
        };
        for (int k = 0; k < deep; k++) fill(k);
        for (int k = 0; e == hipSuccess && chunk_of[k] < chunks && failed.load() == (int)hipSuccess; k = (k + 1) % deep) {
            e = ev[k] ? hipEventSynchronize(ev[k]) : hipStreamSynchronize(L->stream);
            if (e != hipSuccess) break;
            if (OUT) copy(chunk_of[k] * chunk, len_of(k), (double*)slot[t + k]);
            fill(k);
        }
        for (int k = 0; k < 2; k++)
            if (ev[k]) (void)hipEventDestroy(ev[k]);
        if (e != hipSuccess) failed.store((int)e);
    };
    std::thread threads[MAX_SLOTS];
    int started = 1;
    try {
        for (; started < nt; started++) threads[started] = std::thread(work, started, true);
    } catch (const std::system_error&) {
        // fewer threads then: the chunks go to those there are
    }
    work(0, false);
    for (int t = 1; t < started; t++) threads[t].join();
    // (a failed transfer may still have a kernel at work on a slot)
    if (failed.load() != (int)hipSuccess) (void)hipStreamSynchronize(L->stream);
    slots().give(slot);
    const hipError_t e = (hipError_t)failed.load();
    if (e != hipSuccess)
        return drp_fail(DRP_ERR_HIP, "copy %s the host failed: %s", OUT ? "to" : "from", hipGetErrorString(e));
    return DRP_OK;
}

template <typename T>
int to_host(drp_lattice* L, const Grid& G, const T* nodes, int count, const HostRef& ref, double* host) {
    const OnDevice on(L->dev);
    bool found = false;
    const int rc = transfer<true>(
        L, (int64_t)G.nx * G.ny * G.nz * count,
        [&](int64_t first, int64_t len, double* slot) { return launch_pack(G, nodes, ref, first, len, slot, L->stream); },
        [&](int64_t first, int64_t len, double* slot) { std::memcpy(host + first, slot, len * sizeof(double)); }, &found);
    return rc || found ? rc : to_host_unpinned(L, G, nodes, count, ref, host);
}

// values [first, first + len) of the arrays that follow each other, from a chunk to the
// node arrays
__global__ __launch_bounds__(256) void unpack_in(Grid G, const double* __restrict__ in, int64_t first, int64_t len,
                                                 double* __restrict__ nodes) {
    const int64_t n = (int64_t)G.nx * G.ny * G.nz;
    for (int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; j < len; j += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = first + j, a = i / n, s = i - a * n, row = s / G.nx;
        nodes[a * G.ns + G.px * row + (s - row * G.nx)] = in[j];
    }
}

hipError_t launch_unpack(const Grid& G, const double* in, int64_t first, int64_t len, double* nodes, hipStream_t st) {
    const unsigned nb = (unsigned)std::min<int64_t>((len + 255) / 256, 1024);
    hipLaunchKernelGGL(unpack_in, dim3(nb), dim3(256), 0, st, G, in, first, len, nodes);
    return hipGetLastError();
}

// Host arrays by the runtime's own copies: padded rows through a buffer without gaps, as
// many arrays at a time as DIRECT_TOTAL holds, or row by row where there is no memory for
// one; one copy for arrays that lie behind each other on both sides.
int from_host_direct(drp_lattice* L, const double* const* host, int count, double* nodes) {
    const Grid& G = L->G;
    const int64_t n = L->n;
    const size_t row = G.nx * sizeof(double);
    const bool padded = G.px != G.nx;
    int group = padded ? (int)std::max<int64_t>(1, std::min<int64_t>(count, DIRECT_TOTAL / n)) : count;
    double* pack = nullptr;
    while (padded && !(pack = pack_buffer(L, (size_t)group * n)) && group > 1) group /= 2;
    hipError_t e = hipSuccess;
    for (int k0 = 0; k0 < count && e == hipSuccess; k0 += group) {
        const int k1 = std::min(count, k0 + group);
        for (int k = k0, next; k < k1 && e == hipSuccess; k = next) {
            double* const dst = pack ? pack + (k - k0) * n : nodes + k * G.ns;
            next = k + 1;
            if (pack || (!padded && G.ns == n))
                while (next < k1 && host[next] == host[next - 1] + n) next++;
            if (pack || !padded)
                e = hipMemcpyAsync(dst, host[k], (next - k) * n * sizeof(double), hipMemcpyHostToDevice, L->stream);
            else
                e = hipMemcpy2DAsync(dst, G.px * sizeof(double), host[k], row, row, (size_t)G.ny * G.nz,
                                     hipMemcpyHostToDevice, L->stream);
        }
        if (pack && e == hipSuccess) e = launch_unpack(G, pack, 0, (k1 - k0) * n, nodes + k0 * G.ns, L->stream);
    }
    const hipError_t s = hipStreamSynchronize(L->stream);
    if (e == hipSuccess) e = s;
    if (e != hipSuccess) return drp_fail(DRP_ERR_HIP, "copy from the host failed: %s", hipGetErrorString(e));
    return DRP_OK;
}

}  // namespace

void host_io_retain() { slots().retain(); }
void host_io_release() { slots().release(); }

int nodes_to_host(drp_lattice* L, const double* nodes, int count, double* host) {
    return to_host(L, L->G, nodes, count, HostRef{}, host);
}

int nodes_to_host(drp_lattice* L, const float* nodes, int count, const HostRef& ref, double* host) {
    return to_host(L, L->G, nodes, count, ref, host);
}

int dense_to_host(drp_lattice* L, const double* values, double* host) {
    return to_host(L, Grid{L->G.nx, L->G.ny, L->G.nz, L->G.nx, L->n}, values, 1, HostRef{}, host);
}

int nodes_from_host(drp_lattice* L, const double* const* host, int count, double* nodes) {
    const OnDevice on(L->dev);
    const int64_t n = L->n, total = n * count;
    bool found = false;
    if (n < DIRECT_MIN || total > DIRECT_TOTAL) {
        const int rc = transfer<false>(
            L, total,
            [&](int64_t first, int64_t len, double* slot) { return launch_unpack(L->G, slot, first, len, nodes, L->stream); },
            [&](int64_t first, int64_t len, double* slot) {
                while (len > 0) {
                    const int64_t a = first / n, at = first - a * n, m = std::min(len, n - at);
                    std::memcpy(slot, host[a] + at, m * sizeof(double));
                    first += m;
                    slot += m;
                    len -= m;
                }
            },
            &found);
        if (rc || found) return rc;
    }
    return from_host_direct(L, host, count, nodes);
}

int nodes_from_host(drp_lattice* L, const double* host, int count, double* nodes) {
    const double* h[15];
    for (int k = 0; k < count; k++) h[k] = host + k * L->n;
    return nodes_from_host(L, h, count, nodes);
}
