// host_copy.hip -- device arrays to the caller's (pageable) memory.
//
// hipMemcpyAsync to pageable memory moves 16.5 GB/s here, and half of that into memory the caller
// has just allocated, whose pages the one copying thread also has to fault in.  Large copies go
// through pinned slots instead: each of a few threads takes every n-th piece, waits for its
// piece's DMA (57 GB/s over the link) and copies it on, so the page faults and the copies out
// of the slots run side by side and under the DMA of the next pieces.  The slots are shared by
// the process, one copy at a time (a second caller's goes the plain way), and are freed with the
// last grid.  Fields of 256^3 cells (537 MB) into fresh arrays: 55 -> 13 ms.
#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "internal.hpp"

namespace lumagpu {
namespace {

constexpr int kPipeThreads = 6;
constexpr size_t kPipeSlot = size_t(4) << 20;
// below: the plain copy takes no longer than starting the threads and faulting the pages in turn
constexpr size_t kPipeMin = size_t(12) << 20;

std::mutex g_pipe_mu;
int g_pipe_grids = 0;
void *g_pipe_pin = nullptr;

int cpus() {
    cpu_set_t set;
    CPU_ZERO(&set);
    if (sched_getaffinity(0, sizeof set, &set) != 0) return 1;
    return CPU_COUNT(&set);
}

// the grid's device current on this thread while the object lives: the caller's own thread, which copies
// too, gets back the device it had
struct DeviceGuard {
    int had = -1;
    hipError_t e;
    explicit DeviceGuard(int device) {
        e = hipGetDevice(&had);
        if (e == hipSuccess && had == device) had = -1;
        else if (e == hipSuccess) e = hipSetDevice(device);
    }
    DeviceGuard(const DeviceGuard &) = delete;
    DeviceGuard &operator=(const DeviceGuard &) = delete;
    ~DeviceGuard() {
        if (had >= 0) (void)hipSetDevice(had);
    }
};

// the pieces first, first + n, ... of one copy; each waits for its own DMA only
hipError_t copy_pieces(const lumagpu_grid *g, char *dst, const char *src, size_t bytes, int first, int n, char *pin,
                       std::atomic<bool> &stop) {
    const DeviceGuard device(g->device);
    if (device.e != hipSuccess) return device.e;
    hipEvent_t ev = nullptr;
    hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    if (e != hipSuccess) return e;
    for (size_t off = (size_t)first * kPipeSlot; off < bytes && e == hipSuccess && !stop; off += (size_t)n * kPipeSlot) {
        const size_t len = std::min(kPipeSlot, bytes - off);
        e = hipMemcpyAsync(pin, src + off, len, hipMemcpyDeviceToHost, g->stream);
        if (e == hipSuccess) e = hipEventRecord(ev, g->stream);
        if (e == hipSuccess) e = hipEventSynchronize(ev);
        if (e == hipSuccess) std::memcpy(dst + off, pin, len);
    }
    (void)hipEventDestroy(ev);
    if (e != hipSuccess) stop = true;
    return e;
}

}  // namespace

void host_copy_grid_added() {
    std::lock_guard<std::mutex> lock(g_pipe_mu);
    ++g_pipe_grids;
}

void host_copy_grid_gone() {
    std::lock_guard<std::mutex> lock(g_pipe_mu);
    if (--g_pipe_grids == 0 && g_pipe_pin) {
        (void)hipHostFree(g_pipe_pin);
        g_pipe_pin = nullptr;
    }
}

// bytes from device memory to dst, ordered on g's stream; dst is complete when the stream has
// been synchronised
int copy_to_host(const lumagpu_grid *g, void *dst, const void *src, size_t bytes) {
    const int n = (int)std::min<size_t>(std::min(kPipeThreads, cpus() / 2), bytes / kPipeSlot);
    std::unique_lock<std::mutex> lock(g_pipe_mu, std::defer_lock);
    if (bytes < kPipeMin || n < 2 || !lock.try_lock()) {
        HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g->stream));
        return 0;
    }
    if (!g_pipe_pin && hipHostMalloc(&g_pipe_pin, kPipeThreads * kPipeSlot, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        g_pipe_pin = nullptr;
        HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g->stream));
        return 0;
    }
    hipError_t err[kPipeThreads];
    std::fill(err, err + kPipeThreads, hipSuccess);
    std::atomic<bool> stop{false};
    std::thread th[kPipeThreads];
    char *d = static_cast<char *>(dst), *pin = static_cast<char *>(g_pipe_pin);
    const char *s = static_cast<const char *>(src);
    int started = 1;   // threads 1 .. started - 1 run; this thread takes the pieces of the rest
    try {
        for (; started < n; ++started)
            th[started] = std::thread([=, &stop, &err] { err[started] = copy_pieces(g, d, s, bytes, started, n, pin + started * kPipeSlot, stop); });
    } catch (const std::exception &) {
    }
    err[0] = copy_pieces(g, d, s, bytes, 0, n, pin, stop);
    for (int k = started; k < n && err[0] == hipSuccess; ++k) err[0] = copy_pieces(g, d, s, bytes, k, n, pin, stop);
    for (int k = 1; k < started; ++k) th[k].join();
    for (int k = 0; k < n; ++k)
        if (err[k] != hipSuccess) return fail(LUMAGPU_EHIP, std::string("copy to host: ") + hipGetErrorString(err[k]));
    return 0;
}

}  // namespace lumagpu
