// A stand-in for the allocation calls of the HIP runtime that libluma_amd.so makes, loaded before it
// with RTLD_GLOBAL: each goes on to the runtime's own unless a limit set here refuses it.  So a test
// can run the library short of device memory without filling the device.  And its launches: one can be
// made to fail.
#include <dlfcn.h>

#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <thread>

namespace {
constexpr int kOutOfMemory = 2;   // hipErrorOutOfMemory
std::mutex mu;
std::map<void *, size_t> live;
long long budget = -1;            // bytes that may still be allocated; < 0: no limit
size_t refused_size = 0;          // allocations of exactly this many bytes fail
bool until_freed = false;         // ... until something of 1 MiB or more has been freed
size_t total_shown = 0;           // what hipMemGetInfo reports as the device's memory (0: the truth)
int device_shown = -1;            // a current device for the watched thread alone (< 0: the truth)
size_t held = 0;
int calls = 0, refusals = 0;
int failing_launch = 0;           // this launch from now fails (1: the next); 0: none
int launch_error = 0;             // what hipGetLastError then reports, once
std::thread::id watched;
int watched_set_device = 0;

void *runtime() {
    static void *h = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL);
    if (!h) {
        std::fprintf(stderr, "alloc_limit: %s\n", dlerror());
        std::abort();
    }
    return h;
}
template <class F>
F *own(const char *name) {
    void *p = dlsym(runtime(), name);
    if (!p) std::abort();
    return reinterpret_cast<F *>(p);
}
}  // namespace

extern "C" {
int hipMalloc(void **p, size_t n) {
    static auto *f = own<int(void **, size_t)>("hipMalloc");
    std::lock_guard<std::mutex> lock(mu);
    ++calls;
    if ((budget >= 0 && n > (size_t)budget) || (refused_size && n == refused_size)) {
        ++refusals;
        return kOutOfMemory;
    }
    const int e = f(p, n);
    if (e == 0) {
        live[*p] = n;
        held += n;
        if (budget >= 0) budget -= (long long)n;
    }
    return e;
}
int hipFree(void *p) {
    static auto *f = own<int(void *)>("hipFree");
    std::lock_guard<std::mutex> lock(mu);
    const auto it = live.find(p);
    if (it != live.end()) {
        held -= it->second;
        if (budget >= 0) budget += (long long)it->second;
        if (until_freed && it->second >= (size_t(1) << 20)) refused_size = 0;
        live.erase(it);
    }
    return f(p);
}
int hipMemGetInfo(size_t *avail, size_t *total) {
    static auto *f = own<int(size_t *, size_t *)>("hipMemGetInfo");
    const int e = f(avail, total);
    std::lock_guard<std::mutex> lock(mu);
    if (budget >= 0 && *avail > (size_t)budget) *avail = (size_t)budget;
    if (total_shown) *total = total_shown;
    return e;
}
int hipGetDevice(int *d) {
    static auto *f = own<int(int *)>("hipGetDevice");
    const int e = f(d);
    if (device_shown >= 0 && std::this_thread::get_id() == watched) *d = device_shown;
    return e;
}
int hipSetDevice(int d) {
    static auto *f = own<int(int)>("hipSetDevice");
    if (std::this_thread::get_id() == watched) {
        ++watched_set_device;
        if (device_shown >= 0) {
            device_shown = d;
            return 0;
        }
    }
    return f(d);
}

struct Dim3 {
    unsigned x, y, z;
};
int hipLaunchKernel(const void *fn, Dim3 grid, Dim3 block, void **args, size_t lds, void *stream) {
    static auto *f = own<int(const void *, Dim3, Dim3, void **, size_t, void *)>("hipLaunchKernel");
    if (failing_launch > 0 && --failing_launch == 0) return launch_error = 719;   // hipErrorLaunchFailure
    return f(fn, grid, block, args, lds, stream);
}
int hipGetLastError() {
    static auto *f = own<int()>("hipGetLastError");
    const int e = f(), injected = launch_error;
    launch_error = 0;
    return injected ? injected : e;
}

void limit_fail_launch(int nth) { failing_launch = nth; }
void limit_budget(long long bytes) {
    std::lock_guard<std::mutex> lock(mu);
    budget = bytes;
}
void limit_refuse_size(size_t bytes) {
    std::lock_guard<std::mutex> lock(mu);
    refused_size = bytes;
    until_freed = false;
}
void limit_refuse_until_freed(size_t bytes) {
    std::lock_guard<std::mutex> lock(mu);
    refused_size = bytes;
    until_freed = true;
}
void limit_show_total(size_t bytes) {
    std::lock_guard<std::mutex> lock(mu);
    total_shown = bytes;
}
// the calling thread is watched from here on
void limit_show_device(int d) {
    watched = std::this_thread::get_id();
    watched_set_device = 0;
    device_shown = d;
}
int limit_shown_device() { return device_shown; }
int limit_set_device_calls() { return watched_set_device; }
size_t limit_held() { return held; }
int limit_calls() { return calls; }
int limit_refusals() { return refusals; }
}
