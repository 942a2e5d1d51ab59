// Error state, device-memory accounting and device selection for libedx.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <unordered_map>

#include "common.h"

namespace edx {

static thread_local std::string g_last_error;
static thread_local int g_device = 0;
static thread_local int g_corehole_layout = EDX_COREHOLE_REFERENCE;
thread_local hipStream_t g_launch_stream = 0;

int corehole_layout() { return g_corehole_layout; }

int set_error(int code, const char *fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

int hip_fail(hipError_t e, const char *what, const char *file, int line) {
    return set_error(EDX_ERR_HIP, "%s failed: %s (%s:%d)", what, hipGetErrorString(e), file,
                     line);
}

// Device memory.  A freed block is kept for the next request of its size
// instead of going back to the driver: mapping and clearing a released block
// again costs the next build more than the build itself (CSR of H_i at norb 24,
// 1 GB: 1.6 ms of kernels, 25 ms a call through hipMalloc / hipFree, 2 ms
// reusing the blocks).  A block is only kept once the device has finished all
// work (hipFree waits for the same), so any thread on any stream may have it
// next.  Kept blocks are memory that other users of the device do not get, so
// they are bounded, on each device, by 1/16 of its memory and by a quarter of
// what would be free without them, looked at again for every eighth of that
// freed (64 MB at least; a look costs a build of 1 GB 1 % of its time).  The blocks
// unused longest go first.  All are given back when an allocation here fails and
// by mem_trim, and all but 64 MB when the last library object is freed.
namespace {

struct Live {
    size_t bytes, cap;   // asked for, allocated
    int dev;
};
struct Idle {
    void *p;
    uint64_t freed;      // order of the frees
};
struct DevPool {
    std::multimap<size_t, Idle> idle;   // by allocated size
    size_t idle_bytes = 0;
    size_t unlooked = 0;                // bytes freed since the device's memory was looked at
    size_t limit = 0;                   // bound of idle_bytes found then
};
struct Pool {
    std::mutex mu;
    std::unordered_map<void *, Live> live;
    std::map<int, DevPool> devs;
    int64_t in_use = 0, live_bytes = 0;   // asked for, allocated
    uint64_t frees = 0;
};
Pool &pool() {
    static Pool *p = new Pool;   // never destroyed: objects may be freed at exit
    return *p;
}

constexpr size_t POOL_SMALL = 64ull << 20;   // kept even when nothing is live

size_t pool_cap(size_t bytes) {
    const size_t g = bytes <= (1u << 20) ? 512 : 2u << 20;
    return (bytes + g - 1) / g * g;
}

// Releases a device's idle blocks, oldest first, until at most keep bytes stay (mu held).
void pool_trim(DevPool &d, size_t keep) {
    while (d.idle_bytes > keep && !d.idle.empty()) {
        auto old = d.idle.begin();
        for (auto it = d.idle.begin(); it != d.idle.end(); ++it)
            if (it->second.freed < old->second.freed) old = it;
        (void)hipFree(old->second.p);
        d.idle_bytes -= old->first;
        d.idle.erase(old);
    }
}

void pool_trim_all(Pool &q, size_t keep) {
    for (auto &d : q.devs) pool_trim(d.second, keep);
}

// The bound of the current device's idle bytes (mu held).
size_t pool_limit(DevPool &d, size_t freed) {
    d.unlooked += freed;
    if (!d.limit || d.unlooked >= std::max(POOL_SMALL, d.limit / 8)) {
        size_t fr = 0, tot = 0;
        if (hipMemGetInfo(&fr, &tot) != hipSuccess) {
            (void)hipGetLastError();
            fr = tot = 0;
        }
        d.limit = std::max(std::min(tot / 16, (fr + d.idle_bytes) / 4), (size_t)1);
        d.unlooked = 0;
    }
    return d.limit;
}

}  // namespace

void *dmalloc(size_t bytes, const char *what) {
    if (bytes == 0) bytes = 16;
    const size_t cap = pool_cap(bytes);
    int dev = 0;
    (void)hipGetDevice(&dev);
    Pool &q = pool();
    auto take = [&](void *p, size_t size) {
        q.live[p] = Live{bytes, size, dev};
        q.in_use += (int64_t)bytes;
        q.live_bytes += (int64_t)size;
        return p;
    };
    {
        std::lock_guard<std::mutex> lk(q.mu);
        DevPool &d = q.devs[dev];
        auto it = d.idle.lower_bound(cap);
        if (it != d.idle.end() && it->first <= cap + cap / 8) {
            void *p = take(it->second.p, it->first);
            d.idle_bytes -= it->first;
            d.idle.erase(it);
            return p;
        }
    }
    void *p = nullptr;
    hipError_t e = hipMalloc(&p, cap);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        {
            std::lock_guard<std::mutex> lk(q.mu);
            pool_trim_all(q, 0);
        }
        e = hipMalloc(&p, cap);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        set_error(EDX_ERR_NOMEM, "device allocation of %zu bytes for %s failed: %s", bytes, what,
                  hipGetErrorString(e));
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(q.mu);
    return take(p, cap);
}

void dfree(void *p) {
    if (!p) return;
    Pool &q = pool();
    Live l{0, 0, -1};
    {
        std::lock_guard<std::mutex> lk(q.mu);
        auto it = q.live.find(p);
        if (it != q.live.end()) {
            l = it->second;
            q.in_use -= (int64_t)l.bytes;
            q.live_bytes -= (int64_t)l.cap;
            q.live.erase(it);
        }
    }
    int dev = 0;
    const bool keep = l.dev >= 0 && hipGetDevice(&dev) == hipSuccess && dev == l.dev &&
                      hipDeviceSynchronize() == hipSuccess;
    if (!keep) {
        (void)hipGetLastError();
        (void)hipFree(p);
        return;
    }
    std::lock_guard<std::mutex> lk(q.mu);
    DevPool &d = q.devs[dev];
    d.idle.emplace(l.cap, Idle{p, ++q.frees});
    d.idle_bytes += l.cap;
    pool_trim(d, pool_limit(d, l.cap));
    if (q.in_use == 0) pool_trim_all(q, POOL_SMALL);
}

int64_t mem_in_use() {
    Pool &q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    return q.in_use;
}

void mem_reserved(int64_t *live, int64_t *idle) {
    Pool &q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    *live = q.live_bytes;
    *idle = 0;
    for (auto &d : q.devs) *idle += (int64_t)d.second.idle_bytes;
}

void mem_trim() {
    Pool &q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    pool_trim_all(q, 0);
}

int current_device() { return g_device; }

int num_cus() {
    static int cached = -1;
    if (cached < 0) {
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, g_device) == hipSuccess)
            cached = prop.multiProcessorCount;
        else
            cached = 256;
    }
    return cached;
}

}  // namespace edx

extern "C" {

const char *edx_last_error(void) { return edx::g_last_error.c_str(); }

int edx_set_corehole_layout(int layout, int *previous) {
    EDX_CHECK(layout == EDX_COREHOLE_REFERENCE || layout == EDX_COREHOLE_INTERLEAVED, EDX_ERR_ARG,
              "unknown core-hole layout %d", layout);
    if (previous) *previous = edx::g_corehole_layout;
    edx::g_corehole_layout = layout;
    return EDX_OK;
}

int edx_init(int device) {
    int n = 0;
    EDX_HIP(hipGetDeviceCount(&n));
    EDX_CHECK(device >= 0 && device < n, EDX_ERR_ARG, "device %d out of range (%d devices)",
              device, n);
    EDX_HIP(hipSetDevice(device));
    edx::g_device = device;
    return edx::ensure_binomials();
}

int edx_mem_in_use(int64_t *bytes) {
    EDX_CHECK(bytes, EDX_ERR_ARG, "null output");
    *bytes = edx::mem_in_use();
    return EDX_OK;
}

int edx_mem_reserved(int64_t *live, int64_t *idle) {
    EDX_CHECK(live && idle, EDX_ERR_ARG, "null output");
    edx::mem_reserved(live, idle);
    return EDX_OK;
}

int edx_mem_trim(void) {
    edx::mem_trim();
    return EDX_OK;
}

int edx_set_stream(void *stream) {
    edx::g_launch_stream = (hipStream_t)stream;
    return EDX_OK;
}

}  // extern "C"
