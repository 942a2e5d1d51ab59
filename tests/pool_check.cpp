// Checks of the library's device-memory pool (edrixs_amd/csrc/runtime.cpp) on the host: the
// device is a stand-in of 16 GiB whose allocations are small host blocks.  Exits with the line
// of the first check that fails, modulo 256, or 0.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <random>
#include <thread>
#include <vector>

#include "../edrixs_amd/csrc/common.h"

namespace {
constexpr size_t GB = 1ull << 30, MB = 1ull << 20, TOTAL = 16 * GB;
std::mutex g_mu;
std::map<void *, size_t> g_blocks;
size_t g_used = 0, g_others = 0;   // by the library, by other users of the device
int g_mallocs = 0, g_looks = 0;
thread_local int g_current = 0;
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_used + g_others + n > TOTAL) return hipErrorOutOfMemory;
    *p = malloc(64);
    g_blocks[*p] = n;
    g_used += n;
    ++g_mallocs;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_blocks.find(p);
    if (it == g_blocks.end()) abort();
    g_used -= it->second;
    g_blocks.erase(it);
    free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
    std::lock_guard<std::mutex> lk(g_mu);
    ++g_looks;
    *f = TOTAL - g_used - g_others;
    *t = TOTAL;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = g_current;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    g_current = d;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "out of memory"; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *, int) { return hipErrorUnknown; }
}

namespace edx {
int ensure_binomials() { return 0; }
}  // namespace edx

#define CHECK(c)                                            \
    do {                                                    \
        if (!(c)) {                                         \
            fprintf(stderr, "line %d: %s\n", __LINE__, #c); \
            exit(__LINE__ % 256 ? __LINE__ % 256 : 1);      \
        }                                                   \
    } while (0)

using edx::dfree;
using edx::dmalloc;

int64_t live() {
    int64_t l, i;
    edx::mem_reserved(&l, &i);
    return l;
}
int64_t idle() {
    int64_t l, i;
    edx::mem_reserved(&l, &i);
    return i;
}

int main() {
    void *held = dmalloc(4096, "held");
    CHECK(edx::mem_in_use() == 4096 && live() == 4096 && idle() == 0);

    // a freed block serves the next request of about its size, none far smaller or larger
    void *a = dmalloc(100 * MB, "a");
    dfree(a);
    CHECK(edx::mem_in_use() == 4096 && idle() == (int64_t)(100 * MB));
    const int mallocs = g_mallocs;
    CHECK(dmalloc(50 * MB, "half") != a && dmalloc(101 * MB, "more") != a && g_mallocs == mallocs + 2);
    void *b = dmalloc(95 * MB, "b");
    CHECK(b == a && g_mallocs == mallocs + 2 && idle() == 0);
    CHECK(live() >= (int64_t)(100 * MB) && edx::mem_in_use() == (int64_t)(4096 + 246 * MB));

    // blocks of another device stay there
    g_current = 1;
    dfree(b);   // freed while device 1 is current: given back
    CHECK(idle() == 0);
    void *c = dmalloc(100 * MB, "c");
    dfree(c);
    CHECK(idle() == (int64_t)(100 * MB));
    g_current = 0;
    void *d = dmalloc(100 * MB, "d");
    CHECK(d != c && idle() == (int64_t)(100 * MB));
    edx::mem_trim();
    CHECK(idle() == 0 && g_used == (size_t)live());

    // bounded by 1/16 of the device, oldest first
    std::vector<void *> v;
    for (int i = 0; i < 40; ++i) v.push_back(dmalloc(64 * MB + i * 2 * MB, "v"));
    for (void *p : v) dfree(p);
    CHECK(idle() <= (int64_t)(TOTAL / 16) && idle() > (int64_t)(TOTAL / 32));
    CHECK(g_blocks.count(v.back()) == 1 && g_blocks.count(v.front()) == 0);

    // and by a quarter of what would be free: others have taken nearly all of it
    g_others = TOTAL - g_used - 200 * MB;
    const size_t open = 200 * MB + idle();
    v.clear();
    for (int i = 0; i < 130; ++i) v.push_back(dmalloc(MB, "small"));
    for (void *p : v) dfree(p);
    CHECK(idle() <= (int64_t)(open / 4) && idle() > 0);
    CHECK(g_looks < 50);   // not for every small block

    // what is kept gives way to an allocation that would fail
    edx::mem_trim();
    g_others = 0;
    a = dmalloc(900 * MB, "a");
    dfree(a);
    CHECK(idle() == (int64_t)(900 * MB));
    g_others = TOTAL - g_used - 100 * MB;
    b = dmalloc(980 * MB, "b");
    CHECK(b && idle() == 0);
    CHECK(!dmalloc(2 * GB, "too much"));
    CHECK(strstr(edx_last_error(), "too much"));
    dfree(b);
    g_others = 0;

    // the last object freed leaves 64 MB at the most
    std::vector<void *> rest;
    for (auto &q : g_blocks) rest.push_back(q.first);
    edx::mem_trim();
    for (void *p : rest)
        if (g_blocks.count(p)) dfree(p);
    CHECK(edx::mem_in_use() == 0 && live() == 0 && idle() <= (int64_t)(64 * MB) && g_used == (size_t)idle());

    // threads: no block is anyone else's while it is held
    std::atomic<int> wrong{0};
    std::vector<std::thread> th;
    for (int t = 0; t < 8; ++t)
        th.emplace_back([t, &wrong] {
            std::mt19937 r(t);
            std::vector<std::pair<int *, int>> mine;
            for (int i = 0; i < 3000; ++i) {
                if (mine.size() < 6 && r() % 2) {
                    int *p = (int *)dmalloc((r() % 40 + 1) * 512, "thread");
                    const int tag = t * 10000 + i;
                    *p = tag;
                    mine.push_back({p, tag});
                } else if (!mine.empty()) {
                    const size_t k = r() % mine.size();
                    if (*mine[k].first != mine[k].second) ++wrong;
                    dfree(mine[k].first);
                    mine.erase(mine.begin() + k);
                }
                if (i % 500 == 0) edx::mem_trim();
            }
            for (auto &q : mine) dfree(q.first);
        });
    for (auto &t : th) t.join();
    CHECK(wrong == 0 && edx::mem_in_use() == 0 && g_used == (size_t)(live() + idle()));
    puts("pool ok");
    return 0;
}
