// Host check of the library's held device memory (csrc/pool.cpp) over a
// stand-in HIP runtime: a device of 1 GiB whose memory is host memory.
//   pool_check hold      bound, order of giving back, out of memory, last context
//   pool_check share     a full device: little is held, and given back when asked
//   pool_check wait      a block is handed out again only after a device wait
//   pool_check capture   allocation is refused where hipMalloc is
//   pool_check exit      a handle and its context that go after the library's statics
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "../../kaust-hierarchical-matrices_amd/csrc/hmx_internal.h"

namespace hmx {
std::atomic<int64_t> g_allocCount{0}, g_allocFailAt{-1}, g_liveBytes{0};
}

static constexpr size_t kTotal = size_t(1) << 30;
static std::map<void*, size_t>& blocks() {
    static auto* m = new std::map<void*, size_t>();
    return *m;
}
static size_t g_used = 0;
static int g_mallocs = 0, g_waits = 0;
static bool g_capturing = false;
static std::vector<void*>& freed() {
    static auto* v = new std::vector<void*>();
    return *v;
}

extern "C" {
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* fr, size_t* tot) {
    *fr = kTotal - g_used;
    *tot = kTotal;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
    if (g_capturing) return hipErrorStreamCaptureUnsupported;
    if (g_used + n > kTotal) return hipErrorOutOfMemory;
    *p = std::malloc(1);
    blocks()[*p] = n;
    g_used += n;
    ++g_mallocs;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (g_capturing) return hipErrorStreamCaptureUnsupported;
    if (!p) return hipSuccess;
    g_used -= blocks().at(p);
    blocks().erase(p);
    std::free(p);
    freed().push_back(p);
    ++g_waits;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
    if (g_capturing) return hipErrorStreamCaptureUnsupported;
    ++g_waits;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
}

#define REQUIRE(c)                                                \
    do {                                                          \
        if (!(c)) {                                               \
            std::printf("failed at line %d: %s\n", __LINE__, #c); \
            std::exit(1);                                         \
        }                                                         \
    } while (0)

using namespace hmx;
static constexpr size_t MB = size_t(1) << 20;

static void hold() {
    pool_context_created();
    pool_context_created();
    // 16 blocks of 8 MiB: the 64 MiB bound (1/16 of the device) keeps the last 8
    std::vector<void*> p;
    for (int i = 0; i < 16; ++i) p.push_back(pool_alloc(8 * MB));
    freed().clear();
    for (void* q : p) {
        pool_free(q);
        REQUIRE(pool_held_bytes() <= kTotal / 16);
    }
    REQUIRE(pool_held_bytes() == 64 * MB);
    REQUIRE(freed().size() == 8);
    for (int i = 0; i < 8; ++i) REQUIRE(freed()[i] == p[i]);  // the ones held longest
    // a block above the bound is not held
    void* big = pool_alloc(100 * MB);
    pool_free(big);
    REQUIRE(pool_held_bytes() == 64 * MB && freed().back() == big);
    // device full: what is held goes back and the allocation succeeds
    void* rest = pool_alloc(kTotal - 32 * MB);
    REQUIRE(rest && pool_held_bytes() == 0);
    bool refused = false;
    try {
        pool_alloc(64 * MB);
    } catch (const Error& e) {
        refused = e.status == HMX_ENOMEM;
    }
    REQUIRE(refused);
    pool_free(rest);
    pool_free(pool_alloc(8 * MB));
    REQUIRE(pool_held_bytes() == 8 * MB);
    // the last context gives all back; after it nothing is held
    pool_context_destroyed();
    REQUIRE(pool_held_bytes() == 8 * MB);
    void* late = pool_alloc(4 * MB);
    pool_context_destroyed();
    REQUIRE(pool_held_bytes() == 0);
    pool_free(late);
    REQUIRE(pool_held_bytes() == 0 && g_used == 0);
}

static void share() {
    pool_context_created();
    // somebody else's memory: 104 MiB of the device are left
    g_used += kTotal - 104 * MB;
    std::vector<void*> p;
    for (int i = 0; i < 10; ++i) p.push_back(pool_alloc(4 * MB));
    for (void* q : p) {
        pool_free(q);
        REQUIRE(pool_held_bytes() <= (kTotal - g_used) / 8);
    }
    REQUIRE(pool_held_bytes() > 0 && pool_held_bytes() <= 13 * MB);
    pool_release();
    REQUIRE(pool_held_bytes() == 0 && g_used == kTotal - 104 * MB);
    // in a capture nothing is given back, and nothing is lost
    pool_free(pool_alloc(4 * MB));
    g_capturing = true;
    bool refused = false;
    try {
        pool_release();
    } catch (const Error&) {
        refused = true;
    }
    g_capturing = false;
    REQUIRE(refused && pool_held_bytes() == 4 * MB);
    pool_context_destroyed();
    REQUIRE(g_used == kTotal - 104 * MB);
}

static void wait() {
    pool_context_created();
    void* a = pool_alloc(2 * MB);
    pool_free(a);
    int w = g_waits;
    void* b = pool_alloc(2 * MB);
    REQUIRE(b == a && g_waits == w + 1);  // the same block, after one wait
    void* c = pool_alloc(3 * MB);
    void* d = pool_alloc(5 * MB);
    pool_free(b);
    pool_free(c);
    pool_free(d);
    w = g_waits;
    REQUIRE(pool_alloc(5 * MB) == d && pool_alloc(3 * MB) == c && pool_alloc(2 * MB) == b);
    REQUIRE(g_waits == w + 1);  // one wait serves all blocks released before it
    // not for a much smaller request, nor for a larger one
    pool_free(d);
    void* e = pool_alloc(3 * MB);
    void* f = pool_alloc(6 * MB);
    REQUIRE(e != d && f != d);
    for (void* q : {b, c, e, f}) pool_free(q);
    pool_context_destroyed();
    REQUIRE(g_used == 0);
}

static void capture() {
    pool_context_created();
    void* a = pool_alloc(2 * MB);
    pool_free(a);
    void* b = pool_alloc(2 * MB);  // waited for: the next one needs no wait
    pool_free(pool_alloc(4 * MB));
    pool_free(b);
    void* c = pool_alloc(4 * MB);
    pool_free(c);
    g_capturing = true;
    for (size_t n : {2 * MB, 4 * MB, 32 * MB}) {
        bool refused = false;
        try {
            pool_alloc(n);
        } catch (const Error& e) {
            refused = e.status == HMX_EDEVICE;
        }
        REQUIRE(refused);
    }
    g_capturing = false;
    pool_context_destroyed();
    REQUIRE(g_used == 0);
}

// constructed before the library's statics, so destroyed after them
struct LateHandle {
    void* p = nullptr;
    ~LateHandle() {
        if (!p) return;
        pool_free(p);
        pool_context_destroyed();  // and its context: everything held goes back
        if (g_used != 0) std::_Exit(3);
    }
};
static LateHandle g_late __attribute__((init_priority(101)));

int main(int argc, char** argv) {
    const char* what = argc > 1 ? argv[1] : "";
    if (!std::strcmp(what, "hold")) hold();
    else if (!std::strcmp(what, "share")) share();
    else if (!std::strcmp(what, "wait")) wait();
    else if (!std::strcmp(what, "capture")) capture();
    else if (!std::strcmp(what, "exit")) {
        pool_context_created();
        g_late.p = pool_alloc(2 * MB);
        pool_free(pool_alloc(2 * MB));  // held while the process ends
    } else return 2;
    std::printf("pool check %s ok\n", what);
    return 0;
}
