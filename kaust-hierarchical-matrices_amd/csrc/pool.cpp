// Device memory kept between the library's allocations.  A build makes some
// 150 allocations and frees most of them again; every hipFree waits for the
// device, and a hipMalloc of memory freed a moment ago waits for the driver
// to clear it (10-15 ms of the 2D TLR build at N = 16384, up to 0.5 s of the
// 3D build at N = 65536).  Blocks the library frees are therefore kept for
// its next allocations of about their size:
//
//   * bounded: at most 1/16 of the device's memory is held (18 GB of 288; the
//     3D build at N = 65536 leaves 12 GB, and takes 70 ms, with 1/64 75, with
//     1/256 77, with nothing held 80; the TLR build 21, 21, 31 and 32 ms), and
//     at most 1/8 of what is free on it (asked once per 1/1024 of the device
//     that comes back: 4.7 us), so that on a full card little is kept from
//     other allocators; the blocks held longest go back to the driver first,
//     and blocks above the bound are never held;
//   * given back: when the device has no memory left for an allocation of
//     the library, when the caller asks (hmx_memory_release), and when the
//     last context is destroyed;
//   * as safe as hipFree with several streams and threads: a freed block is
//     handed out again only after a wait for the device that followed its
//     release, so no kernel or copy of any stream still uses it (hipFree made
//     the same wait, for every block); one lock guards the lists;
//   * with stream captures as hipMalloc and hipFree: allocating inside a
//     capture is refused where hipMalloc is, and neither disturbs a capture of
//     another thread;
//   * per device: a block returns to the device that it came from.
#include <algorithm>
#include <cstdint>
#include <list>
#include <mutex>
#include <unordered_map>

#include "hmx_internal.h"

namespace hmx {
namespace {

struct Held {
    void* p;
    size_t bytes;
    uint64_t seq;  // release number
};

struct Pool {
    std::list<Held> held;  // in the order of release
    size_t bytes = 0;      // sum over held
    size_t bound = 0;      // most bytes held (0: not asked yet)
    size_t limit = 0;      // the same by the device's free memory, when last asked
    size_t back = 0;       // bytes released since then
    uint64_t synced = 0;   // blocks released before this number may be handed out
};

struct Place {
    int device;
    size_t bytes;
};

constexpr int kDevices = 64;
std::mutex g_mu;
struct State {
    Pool pool[kDevices];
    std::unordered_map<void*, Place> places;
};
// never destroyed: handles and contexts may go while the process ends
State& state() {
    static auto* s = new State();
    return *s;
}
Pool& pool(int device) { return state().pool[device]; }
std::unordered_map<void*, Place>& places() { return state().places; }
uint64_t g_seq = 1;
int g_contexts = 0;

// Sizes are rounded up to 1/8 of their power of two, so that blocks of about
// one size (factors of two clouds of the same kind) serve each other.
size_t rounded(size_t n) {
    if (n <= 4096) return 4096;
    size_t p = 4096;
    while (p < n) p <<= 1;
    const size_t q = p / 16;
    return (n + q - 1) / q * q;
}

// takes out the smallest held block of bytes or up to a quarter more (exact
// sizes only, or up to twice: the builds take the same time; a quarter wastes
// less of a long-lived object's memory than twice)
void* take(Pool& P, size_t bytes, bool syncedOnly) {
    auto best = P.held.end();
    for (auto it = P.held.begin(); it != P.held.end(); ++it)
        if (it->bytes >= bytes && it->bytes <= bytes + bytes / 4 && (!syncedOnly || it->seq < P.synced) &&
            (best == P.held.end() || it->bytes < best->bytes))
            best = it;
    if (best == P.held.end()) return nullptr;
    if (!syncedOnly) return best->p;  // only looked up
    void* p = best->p;
    P.bytes -= best->bytes;
    P.held.erase(best);
    return p;
}

void flush(Pool& P) {  // hipFree waits for the device
    for (const Held& h : P.held) {
        (void)hipFree(h.p);
        places().erase(h.p);
    }
    P.held.clear();
    P.bytes = 0;
}

// Waits for all work of the device, as every hipFree does (1.4 us when idle).
// hipDeviceSynchronize would wait too, but ends every capture that any thread
// of the process has open.
hipError_t wait_device() {
    void* t = nullptr;
    const hipError_t e = hipMalloc(&t, 4096);
    return e == hipSuccess ? hipFree(t) : e;
}

}  // namespace

void* pool_alloc(size_t bytes) {
    // hipMalloc's rule under capture, for a held block too: a graph would keep
    // its address beyond the block's life (0.2 us)
    HMX_HIP(hipFree(nullptr));
    int dev = 0;
    HMX_HIP(hipGetDevice(&dev));
    HMX_CHECK(dev >= 0 && dev < kDevices, HMX_EUNSUPPORTED, "device index beyond the pool table");
    Pool& P = pool(dev);
    size_t want = rounded(bytes);
    {
        std::unique_lock<std::mutex> lk(g_mu);
        if (P.bound == 0) {
            size_t fr = 0, tot = 0;
            HMX_HIP(hipMemGetInfo(&fr, &tot));
            P.bound = P.limit = tot / 16;
        }
        if (want > P.bound / 4) want = bytes;  // large blocks: no memory given away to rounding
        if (void* p = take(P, want, true)) return p;
        if (take(P, want, false)) {
            const uint64_t upto = g_seq;
            lk.unlock();
            const hipError_t w = wait_device();
            if (w != hipErrorOutOfMemory) HMX_HIP(w);
            else (void)hipGetLastError();  // not a page left: the flush below waits
            lk.lock();
            if (w == hipSuccess && P.synced < upto) P.synced = upto;
            if (void* p = take(P, want, true)) return p;  // else another thread took it
        }
    }
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, want);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        {
            std::lock_guard<std::mutex> lk(g_mu);
            flush(P);
        }
        want = bytes;
        e = hipMalloc(&p, want);
    }
    HMX_HIP(e);
    std::lock_guard<std::mutex> lk(g_mu);
    places()[p] = Place{dev, want};
    return p;
}

void pool_free(void* p) {
    std::unique_lock<std::mutex> lk(g_mu);
    auto it = places().find(p);
    if (it == places().end()) return;
    const Place at = it->second;
    Pool& P = pool(at.device);
    if (g_contexts == 0 || at.bytes > P.bound) {
        places().erase(it);
        lk.unlock();
        (void)hipFree(p);
        return;
    }
    P.held.push_back(Held{p, at.bytes, g_seq++});
    P.bytes += at.bytes;
    P.back += at.bytes;
    int dev = -1;
    if (P.back >= P.bound / 64 && hipGetDevice(&dev) == hipSuccess && dev == at.device) {
        size_t fr = 0, tot = 0;
        P.back = 0;
        P.limit = hipMemGetInfo(&fr, &tot) == hipSuccess ? std::min(P.bound, fr / 8) : P.bound;
    }
    std::list<Held> out;  // the blocks held longest, until the bound holds
    while (P.bytes > P.limit) {
        P.bytes -= P.held.front().bytes;
        places().erase(P.held.front().p);
        out.splice(out.end(), P.held, P.held.begin());
    }
    lk.unlock();
    for (const Held& h : out) (void)hipFree(h.p);
}

void pool_release() {
    int dev = 0;
    HMX_HIP(hipGetDevice(&dev));
    HMX_HIP(hipFree(nullptr));  // not inside a capture
    std::lock_guard<std::mutex> lk(g_mu);
    if (dev >= 0 && dev < kDevices) flush(pool(dev));
}

size_t pool_held_bytes() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kDevices) return 0;
    std::lock_guard<std::mutex> lk(g_mu);
    return pool(dev).bytes;
}

void pool_context_created() {
    std::lock_guard<std::mutex> lk(g_mu);
    ++g_contexts;
}

void pool_context_destroyed() {
    std::lock_guard<std::mutex> lk(g_mu);
    if (--g_contexts > 0) return;
    for (Pool& P : state().pool) flush(P);
}

}  // namespace hmx
