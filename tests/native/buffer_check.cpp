// Host check of the library's workspace growth (csrc/hmx_internal.h) with the
// device allocator replaced by malloc: a failed growth leaves the buffer empty
// and recorded as empty, so the next request, however small, allocates.
#include <cstdio>
#include <cstdlib>

#include "../../kaust-hierarchical-matrices_amd/csrc/hmx_internal.h"

namespace hmx {
std::atomic<int64_t> g_allocCount{0}, g_allocFailAt{-1}, g_liveBytes{0};
void* pool_alloc(size_t bytes) { return std::malloc(bytes); }
void pool_free(void* p) { std::free(p); }
}  // namespace hmx

#define REQUIRE(c)                                                  \
    do {                                                            \
        if (!(c)) {                                                 \
            std::printf("failed at line %d: %s\n", __LINE__, #c);   \
            return 1;                                               \
        }                                                           \
    } while (0)

int main() {
    using namespace hmx;
    DBuf<double> b;
    REQUIRE(grow(b, 16) && b.n == 16 && b.p);
    REQUIRE(!grow(b, 16) && !grow(b, 3));
    g_allocFailAt = g_allocCount.load();
    bool failed = false;
    try {
        grow(b, 64);
    } catch (const Error& e) {
        failed = e.status == HMX_ENOMEM;
    }
    REQUIRE(failed && b.p == nullptr && b.n == 0 && g_liveBytes == 0);
    g_allocFailAt = -1;
    REQUIRE(grow(b, 16) && b.n == 16 && b.p);
    REQUIRE(g_liveBytes == 16 * 8);
    b.release();
    REQUIRE(g_liveBytes == 0);
    std::printf("buffer check ok\n");
    return 0;
}
