/* Drives cudec_amd/csrc/host_copy.h on the CPU: TEST INFRASTRUCTURE ONLY. */
#include "host_copy.h"

#include <cstdint>
#include <cstdlib>
#include <new>

namespace {
std::atomic<bool> g_refuse{false};
std::atomic<uint64_t> g_refused{0};
}  // namespace

void* operator new(std::size_t n) {
    if (g_refuse.load()) {
        g_refused++;
        throw std::bad_alloc();
    }
    void* p = std::malloc(n == 0 ? 1 : n);
    if (p == nullptr) {
        throw std::bad_alloc();
    }
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

extern "C" {

/* `rounds` rounds of each() over n items by a crew for `bytes` bytes, with
 * every allocation refused meanwhile. hits[i] counts the calls for item i.
 * Returns the allocations refused, or -1 when a round threw. */
int64_t host_copy_rounds(uint64_t bytes, uint64_t n, uint64_t rounds, uint32_t* hits) {
    cudec_amd::CopyCrew crew(bytes, n);
    g_refused = 0;
    g_refuse = true;
    bool threw = false;
    try {
        for (uint64_t r = 0; r < rounds; r++) {
            /* as many captures as the streaming call's copies have */
            const uint64_t a = r, b = n, c = bytes;
            crew.each(n, [&, hits](size_t i) {
                __atomic_fetch_add(&hits[i], a + b + c == r + n + bytes ? 1u : 0u,
                                   __ATOMIC_RELAXED);
            });
        }
    } catch (...) {
        threw = true;
    }
    g_refuse = false;
    return threw ? -1 : (int64_t)g_refused.load();
}

/* One round over n items of `bytes` bytes; owner[i] tells the threads apart. */
void host_copy_owners(uint64_t bytes, uint64_t n, uint64_t* owner) {
    cudec_amd::CopyCrew crew(bytes, n);
    crew.each(n, [&](size_t i) {
        static thread_local char here;
        owner[i] = (uint64_t)(uintptr_t)&here;
    });
}

}  // extern "C"
