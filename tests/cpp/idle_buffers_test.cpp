// The device buffers kept between calls (cuev_amd/csrc/idle_buffers.cpp) against a stand-in for the HIP
// allocator that counts bytes: no call holds more than it did with a buffer of its own per call.
#include <cstdarg>
#include <cstdio>
#include <map>

#include "../../cuev_amd/csrc/idle_buffers.hpp"

static size_t g_capacity = 0, g_used = 0, g_peak = 0;
static std::map<void *, size_t> g_live;
static hipError_t g_last = hipSuccess;
static char g_heap[1 << 20];
static size_t g_next = 0;

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    if (g_used + n > g_capacity) {
        *p = nullptr;
        return g_last = hipErrorOutOfMemory;
    }
    g_used += n;
    if (g_used > g_peak) g_peak = g_used;
    *p = g_heap + g_next++;
    g_live[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!g_live.count(p)) return hipErrorInvalidValue;
    g_used -= g_live[p];
    g_live.erase(p);
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = g_last; g_last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t) { return ""; }
}
namespace cuev {
namespace detail {
void set_error(const char *, ...) {}
} // namespace detail
} // namespace cuev

using namespace cuev;

#define CHECK(c)                                        \
    do {                                                \
        if (!(c)) {                                     \
            std::printf("line %d: %s\n", __LINE__, #c); \
            return 1;                                   \
        }                                               \
    } while (0)

static IdleBuffers g_a, g_b;

int main() {
    IdleBuffers::Buffer x, y;
    g_capacity = 100;
    // kept, and handed out again
    CHECK(g_a.take(x, 60) == CUEV_STATUS_SUCCESS && g_used == 60);
    void *first = x.p;
    g_a.give(x);
    CHECK(g_used == 60 && g_a.take(x, 50) == CUEV_STATUS_SUCCESS && x.p == first && x.bytes == 60);
    g_a.give(x);
    // a larger one: the smaller is freed first
    CHECK(g_a.take(x, 80) == CUEV_STATUS_SUCCESS && g_used == 80 && g_peak == 80);
    g_a.give(x);
    // calls that overlap: the larger stays
    g_capacity = 200;
    CHECK(g_a.take(x, 80) == CUEV_STATUS_SUCCESS && g_a.take(y, 90) == CUEV_STATUS_SUCCESS && g_used == 170);
    g_a.give(y);
    g_a.give(x);
    CHECK(g_used == 90);
    // another user's allocation comes before idle buffers
    g_capacity = 100;
    void *p = nullptr;
    CHECK(device_alloc(&p, 70) == hipSuccess && g_used == 70);
    CHECK(g_b.take(y, 40) == CUEV_STATUS_ALLOC_FAILED && g_last == hipSuccess && y.p == nullptr && g_used == 70);
    CHECK(g_b.take(y, 30) == CUEV_STATUS_SUCCESS && g_used == 100);
    void *q = nullptr;
    CHECK(device_alloc(&q, 30) == hipErrorOutOfMemory && q == nullptr && g_last == hipSuccess); // in use, not idle
    g_b.give(y);
    CHECK(device_alloc(&q, 30) == hipSuccess && g_used == 100);
    CHECK(hipFree(p) == hipSuccess && hipFree(q) == hipSuccess);
    CHECK(g_a.take(x, 10) == CUEV_STATUS_SUCCESS);
    g_a.give(x);
    g_a.release_all();
    g_b.release_all();
    CHECK(g_used == 0 && g_live.empty());
    std::puts("idle buffers ok");
    return 0;
}
