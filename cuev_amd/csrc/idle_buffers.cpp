// idle_buffers.cpp — device buffers kept between blocking calls.
#include "idle_buffers.hpp"

#include <vector>

namespace cuev {
namespace {
// every IdleBuffers (objects of static storage, created while the library is loaded)
std::vector<IdleBuffers *> &pools() {
    static std::vector<IdleBuffers *> p;
    return p;
}
} // namespace

IdleBuffers::IdleBuffers() { pools().push_back(this); }

int IdleBuffers::take(Buffer &b, size_t bytes) {
    int dev = 0;
    CUEV_HIP(hipGetDevice(&dev));
    {
        std::lock_guard<std::mutex> lk(mu_);
        Buffer &slot = idle_[dev & 63];
        if (slot.p && slot.device == dev && slot.bytes >= bytes) {
            b = slot;
            slot = Buffer{};
            return CUEV_STATUS_SUCCESS;
        }
    }
    release(dev);
    b.device = dev;
    b.bytes = bytes;
    if (device_alloc(&b.p, bytes) != hipSuccess)
        CUEV_FAIL(CUEV_STATUS_ALLOC_FAILED, "device allocation of %zu bytes failed", bytes);
    return CUEV_STATUS_SUCCESS;
}

void IdleBuffers::give(Buffer &b) {
    Buffer victim;
    {
        std::lock_guard<std::mutex> lk(mu_);
        Buffer &slot = idle_[b.device & 63];
        if (slot.p && slot.bytes >= b.bytes) {
            victim = b;
        } else {
            victim = slot;
            slot = b;
        }
    }
    b = Buffer{};
    if (victim.p) (void)hipFree(victim.p);
}

void IdleBuffers::release(int device) {
    Buffer victim;
    {
        std::lock_guard<std::mutex> lk(mu_);
        Buffer &slot = idle_[device & 63];
        if (slot.device == device) {
            victim = slot;
            slot = Buffer{};
        }
    }
    if (victim.p) (void)hipFree(victim.p);
}

void IdleBuffers::release_all() {
    Buffer victims[64];
    {
        std::lock_guard<std::mutex> lk(mu_);
        for (int i = 0; i < 64; ++i) {
            victims[i] = idle_[i];
            idle_[i] = Buffer{};
        }
    }
    int cur = 0;
    (void)hipGetDevice(&cur);
    for (Buffer &v : victims)
        if (v.p) {
            (void)hipSetDevice(v.device);
            (void)hipDeviceSynchronize();
            (void)hipFree(v.p);
        }
    (void)hipSetDevice(cur);
}

hipError_t device_alloc(void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) return e;
    (void)hipGetLastError();
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess) {
        for (IdleBuffers *pool : pools()) pool->release(dev);
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
    }
    return e;
}

} // namespace cuev
