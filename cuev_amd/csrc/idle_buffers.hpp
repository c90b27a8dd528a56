// idle_buffers.hpp — device buffers kept between blocking calls (host code only).
#pragma once

#include <mutex>

#include "common.hpp"

namespace cuev {

// One idle device buffer per GPU, kept between blocking calls: take() hands it out if it is
// large enough and free, else allocates (a smaller idle one is freed first); give() (after the call's
// work has finished) keeps the larger of the two. Calls that overlap each have a buffer of their own.
class IdleBuffers {
  public:
    struct Buffer {
        void *p = nullptr;
        size_t bytes = 0;
        int device = -1;
    };
    IdleBuffers();
    int take(Buffer &b, size_t bytes); // on the current device
    void give(Buffer &b);
    void release_all();
    void release(int device); // the idle buffer of one device

  private:
    std::mutex mu_;
    Buffer idle_[64];
};

// hipMalloc on the current device; where that fails, once more without the idle buffers of every
// IdleBuffers on it. *p is nullptr and no error stays pending on failure.
hipError_t device_alloc(void **p, size_t bytes);

} // namespace cuev
