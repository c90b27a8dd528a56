// util.hpp — small element-wise kernels and error bookkeeping.
#pragma once

#include <mutex>

#include "common.hpp"

namespace cuev {

// One idle device buffer per GPU, kept between blocking calls: take() hands it out if it is
// large enough and free, else allocates; give() (after the call's work has finished) keeps the
// larger of the two. Calls that overlap each have a buffer of their own.
class IdleBuffers {
  public:
    struct Buffer {
        void *p = nullptr;
        size_t bytes = 0;
        int device = -1;
    };
    int take(Buffer &b, size_t bytes); // on the current device
    void give(Buffer &b);
    void release_all();

  private:
    std::mutex mu_;
    Buffer idle_[64];
};

namespace detail {
const char *last_error();
void clear_error();
} // namespace detail

// A[i,j] = (i == j) ? diag : v for the m x n block at A (ld lda).
template <typename T> int fill2d(hipStream_t s, T *A, i64 lda, i64 m, i64 n, T v, T diag);
// D[0:m, 0:n] = S[0:m, 0:n]
template <typename T> int copy2d(hipStream_t s, const T *S, i64 lds, T *D, i64 ldd, i64 m, i64 n);
// dst = (D) src, element-wise over an m x n block
template <typename S, typename D>
int convert2d(hipStream_t s, const S *src, i64 lds, D *dst, i64 ldd, i64 m, i64 n);
// p[0:n] = v
int fill_int(hipStream_t s, int *p, i64 n, int v);

// Solves whose band reduction and chase need more than a quarter of the CUs take turns on the GPU for
// these two stages. Their kernels wait for workgroups of their own to become resident, one per CU:
// four of up to a quarter each (as many as a process has hardware queues by default) always
// fit at once, of larger ones each could get a part of the CUs and none all it waits for. begin() makes
// the stream wait for the turn before (one event per device), end() ends the turn; other threads queue
// their work once this one's is queued.
class PersistentTurn {
  public:
    int begin(hipStream_t s, int n, int b);
    int end();

  private:
    std::unique_lock<std::mutex> lock_;
    int dev_ = -1;
    hipStream_t s_ = nullptr;
};

} // namespace cuev
