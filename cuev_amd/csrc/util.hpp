// util.hpp — small element-wise kernels and error bookkeeping.
#pragma once

#include "common.hpp"

namespace cuev {

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

// A solve's hold on the CUs of the current device for its band reduction and chase (residency.hpp).
// give() once they have finished on the GPU; left to the destructor (an error on the way), the
// stream is waited for first. A thread holds at most one.
class CuClaim {
  public:
    CuClaim() = default;
    CuClaim(const CuClaim &) = delete;
    CuClaim &operator=(const CuClaim &) = delete;
    ~CuClaim();
    int take(hipStream_t s, i64 n, int b);
    void give();

  private:
    int dev_ = -1, shares_ = 0;
    hipStream_t s_ = nullptr;
};

} // namespace cuev
