// small.hpp — dense symmetric eigenproblems that fit one workgroup's LDS.
#pragma once

#include "common.hpp"

namespace cuev {

constexpr int kSmallMaxN = 128;

// batch matrices of order n <= kSmallMaxN (column-major, contiguous, lower triangle read). With V: all n eigenvalues, ascending, to W (batch x n) and
// the eigenvectors to V; with V == nullptr: eigenvalues il..iu to W (batch x (iu - il + 1)).
// Blocking. *n_failed: matrices whose QL iteration did not converge; *n_not_finite: matrices
// with a NaN or infinite entry (their outputs are NaN). n_need_ql: nullptr, or the matrices
// with eigenvalues too close for the fast path are left unsolved and counted there.
template <typename T>
int small_eig(hipStream_t s, const T *A, int n, int batch, T *W, T *V, int il, int iu, int *n_failed,
              int *n_not_finite, int *n_need_ql = nullptr);

// frees the failure counters kept between calls, where no call is using them
void small_release_all();

} // namespace cuev
