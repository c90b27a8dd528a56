// small.hpp — dense symmetric eigenproblems that fit one workgroup's LDS.
#pragma once

#include "common.hpp"

namespace cuev {

constexpr int kSmallMaxN = 128;

// batch matrices of order n <= kSmallMaxN (column-major, contiguous, lower triangle read). With V: all n eigenvalues, ascending, to W (batch x n) and
// the eigenvectors to V; with V == nullptr: eigenvalues il..iu to W (batch x (iu - il + 1)).
// Blocking. *n_failed: matrices whose QL iteration did not converge; *n_not_finite: matrices
// with a NaN or infinite entry (their outputs are NaN). n_need_ql: nullptr, or the matrices
// with eigenvalues too close for the fast path are left unsolved and counted there, unless their
// scale is too large or too small for the staged pipeline (kStagedExp in small.hip).
template <typename T>
int small_eig(hipStream_t s, const T *A, int n, int batch, T *W, T *V, int il, int iu, int *n_failed,
              int *n_not_finite, int *n_need_ql = nullptr);

// Diagonal blocks of a tridiagonal matrix, of order <= kSmallTridiMaxN each (device array, max_sz the
// largest): block [off, off + sz) of the diagonal d, with couplings e[off .. off + sz - 2]. Eigenvalues,
// ascending, to W[off ..], eigenvectors to the diagonal blocks of V (ld ldv; the rest of V is not
// touched). Not blocking. Eigenvalues are NaN where the QL iteration did not converge.
constexpr int kSmallTridiMaxN = 64;
struct SmallLeaf {
    int off, sz;
};
template <typename T>
int small_tridi(hipStream_t s, const T *d, const T *e, const SmallLeaf *leaves, int nleaves, int max_sz, T *W, T *V,
                i64 ldv);

// frees the failure counters kept between calls, where no call is using them
void small_release_all();

} // namespace cuev
