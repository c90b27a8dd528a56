// sturm.hpp — Sturm counts by the three-term recurrence, shared by the tridiagonal
// eigenvalue kernel (tridi_values.hip, where the method is described) and the small
// dense solver (small.hip).
#pragma once

#include "common.hpp"

#if defined(__HIPCC__)
namespace cuev {

// Sign changes of p over `rows` rows (a multiple of 8) of (d_i, e_{i-1}^2): pp = p_{i-2},
// p = p_{i-1} on entry and exit. The next 8 rows are read from LDS while 8 are computed
// (de holds 8 rows more than `rows`). p and pp are rescaled every 8 rows.
__device__ __forceinline__ int sturm_rows(const double2 *de, int rows, double x, double &pp, double &p) {
    int cnt = 0;
    double2 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = de[u];
    for (int i = 0; i < rows; i += 8) {
        double2 nx[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) nx[u] = de[i + 8 + u];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const double q = fma(v[u].x - x, p, -(v[u].y * pp));
            cnt += (int)((unsigned)(__double2hiint(q) ^ __double2hiint(p)) >> 31);
            pp = p;
            p = q;
        }
        const int ex = __builtin_amdgcn_frexp_exp(fmax(fabs(pp), fabs(p)));
        pp = ldexp(pp, -ex);
        p = ldexp(p, -ex);
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = nx[u];
    }
    return cnt;
}

} // namespace cuev
#endif
