// tridi_values.hip — eigenvalues of a symmetric tridiagonal matrix on the GPU by
// Sturm-sequence multisection (no reference counterpart: the reference always
// computes every eigenpair with its D&C, src/cuda/tridi.cu:12-13).
//
// The number of eigenvalues of T = tridiag(e, d, e) below x is the number of sign changes
// in the sequence p_{-1} = 1, p_0 = d_0 - x,
//   p_i = (d_i - x) p_{i-1} - e_{i-1}^2 p_{i-2}
// (Givens 1954; Wilkinson: the computed signs are exact for a matrix with off-diagonals
// and differences d_i - x within a few roundings of T's). Its chain is one FMA per row,
// where the pivots q_i = (d_i - x) - e_{i-1}^2 / q_{i-1} of the LDL^T form take a division
// per row. Two safeguards replace that form's smallest pivot:
//   * e_{i-1}^2 is raised to 2^-120 ||T||^2 (the off-diagonal moves by at most 2^-60 ||T||, far
//     below the stopping width), so a zero p_i never makes the following ones zero: its
//     sign does not matter, p_{i-1} and p_{i+1} differ in sign;
//   * T is scaled by a power of two to ||T|| < 1 and p_{i-1}, p_i are rescaled every 8 rows
//     by the larger one's exponent, so 8 rows grow by at most 2^16 and shrink by at
//     most 2^-500.
// Eigenvalue j (0-based, ascending) is the point where the count passes j.
//
// L consecutive lanes of a wave share one eigenvalue: each iteration they count
// at L interior points of the current interval [lo, hi], split into L + 1 equal
// parts, and keep the part in which the count passes j (a ballot over the
// group: the counts are monotone in x, so the lanes with count <= j form a
// prefix). The interval shrinks by L + 1 per iteration, until its width is below
// max(2 eps max(|lo|, |hi|), eps ||T||) — the stopping rule of dstebz. The Gershgorin
// interval that starts it, widened by 2.1 eps ||T|| as in dstebz, is formed by every
// wave from (d, e) itself, so the kernel needs no scratch memory. Everything runs in
// FP64 (the float entry converts on load).
//
// Bound: the chain, about 45 cycles per row (measured; the instructions of a row issue in
// about 25). L is the largest of 4 .. 64 that keeps to about one wave per SIMD: more lanes
// take fewer iterations (log 2^53 / log (L + 1)), but past one wave per SIMD they wait for
// each other. (d_i, e_{i-1}^2) pairs come from LDS, 4080 rows at a time, one broadcast read
// per row. All eigenvalues, the pivot form with L = 8 throughout and this one: n = 1000 1.75
// and 0.20 ms, n = 3001 6.7 and 0.8, n = 8192 18.1 and 2.7, n = 16384 40.4 and 7.3.
#include "tridi_values.hpp"

#include <cfloat>

#include "sturm.hpp"

namespace cuev {
namespace {

constexpr int kTvThreads = 256;
constexpr int kTvRows = 4080; // (d, e^2) pairs per LDS stage, a multiple of 8 (64 KiB with the 8 more)
inline int tv_stage_rows(int n) { return n < kTvRows ? (n + 7) / 8 * 8 : kTvRows; }

template <typename T, int L>
__global__ __launch_bounds__(kTvThreads) void sturm_multisect_kernel(const T *__restrict__ d,
                                                                     const T *__restrict__ e, int n,
                                                                     int il, int iu, T *__restrict__ w) {
    extern __shared__ __align__(16) unsigned char tv_smem[];
    double2 *de = reinterpret_cast<double2 *>(tv_smem); // tv_stage_rows(n) + 8 rows
    const int tid = threadIdx.x, lane = tid & 63;
    // --- Gershgorin bounds and ||T||_inf, over the whole matrix (every wave)
    double gl = DBL_MAX, gu = -DBL_MAX;
    for (int i = lane; i < n; i += 64) {
        const double di = (double)d[i];
        const double el = (i > 0) ? fabs((double)e[i - 1]) : 0.0;
        const double er = (i < n - 1) ? fabs((double)e[i]) : 0.0;
        gl = fmin(gl, di - el - er);
        gu = fmax(gu, di + el + er);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        gl = fmin(gl, __shfl_xor(gl, o, 64));
        gu = fmax(gu, __shfl_xor(gu, o, 64));
    }
    const double eps = DBL_EPSILON * 0.5; // unit roundoff, as LAPACK's dlamch('P') / 2
    double tnorm = fmax(fabs(gl), fabs(gu));
    // scaled by 2^-ts, ||T|| < 1 (exact; a zero or non-finite ||T|| is left as it is)
    const int ts = (tnorm > 0.0 && tnorm < DBL_MAX) ? ilogb(tnorm) + 1 : 0;
    gl = ldexp(gl, -ts);
    gu = ldexp(gu, -ts);
    tnorm = ldexp(tnorm, -ts);
    const double fudge = 2.1 * eps * tnorm + 2.0 * DBL_MIN;
    gl -= fudge;
    gu += fudge;
    const double atol = 2.0 * eps * tnorm; // absolute part of the stopping width
    const double e2min = 0x1p-120;

    // --- one eigenvalue per group of L lanes
    const i64 grp = (blockIdx.x * (i64)kTvThreads + tid) / L;
    const i64 j = il + grp;
    const bool active = j <= iu;
    const int sub = lane % L;
    const int gbase = lane - sub;
    double lo = gl, hi = gu;
    const int nst = (n + kTvRows - 1) / kTvRows;
    for (int it = 0; it < 64; ++it) {
        const double width = hi - lo;
        const double tol = fmax(fmax(2.0 * eps * fmax(fabs(lo), fabs(hi)), atol), DBL_MIN);
        // groups stop independently; the others still join the barriers and the ballot
        const bool go = active && width > tol;
        if (!__syncthreads_or(go)) break;
        const double x = lo + width * (double)(sub + 1) / (double)(L + 1);
        const bool wave_go = __any(go);
        int cnt = 0;
        double pp = 0.0, p = 1.0;
        for (int st = 0; st < nst; ++st) {
            const int i0 = st * kTvRows, rows = min(kTvRows, n - i0);
            if (nst > 1 || it == 0) {
                __syncthreads(); // the stage before is read
                // rows past the last one, up to a multiple of 8: d - x > 0, e = 0, no sign change
                for (int i = tid; i < (int)((rows + 7) & ~7); i += kTvThreads) {
                    const double ei = (i < rows && i0 + i > 0) ? ldexp((double)e[i0 + i - 1], -ts) : 0.0;
                    de[i] = i < rows ? make_double2(ldexp((double)d[i0 + i], -ts), fmax(ei * ei, e2min))
                                     : make_double2(3.0, 0.0);
                }
                __syncthreads();
            }
            if (wave_go) cnt += sturm_rows(de, rows, x, pp, p);
        }
        // lanes of this group whose point has count <= j form a prefix of length q
        const unsigned long long below = __ballot(go && cnt <= j);
        const int q = __popcll((below >> gbase) & (~0ull >> (64 - L)));
        const double xl = __shfl(x, gbase + (q > 0 ? q - 1 : 0), 64);
        const double xh = __shfl(x, gbase + (q < L ? q : L - 1), 64);
        if (go) {
            if (q > 0) lo = xl;
            if (q < L) hi = xh;
        }
    }
    if (active && sub == 0) w[j - il] = (T)ldexp(0.5 * (lo + hi), ts);
}

template <typename T, int L>
void launch_multisect(hipStream_t s, const T *d, const T *e, int n, int il, int iu, T *w) {
    const i64 threads = (i64)(iu - il + 1) * L;
    hipLaunchKernelGGL((sturm_multisect_kernel<T, L>), dim3((unsigned)ceil_div(threads, kTvThreads)),
                       dim3(kTvThreads), sizeof(double2) * (size_t)(tv_stage_rows(n) + 8), s, d, e, n, il, iu, w);
}

} // namespace

template <typename T> int tridi_values(hipStream_t s, const T *d, const T *e, int n, int il, int iu, T *w) {
    if (n < 1 || !d || !w || (n > 1 && !e))
        CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "tridi_values: n=%d d=%p e=%p w=%p", n, (const void *)d,
                  (const void *)e, (void *)w);
    if (il < 0 || iu >= n || il > iu)
        CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "tridi_values: index range [%d, %d] outside [0, %d)", il, iu, n);
    // lanes per eigenvalue: about one wave per SIMD (4 per CU) for a whole spectrum. The
    // number asked for does not count, so a range gives the very values of the whole.
    const i64 lanes = (i64)device_cu_count() * 4 * 64;
    if ((i64)n * 64 <= lanes) launch_multisect<T, 64>(s, d, e, n, il, iu, w);
    else if ((i64)n * 32 <= lanes) launch_multisect<T, 32>(s, d, e, n, il, iu, w);
    else if ((i64)n * 16 <= lanes) launch_multisect<T, 16>(s, d, e, n, il, iu, w);
    else if ((i64)n * 8 <= lanes) launch_multisect<T, 8>(s, d, e, n, il, iu, w);
    else launch_multisect<T, 4>(s, d, e, n, il, iu, w);
    CUEV_LAUNCH_CHECK();
    return CUEV_STATUS_SUCCESS;
}

template int tridi_values<float>(hipStream_t, const float *, const float *, int, int, int, float *);
template int tridi_values<double>(hipStream_t, const double *, const double *, int, int, int, double *);

} // namespace cuev
