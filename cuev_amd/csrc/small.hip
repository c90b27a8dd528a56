// small.hip — dense symmetric eigenproblems of order <= 128, one workgroup per matrix
// with everything in LDS (no reference counterpart: the reference runs its two-stage
// pipeline at every order, src/cuda/solver.cu:25-79).
//
// Per matrix, FP64 throughout (also for float matrices), scaled by a power of two:
//   1. Householder tridiagonalization of the full matrix in registers, H_k = I - 2 w_k w_k^T;
//      the w_k go to the caller's V buffer as pairs of 32-bit words until step 5.
//   2. Eigenvalues of T by Sturm multisection (tridi_values.hip), all lanes of the
//      workgroup spread over them.
//   3. Eigenvectors of T, one thread each, by the twisted factorization (Dhillon and
//      Parlett): forward and backward pivots q+_i, q-_i of T - lambda, the twist r where
//      |gamma_i| = |q+_i + q-_i - (d_i - lambda)| is smallest, z_r = 1 and the two
//      recurrences outwards; lambda + gamma_r / ||z||^2 is its Rayleigh quotient.
//   4. One step of symmetric orthogonalization, Z <- Z (I - E/2), E = Z^T Z - I, on MFMA:
//      two vectors with a gap g carry an error of about eps ||T|| / g along each other, and
//      the step squares it (a second one follows for gaps below 1e-7 ||T||). The correction
//      between them is of that size and moves the residual by it times g, so residuals
//      stay at eps ||T||.
//   5. V = H_0 ... H_{n-3} Z, each column in the registers of a few neighbouring lanes.
// T is first split where |e_i| <= 8 u ||T|| (the deflation tolerance of the large solver's divide
// and conquer): blocks have their own eigenvalues, and vectors of different blocks
// are orthogonal whatever the gap, which covers multiple eigenvalues. Where two
// eigenvalues of one block are closer than 1e-10 ||T||, steps 2-4 give way to implicit QL with Wilkinson's shift on T (EISPACK tql2; Bowdler, Martin,
// Reinsch, Wilkinson 1968), which needs no gaps.
//
// Bound: latency. Steps 1 and 5 are chains of n short steps with barriers or lane
// exchanges, 2 and 3 chains of n multiply-adds or reciprocals. One workgroup per matrix and n x n
// of LDS keep 1 (n = 128) to 16 (n <= 32) matrices on a CU. The cyclic Jacobi method this
// replaces (batched.hip, kept for n > 128) needs 6 to 10 sweeps of n - 1 barriers each and
// about ten times the operations.
// Measured (whole calls, FP64): 2048 matrices of n = 32 1.28 ms by Jacobi and 0.20 here,
// 1024 of 64 5.6 and 0.50, 256 of 100 10.7 and 0.49, 512 of 128 48 and 1.2; one matrix of
// 48, 64 and 128 by the staged pipeline 0.50, 0.75 and 1.67 ms and 0.16, 0.20 and 0.54 here.
// A step of 1 takes about 1.1 us with one wave per SIMD and 2 us with two (n > 64).
#include "small.hpp"

#include <cfloat>
#include <mutex>

#include "sturm.hpp"
#include "wave.hpp"

namespace cuev {
namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

// Gaps, of ||T||, below which step 4 runs twice and below which QL takes over: E is about
// 1e-15 / gap, and after one step E^2, after two E^4, is left.
template <typename T> struct Gap;
template <> struct Gap<double> { static constexpr double once = 1e-7, min = 1e-10; };
template <> struct Gap<float> { static constexpr double once = 1e-10, min = 1e-11; }; // of 6e-8
// Largest exponent, either way, of a matrix that may be left to the staged pipeline, which is not scaled: it
// squares entries in FP64 (2^300: sums to 2^614; 2^-300: entries below 2^-510 are lost, 2^-210 of
// the largest) and works in T (FP32 with 26 binary digits of room at either end).
template <typename T> constexpr int kStagedExp = sizeof(T) == 8 ? 300 : 100;

// LDS in doubles: the n x n region (A, then Z, then the reflectors), then vectors
struct SmallLds {
    int np, ldz;                          // order rounded up to 16, Z's leading dimension
    int region, d, e, lam, w, y, de, part; // offsets
    int total;
};
__host__ __device__ inline SmallLds small_lds(int n, int waves) {
    SmallLds L{};
    L.np = (n + 15) / 16 * 16;
    L.ldz = L.np + 2;
    const int cols = L.np <= 32 ? 32 : L.np <= 64 ? 64 : 128; // step 1's columns
    int o = L.np * L.ldz > cols * (1 + 2 * waves) ? L.np * L.ldz : cols * (1 + 2 * waves);
    auto take = [&](int k) {
        const int at = o;
        o += k;
        return at;
    };
    L.d = take(L.np);
    L.e = take(L.np);
    L.lam = take(L.np);
    L.w = take(L.np);
    L.y = take(L.np);
    L.de = take(2 * (L.np + 8));
    L.part = take(waves * (L.np > 64 ? 128 : 64));
    L.total = o;
    return L;
}

__device__ __forceinline__ double fast_rcp(double q) {
    // v_rcp_f64 and two Newton steps; q is a guarded pivot, |q| in [2^-200, 2^200]
    double r = __builtin_amdgcn_rcp(q);
    r = fma(fma(-q, r, 1.0), r, r);
    return fma(fma(-q, r, 1.0), r, r);
}
__device__ __forceinline__ double guarded(double q) { return fabs(q) < 0x1p-200 ? -0x1p-200 : q; }

// One QL sweep's bookkeeping on (d, e) of order n by one wave (every lane alike): the next
// unreduced block l .. m is swept once, its rotations (c, s) of the planes (i, i + 1),
// i = m - 1 .. lo, left in cc, ss (lo = l unless the block splits on the way). Returns false
// when T is diagonal. tql2's recurrences.
__device__ bool ql_sweep(double *d, double *e, int n, int &l, int &m, int &lo, double *cc, double *ss) {
    const int lane = threadIdx.x & 63;
    unsigned long long cut[2]; // bit i: no coupling between i and i + 1
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int i = lane + 64 * u;
        bool z = i >= n - 1;
        if (!z) {
            const double ae = fabs(e[i]);
            z = ae <= 0.5 * DBL_EPSILON * (fabs(d[i]) + fabs(d[i + 1])) || ae < DBL_MIN;
        }
        cut[u] = __ballot(z);
    }
    for (; l < n - 1 && (cut[l >> 6] >> (l & 63) & 1); ++l) {}
    if (l >= n - 1) return false;
    m = l < 64 && (cut[0] >> l) ? l + __builtin_ctzll(cut[0] >> l)
                                : max(l, 64) + __builtin_ctzll(cut[1] >> (max(l, 64) - 64));
    if (m < n - 1) e[m] = 0.0;
    double g = (d[l + 1] - d[l]) / (2.0 * e[l]);
    g = d[m] - d[l] + e[l] / (g + copysign(sqrt(g * g + 1.0), g));
    double s = 1.0, c = 1.0, p = 0.0;
    int i = m - 1;
    double ei = e[i], di = d[i], dn = d[m]; // e_i, d_i, d_{i+1}, read ahead of the chain
    for (; i >= l; --i) {
        const double ep = i > l ? e[i - 1] : 0.0, dp = i > l ? d[i - 1] : 0.0;
        const double f = s * ei, b = c * ei;
        const double h = fma(g, g, f * f);
        if (h < DBL_MIN) { // the block splits here (T is scaled to entries of about 1)
            if (i + 1 < m) e[i + 1] = 0.0;
            d[i + 1] = dn - p;
            break;
        }
        double r, ri;
        fast_sqrt(h, r, ri);
        if (i + 1 < m) e[i + 1] = r;
        s = f * ri;
        c = g * ri;
        g = dn - p;
        const double q = fma(di - g, s, 2.0 * c * b);
        p = s * q;
        d[i + 1] = g + p;
        g = fma(c, q, -b);
        cc[i] = c;
        ss[i] = s;
        dn = di;
        di = dp;
        ei = ep;
    }
    lo = i + 1;
    if (i < l) {
        d[l] -= p;
        e[l] = g;
    }
    return true;
}

// One matrix per workgroup of NT threads, orders up to 16 NB. TRI: the matrix is tridiagonal, block
// `leaf` of the rows of (Ag, Eg), and steps 1 and 5 fall away; the eigenvalues go to W and the
// eigenvectors to the diagonal block of V (ld ldv) at the block's rows; eigenvalues NaN if QL fails.
template <typename T, int NT, int NB, bool TRI>
__device__ __forceinline__ void small_eig_body(const T *Ag, const T *Eg, int n, SmallLeaf leaf, T *W, T *V, i64 ldv, int il,
                                               int iu, int allow_ql, int *dflags, int *hflag) {
    constexpr int NW = NT / 64;
    constexpr int NBW = NB / NW > 1 ? NB / NW : 1; // column blocks of Z per wave in step 4
    constexpr int LPC = NT / (16 * NB);            // lanes per column in step 5
    constexpr int RP = 16 * NB / (2 * LPC);        // row pairs per lane
    extern __shared__ __align__(16) unsigned char small_smem[];
    double *sm = reinterpret_cast<double *>(small_smem);
    const SmallLds S = small_lds(n, NW);
    const int np = S.np, ldz = S.ldz, ld = n | 1;
    double *R = sm, *sd = sm + S.d, *se = sm + S.e, *slam = sm + S.lam, *sw = sm + S.w, *sy = sm + S.y,
           *part = sm + S.part;
    double2 *de = reinterpret_cast<double2 *>(sm + S.de);
    __shared__ int s_l, s_m, s_lo, s_more;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const i64 mat = (i64)n * n;
    const T *A = Ag + (TRI ? leaf.off : (i64)blockIdx.x * mat);
    unsigned *wg = reinterpret_cast<unsigned *>(V + (V ? (i64)blockIdx.x * mat : 0)); // packed reflectors, n (n - 1) words
    const int nout = V ? n : iu - il + 1;
    T *Wo = W + (TRI ? leaf.off : (i64)blockIdx.x * nout);
    bool unconverged = false; // TRI

    auto fail = [&](int which) { // host flag only on failure: a good call needs no copy back
        if (TRI) unconverged = true;
        else if (tid == 0) {
            atomicAdd(dflags + which, 1);
            __hip_atomic_store(hflag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    };

    int ts;
    if constexpr (TRI) {
        double amax = 0.0;
        for (int i = tid; i < n; i += NT) {
            sd[i] = (double)A[i];
            se[i] = i < n - 1 ? (double)Eg[leaf.off + i] : 0.0;
        }
        __syncthreads();
        for (int i = lane; i < n; i += 64) amax = fmax(amax, fmax(fabs(sd[i]), fabs(se[i])));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) amax = fmax(amax, __shfl_xor(amax, o, 64));
        ts = amax > 0.0 ? ilogb(amax) + 1 : 0;
        __syncthreads();
        for (int i = tid; i < n; i += NT) {
            sd[i] = ldexp(sd[i], -ts);
            se[i] = ldexp(se[i], -ts);
        }
        __syncthreads();
    } else {
    // ---- load the lower triangle, scale so that the largest entry is in [1/2, 1)
    double amax = 0.0;
    bool bad = false;
    for (int j = wave; j < n; j += NW)
        for (int i = j + lane; i < n; i += 64) {
            const double v = (double)A[i + (i64)j * n];
            bad |= !(fabs(v) <= DBL_MAX);
            amax = fmax(amax, fabs(v));
            R[j * ld + i] = v;
        }
    if (__syncthreads_or(bad)) {
        fail(1);
        const T nan = (T)__builtin_nan("");
        for (int i = tid; i < nout; i += NT) Wo[i] = nan;
        if (V)
            for (i64 i = tid; i < mat; i += NT) V[(i64)blockIdx.x * mat + i] = nan;
        return;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) amax = fmax(amax, __shfl_xor(amax, o, 64));
    if (lane == 0) part[wave] = amax;
    __syncthreads();
#pragma unroll
    for (int g = 0; g < NW; ++g) amax = fmax(amax, part[g]);
    ts = amax > 0.0 ? ilogb(amax) + 1 : 0;
    for (int j = wave; j < n; j += NW)
        for (int i = j + lane; i < n; i += 64) {
            const double v = ldexp(R[j * ld + i], -ts);
            R[j * ld + i] = v;
            R[i * ld + j] = v;
        }
    __syncthreads();

    // ---- 1. tridiagonalization, A in registers: thread = row `row` (and row + 64) and the 16
    // columns cg + NG t. Step k reads its column as row k, which one thread of each column
    // group holds; every wave forms the reflector from it, so only that row and the partial
    // sums of A w pass through LDS. w and y are zero up to row k: no masks.
    {
        constexpr int H = NB > 4 ? 2 : 1;     // row halves
        constexpr int RL = NB < 4 ? 32 : 64;  // lanes per column group
        constexpr int NG = NT / RL, CPT = 16;
        constexpr int CK = 4;                 // columns per skipped chunk
        static_assert(NG * CPT == 16 * NB, "columns");
        const int row = tid % RL, cg = tid / RL;
        double a[H][CPT];
#pragma unroll
        for (int u = 0; u < H; ++u)
#pragma unroll
            for (int t = 0; t < CPT; ++t) {
                const int i = row + 64 * u, c = cg + NG * t;
                a[u][t] = (i < n && c < n) ? R[c * ld + i] : 0.0;
            }
        // column c at [cg][t], so a group's columns are consecutive
        auto at = [&](int c) { return (c % NG) * CPT + c / NG; };
        // the region is free from here on: row k for all, and each wave's own copies of w
        // and y, which turn them from row to column order
        constexpr int C = 16 * NB;
        double *sx = R, *pw = R + C * (1 + 2 * wave), *py = pw + C;
        auto turn = [&](double *to, const double (&v)[H]) {
#pragma unroll
            for (int u = 0; u < H; ++u) to[at(row + 64 * u)] = v[u];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // this wave's reads only
        };
        __syncthreads();
        int off = 0; // of w_k in the packed reflectors
        for (int k = 0; k < n; ++k) {
            if (row == (k & 63)) {
#pragma unroll
                for (int t = 0; t < CPT; ++t) sx[cg * CPT + t] = (H == 2 && k >= 64) ? a[H - 1][t] : a[0][t];
            }
            __syncthreads();
            if (k >= n - 2) {
                if (tid == 0) {
                    sd[k] = sx[at(k)];
                    se[k] = k == n - 2 ? sx[at(n - 1)] : 0.0;
                }
                __syncthreads();
                continue;
            }
            double x[H], w[H];
            double sq = 0.0;
#pragma unroll
            for (int u = 0; u < H; ++u) {
                const int i = row + 64 * u;
                x[u] = (i > k && i < n) ? sx[at(i)] : 0.0;
                sq += i > k + 1 ? x[u] * x[u] : 0.0;
            }
            const double alpha = sx[at(k + 1)], diag = sx[at(k)];
            const double tail = group_sum<RL>(sq);
            // (entries are below about n: a tail below 2^-900 is zero to every digit)
            const bool zero = tail < 0x1p-900;
            double beta = alpha, t0 = 0.0, inv = 0.0;
            if (!zero) {
                double nrm, ri;
                fast_sqrt(alpha * alpha + tail, nrm, ri);
                beta = alpha >= 0.0 ? -nrm : nrm;
                t0 = alpha - beta;
                fast_sqrt(t0 * t0 + tail, ri, inv);
            }
#pragma unroll
            for (int u = 0; u < H; ++u) w[u] = (row + 64 * u == k + 1 ? t0 : x[u]) * inv;
            if (tid == 0) {
                sd[k] = diag;
                se[k] = beta;
            }
            if (V && cg == NG - 1) {
#pragma unroll
                for (int u = 0; u < H; ++u) {
                    const int i = row + 64 * u;
                    if (i > k && i < n) {
                        unsigned *o = wg + 2 * (off + i - k - 1);
                        o[0] = (unsigned)__double2loint(w[u]);
                        o[1] = (unsigned)__double2hiint(w[u]);
                    }
                }
            }
            off += n - 1 - k;
            if (zero) { // the identity (the same in every wave)
                __syncthreads();
                continue;
            }
            double wc[CPT], ac[H][CK], acc[H], y[H];
#pragma unroll
            for (int u = 0; u < H; ++u)
#pragma unroll
                for (int t = 0; t < CK; ++t) ac[u][t] = 0.0;
            turn(pw, w);
#pragma unroll
            for (int c0 = 0; c0 < CPT; c0 += CK)
                if (NG * (c0 + CK) - 1 > k) { // some column of the chunk past k
#pragma unroll
                    for (int t = c0; t < c0 + CK; ++t) wc[t] = pw[cg * CPT + t];
#pragma unroll
                    for (int t = c0; t < c0 + CK; ++t)
#pragma unroll
                        for (int u = 0; u < H; ++u) ac[u][t - c0] = fma(a[u][t], wc[t], ac[u][t - c0]);
                }
#pragma unroll
            for (int u = 0; u < H; ++u) acc[u] = (ac[u][0] + ac[u][1]) + (ac[u][2] + ac[u][3]);
            if constexpr (NW == 1) {
                double o = acc[0];
                lane_swap<32>(acc[0], o);
                acc[0] += o;
            } else {
#pragma unroll
                for (int u = 0; u < H; ++u) part[wave * (64 * H) + row + 64 * u] = acc[u];
                __syncthreads();
#pragma unroll
                for (int u = 0; u < H; ++u) {
                    double v[NW];
#pragma unroll
                    for (int g = 0; g < NW; ++g) v[g] = part[g * (64 * H) + row + 64 * u];
#pragma unroll
                    for (int d = NW / 2; d > 0; d /= 2)
#pragma unroll
                        for (int g = 0; g < d; ++g) v[g] += v[g + d];
                    acc[u] = v[0];
                }
            }
            double kp = 0.0;
#pragma unroll
            for (int u = 0; u < H; ++u) kp += w[u] * (2.0 * acc[u]);
            const double kap = group_sum<RL>(kp);
#pragma unroll
            for (int u = 0; u < H; ++u) y[u] = 2.0 * acc[u] - kap * w[u];
            turn(py, y);
#pragma unroll
            for (int c0 = 0; c0 < CPT; c0 += CK)
                if (NG * (c0 + CK) - 1 > k) {
                    double yc[CK];
#pragma unroll
                    for (int t = 0; t < CK; ++t) yc[t] = py[cg * CPT + c0 + t];
#pragma unroll
                    for (int t = 0; t < CK; ++t)
#pragma unroll
                        for (int u = 0; u < H; ++u)
                            a[u][c0 + t] = fma(-w[u], yc[t], fma(-y[u], wc[c0 + t], a[u][c0 + t]));
                }
        }
    }

    } // !TRI

    // ---- 2. eigenvalues of T: L lanes each
    double tnorm;
    unsigned long long cut[2]; // bit i: T is split between i and i + 1 (the last row's is set)
    auto block = [&](int i, int &b0, int &b1) { // the block [b0, b1] of row i
        const int h = i >> 6, o = i & 63;
        const unsigned long long up = cut[h] >> o;
        b1 = up ? i + __builtin_ctzll(up) : 64 + __builtin_ctzll(cut[1]);
        const unsigned long long dn = o ? cut[h] << (64 - o) : 0ull;
        b0 = dn ? i - __builtin_clzll(dn) : (h && cut[0]) ? 64 - __builtin_clzll(cut[0]) : 0;
    };
    bool split;
    {
        double gl = DBL_MAX, gu = -DBL_MAX;
        for (int i = lane; i < n; i += 64) {
            const double el = i > 0 ? fabs(se[i - 1]) : 0.0, er = fabs(se[i]); // se[n - 1] = 0
            gl = fmin(gl, sd[i] - el - er);
            gu = fmax(gu, sd[i] + el + er);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            gl = fmin(gl, __shfl_xor(gl, o, 64));
            gu = fmax(gu, __shfl_xor(gu, o, 64));
        }
        tnorm = fmax(fabs(gl), fabs(gu));
        const double eps = DBL_EPSILON * 0.5, e2min = 0x1p-120 * tnorm * tnorm;
        const double negligible = 8.0 * eps * tnorm;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int i = lane + 64 * u;
            cut[u] = __ballot(i == n - 1 || (i < n - 1 && fabs(se[i]) <= negligible));
        }
        split = __popcll(cut[0]) + __popcll(cut[1]) > 1;
        const int rows = (n + 7) & ~7;
        for (int i = tid; i < rows; i += NT) {
            const double ei = (i > 0 && i < n && fabs(se[i - 1]) > negligible) ? se[i - 1] : 0.0;
            de[i] = i < n ? make_double2(sd[i], fmax(ei * ei, e2min)) : make_double2(3.0 * tnorm + 1.0, 0.0);
        }
        __syncthreads();
        for (int i = tid; i < n; i += NT)
            if (fabs(se[i]) <= negligible) se[i] = 0.0;
        int L = 64; // lanes per eigenvalue
        while (L * n > NT) L >>= 1;
        const int j = tid / L, sub = lane & (L - 1), gbase = lane - sub;
        const bool active = j < n;
        int b0 = 0, b1 = n - 1; // eigenvalue j - b0 of block [b0, b1]
        if (split && active) block(j, b0, b1);
        int maxlen = b1 - b0 + 1;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) maxlen = max(maxlen, __shfl_xor(maxlen, o, 64));
        const unsigned long long gmask = ~0ull >> (64 - L);
        double lo = gl - 2.1 * eps * tnorm - DBL_MIN, hi = gu + 2.1 * eps * tnorm + DBL_MIN;
        const double atol = 2.0 * eps * tnorm, frac = 1.0 / (double)(L + 1);
        for (int it = 0; it < 64; ++it) {
            const double width = hi - lo;
            const bool go = active && width > fmax(fmax(2.0 * eps * fmax(fabs(lo), fabs(hi)), atol), DBL_MIN);
            if (!__any(go)) break;
            const double x = lo + width * ((double)(sub + 1) * frac);
            double pp = 0.0, p = 1.0;
            int cnt = 0;
            if (!split) {
                cnt = sturm_rows(de, rows, x, pp, p);
            } else { // each lane over its own block
                for (int r = 0; r < maxlen; ++r) {
                    const double2 v = de[min(b0 + r, b1)];
                    const double t = fma(v.x - x, p, -(v.y * pp));
                    if (b0 + r <= b1) {
                        cnt += (int)((unsigned)(__double2hiint(t) ^ __double2hiint(p)) >> 31);
                        pp = p;
                        p = t;
                    }
                    if ((r & 7) == 7) {
                        const int ex = __builtin_amdgcn_frexp_exp(fmax(fabs(pp), fabs(p)));
                        pp = ldexp(pp, -ex);
                        p = ldexp(p, -ex);
                    }
                }
            }
            const unsigned long long below = __ballot(go && cnt <= j - b0);
            const int q = __popcll((below >> gbase) & gmask);
            const double xl = __shfl(x, gbase + (q > 0 ? q - 1 : 0), 64);
            const double xh = __shfl(x, gbase + (q < L ? q : L - 1), 64);
            if (go) {
                if (q > 0) lo = xl;
                if (q < L) hi = xh;
            }
        }
        if (active && sub == 0) slam[j] = b0 == b1 ? sd[j] : 0.5 * (lo + hi);
        __syncthreads();
    }
    // ascending position of eigenvalue j (blocks and QL leave them unordered)
    auto rank = [&](int j) {
        const double lj = slam[j];
        int pos = 0;
        for (int i = 0; i < n; ++i) {
            const double v = slam[i];
            pos += v < lj || (v == lj && i < j);
        }
        return pos;
    };
    if (!V) {
        for (int i = tid; i < n; i += NT) {
            const int pos = split ? rank(i) : i;
            if (pos >= il && pos <= iu) Wo[pos - il] = (T)ldexp(slam[i], ts);
        }
        return;
    }
    int close = 0;
    for (int i = tid; i < n - 1; i += NT)
        if (!(cut[i >> 6] >> (i & 63) & 1)) {
            const double gap = slam[i + 1] - slam[i];
            close |= (gap < Gap<T>::once * tnorm ? 1 : 0) | (gap < Gap<T>::min * tnorm ? 2 : 0);
        }
    const bool twice = __syncthreads_or(close & 1), ql = __syncthreads_or(close & 2);
    if (ql && !allow_ql && ts >= -kStagedExp<T> && ts <= kStagedExp<T>) {
        fail(2);
        return;
    }

    // ---- 3. eigenvectors of T into Z (row i, column j at R[i ldz + j])
    for (int i = tid; i < np * ldz; i += NT) R[i] = 0.0;
    __syncthreads();
    if (!ql) {
        if (tid < n) {
            const int j = tid;
            const double x = slam[j];
            double *z = R + j;
            int b0 = 0, b1 = n - 1;
            if (split) block(j, b0, b1);
            // 1 / q+_i into Z
            double ri = 0.0;
            for (int i = b0; i <= b1; ++i) {
                const double ei = i > b0 ? se[i - 1] : 0.0;
                ri = fast_rcp(guarded((sd[i] - x) - ei * ei * ri));
                z[i * ldz] = ri;
            }
            // backwards: 1 / q-_i and gamma_i = q+_i - e_i^2 / q-_{i+1}; the smallest one
            double rm = 0.0, best = DBL_MAX, gr = 0.0;
            int r = b1;
            for (int i = b1; i >= b0; --i) {
                const double t = se[i] * se[i] * rm, dx = sd[i] - x; // rm = 0 at the block's end
                const double el = i > b0 ? se[i - 1] : 0.0;
                const double gam = dx - (i > b0 ? el * el * z[(i - 1) * ldz] : 0.0) - t;
                rm = fast_rcp(guarded(dx - t));
                if (fabs(gam) < best) {
                    best = fabs(gam);
                    gr = gam;
                    r = i;
                }
            }
            double nrm = 1.0, v = 1.0;
            for (int i = r - 1; i >= b0; --i) {
                v = -se[i] * v * z[i * ldz];
                z[i * ldz] = v;
                nrm += v * v;
            }
            rm = 0.0;
            for (int i = b1; i > r; --i) {
                rm = fast_rcp(guarded((sd[i] - x) - se[i] * se[i] * rm));
                z[i * ldz] = rm;
            }
            v = 1.0;
            z[r * ldz] = 1.0;
            for (int i = r + 1; i <= b1; ++i) {
                v = -se[i - 1] * v * z[i * ldz];
                z[i * ldz] = v;
                nrm += v * v;
            }
            const double inv = 1.0 / sqrt(nrm);
            for (int i = b0; i <= b1; ++i) z[i * ldz] *= inv;
            slam[j] = x + gr / nrm;
        }
        __syncthreads();

        // ---- 4. Z <- Z - Z E / 2. A wave owns 16-column blocks of Z; its blocks of E = Z^T Z - I
        // stay in the accumulators, whose layout (row l/16 + 4r, column l%16) is that of the
        // next product's second operand.
        const int li = lane & 15, lj = lane >> 4, nb = np / 16;
        for (int rep = twice ? 2 : 1; rep > 0; --rep) {
            v4d out[NBW][NB];
#pragma unroll
            for (int q = 0; q < NBW; ++q) {
                const int b = wave + NW * q;
                if (b >= nb) continue;
                v4d g[NB];
#pragma unroll
                for (int a = 0; a < NB; ++a) g[a] = v4d{0, 0, 0, 0};
                for (int k = 0; k < np; k += 4) {
                    const double *zr = R + (k + lj) * ldz + li;
                    const double bf = zr[16 * b];
#pragma unroll
                    for (int a = 0; a < NB; ++a)
                        if (a < nb) g[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(zr[16 * a], bf, g[a], 0, 0, 0);
                }
#pragma unroll
                for (int a = 0; a < NB; ++a) {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        g[a][r] = -0.5 * (g[a][r] - ((a == b && lj + 4 * r == li) ? 1.0 : 0.0));
                    out[q][a] = v4d{0, 0, 0, 0};
                }
#pragma unroll
                for (int a = 0; a < NB; ++a)
                    if (a < nb)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
#pragma unroll
                            for (int i = 0; i < NB; ++i)
                                if (i < nb)
                                    out[q][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                        R[(16 * i + li) * ldz + 16 * a + 4 * r + lj], g[a][r], out[q][i], 0, 0, 0);
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < NBW; ++q) {
                const int b = wave + NW * q;
                if (b >= nb) continue;
#pragma unroll
                for (int i = 0; i < NB; ++i)
                    if (i < nb)
#pragma unroll
                        for (int r = 0; r < 4; ++r) R[(16 * i + lj + 4 * r) * ldz + 16 * b + li] += out[q][i][r];
            }
            __syncthreads();
        }
    } else {
        // QL: wave 0 sweeps (d, e), the threads apply each sweep to their row of Z
        for (int i = tid; i < n; i += NT) R[i * ldz + i] = 1.0;
        if (tid == 0) s_l = 0;
        __syncthreads();
        for (int it = 0;; ++it) {
            if (wave == 0) {
                int l = s_l, m = 0, lo = 0;
                const bool more = it < 60 * n && ql_sweep(sd, se, n, l, m, lo, sw, sy);
                if (lane == 0) {
                    s_more = more;
                    s_l = l;
                    s_m = m;
                    s_lo = lo;
                }
                if (it == 60 * n) fail(0);
            }
            __syncthreads();
            if (!s_more) break;
            if (tid < n) {
                double *z = R + tid * ldz;
                double hi = z[s_m];
                for (int i = s_m - 1; i >= s_lo; i -= 4) { // four rotations' reads at once
                    double c[4], r[4], x[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int k = max(i - u, s_lo);
                        c[u] = sw[k];
                        r[u] = sy[k];
                        x[u] = z[k];
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (i - u >= s_lo) {
                            z[i - u + 1] = r[u] * x[u] + c[u] * hi;
                            hi = c[u] * x[u] - r[u] * hi;
                        }
                }
                z[s_lo] = hi;
            }
            __syncthreads();
        }
        for (int i = tid; i < n; i += NT) slam[i] = sd[i];
        __syncthreads();
    }

    if constexpr (TRI) {
        const double bad = __syncthreads_or(unconverged) ? __builtin_nan("") : 0.0;
        for (int j = wave; j < n; j += NW) {
            const int pos = rank(j);
            if (lane == 0) Wo[pos] = (T)(ldexp(slam[j], ts) + bad);
            for (int i = lane; i < n; i += 64) V[leaf.off + i + (i64)(leaf.off + pos) * ldv] = (T)R[i * ldz + j];
        }
        return;
    }

    // ---- 5. V = H_0 ... H_{n-3} Z: LPC neighbouring lanes per column, rows 2 (t LPC + q) + {0, 1}
    const int j = tid / LPC, q = tid % LPC;
    double2 z[RP];
#pragma unroll
    for (int t = 0; t < RP; ++t) {
        const int i = 2 * (t * LPC + q);
        z[t] = (i < np && j < np) ? make_double2(R[i * ldz + j], R[(i + 1) * ldz + j]) : make_double2(0.0, 0.0);
    }
    const int pos = j < n ? rank(j) : 0;
    if (j < n && q == 0) Wo[pos] = (T)ldexp(slam[j], ts);
    __syncthreads();
    for (int k = wave; k < n - 2; k += NW) {
        const unsigned *o = wg + 2 * (k * (n - 1) - k * (k - 1) / 2) - 2 * (k + 1);
        for (int i = lane; i < np; i += 64)
            R[k * np + i] = (i > k && i < n) ? __hiloint2double((int)o[2 * i + 1], (int)o[2 * i]) : 0.0;
    }
    __syncthreads();
    for (int k = n - 3; k >= 0; --k) {
        const double2 *wk = reinterpret_cast<const double2 *>(R + k * np) + q;
        double2 w[RP];
        double s = 0.0;
        constexpr int CK = 4; // row pairs per skipped chunk: w_k starts at row k + 1
#pragma unroll
        for (int t0 = 0; t0 < RP; t0 += CK) {
            const bool on = 2 * (t0 + CK) * LPC > k + 1 && 2 * t0 * LPC < n; // uniform
            if (on) {
#pragma unroll
                for (int t = t0; t < t0 + CK; ++t) {
                    w[t] = 2 * (t * LPC + q) < np ? wk[t * LPC] : make_double2(0.0, 0.0);
                    s += z[t].x * w[t].x + z[t].y * w[t].y;
                }
            }
        }
        if constexpr (LPC >= 2) s += dpp_mov<kQuadXor1>(s);
        if constexpr (LPC >= 4) s += dpp_mov<kQuadXor2>(s);
        s *= 2.0;
#pragma unroll
        for (int t0 = 0; t0 < RP; t0 += CK) {
            const bool on = 2 * (t0 + CK) * LPC > k + 1 && 2 * t0 * LPC < n;
            if (on) {
#pragma unroll
                for (int t = t0; t < t0 + CK; ++t) {
                    z[t].x -= s * w[t].x;
                    z[t].y -= s * w[t].y;
                }
            }
        }
    }
    if (j < n) {
        T *vo = V + (i64)blockIdx.x * mat + (i64)pos * n;
#pragma unroll
        for (int t = 0; t < RP; ++t) {
            const int i = 2 * (t * LPC + q);
            if (i < n) vo[i] = (T)z[t].x;
            if (i + 1 < n) vo[i + 1] = (T)z[t].y;
        }
    }
}

template <typename T, int NT, int NB>
__global__ __launch_bounds__(NT) void small_eig_kernel(const T *A, int n, T *W, T *V, int il, int iu, int allow_ql,
                                                       int *dflags, int *hflag) {
    small_eig_body<T, NT, NB, false>(A, nullptr, n, SmallLeaf{}, W, V, 0, il, iu, allow_ql, dflags, hflag);
}
template <typename T, int NT, int NB>
__global__ __launch_bounds__(NT) void small_tridi_kernel(const T *d, const T *e, const SmallLeaf *leaves, T *W, T *V, i64 ldv) {
    const SmallLeaf L = leaves[blockIdx.x];
    small_eig_body<T, NT, NB, true>(d, e, L.sz, L, W, V, ldv, 0, L.sz - 1, 1, nullptr, nullptr);
}

template <typename T, int NT, int NB>
int launch_small(hipStream_t s, const T *A, int n, int batch, T *W, T *V, int il, int iu, int allow_ql, int *dflags,
                 int *hflag) {
    const size_t lds = sizeof(double) * (size_t)small_lds(n, NT / 64).total;
    CUEV_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(small_eig_kernel<T, NT, NB>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((small_eig_kernel<T, NT, NB>), dim3((unsigned)batch), dim3(NT), lds, s, A, n, W, V, il, iu,
                       allow_ql, dflags, hflag);
    CUEV_LAUNCH_CHECK();
    return CUEV_STATUS_SUCCESS;
}

// ---- failure counters: three device ints and a pinned host flag per call in flight, kept
// between calls (at most kKeep per device)
struct Counters {
    int *dev = nullptr;  // [3], zero while idle
    int *host = nullptr; // zero while idle
    int device = -1;
};
constexpr int kKeep = 8;
std::mutex g_mu;
Counters g_idle[64][kKeep];

void counters_free(Counters &c) {
    if (c.dev) (void)hipFree(c.dev);
    if (c.host) (void)hipHostFree(c.host);
    c = Counters{};
}
int counters_take(Counters &c, int dev, hipStream_t s) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        for (Counters &x : g_idle[dev & 63])
            if (x.dev && x.device == dev) {
                c = x;
                x = Counters{};
                return CUEV_STATUS_SUCCESS;
            }
    }
    c.device = dev;
    const int zero[3] = {0, 0, 0};
    if (hipMalloc(reinterpret_cast<void **>(&c.dev), sizeof(zero)) != hipSuccess ||
        hipHostMalloc(reinterpret_cast<void **>(&c.host), sizeof(int), hipHostMallocDefault) != hipSuccess) {
        counters_free(c);
        CUEV_FAIL(CUEV_STATUS_ALLOC_FAILED, "small_eig: allocation of the failure counters failed");
    }
    *c.host = 0;
    const hipError_t e = hipMemcpyAsync(c.dev, zero, sizeof(zero), hipMemcpyHostToDevice, s);
    if (e != hipSuccess) {
        counters_free(c);
        CUEV_FAIL(CUEV_STATUS_HIP_ERROR, "small_eig: %s", hipGetErrorString(e));
    }
    return CUEV_STATUS_SUCCESS;
}
void counters_give(Counters &c) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        for (Counters &x : g_idle[c.device & 63])
            if (!x.dev) {
                x = c;
                c = Counters{};
                return;
            }
    }
    counters_free(c);
}

} // namespace

void small_release_all() {
    Counters victims[64][kKeep];
    {
        std::lock_guard<std::mutex> lk(g_mu);
        for (int d = 0; d < 64; ++d)
            for (int k = 0; k < kKeep; ++k) {
                victims[d][k] = g_idle[d][k];
                g_idle[d][k] = Counters{};
            }
    }
    int cur = 0;
    (void)hipGetDevice(&cur);
    for (auto &row : victims)
        for (Counters &c : row)
            if (c.dev) {
                (void)hipSetDevice(c.device);
                counters_free(c);
            }
    (void)hipSetDevice(cur);
}

template <typename T>
int small_eig(hipStream_t s, const T *A, int n, int batch, T *W, T *V, int il, int iu, int *n_failed, int *n_not_finite,
              int *n_need_ql) {
    *n_failed = *n_not_finite = 0;
    if (n_need_ql) *n_need_ql = 0;
    if (n < 1 || n > kSmallMaxN)
        CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "small_eig: n=%d outside [1, %d]", n, kSmallMaxN);
    if (batch < 1) return CUEV_STATUS_SUCCESS;
    int dev = 0;
    CUEV_HIP(hipGetDevice(&dev));
    Counters c;
    CUEV_TRY(counters_take(c, dev, s));
    // threads by order: one wave up to 32, so a CU holds many matrices; eight waves above 64
    int st;
    if (n <= 32) st = launch_small<T, 64, 2>(s, A, n, batch, W, V, il, iu, n_need_ql == nullptr, c.dev, c.host);
    else if (n <= 64) st = launch_small<T, 256, 4>(s, A, n, batch, W, V, il, iu, n_need_ql == nullptr, c.dev, c.host);
    else st = launch_small<T, 512, 8>(s, A, n, batch, W, V, il, iu, n_need_ql == nullptr, c.dev, c.host);
    const hipError_t e = hipStreamSynchronize(s);
    if (st != CUEV_STATUS_SUCCESS || e != hipSuccess) {
        counters_free(c);
        if (st != CUEV_STATUS_SUCCESS) return st;
        CUEV_FAIL(CUEV_STATUS_HIP_ERROR, "small_eig: %s", hipGetErrorString(e));
    }
    if (*static_cast<volatile int *>(c.host)) {
        int h[3] = {0, 0, 0};
        const hipError_t ce = hipMemcpy(h, c.dev, sizeof(h), hipMemcpyDeviceToHost);
        counters_free(c); // not zero any more
        if (ce != hipSuccess) CUEV_FAIL(CUEV_STATUS_HIP_ERROR, "small_eig: %s", hipGetErrorString(ce));
        *n_failed = h[0];
        *n_not_finite = h[1];
        if (n_need_ql) *n_need_ql = h[2];
        return CUEV_STATUS_SUCCESS;
    }
    counters_give(c);
    return CUEV_STATUS_SUCCESS;
}

template <typename T>
int small_tridi(hipStream_t s, const T *d, const T *e, const SmallLeaf *leaves, int nleaves, int max_sz, T *W, T *V,
                i64 ldv) {
    if (max_sz < 1 || max_sz > kSmallTridiMaxN)
        CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "small_tridi: order %d outside [1, %d]", max_sz, kSmallTridiMaxN);
    const size_t lds = sizeof(double) * (size_t)small_lds(max_sz, 4).total;
    CUEV_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(small_tridi_kernel<T, 256, 4>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((small_tridi_kernel<T, 256, 4>), dim3((unsigned)nleaves), dim3(256), lds, s, d, e, leaves, W, V, ldv);
    CUEV_LAUNCH_CHECK();
    return CUEV_STATUS_SUCCESS;
}

template int small_tridi<float>(hipStream_t, const float *, const float *, const SmallLeaf *, int, int, float *, float *, i64);
template int small_tridi<double>(hipStream_t, const double *, const double *, const SmallLeaf *, int, int, double *, double *,
                                 i64);
template int small_eig<float>(hipStream_t, const float *, int, int, float *, float *, int, int, int *, int *, int *);
template int small_eig<double>(hipStream_t, const double *, int, int, double *, double *, int, int, int *, int *,
                               int *);

} // namespace cuev
