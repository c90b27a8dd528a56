// panel_qr.hip — Householder QR of one DBBR panel as a single persistent kernel.
//
// Replaces the reference's panel step dbbr_panel_qr (src/cuda/dbbr.cu:124-143):
// cuSOLVER geqrf + dbbr_extract_reflectors (:55-71) + syrk G = Y^T Y (:140) +
// dbbr_larft (:86-109), and additionally forms W = Y T (the reference's GEMM at
// src/cuda/dbbr.cu:171) for the rows each workgroup owns.
//
// Convention (LAPACK dgeqr2/dlarfg, which the reference obtains from geqrf):
// for column c with pivot alpha = A[c,c] and tail x = A[c+1:, c],
//   xnorm == 0  ->  tau = 0, H = I, the column is left as is;
//   otherwise   ->  beta = -sign(alpha) * sqrt(alpha^2 + xnorm^2),
//                   tau  = (beta - alpha) / beta,  v = [1; x / (alpha - beta)],
//                   A[c,c] = beta, A[c+1:, c] = v[1:].
// T is the upper-triangular factor with H_0 ... H_{b-1} = I - Y T Y^T, built by
// the recurrence T[j,j] = tau_j, T[0:j, j] = -tau_j T[0:j,0:j] (Y^T Y)[0:j, j].
//
// Parallel structure: G workgroups, each owns CH consecutive panel rows and
// keeps them in LDS for the whole factorization. Per column one grid-wide
// reduction carries ||x||^2, the b-c-1 dot products x^T a_j and the Gram
// column of the previous reflector; every workgroup sums the G partial vectors
// in the same order, so all of them hold bit-identical scalars. Norms, dot
// products, tau and T are FP64 for both float and double panels.
// The grid is sized to be co-resident (one workgroup per CU at this LDS size);
// every wait is bounded and reports through *err.
#include "panel_qr.hpp"

#include <algorithm>
#include <type_traits>

#include "wave.hpp"

namespace cuev {
namespace {

constexpr int kPQThreads = 256;
constexpr size_t kPQGateBytes = 256; // scratch head: the CholQR -> Householder gate word

template <typename T> struct PQArgs {
    T *A;
    i64 lda;
    T *Y;
    i64 ldy;
    T *W;
    i64 ldw;
    T *Tm;
    T *tau;
    int rows, b, CH, G;
    double *part;   // [2][G][2b]
    double *pivot;  // [2][b]
    const int *gate; // when set: run only if *gate != 0 (the CholQR kernel declined the panel)
    unsigned *counter;
    unsigned *reset; // the CholQR kernel's barrier counter, zeroed for the next panel
    int *err;
};

// Grid barrier: all G workgroups arrive (counter reaches `target`), then all leave.
__device__ __forceinline__ bool grid_barrier(unsigned *counter, unsigned target, int *err) {
    wg_publish_fence();
    __shared__ int s_ok;
    if (threadIdx.x == 0) {
        counter_add_release(counter, 1u);
        long long it = 0;
        int ok = 1;
        while (counter_load_relaxed(counter) < target) {
            __builtin_amdgcn_s_sleep(1);
            if (++it > kSpinLimit) {
                __hip_atomic_store(err, (int)DEV_WATCHDOG, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
                ok = 0;
                break;
            }
        }
        fence_acquire_agent();
        s_ok = ok;
    }
    __syncthreads();
    return s_ok != 0;
}

// Write-through exchange for the CholQR kernel: every global access to data that
// another workgroup of the same launch reads (Gram partials, their sums, U and Mw)
// is an agent-scope relaxed atomic access. On gfx950 these carry the sc1 bit: the
// store is written through past the XCD-private L2 and the load reads from the
// device-coherent level. A grid barrier then needs neither an L2 write-back before
// the arrival nor an L2 invalidate after the wait: each wave waits until its own
// stores have completed (vmcnt(0)), the workgroup meets, one thread increments the
// counter and polls it, and the workgroup meets again.
__device__ __forceinline__ double ld_wt(const double *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_wt(double *p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool grid_wait_wt(unsigned *counter, unsigned target, int *err) {
    __shared__ int s_ok;
    if (threadIdx.x == 0) {
        long long it = 0;
        int ok = 1;
        while (counter_load_relaxed(counter) < target) {
            __builtin_amdgcn_s_sleep(1);
            if (++it > kSpinLimit) {
                __hip_atomic_store(err, (int)DEV_WATCHDOG, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
                ok = 0;
                break;
            }
        }
        s_ok = ok;
    }
    __syncthreads();
    return s_ok != 0;
}
__device__ __forceinline__ bool grid_barrier_wt(unsigned *counter, unsigned target, int *err) {
    vm_drain();
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return grid_wait_wt(counter, target, err);
}

template <typename T> __global__ __launch_bounds__(kPQThreads) void panel_qr_kernel(PQArgs<T> a) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    // the CholQR kernel before this one has finished: its counter is free
    if (blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(a.reset, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (a.gate && *a.gate == 0) return;
    const int b = a.b, CH = a.CH, CHp = CH + 1;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = blockIdx.x;

    // LDS layout
    double *GT = reinterpret_cast<double *>(smem_raw);   // [b][b+1]: Gram, then T (column-major)
    double *sums = GT + (size_t)b * (b + 1);             // [2b] reduced payload
    double *tauv = sums + 2 * b;                         // [b]
    double *prow = tauv + b;                             // [b] pivot row
    double *red4 = prow + b;                             // [256] partial-sum combine buffer
    double *red4b = red4 + 256;                          // [256] second combine buffer
    double *sx = red4b + 256;                            // [CH] x = column c below the diagonal
    double *sv = sx + CH;                                // [CH] reflector c-1 (unit at row c-1)
    double *sjv = sv + CH;                               // [b] tau * v^T a_j of the trailing columns
    T *P = reinterpret_cast<T *>(sjv + b);               // [b][CHp] panel rows of this workgroup

    const int r0g = g * CH;                              // first global panel row owned
    const int chl = max(0, min(CH, a.rows - r0g));       // rows owned
    const int PS = 2 * b;                                // payload stride

    // load the owned rows
    for (int idx = tid; idx < b * CH; idx += kPQThreads) {
        const int j = idx / CH, rl = idx - j * CH;
        P[j * CHp + rl] = (rl < chl) ? a.A[(i64)(r0g + rl) + (i64)j * a.lda] : T(0);
    }
    for (int idx = tid; idx < b * (b + 1); idx += kPQThreads) GT[idx] = 0.0;
    __syncthreads();

    bool alive = true;
    // past the last row there is only the Gram column of the last reflector left to form
    const int steps = min(b, a.rows);
    for (int c = 0; c <= steps; ++c) {
        const int buf = c & 1;
        const bool has_col = c < b && c < a.rows;
        const int ndot = has_col ? b - c : 0;           // q = 0: ||x||^2, q >= 1: x^T a_{c+q}
        const int ngram = (c >= 2 && c - 1 < a.rows) ? c - 1 : 0; // v_i^T v_{c-1}, i < c-1

        // (1) local partial sums: x^T a_j for j >= c (j = c: ||x||^2) and the Gram
        // column v_i^T v_{c-1}, i < c-1, from masked copies of x and v_{c-1}. Each
        // thread owns one column q and a quarter of the rows; no wave reductions.
        double *mypart = a.part + ((size_t)buf * a.G + g) * PS;
        const int nq = ndot + ngram;
        for (int rl = tid; rl < CH; rl += kPQThreads) {
            const int r = r0g + rl;
            const bool own = rl < chl;
            sx[rl] = (own && has_col && r > c) ? (double)P[c * CHp + rl] : 0.0;
            double v = 0.0;
            if (own && ngram) v = (r > c - 1) ? (double)P[(c - 1) * CHp + rl] : (r == c - 1 ? 1.0 : 0.0);
            sv[rl] = v;
        }
        __syncthreads();
        {
            const int qc = tid & 63, quarter = tid >> 6;
            const int QR = (CH + 3) >> 2;
            const int rb = quarter * QR, re = min(chl, rb + QR);
            double s1 = 0.0, s2 = 0.0;
            if (qc < b) {
                const T *pc = P + (size_t)qc * CHp;
                for (int rl = rb; rl < re; ++rl) {
                    const double pv = (double)pc[rl];
                    s1 += pv * sx[rl];
                    s2 += pv * sv[rl];
                }
            }
            red4[quarter * 64 + qc] = s1;
            red4b[quarter * 64 + qc] = s2;
        }
        __syncthreads();
        if (tid < b) {
            const int qc = tid;
            if (qc >= c && ndot)
                mypart[qc - c] = ((red4[qc] + red4[64 + qc]) + red4[128 + qc]) + red4[192 + qc];
            if (qc < ngram)
                mypart[b + qc] = ((red4b[qc] + red4b[64 + qc]) + red4b[128 + qc]) + red4b[192 + qc];
        }
        // pivot row A[c, c:b] from its owner
        if (has_col && c >= r0g && c < r0g + chl) {
            const int cl = c - r0g;
            for (int j = c + tid; j < b; j += kPQThreads)
                a.pivot[buf * b + j] = (double)P[j * CHp + cl];
        }

        // (2) grid-wide reduction
        if (a.G == 1) { // one workgroup (the last panels): no grid to wait for
            wave_stores_done();
            __syncthreads();
        } else if (!grid_barrier(a.counter, (unsigned)a.G * (unsigned)(c + 1), a.err)) alive = false;

        // Sum the G partial vectors: 4 threads per payload entry, each taking every
        // 4th workgroup with its loads issued back to back, then a fixed-order
        // combine, so every workgroup obtains bit-identical sums.
        {
            const int q = tid & 63, part = tid >> 6;
            double s = 0.0;
            if (q < nq) {
                const int slot = (q < ndot) ? q : b + (q - ndot);
                const double *src = a.part + (size_t)buf * a.G * PS + slot;
                // batches of 32 independent loads (one memory round trip per batch)
                for (int g0 = part; g0 < a.G; g0 += 4 * 32) {
                    double v[32];
#pragma unroll
                    for (int u = 0; u < 32; ++u) {
                        const int gg = g0 + 4 * u;
                        v[u] = (gg < a.G) ? src[(size_t)gg * PS] : 0.0;
                    }
#pragma unroll
                    for (int u = 0; u < 32; ++u) s += v[u];
                }
            }
            red4[part * 64 + q] = s;
        }
        __syncthreads();
        if (tid < nq) {
            const int slot = (tid < ndot) ? tid : b + (tid - ndot);
            sums[slot] = ((red4[tid] + red4[64 + tid]) + red4[128 + tid]) + red4[192 + tid];
        }
        if (has_col)
            for (int j = c + tid; j < b; j += kPQThreads) prow[j] = a.pivot[buf * b + j];
        __syncthreads();

        // Gram column c-1
        if (ngram)
            for (int i = tid; i < ngram; i += kPQThreads) GT[i + (size_t)(c - 1) * (b + 1)] = sums[b + i];
        if (!has_col) {
            for (int j = c + tid; j < b; j += kPQThreads) tauv[j] = 0.0;
            __syncthreads();
            continue;
        }

        // (3) reflector scalars (identical in every workgroup)
        const double alpha = prow[c];
        const double xnorm2 = sums[0];
        double beta, tau, scal;
        if (xnorm2 == 0.0) {
            beta = alpha;
            tau = 0.0;
            scal = 0.0;
        } else {
            const double nrm = sqrt(alpha * alpha + xnorm2);
            beta = (alpha >= 0.0) ? -nrm : nrm;
            tau = (beta - alpha) / beta;
            scal = 1.0 / (alpha - beta);
        }
        if (tid == 0) tauv[c] = tau;

        // (4) apply H = I - tau v v^T to columns c+1..b-1 of the owned rows:
        // a_j -= (tau v^T a_j) v with v^T a_j = a_j[c] + scal * (x^T a_j); each wave
        // takes every 4th column, each lane fixed rows (no index division)
        const int ntrail = b - c - 1;
        if (tau != 0.0) {
            for (int jj = tid; jj < ntrail; jj += kPQThreads)
                sjv[jj] = tau * (prow[c + 1 + jj] + scal * sums[1 + jj]);
            __syncthreads();
            for (int rl = lane; rl < chl; rl += 64) {
                const int r = r0g + rl;
                if (r < c) continue;
                const double vr = (r == c) ? 1.0 : (double)P[c * CHp + rl] * scal;
                for (int jj = wave; jj < ntrail; jj += kPQThreads / 64) {
                    T &e = P[(c + 1 + jj) * CHp + rl];
                    e = (T)((double)e - sjv[jj] * vr);
                }
            }
        }
        __syncthreads();
        for (int rl = tid; rl < chl; rl += kPQThreads) {
            const int r = r0g + rl;
            if (r == c) P[c * CHp + rl] = (T)beta;
            else if (r > c) P[c * CHp + rl] = (T)((double)P[c * CHp + rl] * scal);
        }
        __syncthreads();
    }
    (void)alive;

    // (5) T from the Gram matrix: column j overwrites Gram column j (zero past the last row)
    for (int j = 0; j < steps; ++j) {
        double t = 0.0;
        if (tid < j) {
            for (int q = tid; q < j; ++q) t += GT[tid + (size_t)q * (b + 1)] * GT[q + (size_t)j * (b + 1)];
            t *= -tauv[j];
        }
        __syncthreads();
        if (tid < j) GT[tid + (size_t)j * (b + 1)] = t;
        if (tid == j) GT[j + (size_t)j * (b + 1)] = tauv[j];
        __syncthreads();
    }
    for (int idx = tid; idx < b * b; idx += kPQThreads) {
        const int i = idx % b, j = idx / b;
        if (i > j) GT[i + (size_t)j * (b + 1)] = 0.0;
    }
    __syncthreads();

    // (6) outputs for the owned rows: A (R + reflector tails), Y (explicit), W = Y T
    for (int idx = tid; idx < b * chl; idx += kPQThreads) {
        const int j = idx / chl, rl = idx - j * chl;
        const int r = r0g + rl;
        const T pv = P[j * CHp + rl];
        a.A[(i64)r + (i64)j * a.lda] = pv;
        if (a.Y) a.Y[(i64)r + (i64)j * a.ldy] = (r > j) ? pv : (r == j ? T(1) : T(0));
    }
    if (a.W) {
        for (int idx = tid; idx < b * chl; idx += kPQThreads) {
            const int j = idx / chl, rl = idx - j * chl;
            const int r = r0g + rl;
            double s = 0.0;
            const int imax = min(j, r); // Y[r,i] = 0 for i > r
            for (int i = 0; i <= imax; ++i) {
                const double y = (r > i) ? (double)P[i * CHp + rl] : 1.0;
                s += y * GT[i + (size_t)j * (b + 1)];
            }
            a.W[(i64)r + (i64)j * a.ldw] = (T)s;
        }
    }
    if (g == 0) {
        for (int idx = tid; idx < b * b; idx += kPQThreads) {
            const int i = idx % b, j = idx / b;
            a.Tm[idx] = (T)GT[i + (size_t)j * (b + 1)];
        }
        for (int j = tid; j < b; j += kPQThreads) a.tau[j] = (T)tauv[j];
    }
}

// ---------------------------------------------------------------------------
// CholQR2 panel factorization with Householder reconstruction (the fast path).
//
// Two passes of Cholesky QR make an orthonormal Q with A = Q R (each pass: the
// Gram matrix P^T P of the panel, its Cholesky factor R_p and P <- P R_p^-1, so
// R = R_2 R_1). The Householder form of the same factorization follows from an
// LU factorization without pivoting of the top b x b block of Q with signs
// S = diag(s_k), s_k = -sign of the k-th pivot before the shift:
//   Q_1 - S = L U,  Y = [L; Q_2 U^-1],  T = -U S L^-T,  R_house = S R,
// so that (I - Y T Y^T)[:, :b] = Q S (Ballard, Demmel, Grigori, Jacquelin, Knight,
// Nguyen, "Reconstructing Householder vectors from tall-skinny QR", J. Parallel
// Distrib. Comput. 85, 2015). In exact arithmetic these are the reflectors,
// T and R of Householder QR on the panel itself, the LAPACK convention above.
// CholQR2 keeps Q orthonormal to working precision when cond(panel) is well
// below eps^-1/2; a panel whose first Gram pivots reveal a (nearly) dependent
// column (d_k <= 1e-10 G_kk, or not finite) is left untouched and flagged for
// the Householder kernel, which then runs in full (*gate = 1).
//
// Parallel structure: G workgroups (one per CU), each with CH rows in LDS.
// Per pass: partial Gram -> global, grid barrier, each workgroup sums a slice of
// the entries over all partials in a fixed order, grid barrier, then every
// workgroup factors the same b x b Gram matrix redundantly (bit-identical
// results everywhere), its rows of P stacked under it: the column operations that
// turn G into its Cholesky factor turn P into P R_p^-1, so no inverse is formed.
// Workgroup 0 then factors Q_1 and publishes U^-1 and Mw = -S L^-T: every workgroup
// forms its rows of W = Y T = (Q - [S; 0]) Mw and Y = Q_2 U^-1, workgroup 0 also
// T = U Mw and R = R_2 R_1. All arithmetic is FP64.
//
// Bound: latency, of the two eliminations (b dependent pivots each) and of the grid
// barriers. An elimination holds its matrix in registers, a row in each lane and the
// columns in groups of four dealt out to the waves: the wave that owns the next group
// brings it up to date, eliminates its four columns by itself (pivots and multipliers by
// lane reads) and passes them on through LDS, so there is one barrier for four columns;
// what the columns further right still miss is made up beside the next group. The products
// run on the FP64 matrix cores. Kernel time per panel at b = 64, averaged over a solve: 65 us at n = 333,
// 66 at 2500, 67 at 4096, 81 at 16384 (62 for its last panels, 114 for the first, where the barriers and
// sums over 255 workgroups add up); at b = 32 32 us at n = 1024. With a barrier for every column, 4 x 4
// blocks per thread, vector products and explicit inverses it took 150 (b = 32: 80), and 202 for the first at
// n = 16384. Of 60 us between stamps in the kernel, the first elimination takes 14, Q_1's 20, both Gram matrices
// 3.7 and their sums 8, the second pass 3.2 and W, Y and the top rows 8 (before: elimination and
// P R_1^-1 41, Q_1 33, Gram 9, second pass 16, W and Y 25).
constexpr int kCQThreads = 512;
constexpr int kCQWaves = kCQThreads / 64;
constexpr int kCQMaxCH = 96;

template <typename T> struct CQArgs {
    T *A;
    i64 lda;
    T *Y;
    i64 ldy;
    T *W;
    i64 ldw;
    T *Tm;
    T *tau;
    int rows, CH, G;
    double *part; // [G][tiles * 256] partial Gram matrices
    double *gsum; // [tiles * 256]
    double *bc;   // [2*b*b]: U^-1 (column-major), then Mw = -S L^-T (row-major)
    int *gate;
    unsigned *counter;
    unsigned *reset; // the Householder kernel's barrier counter, zeroed for the launch after this one
    int *err;
};

typedef double cq_v4 __attribute__((ext_vector_type(4)));
// D += A B, 16 x 16 x 4: lane l holds A(l % 16, l / 16), B(l / 16, l % 16), D(l / 16 + 4 r, l % 16)
__device__ __forceinline__ cq_v4 cq_mma(double a, double b, cq_v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Panel slice in LDS: element (r, c) at c * ld + r. A half wave's fragment read is 16 rows of two
// columns, or two rows of 16 columns (P^T P): a leading dimension of 18 modulo 32 spreads both
// over the banks (16 would put the second on four of 64). The b x b matrices, read two rows of 16
// columns at a time, have b + 2.
__host__ __device__ constexpr int cq_ldp(int CH) { return CH + (50 - CH % 32) % 32; }

// x as a value the compiler knows nothing about: addresses formed with it in a loop, or after an
// elimination, are formed there and not kept in registers from before.
__device__ __forceinline__ int cq_fresh(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// lower 16 x 16 tile q of a Gram matrix, row by row
__device__ __forceinline__ void cq_tile(int q, int &I, int &J) {
    I = q >= 6 ? 3 : (q >= 3 ? 2 : (q >= 1 ? 1 : 0));
    J = q - I * (I + 1) / 2;
}

// out (lower tiles, each as the accumulator's four registers x 64 lanes) = P^T P
template <int B> __device__ __forceinline__ void cq_gram(const double *P, int ldp, int CH, double *out, int wave, int lane) {
    constexpr int NT = (B / 16) * (B / 16 + 1) / 2;
    const int lr = lane & 15, lk = lane >> 4;
    for (int q = wave; q < NT; q += kCQWaves) {
        int I, J;
        cq_tile(q, I, J);
        const double *x = P + (size_t)(16 * I + lr) * ldp + lk, *y = P + (size_t)(16 * J + lr) * ldp + lk;
        cq_v4 acc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
        for (int r = 0; r < CH; r += 16) {
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[u & 1] = cq_mma(x[r + 4 * u], y[r + 4 * u], acc[u & 1]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) st_wt(out + q * 256 + u * 64 + lane, acc[0][u] + acc[1][u]);
    }
}

// 1 / sqrt(h), h in [1e-290, 1e290], and 1 / p, |p| in [1, 2^1000]: one step of third order from
// the instruction's 24 bits or more
__device__ __forceinline__ double cq_rsqrt(double h) {
    const double y = __builtin_amdgcn_rsq(h), e = fma(-h * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ double cq_rcp(double p) {
    const double r = __builtin_amdgcn_rcp(p), e = fma(-p, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

// Columns of a b-column matrix held by the waves: group c (columns 4 c .. 4 c + 3) in wave
// c % kCQWaves, as its local group c / kCQWaves.
template <int B> struct CQCols {
    static constexpr int NCH = B / 4;                                        // groups
    static constexpr int LC = NCH <= kCQWaves ? 1 : NCH / kCQWaves;          // local groups
    static constexpr int NC = 4 * LC;                                        // local columns
};

// Drives an elimination over the groups. factor(lc, c): the wave eliminates its local group
// lc = group c and writes it to buffer c % 3; load(c): reads group c from its buffer; apply(lc,
// c): brings local group lc up to date with the group read; rest(lc, c): other work on group
// c for local group lc that nothing waits for (the group's own columns included). A wave that
// has just eliminated group c + 1 leaves its other columns until the next step, beside the next
// wave's elimination.
template <int LC, typename F> __device__ __forceinline__ void cq_each(F &&f) {
    static_assert(LC <= 2, "local groups");
    f(std::integral_constant<int, 0>{});
    if constexpr (LC > 1) f(std::integral_constant<int, 1>{});
}
template <int B, typename Fa, typename Lo, typename Ap, typename Re>
__device__ __forceinline__ void cq_eliminate(int wave, Fa &&factor, Lo &&load, Ap &&apply, Re &&rest) {
    using C = CQCols<B>;
    if (wave == 0) factor(std::integral_constant<int, 0>{}, 0);
    int done = 0; // groups whose other work is done
#pragma unroll 1
    for (int c = 0; c < C::NCH; ++c) {
        __syncthreads(); // group c is in its buffer
        if (c + 1 < C::NCH && (c + 1) % kCQWaves == wave) {
            __builtin_amdgcn_s_setprio(3); // before the other wave of this SIMD
            load(c);
            cq_each<C::LC>([&](auto lc) {
                if (kCQWaves * lc() + wave == c + 1) {
                    apply(lc, c);
                    factor(lc, c + 1);
                }
            });
            __builtin_amdgcn_s_setprio(0);
            continue;
        }
#pragma unroll 1
        for (; done <= c; ++done) {
            load(done);
            cq_each<C::LC>([&](auto lc) {
                const int own = kCQWaves * lc() + wave;
                if (own > done + 1 && own < C::NCH) apply(lc, done);
                if (own < C::NCH) rest(lc, done);
            });
        }
    }
    __syncthreads(); // the buffers are free
}

// Cholesky factor of the b x b Gram matrix Gm (LDS, full, ld b + 2) with the panel rows below
// it: P <- P R^-1 in place; R (upper, column-major, ld b + 2) into Rout if it is set. False in
// every thread if a pivot falls below tol of its diagonal entry or is not finite.
template <int B, int NSET>
__device__ __forceinline__ bool cq_chol(double *P, int ldp, int CH, const double *Gm, double *buf, double *Rout,
                                        double tol, int *s_bad, int wave, int lane) {
    using C = CQCols<B>;
    constexpr int LD = B + 2, NR = 64 * NSET;
    double g[NSET][C::NC];
    // row q = 64 t + lane of [G; P]
#pragma unroll
    for (int lc = 0; lc < C::LC; ++lc)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = 4 * (kCQWaves * lc + wave) + u;
#pragma unroll
            for (int t = 0; t < NSET; ++t) {
                const int q = 64 * t + lane;
                double v = 0.0;
                if (j < B && q < B) v = Gm[q + j * LD];
                else if (j < B && q < B + CH) v = P[(size_t)j * ldp + q - B];
                g[t][4 * lc + u] = v;
            }
        }
    const double diag = lane < B ? Gm[lane + lane * LD] : 0.0;
    double piv[C::NC], l[4][NSET];
    auto factor = [&](auto lcc, int c) {
        constexpr int lc = decltype(lcc)::value;
        double *dst = buf + (size_t)(c % 3) * 4 * NR + lane;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int k = 4 * c + v;
            const double dk = read_lane(g[0][4 * lc + v], k), rs = cq_rsqrt(dk);
            piv[4 * lc + v] = dk; // looked at afterwards
            double w[NSET]; // in G's rows above k: what rounding left of zero, read by no one
#pragma unroll
            for (int t = 0; t < NSET; ++t) w[t] = g[t][4 * lc + v] *= rs;
#pragma unroll
            for (int u = v + 1; u < 4; ++u) {
                const double m = read_lane(w[0], 4 * c + u);
#pragma unroll
                for (int t = 0; t < NSET; ++t) g[t][4 * lc + u] -= w[t] * m;
            }
#pragma unroll
            for (int t = 0; t < NSET; ++t) dst[v * NR + 64 * t] = w[t];
        }
    };
    auto load = [&](int c) {
        const double *src = buf + (size_t)(c % 3) * 4 * NR + lane;
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int t = 0; t < NSET; ++t) l[v][t] = src[v * NR + 64 * t];
    };
    auto apply = [&](auto lcc, int) {
        constexpr int lc = decltype(lcc)::value;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = 4 * (kCQWaves * lc + wave) + u;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const double m = read_lane(l[v][0], j);
#pragma unroll
                for (int t = 0; t < NSET; ++t) g[t][4 * lc + u] -= l[v][t] * m;
            }
        }
    };
    cq_eliminate<B>(wave, factor, load, apply, [](auto, int) {});
#pragma unroll
    for (int lc = 0; lc < C::LC; ++lc)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = 4 * (kCQWaves * lc + wave) + u;
            const double d = piv[4 * lc + u];
            if (j < B && !(d > tol * read_lane(diag, j) && d > 1e-290 && d < 1e290)) *s_bad = 1;
        }
    __syncthreads();
    if (*s_bad) return false;
    const int ln = cq_fresh(lane);
#pragma unroll
    for (int lc = 0; lc < C::LC; ++lc)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = 4 * (kCQWaves * lc + wave) + u;
#pragma unroll
            for (int t = 0; t < NSET; ++t) {
                const int q = 64 * t + ln;
                if (j < B && q < B) {
                    if (Rout) Rout[j + q * LD] = q < j ? 0.0 : g[t][4 * lc + u];
                } else if (j < B && q < B + CH) P[(size_t)j * ldp + q - B] = g[t][4 * lc + u];
            }
        }
    __syncthreads();
    return true;
}

// Workgroup 0: Q_1 - S = L U for the top b rows of P, with L^-1 (row operations on I) and U^-1
// (column operations on I) alongside. L and U into LU (packed, ld b + 2; its memory, buf, is
// free before), U^-1 and Mw to bc, S to sv and into P's diagonal (Q_1 - S).
template <int B>
__device__ __forceinline__ void cq_lu(double *P, int ldp, double *LU, double *buf, double *bc, double *sv, int wave,
                                      int lane) {
    using C = CQCols<B>;
    constexpr int LD = B + 2;
    double m[C::NC], x[C::NC], z[C::NC], sg[C::NC];
#pragma unroll
    for (int lc = 0; lc < C::LC; ++lc)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = 4 * (kCQWaves * lc + wave) + u, q = 4 * lc + u;
            m[q] = (j < B && lane < B) ? P[(size_t)j * ldp + lane] : 0.0;
            x[q] = z[q] = lane == j ? 1.0 : 0.0;
            sg[q] = 1.0;
        }
    double l[4], xk[4];
    auto factor = [&](auto lcc, int c) {
        constexpr int lc = decltype(lcc)::value;
        double *dst = buf + (size_t)(c % 3) * 512 + lane;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int k = 4 * c + v, q = 4 * lc + v;
            const double mkk = read_lane(m[q], k);
            const double s = (mkk >= 0.0) ? -1.0 : 1.0;
            const double piv = mkk - s, rp = cq_rcp(piv);
            const double w = lane > k ? m[q] * rp : 0.0;
            sg[q] = s;
            m[q] = lane > k ? w : m[q];
            x[q] *= rp;
#pragma unroll
            for (int u = v + 1; u < 4; ++u) {
                const double mu = read_lane(m[4 * lc + u], k);
                m[4 * lc + u] -= w * mu;
                x[4 * lc + u] -= x[q] * mu;
            }
            dst[v * 64] = w;
            dst[256 + v * 64] = x[q];
        }
    };
    auto load = [&](int c) {
        const double *src = buf + (size_t)(c % 3) * 512 + lane;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            l[v] = src[v * 64];
            xk[v] = src[256 + v * 64];
        }
    };
    auto apply = [&](auto lcc, int c) {
        constexpr int lc = decltype(lcc)::value;
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const double mu = read_lane(m[4 * lc + u], 4 * c + v);
                m[4 * lc + u] -= l[v] * mu;
                x[4 * lc + u] -= xk[v] * mu;
            }
    };
    auto rest = [&](auto lcc, int c) {
        constexpr int lc = decltype(lcc)::value;
        if (kCQWaves * lc + wave > c) return; // columns of L^-1 that are still those of I
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int u = 0; u < 4; ++u) z[4 * lc + u] -= l[v] * read_lane(z[4 * lc + u], 4 * c + v);
    };
    cq_eliminate<B>(wave, factor, load, apply, rest);
    lane = cq_fresh(lane);
#pragma unroll
    for (int lc = 0; lc < C::LC; ++lc)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = 4 * (kCQWaves * lc + wave) + u, q = 4 * lc + u;
            if (j < B && lane < B) {
                st_wt(bc + lane + j * B, x[q]);
                st_wt(bc + B * B + lane + j * B, -sg[q] * z[q]); // Mw(j, lane) = -s_j L^-1(lane, j)
                LU[lane + j * LD] = lane == j ? m[q] - sg[q] : m[q];
                if (lane == j) {
                    sv[j] = sg[q];
                    P[(size_t)j * ldp + j] -= sg[q];
                }
            }
        }
}

// acc = tile (I, J), I <= J, of X Y for upper triangular X and Y (column-major, ld b + 2;
// entries of X below its diagonal are not read as zeros but masked)
template <int B> __device__ __forceinline__ cq_v4 cq_upper_mm(const double *X, const double *Y, int I, int J, cq_v4 acc, int lane) {
    constexpr int LD = B + 2;
    const int lr = lane & 15, lk = lane >> 4, i = 16 * I + lr;
    for (int k0 = 16 * I; k0 < 16 * (J + 1); k0 += 4) {
        const int k = k0 + lk;
        acc = cq_mma(k >= i ? X[i + k * LD] : 0.0, Y[k + (16 * J + lr) * LD], acc);
    }
    return acc;
}

// Up to 64 rows per workgroup four waves per SIMD (112 VGPRs, as fast as 174): the registers leave room for
// another kernel's waves on the CU, in LDS a panel of 64 columns (141 KB) for an unpadded bulge
// chase of another solve, not for a padded one or another panel. That every workgroup gets a CU
// does not depend on it (residency.hpp).
template <typename T, int B, int NSET>
__global__ __launch_bounds__(kCQThreads, NSET == 2 ? 4 : 2) void panel_cholqr_kernel(CQArgs<T> a) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    constexpr int LD = B + 2, BB = B * B, NTB = B / 16, NT = NTB * (NTB + 1) / 2, NE = 256 * NT;
    constexpr int NP = NTB > 2 ? NTB / 2 : 1; // pairs of column tiles {p, NTB - 1 - p}: equal work for triangular factors
    constexpr int KC = (B * LD > 768 * NSET) ? B * LD : 768 * NSET;
    const int CH = a.CH, ldp = cq_ldp(CH);
    const int tid = threadIdx.x, lane = tid & 63, g = blockIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lk = lane >> 4;
    double *P = reinterpret_cast<double *>(smem_raw); // [B][ldp]: panel(r, c) at P[c * ldp + r]
    double *MA = P + (size_t)B * ldp;                 // [B][LD]: Gram matrix; F or R_2; U^-1
    double *MB = MA + B * LD;                         // [B][LD]: R_1; Mw
    double *MC = MB + B * LD;                         // [KC]: column groups of the eliminations; L and U
    double *sv = MC + KC;                             // [B] signs S
    int *s_bad = reinterpret_cast<int *>(sv + B);     // [2]

    if (g == 0 && tid == 0) __hip_atomic_store(a.reset, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tid < 2) s_bad[tid] = 0;
    const int r0g = g * CH;
    const int chl = max(0, min(CH, a.rows - r0g));
    {
        // the panel slice: rounds of LB loads per thread, all issued before their LDS stores
        constexpr int LB = 8;
        for (int base = 0; base < B * CH; base += LB * kCQThreads) {
            double v[LB];
#pragma unroll
            for (int q = 0; q < LB; ++q) {
                const int idx = base + q * kCQThreads + tid;
                const int j = idx / CH, rl = idx - j * CH;
                v[q] = (idx < B * CH && rl < chl) ? (double)a.A[(i64)(r0g + rl) + (i64)j * a.lda] : 0.0;
            }
#pragma unroll
            for (int q = 0; q < LB; ++q) {
                const int idx = base + q * kCQThreads + tid;
                const int j = idx / CH, rl = idx - j * CH;
                if (idx < B * CH) P[(size_t)j * ldp + rl] = v[q];
            }
        }
    }
    __syncthreads();

    // tasks of the products with a panel slice: (row tile, pair of column tiles), round robin
    const int ntask = (CH / 16) * NP;
    bool tiny = false;
    unsigned nbar = 0;
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
        const int tid = cq_fresh(threadIdx.x), lane = tid & 63, lr = lane & 15, lk = lane >> 4;
        // ---- Gram matrix of the panel: partials, then fixed-order slice sums
        cq_gram<B>(P, ldp, CH, a.part + (size_t)g * NE, wave, lane);
        if (!grid_barrier_wt(a.counter, (unsigned)a.G * ++nbar, a.err)) return;
        {
            const int S = (NE + a.G - 1) / a.G;
            const int e0 = g * S, ne = max(0, min(NE, e0 + S) - e0);
            int tpe = 1; // threads per entry (power of two)
            while (tpe < 64 && tpe * 2 * max(ne, 1) <= kCQThreads) tpe *= 2;
            const int per_round = kCQThreads / tpe;
            for (int base = 0; base < ne; base += per_round) {
                const int el = base + tid / tpe, pt = tid % tpe;
                double s = 0.0;
                if (el < ne) {
                    const double *src = a.part + e0 + el;
                    for (int g0 = pt; g0 < a.G; g0 += tpe * 16) {
                        double v[16];
#pragma unroll
                        for (int u = 0; u < 16; ++u) {
                            const int gg = g0 + u * tpe;
                            v[u] = (gg < a.G) ? ld_wt(src + (size_t)gg * NE) : 0.0;
                        }
#pragma unroll
                        for (int u = 0; u < 16; ++u) s += v[u];
                    }
                }
                for (int d = tpe / 2; d > 0; d /= 2) s += __shfl_xor(s, d, 64);
                if (el < ne && pt == 0) st_wt(a.gsum + e0 + el, s);
            }
        }
        if (!grid_barrier_wt(a.counter, (unsigned)a.G * ++nbar, a.err)) return;

        {
            double v[(NE + kCQThreads - 1) / kCQThreads];
#pragma unroll
            for (int q = 0; q < (NE + kCQThreads - 1) / kCQThreads; ++q) {
                const int idx = q * kCQThreads + tid;
                v[q] = idx < NE ? ld_wt(a.gsum + idx) : 0.0;
            }
            auto place = [&](bool second) {
#pragma unroll
                for (int q = 0; q < (NE + kCQThreads - 1) / kCQThreads; ++q) {
                    const int idx = q * kCQThreads + tid;
                    if (idx >= NE) continue;
                    int I, J;
                    cq_tile(idx >> 8, I, J);
                    const int i = 16 * I + 4 * ((idx >> 6) & 3) + ((idx & 63) >> 4), j = 16 * J + (idx & 15);
                    if (!second) { // G
                        MA[i + j * LD] = v[q];
                        if (I != J) MA[j + i * LD] = v[q];
                        continue;
                    }
                    // second pass: G = I + E with E tiny (the usual case): R_2 = I + F, R_2^-1 = I - F,
                    // F = up(E) = strict upper of E + diag(E) / 2. |E| <= 1e-10 entrywise: up(E)^T
                    // up(E) and F^2 have entries below b 1e-20, under half an ulp of the diagonal
                    const double e = v[q] - (i == j ? 1.0 : 0.0);
                    if (!(fabs(e) <= 1e-10)) s_bad[1] = 1;
                    MA[i + j * LD] = I != J || i > j ? 0.0 : (i < j ? e : 0.5 * e);
                    if (I != J) MA[j + i * LD] = e;
                }
                __syncthreads();
            };
            place(pass == 1);
            tiny = pass == 1 && s_bad[1] == 0;
            if (pass == 1 && !tiny) {
                __syncthreads();
                place(false);
            }
        }
        if (tiny) {
            // P <- P - P F, transposed (16 rows of one column in 16 lanes)
            for (int t0 = 0; t0 < ntask; t0 += kCQWaves) {
                const int t = t0 + wave, I = t / NP, pr = t % NP;
                cq_v4 acc[2];
                if (t < ntask) {
                    const int Jt[2] = {pr, NTB - 1 - pr};
#pragma unroll
                    for (int c = 0; c < (NTB > 1 ? 2 : 1); ++c)
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            acc[c][u] = P[(size_t)(16 * Jt[c] + 4 * u + lk) * ldp + 16 * I + lr];
                    for (int k0 = 0; k0 < 16 * (Jt[1] + 1); k0 += 4) {
                        const double x = P[(size_t)(k0 + lk) * ldp + 16 * I + lr];
#pragma unroll
                        for (int c = 0; c < (NTB > 1 ? 2 : 1); ++c)
                            if (k0 < 16 * (Jt[c] + 1))
                                acc[c] = cq_mma(-MA[k0 + lk + (16 * Jt[c] + lr) * LD], x, acc[c]);
                    }
                }
                __syncthreads();
                if (t < ntask) {
                    const int Jt[2] = {pr, NTB - 1 - pr};
#pragma unroll
                    for (int c = 0; c < (NTB > 1 ? 2 : 1); ++c)
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            P[(size_t)(16 * Jt[c] + 4 * u + lk) * ldp + 16 * I + lr] = acc[c][u];
                }
            }
            __syncthreads();
        } else if (!cq_chol<B, NSET>(P, ldp, CH, MA, MC, g == 0 ? (pass == 0 ? MB : MA) : nullptr, pass == 0 ? 1e-10 : 1e-3,
                                     s_bad, wave, lane)) {
            if (g == 0 && tid == 0) *a.gate = 1;
            return; // every workgroup takes the same decision
        }
    }

    // with b rows the last column has nothing below its pivot, where LAPACK's H is the identity (tau
    // = 0) and the one found here only changes the sign of R's last entry: leave it out
    const bool square = a.rows == B;
    if (g == 0) {
        cq_lu<B>(P, ldp, MC, MC, a.bc, sv, wave, lane);
        if (tid == 0) *a.gate = 0;
        vm_drain();
        __syncthreads();
        if (tid == 0) __hip_atomic_fetch_add(a.counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // R = R_2 R_1, or R_1 + F R_1, into MA
        cq_v4 acc[(NT + kCQWaves - 1) / kCQWaves];
#pragma unroll
        for (int q = 0; q < (NT + kCQWaves - 1) / kCQWaves; ++q) {
            const int t = wave + kCQWaves * q;
            if (t >= NT) continue;
            int I, J;
            cq_tile(t, J, I); // upper tiles
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[q][u] = tiny ? MB[16 * I + 4 * u + lk + (16 * J + lr) * LD] : 0.0;
            acc[q] = cq_upper_mm<B>(MA, MB, I, J, acc[q], lane);
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < (NT + kCQWaves - 1) / kCQWaves; ++q) {
            const int t = wave + kCQWaves * q;
            if (t >= NT) continue;
            int I, J;
            cq_tile(t, J, I);
#pragma unroll
            for (int u = 0; u < 4; ++u) MA[16 * I + 4 * u + lk + (16 * J + lr) * LD] = acc[q][u];
        }
        __syncthreads();
        // panel rows 0..b-1 of A: R_house = S R on and above the diagonal, L below
        for (int idx = tid; idx < BB; idx += kCQThreads) {
            const int r = idx % B, j = idx / B;
            const double l = MC[r + j * LD], s = (square && r == B - 1) ? -sv[r] : sv[r];
            a.A[(i64)r + (i64)j * a.lda] = (T)((j >= r) ? s * MA[r + j * LD] : l);
            if (a.Y) a.Y[(i64)r + (i64)j * a.ldy] = (T)((j < r) ? l : (j == r ? 1.0 : 0.0));
        }
        __syncthreads();
    } else {
        // workgroup 0's arrival alone
        if (!grid_wait_wt(a.counter, (unsigned)a.G * nbar + 1u, a.err)) return;
    }
    {
        // U^-1 and Mw: rounds of 2 x LB loads per thread, all issued before their LDS stores
        constexpr int LB = (BB + kCQThreads - 1) / kCQThreads;
        double u[LB], t[LB];
#pragma unroll
        for (int q = 0; q < LB; ++q) {
            const int idx = q * kCQThreads + tid;
            u[q] = (idx < BB) ? ld_wt(a.bc + idx) : 0.0;
            t[q] = (idx < BB) ? ld_wt(a.bc + BB + idx) : 0.0;
        }
#pragma unroll
        for (int q = 0; q < LB; ++q) {
            const int idx = q * kCQThreads + tid;
            const int i = idx % B, j = idx / B;
            if (idx < BB) {
                MA[i + j * LD] = u[q];
                MB[j + i * LD] = t[q];
            }
        }
    }
    __syncthreads();
    // W = Y T = (Q - [S; 0]) Mw (T = -U S L^-T gives Q_2 U^-1 T = -Q_2 S L^-T below the first b
    // rows, and L T = -(Q_1 - S) S L^-T on them), and Y = Q U^-1 for the rows below the
    // first b (workgroup 0 wrote its top rows, L), also the reflector tails in A
    const int ylo = (g == 0) ? B : 0;
    for (int t = wave; t < ntask; t += kCQWaves) {
        const int I = t / NP, pr = t % NP;
        const int Jt[2] = {pr, NTB - 1 - pr};
        cq_v4 w[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, y[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
        for (int k0 = 0; k0 < 16 * (Jt[1] + 1); k0 += 4) {
            const double x = P[(size_t)(k0 + lk) * ldp + 16 * I + lr];
#pragma unroll
            for (int c = 0; c < (NTB > 1 ? 2 : 1); ++c)
                if (k0 < 16 * (Jt[c] + 1)) {
                    const int at = k0 + lk + (16 * Jt[c] + lr) * LD;
                    if (a.W) w[c] = cq_mma(MB[at], x, w[c]);
                    if (16 * I >= ylo) y[c] = cq_mma(MA[at], x, y[c]);
                }
        }
        const int rl = 16 * I + lr;
        const i64 r = r0g + rl;
        if (rl < chl)
#pragma unroll
            for (int c = 0; c < (NTB > 1 ? 2 : 1); ++c)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const i64 j = 16 * Jt[c] + 4 * u + lk;
                    if (a.W) a.W[r + j * a.ldw] = square && j == B - 1 ? T(0) : (T)w[c][u];
                    if (16 * I >= ylo) {
                        a.A[r + j * a.lda] = (T)y[c][u];
                        if (a.Y) a.Y[r + j * a.ldy] = (T)y[c][u];
                    }
                }
    }
    if (g == 0) {
        // T = U Mw (upper triangular), and tau = diag(T)
        for (int t = wave; t < NTB * NTB; t += kCQWaves) {
            const int I = t / NTB, J = t % NTB;
            cq_v4 acc = {0, 0, 0, 0};
            if (I <= J) acc = cq_upper_mm<B>(MC, MB, I, J, acc, lane);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = 16 * I + 4 * u + lk, j = 16 * J + lr;
                const T t_ij = square && j == B - 1 ? T(0) : (T)acc[u];
                a.Tm[i + (size_t)j * B] = t_ij;
                if (i == j) a.tau[j] = t_ij;
            }
        }
    }
}

// sets of 64 lanes that hold the rows of [G; P]
constexpr int cq_sets(int b, int CH) { return (b + CH + 63) / 64; }

template <int B> size_t cq_lds_bytes(int CH) {
    const size_t groups = std::max((size_t)B * (B + 2), (size_t)768 * cq_sets(B, CH));
    return sizeof(double) * ((size_t)B * cq_ldp(CH) + 2 * (size_t)B * (B + 2) + groups + B + 1);
}

__global__ void zero_u32_kernel(unsigned *p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

template <typename T> size_t pq_lds_bytes(int b, int CH) {
    return sizeof(double) * ((size_t)b * (b + 1) + 2 * b + b + b + 512 + 2 * (size_t)CH + b) +
           sizeof(T) * (size_t)b * (CH + 1);
}

} // namespace

template <typename T> int panel_qr_chunk(int b) {
    // largest multiple of 64 rows whose panel slice fits in 160 KB of LDS
    const size_t budget = 160 * 1024;
    int ch = 64;
    while (ch + 64 <= 1024 && pq_lds_bytes<T>(b, ch + 64) <= budget) ch += 64;
    return ch;
}

size_t panel_qr_scratch_bytes(int n, int b) {
    // gate word; Householder: partials [2][G][2b] + pivot [2][b] doubles, G <= n / 64 + 2;
    // CholQR: partial Gram matrices [G][b*b] + sums [b*b] + broadcast [2*b*b], G <= n / 64 + 1
    const size_t G = (size_t)n / 64 + 2;
    const size_t hh = sizeof(double) * (2 * G * 2 * b + 2 * b);
    const size_t cq = sizeof(double) * ((G + 3) * (size_t)b * b);
    return kPQGateBytes + std::max(hh, cq) + 256;
}

namespace {

// CholQR2 launch if the panel qualifies: b in {16, 32, 64}, at least b rows, and rows spread one
// workgroup per CU with at most kCQMaxCH rows each.
template <typename T, int B>
int launch_cholqr(hipStream_t s, T *A, i64 lda, T *Y, i64 ldy, T *W, i64 ldw, T *Tm, T *tau, int rows,
                  void *scratch, size_t scratch_bytes, unsigned *counter, int *err, bool *launched) {
    *launched = false;
    const int ncu = device_cu_count();
    const int CH = std::max(64, (int)round_up(ceil_div(rows, ncu), 16));
    if (CH > kCQMaxCH) return CUEV_STATUS_SUCCESS;
    const int G = (int)ceil_div(rows, CH);
    // [G; P] takes two sets of 64 lanes, for b = 64 and more than 64 rows three
    static_assert(cq_sets(16, kCQMaxCH) <= 2 && cq_sets(32, kCQMaxCH) <= 2 && cq_sets(64, kCQMaxCH) <= 3, "");
    const auto kernel = cq_sets(B, CH) <= 2 ? panel_cholqr_kernel<T, B, 2> : panel_cholqr_kernel<T, B, B == 64 ? 3 : 2>;
    const size_t lds = cq_lds_bytes<B>(CH);
    CUEV_HIP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int per_cu = 0;
    CUEV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kCQThreads, lds));
    if (G > per_cu * ncu) return CUEV_STATUS_SUCCESS;
    const size_t need = kPQGateBytes + sizeof(double) * ((size_t)(G + 3) * B * B);
    if (need > scratch_bytes) return CUEV_STATUS_SUCCESS;
    CQArgs<T> a;
    a.A = A;
    a.lda = lda;
    a.Y = Y;
    a.ldy = ldy;
    a.W = W;
    a.ldw = ldw;
    a.Tm = Tm;
    a.tau = tau;
    a.rows = rows;
    a.CH = CH;
    a.G = G;
    a.gate = static_cast<int *>(scratch);
    a.part = reinterpret_cast<double *>(static_cast<unsigned char *>(scratch) + kPQGateBytes);
    a.gsum = a.part + (size_t)G * B * B;
    a.bc = a.gsum + B * B;
    a.counter = counter;
    a.reset = counter + 1;
    a.err = err;
    hipLaunchKernelGGL(kernel, dim3(G), dim3(kCQThreads), lds, s, a);
    CUEV_LAUNCH_CHECK();
    *launched = true;
    return CUEV_STATUS_SUCCESS;
}

} // namespace

template <typename T>
int panel_qr(hipStream_t s, T *A, i64 lda, T *Y, i64 ldy, T *W, i64 ldw, T *Tm, T *tau, int rows,
             int b, void *scratch, size_t scratch_bytes, unsigned *counter, int *err) {
    if (rows < 1 || b < 1 || b > 64)
        CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "panel_qr: rows=%d b=%d", rows, b);
    if (scratch_bytes < kPQGateBytes)
        CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "panel_qr: scratch too small");
    // counter[0]: CholQR barriers, counter[1]: Householder barriers. Both are zero
    // when a panel starts: the workspace starts them at zero, each kernel zeroes the
    // other's counter when it starts (the CholQR kernel the Householder kernel's that
    // follows it, the Householder kernel, always launched, the CholQR counter for the
    // next panel), and without a CholQR launch counter[1] is zeroed here.
    bool cq = false;
    if (rows >= b) {
        if (b == 64)
            CUEV_TRY((launch_cholqr<T, 64>(s, A, lda, Y, ldy, W, ldw, Tm, tau, rows, scratch, scratch_bytes,
                                           counter, err, &cq)));
        else if (b == 32)
            CUEV_TRY((launch_cholqr<T, 32>(s, A, lda, Y, ldy, W, ldw, Tm, tau, rows, scratch, scratch_bytes,
                                           counter, err, &cq)));
        else if (b == 16)
            CUEV_TRY((launch_cholqr<T, 16>(s, A, lda, Y, ldy, W, ldw, Tm, tau, rows, scratch, scratch_bytes,
                                           counter, err, &cq)));
    }
    const int CH = panel_qr_chunk<T>(b);
    const int G = (int)ceil_div(rows, CH);
    const size_t lds = pq_lds_bytes<T>(b, CH);
    static_assert(kPQThreads == 256, "");
    CUEV_HIP(hipFuncSetAttribute((const void *)panel_qr_kernel<T>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int per_cu = 0;
    CUEV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, panel_qr_kernel<T>, kPQThreads,
                                                          lds));
    const int resident = per_cu * device_cu_count();
    if (G > resident)
        CUEV_FAIL(CUEV_STATUS_NOT_SUPPORTED,
                  "panel_qr: %d rows need %d co-resident workgroups, device holds %d", rows, G,
                  resident);
    const size_t need = kPQGateBytes + sizeof(double) * ((size_t)2 * G * 2 * b + 2 * b);
    if (need > scratch_bytes)
        CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "panel_qr: scratch too small (%zu < %zu)",
                  scratch_bytes, need);
    PQArgs<T> a;
    a.A = A;
    a.lda = lda;
    a.Y = Y;
    a.ldy = ldy;
    a.W = W;
    a.ldw = ldw;
    a.Tm = Tm;
    a.tau = tau;
    a.rows = rows;
    a.b = b;
    a.CH = CH;
    a.G = G;
    a.part = reinterpret_cast<double *>(static_cast<unsigned char *>(scratch) + kPQGateBytes);
    a.pivot = a.part + (size_t)2 * G * 2 * b;
    a.gate = cq ? static_cast<const int *>(scratch) : nullptr;
    a.counter = counter + 1;
    a.reset = counter;
    a.err = err;
    if (!cq) {
        hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(64), 0, s, counter + 1, 1);
        CUEV_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(panel_qr_kernel<T>, dim3(G), dim3(kPQThreads), lds, s, a);
    CUEV_LAUNCH_CHECK();
    return CUEV_STATUS_SUCCESS;
}

template int panel_qr_chunk<float>(int);
template int panel_qr_chunk<double>(int);
template int panel_qr<float>(hipStream_t, float *, i64, float *, i64, float *, i64, float *,
                             float *, int, int, void *, size_t, unsigned *, int *);
template int panel_qr<double>(hipStream_t, double *, i64, double *, i64, double *, i64, double *,
                              double *, int, int, void *, size_t, unsigned *, int *);

} // namespace cuev
