// bulge.hip — band -> tridiagonal reduction (bulge chasing) and (d, e) extraction.
//
// Algorithm (reference: src/cuda/bulge.cu:64-224, Algorithm 2 of Wang et al.):
// sweep s = 0..n-3 eliminates column s below its subdiagonal with a Householder
// reflector on rows [s+1, s+b], then chases the bulge this creates down the band:
// hop h >= 1 eliminates the bulge column cq = s+1+(h-1)b on rows
// [cq+b, cq+2b-1]. Each hop is the similarity A <- H A H with H = I - 2 w w^T,
// ||w|| = 1, applied as A <- A - w y^T - y w^T, p = 2 A w, kappa = w^T p,
// y = p - kappa w. The reflector of hop h of sweep s occupies rows
// [s+1+hb, min(s+(h+1)b, n-1)] and is stored for the back-transform.
//
// Two kernels: the resident form (bc_chase_resident_kernel, described there) wherever its
// workgroups, one per hop of the first sweep, fit on the GPU at once, and the windowed
// form below for the larger n (b = 64 in FP64: n > 49152), where it still is the only one
// (and, asked for by cuev_handle_set_chase, at any n).
//
// Design of the windowed form (not the reference's):
//  * Reflector convention: if the vector below the pivot is exactly zero the
//    hop is the identity (w = 0), as LAPACK's dlarfg does; the reference's
//    normalised reflector would flip the sign of the pivot instead.
//  * Each hop works on its window in LDS: the packed band columns [cq, r1]
//    (all 2b stored rows) hold every entry the hop reads or writes. The window
//    slides with the sweep: consecutive hops share b columns, so a hop loads
//    only the b new columns and writes back only the b columns the sweep has
//    finished with (a ring of 2b column slots). The Householder vector is formed
//    by wave 0 alone (L <= 64 = one wave64), with FP64 norms.
//  * Dependency: hop (s, cq, r1) touches packed columns [cq, r1] only, and the
//    previous sweep's hops touch columns [cq'', r1''] with cq'' increasing. Hop h of
//    sweep s reads columns up to r1 = r0 + b - 1, which sweep s-1 last changes in its
//    hop h+1 (the rank-2 update of that hop's R1 columns and of its column r0'' = r1,
//    and the elimination of column r1 by its hop h+2's reflector). So a hop publishes
//    progress prog[s] = r0 early: after R1 and column r0 are updated, the next hop's
//    reflector is formed from column r0, and R1's columns and column r0 are written
//    back; the rest of its rank-2 update (R2 and R3 beyond column r0) then runs beside
//    the next sweep's hop, which waits for prog[s-1] >= r1. A hop's reflector is thus
//    formed in the hop before, so a hop runs: wait for sweep s-1, load the b new
//    columns, p and kappa, R1 and column r0, the next reflector, write-back and
//    progress, the rest of R2 and R3. The next sweep's first hop waits for columns up
//    to s + 1 + b (published by hop 1), so hop 0 publishes nothing. The sweep-to-sweep
//    lag is about one hop plus the part of the next hop before its publish; the
//    reference waits for a margin of 3b columns (bulge.cu:193-199).
//  * Hand-offs use agent-scope (write-through) band accesses and flags, with no L2
//    write-back or invalidate (see ld_agent / st_agent below); every wait is bounded,
//    and the grid never exceeds the number of co-resident workgroups, so the lowest
//    unfinished sweep can always proceed.
//  * U is stored shifted: U[(r - s - 1) + s*ldu] holds row r of sweep s's
//    reflectors, so the back-transform reads aligned, contiguous segments.
#include "bulge.hpp"

#include <algorithm>

#include "profile.hpp"
#include "util.hpp"
#include "wave.hpp"

namespace cuev {
namespace {

constexpr int kBCThreads = 512; // 8 waves: two per SIMD, so LDS latency overlaps
constexpr int kDone = 0x3fffffff; // prog value of a finished sweep
constexpr int kMaxPhases = 8;

// Sweep schedule in phases: sweeps [s0[p], s0[p+1]) go round-robin to workgroups
// 0 .. g[p]-1 (g non-increasing). A sweep of h hops is active for ~h hop times and a
// new one starts every ~2 hop times, so fewer sweeps are in flight as they shorten;
// a workgroup with no sweep left in the later phases exits and frees its CU for the
// back-transform products running beside the chase.
struct ChasePhases {
    int np;
    int s0[kMaxPhases + 1];
    int g[kMaxPhases];
};

// Band traffic between workgroups. Every global load and store of the packed band is
// an agent-scope relaxed atomic access: on gfx950 these carry the sc1 bit, so a store
// is written through to the device-coherent level (past the XCD-private L2) and a
// load reads from it. A hand-off then needs no L2 write-back and no L2 invalidate:
//   producer: band stores (sc1), s_waitcnt vmcnt(0) in every wave (the stores have
//             completed at agent scope), workgroup barrier, one flag store (sc1);
//   consumer: one thread polls the flag (sc1 loads), workgroup barrier, band loads
//             (sc1), issued only after the flag was seen.
// The reflectors (U) are read only by later kernels and use plain stores.
template <typename T> __device__ __forceinline__ T ld_agent(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T> __device__ __forceinline__ void st_agent(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// progress flag store after wg_publish_fence (every wave's band stores complete)
__device__ __forceinline__ void flag_store_agent(int *p, int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T, int B>
__global__ __launch_bounds__(kBCThreads) void bc_chase_kernel(T *Bp, T *U, i64 ldu, int n,
                                                              int *prog, int *err, const ChasePhases ph) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    constexpr int b = B;
    constexpr int NEW_PER_THREAD = 2 * B * B / kBCThreads; // b new columns of 2b rows per hop
    const int ldb = 2 * b;       // packed band leading dimension
    // LDS leading dimension of a window column: odd, so that reading along a row
    // (stride WLD doubles across lanes) spreads over the banks
    const int WLD = 2 * b + 1;
    const int NSLOT = 2 * b;     // ring of window columns: matrix column j lives in slot j % NSLOT
    constexpr int NW = kBCThreads / 64;    // waves per workgroup
    // k segments of the p product: (row, segment) pairs cover the workgroup's threads
    constexpr int NSEG = (kBCThreads / (3 * B)) < 1 ? 1 : (kBCThreads / (3 * B));
    T *win = reinterpret_cast<T *>(smem_raw);          // [NSLOT][WLD]
    T *sw = win + (size_t)NSLOT * WLD;                 // [2][b] reflectors: this hop's, the next hop's
    T *sp = sw + 2 * b;                                // [3b]  p
    T *spart = sp + 3 * b;                             // [NSEG][3b] partial sums of p
    __shared__ T sred[NW];
    __shared__ double s_beta[2];
    __shared__ int s_go;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // window element A(i, j) (i >= j, both in the current window)
    auto W_ = [&](int i, int j) -> T & { return win[(j & (NSLOT - 1)) * WLD + (i - j)]; };
    // symmetric read A(i, k) = A(max, min): the address by min/max, without a branch
    auto Wsym = [&](int i, int k) -> T {
        const int hi_ = max(i, k), lo_ = min(i, k);
        return win[(lo_ & (NSLOT - 1)) * WLD + (hi_ - lo_)];
    };
    // copy packed columns [c0, c1] between global memory and their ring slots: in
    // rounds of FIRST_PER_THREAD loads per thread, all issued before any LDS store (one
    // round trip per round; a sweep's first window of b + 1 columns takes one)
    constexpr int FIRST_PER_THREAD = (2 * B * (B + 1) + kBCThreads - 1) / kBCThreads;
    auto load_cols = [&](int c0, int c1) {
        if (c1 < c0) return;
        const int cnt = (c1 - c0 + 1) * ldb;
        const T *src = Bp + (i64)c0 * ldb;
        for (int base = 0; base < cnt; base += FIRST_PER_THREAD * kBCThreads) {
            T v[FIRST_PER_THREAD];
#pragma unroll
            for (int u = 0; u < FIRST_PER_THREAD; ++u) {
                const int idx = base + tid + u * kBCThreads;
                v[u] = (idx < cnt) ? ld_agent(src + idx) : T(0);
            }
#pragma unroll
            for (int u = 0; u < FIRST_PER_THREAD; ++u) {
                const int idx = base + tid + u * kBCThreads;
                if (idx < cnt) {
                    const int jj = idx / ldb, d = idx - jj * ldb;
                    win[((c0 + jj) & (NSLOT - 1)) * WLD + d] = v[u];
                }
            }
        }
    };
    // exactly b new columns: all loads issued before any LDS store (one round trip)
    auto load_b_cols = [&](int c0) {
        const T *src = Bp + (i64)c0 * ldb;
        T v[NEW_PER_THREAD];
#pragma unroll
        for (int u = 0; u < NEW_PER_THREAD; ++u) v[u] = ld_agent(src + tid + u * kBCThreads);
#pragma unroll
        for (int u = 0; u < NEW_PER_THREAD; ++u) {
            const int idx = tid + u * kBCThreads;
            const int jj = idx / ldb, d = idx - jj * ldb;
            win[((c0 + jj) & (NSLOT - 1)) * WLD + d] = v[u];
        }
    };
    auto store_cols = [&](int c0, int c1) {
        if (c1 < c0) return;
        const int cnt = (c1 - c0 + 1) * ldb;
        T *dst = Bp + (i64)c0 * ldb;
        if (cnt <= NEW_PER_THREAD * kBCThreads) {
            // up to b columns (every hop): all LDS reads before the stores
            T v[NEW_PER_THREAD];
#pragma unroll
            for (int u = 0; u < NEW_PER_THREAD; ++u) {
                const int idx = tid + u * kBCThreads;
                const int jj = idx / ldb, d = idx - jj * ldb;
                v[u] = win[((c0 + jj) & (NSLOT - 1)) * WLD + d];
            }
#pragma unroll
            for (int u = 0; u < NEW_PER_THREAD; ++u) {
                const int idx = tid + u * kBCThreads;
                if (idx < cnt) st_agent(dst + idx, v[u]);
            }
            return;
        }
        for (int idx = tid; idx < cnt; idx += kBCThreads) {
            const int jj = idx / ldb, d = idx - jj * ldb;
            st_agent(dst + idx, win[((c0 + jj) & (NSLOT - 1)) * WLD + d]);
        }
    };

    // Householder vector of x = A[r0_ : r0_ + L_ - 1, c_] (column c_ of the window),
    // by wave 0 alone: w into wd, beta into *bd
    auto householder = [&](int r0_, int c_, int L_, T *wd, double *bd) {
        const double x = (lane < L_) ? (double)W_(r0_ + lane, c_) : 0.0;
        const double alpha = __shfl(x, 0, 64);
        const double tail = wave_sum((lane >= 1) ? x * x : 0.0);
        double wv = 0.0, beta = alpha;
        if (tail != 0.0) {
            const double nrm = sqrt(alpha * alpha + tail);
            beta = (alpha >= 0.0) ? -nrm : nrm;
            const double v0 = alpha - beta;
            const double inv = 1.0 / sqrt(v0 * v0 + tail);
            wv = ((lane == 0) ? v0 : x) * inv;
        }
        if (lane < L_) wd[lane] = (T)wv;
        if (lane == 0) *bd = beta;
    };
    // column c_ is final: write it back, the eliminated entries [o_, o_ + L_) as beta e_0
    // (skip_pivot: all but entry o_)
    auto writeback = [&](int c_, int o_, int L_, double beta_, bool skip_pivot = false) {
        T *dst = Bp + (i64)c_ * ldb;
        const T *srcw = win + (size_t)(c_ & (NSLOT - 1)) * WLD;
        for (int d = tid; d < ldb; d += kBCThreads) {
            if (skip_pivot && d == o_) continue;
            st_agent(dst + d, (d == o_) ? (T)beta_ : ((d > o_ && d < o_ + L_) ? T(0) : srcw[d]));
        }
    };

    // this workgroup's sweeps in increasing order: the next one of the current phase,
    // else its first one in a later phase that still uses it (none left: n)
    int phase = 0;
    auto settle = [&](int s_) {
        while (s_ >= ph.s0[phase + 1]) {
            if (++phase >= ph.np) return n;
            s_ = ((int)blockIdx.x < ph.g[phase]) ? ph.s0[phase] + (int)blockIdx.x : ph.s0[phase + 1];
        }
        return s_;
    };
    int s = settle(((int)blockIdx.x < ph.g[0]) ? ph.s0[0] + (int)blockIdx.x : ph.s0[1]);
    for (; s < n - 2;) {
        int held_lo = 0, held_hi = -1; // window columns currently held in LDS
        T *wc = sw, *wn = sw + b;      // this hop's reflector, the next hop's
        double *bc = &s_beta[0], *bn = &s_beta[1];
        for (int h = 0;; ++h) {
            const int cq = (h == 0) ? s : s + 1 + (h - 1) * b;
            const int r0 = (h == 0) ? s + 1 : cq + b;
            if (r0 > n - 1) break;
            const int r1 = min(r0 + b - 1, n - 1);
            const int L = r1 - r0 + 1;
            if (L < 2) {
                // nothing below the pivot: identity reflector (record it for the back-transform)
                if (tid == 0) U[(i64)(r0 - s - 1) + (i64)s * ldu] = T(0);
                break;
            }
            const int hi = min(n - 1, r1 + b);  // last row touched

            // ---- wait for sweep s-1 to be done with columns <= r1 (acquire), then bring
            // the window [cq, r1] into LDS: columns already held stay, the rest come from
            // global memory (b columns per hop after the first)
            auto wait_and_load = [&]() -> bool {
                if (s > 0) {
                    if (tid == 0) {
                        long long it = 0;
                        int go = 1;
                        while (flag_load_relaxed(prog + (s - 1)) < r1) {
                            __builtin_amdgcn_s_sleep(1);
                            if (++it > kSpinLimit) {
                                __hip_atomic_store(err, (int)DEV_WATCHDOG, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
                                go = 0;
                                break;
                            }
                        }
                        s_go = go;
                    }
                    __syncthreads();
                    if (!s_go) return false;
                }
                if (held_hi < held_lo) load_cols(cq, r1);
                else if (r1 - held_hi == b) load_b_cols(held_hi + 1);
                else load_cols(max(cq, held_hi + 1), r1);
                held_lo = cq;
                held_hi = r1;
                __syncthreads();
                return true;
            };
            if (!wait_and_load()) return;
            if (h == 0) {
                // the sweep's first reflector, on column s; column s is then final (rows
                // above r0 untouched by this sweep, beta e_0 below): write it back and
                // publish progress s. Later hops find their reflector formed and their
                // column cq written back and published by the hop before.
                // No progress is published for column s (or s + 1 below): the next
                // sweep first waits for columns up to s + 1 + b, published by hop 1,
                // whose fence also covers these stores.
                if (wave == 0) householder(r0, cq, L, wc, bc);
                __syncthreads();
                writeback(cq, r0 - cq, L, *bc);
            }

            // ---- p_t = 2 sum_k A(cq+t, r0+k) w_k, t < nrow. Thread = (row t, k segment);
            // each thread walks its segment starting at a row-dependent offset, so the
            // lanes of a wave (consecutive rows) hit distinct LDS banks both for
            // A(i, k), i >= k (column k, stride 1 across lanes) and for A(k, i), i < k
            // (column i: stride WLD - 1 across lanes, which without the rotation puts
            // every lane on one bank)
            const int nrow = hi - cq + 1; // <= 3b
            const int o = r0 - cq;
            // b = 64: rows in six waves of 32 lanes, the two k segments of a row in the
            // two halves of a wave, so p_t is completed with one lane exchange and
            // kappa's partial sums come out of the same phase (one barrier)
            constexpr bool kWaveSeg = 3 * B == 192 && NSEG == 2 && kBCThreads >= 384;
            {
                const int t = kWaveSeg ? wave * 32 + (lane & 31) : tid % (3 * B);
                const int seg = kWaveSeg ? (wave < 6 ? lane >> 5 : NSEG) : tid / (3 * B);
                const int SL = (L + NSEG - 1) / NSEG;
                const int kb = seg * SL, ke = min(L, kb + SL), len = ke - kb;
                T acc = T(0);
                constexpr int FL = B / NSEG; // segment length of a full hop
                if (seg < NSEG && t < nrow && len > 0) {
                    const int i = cq + t;
                    if (B % NSEG == 0 && (FL & (FL - 1)) == 0 && len == FL) {
                        // full segment: unrolled with four partial sums, so the LDS
                        // reads of consecutive steps overlap (same rotation as below)
                        T a4[4] = {T(0), T(0), T(0), T(0)};
#pragma unroll 8
                        for (int j = 0; j < FL; ++j) {
                            const int q = kb + ((t + j) & (FL - 1));
                            const int k = r0 + q;
                            a4[j & 3] += Wsym(i, k) * wc[q];
                        }
                        acc = (a4[0] + a4[1]) + (a4[2] + a4[3]);
                    } else {
                        int qq = t % len;
                        for (int j = 0; j < len; ++j) {
                            const int q = kb + qq;
                            const int k = r0 + q;
                            const T a = Wsym(i, k);
                            acc += a * wc[q];
                            qq = (qq + 1 == len) ? 0 : qq + 1;
                        }
                    }
                }
                if (kWaveSeg) {
                    // ---- p (segment 0 + segment 1, as below), and kappa = w^T p over
                    // the reflector's rows [o, o + L)
                    const T other = __shfl_xor(acc, 32, 64);
                    T kv = T(0);
                    if (seg == 0 && t < nrow) {
                        const T pv = T(2) * (acc + other);
                        sp[t] = pv;
                        if (t >= o && t < o + L) kv = pv * wc[t - o];
                    }
                    kv = wave_sum(kv);
                    if (lane == 0) sred[wave] = kv;
                } else if (seg < NSEG && t < 3 * B) {
                    spart[seg * (3 * B) + t] = acc;
                }
            }
            __syncthreads();
            if (!kWaveSeg) {
                // ---- p, and kappa = w^T p over the reflector's rows [o, o + L)
                T kv = T(0);
                if (tid < nrow) {
                    T ps = T(0);
#pragma unroll
                    for (int v = 0; v < NSEG; ++v) ps += spart[v * (3 * B) + tid];
                    const T pv = T(2) * ps;
                    sp[tid] = pv;
                    if (tid >= o && tid < o + L) kv = pv * wc[tid - o];
                }
                kv = wave_sum(kv);
                if (lane == 0) sred[wave] = kv;
                __syncthreads();
            }

            // ---- rank-2 update A -= w y^T + y w^T with y = p - kappa w, on the three
            // regions of the window where w_i or w_j is non-zero:
            //   R1: rows r0+a (a < L)      x columns cq+c, 0 <= c < o  (w_j = 0); c = 0 is the
            //       eliminated column, set to its exact value beta e_0
            //   R2: rows r0+a (a < L)      x columns r0+c, c <= a     (both non-zero)
            //   R3: rows r1+1+a (a < m3)   x columns r0+c, c < L      (w_i = 0)
            // thread = (row a, column group cg); the column value is a broadcast read.
            // part 1: R1, and column c = 0 of R2 and R3 (column r0, the next hop's
            // reflector column); part 2: the rest of R2 and R3; part 3: all of it
            auto rank2 = [&](int part) {
                const bool dR1 = part != 2, dC0 = part != 2, dRest = part != 1;
                T kap = T(0);
#pragma unroll
                for (int v = 0; v < NW; ++v) kap += sred[v];
                constexpr int NG = kBCThreads / B;
                const int a = tid % B, cg = tid / B;
                const int m3 = hi - r1;
                const T wa = (a < L) ? wc[a] : T(0);
                const T ya = (a < L) ? sp[o + a] - kap * wa : T(0);
                const T y3 = (a < m3) ? sp[o + L + a] : T(0);
                const T bet = (T)*bc;
                constexpr bool kFull = B >= NG && B % NG == 0; // whole columns per thread group
                // R1 has o < B columns in a sweep's first hop (o = 1): it then goes through
                // the general loop, and R2 and R3 through the fast path below
                const bool full23 = kFull && L == B && m3 == B;
                const bool split1 = full23 && o != B;
                if (split1 && dR1 && a < L)
                    for (int cc = cg; cc < o; cc += NG) {
                        T &e = W_(r0 + a, cq + cc);
                        if (cc == 0) e = (a == 0) ? bet : T(0);
                        else e -= wa * sp[cc];
                    }
                if (full23) {
                    const bool fR1 = dR1 && !split1;
                    // full hop (every thread in all three regions, each element read and
                    // written by its own thread only): every LDS read before any write,
                    // so the round trips overlap; same arithmetic as the general path
                    constexpr int NU = kFull ? B / NG : 1;
                    T e1[NU], e2[NU], e3[NU], p1[NU], wcv[NU], pc[NU];
#pragma unroll
                    for (int u = 0; u < NU; ++u) {
                        const int cc = cg + NG * u;
                        const bool d23 = (cc == 0) ? dC0 : dRest;
                        if (fR1) {
                            e1[u] = W_(r0 + a, cq + cc);
                            p1[u] = sp[cc];
                        }
                        if (d23) {
                            e2[u] = W_(r0 + a, r0 + min(cc, a));
                            wcv[u] = wc[cc];
                            pc[u] = sp[o + cc];
                            e3[u] = W_(r1 + 1 + a, r0 + cc);
                        }
                    }
#pragma unroll
                    for (int u = 0; u < NU; ++u) {
                        const int cc = cg + NG * u;
                        const bool d23 = (cc == 0) ? dC0 : dRest;
                        if (fR1) W_(r0 + a, cq + cc) = (cc == 0) ? ((a == 0) ? bet : T(0)) : e1[u] - wa * p1[u];
                        if (d23) {
                            if (cc <= a) W_(r0 + a, r0 + cc) = e2[u] - (wa * (pc[u] - kap * wcv[u]) + ya * wcv[u]);
                            W_(r1 + 1 + a, r0 + cc) = e3[u] - y3 * wcv[u];
                        }
                    }
                } else {
                    if (a < L) {
                        if (dR1)
                            for (int cc = cg; cc < o; cc += NG) {
                                T &e = W_(r0 + a, cq + cc);
                                if (cc == 0) e = (a == 0) ? bet : T(0);
                                else e -= wa * sp[cc];
                            }
                        for (int cc = cg; cc <= a; cc += NG) {
                            if (!((cc == 0) ? dC0 : dRest)) continue;
                            const T wcc = wc[cc];
                            const T yc = sp[o + cc] - kap * wcc;
                            W_(r0 + a, r0 + cc) -= wa * yc + ya * wcc;
                        }
                    }
                    if (a < m3) {
                        for (int cc = cg; cc < L; cc += NG) {
                            if (!((cc == 0) ? dC0 : dRest)) continue;
                            W_(r1 + 1 + a, r0 + cc) -= y3 * wc[cc];
                        }
                    }
                }
            };

            T *ucol = U + (i64)(r0 - s - 1) + (i64)s * ldu;
            // the next hop: cq' = r0, its reflector on rows [r0 + b, ...] of column r0
            const int nr0 = r0 + b, nr1 = min(nr0 + b - 1, n - 1);
            const bool next_hh = nr0 <= n - 1 && nr1 - nr0 + 1 >= 2;
            if (next_hh) {
                // Early publish. The next sweep's hop that waits for this one reads the
                // columns up to r0 only: R1's columns [cq, r0) and column r0, which are
                // final once R1 and column r0 are updated and the next hop's reflector has
                // eliminated column r0 (this sweep later writes column r0 only with those
                // same values, and reads it only in LDS). So: R1 and column r0; the next
                // reflector (wave 0) while the other waves store R1's columns and U; column
                // r0 written back; progress r0 published; then the rest of R2 and R3,
                // beside the next sweep's hop.
                rank2(1);
                __syncthreads();
                if (wave == 0) householder(nr0, r0, nr1 - nr0 + 1, wn, bn);
                for (int t = tid; t < L; t += kBCThreads) ucol[t] = wc[t];
                store_cols(cq + 1, r0 - 1);
                // column r0 except its pivot entry (b, the only value the reflector
                // decides), then the pivot once the reflector is formed
                writeback(r0, b, nr1 - nr0 + 1, T(0), true);
                __syncthreads();
                if (tid == 0) st_agent(Bp + (i64)r0 * ldb + b, (T)*bn);
                if (h > 0) {
                    wg_publish_fence();
                    if (tid == 0) flag_store_agent(prog + s, r0);
                }
                rank2(2);
                held_lo = r0;
                // the next hop's loads overwrite the ring slots of the columns stored above,
                // and its p reads R2 and R3
                __syncthreads();
                T *tw = wc;
                wc = wn;
                wn = tw;
                double *tb = bc;
                bc = bn;
                bn = tb;
            } else {
                // the sweep's last reflector
                rank2(3);
                __syncthreads();
                for (int t = tid; t < L; t += kBCThreads) ucol[t] = wc[t];
                const int keep_lo = min(r0, r1 + 1);
                store_cols(cq + 1, keep_lo - 1);
                held_lo = keep_lo;
                __syncthreads();
            }
        }
        // the rest of the last window
        store_cols(held_lo, held_hi);
        wg_publish_fence();
        if (tid == 0) flag_store_agent(prog + s, kDone);
        s = settle(s + ph.g[phase]);
    }
}

// ---------------------------------------------------------------------------
// Resident form: the band stays in registers, only reflectors and rows travel.
//
// Workgroup h runs hop h of every sweep and holds the two b x b blocks that hop works
// on for the whole chase: D = A[r0..r1, r0..r1] (full square) and L = A[r0..r1,
// r0-b..r0-1], r0 = s + 1 + h b, r1 = r0 + b - 1 (h = 0: of L only column r0 - 1). Row i
// and column j sit in slots i mod b and j mod b, so when the sweep number advances by
// one nothing moves: row and column r0 leave their slot and row and column r1 + 1 = r0 +
// b enter the same one. Thread = (row slot, group of CPT column slots), B lanes per row
// vector, the CPT elements of each block in registers.
//
// Per sweep, workgroup h
//   1. receives w' = w_{h-1}(s) from its left neighbour; column r0 - 1 of D becomes a column
//      of L, a zero row enters L;
//   2. y = 2 L w', x = column r0 - b of L - y w'^T, the reflector w and beta of x (every
//      wave forms it from the same sums, so it is not sent through LDS), w to the right,
//      beta to the left. The value beta that the right neighbour left in the entering row
//      in sweep s - 1 (its only entry, in column r0 - 1) joins after the partial sums;
//   3. L -= y w'^T, L -= w (2 w^T L); its row r0 goes to the left neighbour;
//   4. receives row r1 of sweep s - 1 from the right (new last row and column of D);
//      p = 2 D w, D -= w y^T + y w^T with y = p - (w^T p) w; D(r0, r0) goes to the left.
//      The right's D(r1, r1), the last value it forms, joins after the partial sums.
// Workgroup 0 writes (d, e). Rows and columns from n on are zeros, which need no special
// cases: a one-row hop finds a zero tail and makes the identity. A ninth wave (fifth, for
// b <= 32) does the receiving, each message between the two barriers before its first use,
// so that no round trip of 0.4 us stands in the others' way.
//
// A message word is 64 bits: 32 bits of payload and the sweep number + 1 as a tag, so the
// receiver polls the data itself and one store-to-load latency covers the hand-off (a
// flag behind the data costs a second one). Buffers are double: sweep s + 2 overwrites
// sweep s's words only after an answer that was computed from them came back.
//
// Bound: the sweep-to-sweep lag. Its cycles: a hand-off to the right, steps 1-2 there, beta
// back, the end of step 2; the same with D(r1, r1); and a workgroup's own steps 1-4. All
// three take about 3.1 us at b = 64 (of which a hand-off 0.5, step 2 1.0, step 4 1.2).
// Measured alone, FP64: 3.1 us per sweep at b = 64 and 2.75 at b = 32, against 16.4 and 9.1
// for the windowed kernel, which moves 2 b columns through memory per hop and pays two
// dependent global round trips per hop (n = 16384: 276 -> 52 ms; n = 4096: 67 -> 13 ms;
// n = 1024, b = 32: 9.3 -> 2.7 ms). Beside Q_s^T's products it shares every CU with them
// (n = 16384: 99 ms, and 145 ms for the products). With compute waves polling and both late
// values awaited at the start it took 3.9 us (the form without the ninth wave still does);
// neighbouring workgroups on one XCD, a sleep between polls or two to four polls in flight
// gained nothing; four or sixteen compute waves took 4.9 and 3.8 us against 3.9 for eight.
// The ninth wave's own loop keeps it from holding a block it never uses: 74 VGPRs instead
// of 104, so that two workgroups fit on a CU, and 3.1 us instead of 3.3.
// ---------------------------------------------------------------------------
using u64 = unsigned long long;

template <typename T> struct MsgWord;
template <> struct MsgWord<double> {
    static constexpr int N = 2; // words per value
    __device__ static void put(u64 *p, double v, unsigned tag) {
        const u64 b = (u64)__double_as_longlong(v), t = (u64)tag << 32;
        st_agent(p, (b & 0xffffffffull) | t);
        st_agent(p + 1, (b >> 32) | t);
    }
    __device__ static bool get(const u64 *p, double &v, unsigned tag) {
        const u64 a = ld_agent(p), b = ld_agent(p + 1);
        v = __longlong_as_double((long long)((a & 0xffffffffull) | (b << 32)));
        return (unsigned)(a >> 32) == tag && (unsigned)(b >> 32) == tag;
    }
};
template <> struct MsgWord<float> {
    static constexpr int N = 1;
    __device__ static void put(u64 *p, float v, unsigned tag) {
        st_agent(p, (u64)__float_as_uint(v) | ((u64)tag << 32));
    }
    __device__ static bool get(const u64 *p, float &v, unsigned tag) {
        const u64 a = ld_agent(p);
        v = __uint_as_float((unsigned)a);
        return (unsigned)(a >> 32) == tag;
    }
};

// Message buffers of the link between workgroups h - 1 and h, one set per parity of s:
// w (h - 1 -> h, b values), row (h -> h - 1, b values), beta and the row's diagonal entry
// (h -> h - 1, one value each on a line of its own).
constexpr int kBetaPad = 16; // values
template <typename T> __host__ __device__ constexpr i64 msg_words(int b) { return (2 * b + 2 * kBetaPad) * (i64)(sizeof(T) / 4); }

// v of row slot idx0 + j of the lane's column group: lane slots repeat every B lanes, so
// lanes 0..B-1 hold them all. `first`: the first column slot of the wave (uniform).
template <int B, int CPT, typename V>
__device__ __forceinline__ V slot_value(V v, int first, int j, int lane) {
    if constexpr (B == 64) return read_lane(v, first + j);
    else if constexpr (B == 32) {
        const V a = read_lane(v, first + j), b = read_lane(v, first + CPT + j);
        return lane < 32 ? a : b;
    } else return __shfl(v, first + CPT * (lane / B) + j, 64);
}
// totals over the B lanes of a group of CPT values per lane, all in every lane: halving
// exchanges (each lane keeps half of the columns) instead of CPT butterflies
template <int B, int CPT, typename V> __device__ __forceinline__ void column_sums(V (&v)[CPT], int lane) {
    if constexpr (B == 16) {
#pragma unroll
        for (int j = 0; j < CPT; ++j) v[j] = group_sum<16>(v[j]);
    } else if constexpr (B == 64) {
        static_assert(CPT == 8, "eight lanes per column at the end");
        V t[4], r[2];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            V a = v[i], b = v[i + 4];
            lane_swap<32>(a, b);
            t[i] = a + b;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            V a = t[i], b = t[i + 2];
            lane_swap<16>(a, b);
            r[i] = a + b;
        }
        const bool odd = (lane & 8) != 0;
        const V q = sum8((odd ? r[1] : r[0]) + dpp_mov<kRowRor8>(odd ? r[0] : r[1]));
#pragma unroll
        for (int j = 0; j < CPT; ++j) v[j] = read_lane(q, 8 * j);
    } else if constexpr (B == 32) {
        static_assert(CPT == 4, "eight lanes per column at the end");
        V r[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            V a = v[i], b = v[i + 2];
            lane_swap<16>(a, b);
            r[i] = a + b;
        }
        const bool odd = (lane & 8) != 0;
        const V q = sum8((odd ? r[1] : r[0]) + dpp_mov<kRowRor8>(odd ? r[0] : r[1]));
#pragma unroll
        for (int j = 0; j < CPT; ++j) { // column j of the group in its lanes 8 j ..
            const V a = read_lane(q, 8 * j), b = read_lane(q, 32 + 8 * j);
            v[j] = lane < 32 ? a : b;
        }
    }
}

// f(0) + ... + f(N - 1) pairwise (N a power of two): a short chain
template <int N, typename F> __device__ __forceinline__ auto tree_sum(F &&f) {
    decltype(f(0)) v[N];
#pragma unroll
    for (int g = 0; g < N; ++g) v[g] = f(g);
#pragma unroll
    for (int d = N / 2; d > 0; d /= 2)
#pragma unroll
        for (int g = 0; g < d; ++g) v[g] += v[g + d];
    return v[0];
}

// compute threads (column groups of b rows), and with RECV one wave more that only receives
constexpr int chase_compute(int b) { return b == 64 ? 512 : 256; }
constexpr int chase_threads(int b, bool recv) { return chase_compute(b) + (recv ? 64 : 0); }

template <typename T, int B, bool RECV>
__global__ __launch_bounds__(chase_threads(B, RECV)) void bc_chase_resident_kernel(const T *Bp, T *U, i64 ldu, int n,
                                                                                   T *dd, T *ee, u64 *msg, int *err) {
    constexpr int NG = chase_compute(B) / B; // column groups
    constexpr int CPT = B / NG;              // columns per thread
    constexpr int SPW = CPT * (64 / B);      // column slots per wave
    constexpr int NWD = MsgWord<T>::N;
    constexpr int M = B - 1;
    const int ldb = 2 * B;
    __shared__ T s_wp[B], s_x[B], s_row[B], s_lrow[B];
    __shared__ T s_part[NG][B], s_part2[NG][B];
    __shared__ T s_beta, s_diag;
    __shared__ int s_go;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool receiver = RECV && wave == NG * B / 64;
    const int lam = tid & M, cg = B == 64 ? wave : tid / B; // b = 64: uniform in the wave
    const int c0 = cg * CPT;       // this thread's first column slot
    const int cw = wave * SPW;     // this wave's first column slot
    const int h = blockIdx.x;
    // the chase is a chain of short latency-bound steps; products running beside it are not
    __builtin_amdgcn_s_setprio(3);

    const i64 mw = msg_words<T>(B);
    u64 *left = msg + (i64)h * 2 * mw, *right = left + 2 * mw; // links to h - 1 and h + 1
    constexpr int oRow = B * NWD, oBeta = 2 * B * NWD, oDiag = (2 * B + kBetaPad) * NWD;

    if (tid == 0) {
        s_go = 1;
        if (h == 0) {
            dd[0] = Bp[0];
            ee[n - 1] = T(0);
        }
    }
    __syncthreads();

    // one value per lane from p + lane * NWD, for the lanes that want one; false: the wait expired
    auto poll = [&](const u64 *p, bool want, unsigned tag, T &v) -> bool {
        bool ok = !want;
        for (long long it = 0;; ++it) {
            if (!ok) ok = MsgWord<T>::get(p + lane * NWD, v, tag);
            if (__all(ok)) return true;
            if (it > kPollLimit) {
                if (lane == 0)
                    __hip_atomic_store(err, (int)DEV_WATCHDOG, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return false;
            }
        }
    };

    // the four messages of sweep s, each to be received before its barrier (A to D below)
    auto right_ran = [&](int s) { return s > 0 && s + (h + 1) * B <= n - 1; }; // h + 1 had sweep s - 1
    auto receive_w = [&](int s) { // A
        T v = T(0);
        if (h > 0 && !poll(left + (s & 1) * mw, lane < B, (unsigned)s + 1u, v)) s_go = 0;
        if (lane < B) s_wp[lane] = v; // h = 0: zero
    };
    auto receive_one = [&](int s, int at, T *to) { // B: beta, D: the diagonal entry
        T v = T(0);
        if (right_ran(s) && !poll(right + ((s & 1) ^ 1) * mw + at, lane == 0, (unsigned)s, v)) s_go = 0;
        if (lane == 0) *to = v;
    };
    auto receive_row = [&](int s) { // C; the diagonal slot stays zero
        T v = T(0);
        const bool want = lane < B && lane != ((s + h * B) & M);
        if (right_ran(s) && !poll(right + ((s & 1) ^ 1) * mw + oRow, want, (unsigned)s, v)) s_go = 0;
        if (lane < B) s_row[lane] = v;
    };
    if (receiver) {
        for (int s = 0; s + 1 + h * B <= n - 1; ++s) {
            receive_w(s);
            __syncthreads(); // A
            if (!s_go) return;
            receive_one(s, oBeta, &s_beta);
            __syncthreads(); // B
            receive_row(s);
            __syncthreads(); // C
            receive_one(s, oDiag, &s_diag);
            __syncthreads(); // D
        }
        return;
    }

    T L[CPT], D[CPT];
    {
        const int r0 = 1 + h * B;
        const int gi = r0 + ((lam - r0) & M);
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            const int gc = r0 + ((c0 + j - r0) & M);
            const int hi = max(gi, gc), lo = min(gi, gc);
            D[j] = hi < n ? Bp[(hi - lo) + (i64)lo * ldb] : T(0);
            const int gl = gc - B, diff = gi - gl;
            L[j] = (gi < n && gl >= 0 && diff <= B) ? Bp[diff + (i64)gl * ldb] : T(0);
        }
    }
    for (int s = 0; s + 1 + h * B <= n - 1; ++s) {
        const int r0 = s + 1 + h * B;
        const int kap = r0 & M, kold = (r0 - 1) & M;
        const i64 cur = (s & 1) * mw; // this sweep's buffers
        const unsigned tag = (unsigned)s + 1u;

        if (!RECV && wave == 0) receive_w(s);
        __syncthreads(); // A: w' is here
        if (!s_go) return;
        // column indexes of this thread's group (outside 0 .. CPT - 1: another group's)
        const int jo = kold - c0, jk = kap - c0, jx = h > 0 ? jk : jo; // jx: the column to eliminate
        // ---- 1. the entering column and (zero) row of L; beta, its only entry there, joins below
        if (s > 0) {
#pragma unroll
            for (int j = 0; j < CPT; ++j) L[j] = lam == kold ? T(0) : (j == jo ? D[j] : L[j]);
        }
        // ---- 2. y = 2 L w', the reflector of column x
        {
            T acc[2] = {T(0), T(0)};
#pragma unroll
            for (int j = 0; j < CPT; ++j) acc[j & 1] += L[j] * s_wp[c0 + j];
            s_part[cg][lam] = acc[0] + acc[1];
#pragma unroll
            for (int j = 0; j < CPT; ++j)
                if (j == jx) s_x[lam] = L[j];
        }
        if (!RECV && wave == 1) receive_one(s, oBeta, &s_beta);
        __syncthreads(); // B: the partial sums, and beta
        const T bold = s_beta, wpk = s_wp[kap], wpo = s_wp[kold];
        T y = tree_sum<NG>([&](int g) { return s_part[g][lam]; });
        T xt = s_x[lam];
        if (s > 0 && lam == kold) { // the entering row is beta in column slot kold
            y = bold * wpo;
            if (h == 0) xt = bold;
        }
        y *= T(2);
        double x = (double)(xt - y * wpk);
        double alpha = read_lane(x, kap);
        double tail = group_sum<B>(lam == kap ? 0.0 : x * x);
        double wd = 0.0, beta = alpha;
        if (tail != 0.0) {
            double back = 1.0;
            if (!(tail + alpha * alpha > 0x1p-900 && tail + alpha * alpha < 0x1p900)) {
                // into the short square roots' range
                const bool up = fabs(alpha) < 1.0 && tail < 1.0;
                const double sc = up ? 0x1p500 : 0x1p-500;
                back = up ? 0x1p-500 : 0x1p500;
                x *= sc;
                alpha *= sc;
                tail = group_sum<B>(lam == kap ? 0.0 : x * x);
            }
            double nrm, inv, r;
            fast_sqrt(alpha * alpha + tail, nrm, r);
            if (alpha >= 0.0) nrm = -nrm;
            beta = nrm * back;
            alpha -= nrm;
            fast_sqrt(alpha * alpha + tail, r, inv);
            wd = (lam == kap ? alpha : x) * inv;
        }
        const T w = (T)wd;
        if (wave == 0) {
            if (lane < B && r0 + B <= n - 1) MsgWord<T>::put(right + cur + lane * NWD, w, tag);
        } else if (wave == 1) {
            if (lane == 0) {
                if (h > 0) MsgWord<T>::put(left + cur + oBeta, (T)beta, tag);
                else ee[s] = (T)beta;
            }
        } else if (wave == 3) {
            const int q = (lam - kap) & M;
            if (lane < B && s <= n - 3 && r0 + q <= n - 1) U[(i64)h * B + q + (i64)s * ldu] = w;
        }
        // ---- 3. L -= y w'^T, L -= w (2 w^T L); row r0 of L
        {
            T u[CPT];
#pragma unroll
            for (int j = 0; j < CPT; ++j) {
                if (s > 0 && lam == kold && j == jo) L[j] = bold;
                L[j] -= y * s_wp[c0 + j]; // read again: held, it would cost the registers of a wave
                u[j] = w * L[j];
            }
            column_sums<B, CPT>(u, lane);
            const T w2 = T(2) * w;
#pragma unroll
            for (int j = 0; j < CPT; ++j) L[j] -= w2 * u[j];
            if (lam == kap)
#pragma unroll
                for (int j = 0; j < CPT; ++j) s_lrow[c0 + j] = L[j];
        }
        if (!RECV && wave == 2) receive_row(s);
        __syncthreads(); // C: row r0 of L, and the right's last row but for its diagonal entry
        if (wave == 3 && h > 0 && lane < B && lane != kap)
            MsgWord<T>::put(left + cur + oRow + lane * NWD, s_lrow[lane], tag);
        // ---- 4. D: its new row and column, then the two-sided update
        if (s > 0) {
            const T rl = s_row[lam];
#pragma unroll
            for (int j = 0; j < CPT; ++j) {
                const T rc = s_row[c0 + j];
                D[j] = lam == kold ? rc : (j == jo ? rl : D[j]);
            }
        }
        T wc[CPT];
        {
            T acc[2] = {T(0), T(0)};
#pragma unroll
            for (int j = 0; j < CPT; ++j) {
                wc[j] = slot_value<B, CPT>(w, cw, j, lane);
                acc[j & 1] += D[j] * wc[j];
            }
            s_part2[cg][lam] = acc[0] + acc[1];
        }
        if (!RECV && wave == 3) receive_one(s, oDiag, &s_diag);
        __syncthreads(); // D: the partial sums, and the diagonal entry
        T p = tree_sum<NG>([&](int g) { return s_part2[g][lam]; });
        if (s > 0) {
            const T dg = s_diag;
            if (lam == kold) {
                p += dg * w;
#pragma unroll
                for (int j = 0; j < CPT; ++j)
                    if (j == jo) D[j] = dg;
            }
        }
        p *= T(2);
        const T yv = p - group_sum<B>(w * p) * w;
#pragma unroll
        for (int j = 0; j < CPT; ++j) D[j] -= w * slot_value<B, CPT>(yv, cw, j, lane) + yv * wc[j];
#pragma unroll
        for (int j = 0; j < CPT; ++j)
            if (lam == kap && j == jk) {
                if (h > 0) MsgWord<T>::put(left + cur + oDiag, D[j], tag);
                else dd[s + 1] = D[j];
            }
    }
}

template <typename T>
__global__ void bc_extract_kernel(const T *Bp, T *d, T *e, int n, int b) {
    const i64 ldb = 2 * b;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = Bp[(i64)i * ldb];
    if (i < n - 1) e[i] = Bp[1 + (i64)i * ldb];
    if (i == n - 1) e[i] = T(0);
}

// the tridiagonal matrix (d, e) as a packed band: what the windowed form leaves in Bp
template <typename T>
__global__ __launch_bounds__(256) void bc_band_kernel(T *Bp, const T *d, const T *e, int n, int b) {
    const i64 ldb = 2 * b, idx = (i64)blockIdx.x * 256 + threadIdx.x;
    if (idx >= ldb * n) return;
    const i64 j = idx / ldb;
    const int r = (int)(idx - j * ldb);
    Bp[idx] = r == 0 ? d[j] : (r == 1 && j < n - 1) ? e[j] : T(0);
}

template <typename T> size_t bc_lds_bytes(int b) {
    const size_t nseg = std::max<size_t>(1, kBCThreads / (3 * (size_t)b));
    return sizeof(T) * ((size_t)2 * b * (2 * b + 1) + 2 * b + 3 * b + nseg * 3 * b);
}

// Workgroups of the resident kernel that fit on the GPU together wherever the hardware puts
// their waves: the occupancy query divides a CU's wave slots by a workgroup's waves, but a
// workgroup of nine may take three of one SIMD's slots every time.
template <typename T, int B, bool RECV> int chase_capacity(i64 *out) {
    const void *k = reinterpret_cast<const void *>(bc_chase_resident_kernel<T, B, RECV>);
    hipFuncAttributes fa;
    CUEV_HIP(hipFuncGetAttributes(&fa, k));
    int per_cu = 0;
    CUEV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, bc_chase_resident_kernel<T, B, RECV>,
                                                          chase_threads(B, RECV), 0));
    const int simd_waves = std::min(8, 512 / std::max(8, (fa.numRegs + 7) / 8 * 8));
    const int wg_waves = (chase_threads(B, RECV) / 64 + 3) / 4; // of one SIMD
    *out = (i64)std::min(per_cu, simd_waves / wg_waves) * device_cu_count();
    return CUEV_STATUS_SUCCESS;
}

// LDS that the chase asks for on top of its own where it is to have its CUs to itself: what is left is
// less than any product's tiles need (64 x 64 in FP32, 20 KB). The products that run beside the chase
// in the reordered order otherwise share the chase's CUs and slow its chain of short steps down.
constexpr size_t kCuLds = 160 * 1024, kSmallestTiles = 20 * 1024;
template <typename T, int B> constexpr size_t chase_lds() { // the kernel's own
    return sizeof(T) * (4 * B + 2 * (chase_compute(B) / B) * B + 2) + sizeof(int);
}
template <typename T, int B> constexpr size_t chase_pad() {
    return std::max<size_t>(136 * 1024, kCuLds - kSmallestTiles - chase_lds<T, B>() / 256 * 256);
}
template <typename T, int B> constexpr bool chase_alone() {
    const size_t all = chase_pad<T, B>() + chase_lds<T, B>();
    return all <= kCuLds && all + kSmallestTiles > kCuLds;
}
static_assert(chase_alone<double, 16>() && chase_alone<double, 32>() && chase_alone<double, 64>() &&
                  chase_alone<float, 16>() && chase_alone<float, 32>() && chase_alone<float, 64>(),
              "no product beside a padded chase");

template <typename T, int B, bool RECV>
int launch_chase_resident(Workspace<T> &ws, const T *Bp, T *d, T *e, int hops, size_t pad = 0) {
    const int n = ws.n;
    hipStream_t s = ws.stream;
    if (pad)
        CUEV_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(bc_chase_resident_kernel<T, B, RECV>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)pad));
    const i64 words = (i64)(hops + 1) * 2 * msg_words<T>(B);
    CUEV_TRY(fill_int(s, reinterpret_cast<int *>(ws.chmsg), 2 * words, 0)); // no tag of an earlier chase
    const double nhops = (double)n * n / (2.0 * B);
    // each hop writes and reads two messages of b tagged values and writes b values of U
    prof::Scope sc(s, "bc.chase", nhops * (6.0 * B * B + 16.0 * B * B), nhops * 9.0 * B * sizeof(T));
    hipLaunchKernelGGL((bc_chase_resident_kernel<T, B, RECV>), dim3((unsigned)hops), dim3(chase_threads(B, RECV)), pad, s,
                       Bp, ws.U, ws.ldu, n, d, e, reinterpret_cast<u64 *>(ws.chmsg), ws.err);
    CUEV_LAUNCH_CHECK();
    return CUEV_STATUS_SUCCESS;
}

// Resident form when its workgroups, one per hop of the first sweep, all fit on the GPU at
// once (each waits for both neighbours); *done tells whether it was launched. The caller holds
// a CU per workgroup, or the whole GPU (residency.hpp), so other solves need no room here. The form
// with a receiving wave is taken up to half of what the GPU holds of it (b = 64 in FP64: n <= 16384),
// the one without it, which has more room, up to all it holds (n <= 49152; at n = 16384 3.9 us
// per sweep, windowed 16.4). Between n = 16384 and 32768 a chase with it would fit, but has not been measured.
// A chase of at most a quarter of the CUs' number of hops (b = 64: n <= 4096) takes its CUs for itself.
// Whole solves: FP64 n = 1024 7.14 -> 7.00 ms, 2500 19.65 -> 19.19, 4096 36.3 -> 34.8 (the chase 14.7 ->
// 13.3), FP32 4096 29.7 -> 28.8. Above, n = 8192 alone has been measured (127.5 -> 120.2).
template <typename T, int B> int try_chase_resident(Workspace<T> &ws, const T *Bp, T *d, T *e, bool *done) {
    const int hops = (ws.n - 2) / B + 1;
    i64 with = 0, without = 0;
    CUEV_TRY((chase_capacity<T, B, true>(&with)));
    CUEV_TRY((chase_capacity<T, B, false>(&without)));
    *done = true;
    if (2 * hops <= with)
        return launch_chase_resident<T, B, true>(ws, Bp, d, e, hops, 4 * hops <= device_cu_count() ? chase_pad<T, B>() : 0);
    if (hops <= without) return launch_chase_resident<T, B, false>(ws, Bp, d, e, hops);
    *done = false;
    return CUEV_STATUS_SUCCESS;
}

} // namespace

size_t bc_chase_msg_bytes(int n, int b) {
    const i64 hops = n > 2 ? (n - 2) / b + 1 : 0;
    return sizeof(u64) * (size_t)((hops + 1) * 2 * msg_words<double>(b));
}

template <typename T, int B> int launch_chase(Workspace<T> &ws, T *Bp) {
    const int n = ws.n;
    hipStream_t s = ws.stream;
    const int nsweeps = n - 2;
    CUEV_TRY(fill_int(s, ws.prog, n, -1));
    const size_t lds = bc_lds_bytes<T>(B);
    CUEV_HIP(hipFuncSetAttribute((const void *)bc_chase_kernel<T, B>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int per_cu = 0;
    CUEV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, bc_chase_kernel<T, B>,
                                                          kBCThreads, lds));
    const int resident = std::max(1, per_cu * device_cu_count());
    // a sweep of H hops starts about two hops after the previous one, so up to
    // ~H/2 <= n/(2b) sweeps could be active at once; the grid stays a little below
    // that, leaving CUs to the back-transform GEMMs that run beside the chase
    // (measured at n = 16384, b = 64, with the same factor in the phases below:
    // 84 workgroups, chase 307 ms and 0.966 s per solve; 112, 276 ms and 0.931 s;
    // 136, 278 ms and 0.935 s; 168, 274 ms and 0.931 s, with Q_s^T beside the chase
    // going from 222 to 252 ms)
    const int useful = (int)ceil_div((i64)n * 13, 32 * B) + 8;
    const int grid = std::max(1, std::min({nsweeps, resident, useful}));
    // phases of equal sweep counts; phase p keeps the workgroups its sweeps' lengths
    // call for, by the same rule applied to the n - s0 columns left
    ChasePhases ph{};
    ph.np = std::min(kMaxPhases, std::max(1, nsweeps / 256));
    for (int q = 0; q <= ph.np; ++q) ph.s0[q] = (int)((i64)nsweeps * q / ph.np);
    for (int q = 0; q < ph.np; ++q) {
        const int left = n - ph.s0[q];
        const int want = (int)ceil_div((i64)left * 13, 32 * B) + 8;
        ph.g[q] = std::max(1, std::min(grid, want));
        if (q > 0) ph.g[q] = std::min(ph.g[q], ph.g[q - 1]);
    }
    // algorithmic work: ~n^2/(2b) hops, each reading and writing b columns of the
    // packed band (2 * 2b^2 S bytes) and doing ~ (2 * 3b * b + 4 * 4b^2) flops
    const double hops = (double)n * n / (2.0 * B);
    prof::Scope sc(s, "bc.chase", hops * (6.0 * B * B + 16.0 * B * B), hops * 4.0 * B * B * sizeof(T));
    hipLaunchKernelGGL((bc_chase_kernel<T, B>), dim3(grid), dim3(kBCThreads), lds, s, Bp, ws.U,
                       ws.ldu, n, ws.prog, ws.err, ph);
    CUEV_LAUNCH_CHECK();
    return CUEV_STATUS_SUCCESS;
}

template <typename T> int bc_chase(Workspace<T> &ws, T *Bp, T *d, T *e, bool write_band) {
    const int n = ws.n;
    hipStream_t s = ws.stream;
    if (n - 2 > 0) {
        bool done = false;
        switch (ws.chase_windowed ? 0 : ws.b) {
        case 0: break;
        case 16: CUEV_TRY((try_chase_resident<T, 16>(ws, Bp, d, e, &done))); break;
        case 32: CUEV_TRY((try_chase_resident<T, 32>(ws, Bp, d, e, &done))); break;
        case 64: CUEV_TRY((try_chase_resident<T, 64>(ws, Bp, d, e, &done))); break;
        default: CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "bc_chase: unsupported b=%d", ws.b);
        }
        if (done) {
            if (write_band) {
                hipLaunchKernelGGL(bc_band_kernel<T>, dim3((unsigned)ceil_div((i64)2 * ws.b * n, 256)), dim3(256), 0, s,
                                   Bp, d, e, n, ws.b);
                CUEV_LAUNCH_CHECK();
            }
            return CUEV_STATUS_SUCCESS;
        }
        switch (ws.b) {
        case 16: CUEV_TRY((launch_chase<T, 16>(ws, Bp))); break;
        case 32: CUEV_TRY((launch_chase<T, 32>(ws, Bp))); break;
        case 64: CUEV_TRY((launch_chase<T, 64>(ws, Bp))); break;
        default: CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "bc_chase: unsupported b=%d", ws.b);
        }
    }
    hipLaunchKernelGGL(bc_extract_kernel<T>, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, s, Bp,
                       d, e, n, ws.b);
    CUEV_LAUNCH_CHECK();
    return CUEV_STATUS_SUCCESS;
}

template int bc_chase<float>(Workspace<float> &, float *, float *, float *, bool);
template int bc_chase<double>(Workspace<double> &, double *, double *, double *, bool);

} // namespace cuev
