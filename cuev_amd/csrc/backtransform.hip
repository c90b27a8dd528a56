// backtransform.hip — eigenvector back-transform evec <- Q_s Q_b Q_d.
//
// Reference: src/cuda/backtransform.cu:76-275 (bc_back_kernel, sbr_back,
// back_transform).
//
// bc_back (M <- Q_b M). The bulge-chasing reflectors compose to Q_b in forward
// (sweep-major) order, so Q_b M applies them last-first. Reflector (s, h) covers
// rows [s+1+hb, s+(h+1)b]; two reflectors need a fixed relative order only when
// their row ranges overlap, and then the one of the later sweep goes first.
// Overlaps occur only between (s, h) and (s', h) with |s - s'| < b, and between
// (s, h+1) and (s', h) with s' > s. Hence this order is valid:
//   passes of 4 or 8 hop indices, in increasing order;
//   inside a pass, groups of 16 consecutive sweeps, in decreasing order;
//   inside a group, its hops in increasing order; for one hop the 16
//   reflectors (sweeps s0..s0+15) are one block H_s0 ... H_s0+15 = I - V T V^T
//   (V: (b+15) x 16 parallelogram read straight from the shifted U layout,
//   T = (I/2 + striu(V^T V))^-1 for reflectors H = I - 2 w w^T).
// Each block is three small MFMA products on 16 columns of M:
//   X = V^T M_J, Y = T X, M_J -= V Y.
// A workgroup owns 16 or 32 columns of M, each of its waves one hop of a pass (see
// bc_back_kernel). With v_mfma_*_16x16x4, the accumulator register r of lane l holds row
// kidx(r, l/16) of its 16x16 tile; the K index of every product is ordered by the same kidx, so
// the registers of X and Y are directly the B operand of the next product and the rows of M_J
// kept in registers are at once the B operand of X and the accumulator of the update.
//
// sbr_back (M <- Q_s M): the reference applies the DBBR panels last-first,
// M_b -= W_j (Y_j^T M_b) (backtransform.cu:210-230), one rank-b update of M per
// panel. Here the panels of one reduction block are folded into one block
// reflector first, so M is updated once per block (rank k) on the MFMA engine.
#include "backtransform.hpp"

#include <algorithm>
#include <type_traits>
#include <utility>
#include <vector>

#include "gemm.hpp"
#include "profile.hpp"
#include "util.hpp"

namespace cuev {
namespace {

constexpr int kBTThreads = 256; // T-factor kernel: one wave per block reflector
// apply kernel: hops per pass, one wave each. Transposed it runs beside the tridiagonal solver, to
// whose kernels the registers of one wave per SIMD leave room; otherwise nothing runs beside it, and
// two waves hide each other's waits (FP64: n = 8192 26.7 -> 23.0 ms, n = 16384 205 -> 174; beside
// the solver both together take 38 ms at n = 8192 with four waves and 41 with eight).
constexpr int bt_waves(bool tr) { return tr ? 4 : 8; }
// blocks per launch of the apply kernel (a quarter of the stream at n = 16384; 8000 makes no
// difference there)
constexpr i64 kBtSegBlocks = 33000;

template <typename T> struct MfmaBt;
template <> struct MfmaBt<double> {
    typedef double v4 __attribute__((ext_vector_type(4)));
    __device__ static __forceinline__ v4 mma(double a, double b, v4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // f64 16x16x4: accumulator register r of lane l is row l/16 + 4r of the tile
    __device__ static __forceinline__ int kidx(int r, int q) { return 4 * r + q; }
};
template <> struct MfmaBt<float> {
    typedef float v4 __attribute__((ext_vector_type(4)));
    __device__ static __forceinline__ v4 mma(float a, float b, v4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    // f32 16x16x4: accumulator register r of lane l is row 4(l/16) + r of the tile
    __device__ static __forceinline__ int kidx(int r, int q) { return 4 * q + r; }
};

// Operands of every block (g, h), packed in the apply kernel's lane order: one
// wave per block. V's columns are the hop-h reflectors of sweeps 16g..16g+15
// (zero for sweeps past n-3 and for rows past a sweep's last hop, which U holds
// as zeros); V[i][j] = U[hb + i - j + (16g + j) ldu] for 0 <= i - j < b. The
// block is I - V T V^T with T = (I/2 + striu(V^T V))^-1 (reflectors
// H = I - 2 w w^T); TR packs the transposed block I - V T^T V^T. Per lane
// (q = lane/16, li = lane%16) the block holds 8 NKB values:
//   c <  4 NKB: V[16(c/4) + kidx(c%4, q)][li]            (A operand of X = V^T M_J)
//   c >= 4 NKB: W[16t + li][kidx(r, q)], c = 4 NKB + 4t + r (A operand of M_J += W X)
// with W = -V T (TR: -V T^T), stored as pairs: value c of lane l at
// ((c/2) 64 + l) 2 + c%2, so the apply kernel reads each pair with one 16-byte load.
template <typename T, int B, bool TR>
__global__ __launch_bounds__(kBTThreads, 2) void bt_pack_kernel(const T *__restrict__ U, i64 ldu,
                                                             const i64 *__restrict__ toff,
                                                             int ngroups, i64 nblocks, int n,
                                                             T *__restrict__ ops) {
    using MB = MfmaBt<T>;
    constexpr int NG = kBtGroup;
    constexpr int NKB = B / 16 + 1;
    constexpr int NOP = 8 * NKB;
    __shared__ T sv[4][NG][B];
    __shared__ T sn[4][NG][NG + 1];
    __shared__ T st[4][NG][NG + 1];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const i64 id = (i64)blockIdx.x * 4 + wave;
    const bool act = id < nblocks;
    int g = 0, h = 0;
    if (act) {
        int lo = 0, hi = ngroups - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (toff[mid] <= id) lo = mid;
            else hi = mid - 1;
        }
        g = lo;
        h = (int)(id - toff[g]);
    }
    const int s0 = g * NG;
    {
        // the block's NG reflectors: every load issued before its LDS store (one round trip)
        constexpr int PER = NG * B / 64;
        static_assert(NG * B % 64 == 0, "bt_pack load layout");
        T v[PER];
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int e = lane + 64 * u, j = e / B, k = e - j * B, sw = s0 + j;
            v[u] = (act && sw <= n - 3) ? U[(i64)h * B + k + (i64)sw * ldu] : T(0);
        }
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int e = lane + 64 * u, j = e / B, k = e - j * B;
            sv[wave][j][k] = v[u];
        }
    }
    __syncthreads();
    // strictly upper Gram: N[i][j] = v_i . v_j with v_j shifted down by j - i rows
    for (int pidx = lane; pidx < NG * NG; pidx += 64) {
        const int i = pidx % NG, j = pidx / NG;
        T acc = T(0);
        if (i < j) {
            const int dl = j - i;
            for (int t = 0; t + dl < B; ++t) acc += sv[wave][i][t + dl] * sv[wave][j][t];
        }
        sn[wave][i][j] = acc;
    }
    __syncthreads();
    // T = (I/2 + N)^-1, column j by lane j (back substitution)
    if (lane < NG) {
        const int j = lane;
        st[wave][j][j] = T(2);
        for (int i = j - 1; i >= 0; --i) {
            T acc = T(0);
            for (int k = i + 1; k <= j; ++k) acc += sn[wave][i][k] * st[wave][k][j];
            st[wave][i][j] = T(-2) * acc;
        }
        for (int i = j + 1; i < NG; ++i) st[wave][i][j] = T(0);
    }
    __syncthreads();
    if (!act) {
        if (id == nblocks) // an all-zero block after the last (the identity, for waves without one)
            for (int c = 0; c < NOP; ++c) ops[id * (i64)(NOP * 64) + c * 64 + lane] = T(0);
        return;
    }
    const int q = lane >> 4, li = lane & 15;
    T *ob = ops + id * (i64)(NOP * 64) + 2 * lane;
#pragma unroll
    for (int c = 0; c < 4 * NKB; ++c) {
        const int d = 16 * (c >> 2) + MB::kidx(c & 3, q) - li;
        ob[(c >> 1) * 128 + (c & 1)] = (d >= 0 && d < B) ? sv[wave][li][d] : T(0);
    }
#pragma unroll 1
    for (int t = 0; t < NKB; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = MB::kidx(r, q), i = 16 * t + li;
            T acc = T(0);
            for (int k = 0; k < NG; ++k) {
                const int d = i - k;
                const T v = (d >= 0 && d < B) ? sv[wave][k][d] : T(0);
                acc += v * (TR ? st[wave][j][k] : st[wave][k][j]);
            }
            const int c = 4 * NKB + 4 * t + r;
            ob[(c >> 1) * 128 + (c & 1)] = -acc;
        }
}

// last group with hop h (-1: none)
template <int B> __host__ __device__ __forceinline__ int bt_gmax(int n, int h) {
    const int m = n - 3 < n - 2 - h * B ? n - 3 : n - 2 - h * B;
    return m < 0 ? -1 : m / kBtGroup;
}

// Tile j of one half of a block's packed operands, V (half 0) or W (half 1) of NC values.
template <typename T, int NC>
__device__ __forceinline__ void bt_load_ops(T (&o)[NC], const T *__restrict__ ops, i64 id, int half, int j, int lane) {
    typedef T T2 __attribute__((ext_vector_type(2)));
    const T2 *p = reinterpret_cast<const T2 *>(ops + id * (i64)(2 * NC * 64)) + (half * (NC / 2) + 2 * j) * 64 + lane;
    const T2 v0 = p[0], v1 = p[64];
    o[4 * j] = v0.x;
    o[4 * j + 1] = v0.y;
    o[4 * j + 2] = v1.x;
    o[4 * j + 3] = v1.y;
}

template <int... PH, typename F> __device__ __forceinline__ void bt_rotations(std::integer_sequence<int, PH...>, F &&f) {
    (f(std::integral_constant<int, PH>{}), ...);
}

// M <- Q_b M (TR: M <- Q_b^T M, the blocks in reverse order, each transposed) for columns
// [0, ncols), over the passes p_first to p_last (in application order; a pass leaves all its rows
// in M, so a launch may end and the next begin at any pass). One workgroup per 16 NCT columns.
//
// Pass p applies the hops p NW + w, wave w one of them. Block (g, h) covers the 16 NKB =
// b + 16 rows from 16 g + 1 + h b on, and block (g + 1, h + 1) the b + 16 rows after those; of two
// reflectors whose rows overlap, (s, h + 1) and (s', h) with s' > s, the second goes first. So
// while wave w is at group g, wave w + 1 may be at group g + 1: the waves' blocks of one step are
// independent, and their windows make one contiguous window of NW NKB tiles of 16 rows,
// which moves up by one tile per step (TR: down). Every wave keeps its NKB tiles in registers;
// at each step the tile at one end of a window goes to the next wave through LDS (at the end of
// the row: to M), and one enters at the other (at the beginning: from M, its loads issued two
// steps earlier, behind that step's operand loads, whose waits they would lengthen otherwise).
// It enters the registers of the tile that left, so the roles of the registers rotate: the step
// is written out for each rotation (twice, for the two sets of loads from M). A wave without a block in a step (at a
// pass's ends, or past the last hop) applies the all-zero block, which changes nothing.
// The next block's operands are loaded into the registers of the current ones as these die, tile
// by tile. The tile that leaves is updated first, its hand-over hidden behind the other tiles'
// products; the entering tile is used last in X.
//
// Bound: the MFMA pipe (8 NKB NCT products per step and wave: at b = 64 in FP64 2560 NCT cycles of
// one SIMD) and, where there are fewer of column strips than CUs, their number.
// Measured in FP64 at b = 64 (direct order, nothing beside it): n = 2500 1.5 ms, 4096 3.8, 8192 23,
// 16384 172 (2 n^3 flops at 51 TF/s; the products' pipe is busy 85% of the time). With one wave per
// 16 columns that walked every block, n = 2500 5.7 ms (on 157 of 1024 SIMDs), 4096 14.8, 8192 63,
// 16384 242; with M's and the operands' loads issued together, one step ahead, 16384 258.
template <typename T, int B, bool TR, int NCT>
__global__ __launch_bounds__(64 * bt_waves(TR)) void bc_back_kernel(const T *__restrict__ ops, const i64 *__restrict__ toff,
                                                             i64 nblocks, const T *__restrict__ zp, T *M, i64 ldm,
                                                             int n, int ncols, int p_first, int p_last) {
    using MB = MfmaBt<T>;
    using V4 = typename MB::v4;
    constexpr int NKB = B / 16 + 1; // tiles of a block
    constexpr int NC = 4 * NKB;     // 4-row K chunks of a block; values per operand half
    constexpr int NW = bt_waves(TR); // hops of a pass
    constexpr int kSrc = TR ? NW - 1 : 0, kSink = TR ? 0 : NW - 1; // waves next to M
    constexpr int kIn = TR ? NKB - 1 : 0, kOut = TR ? 0 : NKB - 1; // entering and leaving tile of a window
    __shared__ T hand[2][NW][NCT][4][64]; // [parity of the step][from wave]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, q = lane >> 4, li = lane & 15;
    const int wcol = blockIdx.x * (16 * NCT);

    // tile rows [r0, r0 + 16) of the workgroup's columns in accumulator layout; row 0, which no
    // reflector covers, is not one of M's here: the all-zero block would spread a NaN in it
    auto load_tile = [&](int r0, V4(&v)[NCT]) {
#pragma unroll
        for (int c = 0; c < NCT; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = r0 + MB::kidx(r, q), col = wcol + 16 * c + li;
                const bool ok = row > 0 && row < n && col < ncols;
                v[c][r] = *(ok ? M + row + (i64)col * ldm : zp);
            }
    };
    auto store_tile = [&](int r0, const V4(&v)[NCT]) {
#pragma unroll
        for (int c = 0; c < NCT; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = r0 + MB::kidx(r, q), col = wcol + 16 * c + li;
                if (row > 0 && row < n && col < ncols) M[row + (i64)col * ldm] = v[c][r];
            }
    };

    for (int p = p_first; TR ? p >= p_last : p <= p_last; p += TR ? -1 : 1) {
        const int h0 = p * NW, h = h0 + wave, gm = bt_gmax<B>(n, h), gs = bt_gmax<B>(n, h0);
        const int nst = gs + NW; // steps: wave 0 at the groups gs .. -(NW - 1)
        int g = (TR ? -(NW - 1) : gs) + wave;
        int top = g * kBtGroup + 1 + h * B; // first row of this wave's window
        auto block = [&](int g_) { return g_ >= 0 && g_ <= gm ? toff[g_] + h : nblocks; };
        T ov[NC], ow[NC];
        V4 m[NKB][NCT], ent[2][NCT];
        const i64 id0 = block(g);
#pragma unroll
        for (int j = 0; j < NKB; ++j) {
            bt_load_ops<T, NC>(ov, ops, id0, 0, j, lane);
            bt_load_ops<T, NC>(ow, ops, id0, 1, j, lane);
        }
#pragma unroll
        for (int j = 0; j < NKB; ++j) load_tile(top + 16 * j, m[j]);
        if (wave == kSrc) load_tile(TR ? top + 16 * NKB : top - 16, ent[1]);

        // step t in rotation PH, t % (2 NKB): window tile j is m[at(j)]
        auto step = [&](auto rot, int t) {
            constexpr int PH = decltype(rot)::value;
            auto at = [](int j) constexpr { return TR ? (j + PH) % NKB : (j + 2 * NKB - PH) % NKB; };
            const bool last = t + 1 == nst;
            if (t > 0) {
                if (wave == kSrc) {
#pragma unroll
                    for (int c = 0; c < NCT; ++c) m[at(kIn)][c] = ent[PH & 1][c];
                } else {
                    const int from = TR ? wave + 1 : wave - 1;
#pragma unroll
                    for (int c = 0; c < NCT; ++c)
#pragma unroll
                        for (int r = 0; r < 4; ++r) m[at(kIn)][c][r] = hand[(t - 1) & 1][from][c][r][lane];
                }
            }
            const int ng = TR ? g + 1 : g - 1;
            const i64 nid = last ? nblocks : block(ng);

            // ---- X = V^T M_J, two chains per 16 columns, the entering tile last
            V4 x[NCT][2];
#pragma unroll
            for (int c = 0; c < NCT; ++c) x[c][0] = x[c][1] = V4{T(0), T(0), T(0), T(0)};
#pragma unroll
            for (int jj = 1; jj <= NKB; ++jj) {
                const int j = (kIn + (TR ? NKB - jj : jj)) % NKB;
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int c = 0; c < NCT; ++c)
                        x[c][r & 1] = MB::mma(ov[4 * j + r], m[at(j)][c][r], x[c][r & 1]);
                bt_load_ops<T, NC>(ov, ops, nid, 0, j, lane);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int c = 0; c < NCT; ++c) x[c][0] += x[c][1];
            // ---- M_J += W X (W = -V T, or -V T^T): the leaving tile first; two tiles at a time
            // where a tile has one chain only
            constexpr int TW = NCT > 1 ? 1 : 2;
#pragma unroll
            for (int j0 = 0; j0 < NKB; j0 += TW) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int jj = j0; jj < j0 + TW && jj < NKB; ++jj) {
                        const int j = (kOut + jj) % NKB;
#pragma unroll
                        for (int c = 0; c < NCT; ++c)
                            m[at(j)][c] = MB::mma(ow[4 * j + r], x[c][0][r], m[at(j)][c]);
                    }
#pragma unroll
                for (int jj = j0; jj < j0 + TW && jj < NKB; ++jj)
                    bt_load_ops<T, NC>(ow, ops, nid, 1, (kOut + jj) % NKB, lane);
                __builtin_amdgcn_sched_barrier(0);
                if (j0 == (NKB > TW ? TW : 0) && !last && wave != kSink) { // the leaving tile is ready by now
#pragma unroll
                    for (int c = 0; c < NCT; ++c)
#pragma unroll
                        for (int r = 0; r < 4; ++r) hand[t & 1][wave][c][r][lane] = m[at(kOut)][c][r];
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (last) {
#pragma unroll
                for (int j = 0; j < NKB; ++j) store_tile(top + 16 * j, m[at(j)]);
            } else if (wave == kSink) {
                store_tile(top + 16 * kOut, m[at(kOut)]);
            }
            if (wave == kSrc && t + 2 < nst) load_tile(TR ? top + 16 * NKB + 16 : top - 32, ent[PH & 1]);
            __syncthreads();
            g = ng;
            top += TR ? 16 : -16;
        };
        for (int t = 0; t < nst;) {
            bool go = true;
            bt_rotations(std::make_integer_sequence<int, 2 * NKB>{}, [&](auto rot) {
                if (!go) return;
                step(rot, t);
                go = ++t < nst;
            });
        }
        // the next pass reads these rows back through other waves
        wave_stores_done();
        __syncthreads();
    }
}

// The passes over columns [0, nc) of M, 16 NCT of them per workgroup.
template <typename T, int B, int NCT>
int launch_bc_passes(Workspace<T> &ws, hipStream_t s, T *M, i64 ldm, int nc, bool tr, const T *zp) {
    const int n = ws.n;
    // Passes in launches of at least kBtSegBlocks blocks each (the last one fewer): the
    // workgroups of one launch drift apart along the block stream as it goes, and a launch
    // boundary lines them up again.
    const int nw = bt_waves(tr), np = (n - 2) / B / nw + 1;
    std::vector<std::pair<int, int>> segs; // (first, last) pass, in application order
    i64 acc = 0;
    for (int k = 0; k < np; ++k) {
        const int p = tr ? np - 1 - k : k;
        if (bt_gmax<B>(n, p * nw) < 0) continue;
        if (acc == 0) segs.emplace_back(p, p);
        segs.back().second = p;
        for (int w = 0; w < nw; ++w) acc += bt_gmax<B>(n, p * nw + w) + 1;
        if (acc >= kBtSegBlocks) acc = 0;
    }
    const dim3 grid((unsigned)ceil_div(nc, 16 * NCT));
    const auto kernel = tr ? bc_back_kernel<T, B, true, NCT> : bc_back_kernel<T, B, false, NCT>;
    for (const auto &sg : segs) {
        hipLaunchKernelGGL(kernel, grid, dim3(64 * nw), 0, s, ws.BtT, ws.bt_off, ws.bt_blocks, zp, M, ldm, n, nc,
                           sg.first, sg.second);
        CUEV_LAUNCH_CHECK();
    }
    return CUEV_STATUS_SUCCESS;
}

template <typename T, int B>
int launch_bc_back(Workspace<T> &ws, hipStream_t s, const T *U, T *M, i64 ldm, bool tr) {
    const int n = ws.n;
    if (ws.bt_blocks <= 0) return CUEV_STATUS_SUCCESS;
    {
        prof::Scope sc(s, "bt.bc_pack", (double)ws.bt_blocks * kBtGroup * kBtGroup * B);
        const dim3 grid((unsigned)ceil_div(ws.bt_blocks + 1, 4)); // + the zero block
        if (tr)
            hipLaunchKernelGGL((bt_pack_kernel<T, B, true>), grid, dim3(kBTThreads), 0, s, U, ws.ldu,
                               ws.bt_off, ws.bt_groups, ws.bt_blocks, n, ws.BtT);
        else
            hipLaunchKernelGGL((bt_pack_kernel<T, B, false>), grid, dim3(kBTThreads), 0, s, U, ws.ldu,
                               ws.bt_off, ws.bt_groups, ws.bt_blocks, n, ws.BtT);
        CUEV_LAUNCH_CHECK();
    }
    // 4 flops per reflector entry per column: sum_s (n-1-s) entries ~ n^2/2
    prof::Scope sc(s, "bt.bc_back", 2.0 * (double)n * n * n);
    const T *zp = U + ws.ldu * (i64)n; // zeros past U's last column
    // Columns in chunks of one workgroup per CU: every workgroup streams the same block operands,
    // and those that start together share them in L2 (in one launch of more, the later ones
    // would start as earlier ones finish and lose that). 32 columns per workgroup take 1.5 times as
    // long as 16 (each operand read serves two products), so 16 where that covers what is left.
    const i64 ncu = device_cu_count();
    for (i64 c0 = 0; c0 < n;) {
        const bool wide = n - c0 > 16 * ncu;
        const int nc = (int)std::min<i64>(wide ? 32 * ncu : 16 * ncu, n - c0);
        CUEV_TRY((wide ? launch_bc_passes<T, B, 2>(ws, s, M + c0 * ldm, ldm, nc, tr, zp)
                       : launch_bc_passes<T, B, 1>(ws, s, M + c0 * ldm, ldm, nc, tr, zp)));
        c0 += nc;
    }
    return CUEV_STATUS_SUCCESS;
}

template <typename T> int bc_back_any(Workspace<T> &ws, hipStream_t s, const T *U, T *M, i64 ldm, bool tr) {
    if (ldm < ws.n) CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "bc_back: ldm < n");
    if (ws.n < 3) return CUEV_STATUS_SUCCESS;
    switch (ws.b) {
    case 16: return launch_bc_back<T, 16>(ws, s, U, M, ldm, tr);
    case 32: return launch_bc_back<T, 32>(ws, s, U, M, ldm, tr);
    case 64: return launch_bc_back<T, 64>(ws, s, U, M, ldm, tr);
    default: CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "bc_back: unsupported b=%d", ws.b);
    }
}

// What for the block of panels i .. i+np-1 into ws.Z (rows r0 = i+b .., ld ws.ld)
template <typename T>
int build_what(Workspace<T> &ws, hipStream_t s, const T *Y, const T *W, int i, int np, Scratch gs) {
    const int n = ws.n, b = ws.b;
    const i64 ld = ws.ld;
    const int r0 = i + b;
    const i64 R0 = n - r0;
    T *Wh = ws.Z + r0;
    for (int t = 0; t < np; ++t) {
        const int j = i + t * b, rt = j + b; // panel t: columns j.., rows rt..
        T *Wt = ws.Z + (i64)t * b * ld;
        CUEV_TRY(fill2d<T>(s, Wt + r0, ld, rt - r0, b, T(0), T(0)));
        CUEV_TRY(copy2d<T>(s, W + (i64)j * ld + rt, ld, Wt + rt, ld, n - rt, b));
        if (t == 0) continue;
        // C = Yhat_{0:t}^T W_t over rows rt.. (where W_t lives), t b x b
        CUEV_TRY(gemm<T>(s, 1, 0, (i64)t * b, b, n - rt, T(1), Y + (i64)i * ld + rt, ld,
                         W + (i64)j * ld + rt, ld, T(0), ws.Dwk, (i64)t * b, gs));
        // What_t -= What_{0:t} C over rows r0..
        CUEV_TRY(gemm<T>(s, 0, 0, R0, b, (i64)t * b, T(-1), Wh, ld, ws.Dwk, (i64)t * b, T(1), Wt + r0,
                         ld, gs));
    }
    return CUEV_STATUS_SUCCESS;
}

// Yhat of the same block into ws.Yh: its panels' Y with zeros above each (Y holds nothing defined there)
template <typename T> int build_yhat(Workspace<T> &ws, hipStream_t s, const T *Y, int i, int np) {
    const int n = ws.n, b = ws.b, r0 = i + b;
    const i64 ld = ws.ld;
    for (int t = 0; t < np; ++t) {
        const int j = i + t * b, rt = j + b;
        T *Yt = ws.Yh + (i64)t * b * ld;
        CUEV_TRY(fill2d<T>(s, Yt + r0, ld, rt - r0, b, T(0), T(0)));
        CUEV_TRY(copy2d<T>(s, Y + (i64)j * ld + rt, ld, Yt + rt, ld, n - rt, b));
    }
    return CUEV_STATUS_SUCCESS;
}

} // namespace

template <typename T> int bc_back(Workspace<T> &ws, const T *U, T *M, i64 ldm) {
    return bc_back_any<T>(ws, ws.stream, U, M, ldm, false);
}

template <typename T> int bc_back_t(Workspace<T> &ws, hipStream_t s, const T *U, T *M, i64 ldm) {
    return bc_back_any<T>(ws, s, U, M, ldm, true);
}

template <typename T> int sbr_back(Workspace<T> &ws, const T *Y, const T *W, T *M, i64 ldm) {
    const int n = ws.n, b = ws.b, k = ws.k;
    const i64 ld = ws.ld;
    if (ldm < n) CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "sbr_back: ldm < n");
    Scratch gs{ws.gscratch, ws.gscratch_bytes};
    hipStream_t s = ws.stream;
    // Blocks of the reduction (k columns, np = k/b panels), last block first. Block
    // i applies H_i0 H_i1 ... = I - What Yhat^T with Yhat = [Y_i0 .. Y_inp-1] and
    // What built left to right: What_t = W_t - What_{0:t} (Yhat_{0:t}^T W_t)
    // (what panel t's W becomes once the earlier panels' reflectors are folded in).
    // Then Zt = Yhat^T M and M -= What Zt, one product each over the block's rows: a product per
    // panel, over that panel's rows only, spares np b^2 n / 2 multiplications but reads M np times
    // (FP64, n = 16384: 184 -> 163 ms, n = 8192: 30 -> 26).
    int ilast = -1;
    for (int i = 0; i + b < n; i += k) ilast = i;
    for (int i = ilast; i >= 0; i -= k) {
        int np = 0;
        while (np * b < k && i + np * b + b < n) ++np;
        const int r0 = i + b; // first row of the block's reflectors
        const i64 R0 = n - r0;
        {
            prof::Scope sc(s, "bt.sbr_what");
            CUEV_TRY(build_what<T>(ws, s, Y, W, i, np, gs));
            CUEV_TRY(build_yhat<T>(ws, s, Y, i, np));
        }
        prof::Scope sc(s, "bt.sbr_back", 4.0 * (double)R0 * np * b * n);
        CUEV_TRY(gemm<T>(s, 1, 0, (i64)np * b, n, R0, T(1), ws.Yh + r0, ld, M + r0, ldm, T(0), ws.Zt, k, gs));
        CUEV_TRY(gemm<T>(s, 0, 0, R0, n, (i64)np * b, T(-1), ws.Z + r0, ld, ws.Zt, k, T(1), M + r0, ldm,
                         gs));
    }
    return CUEV_STATUS_SUCCESS;
}

template <typename T>
int sbr_back_t(Workspace<T> &ws, hipStream_t s, const T *Y, const T *W, T *M, i64 ldm) {
    const int n = ws.n, b = ws.b, k = ws.k;
    const i64 ld = ws.ld;
    if (ldm < n) CUEV_FAIL(CUEV_STATUS_INVALID_ARGUMENT, "sbr_back_t: ldm < n");
    Scratch gs{ws.gscratch, ws.gscratch_bytes};
    // M = Q_s^T = Q_T^T ... Q_1^T Q_0^T with Q_t^T = I - Yhat_t What_t^T for the
    // reduction's blocks t (Yhat the block's Y columns, zero above each panel's rows,
    // copied into ws.Yh since Y there holds nothing defined). Built from the right,
    // last block first: M = I, then M <- M Q_t^T = M - (M Yhat_t) What_t^T for
    // t = T .. 0. Before block t, M differs from I only in its trailing block from
    // row and column r0_t + k on, and Yhat_t, What_t vanish above row r0_t, so the
    // update touches the trailing (n - r0_t)^2 block alone:
    //   P = M[r0:, r0:] Yhat_t[r0:],   M[r0:, r0:] -= P What_t[r0:]^T
    // (4/3 n^3 flops in all, against 2 n^3 for applying the blocks from the left to
    // every column).
    CUEV_TRY(fill2d<T>(s, M, ldm, n, n, T(0), T(1)));
    int nblk = 0;
    for (int i = 0; i + b < n; i += k) ++nblk;
    for (int bi = nblk - 1; bi >= 0; --bi) {
        const int i = bi * k;
        int np = 0;
        while (np * b < k && i + np * b + b < n) ++np;
        const int r0 = i + b;
        const i64 R0 = n - r0, kb = (i64)np * b;
        {
            prof::Scope sc(s, "bt.sbr_what");
            CUEV_TRY(build_what<T>(ws, s, Y, W, i, np, gs));
            CUEV_TRY(build_yhat<T>(ws, s, Y, i, np));
        }
        prof::Scope sc(s, "bt.sbr_back", 4.0 * (double)R0 * R0 * kb);
        T *Mt = M + r0 + (i64)r0 * ldm;
        // P (R0 x kb, ld n) in ws.Zt, which holds k x n elements
        CUEV_TRY(gemm<T>(s, 0, 0, R0, kb, R0, T(1), Mt, ldm, ws.Yh + r0, ld, T(0), ws.Zt, n, gs));
        CUEV_TRY(gemm<T>(s, 0, 1, R0, R0, kb, T(-1), ws.Zt, n, ws.Z + r0, ld, T(1), Mt, ldm, gs));
    }
    return CUEV_STATUS_SUCCESS;
}

template int bc_back<float>(Workspace<float> &, const float *, float *, i64);
template int bc_back<double>(Workspace<double> &, const double *, double *, i64);
template int bc_back_t<float>(Workspace<float> &, hipStream_t, const float *, float *, i64);
template int bc_back_t<double>(Workspace<double> &, hipStream_t, const double *, double *, i64);
template int sbr_back_t<float>(Workspace<float> &, hipStream_t, const float *, const float *, float *, i64);
template int sbr_back_t<double>(Workspace<double> &, hipStream_t, const double *, const double *, double *,
                                i64);
template int sbr_back<float>(Workspace<float> &, const float *, const float *, float *, i64);
template int sbr_back<double>(Workspace<double> &, const double *, const double *, double *, i64);

} // namespace cuev
