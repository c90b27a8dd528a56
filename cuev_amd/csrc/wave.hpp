// wave.hpp — exchanges between the lanes of a wave64 by DPP and permlane swaps (no LDS
// round trip), for the latency-bound kernels.
#pragma once

#include "common.hpp"

#if defined(__HIPCC__)
namespace cuev {

template <int CTRL> __device__ __forceinline__ float dpp_mov(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL> __device__ __forceinline__ double dpp_mov(double v) {
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true));
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E, kHalfMirror = 0x141, kRowRor8 = 0x128;

// upper half of a <-> lower half of b, of the 64 lanes (32) or of each 32 lanes (16)
template <int W> __device__ __forceinline__ void lane_swap(unsigned &a, unsigned &b) {
    if constexpr (W == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        a = r[0];
        b = r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = r[0];
        b = r[1];
    }
}
template <int W> __device__ __forceinline__ void lane_swap(float &a, float &b) {
    unsigned x = __float_as_uint(a), y = __float_as_uint(b);
    lane_swap<W>(x, y);
    a = __uint_as_float(x);
    b = __uint_as_float(y);
}
template <int W> __device__ __forceinline__ void lane_swap(double &a, double &b) {
    unsigned xl = (unsigned)__double2loint(a), xh = (unsigned)__double2hiint(a);
    unsigned yl = (unsigned)__double2loint(b), yh = (unsigned)__double2hiint(b);
    lane_swap<W>(xl, yl);
    lane_swap<W>(xh, yh);
    a = __hiloint2double((int)xh, (int)xl);
    b = __hiloint2double((int)yh, (int)yl);
}

// sums over groups of 8 lanes, of B lanes: every lane gets its group's total
template <typename V> __device__ __forceinline__ V sum8(V v) {
    v += dpp_mov<kQuadXor1>(v);
    v += dpp_mov<kQuadXor2>(v);
    v += dpp_mov<kHalfMirror>(v);
    return v;
}
template <int B, typename V> __device__ __forceinline__ V group_sum(V v) {
    v = sum8(v);
    v += dpp_mov<kRowRor8>(v);
    if constexpr (B >= 32) {
        V a = v, b = v;
        lane_swap<16>(a, b);
        v = a + b;
    }
    if constexpr (B >= 64) {
        V a = v, b = v;
        lane_swap<32>(a, b);
        v = a + b;
    }
    return v;
}
__device__ __forceinline__ float read_lane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double read_lane(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

// sqrt(h) and 1 / sqrt(h), h in [2^-1000, 2^1000]: v_rsq_f64, two Newton steps
__device__ __forceinline__ void fast_sqrt(double h, double &r, double &ri) {
    double y = __builtin_amdgcn_rsq(h);
    y = fma(0.5 * y, fma(-h * y, y, 1.0), y);
    const double t = h * y;
    r = fma(0.5 * y, fma(-t, t, h), t);
    ri = fma(y, fma(-r, y, 1.0), y);
}

} // namespace cuev
#endif
