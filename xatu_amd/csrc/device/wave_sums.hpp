// Sums over the lanes of a wave by DPP moves: a few cycles a step where a shuffle through LDS takes
// its latency.
#pragma once
#include <hip/hip_runtime.h>

namespace xatu_dev {

// Cross-lane moves of a double by DPP (two 32-bit halves); lanes whose row is outside
// row_mask receive 0.
template <int kCtrl, int kRowMask = 0xF>
__device__ inline double dpp(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), kCtrl, kRowMask, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), kCtrl, kRowMask, 0xF, false);
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}
template <int kCtrl, int kRowMask = 0xF>
__device__ inline float dpp(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, kRowMask, 0xF, false));
}
__device__ inline double lane63(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane(static_cast<int>(b), 63);
    const int hi = __builtin_amdgcn_readlane(static_cast<int>(b >> 32), 63);
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}
__device__ inline float lane63(float x) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63)); }
constexpr int kDppXor1 = 0xB1;        // quad_perm [1, 0, 3, 2]
constexpr int kDppXor2 = 0x4E;        // quad_perm [2, 3, 0, 1]
constexpr int kDppHalfMirror = 0x141; // lane i <-> 7 - i within 8
constexpr int kDppMirror = 0x140;     // lane i <-> 15 - i within 16
constexpr int kDppBcast15 = 0x142;    // lane 15 of a row to the next row
constexpr int kDppBcast31 = 0x143;    // lane 31 to rows 2 and 3

// Sum over the 8 lanes l ^ 0..7 (every lane of the group receives it).
template <typename T>
__device__ inline T sum8(T x) {
    x += dpp<kDppXor1>(x);
    x += dpp<kDppXor2>(x);
    x += dpp<kDppHalfMirror>(x);
    return x;
}
// Sum over the 16 lanes of a DPP row (every lane of the row receives it).
template <typename T>
__device__ inline T sum16_row(T x) {
    x = sum8(x);
    x += dpp<kDppMirror>(x);
    return x;
}
// Sum over the wave of a value that is the same within groups of 8 lanes: one term per group.
template <typename T>
__device__ inline T wave_sum_groups8(T x) {
    x += dpp<kDppMirror>(x);             // two groups, every lane of a row of 16
    x += dpp<kDppBcast15, 0xA>(x);       // rows 1, 3 += rows 0, 2
    x += dpp<kDppBcast31, 0xC>(x);       // rows 2, 3 += row 1
    return lane63(x);
}
// Sum over the wave, the same in every lane.
template <typename T>
__device__ inline T wave_sum(T x) { return wave_sum_groups8(sum8(x)); }

// Inclusive prefix sum over the lanes of the wave (shifts by 1, 2, 4 and 8 within the rows of 16, then
// the rows' ends broadcast).
__device__ inline double wave_scan(double x) {
    x += dpp<0x111>(x);
    x += dpp<0x112>(x);
    x += dpp<0x114>(x);
    x += dpp<0x118>(x);
    x += dpp<kDppBcast15, 0xA>(x);
    x += dpp<kDppBcast31, 0xC>(x);
    return x;
}

}  // namespace xatu_dev
