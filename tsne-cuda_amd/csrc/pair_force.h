// The attractive force of one stored pair, and how forces over a prepared pattern are summed (gfx950).  The kernels that
// hold an entry in several pieces (attractive.hip, attractive_blocked.hip) spell the force out: the same operations.
#ifndef TSNE_HIP_PAIR_FORCE_H_
#define TSNE_HIP_PAIR_FORCE_H_

#include "common.h"

namespace tsnehip {

constexpr double kRoundMagic = 6755399441055744.0;  // 1.5 * 2^52: adding it rounds a double to an integer

#ifdef __HIPCC__
// p (y_i - y_j) / (1 + |y_i - y_j|^2)
__device__ __forceinline__ float2 pair_force(float p, float2 yi, float2 yj) {
    const float dx = yi.x - yj.x, dy = yi.y - yj.y;
    const float w = p * __builtin_amdgcn_rcpf(1.0f + dx * dx + dy * dy);
    return make_float2(w * dx, w * dy);
}

// A contribution is below p_max / 2, so that this scale keeps each below 2^50 and a row's sum in 64 bits.
__device__ __forceinline__ double force_scale(float p_max) {
    return p_max > 0.0f ? 2251799813685248.0 / (double)p_max : 1.0;  // 2^51 / p_max
}

// magic + v * scale is a double in [2^52, 2^53), where doubles are the integers: its bit pattern is the
// magic's plus round(v * scale).  The patterns themselves are summed; every row has exactly K entries, so
// its accumulators start at -K times the magic's pattern (mod 2^64) and end at the sum of the integers.
__device__ __forceinline__ unsigned long long fixed_force(float v, double scale) {
    return (unsigned long long)__double_as_longlong(fma((double)v, scale, kRoundMagic));
}
__device__ __forceinline__ unsigned long long fixed_force_start(int K) {
    return 0ull - (unsigned long long)K * (unsigned long long)__double_as_longlong(kRoundMagic);
}
#endif  // __HIPCC__

}  // namespace tsnehip

#endif  // TSNE_HIP_PAIR_FORCE_H_
