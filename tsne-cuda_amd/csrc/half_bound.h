// The rounding bound of the neighbour search's sweeps on halves (knn.hip): what is subtracted from a distance of such a
// sweep to make it a lower bound.  By itself, so that a test can compile it for the host.
#ifndef TSNE_HIP_HALF_BOUND_H_
#define TSNE_HIP_HALF_BOUND_H_

#include <cmath>

#ifdef __HIPCC__
#define TSNE_HALF_BOUND __host__ __device__ __forceinline__
#else
#define TSNE_HALF_BOUND inline
#endif

namespace tsnehip {

constexpr float kLeastNormal = 1.17549435e-38f;  // 2^-126: more than an operation that underflows is off by

// Upper bound of a vector's length from the sum of its D squares in fp32.  Squares below 2^-126 lose bits or vanish, so
// that much is added for each.  (Without it a point whose coordinates lie about 1e-19 from their frame's appears to lose
// nothing as halves, and keys exceed distances: by 2 % at 2e-20 in five dimensions.)
TSNE_HALF_BOUND float length_bound(float sum_of_squares, int D) {
    return sqrtf(sum_of_squares + (float)D * kLeastNormal) * (1.0f + 1e-3f);
}

// A query's side of the bound.
//  - q' and x' are kept as halves: |q'.x' - (their halves)| <= |q'| e_x + e_q (|x'| + e_x), e what the halves lose;
//  - D products are accumulated in fp32 onto -beta / 2, in the matrix unit's order, and beta itself is a sum of D
//    rounded terms: 5 (D + 8) 2^-24 (the factor covers that order) times the magnitudes, 2 |q'||x'| + |x'|^2 + 2 |f - c||x'|;
//  - |q - c|^2 is a sum of D rounded terms too, (|q'| + |f - c|)^2 at most, taken in a known order: 1.25 (D + 8) 2^-24;
//  - what underflows on the way: fewer than 8 D + 20 operations on distances and D + 2 on products, which are distances
//    times s^2 / 2 (s: the halves' scale), and the D of the distance that the re-rank forms.
struct HalfQuery {
    float len, eps, kap;      // |q'|, what its halves lose, 5 (D + 8) 2^-24
    float least;              // what may underflow
    float off, frame_len;     // lower bound of |q - c|^2, and |f - c|, of the candidate frame at hand
    int frame;                // that frame (-1: none yet)
};
// (back: -2 / s^2, a distance per product)
TSNE_HALF_BOUND HalfQuery half_query(float len, float eps, int D, float back) {
    return {len, eps, 5.0f * (float)(D + 8) * 5.9604644775390625e-08f,
            (16.0f * (float)D + 64.0f) * kLeastNormal * fmaxf(1.0f, -back), 0.0f, 0.0f, -1};
}
// (d2, frame_len: |f - c|^2, and length_bound of it)
TSNE_HALF_BOUND void enter_frame(HalfQuery &hq, int frame, float beta_q, float d2, float frame_len) {
    hq.frame = frame;
    hq.frame_len = frame_len;
    const float reach = hq.len + hq.frame_len;
    hq.off = beta_q + d2 - 0.25f * hq.kap * reach * reach - hq.least;
}
// |q - c|^2 less the bound for a tile (its tile_info).
TSNE_HALF_BOUND float tile_offset(const HalfQuery &hq, float tile_eps, float tile_len) {
    const float split = hq.len * tile_eps + hq.eps * (tile_len + tile_eps);
    const float sums = tile_len * (2.0f * hq.len + tile_len + 2.0f * hq.frame_len);
    return hq.off - (2.02f * split + hq.kap * sums);
}

}  // namespace tsnehip

#endif  // TSNE_HIP_HALF_BOUND_H_
