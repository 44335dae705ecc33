// Host half of the locality ordering: plain C++, so that it can be compiled and tested without a device.
#ifndef TSNE_HIP_LOCALITY_CHAIN_H_
#define TSNE_HIP_LOCALITY_CHAIN_H_

#include <cstddef>
#include <cstdint>
#include <limits>
#include <vector>

namespace tsnehip {

// Greedy chain over M pivots (rows: M x D): starts at pivot 0 and always continues with the nearest pivot not yet
// placed, or, where no distance from the last one is a finite number (a row with a NaN or an infinity), with the first
// of them.  Returns the place of every pivot, a permutation of 0 .. M - 1 whatever the rows hold.
inline std::vector<int> chain_pivots(const float *rows, int M, int D) {
    std::vector<int> place(M, -1);
    int cur = 0;
    for (int pos = 0; pos < M; ++pos) {
        place[cur] = pos;
        double best = std::numeric_limits<double>::infinity();
        int next = -1, first = -1;
        for (int j = 0; j < M; ++j) {
            if (place[j] >= 0) continue;
            if (first < 0) first = j;
            double d2 = 0.0;
            for (int d = 0; d < D; ++d) {
                const double diff = (double)rows[(size_t)cur * D + d] - (double)rows[(size_t)j * D + d];
                d2 += diff * diff;
            }
            if (d2 < best) {
                best = d2;
                next = j;
            }
        }
        cur = next >= 0 ? next : first;
    }
    return place;
}

// Stable counting sort of N points by the place of their pivot (labels: a pivot in [0, place.size()) per point, or
// negative: no pivot is at a finite distance, the point goes with pivot 0).  Whether no label is negative.
inline bool order_by_place(const int *labels, int N, const std::vector<int> &place, int *order) {
    std::vector<int64_t> start(place.size() + 1, 0);
    bool all_near = true;
    for (int i = 0; i < N; ++i) {
        all_near = all_near && labels[i] >= 0;
        start[place[labels[i] < 0 ? 0 : labels[i]] + 1] += 1;
    }
    for (size_t c = 0; c < place.size(); ++c) start[c + 1] += start[c];
    for (int i = 0; i < N; ++i) order[start[place[labels[i] < 0 ? 0 : labels[i]]]++] = i;
    return all_near;
}

}  // namespace tsnehip

#endif  // TSNE_HIP_LOCALITY_CHAIN_H_
