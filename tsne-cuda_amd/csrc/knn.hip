// Exact brute-force k nearest neighbours for gfx950.
//
// Stands in for the FAISS IVF-Flat search of the reference
// (src/util/distance_utils.cu:79-121), which is approximate; this one is exact
// and reproducible: the squared distance of a pair is accumulated in fp32 over
// ascending dimension with one fused multiply-add per dimension ("canonical"
// distance), neighbours are ordered by (distance, index), and the point itself
// is forced into slot 0 with distance exactly 0 (the perplexity search depends
// on that, src/kernels/perplexity_search.cu:30-32).
//
// Two sweeps share the selection machinery (a per-query candidate list filtered
// against the query's current k-th best and compacted by an LDS bitonic sort):
//
//  * VALU sweep: canonical distances directly, 64 queries x 128-candidate tiles,
//    4 x 8 register block per thread.  Exact by construction; any dimension.
//
//  * MFMA sweep (up to 126 dimensions): v_mfma_f32_32x32x2f32 evaluates
//    |c|^2 - 2 q.c for 32 candidates x 32 queries at a time.  The queries are
//    the B operand and stay in registers for the whole sweep (scaled by -2,
//    with one extra dimension that multiplies the candidate's |c|^2 by 1); the
//    candidates stream through LDS in the A operand's lane layout.  A lane owns
//    one query column of the 32 x 32 result, so filtering is a min over its 16
//    accumulators against one threshold register.  These distances are only
//    approximate (cancellation), so the sweep keeps K' > K candidates; a second
//    kernel recomputes their canonical distances, sorts, and proves that nothing
//    outside the list can belong to the top K: every discarded candidate has an
//    approximate distance >= tau (the K'-th best), hence a canonical distance
//    >= tau - g for a rigorous rounding bound g, and the query passes when its
//    K-th canonical distance is below that.  Queries that do not pass are redone
//    by the VALU sweep, so the result is exact either way.
//    By default the products run on halves relative to a few frames that the
//    tiles are spread over (v_mfma_f32_32x32x16_f16, one product;
//    knn_half_sweep_kernel, and the chunked sweep below), with the distances less
//    a rigorous bound of what that loses as keys.  Where that bound is much larger
//    than the next one's, or more than a few queries fail because of it, and where
//    a caller asks for that sweep, they run on the bf16 matrix pipe
//    (v_mfma_f32_32x32x16_bf16, two bf16 terms per coordinate, three products;
//    not at 126 dimensions):
//    the candidates are stored relative to the centre m of their own 128-point
//    tile, which keeps what the split leaves out small, |q - m|^2 is added on
//    the vector ALU per (query, tile), and the keys are the distances less the
//    tile's error bound - lower bounds, so the proof above needs no g.
//
//  * Chunked MFMA sweep (more than 126 dimensions): the same products (bf16
//    terms by default), but the queries no longer fit a wave's registers, so
//    both operands stream in chunks of 64 dimensions (32 on bf16 terms; candidates through LDS,
//    queries straight into registers from a pre-scaled packed copy) while the
//    32 x 128 results of a wave accumulate in registers; |q - m|^2 is formed
//    chunk by chunk from the query-side operand and the centre's chunk.  With hundreds of dimensions a query's neighbour
//    distances lie close together and the rounding bound g grows, so the margin
//    K' - K is first tried on a sample of query tiles and doubled until the
//    sample verifies (or the vector sweep is taken instead); the query tiles of
//    the few queries that still fail are swept once more with twice the margin
//    before the vector sweep gets what is left.  Sweeps of few query tiles split
//    every tile's candidates over several workgroups; a merge kernel reduces
//    their lists to what a single list would have kept.
#include "common.h"
#include "half_bound.h"
#include "stages.h"

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <new>
#include <type_traits>
#include <vector>

namespace tsnehip {

namespace {

typedef unsigned long long u64;
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v8f __attribute__((ext_vector_type(8)));
typedef float v32f __attribute__((ext_vector_type(32)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// What the matrix sweeps multiply: floats, two bf16 terms per coordinate, or one half each (see half_pack_kernel).
enum class Products { kFloats, kBf16, kHalf };

constexpr int kQT = 64;   // VALU sweep: queries per workgroup
constexpr int kCT = 128;  // candidates per tile (both sweeps)
constexpr int kDC = 32;   // VALU sweep: dimensions staged per chunk
constexpr int kMQ = 128;  // MFMA sweep: queries per workgroup (4 waves x 32)
constexpr int kMfmaMaxSteps = 64;  // k-steps of 2 dimensions: up to 126 dimensions + 2 augmented
static_assert(kMQ == kCT, "query tiles and candidate tiles share the packed layout");

// From memory to LDS with no register in between: lane l's 16 bytes, at src + its offset, go to dst + 16 l.  The
// compiler knows nothing of the load: s_waitcnt vmcnt(0) and a barrier stand between it and the words' readers, a barrier
// between their last readers and it.  (As a builtin, every read of LDS that follows waits for it.)
// The address is copied here, on the scalar unit: a memory instruction may not read a scalar register within five wait states
// of the vector instruction that wrote it (a readfirstlane of an address, say), and the compiler counts those for instructions
// it knows only.  The copy is also the wait state between M0's writing and its use.  (M0 is a reserved register: naming it tells
// the compiler that it is written, and draws a warning that it would not be saved, which nobody asks for.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
typedef __attribute__((address_space(3))) unsigned char LdsByte;
__device__ __forceinline__ void load_to_lds(const void *src, unsigned int offset, unsigned int dst) {
    const void *at;
    asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 %0, %1\n\tglobal_load_lds_dwordx4 %2, %0" : "=&s"(at) : "s"(src), "v"(offset), "s"(dst) : "memory", "m0");
}
#pragma clang diagnostic pop
// (The builtin: a wait inside inline assembly leaves the compiler waiting once more for loads it knows of, and with them
// for those it does not.)
__device__ __forceinline__ void wait_for_loads() {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    asm volatile("" ::: "memory");
}

// Of a branch, where it stands: the path that is seldom taken is laid out elsewhere, and the other runs straight on.
#define TSNE_LIKELY(c) __builtin_expect(!!(c), 1)
#define TSNE_UNLIKELY(c) __builtin_expect(!!(c), 0)

// v_min3_f32 / v_min_f32 without the quieting moves the library fminf adds for signalling NaNs.
// The compiler's wait states between a matrix instruction and a vector instruction that reads its result do
// not cover instructions inside inline assembly: a chain of these over an accumulator has to start from
// matrix_result(), an ordinary instruction on one of the accumulator's registers, and depend on its value.
__device__ __forceinline__ float min3(float a, float b, float c) {
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float min2(float a, float b) {
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float max2(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// The smaller of three, or the larger (MAX).
template <bool MAX>
__device__ __forceinline__ float extreme3(float a, float b, float c) {
    return MAX ? max3(a, b, c) : min3(a, b, c);
}
template <bool MAX>
__device__ __forceinline__ float extreme2(float a, float b) {
    return MAX ? max2(a, b) : min2(a, b);
}
__device__ __forceinline__ float matrix_result(float x) { return __builtin_canonicalizef(x); }

__device__ __forceinline__ u64 pack_key(float d, int j) {
    return ((u64)float_to_ordered(d) << 32) | (unsigned int)j;
}
// ... of a distance that is not negative (or of -0).
__device__ __forceinline__ u64 pack_key_positive(float d, int j) {
    return ((u64)(__float_as_uint(d) | 0x80000000u) << 32) | (unsigned int)j;
}
__device__ __forceinline__ float key_distance(u64 key) { return ordered_to_float((unsigned int)(key >> 32)); }
__device__ __forceinline__ int key_index(u64 key) { return (int)(unsigned int)(key & 0xffffffffu); }

// Transposed copy of the points, [dim][point], padded to Npad points (vector sweep).
__global__ __launch_bounds__(256) void transpose_points_kernel(const float *__restrict__ X, int N, int D, int Npad,
                                                               float *__restrict__ Xt) {
    __shared__ float tile[32][33];
    const int i0 = blockIdx.x * 32, d0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
    for (int r = ty; r < 32; r += 8) {
        const int i = i0 + r, d = d0 + tx;
        tile[r][tx] = (i < N && d < D) ? X[(size_t)i * D + d] : 0.0f;
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int d = d0 + r, i = i0 + tx;
        if (d < D && i < Npad) Xt[(size_t)d * Npad + i] = tile[tx][r];
    }
}

// |x|^2 of every point (fp32, one fma per dimension) and the largest of them.
__global__ __launch_bounds__(256) void norms_kernel(const float *__restrict__ X, int N, int D, int Npad,
                                                    float *__restrict__ norms, float *__restrict__ max_norm) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    float nrm = 0.0f;
    if (i < N) {
        const float *x = X + (size_t)i * D;
        for (int d = 0; d < D; ++d) nrm = fmaf(x[d], x[d], nrm);
    }
    if (i < Npad) norms[i] = nrm;
    nrm = group_max<kWave>(nrm);
    if ((threadIdx.x & (kWave - 1)) == 0) atomicMax(reinterpret_cast<unsigned int *>(max_norm), __float_as_uint(nrm));
}

// Points in the A-operand layout of v_mfma_f32_32x32x2f32, tile by tile, so that
// a 128-candidate tile is one contiguous run of float4:
//   Xp[tile][block of 32 points (4)][group of 4 k-steps (S4)][lane (64)] float4
// where lane = (dimension % 2) * 32 + point % 32 and component = k-step % 4,
// k-step = dimension / 2.  Dimension Dnorm carries |x|^2, padding is zero.
__global__ __launch_bounds__(256) void pack_points_kernel(const float *__restrict__ X,
                                                          const float *__restrict__ norms, int N, int D, int Dnorm,
                                                          int S4, int Npad, float4 *__restrict__ Xp,
                                                          bool query_side) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // one float4 of Xp per thread
    const int64_t total = (int64_t)Npad * S4 * 2;
    if (t >= total) return;
    const int lane = (int)(t & 63);
    const int64_t rest = t >> 6;
    const int s4 = (int)(rest % S4);
    const int64_t blk = rest / S4;  // tile * 4 + block
    const int i = (int)(blk * 32 + (lane & 31));
    const int h = lane >> 5;
    float v[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int d = 2 * (4 * s4 + c) + h;
        v[c] = 0.0f;
        if (i < N) {
            if (d < D) v[c] = query_side ? -2.0f * X[(size_t)i * D + d] : X[(size_t)i * D + d];
            else if (d == Dnorm) v[c] = query_side ? 1.0f : norms[i];
        }
    }
    Xp[t] = make_float4(v[0], v[1], v[2], v[3]);
}

// Nearest bf16 of a finite float (ties to even), as its 16 bits, and the float such bits stand for.
__device__ __forceinline__ unsigned int bf16_bits(float v) {
    const unsigned int u = __float_as_uint(v);
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ float bf16_value(unsigned int bits) { return __uint_as_float(bits << 16); }

// Points for the bf16 sweep: relative to the centre m of their own tile's bounding ball (small numbers, so
// that what the bf16 terms leave out is small), every coordinate split into two bf16 terms (high = nearest
// bf16, low = nearest bf16 of the rest), in the A-operand layout of v_mfma_f32_32x32x16_bf16.  Per tile
//   [block of 32 points (4)][term (2: high, low)][step of 16 dimensions (S16)][lane (64)] 8 x bf16
// (lane = 32 * (dimension % 16 / 8) + point % 32, element = dimension % 8), then 64 float4 written by
// pack_tile_centres_kernel.  Dimensions D, D + 1 and D + 2 of the high term carry
// beta = |x - m|^2 + 2 m.(x - m) as three bf16 terms (24 bits: the float exactly), so that against the
// query-side operand (-2 q_d, and 1 in those three dimensions) the product is |q - x|^2 - |q - m|^2.
__global__ __launch_bounds__(256) void pack_points_bf16_kernel(const float *__restrict__ X,
                                                               const float *__restrict__ centers_t, int N, int D,
                                                               int S16, int T, int Npad, uint4 *__restrict__ Xb) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // one lane's 8 values per thread
    const int64_t total = (int64_t)Npad * S16 * 4;
    if (t >= total) return;
    const int lane = (int)(t & 63);
    int64_t rest = t >> 6;
    const int s16 = (int)(rest % S16);
    rest /= S16;
    const int term = (int)(rest & 1);
    const int64_t blk = rest >> 1;  // tile * 4 + block
    const int tile = (int)(blk >> 2);
    const int i = (int)(blk * 32 + (lane & 31));
    const int d0 = 16 * s16 + 8 * (lane >> 5);
    unsigned int h[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
    if (i < N) {
        float beta = 0.0f;
        if (term == 0 && d0 + 8 > D && d0 < D + 3) {
            float sq = 0.0f, dot = 0.0f;
            for (int d = 0; d < D; ++d) {
                const float m = centers_t[(size_t)d * T + tile];
                const float delta = X[(size_t)i * D + d] - m;
                sq = fmaf(delta, delta, sq);
                dot = fmaf(m, delta, dot);
            }
            beta = fmaf(2.0f, dot, sq);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int d = d0 + j;
            if (d < D) {
                const float v = X[(size_t)i * D + d] - centers_t[(size_t)d * T + tile];
                const unsigned int hi = bf16_bits(v);
                h[j] = term == 0 ? hi : bf16_bits(v - bf16_value(hi));
            } else if (d < D + 3 && term == 0) {
                float r = beta;
                unsigned int part = bf16_bits(r);
                for (int k = D; k < d; ++k) {
                    r -= bf16_value(part);
                    part = bf16_bits(r);
                }
                h[j] = part;
            }
        }
    }
    const int64_t in_tile = t - (int64_t)tile * (S16 * 512);
    Xb[(int64_t)tile * (S16 * 512 + 64) + in_tile] =
        make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16));
}

// The 64 float4 that close a tile of the bf16 sweep's points: floats 0 .. 16 S16 - 1 the centre m (zero beyond
// D), floats 128 and 129 the tile's error coefficients ga, gb.  A candidate distance the sweep computes for
// a query q against this tile is off by at most |q| ga + gb:
//  - the two bf16 terms leave out, per dimension, low x low and what they do not represent: with u = 2^-8
//    less than 3.1 * 2^-16 |q_d delta_d|, twice that after the factor -2, and sum |q_d delta_d| <= |q| r
//    (r: the ball's radius);
//  - the 3 D + 3 products are accumulated in fp32 in the matrix unit's order: 4 (3 D + 6) 2^-24 (the factor
//    four covers that order) times the sum of the terms' magnitudes, at most 2 |q| r + r^2 + 2 |m| r;
//  - the rounding of x - m, of beta and of the final additions is below a hundredth of the above.
__global__ __launch_bounds__(64) void pack_tile_centres_kernel(const float *__restrict__ centers_t,
                                                               const float *__restrict__ radius, int D, int S16,
                                                               int T, float4 *__restrict__ Xb) {
    const int tile = blockIdx.x, l = threadIdx.x;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (l < 32) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (4 * l + c < D) v[c] = centers_t[(size_t)(4 * l + c) * T + tile];
    } else if (l == 32) {
        float m2 = 0.0f;
        for (int d = 0; d < D; ++d) {
            const float m = centers_t[(size_t)d * T + tile];
            m2 = fmaf(m, m, m2);
        }
        const float r = radius[tile], mlen = sqrtf(m2) * (1.0f + 1e-6f);
        const float split = 6.2f / 65536.0f, acc = 4.0f * (float)(3 * D + 6) * 5.9604644775390625e-08f;
        v[0] = 1.01f * (split + 2.0f * acc) * r;
        v[1] = 1.01f * acc * (r * r + 2.0f * mlen * r) + 1e-30f;
    }
    Xb[(size_t)tile * (S16 * 512 + 64) + S16 * 512 + l] = make_float4(v[0], v[1], v[2], v[3]);
}

// The bf16 operands of the chunked sweep, in its layout [tile][block of 32 points (4)][chunk of 32 dimensions]
// [slot (4)][lane (64)] 8 x bf16 with slot = 2 * term + step (step: 16 dimensions of the chunk; lane and
// element as in pack_points_bf16_kernel).  Candidate side: the points relative to their tile's centre in two
// terms, beta in dimensions D .. D + 2 of the high term.  Query side: -2 x in two terms, 1 in those three.
__global__ __launch_bounds__(256) void pack_points_bf16_chunked_kernel(const float *__restrict__ X,
                                                                       const float *__restrict__ centers_t, int N,
                                                                       int D, int n_chunks, int T, int Npad,
                                                                       uint4 *__restrict__ Xb, bool query_side) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // one lane's 8 values per thread
    const int64_t total = (int64_t)Npad * n_chunks * 8;
    if (t >= total) return;
    const int lane = (int)(t & 63);
    int64_t rest = t >> 6;
    const int slot = (int)(rest & 3);
    rest >>= 2;
    const int chunk = (int)(rest % n_chunks);
    const int64_t blk = rest / n_chunks;  // tile * 4 + block
    const int tile = (int)(blk >> 2);
    const int term = slot >> 1, step = slot & 1;
    const int i = (int)(blk * 32 + (lane & 31));
    const int d0 = 32 * chunk + 16 * step + 8 * (lane >> 5);
    unsigned int h[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
    if (i < N) {
        float beta = 0.0f;
        if (!query_side && term == 0 && d0 + 8 > D && d0 < D + 3) {
            float sq = 0.0f, dot = 0.0f;
            for (int d = 0; d < D; ++d) {
                const float m = centers_t[(size_t)d * T + tile];
                const float delta = X[(size_t)i * D + d] - m;
                sq = fmaf(delta, delta, sq);
                dot = fmaf(m, delta, dot);
            }
            beta = fmaf(2.0f, dot, sq);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int d = d0 + j;
            if (d < D) {
                const float x = X[(size_t)i * D + d];
                const float v = query_side ? -2.0f * x : x - centers_t[(size_t)d * T + tile];
                const unsigned int hi = bf16_bits(v);
                h[j] = term == 0 ? hi : bf16_bits(v - bf16_value(hi));
            } else if (d < D + 3 && term == 0) {
                if (query_side) {
                    h[j] = 0x3f80u;
                } else {
                    float r = beta;
                    unsigned int part = bf16_bits(r);
                    for (int k = D; k < d; ++k) {
                        r -= bf16_value(part);
                        part = bf16_bits(r);
                    }
                    h[j] = part;
                }
            }
        }
    }
    Xb[t] = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16));
}

// Tile centres for the chunked bf16 sweep: centres_p[tile][32 n_chunks] and the two error coefficients of
// pack_tile_centres_kernel in tile_coef[2 tile], [2 tile + 1].  Beyond D the centre is zero, except -1/2 in
// dimensions D .. D + 2: the sweep forms |q - m|^2 from the query-side operand, which holds 1 there and
// stands for -2 q, so those three dimensions add nothing.
__global__ __launch_bounds__(64) void pack_chunked_centres_kernel(const float *__restrict__ centers_t,
                                                                  const float *__restrict__ radius, int D,
                                                                  int n_chunks, int T, float *__restrict__ centres_p,
                                                                  float *__restrict__ tile_coef) {
    const int tile = blockIdx.x, l = threadIdx.x;
    float m2 = 0.0f;
    for (int d = l; d < 32 * n_chunks; d += 64) {
        const float m = d < D ? centers_t[(size_t)d * T + tile] : 0.0f;
        centres_p[(size_t)tile * 32 * n_chunks + d] = d >= D && d < D + 3 ? -0.5f : m;
        m2 = fmaf(m, m, m2);
    }
    m2 = group_sum<kWave>(m2);
    if (l == 0) {
        const float r = radius[tile], mlen = sqrtf(m2) * (1.0f + 1e-5f);
        const float split = 6.2f / 65536.0f, acc = 4.0f * (float)(3 * D + 6) * 5.9604644775390625e-08f;
        tile_coef[2 * tile] = 1.01f * (split + 2.0f * acc) * r;
        tile_coef[2 * tile + 1] = 1.01f * acc * (r * r + 2.0f * mlen * r) + 1e-30f;
    }
}

// Sorts sortbuf[0..cap) ascending (cap a power of two), all 256 threads.
__device__ __forceinline__ void bitonic_sort(u64 *sortbuf, int cap, int tid) {
    for (int k = 2; k <= cap; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int t = tid; t < cap / 2; t += 256) {
                const int lo = ((t & ~(j - 1)) << 1) | (t & (j - 1));
                const int hi = lo | j;
                const bool up = (lo & k) == 0;
                const u64 a = sortbuf[lo], b = sortbuf[hi];
                if ((a > b) == up) {
                    sortbuf[lo] = b;
                    sortbuf[hi] = a;
                }
            }
            __syncthreads();
        }
    }
}

// Bitonic sort of one wave's own keys in LDS (sort_n a power of two, at least 64): no workgroup barrier, a wave's
// LDS operations execute in order and the wavefront fences only keep the compiler from reordering them.
__device__ __forceinline__ void wave_sort(u64 *keys, int sort_n, int lane) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int k = 2; k <= sort_n; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int t = lane; t < sort_n / 2; t += kWave) {
                const int lo = ((t & ~(j - 1)) << 1) | (t & (j - 1));
                const int hi = lo | j;
                const bool up = (lo & k) == 0;
                const u64 a = keys[lo], b = keys[hi];
                if ((a > b) == up) {
                    keys[lo] = b;
                    keys[hi] = a;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
}

// Keeps the `want` best entries of query slot qq and tightens its threshold.
__device__ __forceinline__ void compact_query(u64 *list, int cap, int want, int *cnt, u64 *thr, int qq,
                                              u64 *sortbuf, int tid) {
    const int n = cnt[qq];
    for (int e = tid; e < cap; e += 256) sortbuf[e] = e < n ? list[(size_t)qq * cap + e] : ~0ull;
    __syncthreads();
    bitonic_sort(sortbuf, cap, tid);
    const int keep = min(n, want);
    for (int e = tid; e < keep; e += 256) list[(size_t)qq * cap + e] = sortbuf[e];
    if (tid == 0) {
        cnt[qq] = keep;
        if (n >= want) thr[qq] = sortbuf[want - 1];
    }
    __syncthreads();
}

// Wave-private selection for the matrix sweep, where a query's list, counter and threshold are
// only ever touched by the wave that owns the query.  The sweep never needs its candidates in
// order, only the `want` smallest of them and the distance of the last one kept, so a compaction
// is a radix select on the distance bits, six bits per pass: lane l owns histogram bin l, a wave
// scan finds the bin that holds the want-th smallest.  The bits are taken relative to the smallest
// distance present, which skips the leading bits all keys share.  No workgroup barrier is involved
// (LDS operations of a wave execute in order; the wavefront fences only stop the compiler from
// reordering them), so the other waves keep issuing matrix instructions meanwhile.
__device__ __forceinline__ int wave_inclusive_scan(int v, int lane) {
    // Within the rows of 16 lanes by DPP row shifts (a lane without a source adds 0), then the row totals
    // across the rows by the two row broadcasts (lane 15 of a row to the next row: rows 1 and 3; lane 31 to
    // rows 2 and 3).  Twelve vector instructions; six ds_bpermute round trips through LDS before.
    (void)lane;
    int x = v;
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);   // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);   // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);   // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return x;
}

// list: this query's entries in global memory (n = *cnt of them); buf: cap keys of LDS; hist: 64 words
// of LDS.  Afterwards list[0, min(n, want)) holds the entries kept (in no particular order), *cnt their
// number, and *thr is lowered to (distance of the want-th smallest, all index bits set) when n >= want.
// Returns the number of entries kept.
// With slack > 0 the selection may stop early: once the histogram bin that holds the want-th smallest
// has few enough entries that keeping all of them stays within want + slack, everything up to the
// bin's upper edge is kept and that edge becomes the threshold.  A compaction in the middle of a sweep
// only needs some threshold below which everything was kept; the last one of a query passes slack = 0.
//
// HALVES: the list is two regions of `half` entries, each appended to by one of the query's two lanes
// (entries 0 .. c0-1 of the first, the rest of the *cnt entries in the second); the entries kept go back
// alternately into the two regions (entry p to region p & 1, position p >> 1), so both keep room.
template <bool HALVES = false>
__device__ __forceinline__ int wave_select(u64 *list, int want, int *cnt, u64 *thr, u64 *buf, unsigned int *hist,
                                           int lane, int slack = 0, int half = 0, int c0 = 0) {
    __threadfence_block();  // this wave's appends to the list are complete
    const int n = *cnt;
    if (n < want) return n;
    auto wr = [&](int p, u64 key) {
        if (HALVES) list[(p & 1) * half + (p >> 1)] = key;
        else list[p] = key;
    };
    unsigned int lo = ~0u, hi = 0u;
    // Four loads in flight: the list comes from global memory and a load at a time would cost its latency each.
    auto load_run = [&](const u64 *src, int count, u64 *dst) {
        for (int e0 = lane; e0 < count; e0 += 4 * kWave) {
            u64 key[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) key[u] = src[min(e0 + u * kWave, count - 1)];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = e0 + u * kWave;
                if (e < count) {
                    dst[e] = key[u];
                    const unsigned int bits = (unsigned int)(key[u] >> 32);
                    lo = min(lo, bits);
                    hi = max(hi, bits);
                }
            }
        }
    };
    if (HALVES) {
        load_run(list, c0, buf);
        load_run(list + half, n - c0, buf + c0);
    } else {
        load_run(list, n, buf);
    }
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) {
        lo = min(lo, (unsigned int)__shfl_xor((int)lo, m, kWave));
        hi = max(hi, (unsigned int)__shfl_xor((int)hi, m, kWave));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // Radix select of the want-th smallest value of (bits - lo).
    unsigned int prefix = 0u;
    int rank = want;  // 1-based rank among the keys that match the prefix
    int shift = 32 - __clz((int)(hi - lo));  // significant bits of the range (0 when all distances are equal)
    if (hi == lo) shift = 0;
    while (shift > 0) {
        const int w = shift < 6 ? shift : 6;
        shift -= w;
        hist[lane] = 0u;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        for (int e = lane; e < n; e += kWave) {
            const unsigned int v = (unsigned int)(buf[e] >> 32) - lo;
            if ((unsigned int)((u64)v >> (shift + w)) == prefix) atomicAdd(&hist[(v >> shift) & ((1u << w) - 1u)], 1u);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const int c = (int)hist[lane];
        const int incl = wave_inclusive_scan(c, lane);
        const int b = __ffsll((long long)__ballot(incl >= rank)) - 1;  // some lane qualifies: the last one holds all matches
        rank -= __builtin_amdgcn_readlane(incl - c, b);  // (b is the same in every lane)
        prefix = (prefix << w) | (unsigned int)b;
        if (slack > 0 && shift > 0) {
            const int kept = (want - rank) + __builtin_amdgcn_readlane(c, b);  // below the bin + the whole bin
            if (kept <= want + slack) {
                // Keep everything up to the upper edge of the bin.
                const u64 edge = (u64)lo + ((((u64)prefix + 1ull) << shift) - 1ull);
                const unsigned int dedge = edge > 0xffffffffull ? 0xffffffffu : (unsigned int)edge;
                int base = 0;
                const u64 below_lanes = (1ull << lane) - 1ull;
                for (int e0 = 0; e0 < n; e0 += kWave) {
                    const int e = e0 + lane;
                    const u64 key = e < n ? buf[e] : 0ull;
                    const bool keep = e < n && (unsigned int)(key >> 32) <= dedge;
                    const u64 m = __ballot(keep);
                    if (keep) wr(base + __popcll(m & below_lanes), key);
                    base += __popcll(m);
                }
                if (lane == 0) {
                    *cnt = base;
                    *thr = ((u64)dedge << 32) | 0xffffffffull;
                }
                __threadfence_block();
                return base;
            }
        }
    }
    const unsigned int dstar = lo + prefix;
    // Keep everything below dstar and the first `rank` entries equal to it.
    const int need_eq = rank, c_lt = want - rank;
    int base_lt = 0, base_eq = 0;
    const u64 below = (1ull << lane) - 1ull;
    for (int e0 = 0; e0 < n; e0 += kWave) {
        const int e = e0 + lane;
        const u64 key = e < n ? buf[e] : 0ull;
        const unsigned int bits = (unsigned int)(key >> 32);
        const bool lt = e < n && bits < dstar, eq = e < n && bits == dstar;
        const u64 m_lt = __ballot(lt), m_eq = __ballot(eq);
        if (lt) wr(base_lt + __popcll(m_lt & below), key);
        if (eq) {
            const int k = base_eq + __popcll(m_eq & below);
            if (k < need_eq) wr(c_lt + k, key);
        }
        base_lt += __popcll(m_lt);
        base_eq += __popcll(m_eq);
    }
    if (lane == 0) {
        *cnt = want;
        *thr = ((u64)dstar << 32) | 0xffffffffull;
    }
    __threadfence_block();
    return want;
}

// Smallest (MIN) or largest of a value over the wave, in every lane, by DPP (see wave_inclusive_scan).
template <bool MIN>
__device__ __forceinline__ unsigned int wave_extreme(unsigned int v) {
    constexpr unsigned int none = MIN ? ~0u : 0u;
    auto step = [](unsigned int a, unsigned int b) { return MIN ? min(a, b) : max(a, b); };
    v = step(v, (unsigned int)__builtin_amdgcn_update_dpp((int)none, (int)v, 0x111, 0xf, 0xf, false));
    v = step(v, (unsigned int)__builtin_amdgcn_update_dpp((int)none, (int)v, 0x112, 0xf, 0xf, false));
    v = step(v, (unsigned int)__builtin_amdgcn_update_dpp((int)none, (int)v, 0x114, 0xf, 0xf, false));
    v = step(v, (unsigned int)__builtin_amdgcn_update_dpp((int)none, (int)v, 0x118, 0xf, 0xf, false));
    v = step(v, (unsigned int)__builtin_amdgcn_update_dpp((int)none, (int)v, 0x142, 0xa, 0xf, false));
    v = step(v, (unsigned int)__builtin_amdgcn_update_dpp((int)none, (int)v, 0x143, 0xc, 0xf, false));
    return (unsigned int)__builtin_amdgcn_readlane((int)v, kWave - 1);
}

// wave_select over a list of at most 64 NK entries that the wave holds in registers (load_halves): the want-th smallest
// distance is found by counting how many lie below a trial value (a ballot per register), trial values by interpolation
// between the counts at either end and by halving in turn.  The list is two regions of `half` entries, c0 and n - c0 of
// them in use; the entries kept go back alternately into the two (entry p to region p & 1, position p >> 1).  Keeps the
// `want` smallest, or with slack > 0 any want .. want + slack smallest; lowers *thr to a value that everything kept is
// within and everything dropped at or beyond.  Fewer than `want` entries: all kept, dealt out afresh.
// counted: the rank is taken among the entries without kNotCounted; fewer than `want` of those: all entries kept.
// (A wave's loads find what its stores before them wrote: nothing is waited for but the loads themselves.)
constexpr u64 kNotCounted = 0x80000000ull;  // in a key's point number
template <int NK>
__device__ __forceinline__ void load_halves(const u64 *list, int half, int c0, int n, int lane, u64 (&key)[NK]) {
#pragma unroll
    for (int u = 0; u < NK; ++u) {
        const int e = u * kWave + lane;
        key[u] = ~0ull;
        if (e < n) key[u] = list[e < c0 ? e : half + e - c0];
    }
}
// A value that at least `want` of the wave's `ranked` rated words (of 64 NK; all bits set: not rated) do not exceed, and, but
// for equal ones, at most want + slack.  at_under: how many lie below it, at_hi: how many do not exceed it.
template <int NK>
__device__ __forceinline__ unsigned int ranked_limit(const unsigned int (&rated)[NK], int ranked, int want, int slack,
                                                     int &at_under, int &at_hi) {
    unsigned int lo = ~0u, hi = 0u;
#pragma unroll
    for (int u = 0; u < NK; ++u) {
        lo = min(lo, rated[u]);
        hi = max(hi, rated[u] == ~0u ? 0u : rated[u]);
    }
    lo = wave_extreme<true>(lo);
    hi = wave_extreme<false>(hi);
    // Fewer than `want` lie below or at `lo - 1` (at_under of them), at least `want` at or below hi (at_hi of them).
    unsigned int under = lo - 1u;
    at_under = 0;
    at_hi = ranked;
    for (int round = 0; at_hi > want + slack && hi - under > 1u; ++round) {
        const float share = (round & 1) ? 0.5f : (float)(want + slack / 2 - at_under) * __builtin_amdgcn_rcpf((float)(at_hi - at_under));
        const unsigned int span = hi - under;
        unsigned int step = (unsigned int)((float)span * share);
        step = min(max(step, 1u), span - 1u);
        const unsigned int trial = __builtin_amdgcn_readfirstlane(under + step);
        int c = 0;
#pragma unroll
        for (int u = 0; u < NK; ++u) c += __popcll(__ballot(rated[u] <= trial));
        if (c >= want) {
            hi = trial;
            at_hi = c;
        } else {
            under = trial;
            at_under = c;
        }
    }
    return hi;
}
template <int NK>
__device__ __forceinline__ int select_halves(u64 *list, int want, int slack, bool counted, int half, int n, u64 *thr,
                                             int lane, const u64 (&key)[NK]) {
    unsigned int rated[NK];  // distances, the largest number for an entry that is not counted
    int ranked = 0;
#pragma unroll
    for (int u = 0; u < NK; ++u) {
        rated[u] = counted && (key[u] & kNotCounted) ? ~0u : (unsigned int)(key[u] >> 32);
        ranked += __popcll(__ballot(rated[u] != ~0u));
    }
    const u64 below = (1ull << lane) - 1ull;
    unsigned int limit = ~0u;  // distances up to this are kept ...
    int ties = INT_MAX;        // ... of those equal to it so many
    if (ranked >= want) {
        int at_under, at_hi;
        limit = ranked_limit<NK>(rated, ranked, want, slack, at_under, at_hi);
        if (at_hi > want + slack && !counted) ties = want - at_under;  // (equal distances: as many of them as there is room for)
        // (Entries pass up to 4e-7 beyond the threshold of the moment: with fewer than `want` within it, as a rank among
        // few leaves them, the want-th may be one of those.)
        if (lane == 0) *thr = min(*thr, ((u64)limit << 32) | 0xffffffffull);
    }
    int base = 0, equal = 0;
#pragma unroll
    for (int u = 0; u < NK; ++u) {
        const unsigned int bits = (unsigned int)(key[u] >> 32);
        bool keep = u * kWave + lane < n && bits <= limit;
        if (ties != INT_MAX) {
            const u64 eq = __ballot(keep && bits == limit);
            if (keep && bits == limit && equal + __popcll(eq & below) >= ties) keep = false;
            equal += __popcll(eq);
        }
        const u64 m = __ballot(keep);
        const int p = base + __popcll(m & below);
        if (keep) list[(p & 1) * half + (p >> 1)] = key[u];
        base += __popcll(m);
    }
    return base;
}

__device__ __forceinline__ int group_sum_int(int v) {
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) v += __shfl_xor(v, m, kWave);
    return v;
}

// Bounding ball of every tile of kCT consecutive points: the centre is the tile's mean, the
// radius the largest distance of a member to it, inflated by 1e-3 (far more than the fp32
// rounding of the sums) so that it is an upper bound.  centers_t is D x T (dimension-major).
// One workgroup of 128 threads per tile; dynamic LDS: D floats.
__global__ __launch_bounds__(128) void tile_balls_kernel(const float *__restrict__ X, int N, int D, int T,
                                                         float *__restrict__ centers_t, float *__restrict__ radius) {
    extern __shared__ float c[];
    __shared__ float wmax[2];
    const int t = blockIdx.x, tid = threadIdx.x;
    const int first = t * kCT;
    const int count = min(kCT, N - first);
    for (int d = tid; d < D; d += 128) {
        float sum = 0.0f;
        for (int i = 0; i < count; ++i) sum += X[(size_t)(first + i) * D + d];
        sum /= (float)count;
        c[d] = sum;
        centers_t[(size_t)d * T + t] = sum;
    }
    __syncthreads();
    float d2 = 0.0f;
    if (tid < count) {
        const float *x = X + (size_t)(first + tid) * D;
        for (int d = 0; d < D; ++d) {
            const float diff = x[d] - c[d];
            d2 = fmaf(diff, diff, d2);
        }
    }
    d2 = group_max<kWave>(d2);
    if ((tid & (kWave - 1)) == 0) wmax[tid / kWave] = d2;
    __syncthreads();
    if (tid == 0) radius[t] = sqrtf(fmaxf(wmax[0], wmax[1])) * (1.0f + 1e-3f) + 1e-30f;
}

constexpr int kHomeTiles = 8;  // candidate tiles on either side of the query tile that are always swept

// Whether tile t may hold a point closer than sqrt(tmax) to some point of the tile whose ball is
// (qcenter, ra): with c, r the balls, every pair of members is at least |c_a - c_t| - r_a - r_t apart
// (triangle inequality); 1e-3 relative slack on the centre distance, the radii are upper bounds.
// Anything that is not a number keeps the tile.
// Eight loads in flight and two partial sums: one load at a time would cost its latency per dimension
// (any summation order will do, the slack covers the rounding).
__device__ __forceinline__ bool tile_may_matter(const float *qcenter, float ra, const float *__restrict__ centers_t,
                                                const float *__restrict__ radius, int D, int T, int t, float tmax) {
    float s0 = 0.0f, s1 = 0.0f;
    int d = 0;
    for (; d + 8 <= D; d += 8) {
        float c[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) c[u] = centers_t[(size_t)(d + u) * T + t];
#pragma unroll
        for (int u = 0; u < 8; u += 2) {
            const float e0 = qcenter[d + u] - c[u], e1 = qcenter[d + u + 1] - c[u + 1];
            s0 = fmaf(e0, e0, s0);
            s1 = fmaf(e1, e1, s1);
        }
    }
    for (; d < D; ++d) {
        const float diff = qcenter[d] - centers_t[(size_t)d * T + t];
        s0 = fmaf(diff, diff, s0);
    }
    const float lb = sqrtf(s0 + s1) * (1.0f - 1e-3f) - (ra + radius[t]);
    return !(lb > 0.0f && lb * lb > tmax);
}

// ---------------------------------------------------------------------------
// VALU sweep.  qlist == nullptr: queries are 0..N-1; otherwise the nq listed ones.
// Sweeping all queries with tile balls given (bitmap_words > 0), the candidate tiles are visited in
// two phases as in the matrix sweep: the query tile's neighbourhood in the numbering first, then
// only the tiles whose ball may hold a point below the largest k-th distance found so far.  The
// distances here are the canonical ones, so a skipped tile is strictly farther than every threshold.
// Dynamic LDS: cap keys, then D floats (the query tile's ball centre), then the visit bitmap.
//
// slices > 1 (listed queries only): a handful of queries would occupy a handful of workgroups for a sweep over
// all points, so the candidate tiles are cut into `slices` ranges and a (query tile, range) pair is one unit of
// work; each unit leaves its K-1 best keys in slice_keys[(slot * slices + range) * (K-1) ...] (padded with ~0)
// and knn_merge_slices_kernel forms the rows.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void knn_sweep_kernel(const float *__restrict__ Xt, int N, int Npad, int D, int K,
                                                        int cap, u64 *__restrict__ lists, int num_qtiles,
                                                        const int *__restrict__ qlist, int nq,
                                                        int *__restrict__ out_idx, float *__restrict__ out_d,
                                                        const float *__restrict__ centers_t,
                                                        const float *__restrict__ radius, int bitmap_words,
                                                        int slices, u64 *__restrict__ slice_keys) {
    __shared__ __attribute__((aligned(16))) float xq[kDC][kQT];
    __shared__ __attribute__((aligned(16))) float xc[kDC][kCT];
    __shared__ u64 thr[kQT];
    __shared__ int cnt[kQT];
    __shared__ int qid[kQT];
    extern __shared__ u64 sortbuf[];
    float *qcenter = reinterpret_cast<float *>(sortbuf + cap);
    unsigned int *bitmap = reinterpret_cast<unsigned int *>(qcenter + D);
    __shared__ float tmax_part[kQT / kWave];

    const int tid = threadIdx.x;
    const int tq = tid >> 4, tc = tid & 15;
    const int want = K - 1;
    const int T = (N + kCT - 1) / kCT;
    u64 *list = lists + (size_t)blockIdx.x * kQT * cap;

    for (int unit = blockIdx.x; unit < num_qtiles * slices; unit += gridDim.x) {
        const int qt = unit / slices, slice = unit - qt * slices;
        if (tid < kQT) {
            const int slot = qt * kQT + tid;
            thr[tid] = ~0ull;
            cnt[tid] = 0;
            qid[tid] = slot < nq ? (qlist ? qlist[slot] : slot) : -1;
        }
        __syncthreads();
        auto process = [&](int c0) {
            float acc[4][8];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 8; ++b) acc[a][b] = 0.0f;
            for (int d0 = 0; d0 < D; d0 += kDC) {
                const int dn = min(kDC, D - d0);
                __syncthreads();
                for (int e = tid; e < dn * kQT; e += 256) {
                    const int dd = e / kQT, ql = e % kQT;
                    const int q = qid[ql];
                    xq[dd][ql] = q >= 0 ? Xt[(size_t)(d0 + dd) * Npad + q] : 0.0f;
                }
                for (int e = tid; e < dn * (kCT / 4); e += 256) {
                    const int dd = e / (kCT / 4), v = e % (kCT / 4);
                    *reinterpret_cast<float4 *>(&xc[dd][v * 4]) =
                        *reinterpret_cast<const float4 *>(Xt + (size_t)(d0 + dd) * Npad + c0 + v * 4);
                }
                __syncthreads();
                for (int dd = 0; dd < dn; ++dd) {
                    const float4 qv = *reinterpret_cast<const float4 *>(&xq[dd][tq * 4]);
                    const float4 ca = *reinterpret_cast<const float4 *>(&xc[dd][tc * 8]);
                    const float4 cb = *reinterpret_cast<const float4 *>(&xc[dd][tc * 8 + 4]);
                    const float qs[4] = {qv.x, qv.y, qv.z, qv.w};
                    const float cs[8] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
#pragma unroll
                    for (int a = 0; a < 4; ++a)
#pragma unroll
                        for (int b = 0; b < 8; ++b) {
                            const float df = qs[a] - cs[b];
                            acc[a][b] = fmaf(df, df, acc[a][b]);
                        }
                }
            }
            // Filter against the current k-th best of each query.
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const int ql = tq * 4 + a;
                const int q = qid[ql];
                const u64 limit = thr[ql];
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    const int j = c0 + tc * 8 + b;
                    const u64 key = pack_key(acc[a][b], j);
                    if (j < N && q >= 0 && j != q && key < limit) {
                        const int slot = atomicAdd(&cnt[ql], 1);
                        list[(size_t)ql * cap + slot] = key;
                    }
                }
            }
            __syncthreads();
            const int crowded = (tid < kQT) && (cnt[tid] > cap - kCT);
            if (__syncthreads_or(crowded)) {
                for (int ql = 0; ql < kQT; ++ql)
                    if (cnt[ql] > cap - kCT) compact_query(list, cap, want, cnt, thr, ql, sortbuf, tid);
            }
        };
        const bool prune = bitmap_words > 0 && qlist == nullptr;
        const int bt = (qt * kQT) / kCT;  // the ball tile this query tile lies in
        int h0 = prune ? max(bt - kHomeTiles, 0) : 0, h1 = prune ? min(bt + kHomeTiles, T - 1) : T - 1;
        if (slices > 1) {  // this unit's range of the candidate tiles
            h0 = (int)(((long long)T * slice) / slices);
            h1 = (int)(((long long)T * (slice + 1)) / slices) - 1;
        }
        for (int ct = h0; ct <= h1; ++ct) process(ct * kCT);
        if (prune && (h0 > 0 || h1 < T - 1)) {
            // Thresholds from what the neighbourhood held, then the tiles that may still matter.
            for (int ql = 0; ql < kQT; ++ql)
                if (qid[ql] >= 0) compact_query(list, cap, want, cnt, thr, ql, sortbuf, tid);
            for (int w = tid; w < bitmap_words; w += 256) bitmap[w] = 0u;
            for (int d = tid; d < D; d += 256) qcenter[d] = centers_t[(size_t)d * T + bt];
            if (tid < kQT) {
                float v = -INFINITY;
                if (qid[tid] >= 0) {
                    const u64 t = thr[tid];
                    v = t == ~0ull ? INFINITY : key_distance(t);
                    v += 1e-5f * fabsf(v) + 1e-30f;
                }
                v = group_max<kWave>(v);
                if ((tid & (kWave - 1)) == 0) tmax_part[tid / kWave] = v;
            }
            __syncthreads();
            float tmax = tmax_part[0];
#pragma unroll
            for (int w = 1; w < kQT / kWave; ++w) tmax = fmaxf(tmax, tmax_part[w]);
            const float ra = radius[bt];
            for (int t = tid; t < T; t += 256)
                if ((t < h0 || t > h1) && tile_may_matter(qcenter, ra, centers_t, radius, D, T, t, tmax))
                    atomicOr(&bitmap[t >> 5], 1u << (t & 31));
            __syncthreads();
            for (int w = 0; w < bitmap_words; ++w) {
                unsigned int word = bitmap[w];
                while (word) {
                    const int t = w * 32 + __ffs((int)word) - 1;
                    word &= word - 1u;
                    process(t * kCT);
                }
            }
        }
        // Final ordering and output: self first, then the K-1 best others.
        for (int ql = 0; ql < kQT; ++ql) {
            const int q = qid[ql];
            if (q < 0) break;
            compact_query(list, cap, want, cnt, thr, ql, sortbuf, tid);
            if (slices > 1) {
                // (compact_query leaves the sorted keys in sortbuf, ~0 beyond the entries there were)
                u64 *dst = slice_keys + ((size_t)(qt * kQT + ql) * slices + slice) * want;
                for (int e = tid; e < want; e += 256) dst[e] = sortbuf[e];
                __syncthreads();
                continue;
            }
            for (int e = tid; e < K; e += 256) {
                int j = q;
                float d = 0.0f;
                if (e > 0) {
                    const u64 key = sortbuf[e - 1];
                    j = key_index(key);
                    d = key_distance(key);
                }
                out_idx[(size_t)q * K + e] = j;
                out_d[(size_t)q * K + e] = d;
            }
            __syncthreads();
        }
    }
}

// Rows of the listed queries from the keys their `slices` units left: one workgroup per query sorts the
// slices * (K-1) keys (sort_n: that count rounded up to a power of two; dynamic LDS: sort_n keys).
__global__ __launch_bounds__(256) void knn_merge_slices_kernel(const u64 *__restrict__ slice_keys, int slices, int K,
                                                               int sort_n, const int *__restrict__ qlist,
                                                               int *__restrict__ out_idx, float *__restrict__ out_d) {
    extern __shared__ u64 merge_sortbuf[];
    const int tid = threadIdx.x, slot = blockIdx.x, want = K - 1;
    const int q = qlist[slot];
    const int total = slices * want;
    for (int e = tid; e < sort_n; e += 256) merge_sortbuf[e] = e < total ? slice_keys[(size_t)slot * total + e] : ~0ull;
    __syncthreads();
    bitonic_sort(merge_sortbuf, sort_n, tid);
    for (int e = tid; e < K; e += 256) {
        int j = q;
        float d = 0.0f;
        if (e > 0) {
            const u64 key = merge_sortbuf[e - 1];
            j = key_index(key);
            d = key_distance(key);
        }
        out_idx[(size_t)q * K + e] = j;
        out_d[(size_t)q * K + e] = d;
    }
}

// ---------------------------------------------------------------------------
// Direct search (small problems): every canonical distance of a block of query rows is written to memory
// (pair_distances_kernel), then one wave per query reads its row and keeps the K - 1 smallest keys
// (select_row_kernel).  The sweeps above and below give a query tile to one workgroup, which walks all the
// candidates by itself: 47 workgroups at 3000 points, on a chip that holds hundreds.  Here the pairs are spread
// over the chip, and the selection has no barrier.
// ---------------------------------------------------------------------------
constexpr int kDirectDims = 16;  // dimensions staged per chunk

// Distances of rows row0 .. row0 + rows - 1 of Q (NQ x D; rows of `dist`, pitch floats each, pitch a multiple of the
// tile's side 16 R and at least N) to the N rows of X; columns from N on are left as distances to a point at 0.
// A workgroup computes a square tile, R x R distances per thread, both operands staged in LDS a chunk of
// dimensions ahead; same fma chain as everywhere (dimensions past D are zeros on both sides, which leave a sum
// as it is).  Bound by the vector ALU, two instructions per pair and dimension.
//
// MIRROR (Q = X): of the square of the rows' own columns only the tiles on and above the diagonal are formed, and those above
// it are written a second time, mirrored: (a - b)^2 is (b - a)^2, bit for bit, and so are the sums, but for the sign of what
// is not a number, which tells first from last neighbours: a tile with such a distance is formed once more with rows and
// columns exchanged, as if nothing were mirrored.  (Those distances alone, by the threads that have them: 3000 x 64 with a fifth of
// the points not numbers 1.34 ms, every tile formed 0.68.)
template <int R, bool MIRROR>
__global__ __launch_bounds__(256) void pair_distances_kernel(const float *__restrict__ Q, int NQ,
                                                             const float *__restrict__ X, int N, int D, int row0,
                                                             int rows, int pitch, float *__restrict__ dist) {
    constexpr int kSide = 16 * R;
    constexpr int kRow = kSide + 4;              // LDS row: 16-byte aligned, chunk rows off each other's banks
    constexpr int kLoads = kSide * kDirectDims / (4 * 256);  // pieces of four dimensions per thread and operand
    __shared__ __attribute__((aligned(16))) float xs[2][2][kDirectDims][kRow];
    const int tid = threadIdx.x, tq = tid >> 4, tc = tid & 15;
    int q0 = row0 + blockIdx.y * kSide, c0 = blockIdx.x * kSide;
    if (MIRROR && c0 >= row0 && c0 < q0) return;  // (row0 is a multiple of the side)
    const bool wide =
        (D & 3) == 0 && ((reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(Q)) & 15) == 0;
    float4 ahead[2][kLoads];
    auto load = [&](int d0) {
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int u = 0; u < kLoads; ++u) {
                const int e = tid + u * 256, p = (o ? c0 : q0) + (e >> 2), d = d0 + 4 * (e & 3);
                float4 v = {0.0f, 0.0f, 0.0f, 0.0f};
                if (p < (o ? N : NQ) && d < D) {
                    const float *x = (o ? X : Q) + (size_t)p * D + d;
                    if (wide) {
                        v = *reinterpret_cast<const float4 *>(x);
                    } else {
                        v.x = x[0];
                        if (d + 1 < D) v.y = x[1];
                        if (d + 2 < D) v.z = x[2];
                        if (d + 3 < D) v.w = x[3];
                    }
                }
                ahead[o][u] = v;
            }
    };
    auto stage = [&](int buffer) {
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int u = 0; u < kLoads; ++u) {
                const int e = tid + u * 256, p = e >> 2, dd = 4 * (e & 3);
                xs[buffer][o][dd][p] = ahead[o][u].x;
                xs[buffer][o][dd + 1][p] = ahead[o][u].y;
                xs[buffer][o][dd + 2][p] = ahead[o][u].z;
                xs[buffer][o][dd + 3][p] = ahead[o][u].w;
            }
    };
    for (bool mirror = MIRROR && c0 > q0 && c0 < row0 + rows;; mirror = false) {
        float acc[R][R];
#pragma unroll
        for (int a = 0; a < R; ++a)
#pragma unroll
            for (int b = 0; b < R; ++b) acc[a][b] = 0.0f;
        load(0);
        stage(0);
        for (int d0 = 0, buffer = 0; d0 < D; d0 += kDirectDims, buffer ^= 1) {
            const bool more = d0 + kDirectDims < D;
            if (more) load(d0 + kDirectDims);
            // One barrier per chunk: the buffer written below was last read before this barrier.
            __syncthreads();
            const int dn = min(kDirectDims, D - d0);
#pragma unroll 2
            for (int dd = 0; dd < dn; ++dd) {
                float qs[R], cs[R];
#pragma unroll
                for (int a = 0; a < R; a += 4) {
                    const float4 v = *reinterpret_cast<const float4 *>(&xs[buffer][0][dd][tq * R + a]);
                    const float4 w = *reinterpret_cast<const float4 *>(&xs[buffer][1][dd][tc * 4 + 16 * a]);
                    qs[a] = v.x, qs[a + 1] = v.y, qs[a + 2] = v.z, qs[a + 3] = v.w;
                    cs[a] = w.x, cs[a + 1] = w.y, cs[a + 2] = w.z, cs[a + 3] = w.w;
                }
#pragma unroll
                for (int a = 0; a < R; ++a)
#pragma unroll
                    for (int b = 0; b < R; ++b) {
                        const float df = qs[a] - cs[b];
                        acc[a][b] = fmaf(df, df, acc[a][b]);
                    }
            }
            if (more) stage(buffer ^ 1);
        }
        bool exchange = false;
        if (mirror) {
            bool numbers = true;
#pragma unroll
            for (int a = 0; a < R; ++a)
#pragma unroll
                for (int b = 0; b < R; ++b) numbers = numbers && acc[a][b] == acc[a][b];
            exchange = __syncthreads_or(!numbers);  // (ahead of the stores, which a barrier would wait for)
        }
#pragma unroll
        for (int a = 0; a < R; ++a) {
            const int r = q0 - row0 + tq * R + a;
            if (r >= rows) break;
            float *dst = dist + (size_t)r * pitch + c0 + tc * 4;
#pragma unroll
            for (int b = 0; b < R; b += 4)
                *reinterpret_cast<float4 *>(dst + 16 * b) = float4{acc[a][b], acc[a][b + 1], acc[a][b + 2], acc[a][b + 3]};
        }
        if (!mirror) return;
        if (!exchange) {
#pragma unroll
            for (int b = 0; b < R; ++b) {
                const int r = c0 - row0 + tc * 4 + 16 * (b & ~3) + (b & 3);
                if (r >= rows) continue;
                float *dst = dist + (size_t)r * pitch + q0 + tq * R;
#pragma unroll
                for (int a = 0; a < R; a += 4)
                    *reinterpret_cast<float4 *>(dst + a) = float4{acc[a][b], acc[a + 1][b], acc[a + 2][b], acc[a + 3][b]};
            }
            return;
        }
        const int first = q0;
        q0 = c0, c0 = first;
    }
}

// The K - 1 smallest keys (distance, number) of every row of `dist`, in order, after the point itself; one wave
// per row.  First reading: the row is cut into 64 S groups, which leave their minima; the (K-1)-th smallest
// minimum bounds the (K-1)-th smallest distance, because every minimum is an entry of its own.  A group takes
// pieces of four neighbouring entries, S 256 entries apart and one lane further each time, so that points whose
// clusters come in turn (any period) spread over the groups.  Second reading: the entries within the bound (1.4
// (K-1) of them where 64 S is 2 (K-1) and the order is random) go to LDS and are sorted.  If there are more than
// LDS has room for, the (K-1)-th smallest of those that found room is a better bound for another reading; if it
// is no better (many equal distances), the (K-1)-th smallest distance is found bit by bit and the entries equal
// to it are taken by number.  Needs 2 (K-1) <= 64 S.  listed (optional): the point every row is of.
template <int S>
__global__ __launch_bounds__(256) void select_row_kernel(const float *__restrict__ dist, int N, int row0, int rows,
                                                         int pitch, int K, const int *__restrict__ listed,
                                                         int *__restrict__ out_idx, float *__restrict__ out_d) {
    constexpr int kRoom = 128 * S;
    __shared__ u64 keys_all[4][kRoom];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = blockIdx.x * 4 + wave, want = K - 1;
    if (r >= rows) return;  // (no barrier below)
    const int q = listed ? listed[r] : row0 + r;
    u64 *keys = keys_all[wave];
    const float *row = dist + (size_t)r * pitch;
    const float4 *row4 = reinterpret_cast<const float4 *>(row);
    const int n4 = (N + 3) / 4;
    const u64 below = (1ull << lane) - 1ull;

    unsigned int least[S];
#pragma unroll
    for (int s = 0; s < S; ++s) least[s] = ~0u;
    for (int e0 = 0, turn = 0; e0 < n4; e0 += kWave * S, ++turn) {
        float4 v[S];  // (S loads in flight; past the end the last piece again, which is not counted)
#pragma unroll
        for (int s = 0; s < S; ++s) v[s] = row4[min(e0 + s * kWave + ((lane + turn) & (kWave - 1)), n4 - 1)];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int e = e0 + s * kWave + ((lane + turn) & (kWave - 1));
            const float f[4] = {v[s].x, v[s].y, v[s].z, v[s].w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int j = e * 4 + c;
                if (j < N && j != q) least[s] = min(least[s], float_to_ordered(f[c]));
            }
        }
    }
    unsigned int bound = 0u;  // the want-th smallest minimum: the largest value with fewer than `want` below it
    for (int b = 31; b >= 0; --b) {
        const unsigned int trial = bound | (1u << b);
        int c = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) c += __popcll(__ballot(least[s] < trial));
        if (c < want) bound = trial;
    }
    int n = 0;
    for (;;) {
        n = 0;
        for (int e0 = 0; e0 < n4; e0 += 4 * kWave) {
            float4 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = row4[min(e0 + u * kWave + lane, n4 - 1)];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = e0 + u * kWave + lane;
                const float f[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int j = e * 4 + c;
                    const bool in = j < N && j != q && float_to_ordered(f[c]) <= bound;
                    const u64 m = __ballot(in);
                    if (m) {
                        const int p = n + __popcll(m & below);
                        if (in && p < kRoom) keys[p] = pack_key(f[c], j);
                        n += __popcll(m);
                    }
                }
            }
        }
        if (n <= kRoom) break;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        unsigned int better = 0u;  // the want-th smallest distance of the kRoom entries in LDS
        for (int b = 31; b >= 0; --b) {
            const unsigned int trial = better | (1u << b);
            int c = 0;
            for (int p = lane; p < kRoom; p += kWave) c += __popcll(__ballot((unsigned int)(keys[p] >> 32) < trial));
            if (c < want) better = trial;
        }
        if (better == bound) break;
        bound = better;
    }
    if (n > kRoom) {
        unsigned int kth = 0u;
        for (int b = 31; b >= 0; --b) {
            const unsigned int trial = kth | (1u << b);
            int c = 0;
            for (int j = lane; j < N; j += kWave) c += j != q && float_to_ordered(row[j]) < trial;
#pragma unroll
            for (int m = kWave / 2; m > 0; m >>= 1) c += __shfl_xor(c, m, kWave);
            if (c < want) kth = trial;
        }
        int closer = 0;  // entries below the want-th smallest distance
        for (int j = lane; j < N; j += kWave) closer += j != q && float_to_ordered(row[j]) < kth;
#pragma unroll
        for (int m = kWave / 2; m > 0; m >>= 1) closer += __shfl_xor(closer, m, kWave);
        int n_closer = 0, n_equal = 0;
        for (int j0 = 0; j0 < N; j0 += kWave) {
            const int j = j0 + lane;
            const float f = row[min(j, N - 1)];
            const bool valid = j < N && j != q;
            const bool lt = valid && float_to_ordered(f) < kth, eq = valid && float_to_ordered(f) == kth;
            const u64 m_lt = __ballot(lt), m_eq = __ballot(eq);
            if (lt) keys[n_closer + __popcll(m_lt & below)] = pack_key(f, j);
            const int at = closer + n_equal + __popcll(m_eq & below);
            if (eq && at < want) keys[at] = pack_key(f, j);
            n_closer += __popcll(m_lt);
            n_equal += __popcll(m_eq);
        }
        n = want;
    }
    int sort_n = kWave;
    while (sort_n < n) sort_n <<= 1;
    for (int e = n + lane; e < sort_n; e += kWave) keys[e] = ~0ull;
    wave_sort(keys, sort_n, lane);
    for (int e = lane; e < K; e += kWave) {
        out_idx[(size_t)q * K + e] = e == 0 ? q : key_index(keys[e - 1]);
        out_d[(size_t)q * K + e] = e == 0 ? 0.0f : key_distance(keys[e - 1]);
    }
}

// ---------------------------------------------------------------------------
// Operands of the sweeps on halves.  Every tile belongs to one of kFrames frames (the nearest of as many points, see
// frame_kernel), and a point x of a tile of frame c is kept as x' = x - c, one half per coordinate, for either side of
// the products.  With f the query's frame and c the candidate's,
//   |q - x|^2 = |q - c|^2 + beta_f(x) - 2 q'.x',   beta_f(x) = |x'|^2 - 2 (f - c).x':
// |q - c|^2 = beta_c(q) + |f - c|^2 is a number per query while the frame lasts, beta a number per candidate that the
// accumulator starts from, and nothing but the products depends on the pair.  One product per pair and coordinate
// where two bf16 terms take three, and half the operand bytes; what it loses is bounded below.
// ---------------------------------------------------------------------------
constexpr int kFrames = 16, kSeedFrames = 8;

// What the frames and the choice between the sweeps take from the tiles.
struct HalfScale {
    unsigned int reach;     // float bits: most a point lies from its frame (an upper bound)
    int not_finite;         // tiles without a finite ball
    float bound, bound_bf16;  // sums over the tiles of about what a distance within the tile may be off by, on either operand
    float log_reach;        // sum over the tiles of log2 of the most a point of theirs lies from the frame
    int unsure;             // sampled queries whose neighbours the bound may not tell from the rest (gap_kernel)
    float pad[2];
};

// Frames first .. last - 1: distances of all tile centres to them, and every tile's nearest frame so far.  The first
// kSeedFrames are centres of tiles spread evenly over the numbering (where points have an order, as densely as the
// points lie), the others each the centre that lies farthest from all frames before it, which reaches the parts of the
// points that the even spread missed.  best[f]: that centre, by the launch whose last frame is f.  The launch of the last
// frame also fills `scale`.  64 threads per tile.
constexpr int kFrameTiles = 16;
__global__ __launch_bounds__(1024) void frame_kernel(const float *__restrict__ centers_t, const float *__restrict__ radius,
                                                     int D, int T, int first, int last, u64 *best, int *frame_tile,
                                                     float *__restrict__ nearest, int *__restrict__ tile_frame,
                                                     HalfScale *scale) {
    __shared__ float part[64][kFrameTiles];
    const int l = threadIdx.x % kFrameTiles, slice = threadIdx.x / kFrameTiles;
    const int t = blockIdx.x * kFrameTiles + l, tc = min(t, T - 1);
    const int per = (D + 63) / 64, d0 = slice * per, d1 = min(d0 + per, D);
    float near2 = INFINITY;
    int frame = 0;
    if (first > 0) {
        near2 = nearest[tc];
        frame = tile_frame[tc];
    }
    for (int f = first; f < last; ++f) {
        const int seed = f < kSeedFrames ? (int)((2 * f + 1) * (long long)T / (2 * kSeedFrames))
                                         : min((int)(unsigned int)(best[f - 1] & 0xffffffffu), T - 1);
        if (blockIdx.x == 0 && threadIdx.x == 0) frame_tile[f] = seed;
        float sum = 0.0f;
#pragma unroll 8
        for (int d = d0; d < d1; ++d) {
            const float diff = centers_t[(size_t)d * T + tc] - centers_t[(size_t)d * T + seed];
            sum = fmaf(diff, diff, sum);
        }
        part[slice][l] = sum;
        __syncthreads();
        if (slice == 0) {
            float d2 = 0.0f;
#pragma unroll
            for (int k = 0; k < 64; ++k) d2 += part[k][l];
            if (d2 < near2) {
                near2 = d2;
                frame = f;
            }
        }
        __syncthreads();
    }
    float m2 = 0.0f;  // (of the launch of the last frame)
    if (last == kFrames) {
        float sum = 0.0f;
#pragma unroll 8
        for (int d = d0; d < d1; ++d) {
            const float m = centers_t[(size_t)d * T + tc];
            sum = fmaf(m, m, sum);
        }
        part[slice][l] = sum;
        __syncthreads();
        if (slice == 0)
#pragma unroll
            for (int k = 0; k < 64; ++k) m2 += part[k][l];
    }
    if (threadIdx.x >= kWave) return;
    const bool mine = slice == 0 && t < T;  // (the other lanes of the wave take part in its sums with nothing)
    if (mine) {
        nearest[t] = near2;
        tile_frame[t] = frame;
    }
    const bool finite = mine && near2 < INFINITY;
    u64 far = finite ? ((u64)__float_as_uint(near2) << 32) | (unsigned int)t : 0ull;
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) {
        const u64 other = __shfl_xor(far, m, kWave);
        far = far > other ? far : other;
    }
    if (threadIdx.x == 0) atomicMax(&best[last - 1], far);
    if (last < kFrames) return;
    const float r = radius[tc], mlen = sqrtf(m2), reach = (sqrtf(near2) * (1.0f + 1e-3f) + r) * (1.0f + 1e-3f);
    const bool good = finite && reach < 1e18f && mlen < 1e18f;  // (its square is a float)
    const float acc = 4.0f * (float)(3 * D + 6) * 5.9604644775390625e-08f;
    const float b = good ? 4.0f / 4096.0f * reach * reach : 0.0f;
    const float b16 = good ? (6.2f / 65536.0f + 2.0f * acc) * r * (mlen + r) + acc * (r * r + 2.0f * mlen * r) : 0.0f;
    const float sl = group_sum<kWave>(good ? log2f(fmaxf(reach, 1e-30f)) : 0.0f);
    const float sb = group_sum<kWave>(b), sb16 = group_sum<kWave>(b16), top = group_max<kWave>(good ? reach : 0.0f);
    const int bad = __popcll(__ballot(mine && !good));
    if (threadIdx.x == 0) {
        atomicMax(&scale->reach, __float_as_uint(top));
        if (bad) atomicAdd(&scale->not_finite, bad);
        atomicAdd(&scale->bound, sb);
        atomicAdd(&scale->bound_bf16, sb16);
        atomicAdd(&scale->log_reach, sl);
    }
}

// A sampled tile's query and its neighbourhood in the numbering.
constexpr int kGapMost = (2 * kHomeTiles + 1) * kCT;
constexpr int kGapStride = 2, kGapGiven = kGapMost / kGapStride;  // gap_distances_kernel: every second point of it
struct GapQuery {
    int tile, q, first, last;
    __device__ GapQuery(int sample, int step, int N, int T) {
        tile = min(sample * step + step / 2, T - 1);
        q = min(tile * kCT + 5, N - 1);
        first = max(tile - kHomeTiles, 0) * kCT;
        last = min((tile + kHomeTiles + 1) * kCT, N);
    }
};
// Squared distances of the sampled queries to their neighbourhoods where rows are long (as bits; all ones beyond the
// points there are, and for the query): four rows per wave and turn, kGapSplit workgroups per sample.  Bound by the rows it
// reads (64 samples of 2176 rows of 784 dimensions 76 us, 5.7 TB/s; a workgroup per sample 0.3 ms): hence every second one.
constexpr int kGapSplit = 8;
__global__ __launch_bounds__(1024) void gap_distances_kernel(const float *__restrict__ X, int N, int D, int T, int step,
                                                             unsigned int *__restrict__ dist) {
    constexpr int kAtOnce = 4, kRows = kGapGiven / kGapSplit;
    static_assert(kRows % kAtOnce == 0 && kGapGiven % kGapSplit == 0, "whole turns");
    const GapQuery g((int)blockIdx.y, step, N, T);
    const int lane = threadIdx.x & (kWave - 1), row0 = (int)blockIdx.x * kRows;
    const float *xq = X + (size_t)g.q * D;
    for (int p = threadIdx.x / kWave * kAtOnce; p < kRows; p += 1024 / kWave * kAtOnce) {
        float sum[kAtOnce];
        const float *x[kAtOnce];
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            sum[u] = 0.0f;
            x[u] = X + (size_t)min(g.first + kGapStride * (row0 + p + u), g.last - 1) * D;
        }
#pragma unroll 8
        for (int d = lane; d < D; d += kWave) {
            const float v = xq[d];
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u) {
                const float diff = v - x[u][d];
                sum[u] = fmaf(diff, diff, sum[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            const int j = g.first + kGapStride * (row0 + p + u);
            const float total = group_sum<kWave>(sum[u]);
            if (lane == 0) dist[(size_t)blockIdx.y * kGapGiven + row0 + p + u] = j < g.last && j != g.q ? __float_as_uint(total) : ~0u;
        }
    }
}

// Whether the bound leaves room between a query's K-th neighbour and the last candidate kept of it: for one point of each
// sampled tile (`step` apart), the distances to the points of its neighbourhood in the numbering (`given`, or formed here),
// those of the ranks `near_rank` and `far_rank` among them, and `loss` times the squared reach of the tile from its frame.  The
// gap among all points is smaller than that, a third to all of it.  One workgroup of 256 threads per sampled tile.
__global__ __launch_bounds__(256) void gap_kernel(const float *__restrict__ X, int N, int D, int T, int step, int near_rank,
                                                  int far_rank, float loss, const unsigned int *__restrict__ given,
                                                  const float *__restrict__ nearest, const float *__restrict__ radius,
                                                  HalfScale *scale) {
    constexpr int kEach = (kGapMost + 255) / 256;
    __shared__ int below[2][2];
    const int tid = threadIdx.x;
    const GapQuery g((int)blockIdx.x, step, N, T);
    const float *xq = X + (size_t)g.q * D;
    unsigned int dist[kEach];
#pragma unroll
    for (int u = 0; u < kEach; ++u) {
        const int r = u * 256 + tid, j = g.first + r;
        if (given) {
            dist[u] = r < kGapGiven ? given[(size_t)blockIdx.x * kGapGiven + r] : ~0u;
            continue;
        }
        const float *x = X + (size_t)min(j, g.last - 1) * D;
        float sum = 0.0f;
#pragma unroll 4
        for (int d = 0; d < D; ++d) {
            const float diff = xq[d] - x[d];
            sum = fmaf(diff, diff, sum);
        }
        dist[u] = j < g.last && j != g.q ? __float_as_uint(sum) : ~0u;  // (not negative: ordered as its bits)
    }
    // The largest values that fewer distances than the ranks lie below, bit by bit, side by side.
    unsigned int near_bits = 0u, far_bits = 0u;
    for (int b = 30, turn = 0; b >= 8; --b, turn ^= 1) {  // (23 bits: a relative 3e-5)
        const unsigned int near_trial = near_bits | (1u << b), far_trial = far_bits | (1u << b);
        if (tid < 2) below[turn][tid] = 0;
        __syncthreads();
        int c_near = 0, c_far = 0;
#pragma unroll
        for (int u = 0; u < kEach; ++u) {
            c_near += __popcll(__ballot(dist[u] < near_trial));
            c_far += __popcll(__ballot(dist[u] < far_trial));
        }
        if ((tid & (kWave - 1)) == 0) {
            atomicAdd(&below[turn][0], c_near);
            atomicAdd(&below[turn][1], c_far);
        }
        __syncthreads();  // (these words are cleared two turns on, past the barrier of the next)
        if (below[turn][0] < near_rank) near_bits = near_trial;
        if (below[turn][1] < far_rank) far_bits = far_trial;
    }
    if (tid == 0) {
        const float near_d = __uint_as_float(near_bits), far_d = __uint_as_float(far_bits);
        // (in many dimensions a point lies about across from the frame, seen from the tile's centre)
        const float r = radius[g.tile], reach = sqrtf(nearest[g.tile]) + r, reach2 = given ? nearest[g.tile] + r * r : reach * reach;
        if (!(loss * reach2 < far_d - near_d)) atomicAdd(&scale->unsure, 1);
    }
}

// frames[d][f]: coordinate d of frame f (rows of kFrames floats), and |frame f - frame g|^2.  One workgroup.
__global__ __launch_bounds__(1024) void frame_rows_kernel(const float *__restrict__ centers_t, int D, int T,
                                                          const int *__restrict__ frame_tile, float *__restrict__ frames,
                                                          float *__restrict__ frame_d2) {
    constexpr int kDims = 512;  // at a time
    __shared__ float rows[kDims * kFrames];
    __shared__ float part[4][kFrames * kFrames];
    const int tid = threadIdx.x, pair = tid & 255, quarter = tid >> 8;
    static_assert(kFrames * kFrames == 256, "four threads per pair of frames");
    float sum = 0.0f;
    for (int first = 0; first < D; first += kDims) {
        const int dims = min(kDims, D - first);
        __syncthreads();
        for (int e = tid; e < dims * kFrames; e += 1024) {
            rows[e] = centers_t[(size_t)(first + e / kFrames) * T + frame_tile[e % kFrames]];
            frames[(size_t)first * kFrames + e] = rows[e];
        }
        __syncthreads();
        for (int d = quarter; d < dims; d += 4) {
            const float diff = rows[d * kFrames + pair / kFrames] - rows[d * kFrames + pair % kFrames];
            sum = fmaf(diff, diff, sum);
        }
    }
    part[quarter][pair] = sum;
    __syncthreads();
    if (quarter == 0) frame_d2[pair] = (part[0][pair] + part[1][pair]) + (part[2][pair] + part[3][pair]);
}

// Halves are kept times a power of two that brings the largest distance from a frame to at most 2^14; what would be
// a subnormal half is kept as zero, so it does not matter what the matrix unit makes of those.
__device__ __forceinline__ float half_scale_factor(const HalfScale *scale) {
    const float reach = fmaxf(__uint_as_float(scale->reach), 1e-30f);
    return ldexpf(1.0f, min(max(13 - ilogbf(reach), -60), 60));
}

// One workgroup per tile.  Xh: [tile][block of 32 points (4)][step of 16 dimensions (S)][lane (64)] 8 halves, lane = 32 *
// (dimension % 16 / 8) + point % 32, element = dimension % 8 (the layout of pack_points_bf16_kernel, one term).
// beta: row f of `pitch` floats holds beta_f of every point times -s^2 / 2 (s: the halves' scale), which is what the
// accumulators start from; -infinity beyond the points there are, so that nothing passes there.  point_len: |x'| and |x' - what the halves stand for|,
// rounded up (half_bound.h has what the sweeps make of them).  tile_info: the largest of the second and of |x'| among a
// tile's points, and the tile's frame.
__global__ __launch_bounds__(256) void half_pack_kernel(const float *__restrict__ X, int N, int D, int S,
                                                        const float *__restrict__ frames, const int *__restrict__ tile_frame,
                                                        const HalfScale *scale, int pitch, uint4 *__restrict__ Xh,
                                                        float *__restrict__ beta, float2 *__restrict__ point_len,
                                                        float4 *__restrict__ tile_info) {
    __shared__ float wave_eps[4], wave_len[4];
    const int tile = blockIdx.x, tid = threadIdx.x, lane = tid & 63, block = tid >> 6;
    const int i = tile * kCT + block * 32 + (lane & 31), h = lane >> 5;
    const int own = tile_frame[tile];
    const float s = half_scale_factor(scale), inv = 1.0f / s;
    const float *x = X + (size_t)(i < N ? i : 0) * D;
    float dot[kFrames], len = 0.0f, eps = 0.0f;
#pragma unroll
    for (int f = 0; f < kFrames; ++f) dot[f] = 0.0f;
    uint4 *dst = Xh + ((size_t)tile * 4 + block) * S * 64 + lane;
    for (int step = 0; step < S; ++step) {
        const int d0 = 16 * step + 8 * h;
        unsigned int bits[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            bits[j] = 0u;
            if (i < N && d0 + j < D) {
                const float *fr = frames + (size_t)(d0 + j) * kFrames;
                const float c = fr[own], v = x[d0 + j] - c, w = v * s;
                const _Float16 hv = fabsf(w) < 6.103515625e-05f ? (_Float16)0.0f : (_Float16)w;  // (2^-14)
                const float lost = v - (float)hv * inv;
                bits[j] = (unsigned int)__builtin_bit_cast(unsigned short, hv);
                len = fmaf(v, v, len);
                eps = fmaf(lost, lost, eps);
#pragma unroll
                for (int f = 0; f < kFrames; ++f) dot[f] = fmaf(fr[f] - c, v, dot[f]);
            }
        }
        dst[step * 64] = make_uint4(bits[0] | (bits[1] << 16), bits[2] | (bits[3] << 16), bits[4] | (bits[5] << 16),
                                    bits[6] | (bits[7] << 16));
    }
    len += __shfl_xor(len, 32, kWave);
    eps += __shfl_xor(eps, 32, kWave);
#pragma unroll
    for (int f = 0; f < kFrames; ++f) {
        const float other = dot[f] + __shfl_xor(dot[f], 32, kWave);
        if ((f & 1) == h) beta[(size_t)f * pitch + i] = (i < N ? fmaf(-2.0f, other, len) : INFINITY) * (-0.5f * s * s);
    }
    const float xl = length_bound(len, D), xe = length_bound(eps, D);
    if (h == 0) point_len[i] = make_float2(xl, xe);
    const float me = group_max<kWave>(xe), ml = group_max<kWave>(xl);
    if (lane == 0) {
        wave_eps[block] = me;
        wave_len[block] = ml;
    }
    __syncthreads();
    if (tid == 0)
        tile_info[tile] = make_float4(fmaxf(fmaxf(wave_eps[0], wave_eps[1]), fmaxf(wave_eps[2], wave_eps[3])),
                                      fmaxf(fmaxf(wave_len[0], wave_len[1]), fmaxf(wave_len[2], wave_len[3])),
                                      __int_as_float(own), 0.0f);
}

constexpr int kRankRounds = 4;  // (every 256th, 64th, 16th, 4th tile; then all)
// Memory that no kernel writes while this one runs: with a uniform address, loads on the scalar unit.
typedef const __attribute__((address_space(4))) float ConstFloat;
__device__ __forceinline__ ConstFloat *as_const(const void *p) { return (ConstFloat *)p; }

struct SweepArgs {
    const float4 *Xp;
    const float *X;  // the points as given (bf16 sweep: the query side is formed from them)
    const float *centres_p, *tile_coef;  // chunked bf16 sweep: tile centres by chunk, error coefficients
    const float *centre_dist;  // chunked bf16 sweep, TABLE: |query - tile centre|^2, a row of centre_pitch per tile
    int centre_pitch;
    int N, D, Dnorm, want, cap;
    u64 *lists;
    int num_qtiles;
    int *cand;
    float *tau;
    const float *norms;      // |x|^2 per point
    const float *centers_t;  // D x T tile centres
    const float *radius;     // T tile radii (upper bounds)
    int bitmap_words;        // ceil(T / 32)
    int trigger;             // a list longer than this is compacted after the tile (<= cap - kCT)
    unsigned long long *tiles_swept;  // statistics: (query tile, candidate tile) pairs that were not skipped, each once
    const float4 *Bp;  // chunked sweep only: query-side packed copy (-2 x_d, 1 in the |c|^2 row)
    int n_chunks;      // chunked sweep only: chunks of kChunkSteps k-steps per point
    // Chunked sweep only.  The num_qtiles query tiles are qtile_list[i], or first + i step without a list.
    // Every query tile is swept by `parts` workgroups, part p taking the candidate tiles t with t % parts == p.
    // One part writes cand / tau directly (row i * kMQ + query in tile); several parts write the keys they
    // keep (all bits set where a part has fewer) to row (i * kMQ + query in tile) * parts + p of part_keys,
    // and knn_merge_parts_kernel picks the `want` best of a query's parts afterwards.
    const int *qtile_list;
    int qtile_first, qtile_step;
    int parts;
    u64 *part_keys;
    int select_slack;  // entries beyond `want` a compaction in mid-sweep may keep (see wave_select)
    // Approximate search (register-resident sweep only; null = exact): the points are numbered list by list of
    // an inverted file, and after its neighbourhood in the numbering a query tile only visits the tiles that
    // overlap the lists some query of the tile probes.  probe_tile_lists: per query tile a bitmap over the
    // lists (probe_list_words words); probe_list_tiles: first and last tile of every list (first > last: empty).
    const unsigned int *probe_tile_lists;
    int probe_list_words, probe_nlist;
    const int *probe_list_tiles;
    // Sweeps on halves (see half_pack_kernel).
    const float *beta;
    int beta_pitch;
    const float2 *point_len;
    const float4 *tile_info;
    const float *frame_d2;
    const HalfScale *half_scale;
    int ranks[kRankRounds];  // see knn_half_sweep_kernel
};

// ---------------------------------------------------------------------------
// MFMA sweep, in two arithmetic variants.
// BF16 = false: KSTEPS = Daug / 2 k-steps of v_mfma_f32_32x32x2f32 on the points as floats.
// BF16 = true: KSTEPS steps of 16 dimensions of v_mfma_f32_32x32x16_bf16 on the points relative to their
// tile's centre, split into two bf16 terms per coordinate; high x high, high x low and low x high are
// accumulated (three instructions per step), which leaves out terms below 3.1 * 2^-16 of |q_d delta_d| per
// dimension.  The keys stored are the products plus |q - centre|^2 less the tile's error bound (see
// pack_tile_centres_kernel): lower bounds of the distances.  A step of 16 dimensions takes half the
// matrix-pipe time of one fp32 step of 2.
// Dynamic LDS: one candidate tile, copied verbatim from the packed points
//   a[cand block (4)][step group (S4)][lane (64)] float4   (4 steps per float4)            fp32
//   a[cand block (4)][term (2)][step (KSTEPS)][lane (64)] 8 x bf16                          bf16
// followed by one sort buffer (cap keys) per wave and the visit bitmap (one bit per tile).
//
// Tiles are visited in two phases.  First the query tile's own neighbourhood in the point
// numbering (kHomeTiles tiles on either side), which gives every query a finite threshold.
// Then only the tiles whose bounding ball can still hold a point below the largest of those
// thresholds: with c, r the centre and radius of a tile's ball, every point x of tile t has
// |q - x| >= |c_a - c_t| - r_a - r_t for every query q of tile a (triangle inequality), so the
// tile is skipped when that bound, squared, exceeds max_q (threshold_q + |q|^2).  A threshold
// only ever decreases and the final verification of a query compares with its final threshold,
// so a skipped tile cannot hold one of its neighbours.  On numberings without locality the
// balls are large and nothing is skipped.
// Output per query: the `want` best candidates by approximate distance
// (cand, -1 padded) and tau = the approximate distance of the last one kept
// (+inf when fewer than `want` candidates exist), both without the |q|^2 term.
// ---------------------------------------------------------------------------
// Workgroups per compute unit the register budget is set for (bf16: the query's coordinates stay in
// registers beside the two operand terms).  Measured: three workgroups with 330 bytes of spills per lane
// ran at half the speed of two at 4 steps; two workgroups beat one at 5 to 7 steps in spite of 100 to 380
// bytes of spills (300,000 points, 64 / 90 / 100 dimensions: 0.040 -> 0.027 s, 0.044 -> 0.033 s,
// 0.045 -> 0.040 s); at 8 steps two tiles of 66 KB do not fit a compute unit's LDS.
constexpr int bf16_sweep_occupancy(int steps) { return steps <= 2 ? 3 : (steps <= 7 ? 2 : 1); }
constexpr size_t kUnitLds = 160 * 1024, kSweepLds = 4112;  // bytes of a compute unit, and of a workgroup beside its dynamic ones
constexpr int float_sweep_occupancy(int ksteps) { return ksteps <= 28 ? 3 : 1; }
template <int KSTEPS, bool BF16>
constexpr int sweep_occupancy() {
    return BF16 ? bf16_sweep_occupancy(KSTEPS) : float_sweep_occupancy(KSTEPS);
}

template <int KSTEPS, bool BF16>
__global__ __launch_bounds__(256, (sweep_occupancy<KSTEPS, BF16>())) void knn_mfma_sweep_kernel(const SweepArgs args) {
    const float4 *__restrict__ Xp = args.Xp;
    const int N = args.N, D = args.D, Dnorm = args.Dnorm, want = args.want, cap = args.cap;
    const int num_qtiles = args.num_qtiles;
    u64 *__restrict__ lists = args.lists;
    int *__restrict__ cand = args.cand;
    float *__restrict__ tau = args.tau;
    constexpr int S4 = BF16 ? 2 * KSTEPS : (KSTEPS + 3) / 4;  // 16-byte slots per lane and candidate block
    constexpr int kMainFloat4 = 4 * S4 * 64;              // float4 of matrix operands per candidate tile
    constexpr int kTileFloat4 = kMainFloat4 + (BF16 ? 64 : 0);  // ... and the centre block of the bf16 layout
    constexpr int kLoadsPerThread = kMainFloat4 / 256;    // == S4
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    float4 *a_lds = reinterpret_cast<float4 *>(lds_raw);
    u64 *sortbuf = reinterpret_cast<u64 *>(a_lds + kTileFloat4) + (size_t)(threadIdx.x >> 6) * cap;  // per wave
    unsigned int *bitmap = reinterpret_cast<unsigned int *>(reinterpret_cast<u64 *>(a_lds + kTileFloat4) + 4 * (size_t)cap);
    __shared__ u64 thr[kMQ];
    __shared__ int cnt[kMQ];
    __shared__ int fill[256];  // entries in each lane's region of its query's list
    __shared__ float qcenter[128];
    __shared__ unsigned int hist_all[4][kWave];
    __shared__ float tmax_part[2];

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int qn = lane & 31, kh = lane >> 5;
    u64 *list = lists + (size_t)blockIdx.x * kMQ * cap;

    // One candidate tile: global -> registers (in flight during the matrix instructions) -> LDS.
    // The staging array is a native vector type with compile-time indices: as an array of
    // HIP float4 structs it was placed in scratch memory, where every load waited for the last.
    v4f stage[kLoadsPerThread], stage_centre;
    auto fetch = [&](int tile) {
        const v4f *src = reinterpret_cast<const v4f *>(Xp) + (size_t)tile * kTileFloat4 + tid;
#pragma unroll
        for (int r = 0; r < kLoadsPerThread; ++r) stage[r] = src[r * 256];
        if (BF16 && tid < 64) stage_centre = src[kMainFloat4];
    };
    auto stash = [&](int buf) {
        v4f *dst = reinterpret_cast<v4f *>(a_lds) + buf * kTileFloat4 + tid;
#pragma unroll
        for (int r = 0; r < kLoadsPerThread; ++r) dst[r * 256] = stage[r];
        if (BF16 && tid < 64) dst[kMainFloat4] = stage_centre;
    };
    const int num_ctiles = (N + kCT - 1) / kCT;

    for (int qt = blockIdx.x; qt < num_qtiles; qt += gridDim.x) {
        const int q0 = qt * kMQ;
        const int q = q0 + wave * 32 + qn;  // this lane's query (>= N in the last tile: padded zeros)
        if (tid < kMQ) {
            thr[tid] = ~0ull;
            cnt[tid] = 0;
        }
        // A query's list is two regions of cap / 2 entries, one per lane of the pair that shares the query:
        // a lane appends to its own region with a counter of its own, so an append needs neither a count of
        // the passing elements nor an atomic to reserve room.
        const int half = cap >> 1;
        // The counter is a register; around a selection it passes through LDS (fill[tid]), where the whole
        // wave can read and set it.
        int my_n = 0;
        // Selection over the list of query b of this wave (all lanes take part); returns the caller's updated
        // counter: the entries kept go back alternately into the two regions.
        // With fewer than `want` entries nothing is dropped; `spread` then still deals them out alternately,
        // for a query whose one region fills up while the other stays empty (and for the output pass, which
        // reads that order).
        auto select_query = [&](int b, int slack, bool spread) {
            const int ql = wave * 32 + b;
            const int c0n = fill[wave * 64 + b], c1n = fill[wave * 64 + b + 32];
            int kept = c0n + c1n;
            if (kept < want) {
                if (!spread) return;
                u64 *lq = list + (size_t)ql * cap;
                __threadfence_block();  // this wave's appends to the list are complete
                for (int e = lane; e < kept; e += kWave) sortbuf[e] = e < c0n ? lq[e] : lq[half + e - c0n];
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                for (int e = lane; e < kept; e += kWave) lq[(e & 1) * half + (e >> 1)] = sortbuf[e];
                __threadfence_block();
            } else {
                if (lane == 0) cnt[ql] = kept;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                kept = wave_select<true>(list + (size_t)ql * cap, want, &cnt[ql], &thr[ql], sortbuf,
                                         hist_all[wave], lane, slack, half, c0n);
            }
            if (lane == 0) {
                fill[wave * 64 + b] = (kept + 1) >> 1;
                fill[wave * 64 + b + 32] = kept >> 1;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        };
        // B operand from the same packed layout (query tiles and candidate tiles coincide: kMQ == kCT):
        // -2 q_d for the real dimensions, 1 for the |c|^2 row, 0 elsewhere.
        float bq[BF16 ? 1 : 4 * S4];
        v8bf bq_hi[BF16 ? KSTEPS : 1], bq_lo[BF16 ? KSTEPS : 1];
        float qf[BF16 ? 8 * KSTEPS : 1];  // this lane's half of the query's coordinates
        float q_len = 0.0f;               // |q|, rounded up
        if constexpr (BF16) {
            // -2 q_d in two bf16 terms; 1 in the three dimensions of the high term that carry beta.
            const float *xq = args.X + (size_t)(q < N ? q : 0) * D;
            if (q < N) q_len = sqrtf(args.norms[q]) * (1.0f + 1e-6f);
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) {
                unsigned int oh[4], ol[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    unsigned int h2[2], l2[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int d = 16 * s + 8 * kh + 2 * k + e;
                        const float v = q < N && d < D ? xq[d] : 0.0f;
                        qf[8 * s + 2 * k + e] = v;
                        const float w = -2.0f * v;
                        const unsigned int hi = bf16_bits(w);
                        h2[e] = d < D ? hi : (d < D + 3 ? 0x3f80u : 0u);
                        l2[e] = d < D ? bf16_bits(w - bf16_value(hi)) : 0u;
                    }
                    oh[k] = h2[0] | (h2[1] << 16);
                    ol[k] = l2[0] | (l2[1] << 16);
                }
                bq_hi[s] = __builtin_bit_cast(v8bf, make_uint4(oh[0], oh[1], oh[2], oh[3]));
                bq_lo[s] = __builtin_bit_cast(v8bf, make_uint4(ol[0], ol[1], ol[2], ol[3]));
            }
        } else {
            const float4 *src = Xp + (size_t)qt * kTileFloat4 + (size_t)wave * S4 * 64 + lane;
#pragma unroll
            for (int s4 = 0; s4 < S4; ++s4) {
                const float4 v = src[s4 * 64];
                const float c[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int d = 2 * (4 * s4 + k) + kh;
                    bq[4 * s4 + k] = d < D ? -2.0f * c[k] : (d == Dnorm ? 1.0f : 0.0f);
                }
            }
        }
        const int buf = 0;  // one LDS tile: the next tile waits in registers until this one has been read
        // One tile: compute it from LDS buffer `buf` while the next one travels through registers.
        auto process = [&](int ct, int next_ct) {
            const int c0 = ct * kCT;
            if (next_ct >= 0) fetch(next_ct);
            const u64 limit = thr[wave * 32 + qn];
            // ~0 is "no threshold yet": its distance field does not decode to a number.
            const float limit_d = limit == ~0ull ? INFINITY : key_distance(limit);
            // bf16: the matrix product lacks |q - m|^2 (m: the tile's centre), and the keys carry a lower bound
            // of the distance: the product plus `off` = |q - m|^2 (rounded down) - the tile's error bound.
            // The products are tested against the threshold less `off`, rounded up.
            float off = 0.0f, limit_acc = limit_d;
            if constexpr (BF16) {
                const float4 *cen = a_lds + buf * kTileFloat4 + kMainFloat4;
                float f = 0.0f;
#pragma unroll
                for (int s = 0; s < KSTEPS; ++s) {
                    const float4 m0 = cen[4 * s + 2 * kh], m1 = cen[4 * s + 2 * kh + 1];
                    const float m[8] = {m0.x, m0.y, m0.z, m0.w, m1.x, m1.y, m1.z, m1.w};
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const float diff = qf[8 * s + j] - m[j];
                        f = fmaf(diff, diff, f);
                    }
                }
                f += __shfl_xor(f, 32);
                const float4 g = cen[32];
                off = f * (1.0f - (float)(D + 4) * 5.9604644775390625e-08f) - fmaf(q_len, g.x, g.y);
                limit_acc = limit_d - off;
                limit_acc += 2.4e-7f * (fabsf(limit_d) + fabsf(off));  // (inf stays inf)
            }
            // Two candidate blocks at a time: two independent accumulator chains keep the matrix pipe busy.
            auto multiply = [&](int cb, v16f &acc0, v16f &acc1) {
                acc0 = v16f{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                acc1 = acc0;
                const float4 *a0 = a_lds + (size_t)(buf * 4 + cb) * S4 * 64 + lane;
                const float4 *a1 = a0 + S4 * 64;
                if constexpr (BF16) {
                    const v4f *b0 = reinterpret_cast<const v4f *>(a0), *b1 = reinterpret_cast<const v4f *>(a1);
                    // The operands of step s + 1 are read from LDS while the products of step s run.
                    v4f next[4] = {b0[0], b1[0], b0[KSTEPS * 64], b1[KSTEPS * 64]};
#pragma unroll
                    for (int s = 0; s < KSTEPS; ++s) {
                        const v8bf xh = __builtin_bit_cast(v8bf, next[0]);
                        const v8bf yh = __builtin_bit_cast(v8bf, next[1]);
                        const v8bf xl = __builtin_bit_cast(v8bf, next[2]);
                        const v8bf yl = __builtin_bit_cast(v8bf, next[3]);
                        if (s + 1 < KSTEPS) {
                            next[0] = b0[(s + 1) * 64];
                            next[1] = b1[(s + 1) * 64];
                            next[2] = b0[(KSTEPS + s + 1) * 64];
                            next[3] = b1[(KSTEPS + s + 1) * 64];
                        }
                        acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xh, bq_hi[s], acc0, 0, 0, 0);
                        acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(yh, bq_hi[s], acc1, 0, 0, 0);
                        acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xh, bq_lo[s], acc0, 0, 0, 0);
                        acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(yh, bq_lo[s], acc1, 0, 0, 0);
                        acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xl, bq_hi[s], acc0, 0, 0, 0);
                        acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(yl, bq_hi[s], acc1, 0, 0, 0);
                    }
                } else {
#pragma unroll
                    for (int s4 = 0; s4 < S4; ++s4) {
                        const float4 x = a0[s4 * 64], y = a1[s4 * 64];
                        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, bq[4 * s4], acc0, 0, 0, 0);
                        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(y.x, bq[4 * s4], acc1, 0, 0, 0);
                        if (4 * s4 + 1 < KSTEPS) {
                            acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, bq[4 * s4 + 1], acc0, 0, 0, 0);
                            acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(y.y, bq[4 * s4 + 1], acc1, 0, 0, 0);
                        }
                        if (4 * s4 + 2 < KSTEPS) {
                            acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(x.z, bq[4 * s4 + 2], acc0, 0, 0, 0);
                            acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(y.z, bq[4 * s4 + 2], acc1, 0, 0, 0);
                        }
                        if (4 * s4 + 3 < KSTEPS) {
                            acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(x.w, bq[4 * s4 + 3], acc0, 0, 0, 0);
                            acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(y.w, bq[4 * s4 + 3], acc1, 0, 0, 0);
                        }
                    }
                }
            };
            auto filter = [&](int cb, v16f &acc0, v16f &acc1) {
                // Register v of lane l holds candidate row 8*(v/4) + 4*(l/32) + v%4 of the block, query column l%32.
                // Smallest of the lane's 32 values, three operands per instruction (the accumulators are
                // never signalling NaNs, so the library fminf's quieting moves are left out).
                // The minima of the four runs of eight registers are kept: the filter skips a run in which no
                // lane of the wave has a passing element.
                float run_min[4];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const v16f &a = g < 2 ? acc0 : acc1;
                    const int o = 8 * (g & 1);
                    float m = matrix_result(a[o + 7]);
                    m = min3(m, a[o], a[o + 1]);
                    m = min3(m, a[o + 2], a[o + 3]);
                    m = min3(m, a[o + 4], a[o + 5]);
                    run_min[g] = min2(m, a[o + 6]);
                }
                const float best = fminf(min3(run_min[0], run_min[1], run_min[2]), run_min[3]);
                // A query meets about K' ln(N / K') passing candidates during the sweep and the 64 lanes
                // serve different queries, so most block pairs have some lane that passes.  A passing lane
                // stores its keys one after the other at the end of its own region of the query's list.
                // The test is on the distance alone; an element that ties with the threshold's distance
                // but not its index is appended too and sorted out by the next compaction.
                if (best <= limit_acc) {
                    const int jbase = c0 + cb * 32 + 4 * kh;  // element (half, v) is candidate jbase + 32 half + 8 (v / 4) + v % 4
                    // Only the last tile has candidates beyond N and only the query's own tile holds the
                    // query: those two tiles knock the excluded elements out by raising them to +inf.
                    if (c0 + kCT > N || (unsigned int)(q0 - c0) < (unsigned int)kCT) {
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            const int j = jbase + 8 * (e >> 2) + (e & 3);
                            if (j >= N || j == q) acc0[e] = INFINITY;
                            if (j + 32 >= N || j + 32 == q) acc1[e] = INFINITY;
                        }
                    }
                    const float lim = q < N ? limit_acc : -INFINITY;
                    u64 *const dst0 = list + ((wave * 32 + qn) * cap + kh * half + my_n);
                    u64 *dst = dst0;
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        // (the minima are from before the exclusions above: lower bounds, which is all this needs)
                        if (__ballot(run_min[g] <= lim) == 0) continue;
#pragma unroll
                        for (int v = 0; v < 8; ++v) {
                            const int e = 8 * g + v;
                            const float dist = e < 16 ? acc0[e & 15] : acc1[e & 15];
                            if (dist <= lim) {
                                int jb = jbase;
                                asm volatile("" : "+v"(jb));  // the index is formed here, not held in 32 registers
                                *dst++ = pack_key(BF16 ? dist + off : dist, jb + 32 * (e >> 4) + 8 * ((e & 15) >> 2) + (e & 3));
                            }
                        }
                    }
                    my_n += (int)(dst - dst0);
                }
            };
            // The filter's stores to the lists count among the outstanding memory operations that the wait for
            // the next tile's registers has to see through, so the second block pair is filtered only after the
            // next tile has gone to LDS: what that wait then meets are the first pair's stores, a whole pair of
            // matrix products old.
            v16f acc0, acc1;
            multiply(0, acc0, acc1);
            filter(0, acc0, acc1);
            multiply(2, acc0, acc1);
            __syncthreads();  // all waves are done with tile `buf`
            if (next_ct >= 0) {
                stash(buf);
                __syncthreads();
            }
            filter(2, acc0, acc1);
            // Lists that a further tile could overflow are compacted by their own wave, right away.
            {
                // (a region takes at most 64 entries per tile)
                u64 crowded = __ballot(my_n > half - kCT / 2);
                crowded = (crowded | (crowded >> 32)) & 0xffffffffull;  // lanes l, l+32 share a query
                if (crowded) {
                    fill[tid] = my_n;
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    while (crowded) {
                        const int b = __ffsll((long long)crowded) - 1;
                        crowded &= crowded - 1;
                        select_query(b, args.select_slack, true);
                    }
                    my_n = fill[tid];
                }
            }
        };

        // Phase 1: the query tile's neighbourhood; phase 2: the tiles the bitmap keeps.
        const int T = num_ctiles;
        const int h0 = max(qt - kHomeTiles, 0), h1 = min(qt + kHomeTiles, T - 1);
        int word_idx = -1;
        unsigned int cur_word = 0u;
        // Next set bit of the bitmap, ascending; every wave walks the same words.
        auto next_tile = [&]() -> int {
            while (cur_word == 0u) {
                ++word_idx;
                if (word_idx >= args.bitmap_words) return -1;
                cur_word = bitmap[word_idx];
            }
            const int b = __ffs((int)cur_word) - 1;
            cur_word &= cur_word - 1u;
            return word_idx * 32 + b;
        };
        fetch(h0);
        __syncthreads();
        stash(0);
        __syncthreads();
        bool home = true;
        int cur = h0;
        unsigned int swept = 0;
        while (cur >= 0) {
            ++swept;
            int nxt = home ? (cur < h1 ? cur + 1 : -1) : next_tile();
            process(cur, nxt);
            if (nxt < 0 && home && (h0 > 0 || h1 < T - 1)) {
                home = false;
                // Thresholds from what the neighbourhood held.
                fill[tid] = my_n;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                for (int b = 0; b < 32; ++b)
                    if (q0 + wave * 32 + b < N) select_query(b, 0, false);
                my_n = fill[tid];
                for (int w = tid; w < args.bitmap_words; w += 256) bitmap[w] = 0u;
                if (tid < D) qcenter[tid] = args.centers_t[(size_t)tid * T + qt];
                __syncthreads();
                if (tid < kMQ) {
                    // Largest squared distance any query of the tile would still accept (rounded up).
                    float v = -INFINITY;
                    if (q0 + tid < N) {
                        const u64 t = thr[tid];
                        v = t == ~0ull ? INFINITY : key_distance(t) + (BF16 ? 0.0f : args.norms[q0 + tid]);
                        v += 1e-5f * fabsf(v) + 1e-30f;
                    }
                    v = group_max<kWave>(v);
                    if (lane == 0) tmax_part[wave] = v;
                }
                __syncthreads();
                const float tmax = fmaxf(tmax_part[0], tmax_part[1]);
                const float ra = args.radius[qt];
                if (args.probe_tile_lists) {
                    // Approximate search: only tiles of probed lists are eligible (the ball test still drops
                    // those among them that cannot matter, which changes nothing in the result).
                    const unsigned int *mine = args.probe_tile_lists + (size_t)qt * args.probe_list_words;
                    for (int l = tid; l < args.probe_nlist; l += 256) {
                        if (!((mine[l >> 5] >> (l & 31)) & 1u)) continue;
                        const int t0 = args.probe_list_tiles[2 * l], t1 = args.probe_list_tiles[2 * l + 1];
                        for (int t = t0; t <= t1; ++t)
                            if ((t < h0 || t > h1) &&
                                tile_may_matter(qcenter, ra, args.centers_t, args.radius, D, T, t, tmax))
                                atomicOr(&bitmap[t >> 5], 1u << (t & 31));
                    }
                } else {
                    for (int t = tid; t < T; t += 256)
                        if ((t < h0 || t > h1) &&
                            tile_may_matter(qcenter, ra, args.centers_t, args.radius, D, T, t, tmax))
                            atomicOr(&bitmap[t >> 5], 1u << (t & 31));
                }
                __syncthreads();
                nxt = next_tile();
                if (nxt >= 0) {
                    fetch(nxt);
                    stash(buf);  // the barrier that ended the last tile freed both buffers
                    __syncthreads();
                }
                // Nothing this block loaded is left in flight as far as the compiler can tell: a load it
                // takes to be possibly outstanding here makes it wait for all loads, the next tile's
                // included, at the first register reuse after process() has issued them.
                __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
            }
            cur = nxt;
        }
        if (tid == 0) atomicAdd(args.tiles_swept, (unsigned long long)swept);
        // Final ordering and output, every wave for its own 32 queries.
        fill[tid] = my_n;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        for (int b = 0; b < 32; ++b) {
            const int ql = wave * 32 + b;
            const int qq = q0 + ql;
            if (qq >= N) break;
            select_query(b, 0, true);
            const int n = fill[wave * 64 + b] + fill[wave * 64 + b + 32];
            const u64 *lq = list + (size_t)ql * cap;  // entry e of the n kept: region e & 1, position e >> 1
            for (int e = lane; e < want; e += kWave)
                cand[(size_t)qq * want + e] = e < n ? key_index(lq[(e & 1) * half + (e >> 1)]) : -1;
            // Every candidate that was dropped, by a compaction or by the filter, had a distance >= the
            // threshold of the moment, and thresholds only decrease.
            if (lane == 0) tau[qq] = thr[ql] == ~0ull ? INFINITY : key_distance(thr[ql]);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        __syncthreads();  // before the next query tile re-initialises thr / cnt and the LDS tiles
    }
}

// ---------------------------------------------------------------------------
// The sweep on halves, up to 126 dimensions (see half_pack_kernel).  Query tiles, visiting order, tile skipping, lists and
// output are those of knn_mfma_sweep_kernel; the accumulators start from the candidates' betas and fall as the
// distance grows, so what is looked for is the largest.
//
// What bounds the kernel (1,000,000 x 50): 220 vector instructions a wave and tile, 880 cycles of a SIMD, and 640 of the matrix
// unit, of the 2100 that pass, so they hide little of each other; a wave waits 44 % of its time.  So: three waves, nothing of
// the tile loop in scratch memory (a wait for a spilled register is a wait for the next tile's loads too: one of them took
// the sweep of 1,000,000 x 50 from 74 to 100 ms; four waves of 128 registers 86), and to that end what is seldom run takes
// its arguments and its lane number where it stands (`cold`, `here`).  Tiles go from memory to LDS without registers; all
// operands of a pair of blocks are asked for ahead of its products, and all products are under way before the first results
// are looked at; seldom taken paths lie outside the straight run of the loop.
// Whole searches, ms, with staging through registers, thresholds from the lists alone and the accumulators loaded from LDS /
// here: 1,000,000 x 50 in four clusters, 90 neighbours 82.8 / 71.6; 300000 x 50 without structure 28.3 / 25.3;
// 300000 x 100, 45 neighbours 40.3 / 33.4; 199999 x 30, 33 neighbours 7.6 / 6.3; 300000 x 10, 30 neighbours 11.7 / 10.0.
//
// Thresholds ahead of the lists.  A list's own threshold, the `want`-th best of what has been seen, lets 133 ln(N / n)
// candidates of a query with 90 neighbours through (more, as it is only lowered when a list is full), ten times what is
// wanted in the end, and each costs a store and a share of the selections.  So tiles are measured before any entry is
// stored.  The neighbourhood: of each run of eight results the smallest distance is kept, and the want-th of those that hold
// a candidate is a threshold that `want` candidates meet.  Then a sample of the tiles beyond it, every 16th (64th, 256th of
// many): the smallest distance of each tile and lane, and the r-th of those is the threshold: the r-th nearest point of a
// share p of the tiles is farther than the wanted number of all of them unless r or more of those lie in that share, and
// ranks[] has the r for which that does not happen (p wanted + 5.5 sqrt(p wanted) + 5: about 1e-8).  The lists are filled
// after that, round by round: every 4th tile (16th, 64th) first, with another such threshold from the entries after it.
// Neighbours may lie many to a tile, so at most one entry per query, tile and lane counts, the first that passes: r entries
// are in r halves of tiles then, and all tiles have r / p with one at least as near.  A query for which it happens all the
// same is left with too few candidates, fails its verification and is searched again.  Entries per query of the 1,000,000 x
// 50 search: 1050 from lists and rounds alone, 530 so, for 122 more tiles; selections 8 and 3.
//
// Parts: as in the chunked sweep (no rounds: a part's threshold must be that of a list that lacks nothing).
// Dynamic LDS: two candidate tiles, each
//   a[cand block (4)][step (S)][lane (64)] 8 halves, 128 betas (times -s^2 / 2), its tile_info
// and the visit bitmap.
// ---------------------------------------------------------------------------
constexpr int kRoundTiles = 256;   // fewer tiles to visit after the neighbourhood: no rounds
constexpr int kSampleTiles = 240;  // measured beyond the neighbourhood, about, at most (a lane has room for kHalfCap / 2 distances)
// Entries of a list, which a selection holds in registers (eight per lane; with sixteen the tile loop's own go to
// memory: 20000 x 8, 300 neighbours 3.1 ms on bf16 terms, 3.8), and the most candidates kept of them.
constexpr int kHalfCap = 512, kHalfWant = 256;
// Workgroups per compute unit the register budget is set for.
constexpr int half_sweep_occupancy(int steps) { return steps <= 5 ? 3 : 2; }
constexpr int half_tile_float4(int steps) { return 256 * steps + kCT / 4 + 1; }
template <int S>
__global__ __launch_bounds__(256, half_sweep_occupancy(S)) void knn_half_sweep_kernel(const SweepArgs args) {
    constexpr int cap = kHalfCap, half = cap / 2, NK = cap / kWave;
    const int N = args.N, want = args.want;
    // (loaded once)
    const float4 *tile_info = args.tile_info, *points = args.Xp;
    asm volatile("" : "+s"(tile_info), "+s"(points));
    constexpr int kMain = 256 * S, kTile = half_tile_float4(S);
    // Arguments of the code outside the tile loop, read where they are used: kept in registers from the start, they push
    // those of the loop out.
    typedef const __attribute__((address_space(4))) SweepArgs ConstArgs;
    auto cold = []() {
        ConstArgs *p = (ConstArgs *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(p));
        return p;
    };
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    unsigned int *bitmap = reinterpret_cast<unsigned int *>(lds_raw + 2 * kTile * 16);
    __shared__ u64 thr[kMQ];
    __shared__ int fill[256];  // entries in each lane's region of its query's list, around a selection
    __shared__ float qcenter[128];
    __shared__ float tmax_part[2];

    // (A copy that the compiler takes for a new value: what is seldom run forms its addresses from that where it stands, or
    // they would be formed ahead of the loops and held in the tile loop's registers.)
    auto here = [](int v) {
        asm volatile("" : "+v"(v));
        return v;
    };
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int qn = lane & 31, kh = lane >> 5;
    u64 *list = args.lists + (size_t)blockIdx.x * kMQ * cap;
    // (The same in every lane: kept on the scalar side.)
    auto uniform = [](float v) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v))); };
    const float s = half_scale_factor(cold()->half_scale), s2 = uniform(0.5f * s * s), back = uniform(-1.0f / s2);  // (powers of two)
    const int T = (N + kCT - 1) / kCT, P = args.parts;

    // A candidate tile goes to LDS without a register in between: every wave its blocks of 64 slots of 16 bytes, the first
    // wave the betas (lanes 0 .. 31) and what the tile's bound takes (lane 0) as well.
    const unsigned int lds_base = __builtin_amdgcn_readfirstlane((unsigned int)(size_t)(LdsByte *)lds_raw);
    const unsigned int lane_byte = (unsigned int)(wave * 64 + lane) * 16u;
    const float *tile_beta = nullptr;  // of the query tile's frame
    const unsigned int wave_dst = lds_base + (unsigned int)wave * 1024u;
    auto fetch = [&](int tile, unsigned int buf) {
        unsigned int to = wave_dst + buf;
        asm volatile("" : "+s"(to));  // (what is added to it is, where it is used)
#pragma unroll
        for (int r = 0; r < S; ++r) load_to_lds(points + (size_t)tile * kMain + r * 256, lane_byte, to + r * 4096u);
        if (wave == 0) {
            const unsigned int dst = lds_base + buf + kMain * 16;
            if (lane < kCT / 4) load_to_lds(tile_beta + (size_t)tile * kCT, lane_byte, dst);
            if (lane == 0) load_to_lds(tile_info + tile, lane_byte, dst + kCT * 4);
        }
    };

    for (int w = blockIdx.x; w < args.num_qtiles * P; w += gridDim.x) {
        const int qi = w / P, part = w - qi * P;
        const int qt = cold()->qtile_first + qi * cold()->qtile_step;
        const int q0 = qt * kMQ;
        const int q = q0 + wave * 32 + qn;  // this lane's query (>= N in the last tile: padded zeros)
        const bool live = q < N;
        if (tid < kMQ) thr[tid] = ~0ull;
        // A query's list is two regions of cap / 2 entries, one per lane of the pair that shares the query; a lane
        // appends at my_at, a byte offset into the workgroup's lists.
        const unsigned int region = (unsigned int)(((wave * 32 + qn) * cap + kh * half) * (int)sizeof(u64));
        unsigned int my_at = region;
        float limit_d = INFINITY;  // the query's threshold
        unsigned int not_counted = (unsigned int)kNotCounted;  // of the next entry of this lane
        bool home = true;
        // Measuring: of each lane's results only the smallest distances, of runs of eight (in the neighbourhood) or of the
        // tile, go to the second half of its region, `minima` of them so far, and nothing to the list.
        bool measure = false;
        int minima = 0;
        auto my_fill = [&]() { return (int)((my_at - region) / (unsigned int)sizeof(u64)); };
        // Selections over the lists of this wave's queries in `mask`, the next list on its way into registers meanwhile.
        auto select_queries = [&](unsigned int mask, int rank, int slack, bool counted) {
            const int tid = here(threadIdx.x), lane = tid & 63, qn = lane & 31;
            fill[tid] = my_fill();
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            auto counts = [&](int b, int &c0, int &n) {
                c0 = __builtin_amdgcn_readfirstlane(fill[wave * 64 + b]);
                n = c0 + __builtin_amdgcn_readfirstlane(fill[wave * 64 + b + 32]);
            };
            u64 next[NK];
            int c0, n, next_n = 0;
            auto load = [&](int b) {
                counts(b, c0, next_n);
                load_halves<NK>(list + (size_t)(wave * 32 + b) * cap, half, c0, next_n, lane, next);
            };
            if (mask) load(__ffs((int)mask) - 1);
            while (mask) {
                const int b = __ffs((int)mask) - 1;
                mask &= mask - 1u;
                u64 key[NK];
#pragma unroll
                for (int u = 0; u < NK; ++u) key[u] = next[u];
                n = next_n;
                if (mask) load(__ffs((int)mask) - 1);
                const int ql = wave * 32 + b;
                const int kept = select_halves<NK>(list + (size_t)ql * cap, rank, slack, counted, half, n, &thr[ql], lane, key);
                if (lane == 0) {
                    fill[wave * 64 + b] = (kept + 1) >> 1;
                    fill[wave * 64 + b + 32] = kept >> 1;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            my_at = region + (unsigned int)(fill[tid] * (int)sizeof(u64));
            const u64 limit = thr[wave * 32 + qn];
            // ~0 is "no threshold yet": its distance field does not decode to a number.
            limit_d = limit == ~0ull ? INFINITY : key_distance(limit);
        };
        const int valid = min(max(N - (q0 + wave * 32), 0), 32);  // this wave's queries
        const unsigned int all_queries = valid == 32 ? ~0u : (1u << valid) - 1u;

        v8h bq[S];
        HalfQuery hq;
        {
            const v4f *src = reinterpret_cast<const v4f *>(points) + (size_t)qt * kMain + (size_t)wave * S * 64 + lane;
#pragma unroll
            for (int k = 0; k < S; ++k) bq[k] = __builtin_bit_cast(v8h, src[k * 64]);
        }
        const float2 len = cold()->point_len[q];
        hq = half_query(len.x, len.y, cold()->D, back);
        hq.kap = uniform(hq.kap);
        hq.least = uniform(hq.least);
        const int own_frame = __builtin_amdgcn_readfirstlane(__float_as_int(cold()->tile_info[qt].z));
        tile_beta = cold()->beta + (size_t)own_frame * cold()->beta_pitch;
        // The query's betas: the two lanes of a query have the even and the odd frames'.
        v8f query_beta;
        const int odd = here(kh);
#pragma unroll
        for (int f = 0; f < kFrames / 2; ++f) query_beta[f] = cold()->beta[(size_t)(2 * f + odd) * cold()->beta_pitch + q];
        const float my_d2 = cold()->frame_d2[own_frame * kFrames + (lane & (kFrames - 1))];  // a frame per lane
        const float my_frame_len = length_bound(my_d2, cold()->D);

        unsigned int buf = 0;  // byte offset of the LDS buffer that holds the tile at hand: 0 or kTile * 16
        // One tile: compute it from LDS buffer `buf` while the next one travels into the other.
        auto process = [&](int ct, int next_ct) {
            const int c0 = ct * kCT;
            const v4f *tile = reinterpret_cast<const v4f *>(lds_raw + buf);
            // All operands of the first two blocks of candidates are asked for before their first product, those of the others
            // as registers come free; and all products are under way before the first result is looked at: the filter of
            // the first two blocks runs beside the products of the others.
            v4f a[4][S];
            float start[2];
            auto load_start = [&](int pair) { start[pair] = reinterpret_cast<const float *>(tile + kMain)[64 * pair + lane]; };
            auto load_step = [&](int pair, int k) {
                a[2 * pair][k] = tile[(2 * pair * S + k) * 64 + lane];
                a[2 * pair + 1][k] = tile[((2 * pair + 1) * S + k) * 64 + lane];
            };
            // The accumulators start from the betas by a product of a column of them and a row of ones: one word of LDS per
            // lane and two blocks, where loading every lane's sixteen of a block takes as much of the LDS as the operands.
            v16f acc[4];
            auto multiply = [&](int pair) {
                const v32f both = __builtin_amdgcn_mfma_f32_32x32x1f32(start[pair], 1.0f, v32f{}, 0, 0, 0);
                acc[2 * pair] = __builtin_shufflevector(both, both, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
                acc[2 * pair + 1] = __builtin_shufflevector(both, both, 16, 17, 18, 19, 20, 21, 22, 23, 24, 25, 26, 27, 28, 29, 30, 31);
                if (pair == 0) load_start(1);
#pragma unroll
                for (int k = 0; k < S; ++k) {
#pragma unroll
                    for (int b = 2 * pair; b < 2 * pair + 2; ++b)
                        acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a[b][k]), bq[k], acc[b], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (pair == 0) load_step(1, k);
                }
            };
            load_start(0);
#pragma unroll
            for (int k = 0; k < S; ++k) load_step(0, k);
            const v4f info = tile[kMain + kCT / 4];
            __builtin_amdgcn_sched_barrier(0);
            multiply(0);
            __builtin_amdgcn_sched_barrier(0);
            fetch(next_ct >= 0 ? next_ct : ct, kTile * 16 - buf);  // (last read a tile ago, before the barrier that ended that tile)
            __builtin_amdgcn_sched_barrier(0);
            multiply(1);
            __builtin_amdgcn_sched_barrier(0);
            const int frame = __builtin_amdgcn_readfirstlane(__float_as_int(info[2]));
            if (frame != hq.frame) {
                const unsigned int mine = __float_as_uint(query_beta[frame >> 1]);
                const auto halves = __builtin_amdgcn_permlane32_swap(mine, mine, false, false);
                const float beta = __uint_as_float((frame & 1) ? halves[1] : halves[0]) * back;
                enter_frame(hq, frame, beta, __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(my_d2), frame)),
                            __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(my_frame_len), frame)));
            }
            // Distance less its bound = off + product * back; what is tested is the product.  (Never -inf: excluded
            // elements must fail also while the query has no threshold.)
            not_counted = home ? (unsigned int)kNotCounted : 0u;
            const float off = tile_offset(hq, info[0], info[1]);
            const float limit_acc = ((off - limit_d) - 4e-7f * (fabsf(off) + fabsf(limit_d))) * s2;
            const float lim = live ? fmaxf(limit_acc, -3.4028234663852886e38f) : INFINITY;
            // The largest of each run of eight results: a run in which no lane of the wave passes is skipped.  (Element v of
            // run r is candidate c0 + 16 r + 4 kh + v + (v & 4).)
            float run_max[8];
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const v16f &x = acc[r >> 1];
                const int o = 8 * (r & 1);
                float m = matrix_result(x[o + 7]);
                m = max3(m, x[o], x[o + 1]);
                m = max3(m, x[o + 2], x[o + 3]);
                m = max3(m, x[o + 4], x[o + 5]);
                run_max[r] = max2(m, x[o + 6]);
            }
            if (TSNE_UNLIKELY(measure)) {
                float *to = reinterpret_cast<float *>(reinterpret_cast<char *>(list) + region + half * (sizeof(u64) / 2)) + min(minima, half - 1);
                auto key = [&](float p) { return fmaxf(fmaf(p, back, off), 0.0f); };
                if (home) {
                    v4f *const to4 = reinterpret_cast<v4f *>(to);
                    to4[0] = v4f{key(run_max[0]), key(run_max[1]), key(run_max[2]), key(run_max[3])};
                    to4[1] = v4f{key(run_max[4]), key(run_max[5]), key(run_max[6]), key(run_max[7])};
                    minima += 8;
                } else {
                    float m = max3(run_max[0], run_max[1], run_max[2]);
                    m = max3(m, run_max[3], run_max[4]);
                    *to = key(max2(max3(m, run_max[5], run_max[6]), run_max[7]));
                    ++minima;
                }
            } else {
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    if (TSNE_LIKELY(__ballot(run_max[r] >= lim) == 0)) continue;
                    const v16f &x = acc[r >> 1];
                    const int o = 8 * (r & 1);
                    // All eight comparisons first: a branch on a comparison just made waits for it.
                    u64 any[8];
#pragma unroll
                    for (int v = 0; v < 8; ++v) any[v] = __ballot(x[o + v] >= lim);
#pragma unroll
                    for (int v = 0; v < 8; ++v) {
                        if (TSNE_LIKELY(any[v] == 0)) continue;
                        asm volatile("");  // (a scalar branch, not a condition more for the lanes)
                        const float p = x[o + v];
                        const int j = c0 + 16 * r + 4 * (here(lane) >> 5) + v + (v & 4);  // (formed here, not held in registers)
                        if (p >= lim && j != q) {
                            *reinterpret_cast<u64 *>(reinterpret_cast<char *>(list) + my_at) =
                                pack_key_positive(fmaxf(fmaf(p, back, off), 0.0f), (int)((unsigned int)j | not_counted));
                            my_at += (unsigned int)sizeof(u64);
                            not_counted = (unsigned int)kNotCounted;
                        }
                    }
                }
            }
            wait_for_loads();  // (the next tile is in LDS)
            __syncthreads();
            buf = kTile * 16 - buf;
        };

        const int reach = max(kHomeTiles / P, 2) * P;  // (at least two tiles either side of every part)
        const int h0 = max(qt - reach, 0), h1 = min(qt + reach, T - 1);
        int word_idx = -1;
        unsigned int cur_word = 0u;
        // Next set bit of the bitmap, ascending within a round; every wave walks the same words, sixty-four at a time.  Round
        // k takes the tiles that are `first` modulo 256, 64, 16, 4 and 1, without those of the rounds before it.
        int round = kRankRounds, first_round = kRankRounds, last_round = kRankRounds;
        const int first = (int)((unsigned int)(w / (int)gridDim.x) * 0x9E3779B1u >> 24);
        auto round_mask = [&](int k, int word) -> unsigned int {
            return k == 0   ? ((word & 7) == first >> 5 ? 1u << (first & 31) : 0u)
                   : k == 1 ? ((word & 1) == ((first >> 5) & 1) ? 1u << (first & 31) : 0u)
                   : k == 2 ? 0x00010001u << (first & 15)
                   : k == 3 ? 0x11111111u << (first & 3)
                            : ~0u;
        };
        bool round_over = false;  // the tile returned last was the last of its round
        auto next_tile = [&]() -> int {
            if (TSNE_UNLIKELY(cur_word == 0u)) {
                const int lane = here(threadIdx.x) & 63;
                for (;;) {
                    const int word = word_idx + 1 + lane;
                    unsigned int bits = word < cold()->bitmap_words ? bitmap[word] : 0u;
                    bits &= round_mask(round, word) & ~(round > first_round ? round_mask(round - 1, word) : 0u);
                    const u64 some = __ballot(bits != 0u);
                    if (some) {
                        const int l = __ffsll((long long)some) - 1;
                        cur_word = (unsigned int)__builtin_amdgcn_readlane((int)bits, l);
                        word_idx += 1 + l;
                        break;
                    }
                    word_idx += kWave;
                    if (word_idx + 1 >= cold()->bitmap_words) {
                        if (round == last_round) return -1;
                        ++round;
                        round_over = true;
                        word_idx = -1;
                    }
                }
            }
            const int b = __ffs((int)cur_word) - 1;
            cur_word &= cur_word - 1u;
            return word_idx * 32 + b;
        };
        // From rounds `from` to `to`: the first tile of theirs.
        auto start_rounds = [&](int from, int to) -> int {
            home = false;
            round = first_round = from;
            last_round = to;
            word_idx = -1;
            cur_word = 0u;
            const int t = next_tile();
            round_over = false;
            return t;
        };
        // Thresholds from the measured distances: the one of rank `rank` of a query's two lanes'.
        auto take_thresholds = [&](int rank) {
            asm volatile("" ::: "memory");
            minima = min(minima, half);
            const int lane = here(threadIdx.x) & 63;
            for (int b = 0; b < valid; ++b) {
                const unsigned int *from = reinterpret_cast<const unsigned int *>(list + (size_t)(wave * 32 + b) * cap + half / 2);
                unsigned int rated[NK];
                int ranked = 0;
#pragma unroll
                for (int u = 0; u < NK; ++u) {
                    const int e = u * kWave + lane;
                    rated[u] = ~0u;
                    if (e < 2 * minima) rated[u] = from[e < minima ? e : 2 * half + e - minima] | 0x80000000u;
                    if (rated[u] >= 0xff800000u) rated[u] = ~0u;  // (no candidate in it)
                    ranked += __popcll(__ballot(rated[u] != ~0u));
                }
                if (ranked < rank) continue;
                int at_under, at_hi;
                const unsigned int limit = ranked_limit<NK>(rated, ranked, rank, rank / 16, at_under, at_hi);
                if (lane == 0) thr[wave * 32 + b] = min(thr[wave * 32 + b], ((u64)limit << 32) | 0xffffffffull);
            }
            minima = 0;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const u64 limit = thr[wave * 32 + (lane & 31)];
            limit_d = limit == ~0ull ? INFINITY : key_distance(limit);
        };
        // The tiles that some query of the tile may want, by the thresholds so far: their number.
        auto map_tiles = [&]() -> int {
            const int tid = here(threadIdx.x), lane = tid & 63;
            for (int k = tid; k < cold()->bitmap_words; k += 256) bitmap[k] = 0u;
            if (tid < cold()->D) qcenter[tid] = cold()->centers_t[(size_t)tid * T + qt];
            __syncthreads();
            if (tid < kMQ) {
                // Largest squared distance any query of the tile would still accept (rounded up).
                float v = -INFINITY;
                if (q0 + tid < N) {
                    const u64 t = thr[tid];
                    v = t == ~0ull ? INFINITY : key_distance(t);
                    v += 1e-5f * fabsf(v) + 1e-30f;
                }
                v = group_max<kWave>(v);
                if (lane == 0) tmax_part[tid >> 6] = v;
            }
            __syncthreads();
            const float tmax = fmaxf(tmax_part[0], tmax_part[1]);
            const float *radius = cold()->radius, *centers_t = cold()->centers_t;
            const float ra = radius[qt];
            for (int t = tid; t < T; t += 256)
                if ((t < h0 || t > h1) && t % P == part && tile_may_matter(qcenter, ra, centers_t, radius, cold()->D, T, t, tmax))
                    atomicOr(&bitmap[t >> 5], 1u << (t & 31));
            __syncthreads();
            int visits = 0;
            for (int k = lane; k < cold()->bitmap_words; k += kWave) visits += __popc(bitmap[k]);
            return __builtin_amdgcn_readfirstlane(group_sum_int(visits));
        };
        const int home_first = h0 + (part - h0 % P + P) % P;  // this part's first tile of the neighbourhood
        int cur = home_first <= h1 ? home_first : -1;          // (fewer tiles than parts: nothing for this part, its lists stay empty)
        const bool beyond = h0 > 0 || h1 < T - 1;
        // The passes over a query tile's tiles.  The neighbourhood is measured first, where that gives distances enough, so
        // that the lists begin with a threshold, and so is, where there are many of them, a sample of the tiles beyond.
        enum { kMeasureHome, kListHome, kMeasureRounds, kListRounds, kDone };
        int pass = beyond && cur >= 0 && 16 * ((h1 - home_first) / P + 1) > want + want / 8 ? kMeasureHome : kListHome;
        measure = pass == kMeasureHome;
        int sample = kRankRounds;  // the round whose tiles are measured (kRankRounds: none)
        if (cur >= 0) fetch(cur, 0);
        wait_for_loads();
        __syncthreads();
        unsigned int swept = 0;
        while (cur >= 0) {
            round_over = false;
            int nxt;
            if (TSNE_UNLIKELY(home)) nxt = cur + P <= h1 ? cur + P : -1;
            else nxt = next_tile();
            process(cur, nxt);
            swept += measure ? 0 : 1;  // (those measured first are not skipped later, and counted then)
            if (TSNE_LIKELY(nxt >= 0 && !round_over && __ballot(my_fill() > half - kCT / 2) == 0)) {
                cur = nxt;
                continue;
            }
            if (nxt >= 0) {
                // Lists that a further tile could overflow are compacted by their own wave, right away (a region takes at
                // most 64 entries per tile); all of them after a round, for thresholds.  (A list whose counted entries are
                // too few for a rank keeps all it has, full or not, and so may one whose entries are equally far: those are
                // compacted like any other before the next tile.)
                const auto crowded = [&]() -> unsigned int {
                    const u64 lanes = __ballot(my_fill() > half - kCT / 2);
                    return (unsigned int)(lanes | (lanes >> 32));  // lanes l, l+32 share a query
                };
                if (round_over) select_queries(all_queries, cold()->ranks[round - 1], 0, true);
                const unsigned int mask = crowded();
                if (mask) select_queries(mask, want, cold()->select_slack, false);
                cur = nxt;
                continue;
            }
            // A pass is over: on to the next that has tiles.
            while (nxt < 0 && pass != kDone) {
                measure = false;
                if (pass == kMeasureHome) {
                    take_thresholds(want + 1);  // (the query itself is the nearest of one run)
                    pass = kListHome;
                    nxt = home_first;
                } else if (pass == kListHome && beyond) {
                    select_queries(all_queries, want, 0, false);
                    const int visits = map_tiles();
                    if (P == 1 && visits >= kRoundTiles) sample = visits <= 16 * kSampleTiles ? 2 : visits <= 64 * kSampleTiles ? 1 : 0;
                    measure = sample < kRankRounds;
                    pass = measure ? kMeasureRounds : kListRounds;
                    nxt = start_rounds(sample, sample);
                } else if (pass == kMeasureRounds) {
                    take_thresholds(cold()->ranks[sample]);
                    pass = kListRounds;
                    nxt = start_rounds(sample + 1, kRankRounds);
                } else {
                    pass = kDone;
                }
            }
            if (nxt >= 0) fetch(nxt, buf);  // the barrier that ended the last tile freed both buffers
            wait_for_loads();
            __syncthreads();
            cur = nxt;
        }
        select_queries(all_queries, want, 0, false);
        if (tid == 0) atomicAdd(cold()->tiles_swept, (unsigned long long)swept);
        // Output, every wave for its own queries.
        const int lane = here(threadIdx.x) & 63;
        for (int b = 0; b < valid; ++b) {
            const int ql = wave * 32 + b;
            const int n = fill[wave * 64 + b] + fill[wave * 64 + b + 32];
            const u64 *lq = list + (size_t)ql * cap;  // entry e of the n kept: region e & 1, position e >> 1
            const size_t row = (size_t)qt * kMQ + ql;
            if (P == 1) {
                for (int e = lane; e < want; e += kWave)
                    cold()->cand[row * want + e] = e < n ? key_index(lq[(e & 1) * half + (e >> 1)] & ~kNotCounted) : -1;
                // Every candidate that was dropped, by a compaction or by the filter, had a distance >= the
                // threshold of the moment, and thresholds only decrease.
                if (lane == 0) cold()->tau[row] = thr[ql] == ~0ull ? INFINITY : key_distance(thr[ql]);
            } else {
                u64 *dst = cold()->part_keys + (((size_t)qi * kMQ + ql) * P + part) * want;
                for (int e = lane; e < want; e += kWave)
                    dst[e] = e < n ? lq[(e & 1) * half + (e >> 1)] & ~kNotCounted : ~0ull;
            }
        }
        __syncthreads();  // before the next query tile re-initialises thr and the LDS tiles
    }
}

// ---------------------------------------------------------------------------
// MFMA sweep for more dimensions than one wave's registers hold (more than 126).
// The k-steps are cut into chunks of kChunkSteps (64 dimensions).  Per candidate tile and chunk the
// workgroup keeps the chunk of the tile in LDS (on floats 32 KB, layout [block (4)][step group (8)][lane (64)]
// float4, copied verbatim from the packed points), every wave loads the same chunk of its 32 queries
// from the packed query-side copy (already scaled: -2 q_d, 1 in the |c|^2 row) and the products of
// all four candidate blocks accumulate over the chunks in 64 registers.  The next chunk of the queries travels
// into registers meanwhile, and so, on floats and bf16 terms, does the next of the tile (or the first of the next tile); on
// halves that goes straight into a second LDS buffer.  Visiting order, tile skipping, filter, lists and output are those of
// the kernel above.
// Halves: a chunk is 64 dimensions, 16 KB (two LDS buffers) as [block (4)][step of 16 dimensions (4)][lane (64)] 8 halves, one
// product a step, for either side of the products the same packed points (half_pack_kernel), and the accumulators start from
// the betas.
// BF16 = true: a chunk is 32 dimensions, 16 KB (two LDS buffers) as [block (4)][term (2)][step of 16 dimensions (2)][lane (64)]
// 8 x bf16 of the points relative to their tile's centre, the query side two terms of -2 q likewise, and the
// products are those of the kernel above (three v_mfma_f32_32x32x16_bf16 per step); |q - centre|^2 is summed
// over the chunks from the query side's two terms and the centre's chunk (pack_chunked_centres_kernel), and
// the keys are lower bounds of the distances as there.
// Dynamic LDS: 32 KB for one tile chunk or two, one sort buffer (cap keys) per wave, the visit bitmap, D floats
// (centre of the query tile's ball).
// ---------------------------------------------------------------------------
constexpr int kChunkSteps = 32;
constexpr int kChunkS4 = kChunkSteps / 4;            // float4 per lane, block and chunk
constexpr int kChunkFloat4 = 4 * kChunkS4 * 64;      // float4 per tile chunk

// TABLE (bf16): |q - m|^2 comes from a table of all queries and tile centres, formed beforehand; otherwise every wave
// forms it chunk by chunk from the query's own two terms and the centre's chunk, which is five vector instructions
// per coordinate and 16 registers beside the matrix instructions (sweeps of 50000 x 1024: 27.5 -> 24.3 ms and 1.2 for
// the table; 60000 x 784: 13.7 -> 11.9 and 1.1).
constexpr int kSweepXcds = 8;
template <Products PRODUCTS, bool TABLE>
__global__ __launch_bounds__(256, 2) void knn_mfma_chunked_sweep_kernel(const SweepArgs args) {
    constexpr bool BF16 = PRODUCTS == Products::kBf16, HALF = PRODUCTS == Products::kHalf;
    const int N = args.N, D = args.D, want = args.want, cap = args.cap;
    const int num_qtiles = args.num_qtiles, n_chunks = args.n_chunks;
    u64 *__restrict__ lists = args.lists;
    int *__restrict__ cand = args.cand;
    float *__restrict__ tau = args.tau;
    // Slots of 16 bytes per lane, block and chunk: 8 groups of four k-steps (64 dimensions) on floats; on bf16
    // terms 2 terms x 2 steps of 16 dimensions (32 dimensions: with 64 the chunk loop's registers did not fit
    // and the compiler spilled the prefetched chunks the moment they were loaded).
    // halves 4 steps of 16 dimensions (64): sweeps of 50000 x 1024 21.8 -> 11.9 ms, of 60000 x 784 9.2 -> 5.7.  Straight into
    // LDS and with a step's operands ahead of the products of the one before, searches of 60000 x 784 10.5 -> 10.0, of
    // 40000 x 200 5.8 -> 5.5.
    constexpr int kSlots = BF16 || HALF ? 4 : kChunkS4;
    constexpr int kSteps16 = 2;                     // bf16: steps of 16 dimensions per chunk
    constexpr int kChunkF4 = 4 * kSlots * 64;       // float4 per tile chunk
    // bf16 and halves: two LDS buffers of 16 KB, so that the next chunk goes to LDS while the other waves may still read the
    // current one, and one workgroup barrier per chunk does (floats: one buffer of 32 KB, two barriers).
    constexpr int kBufs = BF16 || HALF ? 2 : 1;
    int buf = 0;  // the buffer that holds the chunk being computed
    const size_t tile_stride = (size_t)n_chunks * kChunkF4;  // float4 per packed tile
    const size_t block_stride = (size_t)n_chunks * kSlots * 64;  // float4 per 32-point block of a tile
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    v4f *a_lds = reinterpret_cast<v4f *>(lds_raw);
    u64 *sortbuf = reinterpret_cast<u64 *>(a_lds + kBufs * kChunkF4) + (size_t)(threadIdx.x >> 6) * cap;  // per wave
    unsigned int *bitmap = reinterpret_cast<unsigned int *>(reinterpret_cast<u64 *>(a_lds + kBufs * kChunkF4) + 4 * (size_t)cap);
    float *qcenter = reinterpret_cast<float *>(bitmap + args.bitmap_words);
    __shared__ u64 thr[kMQ];
    __shared__ int cnt[kMQ];
    __shared__ unsigned int hist_all[4][kWave];
    __shared__ float tmax_part[2];
    __shared__ v4f beta_lds[HALF ? 2 * (kCT / 4) : 1];  // halves: what the accumulators start from, by parity of the tile

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int qn = lane & 31, kh = lane >> 5;
    u64 *list = lists + (size_t)blockIdx.x * kMQ * cap;
    const float half_s = HALF ? half_scale_factor(args.half_scale) : 1.0f, half_s2 = 0.5f * half_s * half_s;
    const float half_back = -1.0f / half_s2;  // (a power of two)
    const float *tile_beta = nullptr;         // of the query tile's frame
    int parity = 0;

    // Chunk c of a candidate tile: global -> registers -> LDS.  Element e = 256 r + tid of the chunk is
    // float4 (e % 512) of block e / 512 = r / 2.  (Halves: straight into LDS buffer b, block r by the 256 threads' r-th
    // load; with a tile's first chunk its betas, by the first wave.)
    v4f stage[HALF ? 1 : kSlots];
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    const unsigned int lane_byte = (unsigned int)tid * 16u;
    auto fetch_half = [&](int tile, int c, int b) {
        const float4 *src = args.Xp + (size_t)tile * tile_stride + (size_t)c * (kSlots * 64);
        unsigned int to = __builtin_amdgcn_readfirstlane((unsigned int)(size_t)(LdsByte *)lds_raw) + (unsigned int)(b * kChunkF4 * 16 + wave_u * 1024);
        asm volatile("" : "+s"(to));
#pragma unroll
        for (int r = 0; r < 4; ++r) load_to_lds(src + r * block_stride, lane_byte, to + r * 4096u);
        if (c == 0 && wave_u == 0 && lane < kCT / 4)
            load_to_lds(tile_beta + (size_t)tile * kCT, lane_byte,
                        __builtin_amdgcn_readfirstlane((unsigned int)(size_t)(LdsByte *)beta_lds) + (unsigned int)(parity ^ 1) * (kCT * 4));
    };
    auto fetch = [&](int tile, int c) {
        const v4f *src = reinterpret_cast<const v4f *>(args.Xp) + (size_t)tile * tile_stride + (size_t)c * (kSlots * 64) + tid;
        // element 256 r + tid of the chunk: block (256 r + tid) / (64 kSlots), float4 (256 r + tid) % (64 kSlots) of it
#pragma unroll
        for (int r = 0; r < kSlots; ++r)
            stage[r] = src[(size_t)((256 * r) / (64 * kSlots)) * block_stride + (256 * r) % (64 * kSlots)];
    };
    auto stash = [&](int b) {
#pragma unroll
        for (int r = 0; r < kSlots; ++r) a_lds[b * kChunkF4 + r * 256 + tid] = stage[r];
    };
    const int num_ctiles = (N + kCT - 1) / kCT;

    const int P = args.parts;
    // The parts of a query tile go to workgroups of one XCD, which read the tile's operands at about the same time, and so do
    // query tiles next to each other, which visit much the same candidate tiles.  (Workgroups go to the XCDs round robin; the
    // grid is a multiple of their number times P.  50000 x 1024: 64 % of the requests missed the L2 with the parts dealt to all
    // XCDs, and the sweep went at the rate of the cache behind it, 7 TB/s; 46 % so, 12.0 -> 10.3 ms.)
    const int round_tiles = (int)gridDim.x / P, xcd = (int)blockIdx.x % kSweepXcds;
    const int in_xcd = (int)blockIdx.x / kSweepXcds, part = in_xcd % P;
    for (int round = 0; round < num_qtiles; round += round_tiles) {
        const int tiles = min(round_tiles, num_qtiles - round);  // of this round, dealt out evenly
        const int qi = round + xcd * tiles / kSweepXcds + in_xcd / P;
        if (qi >= round + (xcd + 1) * tiles / kSweepXcds) continue;
        const int qt = args.qtile_list ? args.qtile_list[qi] : args.qtile_first + qi * args.qtile_step;
        const int q0 = qt * kMQ;
        const int q = q0 + wave * 32 + qn;  // this lane's query (>= N in the last tile: padded zeros)
        if (tid < kMQ) {
            thr[tid] = ~0ull;
            cnt[tid] = 0;
        }
        const float q_len = BF16 && q < N ? sqrtf(args.norms[q]) * (1.0f + 1e-6f) : 0.0f;  // |q|, rounded up
        HalfQuery hq = {};
        int own_frame = 0;
        if constexpr (HALF) {
            const float2 len = args.point_len[q];
            hq = half_query(len.x, len.y, D, half_back);
            own_frame = __builtin_amdgcn_readfirstlane(__float_as_int(args.tile_info[qt].z));
            tile_beta = args.beta + (size_t)own_frame * args.beta_pitch;
        }
        // This wave's block of the query-side copy.
        const v4f *bsrc = reinterpret_cast<const v4f *>(args.Bp) + (size_t)qt * tile_stride + (size_t)wave * block_stride + lane;
        v4f bcur[kSlots], bnext[kSlots];
#pragma unroll
        for (int s4 = 0; s4 < kSlots; ++s4) bcur[s4] = bsrc[s4 * 64];

        // One tile: its first chunk is in LDS and the queries' first chunk in bcur on entry; the same holds
        // for next_ct on exit.
        auto process = [&](int ct, int next_ct) {
            const int c0 = ct * kCT;
            // (nothing is in flight as far as the compiler can tell, or it waits in the chunk loop, and for the loads to LDS too)
            if constexpr (HALF) wait_for_loads();
            v16f acc[4];
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    v4f start = {0.0f, 0.0f, 0.0f, 0.0f};
                    if constexpr (HALF) start = beta_lds[parity * (kCT / 4) + 8 * b + 2 * g + kh];
#pragma unroll
                    for (int k = 0; k < 4; ++k) acc[b][4 * g + k] = start[k];
                }
            // bf16: this lane's share of |q - m|^2 (m: the tile's centre), or all of it from the table
            float f_part = 0.0f;
            if constexpr (TABLE) f_part = args.centre_dist[(size_t)ct * args.centre_pitch + q];
            // (`last` a type of its own on halves: with one body for all chunks there is a path, never taken, from the last
            // chunk's loads to the next chunk, and on it the compiler waits for all loads there)
            auto chunk = [&](int c, auto last) {
                v4f mc[2 * kSteps16];  // bf16: the centre's 16 coordinates that go with this lane's 16 of the chunk
                if constexpr (BF16 && !TABLE) {
                    const v4f *msrc = reinterpret_cast<const v4f *>(args.centres_p) + (size_t)ct * (8 * n_chunks) + 8 * c + 2 * kh;
#pragma unroll
                    for (int step = 0; step < kSteps16; ++step) {
                        mc[2 * step] = msrc[4 * step];
                        mc[2 * step + 1] = msrc[4 * step + 1];
                    }
                }
                if constexpr (HALF) {
                    // (the buffer was last read a chunk ago, before the barrier that ended that chunk)
                    if (!last || next_ct >= 0) fetch_half(last ? next_ct : ct, last ? 0 : c + 1, buf ^ 1);
                } else {
                    if (!last) fetch(ct, c + 1);
                    else if (next_ct >= 0) fetch(next_ct, 0);
                }
                {
                    const v4f *bn = bsrc + (size_t)(last ? 0 : c + 1) * (kSlots * 64);
#pragma unroll
                    for (int s4 = 0; s4 < kSlots; ++s4) bnext[s4] = bn[s4 * 64];
                }
                if constexpr (HALF) {
                    // (a step's operands are asked for ahead of the products of the step before)
                    v4f x[2][4];
                    auto load_step = [&](int step) {
#pragma unroll
                        for (int b = 0; b < 4; ++b) x[step & 1][b] = a_lds[buf * kChunkF4 + (b * kSlots + step) * 64 + lane];
                    };
                    load_step(0);
                    load_step(1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int step = 0; step < kSlots; ++step) {
                        const v8h qh = __builtin_bit_cast(v8h, bcur[step]);
#pragma unroll
                        for (int b = 0; b < 4; ++b)
                            acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, x[step & 1][b]), qh, acc[b], 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        if (step + 2 < kSlots) load_step(step + 2);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else if constexpr (BF16) {
#pragma unroll
                    for (int step = 0; step < kSteps16; ++step) {
                        v4f xh[4], xl[4];
#pragma unroll
                        for (int b = 0; b < 4; ++b) {
                            xh[b] = a_lds[buf * kChunkF4 + (b * kSlots + step) * 64 + lane];
                            xl[b] = a_lds[buf * kChunkF4 + (b * kSlots + kSteps16 + step) * 64 + lane];
                        }
                        const v8bf qh = __builtin_bit_cast(v8bf, bcur[step]), ql = __builtin_bit_cast(v8bf, bcur[kSteps16 + step]);
#pragma unroll
                        for (int b = 0; b < 4; ++b)
                            acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, xh[b]), qh, acc[b], 0, 0, 0);
#pragma unroll
                        for (int b = 0; b < 4; ++b)
                            acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, xh[b]), ql, acc[b], 0, 0, 0);
#pragma unroll
                        for (int b = 0; b < 4; ++b)
                            acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, xl[b]), qh, acc[b], 0, 0, 0);
                        if constexpr (!TABLE) {
                            // |q - m|^2 from the query's two terms: q_d = -(high + low) / 2 to within 2^-16 |q_d|.
                            const uint4 uh = __builtin_bit_cast(uint4, bcur[step]), ul = __builtin_bit_cast(uint4, bcur[kSteps16 + step]);
                            const unsigned int wh[4] = {uh.x, uh.y, uh.z, uh.w}, wl[4] = {ul.x, ul.y, ul.z, ul.w};
                            const float m[8] = {mc[2 * step][0], mc[2 * step][1], mc[2 * step][2], mc[2 * step][3],
                                                mc[2 * step + 1][0], mc[2 * step + 1][1], mc[2 * step + 1][2], mc[2 * step + 1][3]};
#pragma unroll
                            for (int k = 0; k < 4; ++k) {
                                const float s0 = __uint_as_float(wh[k] << 16) + __uint_as_float(wl[k] << 16);
                                const float s1 = __uint_as_float(wh[k] & 0xffff0000u) + __uint_as_float(wl[k] & 0xffff0000u);
                                const float e0 = fmaf(-0.5f, s0, -m[2 * k]), e1 = fmaf(-0.5f, s1, -m[2 * k + 1]);
                                f_part = fmaf(e0, e0, f_part);
                                f_part = fmaf(e1, e1, f_part);
                            }
                        }
                    }
                } else {
#pragma unroll
                    for (int s4 = 0; s4 < kChunkS4; ++s4) {
                        v4f x[4];
#pragma unroll
                        for (int b = 0; b < 4; ++b) x[b] = a_lds[(b * kChunkS4 + s4) * 64 + lane];
#pragma unroll
                        for (int k = 0; k < 4; ++k)
#pragma unroll
                            for (int b = 0; b < 4; ++b)
                                acc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[b][k], bcur[s4][k], acc[b], 0, 0, 0);
                    }
                }
                if (!last) {
                    if constexpr (HALF) {
                        wait_for_loads();  // (the next chunk is in LDS)
                        __syncthreads();
                        buf ^= 1;
                    } else if constexpr (BF16) {
                        stash(buf ^ 1);  // (last read a chunk ago, before the barrier that ended that chunk)
                        __syncthreads();
                        buf ^= 1;
                    } else {
                        __syncthreads();  // all waves have read this chunk
                        stash(0);
                        __syncthreads();
                    }
#pragma unroll
                    for (int s4 = 0; s4 < kSlots; ++s4) bcur[s4] = bnext[s4];
                }
            };
            if constexpr (HALF) {
                for (int c = 0; c + 1 < n_chunks; ++c) chunk(c, std::false_type());
                chunk(n_chunks - 1, std::true_type());
            } else {
                for (int c = 0; c < n_chunks; ++c) chunk(c, c + 1 == n_chunks);
            }
            const u64 limit = thr[wave * 32 + qn];
            // ~0 is "no threshold yet": its distance field does not decode to a number.
            const float limit_d = limit == ~0ull ? INFINITY : key_distance(limit);
            // Never +inf: excluded elements are raised to +inf and must fail the test also while the query
            // has no threshold yet (a part can hold fewer than `want` real candidates, so nothing would
            // push them out of the list later).
            // bf16: the keys are lower bounds of the distances: product + `off`, off = |q - m|^2 rounded down
            // (the rounding of its sum, and, formed from the query's two terms, the 2^-16 |q| by which they miss q)
            // less the tile's error bound; the products are tested against the threshold less `off`, rounded up.
            float off = 0.0f, limit_acc = limit_d;
            if constexpr (HALF) {
                // Distance less its bound = off - product / half_s2; what is tested is the product.
                const float4 info = args.tile_info[__builtin_amdgcn_readfirstlane(ct)];
                const int frame = __builtin_amdgcn_readfirstlane(__float_as_int(info.z));
                if (frame != hq.frame) {
                    const float d2 = args.frame_d2[own_frame * kFrames + frame];
                    enter_frame(hq, frame, args.beta[(size_t)frame * args.beta_pitch + q] * half_back, d2, length_bound(d2, D));
                }
                off = tile_offset(hq, info.x, info.y);
                limit_acc = ((off - limit_d) - 4e-7f * (fabsf(off) + fabsf(limit_d))) * half_s2;
            }
            if constexpr (BF16) {
                const float f = TABLE ? f_part : f_part + __shfl_xor(f_part, 32);
                off = f * (1.0f - (float)(D + 4) * 5.9604644775390625e-08f);
                if constexpr (!TABLE) off -= 2.1f / 65536.0f * q_len * sqrtf(f);
                off -= fmaf(q_len, args.tile_coef[2 * ct], args.tile_coef[2 * ct + 1]);
                limit_acc = limit_d - off;
                limit_acc += 2.4e-7f * (fabsf(limit_d) + fabsf(off));
            }
            // (halves: the accumulators fall as the distance grows, and everything is the other way round)
            auto passes = [](float v, float limit) { return HALF ? v >= limit : v <= limit; };
            constexpr float kNever = HALF ? -INFINITY : INFINITY, kMost = 3.4028234663852886e38f;
            const float lim = q < N ? (HALF ? fmaxf(limit_acc, -kMost) : fminf(limit_acc, kMost)) : -kNever;
            const bool edge_tile = c0 + kCT > N || (unsigned int)(q0 - c0) < (unsigned int)kCT;
#pragma unroll
            for (int cb = 0; cb < 4; cb += 2) {
                v16f &acc0 = acc[cb], &acc1 = acc[cb + 1];
                // Register v of lane l holds candidate row 8*(v/4) + 4*(l/32) + v%4 of the block, query column l%32.
                float best = matrix_result(acc0[0]);
#pragma unroll
                for (int v = 1; v + 1 < 16; v += 2) best = extreme3<HALF>(best, acc0[v], acc0[v + 1]);
                best = extreme3<HALF>(best, acc0[15], matrix_result(acc1[0]));
#pragma unroll
                for (int v = 1; v + 1 < 16; v += 2) best = extreme3<HALF>(best, acc1[v], acc1[v + 1]);
                best = extreme2<HALF>(best, acc1[15]);
                if (passes(best, limit_acc)) {
                    const int jbase = c0 + cb * 32 + 4 * kh;  // element (half, v) is candidate jbase + 32 half + 8 (v / 4) + v % 4
                    // Candidates beyond N (last tile) and the query itself (its own tile) are raised to +inf.
                    if (edge_tile) {
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            const int j = jbase + 8 * (e >> 2) + (e & 3);
                            if (j >= N || j == q) acc0[e] = kNever;
                            if (j + 32 >= N || j + 32 == q) acc1[e] = kNever;
                        }
                    }
                    // Count, reserve the list slots with one LDS atomic, then store the keys.
                    int n = 0;
#pragma unroll
                    for (int e = 0; e < 32; ++e) n += passes(e < 16 ? acc0[e & 15] : acc1[e & 15], lim) ? 1 : 0;
                    if (n != 0) {
                        const int slot = atomicAdd(&cnt[wave * 32 + qn], n);
                        u64 *dst = list + (size_t)(wave * 32 + qn) * cap + slot;
                        float lim2 = lim;
                        asm volatile("" : "+v"(lim2));  // compare again rather than keep 32 lane masks alive
#pragma unroll
                        for (int e = 0; e < 32; ++e) {
                            const float dist = e < 16 ? acc0[e & 15] : acc1[e & 15];
                            const int j = jbase + 32 * (e >> 4) + 8 * ((e & 15) >> 2) + (e & 3);
                            if (passes(dist, lim2))
                                *dst++ = HALF ? pack_key_positive(fmaxf(fmaf(dist, half_back, off), 0.0f), j)
                                              : pack_key(BF16 ? dist + off : dist, j);
                        }
                    }
                }
            }
            // Lists that a further tile could overflow are compacted by their own wave, right away.
            {
                u64 crowded = __ballot(cnt[wave * 32 + qn] > args.trigger) & 0xffffffffull;  // lanes l, l+32 share a query
                while (crowded) {
                    const int ql = wave * 32 + (__ffsll((long long)crowded) - 1);
                    crowded &= crowded - 1;
                    wave_select(list + (size_t)ql * cap, want, &cnt[ql], &thr[ql], sortbuf, hist_all[wave], lane,
                                args.select_slack);
                }
            }
            if constexpr (BF16 || HALF) {
                if constexpr (HALF) wait_for_loads();
                else if (next_ct >= 0) stash(buf ^ 1);
                __syncthreads();  // the next tile's first chunk is in LDS; all waves are done with this tile's last
                if (next_ct >= 0) {
                    buf ^= 1;
                    parity ^= 1;
                }
            } else {
                __syncthreads();  // all waves are done with the tile's last chunk
                if (next_ct >= 0) {
                    stash(0);
                    __syncthreads();
                }
            }
#pragma unroll
            for (int s4 = 0; s4 < kSlots; ++s4) bcur[s4] = bnext[s4];
        };

        // Phase 1: the query tile's neighbourhood; phase 2: the tiles the bitmap keeps.
        const int T = num_ctiles;
        const int h0 = max(qt - kHomeTiles * P, 0), h1 = min(qt + kHomeTiles * P, T - 1);  // >= kHomeTiles tiles of every part
        int word_idx = -1;
        unsigned int cur_word = 0u;
        auto next_tile = [&]() -> int {
            while (cur_word == 0u) {
                ++word_idx;
                if (word_idx >= args.bitmap_words) return -1;
                cur_word = bitmap[word_idx];
            }
            const int b = __ffs((int)cur_word) - 1;
            cur_word &= cur_word - 1u;
            return word_idx * 32 + b;
        };
        int cur = h0 + (part - h0 % P + P) % P;  // this part's first tile of the neighbourhood
        if (cur > h1) cur = -1;  // fewer tiles than parts: nothing for this part, its lists stay empty
        if constexpr (!HALF)
            if (cur >= 0) fetch(cur, 0);
        __syncthreads();  // the previous query tile's last reads of the LDS chunk
        buf = 0;
        if (cur >= 0) {
            if constexpr (HALF) fetch_half(cur, 0, 0);
            else stash(0);
            parity ^= 1;
        }
        wait_for_loads();
        __syncthreads();
        bool home = true;
        unsigned int swept = 0;
        while (cur >= 0) {
            ++swept;
            int nxt = home ? (cur + P <= h1 ? cur + P : -1) : next_tile();
            process(cur, nxt);
            if (nxt < 0 && home && (h0 > 0 || h1 < T - 1)) {
                home = false;
                for (int b = 0; b < 32; ++b) {
                    const int ql = wave * 32 + b;
                    if (q0 + ql < N)
                        wave_select(list + (size_t)ql * cap, want, &cnt[ql], &thr[ql], sortbuf, hist_all[wave], lane);
                }
                for (int w = tid; w < args.bitmap_words; w += 256) bitmap[w] = 0u;
                for (int d = tid; d < D; d += 256) qcenter[d] = args.centers_t[(size_t)d * T + qt];
                __syncthreads();
                if (tid < kMQ) {
                    // Largest squared distance any query of the tile would still accept (rounded up).
                    float v = -INFINITY;
                    if (q0 + tid < N) {
                        const u64 t = thr[tid];
                        v = t == ~0ull ? INFINITY : key_distance(t) + (BF16 || HALF ? 0.0f : args.norms[q0 + tid]);
                        v += 1e-5f * fabsf(v) + 1e-30f;
                    }
                    v = group_max<kWave>(v);
                    if (lane == 0) tmax_part[wave] = v;
                }
                __syncthreads();
                const float tmax = fmaxf(tmax_part[0], tmax_part[1]);
                const float ra = args.radius[qt];
                for (int t = tid; t < T; t += 256)
                    if ((t < h0 || t > h1) && t % P == part &&
                        tile_may_matter(qcenter, ra, args.centers_t, args.radius, D, T, t, tmax))
                        atomicOr(&bitmap[t >> 5], 1u << (t & 31));
                __syncthreads();
                nxt = next_tile();
                if (nxt >= 0) {
                    if constexpr (HALF) {
                        fetch_half(nxt, 0, buf);  // the barrier that ended the last tile freed the LDS chunks
                        wait_for_loads();
                    } else {
                        fetch(nxt, 0);
                        stash(buf);
                    }
                    parity ^= 1;
                    __syncthreads();
                }
                __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0), as in the kernel above
            }
            cur = nxt;
        }
        if (tid == 0) atomicAdd(args.tiles_swept, (unsigned long long)swept);
        // Final ordering and output, every wave for its own 32 queries.
        for (int b = 0; b < 32; ++b) {
            const int ql = wave * 32 + b;
            const int qq = q0 + ql;
            if (qq >= N) break;
            const int n = wave_select(list + (size_t)ql * cap, want, &cnt[ql], &thr[ql], sortbuf, hist_all[wave], lane);
            const size_t row = (size_t)qi * kMQ + ql;
            if (P == 1) {
                for (int e = lane; e < want; e += kWave)
                    cand[row * want + e] = e < n ? key_index(list[(size_t)ql * cap + e]) : -1;
                if (lane == 0) tau[row] = thr[ql] == ~0ull ? INFINITY : key_distance(thr[ql]);
            } else {
                u64 *dst = args.part_keys + (row * P + part) * want;
                for (int e = lane; e < want; e += kWave) dst[e] = e < n ? list[(size_t)ql * cap + e] : ~0ull;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        __syncthreads();  // before the next query tile re-initialises thr / cnt and the LDS chunk
    }
}

// ---------------------------------------------------------------------------
// Merge of the parts of the chunked sweep: the `want` best keys of a query's parts * want, exactly what
// a single list would have kept (every part kept its own `want` best), and their threshold.  One wave
// per query row, four rows per workgroup.  Dynamic LDS: 4 x parts * want keys.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void knn_merge_parts_kernel(u64 *__restrict__ part_keys, int parts, int want,
                                                              int n_rows, int *__restrict__ cand,
                                                              float *__restrict__ tau) {
    extern __shared__ u64 merge_buf[];
    __shared__ unsigned int hist_all[4][kWave];
    __shared__ u64 thr[4];
    __shared__ int cnt[4];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + wave;
    if (row >= n_rows) return;  // no workgroup barrier below
    const int total = parts * want;
    u64 *list = part_keys + (size_t)row * total;
    if (lane == 0) {
        thr[wave] = ~0ull;
        cnt[wave] = total;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // The filler keys sort last; a threshold with all distance bits set means "fewer than `want` candidates".
    wave_select(list, want, &cnt[wave], &thr[wave], merge_buf + (size_t)wave * total, hist_all[wave], lane);
    for (int e = lane; e < want; e += kWave) cand[(size_t)row * want + e] = key_index(list[e]);
    if (lane == 0) tau[row] = (thr[wave] >> 32) == 0xffffffffull ? INFINITY : key_distance(thr[wave]);
}

// ---------------------------------------------------------------------------
// Re-rank: canonical distances of a query's candidates, sort by (distance,
// index), verify, write.  One wave per query, four queries per workgroup.
// Dynamic LDS: 4 x sort_n keys.  rename (optional): the caller's number of every point, where the sweep ran on
// renumbered points; rows come out in the caller's numbering, fail_list in the sweep's.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void knn_rerank_kernel(const float *__restrict__ X,
                                                         const float *__restrict__ norms, int N, int D, int K,
                                                         int want, int sort_n, const int *__restrict__ cand,
                                                         const float *__restrict__ tau,
                                                         const float *__restrict__ max_norm,
                                                         int *__restrict__ out_idx, float *__restrict__ out_d,
                                                         int *__restrict__ fail_count, int *__restrict__ fail_list,
                                                         const int *__restrict__ qtile_list, int qtile_first,
                                                         int qtile_step, int n_slots, int lower_bounds,
                                                         const int *__restrict__ rename) {
    extern __shared__ u64 keys_all[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    // Query slot w belongs to query tile qtile_list[w / kMQ], or first + (w / kMQ) step without a list
    // (all queries: first 0, step 1).  cand holds `want` candidates per slot, tau one threshold.
    const int w = blockIdx.x * 4 + wave;
    const int wt = w < n_slots ? w / kMQ : 0;
    const int q = (qtile_list ? qtile_list[wt] : qtile_first + wt * qtile_step) * kMQ + (w % kMQ);
    u64 *keys = keys_all + (size_t)wave * sort_n;
    const bool live = w < n_slots && q < N;
    const float *xq = X + (size_t)(live ? q : 0) * D;
    for (int c = lane; c < sort_n; c += kWave) {
        u64 key = ~0ull;
        if (live && c < want) {
            const int j = cand[(size_t)w * want + c];
            if (j >= 0) {
                const float *xj = X + (size_t)j * D;
                float acc = 0.0f;
                if ((D & 3) == 0 && D >= 64 && (reinterpret_cast<uintptr_t>(X) & 15) == 0) {
                    // Long rows, 16-byte aligned: 128 bytes of the candidate's row per lane and step, so that a
                    // cache line is used whole by the load that fetches it (the lanes walk 64 different rows);
                    // the same fma chain.
                    const v4f *q4 = reinterpret_cast<const v4f *>(xq);
                    const v4f *j4 = reinterpret_cast<const v4f *>(xj);
                    const int n4 = D / 4;
                    int d4 = 0;
                    for (; d4 + 8 <= n4; d4 += 8) {
                        v4f b[8];
#pragma unroll
                        for (int u = 0; u < 8; ++u) b[u] = j4[d4 + u];
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            const v4f a = q4[d4 + u];
#pragma unroll
                            for (int k = 0; k < 4; ++k) {
                                const float df = a[k] - b[u][k];
                                acc = fmaf(df, df, acc);
                            }
                        }
                    }
                    for (; d4 < n4; ++d4) {
                        const v4f a = q4[d4], b = j4[d4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const float df = a[k] - b[k];
                            acc = fmaf(df, df, acc);
                        }
                    }
                } else if ((D & 1) == 0 && (reinterpret_cast<uintptr_t>(X) & 7) == 0) {
                    // rows are 8-byte aligned: two dimensions per load, the same fma chain
                    const float2 *q2 = reinterpret_cast<const float2 *>(xq);
                    const float2 *j2 = reinterpret_cast<const float2 *>(xj);
                    const int n2 = D / 2;
                    int d = 0;
                    // eight loads (64 bytes of the candidate's row) in flight per lane
                    for (; d + 8 <= n2; d += 8) {
                        float2 b[8];
#pragma unroll
                        for (int u = 0; u < 8; ++u) b[u] = j2[d + u];
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            const float2 a = q2[d + u];
                            const float d0 = a.x - b[u].x, d1 = a.y - b[u].y;
                            acc = fmaf(d0, d0, acc);
                            acc = fmaf(d1, d1, acc);
                        }
                    }
                    for (; d < n2; ++d) {
                        const float2 a = q2[d], b = j2[d];
                        const float d0 = a.x - b.x, d1 = a.y - b.y;
                        acc = fmaf(d0, d0, acc);
                        acc = fmaf(d1, d1, acc);
                    }
                } else {
                    for (int d = 0; d < D; ++d) {
                        const float df = xq[d] - xj[d];
                        acc = fmaf(df, df, acc);
                    }
                }
                key = pack_key(acc, rename ? rename[j] : j);
            }
        }
        keys[c] = key;
    }
    wave_sort(keys, sort_n, lane);
    if (!live) return;
    // Sweep on floats: every candidate outside the list has an approximate distance >= tau (without
    // |q|^2), so its canonical distance is >= tau + |q|^2 - g.  g bounds |approximate - canonical|: both are
    // sums of at most D + 3 rounded terms of magnitude <= (|q| + |c|)^2, and the canonical distance carries
    // a relative error of (D + 2) 2^-24 of itself; a factor of four covers the matrix unit's
    // accumulation order and the rounding of the stored norms.
    // Sweep on bf16 terms (lower_bounds): the sweep's keys are lower bounds of the distances, so every
    // candidate outside the list has a distance >= tau, and a canonical distance within (D + 2) 2^-24 of that.
    const float kth = key_distance(keys[K - 2]);
    const float t = tau[w];
    bool pass = isinf(t) && t > 0.0f;
    if (!pass) {
        const double eps = 5.9604644775390625e-08;  // 2^-24
        if (lower_bounds) {
            pass = (double)kth + (D + 4) * eps * ((double)kth + fabs((double)t)) < (double)t;
        } else {
            const double nq = norms[q], nmax = *max_norm;
            const double g = 4.0 * (D + 4) * eps * (nq + nmax + 2.0 * sqrt(nq * nmax)) + (D + 4) * eps * (double)kth;
            pass = (double)kth < (double)t + nq - g;
        }
    }
    if (pass) {
        const int row = rename ? rename[q] : q;
        for (int e = lane; e < K; e += kWave) {
            out_idx[(size_t)row * K + e] = e == 0 ? row : key_index(keys[e - 1]);
            out_d[(size_t)row * K + e] = e == 0 ? 0.0f : key_distance(keys[e - 1]);
        }
    } else if (lane == 0) {
        fail_list[atomicAdd(fail_count, 1)] = q;
    }
}

__global__ __launch_bounds__(256) void knn_self_only_kernel(int N, int *__restrict__ out_idx,
                                                            float *__restrict__ out_d) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) {
        out_idx[i] = i;
        out_d[i] = 0.0f;
    }
}

__global__ __launch_bounds__(256) void rename_list_kernel(const int *__restrict__ order, int count,
                                                          int *__restrict__ list) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) list[i] = order[list[i]];
}

// How far the points of a sampled tile (128 consecutive points) lie from the tile's mean, and how far a point of it
// from the nearest of the other tiles' (one per tile, at a place that no regular numbering lines up with).  Per tile
// out[0 .. D-1] the mean, out[D] the mean squared distance to it, out[D+1] the smallest squared distance.  One workgroup
// of 128 threads per sampled tile, at most 64 of them, `step` tiles apart.
__global__ __launch_bounds__(128) void sample_tiles_kernel(const float *__restrict__ X, int D, int step,
                                                           float *__restrict__ out) {
    __shared__ float part[128 / kWave], between[128];
    const int tile = blockIdx.x, tid = threadIdx.x;
    const float *x = X + (size_t)tile * step * kCT * D;
    float *dst = out + (size_t)tile * (D + 2);
    float within = 0.0f;
    for (int d = tid; d < D; d += 128) {  // (a lane per dimension: neighbouring lanes read neighbouring words)
        float sum = 0.0f;
        for (int p = 0; p < kCT; ++p) sum += x[(size_t)p * D + d];
        const float mean = sum * (1.0f / kCT);
        dst[d] = mean;
        for (int p = 0; p < kCT; ++p) {
            const float off = x[(size_t)p * D + d] - mean;
            within = fmaf(off, off, within);
        }
    }
    within = group_sum<kWave>(within);
    if ((tid & (kWave - 1)) == 0) part[tid / kWave] = within;
    auto member = [&](int t) { return ((size_t)t * step * kCT + ((unsigned int)t * 0x9E3779B1u >> 25)) * D; };
    // (two threads per other tile, half of the dimensions each)
    const int other = tid & (kWave - 1), d0 = tid < kWave ? 0 : D / 2, d1 = tid < kWave ? D / 2 : D;
    const bool counts = other < (int)gridDim.x && other != tile;
    const float *mine = X + member(tile), *theirs = X + member(counts ? other : tile);
    float dist = 0.0f;
#pragma unroll 8
    for (int d = d0; d < d1; ++d) {
        const float off = mine[d] - theirs[d];
        dist = fmaf(off, off, dist);
    }
    between[tid] = dist;
    __syncthreads();
    if (tid < kWave) {
        const float nearest = group_min<kWave>(counts ? between[tid] + between[tid + kWave] : INFINITY);
        if (tid == 0) {
            dst[D] = (part[0] + part[1]) * (1.0f / kCT);
            dst[D + 1] = nearest;
        }
    }
}

struct DeviceMem {
    void *p = nullptr;
    ~DeviceMem() { release(); }
    void release() {
        scratch_free(p);  // (waits for the kernels that use it)
        p = nullptr;
    }
    bool alloc(size_t bytes) {
        release();
        return scratch_malloc(&p, bytes) == hipSuccess;
    }
    // (of a form that the call can do without)
    bool alloc_optional(size_t bytes) {
        release();
        return malloc_optional(&p, bytes ? bytes : 1) == hipSuccess;
    }
    template <typename T>
    T *as() const {
        return static_cast<T *>(p);
    }
};

int next_pow2(int v) {
    int n = 1;
    while (n < v) n <<= 1;
    return n;
}

// lds: SweepGeometry::lds_with
template <int KSTEPS, Products PRODUCTS>
int launch_mfma_sweep(const SweepArgs &args, int grid, size_t lds, hipStream_t s) {
    void (*sweep)(const SweepArgs) = nullptr;
    if constexpr (PRODUCTS == Products::kHalf)
        sweep = knn_half_sweep_kernel<KSTEPS>;
    else
        sweep = knn_mfma_sweep_kernel<KSTEPS, PRODUCTS == Products::kBf16>;
    TSNE_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(sweep), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    sweep<<<grid, 256, lds, s>>>(args);
    TSNE_TRY(hipGetLastError());
    return 0;
}

// Steps of 16 dimensions, of the bf16 sweep (up to 125 dimensions + the three |c|^2 terms) or the one on halves.
template <Products P>
int dispatch_steps16(int steps, const SweepArgs &args, int grid, size_t lds, hipStream_t s) {
    switch (steps) {
        case 1: return launch_mfma_sweep<1, P>(args, grid, lds, s);
        case 2: return launch_mfma_sweep<2, P>(args, grid, lds, s);
        case 3: return launch_mfma_sweep<3, P>(args, grid, lds, s);
        case 4: return launch_mfma_sweep<4, P>(args, grid, lds, s);
        case 5: return launch_mfma_sweep<5, P>(args, grid, lds, s);
        case 6: return launch_mfma_sweep<6, P>(args, grid, lds, s);
        case 7: return launch_mfma_sweep<7, P>(args, grid, lds, s);
        case 8: return launch_mfma_sweep<8, P>(args, grid, lds, s);
        default:
            set_error("knn: no matrix-instruction sweep for %d steps of 16 dimensions", steps);
            return 1;
    }
}

// Instantiated step counts: every count up to 32 (62 dimensions), then multiples of 4.
int dispatch_mfma_sweep(int ksteps, const SweepArgs &args, int grid, size_t lds, hipStream_t s) {
#define TSNE_MFMA_CASE(KS) \
    case KS:               \
        return launch_mfma_sweep<KS, Products::kFloats>(args, grid, lds, s);
    switch (ksteps) {
        TSNE_MFMA_CASE(2) TSNE_MFMA_CASE(3) TSNE_MFMA_CASE(4) TSNE_MFMA_CASE(5) TSNE_MFMA_CASE(6)
        TSNE_MFMA_CASE(7) TSNE_MFMA_CASE(8) TSNE_MFMA_CASE(9) TSNE_MFMA_CASE(10) TSNE_MFMA_CASE(11)
        TSNE_MFMA_CASE(12) TSNE_MFMA_CASE(13) TSNE_MFMA_CASE(14) TSNE_MFMA_CASE(15) TSNE_MFMA_CASE(16)
        TSNE_MFMA_CASE(17) TSNE_MFMA_CASE(18) TSNE_MFMA_CASE(19) TSNE_MFMA_CASE(20) TSNE_MFMA_CASE(21)
        TSNE_MFMA_CASE(22) TSNE_MFMA_CASE(23) TSNE_MFMA_CASE(24) TSNE_MFMA_CASE(25) TSNE_MFMA_CASE(26)
        TSNE_MFMA_CASE(27) TSNE_MFMA_CASE(28) TSNE_MFMA_CASE(29) TSNE_MFMA_CASE(30) TSNE_MFMA_CASE(31)
        TSNE_MFMA_CASE(32) TSNE_MFMA_CASE(36) TSNE_MFMA_CASE(40) TSNE_MFMA_CASE(44) TSNE_MFMA_CASE(48)
        TSNE_MFMA_CASE(52) TSNE_MFMA_CASE(56) TSNE_MFMA_CASE(60) TSNE_MFMA_CASE(64)
        default:
            set_error("knn: no matrix-instruction sweep for %d steps", ksteps);
            return 1;
    }
#undef TSNE_MFMA_CASE
}

// Shape of the matrix-instruction sweep for N points of D dimensions.
struct SweepGeometry {
    int Dnorm;           // |x|^2 row: first even row after the real dimensions
    int ksteps;          // k-steps incl. the augmented pair
    bool chunked;        // more dimensions than one wave's registers hold
    bool half;           // one half per coordinate
    bool bf16, bf16_chunked;
    int n_chunks, steps16, num_tiles, bitmap_words;
    int slots;           // 16-byte slots per lane and block of the packed points
    size_t tile_float4;  // float4 per packed tile
    size_t tile_lds;

    // Two bf16 terms per coordinate are of the points relative to their tile's centre; three more dimensions carry a
    // per-point term, and 126 dimensions, the most the register-resident sweep takes, are multiplied as floats.
    SweepGeometry(int N, int D, Products products) {
        Dnorm = (D + 1) & ~1;
        ksteps = (Dnorm + 2) / 2;
        chunked = ksteps > kMfmaMaxSteps;
        half = products == Products::kHalf;
        bf16 = !chunked && products == Products::kBf16 && D + 3 <= 128;
        bf16_chunked = chunked && products == Products::kBf16;
        n_chunks = !chunked ? 0 : half ? div_up(D, 64) : bf16_chunked ? div_up(D + 3, 32) : div_up(ksteps, kChunkSteps);
        if (chunked) ksteps = n_chunks * (bf16_chunked ? kChunkSteps / 2 : kChunkSteps);  // (slots of 16 bytes per lane x 4)
        else if (ksteps > 32) ksteps = (ksteps + 3) & ~3;
        steps16 = half ? div_up(D, 16) : div_up(D + 3, 16);
        num_tiles = div_up(N, kCT);
        bitmap_words = div_up(num_tiles, 32);
        slots = half ? (chunked ? 4 * n_chunks : steps16) : bf16 ? 2 * steps16 : (ksteps + 3) / 4;
        tile_float4 = (size_t)kCT * slots * 2 + (bf16 ? 64 : 0);
        // (the chunked sweeps on halves and bf16 terms keep two chunks of half the size)
        tile_lds = chunked ? sizeof(float4) * kChunkFloat4 + sizeof(float) * D
                           : sizeof(float4) * (half ? 2 * (size_t)half_tile_float4(steps16) : tile_float4);
    }
    size_t lds_with(int cap) const {
        return tile_lds + (half && !chunked ? 0 : sizeof(u64) * 4 * cap) + sizeof(unsigned int) * bitmap_words;
    }
    // Room for the candidates kept, as many again and one more tile where the LDS sort buffers of that
    // size fit: a list that is nearly full right after a selection would be selected again after every tile.
    int list_cap(int want) const {
        if (half && !chunked) return kHalfCap;
        int cap = next_pow2(2 * want + kCT);
        if (cap > 4096 || lds_with(cap) > 150 * 1024) cap = next_pow2(want + kCT);
        return cap < 256 ? 256 : cap;
    }
    size_t sweep_lds(int want) const { return lds_with(list_cap(want)); }
    bool fits(int want) const {
        return (half && !chunked ? want <= kHalfWant : list_cap(want) <= 4096) && sweep_lds(want) <= 150 * 1024;
    }
};
// Chunked sweep: the table of centre distances takes a pass of N^2 D / 128 and saves one in the sweep, and its launches
// and memory (the square of the points: 80 MB at 50000) cost 0.2 ms.  Calls in a row without / with it, clustered and
// structureless points: 17000 x 127 0.96, 0.97; 30000 x 127 0.92, 0.95; 45000 x 127 0.94, 0.98; 24576 x 400 1.00, 1.03;
// 30000 x 400 1.00, 1.04; 45000 x 250 0.98, 1.03; 60000 x 784 1.03, 1.09.  Larger tables gain as much (150000 x 256 1.02,
// 1.12) but are memory that the driver clears between calls: with 200 to 313 MB (80000 and 100000 points) about one call
// in a hundred took 0.1 to 1.3 s longer, none without a table or with up to 153 MB.
inline bool centre_table_pays(int N, int D) { return (double)N * N * D >= 3e11; }
constexpr size_t kMaxCentreTable = (size_t)128 << 20;  // (64896 points)
constexpr int kMatrixPoints = 8192;  // fewer points: vector sweep
// K' candidates kept per query.
inline int candidates_kept(int N, int K) { return std::min(N - 1, (K - 1) + std::max(32, (K - 1) / 2)); }
// The re-rank takes 64 of them at a time, and as long for a few as for 64: up to eight beyond a multiple may be left out (87 to
// 92 and 130 to 134 neighbours).  Of many points more queries then fail and are searched again.  90 neighbours, on halves, ms, 133 /
// 128 kept: 100000 x 30 4.45 / 4.28, 200000 x 20 7.84 / 7.49, 300000 x 50 25.3 / 25.2, 1,000,000 x 50 in four clusters 71.1 /
// 73.3; 270000 to 1,000,000 points without structure, 90 and 132 neighbours, within 1 % of each other.
// Where they decide more than that the search keeps them all (see there): how long lists are and whether a sample verifies are
// questions of margins, and an answer that eight candidates turn round costs more than they do.
inline int candidates_trimmed(int N, int K) {
    const int want = candidates_kept(N, K), whole = want / kWave * kWave;
    return N <= 262144 && want < 256 && want - whole <= 8 && whole >= (K - 1) + 32 ? whole : want;
}

int valu_cap(int K) {
    int cap = 256;
    while (cap < K - 1 + kCT) cap <<= 1;
    return cap;
}

// Direct search: distances and their selection, by blocks of query rows.  Measured, ms, direct / sweep, points in an
// order with locality: 3000 x 64, 91 neighbours 0.13 / 3.9; 5000 x 50, 90: 0.21 / 4.9; 8000 x 126, 151: 0.68 / 4.8;
// 8192 x 30, 45: 0.35 / 0.93; 16384 x 50, 33: 1.5 / 1.4; 16384 x 125, 90: 2.4 / 3.0; 20000 x 32, 50: 1.6 / 1.9;
// 32000 x 8, 30: 2.8 / 2.7; 32000 x 50, 90: 4.3 / 2.7.  It forms every pair, where the matrix sweep skips tiles and
// multiplies on the matrix pipe: the line lies where the two are near each other.  Beyond 126 dimensions the sweep's
// time depends on how well its margin verifies, the direct form's does not: 14336 x 784, 33: clustered pixels 7.2 / 16,
// no structure 7.1 / 6.0; 16384 x 1024, 33: 11.6 / 44 and 11.4 / 7.5.  A sweep for few neighbours keeps few candidates,
// and the line lies lower: 12288 x 125, 2: 1.35 / 1.53; 16384 x 125, 2: 2.27 / 1.77; 16384 x 50, 10: 1.39 / 1.31.
constexpr int kDirectPoints = 16384, kDirectPointsFew = 12288, kFewNeighbors = 12;
inline bool direct_search_pays(int N, int K) { return N <= (K <= kFewNeighbors ? kDirectPointsFew : kDirectPoints); }
constexpr int kDirectNeighbors = 256;  // most K - 1 that select_row_kernel<8> takes
// Floats per block: 64 MiB, which the driver hands out again at once.  Calls that took 128 or 256 MiB (a third fewer
// launches, none of it measurable: 12288 x 50, 33 neighbours 0.89 ms with either) waited for it to clear what the call
// before had returned, at times: 11000 x 50, medians of 12 calls in a row 0.72 / 7.5 / 15.1 ms with 64 / 128 / 256 MiB.
constexpr size_t kDirectFloats = (size_t)1 << 24;

// (kNoRoom: nothing done, the sweeps need less memory)
int run_direct_search(const float *points, int N, int D, int K, int *indices, float *sq_dist, hipStream_t s) {
    const int pitch = div_up(N, 128) * 128;
    // Tiles of 64 points a side: of 128, with which a thread loads half as much per pair, half of them mirrored leave the chip
    // unevenly filled.  Whole searches, us, every tile formed with the better of the two / mirrored, 64 / 128 a side:
    // 3000 x 64, 91 neighbours 88 / 71 / 79; 4000 x 126, 90: 149 / 121 / 144; 6000 x 200, 45: 445 / 369 / 429;
    // 8000 x 126, 60: 532 / 492 / 518; 12000 x 40, 33: 731 / 697 / 737.
    constexpr int side = 64;
    const int block = std::min(div_up(N, 128) * 128, std::max(128, (int)(kDirectFloats / pitch) / 128 * 128));
    DeviceMem dist;
    if (!dist.alloc_optional(sizeof(float) * (size_t)std::min(block, N) * pitch)) {
        (void)hipGetLastError();
        return kNoRoom;
    }
    for (int row0 = 0; row0 < N; row0 += block) {
        const int rows = std::min(block, N - row0);
        const dim3 grid(div_up(N, side), div_up(rows, side));
        // Mirrored where the tiles are more than two per compute unit (22 a side), and of short rows from 2048 points on: every tile formed /
        // mirrored, 32 neighbours, us, 1025 x 20 40.8 / 41.9; 1408 x 4 41.3 / 42.7, x 100 51.8 / 52.5; 1536 x 20 44.6 / 45.0, x 50
        // 50.8 / 49.2, x 200 68.8 / 63.1; 1900 x 4 44.9 / 46.0, x 20 47.7 / 48.0; 2200 x 20 53.5 / 53.4, x 200 90.1 / 80.7.
        const auto distances = N <= 1408 || (N <= 2048 && D < 32) ? pair_distances_kernel<4, false> : pair_distances_kernel<4, true>;
        distances<<<grid, 256, 0, s>>>(points, N, points, N, D, row0, rows, pitch, dist.as<float>());
        TSNE_TRY(hipGetLastError());
        if (2 * (K - 1) <= 64 * 4)
            select_row_kernel<4><<<div_up(rows, 4), 256, 0, s>>>(dist.as<float>(), N, row0, rows, pitch, K, nullptr,
                                                                 indices, sq_dist);
        else
            select_row_kernel<8><<<div_up(rows, 4), 256, 0, s>>>(dist.as<float>(), N, row0, rows, pitch, K, nullptr,
                                                                 indices, sq_dist);
        TSNE_TRY(hipGetLastError());
    }
    TSNE_TRY(hipStreamSynchronize(s));
    return 0;
}

// A few queries (device list) of a moderate number of points: as above, their rows gathered first.  The vector sweep takes a
// transposed copy of the points and three more launches for them: searches of 20000 x 50 with two such queries 3.4 -> 2.3 ms,
// of 60000 x 784 with 100 of them 15.0 -> 12.2.
constexpr int kListedPoints = 131072;  // (a wave reads a row of distances twice)
int run_listed_search(const float *points, int N, int D, int K, const int *list, int count, int *indices, float *sq_dist,
                      hipStream_t s) {
    const int pitch = div_up(N, 64) * 64;
    if (N > kListedPoints || K - 1 > kDirectNeighbors || (size_t)count * pitch > kDirectFloats) return kNoRoom;
    DeviceMem dist, queries;
    if (!dist.alloc_optional(sizeof(float) * (size_t)count * pitch) ||
        !queries.alloc_optional(sizeof(float) * (size_t)count * D)) {
        (void)hipGetLastError();
        return kNoRoom;
    }
    if (launch_gather_rows(points, list, count, D, queries.as<float>(), s)) return 1;
    pair_distances_kernel<4, false><<<dim3(div_up(N, 64), div_up(count, 64)), 256, 0, s>>>(
        queries.as<float>(), count, points, N, D, 0, count, pitch, dist.as<float>());
    TSNE_TRY(hipGetLastError());
    const auto select = 2 * (K - 1) <= 64 * 4 ? select_row_kernel<4> : select_row_kernel<8>;
    select<<<div_up(count, 4), 256, 0, s>>>(dist.as<float>(), N, 0, count, pitch, K, list, indices, sq_dist);
    TSNE_TRY(hipGetLastError());
    TSNE_TRY(hipStreamSynchronize(s));
    return 0;
}

// VALU sweep over all points (qlist == nullptr) or over the nq listed queries.
int run_valu_sweep(const float *points, const float *Xt, int N, int Npad, int D, int K, const int *qlist, int nq,
                   int cus, int *indices, float *sq_dist, hipStream_t s) {
    const int cap = valu_cap(K);
    const int num_qtiles = div_up(nq, kQT);
    // A few listed queries: cut the candidates into ranges so that the whole chip works on them (as many
    // ranges as keep about four workgroups per CU busy, the merge's sort within 8192 keys, and at least one
    // candidate tile per range).
    int slices = 1;
    if (qlist != nullptr && K > 1)
        while (slices < 64 && num_qtiles * slices * 2 <= 4 * cus && slices * 2 * (K - 1) <= 8192 &&
               slices * 2 <= div_up(N, kCT))
            slices *= 2;
    const int grid = std::min(num_qtiles * slices, cus * 3);
    // Tile balls for skipping far-away candidate tiles: only when all queries are swept and the
    // neighbourhood that is always swept does not cover everything anyway.
    const int T = div_up(N, kCT);
    const bool prune = qlist == nullptr && T > 2 * kHomeTiles + 1;
    const int bitmap_words = prune ? div_up(T, 32) : 0;
    DeviceMem lists, centers, radius, slice_keys;
    if (!lists.alloc(sizeof(u64) * (size_t)grid * kQT * cap) ||
        (slices > 1 && !slice_keys.alloc(sizeof(u64) * (size_t)num_qtiles * kQT * slices * (K - 1))) ||
        (prune && (!centers.alloc(sizeof(float) * (size_t)D * T) || !radius.alloc(sizeof(float) * T)))) {
        set_error("knn: out of device memory for the candidate lists");
        return kNoRoom;
    }
    if (prune) {
        tile_balls_kernel<<<T, 128, sizeof(float) * D, s>>>(points, N, D, T, centers.as<float>(), radius.as<float>());
        TSNE_TRY(hipGetLastError());
    }
    const size_t lds = sizeof(u64) * cap + (prune ? sizeof(float) * D + sizeof(unsigned int) * bitmap_words : 0);
    knn_sweep_kernel<<<grid, 256, lds, s>>>(Xt, N, Npad, D, K, cap, lists.as<u64>(), num_qtiles, qlist, nq, indices,
                                            sq_dist, centers.as<float>(), radius.as<float>(), bitmap_words, slices,
                                            slice_keys.as<u64>());
    TSNE_TRY(hipGetLastError());
    if (slices > 1) {
        int sort_n = 256;
        while (sort_n < slices * (K - 1)) sort_n <<= 1;
        knn_merge_slices_kernel<<<nq, 256, sizeof(u64) * sort_n, s>>>(slice_keys.as<u64>(), slices, K, sort_n, qlist,
                                                                     indices, sq_dist);
        TSNE_TRY(hipGetLastError());
    }
    TSNE_TRY(hipStreamSynchronize(s));
    return 0;
}

// Fewer dimensions: a step of 16 dimensions is mostly padding, tiles are small beside their frame, and bf16 terms
// relative to the tile's own centre keep more.
constexpr int kHalfDims = 5;
// Halves relative to the frames lose more than two bf16 terms relative to the tiles where the points have structure that
// kFrames frames do not follow.  What counts is whether neighbours can be told from the rest, which a sample says (60000 x
// 20 in 300 clusters, 617 queries failed and were searched again, 4.5 ms, 2.5 on bf16 terms); and beyond kHalfLoss times the
// other sweep's bound that one is the better try.
// The chunked sweep widens its margin until a sample of query tiles verifies, and finds there what it has to, but three
// sweeps of a sample and a return to bf16 terms cost up to as much as the search: it is asked what twice the candidates
// would tell apart, or four times from kWideDims dimensions on, where halves save 40 % of a sweep and wider lists pay as well.
// ms, on bf16 terms / without this sample / with it, clusters 20 deviations apart in their order: 20000 x 150, 90
// neighbours, 18 clusters 8.3 / 15.7 / 8.3, 60 clusters 8.4 / 14.4 / 8.3; 60000 x 200, 45: 18 clusters 13.9 / 19.4 / 14.4, 60
// clusters 21.4 / 28.4 / 21.9, 300 clusters 10 apart 16.9 / 14.2 / 14.4; 60000 x 784, 45: 300 clusters 4 apart 37.9 / 24.5 /
// 24.7, pixel vectors 21.8 / 13.6 / 13.7.  With more dimensions more queries may be in doubt, which the vector sweep takes
// (60000 x 784, 17 clusters of which one has no frame, 105 / 46.4 / 46.8: bf16 terms cannot tell those neighbours apart
// either).
struct GapSample {
    int tiles, near_rank, far_rank;
    int most_in_doubt;  // one in so many may be
    float loss;
};
constexpr int kWideDims = 400;
inline GapSample gap_sample(int D, int T, int K, int want, bool chunked) {
    if (!chunked) return {std::min(T, 128), K - 1, want, 32, 4.0f * 4.0f / 4096.0f};
    const bool wide = D >= kWideDims;
    // (no more than a neighbourhood at either end of the numbering has; for more neighbours nothing is sampled)
    const int asked = std::min((wide ? 4 : 2) * want, kHomeTiles * kCT);
    // (the bound of half_bound.h at |q'| = |x'|: a coordinate's half is off by 0.4 of 2^-12 in the mean square)
    const float loss = 1.8f / 4096.0f + 15.0f * (float)(D + 8) * 5.9604644775390625e-08f;
    return {asked > want ? std::min(T, 48) : 0, std::max((K - 1) / kGapStride, 1), asked / kGapStride, wide ? 8 : 32, loss};
}
constexpr float kHalfLoss = 16.0f;

// What the sweeps on halves take beside the points: made in three steps.
struct HalfOperands {
    DeviceMem small, beta, point_len, tile_info;
    int dims = 0, tiles = 0;
    // `small`: kFrames keys, the scale, kFrames tile numbers, the frames' distances, the frames, the tiles' distance
    // to theirs and its number, and in the chunked form the sampled distances.
    u64 *best() const { return small.as<u64>(); }
    HalfScale *scale() const { return reinterpret_cast<HalfScale *>(best() + kFrames); }
    int *frame_tile() const { return reinterpret_cast<int *>(scale() + 1); }
    float *frame_d2() const { return reinterpret_cast<float *>(frame_tile() + kFrames); }
    float *frame_rows() const { return frame_d2() + kFrames * kFrames; }
    float *nearest() const { return frame_rows() + (size_t)dims * kFrames; }
    int *tile_frame() const { return reinterpret_cast<int *>(nearest() + tiles); }
    void release() {
        small.release();
        beta.release();
        point_len.release();
        tile_info.release();
    }
    // Frames of the tiles; *pays: whether the sweeps should multiply halves (false also where there is no room).
    int frames(const float *points, const float *centers_t, const float *radius, int N, int D, int T, int K, int want,
               bool chunked, bool *pays, hipStream_t s) {
        *pays = false;
        dims = D;
        tiles = T;
        const size_t keys = sizeof(u64) * kFrames + sizeof(HalfScale);
        const GapSample sample = gap_sample(D, T, K, want, chunked);
        const size_t given = chunked ? (size_t)sample.tiles * kGapGiven : 0;
        if (!small.alloc_optional(keys + sizeof(int) * (kFrames + kFrames * kFrames + (size_t)D * kFrames + 2 * (size_t)T + given))) {
            (void)hipGetLastError();
            return 0;
        }
        TSNE_TRY(hipMemsetAsync(small.p, 0, keys, s));
        for (int f = 0; f < kFrames; f = f == 0 ? kSeedFrames : f + 1) {
            frame_kernel<<<div_up(T, kFrameTiles), 1024, 0, s>>>(centers_t, radius, D, T, f, f == 0 ? kSeedFrames : f + 1, best(),
                                                        frame_tile(), nearest(), tile_frame(), scale());
            TSNE_TRY(hipGetLastError());
        }
        if (sample.tiles > 0) {
            const int step = T / sample.tiles;
            unsigned int *dist = given ? reinterpret_cast<unsigned int *>(tile_frame() + tiles) : nullptr;
            if (given) gap_distances_kernel<<<dim3(kGapSplit, sample.tiles), 1024, 0, s>>>(points, N, D, T, step, dist);
            gap_kernel<<<sample.tiles, 256, 0, s>>>(points, N, D, T, step, sample.near_rank, sample.far_rank, sample.loss, dist,
                                                    nearest(), radius, scale());
            TSNE_TRY(hipGetLastError());
        }
        HalfScale host;
        TSNE_TRY(hipMemcpyAsync(&host, scale(), sizeof(host), hipMemcpyDeviceToHost, s));
        TSNE_TRY(hipStreamSynchronize(s));
        // (a point that is not a number takes its tile with it, and which points those are the other sweep decides too)
        // ... and one scale serves all: beside a few tiles that reach 2^16 times as far as most, those lose bits.
        float reach;
        std::memcpy(&reach, &host.reach, sizeof(reach));
        // ... and points mostly within 1e-12 of their frames lose their squares to underflow, and the bound its grip.
        *pays = host.not_finite == 0 && host.unsure * sample.most_in_doubt <= sample.tiles && host.bound <= kHalfLoss * host.bound_bf16 &&
                std::log2(std::max(reach, 1e-30f)) <= host.log_reach / (float)T + 16.0f && host.log_reach >= -40.0f * (float)T;
        return 0;
    }
    bool room(int N, const SweepGeometry &g) {
        const size_t Npad = (size_t)g.num_tiles * kCT;
        return beta.alloc_optional(sizeof(float) * kFrames * Npad) && point_len.alloc_optional(sizeof(float2) * Npad) &&
               tile_info.alloc_optional(sizeof(float4) * g.num_tiles);
    }
    int pack(const float *points, const float *centers_t, int N, int D, const SweepGeometry &g, uint4 *Xh, hipStream_t s) {
        frame_rows_kernel<<<1, 1024, 0, s>>>(centers_t, D, g.num_tiles, frame_tile(), frame_rows(), frame_d2());
        TSNE_TRY(hipGetLastError());
        half_pack_kernel<<<g.num_tiles, 256, 0, s>>>(points, N, D, g.slots, frame_rows(), tile_frame(), scale(),
                                                     g.num_tiles * kCT, Xh, beta.as<float>(), point_len.as<float2>(),
                                                     tile_info.as<float4>());
        TSNE_TRY(hipGetLastError());
        return 0;
    }
};

}  // namespace

// mode: 0 = choose, 1 = VALU sweep only, 2 = matrix-instruction sweep on bf16 terms (on floats at 126 dimensions; error
// if the shape does not fit), 3 = as 2 on floats whatever the dimension count.
// stats (optional, 3 ints): [0] = 1 if the matrix-instruction sweep ran, [1] = queries redone by the VALU sweep,
// [2] = per mille of the (query tile, candidate tile) pairs the matrix sweep did not skip, each counted once: on halves those of
// the neighbourhood and of a sample are computed twice (SweepArgs::tiles_swept).
// renumbered != nullptr: `points` are a renumbered copy (point i is the caller's order[i]) and the result is in
// the caller's numbering.  Returns kNoRoom where memory is what it lacks.
struct KnnRenumbered {
    const int *order;            // device
    const float *caller_points;  // device
};
static int search(const float *points, int N, int D, int K, int *indices, float *sq_dist, hipStream_t s, int mode,
                  int *stats, const KnnProbes *probes, const KnnRenumbered *renumbered, bool halves = true) {
    if (stats) stats[0] = stats[1] = stats[2] = 0;
    if (N <= 0 || D <= 0 || K <= 0) {
        set_error("knn: num_points, num_dims and num_neighbors must be positive (got %d, %d, %d)", N, D, K);
        return 1;
    }
    if (K > N) {
        set_error("knn: num_neighbors (%d) exceeds num_points (%d)", K, N);
        return 1;
    }
    if (K == 1) {
        knn_self_only_kernel<<<div_up(N, 256), 256, 0, s>>>(N, indices, sq_dist);
        TSNE_LAUNCHED(s);
        TSNE_TRY(hipStreamSynchronize(s));
        return 0;
    }
    if (valu_cap(K) > 4096) {
        set_error("knn: num_neighbors = %d is not supported (limit %d)", K, 4096 - kCT + 1);
        return 1;
    }
    int device = 0, cus = 256;
    TSNE_TRY(hipGetDevice(&device));
    TSNE_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));

    // TSNE_KNN_PRODUCTS (measurements and tests of the search's own choice): bf16 never multiplies halves, half is an
    // error wherever the rows would not all come from a sweep on halves and its re-rank.
    const char *products = mode == 0 && !probes ? std::getenv("TSNE_KNN_PRODUCTS") : nullptr;
    const bool halves_only = products && std::strcmp(products, "half") == 0;
    if (products && std::strcmp(products, "bf16") == 0) halves = false;
    auto not_on_halves = [](const char *why) {
        set_error("knn: TSNE_KNN_PRODUCTS=half, but this search %s", why);
        return 1;
    };
    SweepGeometry geometry(N, D, mode == 3 ? Products::kFloats : Products::kBf16);
    if (mode == 3) mode = 2;
    const bool chunked = geometry.chunked;
    int want = candidates_kept(N, K);
    const int trimmed = candidates_trimmed(N, K);
    const bool mfma_fits = geometry.fits(want);
    bool use_mfma = mode == 2 || (mode == 0 && mfma_fits && N >= kMatrixPoints);
    if (mode == 2 && !mfma_fits) {
        set_error("knn: the matrix-instruction sweep does not fit %d dimensions / %d neighbours", D, K);
        return kShapeNotSupported;
    }
    if (probes && (!use_mfma || chunked)) {
        set_error("knn: the approximate search runs on the register-resident matrix sweep only (at most 126 "
                  "dimensions; got %d dimensions, %d neighbours)", D, K);
        return kShapeNotSupported;
    }

    const int Npad = div_up(N, kCT) * kCT;
    // Transposed points for the vector sweep (built only when that sweep runs).
    DeviceMem Xt;
    // Table of centre distances (chunked sweep), which goes where another buffer finds no room beside it.
    DeviceMem centre_dist;
    // (the points in the caller's numbering: equal distances are ordered by that)
    const float *caller_points = renumbered ? renumbered->caller_points : points;
    auto build_transposed = [&]() -> int {
        centre_dist.release();
        if (!Xt.alloc(sizeof(float) * (size_t)D * Npad)) {
            set_error("knn: out of device memory for the transposed points");
            return kNoRoom;
        }
        dim3 tgrid(div_up(Npad, 32), div_up(D, 32));
        transpose_points_kernel<<<tgrid, 256, 0, s>>>(caller_points, N, D, Npad, Xt.as<float>());
        TSNE_TRY(hipGetLastError());
        return 0;
    };
    if (halves_only && (!use_mfma || direct_search_pays(N, K))) return not_on_halves("is of few points or many neighbours");
    if (mode == 0 && direct_search_pays(N, K) && K - 1 <= kDirectNeighbors) {
        const int rc = run_direct_search(points, N, D, K, indices, sq_dist, s);
        if (rc != kNoRoom) return rc;
    }
    if (!use_mfma) {
        if (const int rc = build_transposed()) return rc;
        return run_valu_sweep(caller_points, Xt.as<float>(), N, Npad, D, K, nullptr, N, cus, indices, sq_dist, s);
    }

    const int num_qtiles = div_up(N, kMQ), num_tiles = geometry.num_tiles;
    DeviceMem Xp, Bp, norms, scal, fail_list, centers, radius;
    auto no_room = [](const char *what) {
        set_error("knn: out of device memory for the %s", what);
        return kNoRoom;
    };
    if (!scal.alloc(4 * sizeof(int)) || !fail_list.alloc(sizeof(int) * N) ||
        !centers.alloc(sizeof(float) * (size_t)D * num_tiles) || !radius.alloc(sizeof(float) * num_tiles))
        return no_room("candidate buffers");
    TSNE_TRY(hipMemsetAsync(scal.p, 0, 4 * sizeof(int), s));  // [0] max |x|^2 (float bits), [1] fail count, [2..3] tiles swept (64-bit)
    tile_balls_kernel<<<num_tiles, 128, sizeof(float) * D, s>>>(points, N, D, num_tiles, centers.as<float>(),
                                                               radius.as<float>());
    TSNE_TRY(hipGetLastError());
    HalfOperands operands;
    if (mode == 0 && halves && !probes && D >= kHalfDims) {
        const SweepGeometry on_halves(N, D, Products::kHalf);
        bool pays = false;
        if (on_halves.fits(want))
            if (const int rc = operands.frames(points, centers.as<float>(), radius.as<float>(), N, D, num_tiles, K,
                                               chunked ? want : trimmed, chunked, &pays, s))
                return rc;
        if (pays && operands.room(N, on_halves) && Xp.alloc_optional(sizeof(float4) * on_halves.tile_float4 * num_tiles)) {
            geometry = on_halves;
            if (operands.pack(points, centers.as<float>(), N, D, geometry, Xp.as<uint4>(), s)) return 1;
        } else {
            operands.release();
            (void)hipGetLastError();  // (of an allocation that did not fit)
        }
    }
    const bool half = geometry.half, bf16 = geometry.bf16, bf16_chunked = geometry.bf16_chunked;
    // On bf16 terms and on floats the candidates kept set the lists' length, and trimmed from 198 to 192 (130 to 134 neighbours) lists
    // are half as long and selected from twice as often: only where another workgroup then fits on a compute unit.  132 neighbours, all /
    // trimmed, ms: where none does 20000 x 20 2.21 / 2.42, in 20 clusters 1.43 / 1.56, 120000 x 125 42.5 / 44.6 and 20.7 / 21.2, on
    // floats 60000 x 126 15.7 / 16.2; where one does 60000 x 100 11.2 / 7.6, 5.2 / 4.7.  (200000 x 30 37.1 / 35.2, 11.0 / 10.9: points
    // without structure, which would gain there, are searched on halves.)
    if (!chunked && trimmed < want) {
        const int most = bf16 ? bf16_sweep_occupancy(geometry.steps16) : float_sweep_occupancy(geometry.ksteps);
        const auto workgroups = [&](int keep) { return std::min(most, (int)(kUnitLds / (geometry.sweep_lds(keep) + kSweepLds))); };
        if (geometry.list_cap(trimmed) == geometry.list_cap(want) || workgroups(trimmed) > workgroups(want)) want = trimmed;
    }
    if (halves_only && !half) return not_on_halves("does not choose them");
    const int Dnorm = geometry.Dnorm, ksteps = geometry.ksteps, n_chunks = geometry.n_chunks;
    const int steps16 = geometry.steps16, bitmap_words = geometry.bitmap_words;
    const int S4 = geometry.slots;
    if (!half) {
        if (!Xp.alloc(sizeof(float4) * geometry.tile_float4 * num_tiles) || !norms.alloc(sizeof(float) * Npad) ||
            (chunked && !Bp.alloc(sizeof(float4) * (size_t)Npad * S4 * 2)))
            return no_room("candidate buffers");
        norms_kernel<<<div_up(Npad, 256), 256, 0, s>>>(points, N, D, Npad, norms.as<float>(), scal.as<float>());
        TSNE_TRY(hipGetLastError());
    }
    if (!half && !bf16 && !bf16_chunked) {
        pack_points_kernel<<<div_up((int64_t)Npad * S4 * 2, 256), 256, 0, s>>>(points, norms.as<float>(), N, D, Dnorm,
                                                                              S4, Npad, Xp.as<float4>(), false);
        TSNE_TRY(hipGetLastError());
        if (chunked) {
            pack_points_kernel<<<div_up((int64_t)Npad * S4 * 2, 256), 256, 0, s>>>(
                points, norms.as<float>(), N, D, Dnorm, S4, Npad, Bp.as<float4>(), true);
            TSNE_TRY(hipGetLastError());
        }
    }
    if (bf16) {
        pack_points_bf16_kernel<<<div_up((int64_t)Npad * steps16 * 4, 256), 256, 0, s>>>(
            points, centers.as<float>(), N, D, steps16, num_tiles, Npad, Xp.as<uint4>());
        TSNE_TRY(hipGetLastError());
        pack_tile_centres_kernel<<<num_tiles, 64, 0, s>>>(centers.as<float>(), radius.as<float>(), D, steps16,
                                                         num_tiles, Xp.as<float4>());
        TSNE_TRY(hipGetLastError());
    }
    DeviceMem centres_p, tile_coef, centre_rows;
    if (bf16_chunked) {
        if (!centres_p.alloc(sizeof(float) * 32 * (size_t)n_chunks * num_tiles) ||
            !tile_coef.alloc(sizeof(float) * 2 * (size_t)num_tiles)) {
            set_error("knn: out of device memory for the tile centres");
            return kNoRoom;
        }
        const int64_t pieces = (int64_t)Npad * n_chunks * 8;
        pack_points_bf16_chunked_kernel<<<div_up(pieces, 256), 256, 0, s>>>(points, centers.as<float>(), N, D, n_chunks,
                                                                           num_tiles, Npad, Xp.as<uint4>(), false);
        TSNE_TRY(hipGetLastError());
        pack_points_bf16_chunked_kernel<<<div_up(pieces, 256), 256, 0, s>>>(points, centers.as<float>(), N, D, n_chunks,
                                                                           num_tiles, Npad, Bp.as<uint4>(), true);
        TSNE_TRY(hipGetLastError());
        pack_chunked_centres_kernel<<<num_tiles, 64, 0, s>>>(centers.as<float>(), radius.as<float>(), D, n_chunks,
                                                            num_tiles, centres_p.as<float>(), tile_coef.as<float>());
        TSNE_TRY(hipGetLastError());
        const size_t table_bytes = sizeof(float) * (size_t)num_tiles * Npad;
        if (centre_table_pays(N, D) && table_bytes <= kMaxCentreTable && centre_rows.alloc_optional(sizeof(float) * (size_t)num_tiles * D) &&
            centre_dist.alloc_optional(table_bytes)) {
            transpose_points_kernel<<<dim3(div_up(D, 32), div_up(num_tiles, 32)), 256, 0, s>>>(
                centers.as<float>(), D, num_tiles, D, centre_rows.as<float>());
            TSNE_TRY(hipGetLastError());
            pair_distances_kernel<8, false><<<dim3(div_up(N, 128), div_up(num_tiles, 128)), 256, 0, s>>>(
                centre_rows.as<float>(), num_tiles, points, N, D, 0, num_tiles, Npad, centre_dist.as<float>());
            TSNE_TRY(hipGetLastError());
        } else {
            (void)hipGetLastError();  // (of an allocation that did not fit: the sweep then forms them itself)
        }
    }

    // Sweep + re-rank of `count` query tiles: those of tile_list (device), or first, first + step, ... without a
    // list.  Keeps `keep` candidates per query and part.  failed = queries of those tiles whose verification
    // failed (listed in fail_list), swept = tile pairs not skipped.
    auto sweep_and_rerank = [&](int keep, const int *tile_list, int first, int step, int count, int &failed,
                                unsigned long long &swept) -> int {
        const int cap = geometry.list_cap(keep);
        // One workgroup sweeps a query tile against all its candidate tiles, which takes long with hundreds
        // of dimensions, and the tiles differ in how many candidate tiles they can skip: unless there are
        // several query tiles per workgroup slot to even that out, the chunked kernel splits every tile's
        // candidates over up to 8 workgroups.
        const int slots = cus * (chunked ? 2
                                 : half  ? half_sweep_occupancy(steps16)
                                 : bf16  ? bf16_sweep_occupancy(steps16)
                                         : (ksteps <= 28 ? 3 : 2));
        int parts = 1;
        if (chunked)
            while (parts < 8 && count * parts < 3 * slots && parts * 2 * keep <= 2048 && parts * 2 <= num_tiles)
                parts *= 2;
        // On halves below that the last round of the workgroups counts: what does not fill one is swept by several
        // workgroups per tile, in a launch of its own.
        const int whole = half && !chunked ? count / slots * slots : count, rest = count - whole;
        // Every part sweeps a neighbourhood and keeps lists of its own, so parts only pay where they run beside each
        // other on a chip that is half empty.  Whole searches, ms, in 1 / 2 / 4 / 8 parts: 157 tiles on 768 slots 1.58 /
        // 1.33 / 1.43 / 1.77, 313 2.31 / 1.99 / 2.26 / 3.04, 424 2.68 / 2.55 / 3.06 / 3.81, 469 without structure 3.79 / 4.97 /
        // 5.69 / 7.53; what 768 leave of 938 6.79 / 6.64 / 6.69 / 7.43, of 1172 6.81 / 6.15 / 6.33 / 7.18.
        int rest_parts = 1;
        if (rest > 0)
            while (rest_parts < (whole > 0 ? 16 : 2) && rest * rest_parts * 2 <= slots + slots / 16 &&
                   rest_parts * 2 * keep <= 2048 && rest_parts * 4 * (2 * kHomeTiles + 1) <= num_tiles)
                rest_parts *= 2;
        // (chunked: whole rounds of the XCDs, some of which may find nothing to do at the end)
        const int grid = chunked ? std::min(div_up(count, kSweepXcds) * kSweepXcds * parts, std::max(slots / (kSweepXcds * parts), 1) * (kSweepXcds * parts))
                                 : std::min(std::max(whole * parts, rest * rest_parts), slots);
        const size_t n_slots = (size_t)(tile_list || step != 1 ? count * kMQ : N);
        const size_t merged_rows = parts > 1 ? n_slots : rest_parts > 1 ? n_slots - (size_t)whole * kMQ : 0;
        DeviceMem lists, cand, tau, part_keys;
        // (on halves the lists are longer than on bf16 terms, up to three times, and the search goes on without them)
        auto alloc_lists = [&]() -> bool {
            const auto get = [&](DeviceMem &m, size_t bytes) { return half ? m.alloc_optional(bytes) : m.alloc(bytes); };
            return get(lists, sizeof(u64) * (size_t)grid * kMQ * cap) && get(cand, sizeof(int) * n_slots * keep) &&
                   get(tau, sizeof(float) * n_slots) &&
                   (merged_rows == 0 || get(part_keys, sizeof(u64) * merged_rows * std::max(parts, rest_parts) * keep));
        };
        bool room = alloc_lists();
        if (!room && centre_dist.p) {
            centre_dist.release();
            (void)hipGetLastError();
            room = alloc_lists();
        }
        if (!room) {
            (void)hipGetLastError();
            return no_room("candidate lists");
        }
        TSNE_TRY(hipMemsetAsync(scal.as<int>() + 1, 0, 3 * sizeof(int), s));
        SweepArgs args;
        args.Xp = Xp.as<float4>();
        args.X = points;
        args.centres_p = centres_p.as<float>();
        args.tile_coef = tile_coef.as<float>();
        args.centre_dist = centre_dist.as<float>();
        args.centre_pitch = Npad;
        args.N = N;
        args.D = D;
        args.Dnorm = Dnorm;
        args.want = keep;
        args.cap = cap;
        args.lists = lists.as<u64>();
        args.num_qtiles = count;
        args.cand = cand.as<int>();
        args.tau = tau.as<float>();
        args.norms = norms.as<float>();
        args.centers_t = centers.as<float>();
        args.radius = radius.as<float>();
        args.bitmap_words = bitmap_words;
        args.trigger = cap - kCT;  // as late as possible: a later selection costs the same and sees more candidates
        args.select_slack = (cap - kCT - keep) / 4;
        args.tiles_swept = reinterpret_cast<unsigned long long *>(scal.as<int>() + 2);
        args.Bp = half ? Xp.as<float4>() : Bp.as<float4>();
        args.n_chunks = n_chunks;
        args.qtile_list = tile_list;
        args.qtile_first = first;
        args.qtile_step = step;
        args.parts = parts;
        args.part_keys = part_keys.as<u64>();
        args.probe_tile_lists = probes ? probes->tile_lists : nullptr;
        args.probe_list_words = probes ? probes->list_words : 0;
        args.probe_nlist = probes ? probes->nlist : 0;
        args.probe_list_tiles = probes ? probes->list_tiles : nullptr;
        args.beta = operands.beta.as<float>();
        args.beta_pitch = Npad;
        args.point_len = operands.point_len.as<float2>();
        args.tile_info = operands.tile_info.as<float4>();
        args.frame_d2 = operands.frame_d2();
        args.half_scale = operands.scale();
        for (int k = 0; k < kRankRounds; ++k) {
            const double share = (double)(K - 1 + 16 + (K - 1) / 8) / (double)(256 >> (2 * k));
            args.ranks[k] = (int)std::ceil(share + 5.5 * std::sqrt(share) + 5.0);
        }
        const size_t lds = geometry.lds_with(cap);
        if (chunked) {
            const auto sweep = half               ? knn_mfma_chunked_sweep_kernel<Products::kHalf, false>
                               : !bf16_chunked    ? knn_mfma_chunked_sweep_kernel<Products::kFloats, false>
                               : args.centre_dist ? knn_mfma_chunked_sweep_kernel<Products::kBf16, true>
                                                  : knn_mfma_chunked_sweep_kernel<Products::kBf16, false>;
            TSNE_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(sweep),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            sweep<<<grid, 256, lds, s>>>(args);
            TSNE_TRY(hipGetLastError());
        } else if (half) {
            if (whole > 0) {
                args.num_qtiles = whole;
                if (dispatch_steps16<Products::kHalf>(steps16, args, std::min(whole, slots), lds, s)) return 1;
            }
            if (rest > 0) {
                args.num_qtiles = rest;
                args.qtile_first = first + whole * step;
                args.parts = rest_parts;
                if (dispatch_steps16<Products::kHalf>(steps16, args, std::min(rest * rest_parts, slots), lds, s)) return 1;
            }
        } else if (bf16 ? dispatch_steps16<Products::kBf16>(steps16, args, grid, lds, s)
                        : dispatch_mfma_sweep(ksteps, args, grid, lds, s)) {
            return 1;
        }
        if (merged_rows > 0) {
            // rows of a partial last tile are merged too: the sweep left them unwritten, the re-rank skips them
            const int merged = std::max(parts, rest_parts);
            const size_t lds = sizeof(u64) * 4 * merged * keep, done = n_slots - merged_rows;
            TSNE_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(knn_merge_parts_kernel),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            knn_merge_parts_kernel<<<div_up((int)merged_rows, 4), 256, lds, s>>>(
                part_keys.as<u64>(), merged, keep, (int)merged_rows, cand.as<int>() + done * keep, tau.as<float>() + done);
            TSNE_TRY(hipGetLastError());
        }
        const int sort_n = next_pow2(keep) < 64 ? 64 : next_pow2(keep);
        TSNE_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(knn_rerank_kernel),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)(sizeof(u64) * 4 * sort_n)));
        knn_rerank_kernel<<<div_up((int)n_slots, 4), 256, sizeof(u64) * 4 * sort_n, s>>>(
            points, norms.as<float>(), N, D, K, keep, sort_n, cand.as<int>(), tau.as<float>(), scal.as<float>(),
            indices, sq_dist, scal.as<int>() + 1, fail_list.as<int>(), tile_list, first, step, (int)n_slots,
            half || bf16 || bf16_chunked ? 1 : 0, renumbered ? renumbered->order : nullptr);
        TSNE_TRY(hipGetLastError());
        int host_scal[4] = {0, 0, 0, 0};
        TSNE_TRY(hipMemcpyAsync(host_scal, scal.p, sizeof(host_scal), hipMemcpyDeviceToHost, s));
        TSNE_TRY(hipStreamSynchronize(s));
        failed = host_scal[1];
        std::memcpy(&swept, host_scal + 2, sizeof(swept));
        return 0;
    };

    int failed = 0;
    unsigned long long swept = 0;
    // Points that the halves cannot tell apart, or no room for their lists: everything once more on two bf16 terms.
    auto without_halves = [&]() -> int {
        if (halves_only) return not_on_halves("returns from them");
        for (DeviceMem *m : {&Xp, &centers, &radius, &scal, &fail_list}) m->release();
        operands.release();
        return search(points, N, D, K, indices, sq_dist, s, mode, stats, probes, renumbered, false);
    };
    // The verification needs the distance gap between neighbour K and candidate K' to exceed the rounding
    // bound of the approximate distances, which grows with the dimension count and with the points'
    // distance from the origin.  With many dimensions the neighbour distances of a query lie close
    // together, so the chunked sweep first tries its margin on a sample of query tiles and doubles K'
    // while more than a tenth of the sample fails; data that no margin verifies goes to the vector sweep.
    if (chunked && num_qtiles >= 64) {
        const int sample_tiles = 16, step = num_qtiles / sample_tiles;
        bool verified = false;
        const int attempts = half && D < kWideDims ? 2 : 3;  // (see GapSample)
        for (int attempt = 0; attempt < attempts && !verified; ++attempt) {
            if (const int rc = sweep_and_rerank(want, nullptr, step / 2, step, sample_tiles, failed, swept))
                return rc == kNoRoom && half ? without_halves() : rc;
            if (failed * 10 <= sample_tiles * kMQ) {
                verified = true;
                // Sampled with all, and trimmed for the search itself where few queries of the sample fail (trimmed, up to 1.7 times as
                // many do, which stays below the tenth).  Points in 20 clusters, all throughout / trimmed throughout, ms: where that
                // doubled the margin once more, 90 neighbours, 30000 x 300 7.7 / 11.4, 50000 x 784 24.8 / 29.8, 30000 x 1000 19.1 /
                // 28.0; with 134 neighbours 50000 x 784 (6.6 % of the queries fail) 26.8 / 36.1; with 132 40000 x 200 (3.7 %) 12.7 /
                // 10.2.  Without structure 50000 x 1024 17.3 / 16.6, 30000 x 300 with 132 8.3 / 7.7.
                if (attempt == 0 && failed * 20 <= sample_tiles * kMQ) want = trimmed;
            } else {
                const int wider = std::min(N - 1, 2 * want);
                if (wider == want || !geometry.fits(wider)) break;
                want = wider;
            }
        }
        if (!verified && half) return without_halves();
        if (!verified && mode == 0) {
            if (const int rc = build_transposed()) return rc;
            return run_valu_sweep(caller_points, Xt.as<float>(), N, Npad, D, K, nullptr, N, cus, indices, sq_dist, s);
        }
    }
    if (const int rc = sweep_and_rerank(want, nullptr, 0, 1, num_qtiles, failed, swept))
        return rc == kNoRoom && half ? without_halves() : rc;
    if (half && !chunked && failed > N / 64) return without_halves();
    if (stats) {
        stats[0] = 1;
        stats[1] = failed;
        stats[2] = (int)((1000.0 * (double)swept) / ((double)num_tiles * (double)num_tiles) + 0.5);
    }
    // Few failures, or failures scattered thinly over the query tiles, go straight to the vector sweep, which
    // spreads a list of queries over the chip by candidate range.  Where a quarter or more of the queries of the
    // tiles concerned failed, the chunked sweep takes those tiles once more with twice the margin (a vector sweep
    // of that many queries over all points in hundreds of dimensions takes longer than the matrix sweep of their
    // tiles); what fails again, and every failure of the register-resident sweep, goes to the vector sweep.
    if (failed > 4 * kQT && chunked && failed * 10 <= N) {
        const int wider = std::min(N - 1, 2 * want);
        if (wider != want && geometry.fits(wider)) {
            std::vector<int> queries(failed), tiles;
            TSNE_TRY(hipMemcpy(queries.data(), fail_list.p, sizeof(int) * (size_t)failed, hipMemcpyDeviceToHost));
            for (int q : queries) tiles.push_back(q / kMQ);
            std::sort(tiles.begin(), tiles.end());
            tiles.erase(std::unique(tiles.begin(), tiles.end()), tiles.end());
            if ((size_t)failed * 4 >= tiles.size() * kMQ) {
                DeviceMem tile_list;
                if (!tile_list.alloc(sizeof(int) * tiles.size())) {
                    set_error("knn: out of device memory for the retry list");
                    return kNoRoom;
                }
                TSNE_TRY(hipMemcpy(tile_list.p, tiles.data(), sizeof(int) * tiles.size(), hipMemcpyHostToDevice));
                unsigned long long swept_again = 0;
                if (const int rc =
                        sweep_and_rerank(wider, tile_list.as<int>(), 0, 1, (int)tiles.size(), failed, swept_again))
                    return rc == kNoRoom && half ? without_halves() : rc;
            }
        }
    }
    if (failed > 0) {
        Xp.release();  // (room for what follows)
        Bp.release();
        operands.release();
        if (renumbered) {
            rename_list_kernel<<<div_up(failed, 256), 256, 0, s>>>(renumbered->order, failed, fail_list.as<int>());
            TSNE_TRY(hipGetLastError());
        }
        const int rc_listed = run_listed_search(caller_points, N, D, K, fail_list.as<int>(), failed, indices, sq_dist, s);
        if (rc_listed != kNoRoom) return rc_listed;
        if (const int rc = build_transposed()) return rc;
        return run_valu_sweep(caller_points, Xt.as<float>(), N, Npad, D, K, fail_list.as<int>(), failed, cus, indices, sq_dist, s);
    }
    return 0;
}

int run_knn_mode(const float *points, int N, int D, int K, int *indices, float *sq_dist, hipStream_t s, int mode,
                 int *stats, const KnnProbes *probes) {
    const int rc = search(points, N, D, K, indices, sq_dist, s, mode, stats, probes, nullptr);
    return rc == kNoRoom ? 1 : rc;
}

int run_knn(const float *points, int N, int D, int K, int *indices, float *sq_dist, hipStream_t s) {
    return run_knn_mode(points, N, D, K, indices, sq_dist, s, 0, nullptr);
}

// Whether the points come in no order and an order would let the sweep skip tiles.
// No order: consecutive points are no closer to each other than any points are, by the mean squared distance of a
// sampled tile's points to the tile's mean against that of all sampled points to theirs.
// An order pays where points have others much closer to them than points are on average, which a sample shows too:
// `near`, the squared distance to the nearest of 63 others over the spread, is 0.02 for well separated clusters, 0.1 to
// 0.4 in few dimensions, 1 and more for one cloud in many, where no tile can be skipped whatever the order.  Time as
// they come / renumbered, 33 neighbours, 2 to 120 dimensions, by `near` (the ordering costs 0.3 ms and the larger
// copies, so that small searches need more of it):
//   20000 points  < 0.2 0.94-1.25   0.2-0.5 0.94-1.21   > 0.5 0.78-1.17
//   30000         < 0.2 1.04-1.38   0.2-0.5 0.99-1.21   > 0.5 0.84-1.22
//   60000         < 0.2 1.18-1.63   0.2-0.5 1.08-1.34   > 0.5 0.93-1.25
//   100000        < 0.2 1.27-4.08   0.2-0.5 1.23-1.76   0.5-1.3 0.99-1.68   > 1.3 0.93-0.98
//   500000                          0.2-0.5 1.19-1.57   0.5-1.3 1.05-1.50
// (clustered pixels below 28672 points: 127 and 250 dimensions 0.87-0.95 for 15 neighbours, 1.0-1.5 for 90; 400 to 1024
// dimensions 1.1-3.6).
static int renumbering_pays(const float *points, int N, int D, bool *pays, hipStream_t s) {
    const int tiles = N / kCT, sampled = std::min(tiles, 64);  // (whole tiles only)
    DeviceMem out;
    *pays = false;
    if (sampled < 2) return 0;
    if (!out.alloc_optional(sizeof(float) * (size_t)sampled * (D + 2))) {
        set_error("knn: out of device memory");
        return kNoRoom;
    }
    sample_tiles_kernel<<<sampled, 128, 0, s>>>(points, D, tiles / sampled, out.as<float>());
    TSNE_TRY(hipGetLastError());
    std::vector<float> host((size_t)sampled * (D + 2));
    TSNE_TRY(hipMemcpyAsync(host.data(), out.p, sizeof(float) * host.size(), hipMemcpyDeviceToHost, s));
    TSNE_TRY(hipStreamSynchronize(s));
    double within = 0.0, between = 0.0, nearest = 0.0;
    for (int t = 0; t < sampled; ++t) {
        within += host[(size_t)t * (D + 2) + D];
        nearest += host[(size_t)t * (D + 2) + D + 1];
    }
    for (int d = 0; d < D; ++d) {
        double mean = 0.0, square = 0.0;
        for (int t = 0; t < sampled; ++t) mean += host[(size_t)t * (D + 2) + d];
        mean /= sampled;
        for (int t = 0; t < sampled; ++t) {
            const double off = host[(size_t)t * (D + 2) + d] - mean;
            square += off * off;
        }
        between += square;
    }
    // In a numbering without locality the means of 128 points lie within 1/128 of the points' own spread.
    const double near = N < 28672 ? 0.2 : N < 90112 ? 0.5 : 1.3;
    *pays = between < 0.1 * within && nearest < near * within;
    return 0;
}

// run_knn_any_order on a renumbered copy of the points, unless they are searched as they come (*searched false).
static int search_renumbered(const float *points, int N, int D, int K, int *indices, float *sq_dist, hipStream_t s,
                             int *stats, bool *searched) {
    std::vector<int> order_host;
    bool all_near = true;
    if (const int rc = locality_order(points, N, D, order_host, s, true, &all_near)) return rc;
    // The tile of a point that is not made of numbers has no centre, and the sweep loses the other points of that tile:
    // the caller's numbering decides which those are.
    if (!all_near) return 0;
    DeviceMem order, sorted;
    if (!order.alloc_optional(sizeof(int) * (size_t)N) || !sorted.alloc_optional(sizeof(float) * (size_t)N * D))
        return kNoRoom;
    TSNE_TRY(hipMemcpyAsync(order.p, order_host.data(), sizeof(int) * (size_t)N, hipMemcpyHostToDevice, s));
    if (launch_gather_rows(points, order.as<int>(), N, D, sorted.as<float>(), s)) return 1;
    TSNE_TRY(hipStreamSynchronize(s));
    const KnnRenumbered renumbered = {order.as<int>(), points};
    *searched = true;
    return search(sorted.as<float>(), N, D, K, indices, sq_dist, s, 0, stats, nullptr, &renumbered);
}

// The matrix sweep skips candidate tiles whose ball lies out of reach, which needs close points to have close
// numbers.  Points that come in no such order are searched in the locality order and the rows written in the
// caller's: the same rows, because distances do not depend on the numbering and the re-rank orders equal ones by
// the caller's.  (199999 x 30 in four clusters that come in turn, 33 neighbours: 27.2 -> 12.3 ms; on points
// that already are in order the look at the numbering costs 0.05 ms.)  Only where that sweep will run, and where
// there is room for a second copy of the points and the search beside it.
int run_knn_any_order(const float *points, int N, int D, int K, int *indices, float *sq_dist, hipStream_t s,
                      int *stats) {
    if (K > 1 && D > 0 && K <= N && N > kDirectPoints && locality_pivot_count(N) > 0 &&
        SweepGeometry(N, D, Products::kBf16).fits(candidates_kept(N, K))) {
        bool pays = false, searched = false;
        int rc = 0;
        try {
            rc = renumbering_pays(points, N, D, &pays, s);
            if (!rc && pays) {
                rc = search_renumbered(points, N, D, K, indices, sq_dist, s, stats, &searched);
                if (!rc && searched) return 0;
            }
        } catch (const std::bad_alloc &) {  // (host memory for the order)
            rc = kNoRoom;
        }
        if (rc && rc != kNoRoom) return rc;
        if (rc) (void)hipGetLastError();  // (of the allocation that did not fit)
    }
    return run_knn_mode(points, N, D, K, indices, sq_dist, s, 0, stats);
}

}  // namespace tsnehip
