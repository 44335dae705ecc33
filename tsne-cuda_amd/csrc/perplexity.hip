// Max-normalisation and per-row perplexity search for gfx950.
//
// Semantics: src/util/math_utils.cu:66-74 and
// src/kernels/perplexity_search.cu:10-141 of the reference.  The reference
// iterates all rows in lock-step (<= 200 rounds of: exponentiate nnz values,
// two cuBLAS row reductions, an entropy transform, a per-row update kernel and
// a host-side "all found" reduction).  Rows never interact, so here a group of
// lanes owns a row, keeps its distances in registers and runs the whole
// bisection privately: the distances are read once and the probabilities
// written once.
//
// Reproducible arithmetic.  Whether a row stops at one bisection step or the
// next hangs on the last bits of its entropy, so every operation of the search
// is pinned down: exp and log are the fixed operation sequences of det_math.h,
// nothing is contracted, and the two row sums (of p and of p ln p) are formed in
// one stated order whatever the kernel variant:
//   * 64 interleaved partial sums, partial c taking the values of the slots
//     s = c, c + 64, c + 128, ... in ascending order, starting from +0;
//   * then a balanced tree: partial[c] + partial[c ^ m] for m = 32, 16, 8, 4, 2, 1.
// A CPU restatement that follows the same order gets the same probabilities bit
// for bit.  (The reference's sums are cuBLAS sgemv calls whose order is not
// documented, and its exp/log are the fast intrinsics.)
#include "det_math.h"
#include "plan.h"

#include <algorithm>
#include <cfloat>
#include <mutex>

#include "../../include/tsnecuda/tsne_stages.h"

// Scratch of tsne_hip_max_normalize_noalloc: the device scalar that receives the largest absolute value.
// Every GPU holds its own copy of this array at its own address until the process ends; in host code the
// name is only a handle for hipGetSymbolAddress, never a device address.
static __device__ __align__(256) float scratch[64];

namespace tsnehip {

namespace {

// Bound by memory, and by the atomics on one address if there are many: one per workgroup (one per wave of 4096
// workgroups: 90 M values 237 us, this form 93, 3.9 TB/s), and four values per load where the address allows it.
__global__ __launch_bounds__(256) void abs_max_kernel(const float *__restrict__ v, int64_t n, float *out) {
    __shared__ float partial[256 / kWave];
    float m = 0.0f;
    const int64_t first = (int64_t)blockIdx.x * 256 + threadIdx.x, stride = (int64_t)gridDim.x * 256;
    const int64_t quads = (reinterpret_cast<uintptr_t>(v) & 15) == 0 ? n / 4 : 0;
    for (int64_t t = first; t < quads; t += stride) {
        const float4 x = reinterpret_cast<const float4 *>(v)[t];
        m = fmaxf(m, fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))));
    }
    for (int64_t t = 4 * quads + first; t < n; t += stride) m = fmaxf(m, fabsf(v[t]));
    m = group_max<kWave>(m);
    if ((threadIdx.x & (kWave - 1)) == 0) partial[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < 256 / kWave; ++w) m = fmaxf(m, partial[w]);
        // Non-negative floats order like their bit patterns.
        atomicMax(reinterpret_cast<unsigned int *>(out), __float_as_uint(m));
    }
}

__global__ __launch_bounds__(256) void divide_kernel(float *__restrict__ v, int64_t n, const float *denom) {
    const float d = *denom;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x)
        v[t] = v[t] / d;
}

__global__ void zero_scalar_kernel(float *p) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p = 0.0f;
}

// thrust_transform_functions.h:32-37: x*log(x) with NaN/Inf mapped to 0.
__device__ __forceinline__ float entropy_term(float v) {
#pragma clang fp contract(off)
    const float e = v * det_logf(v);
    return (e != e || isinf(e)) ? 0.0f : e;
}

// v plus the value of the lane that DPP control CTRL names (every lane of a 16-lane row active).
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// group_sum's tree, bit for bit, its last four levels inside the vector instructions: rotations of a 16-lane row by
// 8 and by 4 (after the level of 8 a value depends on the lane modulo 8 only, so 4 back is 4 across), then
// permutations of four.
template <int LANES>
__device__ __forceinline__ float lanes_sum(float v) {
#pragma unroll
    for (int m = LANES / 2; m >= 16; m >>= 1) v += __shfl_xor(v, m, kWave);
    v = dpp_add<0x128>(v);
    v = dpp_add<0x124>(v);
    v = dpp_add<0x4E>(v);
    return dpp_add<0xB1>(v);
}

// The stated summation order for a group of LANES lanes whose lane l holds the slots l + v * LANES: a lane
// owns 64 / LANES of the 64 partial sums (classes l + LANES * (v mod (64 / LANES))); it forms them one after
// the other, combines them by the upper levels of the tree, and the lower levels run across the lanes.
template <int LANES, int VPL>
__device__ __forceinline__ float ordered_row_sum(const float (&val)[VPL]) {
#pragma clang fp contract(off)
    constexpr int kClasses = kWave / LANES;
    float q[kClasses];
#pragma unroll
    for (int c = 0; c < kClasses; ++c) q[c] = 0.0f;
#pragma unroll
    for (int v = 0; v < VPL; ++v) q[v % kClasses] += val[v];
    // Class index c * LANES + lane: the tree's level m = 32 pairs classes c and c ^ (32 / LANES), and so on down.
#pragma unroll
    for (int m = kClasses / 2; m > 0; m >>= 1)
#pragma unroll
        for (int c = 0; c < m; ++c) q[c] += q[c + m];
    return lanes_sum<LANES>(q[0]);
}

// H - ln(perplexity) of a row by the hardware's exponential, logarithm and reciprocal, for 0 <= d < infinity, and
// *slack, a bound of how far the same quantity evaluated by det_expf / det_logf in the stated order is from it.
// In units of u = 2^-24, with a_i = beta d_i (rounded once, the same in both), A = sum p_i a_i, L = |ln sum|,
// `depth` the additions a term goes through:
//   exponentials: within 6 u each of e^-a_i on either side; H moves by sum p_i |ln p_i + H| <= 2 (A + L) times that;
//   ln v_i against -a_i: 6 + 4 A, and A for the products;
//   sums: depth (1 + 2 A) on either side, A for the fused ones; quotients and logarithms of the sums: 6 A + 9 L + 4;
//   last additions: 3 (A + L) + 2 |ln perplexity|.
// Terms below the smallest normal number count as zero, which the caller's limit on the sum makes harmless.
template <int LANES, int VPL>
__device__ __forceinline__ float approximate_excess(const float (&d)[VPL], const bool (&use)[VPL], float beta,
                                                    float log_target, float *sum_out, float *slack) {
#pragma clang fp contract(off)
    constexpr int kDepth = VPL + 6;
    float sum = 0.0f, weighted = 0.0f;
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
        const float a = beta * d[v];
        const float x = a * -1.44269502f;  // log2 e, whose remaining 1.925963e-8 goes in with the product's rounding
        float r = fmaf(a, -1.44269502f, -x);
        r = fmaf(a, -1.925963e-8f, r);
        float e = __builtin_amdgcn_exp2f(x);
        e = fmaf(e, r * 0.693147181f, e);
        e = use[v] ? e : 0.0f;
        sum += e;
        weighted = fmaf(e, a, weighted);
    }
    sum = lanes_sum<LANES>(sum);
    weighted = lanes_sum<LANES>(weighted);
    const float A = weighted * __builtin_amdgcn_rcpf(sum);
    const float log_sum = __builtin_amdgcn_logf(sum) * 0.693147181f;  // (the builtin is log2)
    const float L = fabsf(log_sum);
    *sum_out = sum;
    *slack = 5.9604644775390625e-08f *
             ((float)(48 + 4 * kDepth) * (A + L) + (float)(16 + 2 * kDepth) + 4.0f * fabsf(log_target));
    return (A + log_sum) - log_target;
}

// One row per LANES-lane group, VPL values per lane held in registers.
// Bound by the vector ALU: an evaluation by det_expf / det_logf takes about 55 instructions per neighbour, and a row
// evaluates 15 to 20 exponents.  But all that an evaluation decides, until the last, is a sign: so each exponent
// is first evaluated by the hardware's functions (13 instructions), and where that is further from the target than
// the tolerance plus a bound of the two evaluations' difference, the search goes on from its sign - the same path.
// The rows of a wave that cannot tell wait for each other and are then evaluated exactly together.  Sixteen lanes
// per row up to 128 neighbours: four rows share the search's scalar part, and sums stay inside a DPP row.
// 1,000,000 x 90, tolerance 1e-4, us: every exponent exactly, 32 lanes per row 3647; this form 1442.
template <int LANES, int VPL>
__global__ __launch_bounds__(256) void perplexity_kernel(const float *__restrict__ sq_dist, int N, int K,
                                                         float log_target, float eps, float *__restrict__ pij,
                                                         float *__restrict__ betas) {
#pragma clang fp contract(off)
    constexpr int kRowsPerBlock = 256 / LANES;
    const int row = blockIdx.x * kRowsPerBlock + threadIdx.x / LANES;
    const int lane = threadIdx.x % LANES;
    const bool live = row < N;
    const size_t base = (size_t)(live ? row : 0) * K;

    float d[VPL];
    bool use[VPL];
    bool plain = true;
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
        const int s = lane + v * LANES;
        d[v] = (live && s < K) ? sq_dist[base + s] : 0.0f;
        // perplexity_search.cu:32: neighbour 0 at distance 0 is the point itself.
        use[v] = s < K && !(s == 0 && d[v] == 0.0f);
        plain = plain && d[v] >= 0.0f && d[v] < INFINITY;
    }
    const bool filter = __all(plain);

    float beta = 1.0f, lo = -FLT_MAX, hi = FLT_MAX;
    float p[VPL];
    float sum = 1.0f;
    bool done = !live;
    int it = 0;
    auto advance = [&](bool up) {
        if (up) {
            lo = beta;
            beta = (hi == FLT_MAX || hi == -FLT_MAX) ? beta * 2.0f : (beta + hi) / 2.0f;
        } else {
            hi = beta;
            beta = (lo == -FLT_MAX || lo == FLT_MAX) ? beta / 2.0f : (beta + lo) / 2.0f;
        }
        ++it;
    };
    // A row that the approximate evaluation could not tell kUndecided times has come to the end of its search, which a
    // tolerance below the arithmetic's own keeps it from leaving: the rest of its steps are evaluated exactly only.
    // 100,000 x 90, us, tolerance 1e-4 / 0: every exponent exactly 318 / 3287; approximate first throughout 123 / 3431;
    // up to one time 141 / 2811, three 123 / 2805, six 122 / 2818 (all before the rule below).
    constexpr int kUndecided = 3;
    int undecided = 0;
    // A step that leaves beta as it was would be taken again and again: the same beta gives the same excess and direction.
    // Rows whose distances are large beside their spread get there after some forty steps of 199 (their sums underflow
    // where the tolerance would be met): 60000 x 784 pixel vectors, 45 neighbours, 909 -> 178 us;
    // 50000 x 1024, 90 neighbours, 728 -> 204; 100,000 x 90 at tolerance 0 2892 -> 356.
    // (every pass of either loop advances a row that is not done or ends its part; a row takes 199 at most)
    while (!__all(done)) {
        bool open = filter && !done && it < 199 && undecided < kUndecided;
        while (__any(open)) {
            float s, slack;
            const float diff = approximate_excess<LANES, VPL>(d, use, beta, log_target, &s, &slack);
            if (open) {
                open = s >= 1e-24f && fabsf(diff) > fmaxf(eps, 0.0f) + slack;  // (false where one is not a number)
                if (open) {
                    advance(diff > 0.0f);
                    open = it < 199;
                }
            }
        }
        ++undecided;
        if (!done) {
            float et[VPL];
#pragma unroll
            for (int v = 0; v < VPL; ++v) {
                p[v] = use[v] ? det_expf(-beta * d[v]) : 0.0f;
                et[v] = lane + v * LANES < K ? entropy_term(p[v]) : 0.0f;
            }
            sum = ordered_row_sum<LANES, VPL>(p);
            const float ent = ordered_row_sum<LANES, VPL>(et);
            const float H = (-ent / sum) + det_logf(sum);
            const float diff = H - log_target;
            const bool found = (diff < eps && -diff < eps);
            if (found || it == 199) {
                done = true;
            } else {
                const float before = beta;
                advance(diff > 0);
                done = beta == before;  // (as it would be after every step to come, and p and sum are of it)
            }
        }
    }
    if (live) {
#pragma unroll
        for (int v = 0; v < VPL; ++v) {
            const int s = lane + v * LANES;
            if (s < K) pij[base + s] = p[v] / sum;
        }
        if (betas && lane == 0) betas[row] = beta;
    }
}

// Any K: one wave per row, distances re-read from memory every round.
__global__ __launch_bounds__(256) void perplexity_generic_kernel(const float *__restrict__ sq_dist, int N, int K,
                                                                 float log_target, float eps,
                                                                 float *__restrict__ pij,
                                                                 float *__restrict__ betas) {
#pragma clang fp contract(off)
    const int row = blockIdx.x * (256 / kWave) + threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    if (row >= N) return;
    const size_t base = (size_t)row * K;
    float beta = 1.0f, lo = -FLT_MAX, hi = FLT_MAX, sum = 1.0f;
    for (int it = 0; it < 200; ++it) {
        float ls = 0.0f, le = 0.0f;
        for (int s = lane; s < K; s += kWave) {
            const float dv = sq_dist[base + s];
            const float pv = (s == 0 && dv == 0.0f) ? 0.0f : det_expf(-beta * dv);
            ls += pv;
            le += entropy_term(pv);
        }
        sum = group_sum<kWave>(ls);
        const float ent = group_sum<kWave>(le);
        const float H = (-ent / sum) + det_logf(sum);
        const float diff = H - log_target;
        const bool found = (diff < eps && -diff < eps);
        if (found || it == 199) break;
        const float before = beta;
        if (diff > 0) {
            lo = beta;
            beta = (hi == FLT_MAX || hi == -FLT_MAX) ? beta * 2.0f : (beta + hi) / 2.0f;
        } else {
            hi = beta;
            beta = (lo == -FLT_MAX || lo == FLT_MAX) ? beta / 2.0f : (beta + lo) / 2.0f;
        }
        if (beta == before) break;  // (as above)
    }
    for (int s = lane; s < K; s += kWave) {
        const float dv = sq_dist[base + s];
        const float pv = (s == 0 && dv == 0.0f) ? 0.0f : det_expf(-beta * dv);
        pij[base + s] = pv / sum;
    }
    if (betas && lane == 0) betas[row] = beta;
}

}  // namespace

// scratch: one device float.
int launch_max_normalize(float *values, int64_t n, float *scratch, hipStream_t s) {
    zero_scalar_kernel<<<1, 64, 0, s>>>(scratch);
    TSNE_LAUNCHED(s);
    const int blocks = std::max(1, (int)std::min<int64_t>(div_up(n, 256 * 4), 4096));
    abs_max_kernel<<<std::min(blocks, 2048), 256, 0, s>>>(values, n, scratch);
    TSNE_LAUNCHED(s);
    divide_kernel<<<blocks, 256, 0, s>>>(values, n, scratch);
    TSNE_LAUNCHED(s);
    return 0;
}

namespace {
constexpr int kMaxDevices = 64;
constexpr int64_t kNoAllocMaxValues = (int64_t)1 << 32;
std::mutex g_scratch_mutex;
float *g_scratch_ptr[kMaxDevices] = {};
}  // namespace

// The address of `scratch` on the current device, looked up once per device.
int noalloc_scratch(float **out) {
    int dev = -1;
    TSNE_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) {
        set_error("max_normalize_noalloc: device %d is outside the supported range [0, %d)", dev, kMaxDevices);
        return 1;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        float *ptr = nullptr;
        TSNE_TRY(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
        if (!ptr) {
            set_error("max_normalize_noalloc: hipGetSymbolAddress returned a null address");
            return 1;
        }
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

int launch_perplexity(const float *sq_dist, int N, int K, float perplexity, float eps, float *pij, float *betas,
                      hipStream_t s) {
    const float log_target = det_logf(perplexity);
#define TSNE_PERP(LANES, VPL)                                                                                  \
    perplexity_kernel<LANES, VPL><<<div_up(N, 256 / LANES), 256, 0, s>>>(sq_dist, N, K, log_target, eps, pij, \
                                                                         betas)
    if (K <= 32) {
        TSNE_PERP(16, 2);
    } else if (K <= 64) {
        TSNE_PERP(16, 4);
    } else if (K <= 96) {
        TSNE_PERP(16, 6);
    } else if (K <= 128) {
        TSNE_PERP(16, 8);
    } else if (K <= 256) {
        TSNE_PERP(32, 8);
    } else if (K <= 512) {
        TSNE_PERP(64, 8);
    } else if (K <= 1024) {
        TSNE_PERP(64, 16);
    } else {
        perplexity_generic_kernel<<<div_up(N, 256 / kWave), 256, 0, s>>>(sq_dist, N, K, log_target, eps, pij, betas);
    }
#undef TSNE_PERP
    TSNE_LAUNCHED(s);
    return 0;
}

}  // namespace tsnehip

extern "C" int tsne_hip_max_normalize_noalloc(float *values, int64_t n, void *stream) {
    using namespace tsnehip;
    if (!values || n <= 0) {
        set_error("max_normalize_noalloc: need a non-empty array");
        return 1;
    }
    if (n > kNoAllocMaxValues) {
        set_error("max_normalize_noalloc: %lld values exceed the supported maximum of %lld", (long long)n,
                  (long long)kNoAllocMaxValues);
        return 1;
    }
    float *ptr = nullptr;
    if (noalloc_scratch(&ptr)) return 1;
    // launch_max_normalize clears the scalar with a kernel (no memset node, so the call may be captured).
    return launch_max_normalize(values, n, ptr, (hipStream_t)stream);
}
