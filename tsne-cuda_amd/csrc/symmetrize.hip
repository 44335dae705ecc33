// Pattern-restricted symmetrisation of the conditional probabilities for gfx950.
//
//   P[i,s] = (p[i,s] + sum_{t : idx[j,t] == i} p[j,t]) / (2 N),   j = idx[i,s]
//
// Semantics: src/util/math_utils.cu:269-291 of the reference (the N x K pattern
// is kept; pairs present in only one direction keep half their mass).  The
// reference gives every non-zero its own thread that walks row j alone: N K^2
// index reads, 32 GB at a million points and 90 neighbours.  Two forms here:
//   * hashed (the default from 4096 points up): every row's (column, value)
//     pairs go once into a small open-addressing table of the row's own (a power
//     of two >= 1.25 K slots of 8 bytes, in buckets of 16 that overflow into the
//     next, built in LDS by a group of lanes per row); a non-zero looks for its row
//     number in the table of row j.  Large tables hold a byte of each column's hash
//     and its place in the row instead: 16 bytes of a bucket answer most lookups,
//     the row itself the others, and a pair is looked up once for both its entries;
//   * scanning (small problems, more than 1638 neighbours, rows that name a column
//     twice, or when the tables do not fit in memory): a group of lanes owns row i
//     and the whole group scans each row j
//     together, so every index row is fetched with coalesced loads and the match
//     is found with a ballot.
#include "plan.h"
#include "stages.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace tsnehip {

namespace {

template <int LANES>
__global__ __launch_bounds__(256) void symmetrize_kernel(const float *__restrict__ p, const int *__restrict__ idx,
                                                         int N, int K, float *__restrict__ P) {
    constexpr int kRowsPerBlock = 256 / LANES;
    const int row = blockIdx.x * kRowsPerBlock + threadIdx.x / LANES;
    const int lane = threadIdx.x % LANES;
    if (row >= N) return;  // whole groups leave together
    const size_t base = (size_t)row * K;
    const double denom = 2.0 * (double)N;
    for (int s0 = 0; s0 < K; s0 += LANES) {
        const int my_s = s0 + lane;
        const int my_j = my_s < K ? idx[base + my_s] : 0;
        float my_acc = my_s < K ? p[base + my_s] : 0.0f;
        const int count = min(LANES, K - s0);
        for (int t = 0; t < count; ++t) {
            const int j = __shfl(my_j, t, LANES);
            const size_t jb = (size_t)j * K;
            float found = 0.0f;
            // (a column that names no point has no row to scan)
            for (int u = (unsigned int)j < (unsigned int)N ? lane : K; u < K; u += LANES)
                if (idx[jb + u] == row) found += p[jb + u];
            found = group_sum<LANES>(found);
            if (lane == t) my_acc += found;
        }
        if (my_s < K) P[base + my_s] = (float)((double)my_acc / denom);
    }
}

// ---- hashed form ----------------------------------------------------------
struct Slot {
    int key;  // column, -1: empty
    float value;
};
constexpr int kBucket = 16;  // slots; their tags are one 16-byte load
__device__ __forceinline__ unsigned int hash_of(int key) { return (unsigned int)key * 0x9E3779B1u; }
// The tag of a column, 1 to 255 (0: an empty slot), from hash bits below those that choose the slot.
__device__ __forceinline__ unsigned int tag_of(unsigned int hash) {
    const unsigned int t = (hash >> 13) & 0xffu;
    return t ? t : 1u;
}

// The slot after `at`, the seen-th looked at: round the bucket (all of a smaller table), then the next bucket.
__device__ __forceinline__ unsigned int next_slot(unsigned int at, int seen, int log2_slots) {
    const unsigned int slots = 1u << log2_slots, within = min((unsigned int)kBucket, slots) - 1u;
    at = (at & ~within) | ((at + 1u) & within);
    return (seen & (kBucket - 1)) ? at : (at + kBucket) & (slots - 1u);
}

// A neighbour's place in its row, in tables built by LANES lanes per row: up to 204 neighbours by 16, else 64.
template <int LANES>
using PlaceOf = std::conditional_t<LANES == 16, unsigned char, unsigned short>;
// A bucket without slots: the columns' tags, one load, and their places in the row.
template <typename PLACE>
struct alignas(16) Tagged {
    unsigned int tags[kBucket / 4];
    PLACE places[kBucket];
};

// A group of LANES lanes per row builds the row's table in LDS (insertions race for empty slots with a
// compare-and-swap; which slot of its bucket a column ends up in does not matter to a lookup, and it goes to the
// next bucket only when its own is full) and writes it out whole: the slots, or (tagged != nullptr) the columns' tags
// and their places in the row.  flags[0]: some row names a column twice (the caller then takes the scanning form,
// which adds such values up); flags[1]: a column outside [0, N).
template <int LANES>
__global__ __launch_bounds__(256) void build_tables_kernel(const float *__restrict__ p, const int *__restrict__ idx,
                                                           int N, int K, int log2_slots, Slot *__restrict__ table,
                                                           Tagged<PlaceOf<LANES>> *__restrict__ tagged,
                                                           int *__restrict__ flags) {
    extern __shared__ Slot lds_tables[];
    constexpr int kRows = 256 / LANES;
    const int slots = 1 << log2_slots;
    const int group = threadIdx.x / LANES, lane = threadIdx.x % LANES;
    const int row = blockIdx.x * kRows + group;
    Slot *mine = lds_tables + (size_t)group * slots;
    for (int e = lane; e < slots; e += LANES) mine[e] = Slot{-1, 0.0f};
    __syncthreads();
    bool twice = false, outside = false;
    if (row < N) {
        const size_t base = (size_t)row * K;
        for (int t = lane; t < K; t += LANES) {
            const int key = idx[base + t];
            const float v = tagged ? __int_as_float(t) : p[base + t];
            if ((unsigned int)key >= (unsigned int)N) {
                outside = true;
                continue;
            }
            unsigned int at = hash_of(key) >> (32 - log2_slots);
            for (int seen = 1;; ++seen) {  // (more slots than pairs: an empty one is always met)
                const int old = atomicCAS(&mine[at].key, -1, key);
                if (old == -1) {
                    mine[at].value = v;
                    break;
                }
                if (old == key) {
                    twice = true;
                    break;
                }
                at = next_slot(at, seen, log2_slots);
            }
        }
    }
    if (__any(twice) && (threadIdx.x & (kWave - 1)) == 0) atomicOr(&flags[0], 1);
    if (__any(outside) && (threadIdx.x & (kWave - 1)) == 0) atomicOr(&flags[1], 1);
    __syncthreads();
    if (row < N) {
        if (!tagged) {
            Slot *out = table + ((size_t)row << log2_slots);
            for (int e = lane; e < slots; e += LANES) out[e] = mine[e];
            return;
        }
        Tagged<PlaceOf<LANES>> *out = tagged + ((size_t)row << (log2_slots - 4));
        for (int e = lane; e < slots; e += LANES) {  // (whole groups of four lanes: slots and LANES are multiples of 16)
            const Slot here = mine[e];
            out[e / kBucket].places[e % kBucket] = (PlaceOf<LANES>)__float_as_int(here.value);
            unsigned int four = (here.key < 0 ? 0u : tag_of(hash_of(here.key))) << (8 * (lane & 3));
            four |= __builtin_amdgcn_update_dpp(0u, four, 0xB1, 0xf, 0xf, true);  // lane ^ 1
            four |= __builtin_amdgcn_update_dpp(0u, four, 0x4E, 0xf, 0xf, true);  // lane ^ 2
            if ((lane & 3) == 0) out[e / kBucket].tags[e % kBucket / 4] = four;
        }
    }
}

constexpr size_t kTaggedBytes = (size_t)512 << 20;  // slots of more bytes than this are replaced by tags and places

// Tables of slots.  Bound by the cache lines that the lookups touch, random ones.
__global__ __launch_bounds__(256) void symmetrize_hashed_kernel(const float *__restrict__ p, const int *__restrict__ idx,
                                                                int N, int K, int log2_slots,
                                                                const Slot *__restrict__ table,
                                                                const int *__restrict__ flags, float *__restrict__ P) {
    if (flags[0] | flags[1]) return;  // (a column out of range: P stays as it is; one named twice: the scan writes it)
    const size_t nnz = (size_t)N * K;
    const double denom = 2.0 * (double)N;
    for (size_t e0 = (size_t)blockIdx.x * 256; e0 < nnz; e0 += (size_t)gridDim.x * 256) {
        const size_t row0 = e0 / (unsigned int)K, e = e0 + threadIdx.x;
        if (e >= nnz) return;
        const int row = (int)row0 + (int)((unsigned int)(e - row0 * K) / (unsigned int)K);
        const int j = idx[e];
        const float own = p[e];
        float found = 0.0f;
        if ((unsigned int)j < (unsigned int)N) {
            const Slot *theirs = table + ((size_t)j << log2_slots);
            unsigned int at = hash_of(row) >> (32 - log2_slots);
            for (int seen = 1;; ++seen) {  // (an empty slot is always met)
                const Slot here = theirs[at];
                if (here.key == row) {
                    found = here.value;
                    break;
                }
                if (here.key < 0) break;
                at = next_slot(at, seen, log2_slots);
            }
        }
        P[e] = (float)((double)(own + found) / denom);
    }
}

// Tables of tags and places, in two kernels.  A pair that both rows name has one value, p[i,j] + p[j,i] over 2 N, at two
// places: it is looked up once, by the row of the smaller number, which finds the other place and writes both.  Before
// that every entry is written as if its pair were named once (a point that names itself: twice its own).
__global__ __launch_bounds__(256) void halve_entries_kernel(const float *__restrict__ p, const int *__restrict__ idx, int N, int K,
                                                            const int *__restrict__ flags, float *__restrict__ P) {
    if (flags[0] | flags[1]) return;  // (as above)
    const size_t nnz = (size_t)N * K;
    const double denom = 2.0 * (double)N;
    for (size_t e0 = (size_t)blockIdx.x * 1024; e0 < nnz; e0 += (size_t)gridDim.x * 1024) {
        const size_t row0 = e0 / (unsigned int)K;
        const unsigned int in_row0 = (unsigned int)(e0 - row0 * K);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const unsigned int t = u * 256 + threadIdx.x;
            if (e0 + t >= nnz) break;
            const float own = p[e0 + t];
            const bool self = idx[e0 + t] == (int)row0 + (int)((in_row0 + t) / (unsigned int)K);
            P[e0 + t] = (float)((double)(own + (self ? own : 0.0f)) / denom);
        }
    }
}

// 0x80 in every byte of w that is zero.
__device__ __forceinline__ unsigned int zero_bytes(unsigned int w) {
    return ~(((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w | 0x7f7f7f7fu);
}

// Bound by the cache lines that the lookups touch, random ones, four lookups of a thread in flight.  A lookup reads its
// bucket's tags first and ends there unless one matches (50-dimensional Gaussians: one lookup in four finds its column); the
// match's place leads to the row's own column and value.  Tags and places of a million rows of 90 neighbours are 256 MB
// where slots are 1 GB.  1,000,000 x 90, us: lookups in slots 2970; of every entry in this form 2340;
// of a pair once 1397, and 187 for the entries as if named once.
constexpr int kLookups = 4;
template <typename PLACE>
__global__ __launch_bounds__(256) void symmetrize_pairs_kernel(const float *__restrict__ p, const int *__restrict__ idx, int N,
                                                               int K, int log2_slots, const Tagged<PLACE> *__restrict__ tagged,
                                                               const int *__restrict__ flags, float *__restrict__ P) {
    if (flags[0] | flags[1]) return;  // (as above)
    const size_t nnz = (size_t)N * K;
    const double denom = 2.0 * (double)N;
    const unsigned int buckets = 1u << (log2_slots - 4);
    for (size_t e0 = (size_t)blockIdx.x * (256 * kLookups); e0 < nnz; e0 += (size_t)gridDim.x * (256 * kLookups)) {
        const size_t row0 = e0 / (unsigned int)K;
        const unsigned int in_row0 = (unsigned int)(e0 - row0 * K);
        int row[kLookups], col[kLookups];  // (col < 0: nothing to look up)
        uint4 first[kLookups];
#pragma unroll
        for (int u = 0; u < kLookups; ++u) {
            const unsigned int t = u * 256 + threadIdx.x;
            row[u] = (int)row0 + (int)((in_row0 + t) / (unsigned int)K);
            col[u] = e0 + t < nnz ? idx[e0 + t] : -1;
        }
#pragma unroll
        for (int u = 0; u < kLookups; ++u) {
            if (col[u] <= row[u] || col[u] >= N) col[u] = -1;
            const unsigned int bucket = (hash_of(row[u]) >> (32 - log2_slots)) / kBucket;
            first[u] = make_uint4(0u, 0u, 0u, 0u);
            if (col[u] >= 0)
                first[u] = *reinterpret_cast<const uint4 *>(tagged[((size_t)col[u] << (log2_slots - 4)) + bucket].tags);
        }
#pragma unroll
        for (int u = 0; u < kLookups; ++u) {
            if (col[u] < 0) continue;
            const unsigned int hash = hash_of(row[u]), tag = tag_of(hash) * 0x01010101u;
            unsigned int bucket = (hash >> (32 - log2_slots)) / kBucket;
            const Tagged<PLACE> *theirs = tagged + ((size_t)col[u] << (log2_slots - 4));
            const size_t their_row = (size_t)col[u] * K;
            uint4 t = first[u];
            for (unsigned int visited = 0;;) {
                const unsigned int w[4] = {t.x, t.y, t.z, t.w};
                unsigned int empty = 0u, matches = 0u;  // (matches: a bit per slot of the bucket)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    empty |= zero_bytes(w[k]);
                    matches |= (((zero_bytes(w[k] ^ tag) >> 7) * 0x10204080u) >> 28) << (4 * k);
                }
                bool hit = false;
                while (matches && !hit) {
                    const size_t at = their_row + theirs[bucket].places[__ffs((int)matches) - 1];
                    matches &= matches - 1u;
                    const int key = idx[at];
                    const float value = p[at];
                    if (key == row[u]) {
                        const size_t e = e0 + u * 256 + threadIdx.x;
                        P[e] = P[at] = (float)((double)(p[e] + value) / denom);
                        hit = true;
                    }
                }
                if (hit || empty || ++visited == buckets) break;
                bucket = (bucket + 1u) & (buckets - 1u);
                t = *reinterpret_cast<const uint4 *>(theirs[bucket].tags);
            }
        }
    }
}

__global__ __launch_bounds__(256) void index_range_kernel(const int *__restrict__ idx, int64_t n, int N,
                                                          int *__restrict__ flag) {
    bool bad = false;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x)
        bad = bad || (unsigned int)idx[e] >= (unsigned int)N;
    if (__any(bad) && (threadIdx.x & (kWave - 1)) == 0) atomicOr(flag, 1);
}

}  // namespace

// The stages that turn neighbour numbers into addresses of their own (sort keys, LDS bitmaps, row pointers)
// first make sure that every one of them names a point: 0 if all n indices lie in [0, N), else 1 with the error
// set.  Synchronises the stream.
int validate_indices(const int *idx, int64_t n, int N, const char *who, hipStream_t s) {
    int *flag = nullptr;
    TSNE_TRY(device_malloc(&flag, sizeof(int)));
    int host = 0;
    hipError_t e = hipMemsetAsync(flag, 0, sizeof(int), s);
    if (e == hipSuccess) {
        index_range_kernel<<<(int)std::min<int64_t>(div_up(n, 256 * 8), 2048), 256, 0, s>>>(idx, n, N, flag);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(&host, flag, sizeof(int), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipFree(flag);
    TSNE_TRY(e);
    if (host) {
        set_error("%s: a neighbour index lies outside [0, %d)", who, N);
        return 1;
    }
    return 0;
}

int launch_symmetrize(const float *p, const int *idx, int N, int K, float *P, hipStream_t s) {
    // Hashed form: tables of next_pow2(1.25 K) slots per row, at least 8 (1,000,000 x 2: 0.13 ms, with 16 0.39),
    // or where those are many, of tags in whole buckets.
    int log2_slots = 3;
    while ((1 << log2_slots) < K + (K + 3) / 4) ++log2_slots;
    if (((size_t)N << log2_slots) * sizeof(Slot) > kTaggedBytes) log2_slots = std::max(log2_slots, 4);
    const size_t slots = (size_t)N << log2_slots;
    const bool scan_only = std::getenv("TSNE_SYMMETRIZE_SCAN") != nullptr;  // (for measurements and tests)
    if (N >= 4096 && log2_slots <= 11 && slots * sizeof(Slot) <= ((size_t)64 << 30) && !scan_only) {
        void *memory = nullptr;
        const bool tagged = slots * sizeof(Slot) > kTaggedBytes, narrow = log2_slots <= 8;
        const size_t table_bytes = !tagged ? slots * sizeof(Slot) :
                                   slots / kBucket * (narrow ? sizeof(Tagged<PlaceOf<16>>) : sizeof(Tagged<PlaceOf<64>>));
        if (malloc_optional(&memory, table_bytes + 2 * sizeof(int)) == hipSuccess) {
            Slot *table = tagged ? nullptr : static_cast<Slot *>(memory);
            int *flags = reinterpret_cast<int *>(static_cast<char *>(memory) + table_bytes);
            int raised[2] = {0, 0};
            hipError_t e = hipMemsetAsync(flags, 0, sizeof(raised), s);
            if (e == hipSuccess && !narrow)
                e = hipFuncSetAttribute(reinterpret_cast<const void *>(build_tables_kernel<64>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)(sizeof(Slot) * 4 << 11));
            if (e == hipSuccess) {
                auto *bytes = tagged ? static_cast<Tagged<PlaceOf<16>> *>(memory) : nullptr;
                auto *words = tagged ? static_cast<Tagged<PlaceOf<64>> *>(memory) : nullptr;
                if (narrow)
                    build_tables_kernel<16><<<div_up(N, 16), 256, sizeof(Slot) * 16 << log2_slots, s>>>(
                        p, idx, N, K, log2_slots, table, bytes, flags);
                else
                    build_tables_kernel<64><<<div_up(N, 4), 256, sizeof(Slot) * 4 << log2_slots, s>>>(
                        p, idx, N, K, log2_slots, table, words, flags);
                const int grid = (int)std::min<int64_t>(div_up((int64_t)N * K, 256), 1 << 20);
                if (!tagged) {
                    symmetrize_hashed_kernel<<<grid, 256, 0, s>>>(p, idx, N, K, log2_slots, table, flags, P);
                } else {
                    const int by_four = (int)std::min<int64_t>(div_up((int64_t)N * K, 1024), 1 << 18);
                    halve_entries_kernel<<<by_four, 256, 0, s>>>(p, idx, N, K, flags, P);
                    if (narrow)
                        symmetrize_pairs_kernel<<<by_four, 256, 0, s>>>(p, idx, N, K, log2_slots, bytes, flags, P);
                    else
                        symmetrize_pairs_kernel<<<by_four, 256, 0, s>>>(p, idx, N, K, log2_slots, words, flags, P);
                }
                e = hipGetLastError();
            }
            if (e == hipSuccess) e = hipMemcpyAsync(raised, flags, sizeof(raised), hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipStreamSynchronize(s);  // the tables go
            scratch_free(memory);
            if (e != hipSuccess) {
                set_error("symmetrize: %s", hipGetErrorString(e));
                return 1;
            }
            if (raised[1]) {
                set_error("symmetrize: a neighbour index lies outside [0, %d)", N);
                return 1;
            }
            if (!raised[0]) return 0;
            // (some row names a column twice: the scanning form below adds those values up)
        } else {
            (void)hipGetLastError();  // no room for the tables: the scanning form needs none
        }
    }
    if (K <= 16) {
        symmetrize_kernel<16><<<div_up(N, 256 / 16), 256, 0, s>>>(p, idx, N, K, P);
    } else if (K <= 96) {
        symmetrize_kernel<32><<<div_up(N, 256 / 32), 256, 0, s>>>(p, idx, N, K, P);
    } else {
        symmetrize_kernel<64><<<div_up(N, 256 / 64), 256, 0, s>>>(p, idx, N, K, P);
    }
    TSNE_LAUNCHED(s);
    return 0;
}

}  // namespace tsnehip
