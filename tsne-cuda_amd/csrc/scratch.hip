// Large device scratch, kept between calls.
//
// hipMalloc and hipFree of up to 64 MB cost 0.04 ms (the runtime keeps such memory); of 96 MB and more 0.3 ms, or at
// random and for stretches of calls 2 to 15 ms and more, whatever the size: the driver unmaps what is returned and clears
// what it hands out.  A neighbour search of 60000 x 784 points takes and returns five such blocks, a fit a dozen.  So
// blocks of kKeptLeast bytes and more that are returned here are kept for the next call that asks for about as much.
//
// Kept memory is bounded (kKeptMost per device, the longest unused first), and given back: what nobody has asked for in
// kKeptSeconds by the next call that takes or returns any, all of it where the device has no room for a new block, and
// all of it by tsne_hip_release_scratch.  A block is only kept once the device is idle, as hipFree would have waited
// for, so it may be handed to any thread and any stream; where that cannot be had (a capture is going on) it is freed.
#include "common.h"

#include <chrono>
#include <mutex>
#include <vector>

#include "../../include/tsnecuda/tsne_stages.h"

namespace tsnehip {

namespace {

constexpr size_t kKeptLeast = (size_t)32 << 20, kKeptMost = (size_t)2 << 30;
constexpr double kKeptSeconds = 5.0;

struct Block {
    void *p;
    size_t bytes;
    int device;
    std::chrono::steady_clock::time_point since;  // kept
};
struct Pool {
    std::mutex lock;
    std::vector<Block> kept, in_use;
};
// (never destroyed: the runtime may be gone by then, and the process's memory goes with it)
Pool &pool() {
    static Pool *const p = new Pool();
    return *p;
}

// Frees what has been kept too long, the longest unused while more than `most` bytes are kept on `device`, and, for
// device < 0, everything.
void give_back(Pool &pool, int device, size_t most) {
    const auto now = std::chrono::steady_clock::now();
    size_t total = 0;
    for (const Block &b : pool.kept)
        if (b.device == device) total += b.bytes;
    for (size_t k = 0; k < pool.kept.size();) {  // (in the order they were returned)
        const Block b = pool.kept[k];
        const bool old = std::chrono::duration<double>(now - b.since).count() > kKeptSeconds;
        if (!old && device >= 0 && !(b.device == device && total > most)) {
            ++k;
            continue;
        }
        if (b.device == device) total -= b.bytes;
        (void)hipFree(b.p);
        pool.kept.erase(pool.kept.begin() + (long)k);
    }
}

}  // namespace

hipError_t scratch_malloc(void **p, size_t bytes) {
    *p = nullptr;
    if (bytes < kKeptLeast) return hipMalloc(p, bytes ? bytes : 1);
    int device = 0;
    if (const hipError_t e = hipGetDevice(&device)) return e;
    Pool &all = pool();
    std::lock_guard<std::mutex> hold(all.lock);
    size_t best = all.kept.size();
    for (size_t k = 0; k < all.kept.size(); ++k) {
        const Block &b = all.kept[k];
        if (b.device == device && b.bytes >= bytes && b.bytes / 3 * 2 <= bytes &&
            (best == all.kept.size() || b.bytes < all.kept[best].bytes))
            best = k;
    }
    if (best < all.kept.size()) {
        Block b = all.kept[best];
        all.kept.erase(all.kept.begin() + (long)best);
        all.in_use.push_back(b);
        *p = b.p;
        give_back(all, device, kKeptMost);
        return hipSuccess;
    }
    give_back(all, device, kKeptMost);
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        give_back(all, device, 0);
        e = hipMalloc(p, bytes);
    }
    if (e == hipSuccess) all.in_use.push_back({*p, bytes, device, {}});
    return e;
}

void scratch_free(void *p) {
    if (!p) return;
    Pool &all = pool();
    Block b = {};
    {
        std::lock_guard<std::mutex> hold(all.lock);
        for (size_t k = 0; k < all.in_use.size(); ++k)
            if (all.in_use[k].p == p) {
                b = all.in_use[k];
                all.in_use.erase(all.in_use.begin() + (long)k);
                break;
            }
    }
    int device = -1;
    const bool here = b.p && hipGetDevice(&device) == hipSuccess && device == b.device;
    if (!here || hipDeviceSynchronize() != hipSuccess) {
        (void)hipFree(p);
        return;
    }
    std::lock_guard<std::mutex> hold(all.lock);
    b.since = std::chrono::steady_clock::now();
    all.kept.push_back(b);
    give_back(all, b.device, kKeptMost);
}

}  // namespace tsnehip

extern "C" int tsne_hip_release_scratch(void) {
    tsnehip::Pool &all = tsnehip::pool();
    std::lock_guard<std::mutex> hold(all.lock);
    tsnehip::give_back(all, -1, 0);
    return 0;
}
