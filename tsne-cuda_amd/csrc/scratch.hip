// Large device scratch, kept between calls.
//
// hipMalloc and hipFree of 2 to 64 MB cost 15 to 30 us more than a wait for the device, which what is kept takes too; of
// more 0.3 ms, or at random and for stretches of calls 2 to 15 ms and more, whatever the size: the driver unmaps what is
// returned and clears what it hands out.  (A block filled by a kernel, us, taken and returned / kept: 1 MB 12.2 / 11.5, 2 MB
// 35 / 12, 8 MB 26 to 35 / 13, 16 MB 38 / 15, 32 MB 40 / 17, 64 MB 54 / 23, 72 MB 338 / 24, 256 MB 376 / 58.  The runtime has
// less than 2 MB in hand.)  A search of 60000 x 784 points takes and returns five of the large ones, a fit a dozen.  So
// blocks of kKeptLeast bytes, 2 MB, and more that are returned here are kept for the next call that asks for about as much
// (a block may be half as large again as what it is handed out for).
//
// Kept memory is bounded (kKeptMost per device, the longest unused first), and given back: what nobody has asked for in
// kKeptSeconds by the next call that takes or returns any, all of it where the device has no room for anything that the
// library allocates, and all of it by tsne_hip_release_scratch.  A block is only kept once the device is idle, as hipFree
// would have waited for, so it may be handed to any thread and any stream; where that cannot be had (a capture is going
// on) it is freed.
#include "common.h"
#include "scratch_pool.h"

#include <chrono>

#include "../../include/tsnecuda/tsne_stages.h"

namespace tsnehip {

namespace {

struct HipDevice {
    int alloc(void **p, size_t bytes) {
        const hipError_t e = hipMalloc(p, bytes);
        if (e != hipSuccess) *p = nullptr;
        return (int)e;
    }
    void forgive() { (void)hipGetLastError(); }
    void free(void *p) { (void)hipFree(p); }
    int current() {
        int device = -1;
        return hipGetDevice(&device) == hipSuccess ? device : -1;
    }
    bool idle() {
        if (hipDeviceSynchronize() == hipSuccess) return true;
        (void)hipGetLastError();  // (what a kernel left comes up again)
        return false;
    }
    double now() { return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count(); }
};

// (never destroyed: the runtime may be gone by then, and the process's memory goes with it)
ScratchPool<HipDevice> &pool() {
    static ScratchPool<HipDevice> *const p = new ScratchPool<HipDevice>();
    return *p;
}

}  // namespace

hipError_t device_malloc_bytes(void **p, size_t bytes) { return (hipError_t)pool().plain(p, bytes); }
hipError_t scratch_malloc(void **p, size_t bytes) { return (hipError_t)pool().take(p, bytes); }
void scratch_free(void *p) { pool().put(p); }

}  // namespace tsnehip

extern "C" int tsne_hip_release_scratch(void) {
    tsnehip::pool().release();
    return 0;
}
