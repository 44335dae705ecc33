// Bookkeeping of the device scratch that is kept between calls (scratch.hip has the reasons), on any device: a test
// compiles it for the host with an allocator and a clock of its own.
//
// Device: int alloc(void **, size_t), whose errors are its own, 0 for none; void forgive(), an error that is mended;
// void free(void *); int current(), the calling thread's device (-1: unknown); bool idle(), which waits for it;
// double now() in seconds.  Nothing here throws.
#ifndef TSNE_HIP_SCRATCH_POOL_H_
#define TSNE_HIP_SCRATCH_POOL_H_

#include <cstddef>
#include <mutex>
#include <new>
#include <vector>

namespace tsnehip {

constexpr size_t kKeptLeast = (size_t)2 << 20, kKeptMost = (size_t)2 << 30;
constexpr double kKeptSeconds = 5.0;

template <class Device>
class ScratchPool {
  public:
    explicit ScratchPool(Device device = Device()) : device_(device) {}

    // Memory that is not kept; where there is no room for it, kept memory goes first.
    int plain(void **p, size_t bytes) {
        const int e = device_.alloc(p, bytes);
        if (!e) return 0;
        const int here = device_.current();
        if (here < 0) return e;
        std::lock_guard<std::mutex> hold(lock_);
        give_back(here, 0);  // (tried again also if that gave nothing: another thread may just have given it)
        device_.forgive();
        return device_.alloc(p, bytes);
    }

    // Scratch of a call, to be returned by put.
    int take(void **p, size_t bytes) {
        *p = nullptr;
        const int here = device_.current();
        if (bytes < kKeptLeast || here < 0) return plain(p, bytes ? bytes : 1);
        {
            std::lock_guard<std::mutex> hold(lock_);
            size_t best = kept_.size();
            for (size_t k = 0; k < kept_.size(); ++k) {
                const Block &b = kept_[k];
                if (b.device == here && b.bytes >= bytes && b.bytes / 3 * 2 <= bytes &&
                    (best == kept_.size() || b.bytes < kept_[best].bytes))
                    best = k;
            }
            if (best < kept_.size()) {
                const Block b = kept_[best];
                kept_.erase(kept_.begin() + (long)best);
                in_use_.push_back(b);  // (room_for_one, when it was first taken)
                *p = b.p;
            }
            give_back(here, kKeptMost);
            if (*p) return 0;
        }
        if (const int e = plain(p, bytes)) return e;
        std::lock_guard<std::mutex> hold(lock_);
        if (room_for_one()) in_use_.push_back({*p, bytes, here, 0.0});  // (else it is freed when it is returned)
        return 0;
    }

    void put(void *p) {
        if (!p) return;
        Block b = {};
        {
            std::lock_guard<std::mutex> hold(lock_);
            for (size_t k = 0; k < in_use_.size(); ++k)
                if (in_use_[k].p == p) {
                    b = in_use_[k];
                    in_use_.erase(in_use_.begin() + (long)k);
                    ++returning_;  // (its places stay reserved)
                    break;
                }
        }
        const bool keep = b.p && device_.current() == b.device && device_.idle();
        if (!keep) device_.free(p);
        if (!b.p) return;
        std::lock_guard<std::mutex> hold(lock_);
        --returning_;
        if (!keep) return;
        b.since = device_.now();
        kept_.push_back(b);
        give_back(b.device, kKeptMost);
    }

    void release() {
        std::lock_guard<std::mutex> hold(lock_);
        give_back(-1, 0);
    }

    Device &device() { return device_; }

  private:
    struct Block {
        void *p;
        size_t bytes;
        int device;
        double since;  // when it was returned
    };

    // Frees what has been kept too long, the longest unused while more than `most` bytes are kept on `device`, and, for
    // device < 0, everything.
    void give_back(int device, size_t most) {
        const double now = device_.now();
        size_t total = 0;
        for (const Block &b : kept_)
            if (b.device == device) total += b.bytes;
        for (size_t k = 0; k < kept_.size();) {  // (in the order they were returned)
            const Block b = kept_[k];
            if (now - b.since <= kKeptSeconds && device >= 0 && !(b.device == device && total > most)) {
                ++k;
                continue;
            }
            if (b.device == device) total -= b.bytes;
            device_.free(b.p);
            kept_.erase(kept_.begin() + (long)k);
        }
    }

    // Both lists have a place for every block there is and one more, so that no other push_back allocates.
    bool room_for_one() {
        const size_t blocks = kept_.size() + in_use_.size() + returning_ + 1;
        try {
            if (kept_.capacity() < blocks) kept_.reserve(2 * blocks);
            if (in_use_.capacity() < blocks) in_use_.reserve(2 * blocks);
        } catch (const std::bad_alloc &) {
            return false;
        }
        return true;
    }

    Device device_;
    std::mutex lock_;
    std::vector<Block> kept_, in_use_;
    size_t returning_ = 0;  // blocks in neither list, on their way from one to the other
};

}  // namespace tsnehip

#endif  // TSNE_HIP_SCRATCH_POOL_H_
