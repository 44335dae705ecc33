"""The device scratch kept between calls (csrc/scratch_pool.h), compiled for the host with an allocator of limited size and a
clock of its own."""
import glob
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tsne-cuda_amd", "csrc")

PROGRAM = r"""
#include "scratch_pool.h"
#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>

static bool out_of_host_memory = false;
void *operator new(size_t bytes) {
    void *p = out_of_host_memory ? nullptr : std::malloc(bytes);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

#define EXPECT(what)                                                       \
    do {                                                                   \
        if (!(what)) {                                                     \
            std::fprintf(stderr, "line %d: %s\n", __LINE__, #what);        \
            std::exit(1);                                                  \
        }                                                                  \
    } while (0)

struct World {
    size_t room[2] = {(size_t)8 << 30, (size_t)8 << 30};
    std::map<void *, std::pair<size_t, int>> live;
    int here = 0, waits = 0, errors = 0;
    bool known = true, waits_well = true;
    double clock = 0.0;
    char *next = reinterpret_cast<char *>(4096);
    void (*meanwhile)(void *) = nullptr;  // what another thread does while this one asks for its device
    void *with = nullptr;
};
struct Device {
    World *w;
    int alloc(void **p, size_t bytes) {
        *p = nullptr;
        if (bytes > w->room[w->here]) {
            ++w->errors;
            return 2;
        }
        w->room[w->here] -= bytes;
        const bool fails = out_of_host_memory;
        out_of_host_memory = false;
        w->live[w->next] = {bytes, w->here};
        out_of_host_memory = fails;
        *p = w->next;
        w->next += 4096;
        return 0;
    }
    void forgive() { w->errors = 0; }
    void free(void *p) {
        EXPECT(w->live.count(p));
        w->room[w->live[p].second] += w->live[p].first;
        w->live.erase(p);
    }
    int current() {
        if (w->meanwhile) {
            auto act = w->meanwhile;
            w->meanwhile = nullptr;
            act(w->with);
        }
        return w->known ? w->here : -1;
    }
    bool idle() {
        ++w->waits;
        return w->waits_well;
    }
    double now() { return w->clock; }
};
using Pool = tsnehip::ScratchPool<Device>;
constexpr size_t MB = (size_t)1 << 20, GB = (size_t)1 << 30;

int main() {
    const size_t least = tsnehip::kKeptLeast;
    {  // taken again by what needs about as much; small blocks and blocks of an unknown device are not kept
        World w;
        Pool pool(Device{&w});
        void *a, *b, *c;
        EXPECT(!pool.take(&a, 300 * MB) && !pool.take(&b, least - 1));
        pool.put(a), pool.put(b), pool.put(nullptr);
        EXPECT(w.live.size() == 1 && w.waits == 1);
        EXPECT(!pool.take(&b, 301 * MB) && b != a);   // too small
        EXPECT(!pool.take(&c, 190 * MB) && c != a);   // more than half as large again
        pool.put(b);
        EXPECT(!pool.take(&b, 210 * MB) && b == a);   // the smallest that does
        void *d;
        EXPECT(!pool.take(&d, 0) && d);
        for (void *p : {b, c, d}) pool.put(p);
        pool.release();
        EXPECT(w.live.empty() && w.room[0] == 8 * GB);
        w.known = false;
        EXPECT(!pool.take(&a, 300 * MB) && w.live.size() == 1);
        pool.put(a);
        EXPECT(w.live.empty());
    }
    {  // bounded: the longest unused goes first; and what is kept too long goes at the next call
        World w;
        Pool pool(Device{&w});
        void *p[5], *q;
        for (int k = 0; k < 5; ++k) EXPECT(!pool.take(&p[k], (600 + 100 * k) * MB));
        for (int k = 0; k < 5; ++k) w.clock += 0.1, pool.put(p[k]);
        size_t kept = 0;
        for (auto &b : w.live) kept += b.second.first;
        EXPECT(kept <= tsnehip::kKeptMost && w.live.count(p[4]) && w.live.count(p[3]) && !w.live.count(p[0]));
        w.clock += tsnehip::kKeptSeconds - 0.05;
        EXPECT(!pool.take(&q, 100 * MB));
        EXPECT(w.live.count(p[4]) && !w.live.count(p[3]));
        pool.put(q);
        w.clock += tsnehip::kKeptSeconds + 0.05;
        EXPECT(!pool.take(&q, 3 * GB) && w.live.size() == 1);
        pool.put(q);  // more than is ever kept
        EXPECT(w.live.empty());
    }
    {  // no room: kept memory of that device goes first, for large blocks, small ones and those that are never kept
        for (size_t bytes : {least, (size_t)4096, 600 * MB})
            for (bool scratch : {true, false}) {
                World w;
                w.room[0] = 1 * GB;
                Pool pool(Device{&w});
                void *a, *far, *b;
                w.here = 1;
                EXPECT(!pool.take(&far, 500 * MB));
                pool.put(far);
                w.here = 0;
                EXPECT(!pool.take(&a, 1 * GB));
                pool.put(a);
                EXPECT(w.room[0] == 0);
                EXPECT(!(scratch ? pool.take(&b, bytes) : pool.plain(&b, bytes)));
                EXPECT(w.errors == 0 && !w.live.count(a) && w.live.count(far) && w.room[0] == 1 * GB - bytes);
                void *c;
                EXPECT((scratch ? pool.take(&c, 2 * GB) : pool.plain(&c, 2 * GB)) == 2 && !c && w.errors);
            }
    }
    {  // ... also where another thread gives it, just after this one found none
        World w;
        w.room[0] = 1 * GB;
        Pool pool(Device{&w});
        void *a, *b;
        EXPECT(!pool.take(&a, 1 * GB));
        pool.put(a);
        w.with = &pool;
        w.meanwhile = [](void *p) { static_cast<Pool *>(p)->release(); };
        EXPECT(!pool.plain(&b, 4096) && w.errors == 0);
    }
    {  // returned from another device, or while the device cannot be waited for: freed
        World w;
        Pool pool(Device{&w});
        void *a, *b;
        EXPECT(!pool.take(&a, 100 * MB) && !pool.take(&b, 100 * MB));
        w.here = 1;
        pool.put(a);
        w.here = 0;
        w.waits_well = false;
        pool.put(b);
        EXPECT(w.live.empty());
    }
    {  // no host memory for the records: nothing is thrown, nothing lost
        World w;
        Pool pool(Device{&w});
        void *a, *b;
        out_of_host_memory = true;
        const int e = pool.take(&a, 100 * MB);
        out_of_host_memory = false;
        EXPECT(!e && a);
        EXPECT(!pool.take(&b, 100 * MB));
        out_of_host_memory = true;
        pool.put(b), pool.put(a);
        out_of_host_memory = false;
        EXPECT(w.live.size() == 1 && w.live.count(b));
        pool.release();
        EXPECT(w.live.empty());
    }
    return 0;
}
"""


def test_kept_scratch_is_bounded_and_given_back(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    source, program = tmp_path / "pool.cpp", tmp_path / "pool"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D_GLIBCXX_ASSERTIONS", "-I", CSRC, str(source), "-o",
                    str(program)], check=True)
    env = {k: v for k, v in os.environ.items() if k != "LD_PRELOAD"}
    done = subprocess.run([str(program)], env=env, capture_output=True)
    assert done.returncode == 0, done.stderr.decode()[-2000:]


def test_everything_is_allocated_through_the_pool():
    """An allocation that does not know of the kept memory fails while that lies idle."""
    for path in glob.glob(os.path.join(CSRC, "*")):
        with open(path) as f:
            calls = re.findall(r"\bhipMalloc\w*\(", f.read())
        assert calls == (["hipMalloc("] if os.path.basename(path) == "scratch.hip" else []), path
