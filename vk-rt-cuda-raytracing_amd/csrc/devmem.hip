// devmem.hip — device memory of the build and of the traversal stacks, with a
// bounded cache of freed blocks.
//
// Rebuilding a BVH every frame frees and allocates the same few large blocks,
// and each hipFree of a block of tens of megabytes or more costs 70-290 us and
// each hipMalloc 20-90 us (MI355X): 1.9 of the 5.7 ms that a 3.4 M-triangle
// rebuild took. Freed blocks of at least kCacheMin bytes are kept for the next
// allocation of about their size on their device, at most kCacheMax bytes in
// all over the process (the oldest go first; a 3.4 M-triangle scene rebuilt and
// traced every frame holds 1.0 GiB of them between frames, which a bound of
// 1 GiB gave back and took again each time, 0.34 of 4.3 ms); cudaBVH_resetDevice gives them
// back, and so does an allocation that fails. Smaller blocks cost under 3 us
// and go to the runtime directly.
//
// A block enters the cache only when no device work uses it any longer: the
// caller has waited for that work (dev_free), or dev_release waits for the
// device as hipFree does. So a later owner may use it on any stream.
#include <hip/hip_runtime.h>

#include <list>
#include <mutex>
#include <unordered_map>

#include "rt_internal.h"

namespace rt {

namespace {
constexpr size_t kCacheMin = size_t(1) << 20, kCacheMax = size_t(2) << 30;

struct Block { void* p; size_t bytes; int device; };
struct Cache {
    std::mutex mu;
    std::list<Block> free;                          // oldest first
    size_t freeBytes = 0;
    std::unordered_map<void*, Block> live;          // blocks of at least kCacheMin bytes in use
};
// never destroyed: handles may be freed while the process tears down
Cache& cache() {
    static Cache* c = new Cache();
    return *c;
}
size_t rounded(size_t bytes) {
    size_t step = size_t(2) << 20;
    while (step * 16 < bytes) step *= 2;            // at most an eighth over
    return (bytes + step - 1) / step * step;
}
}  // namespace

void dev_trim() {
    std::list<Block> out;
    {
        std::lock_guard<std::mutex> g(cache().mu);
        out.swap(cache().free);
        cache().freeBytes = 0;
    }
    for (const Block& b : out) hipFree(b.p);
}

void* dev_alloc(size_t bytes) {
    void* p = nullptr;
    if (bytes < kCacheMin) {
        if (hipMalloc(&p, bytes ? bytes : 1) == hipSuccess) return p;
        dev_trim();
        return hipMalloc(&p, bytes ? bytes : 1) == hipSuccess ? p : nullptr;
    }
    const size_t need = rounded(bytes);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    Cache& c = cache();
    {
        std::lock_guard<std::mutex> g(c.mu);
        auto best = c.free.end();
        for (auto it = c.free.begin(); it != c.free.end(); ++it)
            if (it->device == dev && it->bytes >= need && it->bytes <= need + need / 4 &&
                (best == c.free.end() || it->bytes < best->bytes))
                best = it;
        if (best != c.free.end()) {
            const Block b = *best;
            c.freeBytes -= b.bytes;
            c.free.erase(best);
            c.live.emplace(b.p, b);
            return b.p;
        }
    }
    if (hipMalloc(&p, need) != hipSuccess) {
        dev_trim();
        if (hipMalloc(&p, need) != hipSuccess) return nullptr;
    }
    std::lock_guard<std::mutex> g(c.mu);
    c.live.emplace(p, Block{p, need, dev});
    return p;
}

void dev_free(void* p) {
    if (!p) return;
    Cache& c = cache();
    std::list<Block> out;
    {
        std::lock_guard<std::mutex> g(c.mu);
        auto it = c.live.find(p);
        if (it == c.live.end()) {
            out.push_back(Block{p, 0, 0});
        } else {
            const Block b = it->second;
            c.live.erase(it);
            if (b.bytes > kCacheMax) {
                out.push_back(b);
            } else {
                c.free.push_back(b);
                c.freeBytes += b.bytes;
                while (c.freeBytes > kCacheMax) {
                    c.freeBytes -= c.free.front().bytes;
                    out.splice(out.end(), c.free, c.free.begin());
                }
            }
        }
    }
    for (const Block& b : out) hipFree(b.p);
}

void dev_release(void* p) {
    if (!p) return;
    hipDeviceSynchronize();
    dev_free(p);
}

}  // namespace rt
