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
// 1 GiB gave back and took again each time, 0.34 of 4.3 ms).
// cudaBVH_resetDevice gives them back, and so does every device allocation of
// the library that finds no memory (dev_plain). Smaller blocks cost under 3 us
// and go to the runtime directly.
//
// A block is handed out again only when no device work uses it any longer: the
// caller has waited for that work (dev_free), or the block is pending
// (dev_release) until its device has been waited for, which the next
// allocation that could take it does. So a later owner may use it on any
// stream. Blocks leave the cache through hipFree, which waits by itself.
#include <hip/hip_runtime.h>

#include <list>
#include <mutex>
#include <unordered_map>

#include "rt_internal.h"

namespace rt {

namespace {
constexpr size_t kCacheMin = size_t(1) << 20, kCacheMax = size_t(2) << 30;

// seq: number of the release after which it has not been waited for (0: idle)
struct Block { void* p; size_t bytes; int device; unsigned long long seq; };
struct Cache {
    std::mutex mu;
    std::list<Block> free;                          // oldest first
    size_t freeBytes = 0;
    unsigned long long releases = 0;
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

// hipMalloc whose failure leaves no error behind for a later launch check.
void* raw_alloc(size_t bytes) {
    void* p = nullptr;
    if (hipMalloc(&p, bytes) == hipSuccess) return p;
    (void)hipGetLastError();
    return nullptr;
}

// Frees blocks taken out of the cache; those that cannot be freed now (a stream
// capture that forbids it) go back as pending.
void give_back(std::list<Block>& out) {
    for (auto it = out.begin(); it != out.end();) {
        if (hipFree(it->p) == hipSuccess) { it = out.erase(it); continue; }
        (void)hipGetLastError();
        ++it;
    }
    if (out.empty()) return;
    Cache& c = cache();
    std::lock_guard<std::mutex> g(c.mu);
    for (Block& b : out) { b.seq = ++c.releases; c.freeBytes += b.bytes; }
    c.free.splice(c.free.begin(), out);
}

// Waits for all work of the current device as hipFree does, by freeing a block.
// (hipDeviceSynchronize ends a capture in relaxed mode on any thread; this does
// not, and still waits.) False where it cannot wait.
bool wait_device() {
    void* p = raw_alloc(1);
    if (p && hipFree(p) == hipSuccess) return true;
    if (p) (void)hipGetLastError();
    return false;
}

// The smallest cached block of device dev that serves need bytes, idle or pending.
std::list<Block>::iterator best_fit(Cache& c, int dev, size_t need, bool idle) {
    auto best = c.free.end();
    for (auto it = c.free.begin(); it != c.free.end(); ++it)
        if (it->device == dev && (it->seq == 0) == idle && it->bytes >= need && it->bytes <= need + need / 4 &&
            (best == c.free.end() || it->bytes < best->bytes))
            best = it;
    return best;
}

void put(void* p, bool idle) {
    if (!p) return;
    Cache& c = cache();
    std::list<Block> out;
    {
        std::lock_guard<std::mutex> g(c.mu);
        auto it = c.live.find(p);
        if (it != c.live.end()) {
            Block b = it->second;
            c.live.erase(it);
            b.seq = idle ? 0 : ++c.releases;
            p = nullptr;
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
    if (p && hipFree(p) != hipSuccess) (void)hipGetLastError();   // a small block
    give_back(out);
}
}  // namespace

void dev_trim() {
    std::list<Block> out;
    {
        std::lock_guard<std::mutex> g(cache().mu);
        out.swap(cache().free);
        cache().freeBytes = 0;
    }
    give_back(out);
}

void* dev_plain(size_t bytes) {
    if (bytes == 0) bytes = 1;
    void* p = raw_alloc(bytes);
    if (!p) {
        dev_trim();
        p = raw_alloc(bytes);
    }
    return p;
}

void* dev_alloc(size_t bytes) {
    if (bytes < kCacheMin) return dev_plain(bytes);
    const size_t need = rounded(bytes);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    Cache& c = cache();
    {
        std::unique_lock<std::mutex> g(c.mu);
        auto it = best_fit(c, dev, need, true);
        if (it == c.free.end() && best_fit(c, dev, need, false) != c.free.end()) {
            // one wait serves every block released before it
            const unsigned long long upTo = c.releases;
            g.unlock();
            const bool waited = wait_device();
            g.lock();
            if (waited) {
                for (Block& b : c.free)
                    if (b.device == dev && b.seq <= upTo) b.seq = 0;
                it = best_fit(c, dev, need, true);
            } else {
                it = c.free.end();
            }
        }
        if (it != c.free.end()) {
            const Block b = *it;
            c.freeBytes -= b.bytes;
            c.free.erase(it);
            c.live.emplace(b.p, b);
            return b.p;
        }
    }
    void* p = dev_plain(need);
    if (!p) return nullptr;
    std::lock_guard<std::mutex> g(c.mu);
    c.live.emplace(p, Block{p, need, dev, 0});
    return p;
}

void dev_free(void* p) { put(p, true); }
void dev_release(void* p) { put(p, false); }

}  // namespace rt
