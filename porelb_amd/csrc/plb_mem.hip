// plb_mem.hip -- device memory of middle size, kept for the next owner.
//
// Allocating a block of tens of MB maps it (9 us per MB: 270 us for 30 MB) and
// releasing it after use costs more (900 us for 60 MB), which for a sample of
// 265 421 nodes was 3.6 ms of a 16 ms study.  Blocks of 1 to 128 MB that are
// released are therefore kept, up to KEEP_MOST in the process, the oldest
// leaving first, and go to the next owner of about that size on that device.
// They are given back when an allocation of the library does not succeed, as soon as newer ones
// take their room, and by plb_release_memory.  (Not with the last context: programs
// that make one lattice after another would lose most of the gain, 9.5 -> 12.8 ms
// for a study of that sample, 45.1 -> 48.1 for one of 1.4 M FP64 nodes.)  Whoever releases a block has waited for the work that
// uses it: a block may serve another stream or thread the moment it is released.
#include <algorithm>
#include <mutex>
#include <new>
#include <unordered_map>

#include "plb_internal.hpp"

namespace plb {

constexpr size_t MB = (size_t)1 << 20;
constexpr size_t KEEP_FROM = MB, KEEP_TO = 128 * MB, KEEP_MOST = 256 * MB;
constexpr int BLOCKS_MOST = KEEP_MOST / KEEP_FROM + 1;   // with the one that takes the others' room

struct Block {
    void* p;
    size_t size;
    int device;
};
struct Pool {
    std::mutex mutex;
    Block kept[BLOCKS_MOST];                   // oldest first
    int n = 0;
    size_t kept_bytes = 0;
    std::unordered_map<void*, Block> live;

    Block take(int k)
    {
        const Block b = kept[k];
        std::move(kept + k + 1, kept + n, kept + k);
        n--;
        kept_bytes -= b.size;
        return b;
    }
};
// Never destroyed: owners may outlive static objects.
static Pool& pool()
{
    alignas(Pool) static char place[sizeof(Pool)];
    static Pool* const p = new (place) Pool();
    return *p;
}

// Frees the oldest blocks until no more than `most` bytes are kept.
static void give_back(size_t most)
{
    Pool& o = pool();
    for (;;) {
        Block b;
        {
            std::lock_guard<std::mutex> lock(o.mutex);
            if (o.kept_bytes <= most) return;
            b = o.take(0);
        }
        (void)hipFree(b.p);
    }
}

void dev_give_back() { give_back(0); }

hipError_t dev_malloc(void** p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipErrorOutOfMemory) return e;
    (void)hipGetLastError();
    dev_give_back();
    return hipMalloc(p, bytes);
}

hipError_t dev_alloc(void** p, size_t bytes)
{
    if (bytes < KEEP_FROM || bytes > KEEP_TO) return dev_malloc(p, bytes);
    Block b = {nullptr, (bytes + MB - 1) / MB * MB, 0};
    hipError_t e = hipGetDevice(&b.device);
    if (e != hipSuccess) return e;
    Pool& o = pool();
    {
        std::lock_guard<std::mutex> lock(o.mutex);
        int best = -1;
        for (int k = 0; k < o.n; k++)
            if (o.kept[k].device == b.device && o.kept[k].size >= b.size && o.kept[k].size <= b.size + b.size / 2 &&
                (best < 0 || o.kept[k].size < o.kept[best].size))
                best = k;
        if (best >= 0) b = o.take(best);
    }
    if (!b.p) {
        e = dev_malloc(&b.p, b.size);
        if (e != hipSuccess) return e;
    }
    try {
        std::lock_guard<std::mutex> lock(o.mutex);
        o.live[b.p] = b;
    } catch (const std::bad_alloc&) {
        (void)hipFree(b.p);
        return hipErrorOutOfMemory;
    }
    *p = b.p;
    return hipSuccess;
}

void dev_free(void* p)
{
    if (!p) return;
    Pool& o = pool();
    bool known;
    {
        std::lock_guard<std::mutex> lock(o.mutex);
        const auto it = o.live.find(p);
        known = it != o.live.end() && o.n < BLOCKS_MOST;
        if (known) {
            o.kept[o.n++] = it->second;
            o.kept_bytes += it->second.size;
        }
        if (it != o.live.end()) o.live.erase(it);
    }
    if (known) give_back(KEEP_MOST);
    else (void)hipFree(p);
}

}  // namespace plb
