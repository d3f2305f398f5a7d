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
#include <unordered_map>
#include <vector>

#include "plb_internal.hpp"

namespace plb {

constexpr size_t MB = (size_t)1 << 20;
constexpr size_t KEEP_FROM = MB, KEEP_TO = 128 * MB, KEEP_MOST = 256 * MB;

struct Block {
    void* p;
    size_t size;
    int device;
};
// Never destroyed: owners may outlive static objects.
struct Pool {
    std::mutex mutex;
    std::vector<Block> kept;                   // oldest first
    std::unordered_map<void*, Block> live;
    size_t kept_bytes = 0;
};
static Pool& pool()
{
    static Pool* const p = new Pool();
    return *p;
}

void dev_give_back()
{
    Pool& o = pool();
    std::vector<Block> gone;
    {
        std::lock_guard<std::mutex> lock(o.mutex);
        gone.swap(o.kept);
        o.kept_bytes = 0;
    }
    for (const Block& b : gone) (void)hipFree(b.p);
}

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
        std::vector<Block>& kept = o.kept;
        size_t best = kept.size();
        for (size_t k = 0; k < kept.size(); k++)
            if (kept[k].device == b.device && kept[k].size >= b.size && kept[k].size <= b.size + b.size / 2 &&
                (best == kept.size() || kept[k].size < kept[best].size))
                best = k;
        if (best < kept.size()) {
            b = kept[best];
            kept.erase(kept.begin() + best);
            o.kept_bytes -= b.size;
        }
    }
    if (!b.p) {
        e = dev_malloc(&b.p, b.size);
        if (e != hipSuccess) return e;
    }
    std::lock_guard<std::mutex> lock(o.mutex);
    o.live[b.p] = b;
    *p = b.p;
    return hipSuccess;
}

void dev_free(void* p)
{
    if (!p) return;
    Pool& o = pool();
    std::vector<Block> gone;
    {
        std::lock_guard<std::mutex> lock(o.mutex);
        const auto it = o.live.find(p);
        if (it == o.live.end()) {
            gone.push_back({p, 0, 0});
        } else {
            o.kept.push_back(it->second);
            o.kept_bytes += it->second.size;
            o.live.erase(it);
            while (o.kept_bytes > KEEP_MOST) {
                o.kept_bytes -= o.kept.front().size;
                gone.push_back(o.kept.front());
                o.kept.erase(o.kept.begin());
            }
        }
    }
    for (const Block& b : gone) (void)hipFree(b.p);
}

}  // namespace plb
