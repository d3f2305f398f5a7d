// plb_xfer.hip -- the copies between the caller's arrays and device layouts.
//
// Into and out of page-locked memory the copy engine moves long passes at the
// PCIe rate (53 GB/s).  Pageable memory it reaches only through the runtime's own
// staging: 17 GB/s, and 7 GB/s into memory that was never touched, because one
// thread takes all the page faults.  Such reads go through page-locked slots
// here, and a few threads move each slot on, so the faults and the copies are
// shared; writes go the other way.  The engine fills the slots of a read-back; a
// write's slots are read by the kernel itself, since for 60 ms after the engine
// has read such slots it writes page-locked memory at 28 GB/s instead of 54.
// (Kernels on page-locked arrays otherwise: 54 GB/s for separate components, as
// plb_read_macros has it; 24 and 4 GB/s for writes and reads of whole states,
// whose 152-byte rows reach the bus in pieces; records 1.1 times slower.)
//
// The slots are kept from call to call (a page-locked allocation costs 140 us,
// a 16 MB device allocation and its release 45 us), at most MAX_KEPT sets in
// the process, and are given back with the last context.  A call has a set to
// itself; a call that finds none free uses one of its own.
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <functional>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "plb_xfer.hpp"

namespace plb {

constexpr size_t SLOT = (size_t)4 << 20;
constexpr int SLOTS = 4;
constexpr size_t LONG_PASS = (size_t)64 << 20;
constexpr int MAX_KEPT = 4;
constexpr int MAX_THREADS = 8;
// From here a pageable copy is worth the threads (a thread starts in about 15 us),
// and without a context the slots, which then last for one call only (250 us:
// records of 54 000 nodes, 8 MB, 0.96 ms with them and 0.86 without).
constexpr size_t THREADED = (size_t)3 << 20, THREADED_ALONE = 4 * THREADED;

struct Staging {
    int device = 0;
    char *host = nullptr, *dev = nullptr;
    hipEvent_t copied[SLOTS] = {};
    bool busy = true;
};

struct Kept {
    std::mutex mutex;
    Staging* pool[MAX_KEPT];
    int n = 0;
    int contexts = 0;
};
// Never destroyed: a context may outlive static objects.
static Kept& kept()
{
    alignas(Kept) static char place[sizeof(Kept)];
    static Kept* const k = new (place) Kept();
    return *k;
}

static void staging_free(Staging* s)
{
    if (!s) return;
    int current = s->device;   // the caller's, which stays
    (void)hipGetDevice(&current);
    (void)hipSetDevice(s->device);
    if (s->host) (void)hipHostFree(s->host);
    dev_free(s->dev);
    for (hipEvent_t e : s->copied)
        if (e) (void)hipEventDestroy(e);
    (void)hipSetDevice(current);
    delete s;
}

// Frees the sets that no call uses.
static void free_idle()
{
    Kept& o = kept();
    for (;;) {
        Staging* gone;
        {
            std::lock_guard<std::mutex> lock(o.mutex);
            Staging** const idle = std::find_if(o.pool, o.pool + o.n, [](Staging* s) { return !s->busy; });
            if (idle == o.pool + o.n) return;
            gone = *idle;
            *idle = o.pool[--o.n];
        }
        staging_free(gone);
    }
}

void xfer_context(int add)
{
    {
        std::lock_guard<std::mutex> lock(kept().mutex);
        kept().contexts += add;
        if (kept().contexts > 0) return;
    }
    free_idle();
}

static bool slots_are_kept()
{
    std::lock_guard<std::mutex> lock(kept().mutex);
    return kept().contexts > 0;
}

static hipError_t staging_new(int device, Staging** out)
{
    Staging* s = new (std::nothrow) Staging();
    if (!s) return hipErrorOutOfMemory;
    s->device = device;
    hipError_t e = hipHostMalloc((void**)&s->host, SLOT * SLOTS, hipHostMallocCoherent);
    if (e == hipSuccess) e = dev_alloc((void**)&s->dev, SLOT * SLOTS);
    for (int k = 0; k < SLOTS && e == hipSuccess; k++) e = hipEventCreateWithFlags(&s->copied[k], hipEventDisableTiming);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        staging_free(s);
        return e;
    }
    *out = s;
    return hipSuccess;
}

// A set of slots on the current device for one call.
struct Lease {
    Staging* s = nullptr;
    hipError_t take(int device)
    {
        Kept& o = kept();
        {
            std::lock_guard<std::mutex> lock(o.mutex);
            for (int k = 0; k < o.n; k++)
                if (!o.pool[k]->busy && o.pool[k]->device == device) {
                    s = o.pool[k];
                    s->busy = true;
                    return hipSuccess;
                }
        }
        const hipError_t e = staging_new(device, &s);
        if (e != hipSuccess) return e;
        std::lock_guard<std::mutex> lock(o.mutex);
        if (o.n < MAX_KEPT) o.pool[o.n++] = s;
        return hipSuccess;
    }
    ~Lease()
    {
        if (!s) return;
        Kept& o = kept();
        Staging* gone = s;
        {
            std::lock_guard<std::mutex> lock(o.mutex);
            s->busy = false;
            Staging** const it = std::find(o.pool, o.pool + o.n, s);
            if (it != o.pool + o.n) {
                if (o.contexts > 0) gone = nullptr;
                else *it = o.pool[--o.n];
            }
        }
        staging_free(gone);
    }
};

// What the runtime knows of p; pageable memory it does not know.
static hipPointerAttribute_t attributes(const void* p)
{
    hipPointerAttribute_t a = {};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        a = {};
        a.type = hipMemoryTypeUnregistered;
    }
    return a;
}

bool page_locked(const void* p)
{
    const hipPointerAttribute_t a = attributes(p);
    return a.type == hipMemoryTypeHost && a.devicePointer == a.hostPointer;  // kernels take the pointer as it is
}

// Threads that run work(chunk, thread, threads) for every chunk that is posted.
class Team {
public:
    Team(int threads, int64_t chunks, std::function<void(int64_t, int, int)> work) : done_(chunks)
    {
        for (int64_t k = 0; k < chunks; k++) done_[k] = 0;
        try {
            for (int t = 0; t < threads; t++) {
                members_.emplace_back([this, t, threads, chunks, work] {
                    for (int64_t k = 0; k < chunks; k++) {
                        while (posted_.load(std::memory_order_acquire) <= k) {
                            if (stop_.load(std::memory_order_relaxed)) return;
                            std::this_thread::yield();
                        }
                        work(k, t, threads);
                        done_[k].fetch_add(1, std::memory_order_release);
                    }
                });
            }
        } catch (...) {  // no more threads to be had
            ok_ = false;
        }
    }
    ~Team()
    {
        stop_ = true;
        for (std::thread& m : members_) m.join();
    }
    bool ok() const { return ok_; }
    void post(int64_t upto) { posted_.store(upto, std::memory_order_release); }
    void wait(int64_t k) const
    {
        while (done_[k].load(std::memory_order_acquire) < (int)members_.size()) std::this_thread::yield();
    }

private:
    std::vector<std::thread> members_;
    std::vector<std::atomic<int>> done_;
    std::atomic<int64_t> posted_{0};
    std::atomic<bool> stop_{false};
    bool ok_ = true;
};

static int threads_for(size_t bytes)
{
    const int cpus = std::max(1, (int)std::thread::hardware_concurrency() / 2);
    return std::max(1, std::min({MAX_THREADS, cpus, (int)(bytes / ((size_t)1 << 20))}));
}

// Both directions: chunks of m nodes, parts of `item` bytes per node, laid out
// [part][m] in a slot and [part][n] at the caller (arrays[part]).  Kernels and
// copies share the caller's stream: a copy stream of its own gained nothing
// over its events (9.2 -> 12.2 ms for 382 MB of FP32 state).
static int move(int device, hipStream_t s, int64_t n, size_t item, const Arrays& arrays, bool to_device,
                const ChunkKernel& kernel)
{
    const size_t row = item * arrays.n, bytes = row * (size_t)n;
    if (bytes == 0) return PLB_OK;
    // Threads move host memory, if any of it is pageable; device and managed memory is left to the runtime's copies.
    bool host = true, locked = true;
    for (size_t p = 0; p < arrays.n; p++) {
        const hipMemoryType type = attributes(arrays.at[p]).type;
        locked = locked && type == hipMemoryTypeHost;
        host = host && (type == hipMemoryTypeHost || type == hipMemoryTypeUnregistered);
    }
    Lease lease;
    bool threaded = host && !locked && bytes >= (slots_are_kept() ? THREADED : THREADED_ALONE);
    if (threaded && lease.take(device) != hipSuccess) threaded = false;

    int rc = PLB_OK;
    auto check = [&](hipError_t e) {
        if (e == hipSuccess) return true;
        plb_set_hip_error(e, "copy between host and device", __FILE__, __LINE__);
        rc = PLB_ERR_HIP;
        return false;
    };
    // the kernel and the copies of m nodes from `first` on, in stream order
    auto transfer = [&](int64_t first, int64_t m, char* dev) {
        if (!to_device && (rc = kernel(first, m, dev))) return false;
        for (size_t p = 0; p < arrays.n; p++) {
            char* const mine = arrays.at[p] + (size_t)first * item;
            char* const part = dev + (size_t)m * p * item;
            if (!check(to_device ? hipMemcpyAsync(part, mine, m * item, hipMemcpyHostToDevice, s)
                                 : hipMemcpyAsync(mine, part, m * item, hipMemcpyDeviceToHost, s)))
                return false;
        }
        return !to_device || (rc = kernel(first, m, dev)) == PLB_OK;
    };
    auto whole_words = [&](size_t room) { return std::max<int64_t>(1, (int64_t)(room / row) & ~(int64_t)63); };

    std::unique_ptr<Team> team;
    const int64_t per = whole_words(SLOT), chunks = (n + per - 1) / per;
    if (threaded) {
        // slice t of T of every part of a chunk, between its host slot and the caller
        team.reset(new Team(threads_for(bytes), chunks, [&](int64_t k, int t, int T) {
            const int64_t first = k * per, m = std::min(per, n - first);
            const int64_t a = m * t / T, b = m * (t + 1) / T;
            for (size_t p = 0; p < arrays.n; p++) {
                char* const mine = arrays.at[p] + (size_t)(first + a) * item;
                char* const staged = lease.s->host + SLOT * (k % SLOTS) + ((size_t)m * p + a) * item;
                if (to_device) memcpy(staged, mine, (size_t)(b - a) * item);
                else memcpy(mine, staged, (size_t)(b - a) * item);
            }
        }));
        threaded = team->ok();
    }
    if (!threaded) {
        // One long copy per array and pass: the copy engine reaches its rate
        // from a few MB on.
        char* room = nullptr;
        size_t have = std::min(bytes + 64 * row, LONG_PASS);
        hipError_t got = dev_alloc((void**)&room, have);
        while (got != hipSuccess && have > SLOT) {  // little memory left: shorter passes
            (void)hipGetLastError();
            got = dev_alloc((void**)&room, have = std::max(SLOT, have / 4));
        }
        PLB_HIP(got);
        const int64_t pass = whole_words(have);
        for (int64_t first = 0; first < n && !rc; first += pass) transfer(first, std::min(pass, n - first), room);
        const hipError_t e = hipStreamSynchronize(s);
        dev_free(room);
        if (!rc) check(e);
        return rc;
    }
    Staging& st = *lease.s;
    auto chunk = [&](int64_t k) {
        const size_t at = SLOT * (k % SLOTS);
        const int64_t m = std::min(per, n - k * per);
        rc = kernel(k * per, m, to_device ? st.host + at : st.dev + at);
        if (rc || (!to_device && !check(hipMemcpyAsync(st.host + at, st.dev + at, row * m, hipMemcpyDeviceToHost, s))))
            return false;
        return check(hipEventRecord(st.copied[k % SLOTS], s));
    };
    if (to_device) {
        team->post(std::min<int64_t>(chunks, SLOTS));
        for (int64_t k = 0; k < chunks; k++) {
            team->wait(k);
            if (!chunk(k)) break;
            // a host slot is filled again once its copy is through; by now the next one is on its way
            if (k > 0 && k - 1 + SLOTS < chunks) {
                if (!check(hipEventSynchronize(st.copied[(k - 1) % SLOTS]))) break;
                team->post(k + SLOTS);
            }
        }
    } else {
        int64_t issued = 0;
        for (int64_t k = 0; k < chunks && !rc; k++) {
            for (; issued < chunks && issued < k + SLOTS && !rc; issued++) {
                if (issued >= SLOTS) team->wait(issued - SLOTS);
                chunk(issued);
            }
            if (rc || !check(hipEventSynchronize(st.copied[k % SLOTS]))) break;
            team->post(k + 1);
        }
        if (!rc)
            for (int64_t k = std::max<int64_t>(0, chunks - SLOTS); k < chunks; k++) team->wait(k);
    }
    const hipError_t e = hipStreamSynchronize(s);  // the slots are free again, also after an error
    if (!rc) check(e);
    return rc;
}

extern "C" void plb_release_memory(void)
{
    free_idle();
    dev_give_back();
}

int download(int device, hipStream_t s, int64_t n, size_t item, const Arrays& arrays, const ChunkKernel& kernel)
{
    return guarded([&] { return move(device, s, n, item, arrays, false, kernel); });
}

int upload(int device, hipStream_t s, int64_t n, size_t item, const void* array, const ChunkKernel& kernel)
{
    return guarded([&] { return move(device, s, n, item, Arrays((void*)array), true, kernel); });
}

}  // namespace plb
