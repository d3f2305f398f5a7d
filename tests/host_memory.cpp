// The transfer slots and the kept device blocks (plb_xfer.hip, plb_mem.hip) on a
// HIP runtime made of malloc: two devices, immediate copies.  Built and run by
// tests/test_host_memory.py under the address sanitizer; argv[1] names the check.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <vector>

#include "plb_xfer.hpp"

static int current = 0, fails = 0;
static size_t on_device = 0, locked_bytes = 0, capacity = ~(size_t)0;
static std::map<void*, size_t>* sizes = new std::map<void*, size_t>();   // outlives every static object

#define CHECK(c)                                                               \
    do {                                                                       \
        if (!(c)) {                                                            \
            fprintf(stderr, "check failed: %s (line %d)\n", #c, __LINE__);     \
            fails++;                                                           \
        }                                                                      \
    } while (0)

extern "C" {
hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n)
{
    if (n > capacity || on_device > capacity - n) return hipErrorOutOfMemory;
    *p = malloc(n);
    (*sizes)[*p] = n;
    on_device += n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    on_device -= (*sizes)[p];
    sizes->erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { locked_bytes += n; (*sizes)[*p = malloc(n)] = n; return hipSuccess; }
hipError_t hipHostFree(void* p) { locked_bytes -= (*sizes)[p]; sizes->erase(p); free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return hipErrorInvalidValue; }
const char* hipGetErrorString(hipError_t) { return ""; }
}
void plb_set_hip_error(hipError_t, const char*, const char*, int) {}

using namespace plb;

constexpr size_t MB = (size_t)1 << 20;

static void transfer(int device)
{
    std::vector<char> array(8 * MB);
    hipSetDevice(device);
    CHECK(download(device, nullptr, (int64_t)array.size(), 1, Arrays(array.data()), [](int64_t, int64_t m, void* d) {
              memset(d, 7, m);
              return PLB_OK;
          }) == PLB_OK);
    CHECK(array.front() == 7 && array.back() == 7);
}

// The slots of another device go without a change of the caller's current one.
static void device()
{
    xfer_context(1);
    xfer_context(1);
    transfer(0);
    transfer(1);
    CHECK(locked_bytes == 32 * MB);
    for (int left : {1, 0}) {
        hipSetDevice(0);
        xfer_context(-1);
        CHECK(current == 0);
        CHECK(locked_bytes == (left ? 32 * MB : 0));
    }
    // a set that lasts for one call
    transfer(0);
    CHECK(current == 0 && locked_bytes == 0);
}

// Kept blocks: 256 MB at most, for the next owner, and back to the system on request or when there is no more.
static void release()
{
    std::vector<void*> p(10);
    for (void*& q : p) CHECK(dev_alloc(&q, 64 * MB) == hipSuccess);
    CHECK(on_device == 640 * MB);
    for (void* q : p) dev_free(q);
    CHECK(on_device == 256 * MB);
    CHECK(dev_alloc(&p[0], 50 * MB) == hipSuccess && on_device == 256 * MB);
    plb_release_memory();
    CHECK(on_device == 64 * MB);   // the one in use
    dev_free(p[0]);
    CHECK(on_device == 64 * MB);
    capacity = 100 * MB;
    CHECK(dev_alloc(&p[0], 80 * MB) == hipSuccess && on_device == 80 * MB);
    CHECK(dev_alloc(&p[1], 80 * MB) == hipErrorOutOfMemory);
    dev_free(p[0]);
    plb_release_memory();
    CHECK(on_device == 0);
    capacity = ~(size_t)0;
    xfer_context(1);
    transfer(1);
    CHECK(locked_bytes == 16 * MB);
    plb_release_memory();
    CHECK(locked_bytes == 0 && on_device == 0);
    transfer(1);
    CHECK(locked_bytes == 16 * MB);
    xfer_context(-1);
    CHECK(locked_bytes == 0);
    plb_release_memory();
    CHECK(on_device == 0);
}

// Kept blocks make room for every allocation of the library, also those that are not blocks of that kind.
static void room()
{
    void* p = nullptr;
    CHECK(dev_alloc(&p, 80 * MB) == hipSuccess);
    dev_free(p);
    CHECK(on_device == 80 * MB);
    capacity = 100 * MB;
    {
        DevBuf<char> b;
        CHECK(b.alloc(60 * MB) == hipSuccess && on_device == 60 * MB);
    }
    CHECK(dev_alloc(&p, 80 * MB) == hipSuccess);
    dev_free(p);
    Arena a;
    CHECK(a.take(&p, (size_t)1000) == hipSuccess && on_device < 81 * MB);
    DevBuf<char> b;
    CHECK(b.alloc(99 * MB) == hipSuccess && on_device < 100 * MB);
}

// An object of the caller's with static storage may go after the library's own static objects.
struct Late {
    std::vector<void*> blocks;
    bool counted = false;
    ~Late()
    {
        if (!counted) return;
        for (void* p : blocks) dev_free(p);
        void* p = nullptr;
        if (dev_alloc(&p, 3 * MB) == hipSuccess) dev_free(p);
        transfer(0);
        xfer_context(-1);
        if (fails) _Exit(1);
    }
};
static Late late;   // made before the library's static objects: its source comes first on the command line

static void at_exit()
{
    xfer_context(1);
    transfer(0);
    late.counted = true;
    late.blocks.resize(5);
    for (void*& p : late.blocks) CHECK(dev_alloc(&p, 2 * MB) == hipSuccess);
    dev_free(late.blocks.back());
    late.blocks.pop_back();
}

int main(int argc, char** argv)
{
    const char* what = argc > 1 ? argv[1] : "";
    if (!strcmp(what, "device")) device();
    else if (!strcmp(what, "release")) release();
    else if (!strcmp(what, "room")) room();
    else if (!strcmp(what, "at_exit")) at_exit();
    else return 2;
    return fails ? 1 : 0;
}
