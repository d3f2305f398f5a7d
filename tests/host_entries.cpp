// The C entries that step, read and write, with host memory running out at every
// place where they may ask for some: an error code or success, and no exception.
// Host build on a HIP runtime made of malloc whose kernels do nothing
// (tests/test_host_entries.py).
#include <stdlib.h>

#include <new>

#include "plb_api.hip"
#include "plb_mem.hip"
#include "plb_onchip.hip"
#include "plb_xfer.hip"

static long allowed = -1;   // allocations until they fail; -1: never

static void* take(size_t n)
{
    if (allowed == 0) throw std::bad_alloc();
    if (allowed > 0) allowed--;
    return malloc(n ? n : 1);
}
void* operator new(size_t n) { return take(n); }
void* operator new[](size_t n) { return take(n); }
void operator delete(void* p) noexcept { free(p); }
void operator delete[](void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
void operator delete[](void* p, size_t) noexcept { free(p); }

extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = calloc(n, 1); return hipSuccess; }
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(n, 1); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return hipErrorInvalidValue; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipLaunchCooperativeKernel(const void*, dim3, dim3, void**, unsigned, hipStream_t) { return hipSuccess; }
int roctxRangePushA(const char*) { return 0; }
int roctxRangePop(void) { return 0; }
// There is no device code in this program.
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
}

namespace plb {
StepArgs make_args(plb_ctx*, int64_t, bool) { return StepArgs(); }
int launch_step(plb_ctx* c, int64_t, bool, const int64_t*) { c->cur ^= 1; return PLB_OK; }
int launch_graph_steps(plb_ctx*, int64_t, int64_t) { return PLB_OK; }
int launch_reduce(plb_ctx*) { return PLB_OK; }
int launch_fault_words(plb_ctx*) { return PLB_OK; }
int launch_init_eq(plb_ctx*) { return PLB_OK; }
int launch_read_pop(plb_ctx*, int64_t, int64_t, double*) { return PLB_OK; }
int launch_write_pop(plb_ctx*, int64_t, int64_t, const double*) { return PLB_OK; }
int launch_read_macros(plb_ctx*, const MacroList&, int64_t, int64_t) { return PLB_OK; }
int launch_copy_state(plb_ctx*, int64_t, int64_t, void*, bool) { return PLB_OK; }
int launch_read_table(plb_ctx*, int64_t, int64_t, int32_t*) { return PLB_OK; }
int build_table_from_V(plb_ctx*, const plb_node_info*, int64_t) { return PLB_ERR_INVALID; }
int build_table_from_flag(plb_ctx*, const uint8_t*) { return PLB_ERR_INVALID; }
int build_key_runs(plb_ctx*) { return PLB_OK; }
int noalloc_setup(int) { return PLB_OK; }

static int fails = 0;

// `entry` with 0, 1, 2 .. allocations until it gets through; `again` before each.
template <typename Again, typename Entry>
static void every_place(const char* name, Again again, Entry entry)
{
    int failed = 0;
    for (long n = 0; n < 1000; n++) {
        again();
        allowed = n;
        int rc = 1;
        try {
            rc = entry();
        } catch (...) {
            rc = 2;
        }
        const bool done = allowed != 0 && rc == PLB_OK;
        allowed = -1;
        if (rc != PLB_OK && rc != PLB_ERR_NOMEM) {
            fprintf(stderr, "%s: %s after %ld allocations\n", name, rc == 2 ? "exception" : "wrong code", n);
            fails++;
            return;
        }
        if (done) {
            printf("%s: %ld allocations, %d codes\n", name, n, failed);
            return;
        }
        failed += rc != PLB_OK;
    }
    fprintf(stderr, "%s: never got through\n", name);
    fails++;
}

static int run()
{
    HostWords words = {{NO_FAULT, NO_FAULT}, {0.0, 0.0}};
    plb_ctx c;
    memset(&c.cfg, 0, sizeof c.cfg);
    c.cfg.precision = PLB_FP32;
    c.elem = 4;
    c.lds_per_cu = 160 * 1024;
    c.host = &words;
    c.N = c.Npad = 65536;
    c.nx = c.ny = c.nz = 48;
    c.fault = (unsigned long long*)calloc(2, 8);
    c.segs.reserve(SEGMENTS_MOST);
    std::vector<char> array((size_t)c.N * Q * 8);
    double* const d = (double*)array.data();
    auto nothing = [] {};
    for (int context = 0; context < 2; context++) {
        every_place("plb_read_macros", nothing, [&] { return plb_read_macros(&c, d, d + c.N, nullptr, nullptr); });
        every_place("plb_read_populations", nothing, [&] { return plb_read_populations(&c, d); });
        every_place("plb_write_populations", nothing, [&] { return plb_write_populations(&c, d); });
        every_place("plb_read_state", nothing, [&] { return plb_read_state(&c, d); });
        every_place("plb_write_state", nothing, [&] { return plb_write_state(&c, d); });
        every_place("plb_read_table", nothing, [&] { return plb_read_table(&c, (int32_t*)d); });
        xfer_context(1);
    }
    int64_t it = 0;
    every_place("plb_step",
                [&] {
                    onchip_destroy(&c);
                    c.chip_state = 0;
                    c.chip_steps = ONCHIP_PLAN_STEPS;
                    it += 16;
                },
                [&] { return plb_step(&c, it, 16); });
    if (c.chip_state != 1) {
        fprintf(stderr, "the last step did not run on chip\n");
        fails++;
    }
    onchip_destroy(&c);
    c.host = nullptr;
    return fails != 0;
}

}  // namespace plb

int main() { return plb::run(); }
