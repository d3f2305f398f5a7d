// plb_api.hip -- the extern "C" boundary of libplb (declared in include/plb.h).
//
// One context = one pore-node lattice resident on one GPU, one HIP stream.
// The reference's SIMULATION lifecycle (porelb.c:402-443) maps as:
//   alloc_memory/check_V/build_send_recv_info -> plb_create / plb_create_from_flag
//   init_dist_macro                            -> plb_init_equilibrium
//   loop of send/stream/recv/collision         -> plb_step
//   save_data                                  -> plb_read_macros (+ host file write)
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>

#include "plb_xfer.hpp"

using namespace plb;

void plb_set_hip_error(hipError_t e, const char* what, const char* file, int line)
{
    fprintf(stderr, "libplb: HIP error %d (%s) in %s at %s:%d\n", (int)e, hipGetErrorString(e),
            what, file, line);
}

extern "C" void plb_config_default(plb_config* cfg)
{
    memset(cfg, 0, sizeof *cfg);
    cfg->tau = 0.8;   // porelb.c:87
    cfg->gx = 1.0e-3; // porelb.c:91
    cfg->rho0 = 1.0;  // porelb.c:228
    cfg->precision = PLB_FP64;
    cfg->bb_mode = PLB_BB_REFCOMPAT;
    cfg->layout = PLB_LAYOUT_SOA;
    cfg->ordering = PLB_ORDER_REFERENCE;
    cfg->brick[0] = 16;
    cfg->brick[1] = 4;
    cfg->brick[2] = 4;
    cfg->block_size = 256;
    cfg->device = 0;
    cfg->fp16_scale_log2 = 0;
    cfg->index_kind = PLB_INDEX_I32;
    cfg->nodes_per_thread = 1;
    cfg->graph_steps = 0;
    cfg->waves_per_simd = 0;
    cfg->fp16_rounding = PLB_ROUND_NEAREST;
    cfg->stream_mode = PLB_STREAM_PULL;
}

extern "C" const char* plb_strerror(int code)
{
    switch (code) {
    case PLB_OK: return "ok";
    case PLB_ERR_FILE: return "input file could not be opened";
    case PLB_ERR_NUM_P: return "rank count does not fit the V.bin / z-slab rule";
    case PLB_ERR_BOUNDS: return "node coordinate or neighbour id out of range";
    case PLB_ERR_PID: return "EXTERN neighbour with invalid rank id";
    case PLB_ERR_READ: return "short read";
    case PLB_ERR_DENSITY: return "density guard: rho > 1.2 or rho < 0.5";
    case PLB_ERR_ARGS: return "bad command line";
    case PLB_ERR_INVALID: return "invalid argument";
    case PLB_ERR_HIP: return "HIP runtime error";
    case PLB_ERR_NOMEM: return "out of memory";
    case PLB_ERR_RANGE: return "too many pore nodes for int32 node ids";
    case PLB_ERR_NODEVICE: return "no usable GPU";
    case PLB_ERR_FLAG: return "voxel flag value other than 0 or 1";
    default: return "unknown error";
    }
}

int plb::check_cfg(const plb_config* cfg)
{
    if (!cfg) return PLB_ERR_INVALID;
    if (!(cfg->tau > 0.0) || !isfinite(cfg->gx) || !(cfg->rho0 > 0.0)) return PLB_ERR_INVALID;
    if (cfg->precision < PLB_FP64 || cfg->precision > PLB_FP16) return PLB_ERR_INVALID;
    if (cfg->bb_mode != PLB_BB_REFCOMPAT && cfg->bb_mode != PLB_BB_HALFWAY) return PLB_ERR_INVALID;
    if (cfg->layout != PLB_LAYOUT_SOA && cfg->layout != PLB_LAYOUT_AOSOA) return PLB_ERR_INVALID;
    if (cfg->ordering != PLB_ORDER_REFERENCE && cfg->ordering != PLB_ORDER_BRICK &&
        cfg->ordering != PLB_ORDER_PENCIL)
        return PLB_ERR_INVALID;
    if (cfg->ordering != PLB_ORDER_REFERENCE &&
        (cfg->brick[0] < 1 || cfg->brick[1] < 1 || cfg->brick[2] < 1 ||
         cfg->brick[0] > 65535 || cfg->brick[1] > 65535 || cfg->brick[2] > 65535))
        return PLB_ERR_INVALID;
    if (cfg->block_size < 64 || cfg->block_size > 1024 || cfg->block_size % 64) return PLB_ERR_INVALID;
    if (cfg->fp16_scale_log2 < 0 || cfg->fp16_scale_log2 > 100) return PLB_ERR_INVALID;
    if (cfg->index_kind != PLB_INDEX_I32 && cfg->index_kind != PLB_INDEX_TILE8 &&
        cfg->index_kind != PLB_INDEX_BITMAP)
        return PLB_ERR_INVALID;
    // BITMAP derives sources from voxel positions: half-way bounce-back, and
    // node orders that are whole x-rows (checked against nx at build time).
    if (cfg->index_kind == PLB_INDEX_BITMAP &&
        (cfg->bb_mode != PLB_BB_HALFWAY ||
         (cfg->ordering != PLB_ORDER_REFERENCE && cfg->ordering != PLB_ORDER_PENCIL) ||
         (cfg->ordering == PLB_ORDER_PENCIL && cfg->brick[2] != 1)))
        return PLB_ERR_INVALID;
    if (cfg->nodes_per_thread != 1 && cfg->nodes_per_thread != 2) return PLB_ERR_INVALID;
    if (cfg->nodes_per_thread == 2 && cfg->block_size > 512) return PLB_ERR_INVALID;
    if (cfg->graph_steps < 0 || cfg->graph_steps > 4096 || cfg->graph_steps % 2) return PLB_ERR_INVALID;
    if (cfg->waves_per_simd < 0 || cfg->waves_per_simd > 8) return PLB_ERR_INVALID;
    if (cfg->fp16_rounding != PLB_ROUND_NEAREST && cfg->fp16_rounding != PLB_ROUND_STOCHASTIC)
        return PLB_ERR_INVALID;
    if (cfg->placement_reserve_gib < 0 || cfg->placement_reserve_gib > 160) return PLB_ERR_INVALID;
    if (cfg->stream_mode != PLB_STREAM_PULL && cfg->stream_mode != PLB_STREAM_AA) return PLB_ERR_INVALID;
    if (cfg->stream_mode == PLB_STREAM_AA &&
        (cfg->bb_mode != PLB_BB_HALFWAY || cfg->nodes_per_thread != 1 || cfg->graph_steps != 0))
        return PLB_ERR_INVALID;
    return PLB_OK;
}

// FP16 storage scale 2^k: deviations of order 1000*|gx| map to ~2048, far
// from both the FP16 overflow (65504) and its subnormal range (< 6.1e-5).
int plb::fp16_scale_log2_for(double gx)
{
    const double g = fabs(gx) > 0 ? fabs(gx) : 1e-9;
    const int k = (int)floor(log2(2048.0 / (1000.0 * g)));
    return std::max(1, std::min(k, 60));
}

int plb::ctx_begin(plb_ctx* c, const plb_config* cfg, int nx, int ny, int nz, int num_p)
{
    xfer_context(1);
    c->counted = true;
    c->segs.reserve(SEGMENTS_MOST);
    c->cfg = *cfg;
    c->nx = nx;
    c->ny = ny;
    c->nz = nz;
    c->num_p = num_p;
    c->elem = cfg->precision == PLB_FP64 ? 8 : (cfg->precision == PLB_FP32 ? 4 : 2);
    c->omega = 1.0 / cfg->tau;  // porelb.c:88
    const int k = cfg->fp16_scale_log2 ? cfg->fp16_scale_log2 : fp16_scale_log2_for(cfg->gx);
    c->scale_log2 = cfg->precision == PLB_FP16 ? k : 0;
    c->scale = cfg->precision == PLB_FP16 ? ldexpf(1.f, k) : 1.f;
    c->inv_scale = cfg->precision == PLB_FP16 ? ldexpf(1.f, -k) : 1.f;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return PLB_ERR_NODEVICE;
    if (cfg->device < 0 || cfg->device >= ndev) return PLB_ERR_INVALID;
    c->device = cfg->device;
    PLB_HIP(hipSetDevice(c->device));
    PLB_HIP(hipDeviceGetAttribute(&c->lds_per_cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor,
                                  c->device));
    const int rc = noalloc_setup(c->device);  // the no-alloc read-back's staging array
    if (rc) return rc;
    PLB_HIP(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    if (cfg->placement_reserve_gib > 0)  // before every buffer of the context
        PLB_HIP(dev_malloc(&c->reserve, (size_t)cfg->placement_reserve_gib << 30));
    PLB_HIP(hipEventCreate(&c->ev0));
    PLB_HIP(hipEventCreate(&c->ev1));
    return PLB_OK;
}

int plb::ctx_alloc_state(plb_ctx* c)
{
    const size_t nf = (size_t)c->Npad * Q * c->elem;
    PLB_HIP(c->mem.take(&c->f[0], nf));
    if (c->cfg.stream_mode == PLB_STREAM_AA)
        c->f[1] = c->f[0];  // one buffer; c->cur is the AA phase
    else
        PLB_HIP(c->mem.take(&c->f[1], nf));
    PLB_HIP(c->mem.take(&c->macros, 4 * c->Npad));
    PLB_HIP(hipMemsetAsync(c->macros, 0, sizeof(double) * 4 * c->Npad, c->stream));
    PLB_HIP(c->mem.take(&c->fault, 2));
    PLB_HIP(hipMemsetAsync(c->fault, 0xff, 2 * sizeof(unsigned long long), c->stream));
    PLB_HIP(hipHostMalloc((void**)&c->host, sizeof(HostWords), hipHostMallocDefault));
    int dev_cus = 256;
    (void)hipDeviceGetAttribute(&dev_cus, hipDeviceAttributeMultiprocessorCount, c->device);
    c->red_blocks = std::max(1, std::min<int>(dev_cus * 4, (int)((c->N + 255) / 256)));
    PLB_HIP(c->mem.take(&c->red, 2 * c->red_blocks));
    PLB_HIP(c->mem.take(&c->it_dev, 1));
    PLB_HIP(hipStreamSynchronize(c->stream));
    if (c->cfg.precision == PLB_FP16 && c->cfg.fp16_rounding == PLB_ROUND_STOCHASTIC) {
        c->key_bytes = 4.0;
        const int rc = build_key_runs(c);
        if (rc) return rc;
    }
    return plb_init_equilibrium(c);
}

extern "C" void plb_destroy(plb_ctx* c)
{
    if (!c) return;
    if (c->stream) {
        (void)hipSetDevice(c->device);
        (void)hipStreamSynchronize(c->stream);
    }
    if (c->host) (void)hipHostFree(c->host);
    onchip_destroy(c);
    if (c->ev0) (void)hipEventDestroy(c->ev0);
    if (c->ev1) (void)hipEventDestroy(c->ev1);
    for (hipGraphExec_t& g : c->gexec)
        if (g) (void)hipGraphExecDestroy(g);
    if (c->reserve) (void)hipFree(c->reserve);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    if (c->counted) xfer_context(-1);
    delete c;
}

extern "C" int plb_create(plb_ctx** out, const plb_config* cfg, const plb_node_info* V,
                          int64_t n_nodes, const int32_t* V_sub_start, int num_p, int nx, int ny,
                          int nz)
{
    if (!out) return PLB_ERR_INVALID;
    *out = nullptr;
    Range range("plb_create");
    int rc = check_cfg(cfg);
    if (rc) return rc;
    if (n_nodes < 0 || (n_nodes > 0 && !V) || !V_sub_start) return PLB_ERR_INVALID;
    if (nx <= 0 || ny <= 0 || nz <= 0 || nx > 65535 || ny > 65535 || nz > 65535)
        return PLB_ERR_INVALID;
    if (num_p < 1 || num_p > 65535) return PLB_ERR_NUM_P;
    if (n_nodes >= INT32_MAX) return PLB_ERR_RANGE;
    // V_sub_start must partition [0, n_nodes) into consecutive rank slices.
    if (V_sub_start[0] != 0) return PLB_ERR_NUM_P;
    for (int p = 1; p < num_p; p++)
        if (V_sub_start[p] < V_sub_start[p - 1]) return PLB_ERR_NUM_P;
    if (V_sub_start[num_p - 1] > n_nodes) return PLB_ERR_NUM_P;

    plb_ctx* c = new plb_ctx();
    rc = ctx_begin(c, cfg, nx, ny, nz, num_p);
    if (!rc) {
        c->V_sub_start.assign(V_sub_start, V_sub_start + num_p);
        c->N = n_nodes;
        c->Npad = std::max<int64_t>(64, (n_nodes + 63) / 64 * 64);
        rc = build_table_from_V(c, V, n_nodes);
    }
    if (!rc) rc = ctx_alloc_state(c);
    if (rc) {
        plb_destroy(c);
        return rc;
    }
    *out = c;
    return PLB_OK;
}

extern "C" int plb_create_from_flag(plb_ctx** out, const plb_config* cfg, const uint8_t* flag,
                                    int nx, int ny, int nz, int num_p)
{
    if (!out) return PLB_ERR_INVALID;
    *out = nullptr;
    Range range("plb_create_from_flag");
    int rc = check_cfg(cfg);
    if (rc) return rc;
    if (!flag || nx <= 0 || ny <= 0 || nz <= 0 || nx > 65535 || ny > 65535 || nz > 65535)
        return PLB_ERR_INVALID;
    // z-slab rule pid = z/(nz/num_p) must stay inside [0, num_p) (preprocess.c:107).
    if (num_p < 1 || num_p > 65535 || nz / num_p == 0) return PLB_ERR_NUM_P;
    if ((nz - 1) / (nz / num_p) >= num_p) return PLB_ERR_NUM_P;
    plb_ctx* c = new plb_ctx();
    rc = ctx_begin(c, cfg, nx, ny, nz, num_p);
    if (!rc) rc = build_table_from_flag(c, flag);
    if (!rc) rc = ctx_alloc_state(c);
    if (rc) {
        plb_destroy(c);
        return rc;
    }
    *out = c;
    return PLB_OK;
}

__global__ void k_fill_macros(double* m, int64_t Npad, double rho0)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= Npad) return;
    m[i] = rho0;
    m[Npad + i] = 0.0;
    m[2 * Npad + i] = 0.0;
    m[3 * Npad + i] = 0.0;
}

// A state written in from outside starts with a clear density guard: the
// fault words are reset and nothing is pending.
static int clear_fault(plb_ctx* c)
{
    PLB_HIP(hipMemsetAsync(c->fault, 0xff, 2 * sizeof(unsigned long long), c->stream));
    if (c->chip) {
        const int rc = onchip_clear(c);
        if (rc) return rc;
    }
    PLB_HIP(hipStreamSynchronize(c->stream));
    c->segs.clear();
    c->fault_seen = c->fault_held = false;
    return PLB_OK;
}

extern "C" int plb_init_equilibrium(plb_ctx* c)
{
    if (!c) return PLB_ERR_INVALID;
    PLB_HIP(hipSetDevice(c->device));
    // AA: the rest state (every slot w_j rho0) is the local-step form, so the
    // first step is a neighbour step, like a pull step
    c->cur = c->cfg.stream_mode == PLB_STREAM_AA ? 1 : 0;
    int rc = launch_init_eq(c);
    if (rc) return rc;
    hipLaunchKernelGGL(k_fill_macros, dim3((unsigned)((c->Npad + 255) / 256)), dim3(256), 0,
                       c->stream, c->macros, c->Npad, c->cfg.rho0);
    PLB_HIP(hipGetLastError());
    return clear_fault(c);
}

// The fault words, once everything queued has run.
static int read_fault_words(plb_ctx* c, unsigned long long* key, unsigned long long* gave_up)
{
    const int rc = launch_fault_words(c);
    if (rc) return rc;
    PLB_HIP(hipStreamSynchronize(c->stream));
    *key = c->host->fault[0];
    *gave_up = c->host->fault[1];
    return PLB_OK;
}

// Waits for the calls that are queued and settles them: none is left in c->segs,
// and c->cur is the buffer of the state.  An on-chip run in which the density
// guard tripped, or which gave up waiting for a block, has left the state before
// it (and the macros) untouched, and everything queued behind it has left the
// state alone: it and the calls after it are repeated with one launch per step,
// which freeze at the end of the faulting step.  (The queued calls' step numbers
// rise, so a fault's step names its call.)
static int settle(plb_ctx* c, unsigned long long* key)
{
    unsigned long long gave_up = NO_FAULT;
    int rc = read_fault_words(c, key, &gave_up);
    if (rc) return rc;
    auto trips = [&](const Segment& s) {
        const int64_t fs = (int64_t)(*key >> 32);
        return *key != HOLD_FAULT && fs >= s.it0 && fs < s.it0 + s.n;
    };
    size_t k = 0;
    if (*key != NO_FAULT)
        while (k < c->segs.size() && !(c->segs[k].serial && (c->segs[k].serial == gave_up || trips(c->segs[k])))) k++;
    if (*key != NO_FAULT && k < c->segs.size()) {
        if (gave_up != NO_FAULT) {
            rc = onchip_gave_up(c);
            if (rc) return rc;
        }
        PLB_HIP(hipMemsetAsync(c->fault, 0xff, 2 * sizeof(unsigned long long), c->stream));
        c->cur = c->segs[k].cur;
        onchip_restore_macros(c, c->segs[k].macros);
        for (; k < c->segs.size(); k++) {
            Segment& s = c->segs[k];
            s.serial = 0;
            s.cur = c->cur;
            if (c->timed && k + 1 == c->segs.size()) PLB_HIP(hipEventRecord(c->ev0, c->stream));
            for (int64_t t = 0; t < s.n; t++) {
                rc = launch_step(c, s.it0 + t, t == s.n - 1);
                if (rc) return rc;
            }
        }
        if (c->timed) PLB_HIP(hipEventRecord(c->ev1, c->stream));
        rc = read_fault_words(c, key, &gave_up);
        if (rc) return rc;
    }
    if (*key != NO_FAULT) {
        // Steps after the faulting one did not run: the faulting step's output
        // buffer holds the current state (a fault from an earlier call made
        // every launch of these a no-op), and the macros are in the array that
        // its call writes, also where on-chip runs behind it have swapped them.
        const int64_t fs = (int64_t)(*key >> 32);
        for (const Segment& s : c->segs)
            if (fs < s.it0 + s.n) {
                c->cur = fs < s.it0 ? s.cur : s.cur ^ (int)((fs - s.it0 + 1) & 1);
                onchip_restore_macros(c, s.macros);
                break;
            }
        if (!c->fault_seen) c->fault_held = true;
    }
    c->segs.clear();
    return PLB_OK;
}

// Before the state or the macros are read without a plb_sync.
int plb::settle_for_read(plb_ctx* c)
{
    for (const Segment& s : c->segs)
        if (s.serial) {
            unsigned long long key;
            return settle(c, &key);
        }
    return PLB_OK;
}

extern "C" int plb_step_async(plb_ctx* c, int64_t it0, int64_t nsteps)
{
    if (!c || nsteps < 0 || it0 < 0 || it0 + nsteps >= ((int64_t)1 << 31)) return PLB_ERR_INVALID;
    Range range("plb_step");
    PLB_HIP(hipSetDevice(c->device));
    // A call whose step numbers start again would not be held off by a fault of
    // the calls before it, and the fault's step would not tell it from them.
    if (c->segs.size() >= SEGMENTS_MOST || (!c->segs.empty() && it0 < c->segs.back().it0 + c->segs.back().n)) {
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;  // it waits, also beside a capture of the caller's
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        unsigned long long key;
        const int rc = settle(c, &key);
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        if (rc) return rc;
    }
    const bool chip = !c->fault_held && onchip_ready(c, nsteps);
    if (c->timed) PLB_HIP(hipEventRecord(c->ev0, c->stream));  // behind the plan
    if (c->fault_held) return PLB_OK;  // the state stays that of a fault until plb_sync has reported it
    Segment seg{it0, nsteps, c->cur, 0, c->macros};
    if (chip) {
        int rc = launch_onchip(c, it0, nsteps, &seg.serial);
        if (rc) return rc;
        if (seg.serial) {
            c->segs.push_back(seg);
            return PLB_OK;
        }
    }
    int64_t s = 0;
    // Runs of graph_steps steps replay a captured graph; the last step of the
    // call is always a plain launch (it writes the macros).
    for (const int64_t G = c->N > 0 ? c->cfg.graph_steps : 0; G > 0 && nsteps - s > G; s += G) {
        int rc = launch_graph_steps(c, it0 + s, G);
        if (rc) return rc;
    }
    for (; s < nsteps; s++) {
        int rc = launch_step(c, it0 + s, s == nsteps - 1);
        if (rc) return rc;
    }
    // steps that go on from launches per step are of one call with them
    Segment* const last = c->segs.empty() ? nullptr : &c->segs.back();
    if (last && !last->serial && last->it0 + last->n == it0) last->n += nsteps;
    else if (nsteps > 0) c->segs.push_back(seg);
    return PLB_OK;
}

extern "C" int plb_sync(plb_ctx* c)
{
    if (!c) return PLB_ERR_INVALID;
    PLB_HIP(hipSetDevice(c->device));
    unsigned long long key = NO_FAULT;
    const int rc = settle(c, &key);
    if (rc) return rc;
    if (key == NO_FAULT) return PLB_OK;
    c->fault_held = false;
    c->fault_seen = true;
    return PLB_ERR_DENSITY;
}

extern "C" int plb_step(plb_ctx* c, int64_t it0, int64_t nsteps)
{
    int rc = plb_step_async(c, it0, nsteps);
    if (rc) return rc;
    return plb_sync(c);
}

extern "C" int plb_step_timed(plb_ctx* c, int64_t it0, int64_t nsteps, double* ms)
{
    if (!c || !ms) return PLB_ERR_INVALID;
    PLB_HIP(hipSetDevice(c->device));
    // Steps that are repeated, since an on-chip run of them did not complete, are timed where they are repeated.
    c->timed = true;
    int rc = plb_step_async(c, it0, nsteps);
    hipError_t e = rc ? hipSuccess : hipEventRecord(c->ev1, c->stream);
    if (!rc && e == hipSuccess) rc = plb_sync(c);
    c->timed = false;
    PLB_HIP(e);
    if (rc && rc != PLB_ERR_DENSITY) return rc;
    float t = 0.f;
    PLB_HIP(hipEventElapsedTime(&t, c->ev0, c->ev1));
    *ms = t;
    return rc;
}

extern "C" int64_t plb_num_nodes(const plb_ctx* c) { return c ? c->N : -1; }

extern "C" void* plb_host_alloc(size_t bytes)
{
    void* p = nullptr;
    if (hipHostMalloc(&p, bytes ? bytes : 1, hipHostMallocDefault) != hipSuccess) return nullptr;
    return p;
}

extern "C" void plb_host_free(void* p)
{
    if (p) (void)hipHostFree(p);
}

extern "C" double plb_bytes_per_update(const plb_ctx* c)
{
    if (!c) return 0.0;
    // FP16 storage with stochastic rounding also reads each node's V-order key:
    // 16 bytes per tile of runs, plus 4 per node in tiles that load their keys
    const bool key = c->cfg.precision == PLB_FP16 && c->cfg.fp16_rounding == PLB_ROUND_STOCHASTIC &&
                     (c->perm || c->key_perm);
    // AA streaming reads the table on odd steps only
    const double idx = c->cfg.stream_mode == PLB_STREAM_AA ? 0.5 * c->index_bytes : c->index_bytes;
    return 2.0 * Q * (double)c->elem + idx + (key ? c->key_bytes : 0.0);
}

extern "C" int plb_read_macros(plb_ctx* c, double* rho, double* ux, double* uy, double* uz)
{
    if (!c) return PLB_ERR_INVALID;
    Range range("plb_read_macros");
    PLB_HIP(hipSetDevice(c->device));
    if (const int rcs = settle_for_read(c)) return rcs;
    return read_macros_range(c, 0, c->N, rho, ux, uy, uz);
}

// The macros that are asked for, of V-order nodes first .. first + n - 1.
int plb::read_macros_range(plb_ctx* c, int64_t first, int64_t n, double* rho, double* ux, double* uy, double* uz)
{
    double* const outs[4] = {rho, ux, uy, uz};
    Arrays arrays;
    MacroList list;
    for (int k = 0; k < 4; k++)
        if (outs[k]) {
            list.out[list.n] = outs[k];
            list.comp[list.n++] = k;
            arrays.add(outs[k]);
        }
    // Page-locked arrays take the kernel's own stores: a row of 64 values of one
    // component is 512 bytes on the bus, 54 GB/s from the first call on.
    bool locked = n > 0 && list.n > 0;
    for (int q = 0; q < list.n && locked; q++) locked = page_locked(list.out[q]) && page_locked(list.out[q] + n - 1);
    if (locked) {
        const int rc = launch_read_macros(c, list, first, n);
        if (rc) return rc;
        PLB_HIP(hipStreamSynchronize(c->stream));
        return PLB_OK;
    }
    return download(c->device, c->stream, n, sizeof(double), arrays, [&](int64_t b, int64_t m, void* d) {
        for (int q = 0; q < list.n; q++) list.out[q] = (double*)d + q * m;
        return launch_read_macros(c, list, first + b, m);
    });
}

extern "C" int plb_read_populations(plb_ctx* c, double* f_aos)
{
    if (!c || (!f_aos && c->N)) return PLB_ERR_INVALID;
    PLB_HIP(hipSetDevice(c->device));
    if (const int rcs = settle_for_read(c)) return rcs;
    return download(c->device, c->stream, c->N, sizeof(double) * Q, f_aos,
                    [&](int64_t b, int64_t m, void* d) { return launch_read_pop(c, b, m, (double*)d); });
}

extern "C" int plb_write_populations(plb_ctx* c, const double* f_aos)
{
    if (!c || (!f_aos && c->N)) return PLB_ERR_INVALID;
    PLB_HIP(hipSetDevice(c->device));
    if (const int rcs = settle_for_read(c)) return rcs;
    const int rc = upload(c->device, c->stream, c->N, sizeof(double) * Q, f_aos,
                          [&](int64_t b, int64_t m, void* d) { return launch_write_pop(c, b, m, (const double*)d); });
    return rc ? rc : clear_fault(c);
}

extern "C" int plb_get_state_info(const plb_ctx* c, plb_state_info* out)
{
    if (!c || !out) return PLB_ERR_INVALID;
    memset(out, 0, sizeof *out);
    out->precision = c->cfg.precision;
    out->elem_bytes = (int)c->elem;
    out->fp16_scale_log2 = c->scale_log2;
    out->rho0 = c->cfg.rho0;
    out->n_nodes = c->N;
    return PLB_OK;
}

// Stored elements between host AoS [n][19] and the device layout.
extern "C" int plb_read_state(plb_ctx* c, void* buf)
{
    if (!c || (!buf && c->N)) return PLB_ERR_INVALID;
    PLB_HIP(hipSetDevice(c->device));
    if (const int rcs = settle_for_read(c)) return rcs;
    return download(c->device, c->stream, c->N, Q * c->elem, buf,
                    [&](int64_t b, int64_t m, void* d) { return launch_copy_state(c, b, m, d, false); });
}

extern "C" int plb_write_state(plb_ctx* c, const void* buf)
{
    if (!c || (!buf && c->N)) return PLB_ERR_INVALID;
    PLB_HIP(hipSetDevice(c->device));
    if (const int rcs = settle_for_read(c)) return rcs;
    const int rc = upload(c->device, c->stream, c->N, Q * c->elem, buf,
                          [&](int64_t b, int64_t m, void* d) { return launch_copy_state(c, b, m, d, true); });
    return rc ? rc : clear_fault(c);
}

extern "C" int plb_read_table(plb_ctx* c, int32_t* tab)
{
    if (!c || (!tab && c->N)) return PLB_ERR_INVALID;
    PLB_HIP(hipSetDevice(c->device));
    Arrays rows;
    for (int j = 0; j < Q - 1; j++) rows.add(tab + (int64_t)j * c->N);
    return download(c->device, c->stream, c->N, sizeof(int32_t), rows,
                    [&](int64_t b, int64_t m, void* d) { return launch_read_table(c, b, m, (int32_t*)d); });
}

// The reduction from its two sums.
static void fill_reduction(const plb_ctx* c, plb_reduction* out)
{
    const double r[2] = {c->N ? c->host->sum[0] : 0.0, c->N ? c->host->sum[1] : 0.0};
    double mass = r[0];
    if (c->cfg.precision != PLB_FP64) {
        double w = 0.0;
        for (int j = 0; j < Q; j++) w += TP[j] * c->cfg.rho0;
        mass += w * (double)c->N;
    }
    out->mass = mass;
    out->sum_ux = r[1];
    out->mean_ux = c->N ? r[1] / (double)c->N : 0.0;
    out->q = r[1] / ((double)c->nx * c->ny * c->nz);
    const double nu = 1.0 / 3.0 * (c->cfg.tau - 0.5);  // porelb.c:89
    out->K = c->cfg.gx != 0.0 ? nu * out->q / c->cfg.gx : 0.0;
    out->n_nodes = c->N;
}

extern "C" int plb_reduce(plb_ctx* c, plb_reduction* out)
{
    if (!c || !out) return PLB_ERR_INVALID;
    Range range("plb_reduce");
    PLB_HIP(hipSetDevice(c->device));
    if (const int rcs = settle_for_read(c)) return rcs;
    if (c->N > 0) {
        int rc = launch_reduce(c);
        if (rc) return rc;
        PLB_HIP(hipStreamSynchronize(c->stream));
    }
    fill_reduction(c, out);
    return PLB_OK;
}

// plb_step and plb_reduce with one wait for both (two waits and copies back
// took 45 us of a check, as long as ten steps of a small lattice).
static int step_and_reduce(plb_ctx* c, int64_t it0, int64_t n, plb_reduction* out)
{
    int rc = plb_step_async(c, it0, n);
    if (rc) return rc;
    if (c->N > 0) {
        rc = launch_reduce(c);
        if (rc) return rc;
        PLB_HIP(hipStreamSynchronize(c->stream));
        if (c->host->fault[0] == NO_FAULT) {
            c->segs.clear();
            fill_reduction(c, out);
            return PLB_OK;
        }
    }
    rc = plb_sync(c);  // a density trip, or steps to repeat
    return rc ? rc : plb_reduce(c, out);
}

extern "C" int plb_run_to_convergence(plb_ctx* c, int64_t it0, int64_t max_steps, int64_t check_every,
                                      double tol, int64_t* steps_done, plb_reduction* out)
{
    if (!c || !steps_done || !out || it0 < 0 || max_steps < 0 || check_every < 1 || !(tol >= 0.0))
        return PLB_ERR_INVALID;
    Range range("plb_run_to_convergence");
    *steps_done = 0;
    int rc = plb_reduce(c, out);  // the state before the first run (macros as stored)
    if (rc) return rc;
    // The rule cannot stop the run before its second check: steps that are sure
    // to come count for the on-chip plan from the start (100 steps of 265 421
    // FP32 nodes: 1.2 ms one by one, 0.4 on chip and 0.5 for the plan, once).
    const int64_t sure = tol > 0.0 && check_every < max_steps / 2 ? 2 * check_every : max_steps;
    if (c->chip_steps + sure >= ONCHIP_PLAN_STEPS) c->chip_steps = std::max(c->chip_steps, ONCHIP_PLAN_STEPS);
    double prev = NAN;
    const double umin = 1e-3 * fabs(c->cfg.gx);
    for (int64_t s = 0; s < max_steps;) {
        const int64_t m = std::min(check_every, max_steps - s);
        rc = step_and_reduce(c, it0 + s, m, out);
        if (rc) return rc;
        s += m;
        *steps_done = s;
        const double mean = out->mean_ux;
        if (tol > 0.0 && !isnan(prev) && fabs(mean - prev) <= tol * std::max(fabs(mean), umin)) break;
        prev = mean;
    }
    return PLB_OK;
}

extern "C" int plb_last_fault(plb_ctx* c, plb_fault* out)
{
    if (!c || !out) return PLB_ERR_INVALID;
    PLB_HIP(hipSetDevice(c->device));
    if (const int rcs = settle_for_read(c)) return rcs;
    memset(out, 0, sizeof *out);
    unsigned long long key = NO_FAULT, gave_up = NO_FAULT;
    const int rc = read_fault_words(c, &key, &gave_up);
    if (rc) return rc;
    if (key == NO_FAULT) return PLB_OK;
    out->tripped = 1;
    out->step = (int64_t)(key >> 32);
    out->node = (int64_t)(key & 0xffffffffull);
    if (out->node >= c->N) return PLB_ERR_BOUNDS;
    int p = 0;
    for (int q = 0; q < c->num_p; q++)
        if (c->V_sub_start[q] <= out->node) p = q;
    out->pid = p;
    out->local_id = out->node - c->V_sub_start[p];
    int64_t k = out->node;
    if (c->inv_perm) {
        uint32_t kk = 0;
        PLB_HIP(hipMemcpy(&kk, c->inv_perm + out->node, sizeof kk, hipMemcpyDeviceToHost));
        if ((int64_t)kk >= c->N) return PLB_ERR_BOUNDS;
        k = kk;
    }
    uint64_t xyz = 0;
    PLB_HIP(hipMemcpy(&xyz, c->node_xyz + k, sizeof xyz, hipMemcpyDeviceToHost));
    PLB_HIP(hipMemcpy(&out->rho, c->macros + k, sizeof(double), hipMemcpyDeviceToHost));
    out->x = (int)(xyz & 0xffff);
    out->y = (int)((xyz >> 16) & 0xffff);
    out->z = (int)((xyz >> 32) & 0xffff);
    return PLB_OK;
}
