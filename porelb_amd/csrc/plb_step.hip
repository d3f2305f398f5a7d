// plb_step.hip -- the fused D3Q19 time step on gfx950, plus the kernels that
// move populations and macros in and out of the device layouts and the FP64
// reductions.
//
// One kernel per time step, one thread per pore node:
//   1. 18 pull-table entries (int32, TILE8 bases + packed u8 offsets, or
//      derived from the BITMAP index);
//   2. 19 population gathers issued back to back (stream: f[j][src];
//      bounce and const: f[re[j]][self], const replaced after the load);
//   3. collision with body force (porelb.c:318-365);
//   4. 19 coalesced non-temporal stores into the other ping-pong buffer.
// This fuses stream_inner_nodes, update_recv_dist and collision
// (porelb.c:285-365); the reference's f1 array never exists.
//
// FP64 (PLB_FP64): unshifted populations, arithmetic in exactly the
// reference's evaluation order (porelb.c:6-13, 326-362); the library is
// compiled with -ffp-contract=off so results match the reference bit for bit.
// FP32/FP16 storage: populations are stored as deviations d_j = f_j - w_j*rho0
// (FP16 scaled by 2^k), and the collision runs in FP32 on the deviations:
//   d'_j = (1-omega) d_j + omega*dfeq_j + S_j*feq_j,
//   dfeq_j = w_j (drho + rho*P_j), P_j = 3 eu + 4.5 eu^2 - 1.5 u^2,
//   S_j = (1 - omega/2)*3*(e_jx - u)*F,
// which is the reference update minus w_j*rho0 on both sides.
#include <algorithm>

#include "plb_device.hpp"

namespace plb {

// Single lattice, one node per thread, XCD-contiguous block order.
template <typename S, int LAYOUT, int IDX>
__global__ void __launch_bounds__(1024) k_step(const StepArgs a)
{
    const int64_t blk = xcd_block(blockIdx.x, gridDim.x);
    const int64_t i = blk * blockDim.x + threadIdx.x;
    if (i >= a.N) return;
    node_any<S, LAYOUT, IDX>(with_step(a), i, *a.fault);
}

// The same with plain stores for `keep` of 16 groups of 16 blocks, for FP64 and
// FP32 lattices that do not fit the L2s (8 x 4 MB) but whose two buffers and index
// fit the 256 MB memory-side cache, all or in part: non-temporal stores go past
// that cache, and the next step then reads from HBM what this one wrote.  Of a
// lattice beyond 208 MB, the share that takes KEEP_BYTES is kept; the rest passes
// by.  (Keeping everything there pushes out what is still to be read.)  us a step
// against non-temporal stores alone: FP64 14.8 / 16.1 at 204 442 nodes (66 MB), 37.5 /
// 40.5 at 629 146 (204 MB), 47.6 / 52.3 at 823 200 (267 MB), 60.5 / 65.0 at 1 053 542
// (341 MB), 95.2 / 99.3 at 1 635 533 (530 MB); FP32 15.7 / 16.6 at 421 478 (72 MB),
// 39.2 / 41.7 at 1 228 800 (211 MB), 64.5 / 69.7 at 2 123 366 (365 MB), 99.3 / 103.8 at
// 3 194 400 (549 MB), 138.8 / 138.7 at 4 251 746 (731 MB).  Below 32 MB plain stores
// lose (FP64 7.1 / 6.5 at 78 643 nodes), and FP16, bound by L2 requests, gains at no
// size.
template <typename S, int LAYOUT, int IDX>
__global__ void __launch_bounds__(1024) k_step_keep(const StepArgs a, int keep)
{
    const int64_t blk = xcd_block(blockIdx.x, gridDim.x);
    const int64_t i = blk * blockDim.x + threadIdx.x;
    if (i >= a.N) return;
    node_any<S, LAYOUT, IDX, false, true>(with_step(a), i, *a.fault, (int)((blk >> 4) & 15) < keep);
}
constexpr double KEEP_ABOVE = 32e6, KEEP_ALL = 208e6, KEEP_MOST = 600e6, KEEP_BYTES = 115e6;

// Single lattice, one buffer, AA pattern (half-way bounce-back).  The
// buffer alternates between two forms of the post-collision populations
// f*_j(y) of the last step: after a neighbour step (and at rest), f*_j(y)
// lies at out_pos<2>(y, j), which is the pre-collision population of the
// node downstream -- so the next step reads each node's own 19 slots (MODE
// 1, no pull table) and leaves f*_j(y) in the node's own slot re[j]
// (out_pos<1>).  The step after that (MODE 2) reads population j of node x
// from slot re[j] of the upstream node t[j] (x - e_j; its own slot j at a
// wall) and stores by out_pos<2>.  A node of a MODE 2 step reads and writes
// the same 19 locations, so nodes never race; every step stores the values
// the pull step computes.  c->cur names the form (1: out_pos<1>, 0:
// out_pos<2>); read-backs map through it.
template <typename S, int LAYOUT, int IDX, int MODE>
__device__ __forceinline__ void step_aa(const StepArgs& a0)
{
    const StepArgs a = with_step(a0);
    const int64_t blk = xcd_block(blockIdx.x, gridDim.x);
    const int64_t i = blk * blockDim.x + threadIdx.x;
    if (i >= a.N) return;
    const S* __restrict__ f = (const S*)a.fin;
    S raw[Q];
    if constexpr (MODE == 1) {
#pragma unroll
        for (int j = 0; j < Q; j++) raw[j] = f[fpos<LAYOUT>(j, i, a.Npad)];
        const uint32_t key = sr_key<S>(a, i);
        const int32_t none[Q] = {};
        collide_any<S, LAYOUT, 1>(a, i, none, raw, *a.fault, key);
    } else {
        Entries<IDX> e;
        issue_entries<LAYOUT, IDX>(a, i, e);
        decode_entries<IDX>(a, i, e);
        raw[0] = f[fpos<LAYOUT>(0, i, a.Npad)];
#pragma unroll
        for (int j = 1; j < Q; j++) {
            const int64_t src = e.t[j] >= 0 ? fpos<LAYOUT>(RE[j], e.t[j], a.Npad) : fpos<LAYOUT>(j, i, a.Npad);
            raw[j] = f[src];
        }
        const uint32_t key = sr_key<S>(a, i);
        collide_any<S, LAYOUT, 2>(a, i, e.t, raw, *a.fault, key);
    }
}
template <typename S, int LAYOUT, int IDX>
__global__ void __launch_bounds__(1024) k_step_aa_even(const StepArgs a)
{
    step_aa<S, LAYOUT, IDX, 1>(a);
}
template <typename S, int LAYOUT, int IDX>
__global__ void __launch_bounds__(1024) k_step_aa_odd(const StepArgs a)
{
    step_aa<S, LAYOUT, IDX, 2>(a);
}

// Single lattice, two nodes per thread: each wave covers two consecutive
// 64-node tiles and keeps both tiles' index loads and gathers in flight
// together (more bytes in flight per wave at the cost of registers).
template <typename S, int LAYOUT, int IDX>
__global__ void __launch_bounds__(512) k_step2(const StepArgs a0)
{
    const StepArgs a = with_step(a0);
    const int64_t blk = xcd_block(blockIdx.x, gridDim.x);
    const int64_t t = blk * blockDim.x + threadIdx.x;
    const int64_t i0 = (t >> 6) * 128 + (t & 63);
    const int64_t i1 = i0 + 64;
    if (i0 >= a.N) return;
    const bool two = i1 < a.N;
    const unsigned long long fk = *a.fault;
    Entries<IDX> e0, e1;
    issue_entries<LAYOUT, IDX>(a, i0, e0);
    if (two) issue_entries<LAYOUT, IDX>(a, i1, e1);
    decode_entries<IDX>(a, i0, e0);
    if (two) decode_entries<IDX>(a, i1, e1);
    S r0[Q], r1[Q];
    gather<S, LAYOUT>(a, i0, e0.t, r0);
    if (two) gather<S, LAYOUT>(a, i1, e1.t, r1);
    const uint32_t k0 = sr_key<S>(a, i0), k1 = two ? sr_key<S>(a, i1) : 0u;
    collide_any<S, LAYOUT>(a, i0, e0.t, r0, fk, k0);
    if (two) collide_any<S, LAYOUT>(a, i1, e1.t, r1, fk, k1);
}

// Batch of samples: the grid enumerates the blocks of active samples
// (active[]), each block lies inside one sample (samples are padded to a
// multiple of the block size), and the sample supplies omega and gx.
struct BatchArgs {
    const int32_t* active;       // global block ids of active samples
    const int32_t* block_sample; // global block -> sample
    const int64_t* sample_end;   // first node after each sample's nodes
    const double* omega;         // per sample
    const double* gx;            // per sample
};

template <typename S, int LAYOUT, int IDX>
__global__ void __launch_bounds__(1024) k_step_batch(StepArgs a, const BatchArgs b)
{
    const int64_t slot = xcd_block(blockIdx.x, gridDim.x);
    const int64_t gb = b.active[slot];
    const int s = b.block_sample[gb];
    const int64_t i = gb * blockDim.x + threadIdx.x;
    if (i >= b.sample_end[s]) return;
    a.omega = b.omega[s];
    a.gx = b.gx[s];
    node_any<S, LAYOUT, IDX>(a, i, *a.fault);
}

// ---------------------------------------------------------------- fixed-order sums
// Sum of one double per thread of the block, in a fixed order; the result
// is valid in thread 0.  lds holds blockDim.x / 64 doubles.
__device__ __forceinline__ double block_sum_fixed(double v, double* lds)
{
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m, 64);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += lds[w];
    __syncthreads();
    return t;
}

// Sum of a sample's chunk partials by one wave (lane 0 holds the result).
__device__ __forceinline__ double wave_sum_chunks(const double* partial, int64_t c0, int64_t nc)
{
    const int lane = threadIdx.x & 63;
    double acc = 0.0;
    for (int64_t k = lane; k < nc; k += 64) acc += partial[c0 + k];
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) acc += __shfl_xor(acc, m, 64);
    return acc;
}

// ---------------------------------------------------------------- persistent batch
// One launch runs every sample of a batch from its first step to its own
// convergence stop.  The grid is resident (cooperative launch); each
// work-group walks the chunks (blocks of the batch layout) of the active
// samples, with each XCD taking contiguous runs of chunks as in xcd_block.
// A grid barrier separates time steps.  On check steps every chunk stores
// its macros and the fixed-order sum of its u_x; after a barrier, one wave
// per sample forms the sample's sum (the same order as k_sample_sums),
// applies the convergence rule and retires the sample; a second barrier
// publishes the decisions.
//
// Barriers follow the cooperative grid-sync pattern: a block barrier, then
// one thread per block releases the block's stores at agent scope and
// arrives; after the whole grid has arrived it acquires, and a second block
// barrier lets the block go on.  Arrivals and waits are spread over eight
// groups of blocks (block id mod 8, the XCD a block is dispatched to), each
// on its own 128-byte line: the last arrival of a group carries the group
// to a grid-wide counter, and the last group releases every group's flag.
// All counters are monotonic (barrier `gen` completes at gen x members), so
// nothing is reset between barriers.  A wait is bounded by wall time
// (wall_clock64 ticks): a block that waits longer sets `abort`, every block
// leaves the loop at its next barrier, and the host reports the failure, so
// the kernel always ends.  The samples' running flags are copied to LDS
// after every barrier that can change them, so the chunk loop reads them
// without a memory round trip.
constexpr int PERSIST_MAX_SAMPLES = PLB_PERSIST_MAX_SAMPLES;
constexpr int BAR_STRIDE = 16;  // u64 words between counters: one 128-byte line each

__device__ __forceinline__ bool grid_barrier(const PersistArgs& p, unsigned long long& gen)
{
    __shared__ int ok;
    __syncthreads();
    gen++;
    if (threadIdx.x == 0) {
        const unsigned G = gridDim.x, g = blockIdx.x & 7u;
        const unsigned long long members = (G - 1 - g) / 8 + 1, groups = G < 8 ? G : 8;
        unsigned long long* cnt = p.bar + g * BAR_STRIDE;
        unsigned long long* all = p.bar + 8 * BAR_STRIDE;
        unsigned long long* rel = p.bar + 9 * BAR_STRIDE;
        int good = 1;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        if (__hip_atomic_fetch_add(cnt, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == gen * members) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "agent");
            if (__hip_atomic_fetch_add(all, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == gen * groups) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "agent");
                for (unsigned k = 0; k < groups; k++)
                    __hip_atomic_store(rel + k * BAR_STRIDE, gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        const uint64_t t0 = wall_clock64();
        while (__hip_atomic_load(rel + g * BAR_STRIDE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < gen) {
            if (__hip_atomic_load(p.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                good = 0;
                break;
            }
            if (wall_clock64() - t0 > p.wait_ticks) {
                __hip_atomic_store(p.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                good = 0;
                break;
            }
            __builtin_amdgcn_s_sleep(8);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        ok = good;
    }
    __syncthreads();
    return ok;
}

template <typename S, int LAYOUT, int IDX>
__global__ void __launch_bounds__(1024) k_batch_persistent(StepArgs a, const PersistArgs p)
{
    __shared__ double lds[16];
    // aprefix[s] = active chunks of the samples before s (so sample s runs
    // iff aprefix[s + 1] > aprefix[s]); rebuilt after every decision barrier.
    __shared__ int aprefix[PERSIST_MAX_SAMPLES + 1];
    __shared__ int stop;
    __shared__ int64_t claim[2];   // the chunks this block claimed, in its stretch (alternating slots)
    const int bs = blockDim.x;
    // The active chunks, in sample order, are split into eight contiguous
    // stretches, one per XCD (block id mod 8).  The blocks of a stretch take
    // its chunks one at a time from the stretch's counter for this step
    // (line 17 + 2 * group + step parity of p.bar), so the XCD sweeps its
    // stretch in order and a block that finishes early takes more, as the
    // hardware dispatcher does in a launch per step.  Each block claims its
    // next chunk before it processes the current one, which hides the
    // atomic's round trip.  (Claims of 2, 4 or 8 chunks, spread so that the
    // chunks in flight stay consecutive, were slower.)
    const unsigned G = gridDim.x, grp = blockIdx.x & 7u, slot = blockIdx.x >> 3;
    const int64_t ngrp = G < 8 ? G : 8;   // groups that have blocks
    unsigned long long gen = 0;
    // Residency check before any work: every block counts itself in and
    // waits, briefly, for the whole grid.  One decision word settles the
    // outcome for all blocks: the first block to see the full count sets it
    // to "go", the first to wait past start_ticks sets it to "leave" (a grid
    // larger than what the CUs really hold never completes the count), and
    // every block then follows it.  On "leave" the blocks exit before any
    // work with abort = 2, and the host launches a smaller grid.
    if (threadIdx.x == 0) {
        unsigned long long* started = p.bar + 33 * BAR_STRIDE;
        unsigned long long* decision = started + 1;   // 0 open, 1 go, 2 leave
        __hip_atomic_fetch_add(started, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t t0 = wall_clock64();
        unsigned long long d;
        while ((d = __hip_atomic_load(decision, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0) {
            unsigned long long open = 0;
            if (__hip_atomic_load(started, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= G)
                __hip_atomic_compare_exchange_strong(decision, &open, 1ull, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
            else if (wall_clock64() - t0 > p.start_ticks)
                __hip_atomic_compare_exchange_strong(decision, &open, 2ull, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
            else
                __builtin_amdgcn_s_sleep(8);
        }
        if (d == 2) __hip_atomic_store(p.abort, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        stop = d != 1;
    }
    __syncthreads();
    if (stop) return;
    auto rebuild = [&]() {
        if (threadIdx.x == 0) {
            int acc = 0;
            for (int k = 0; k < p.nsamples; k++) {
                aprefix[k] = acc;
                if (p.active[k]) acc += (int)((p.sample_n[k] + bs - 1) / bs);
            }
            aprefix[p.nsamples] = acc;
        }
        __syncthreads();
    };
    rebuild();
    for (int64_t t = 0; t < p.max_steps; t++) {
        const bool check = (t + 1) % p.check_every == 0 || t + 1 == p.max_steps;
        const int par = (p.cur0 + (int)(t & 1)) & 1;
        a.fin = p.f[par];
        a.fout = p.f[par ^ 1];
        a.it = t;
        a.write_macros = check ? 1 : 0;
        const int64_t total = aprefix[p.nsamples];
        const int64_t j0 = grp * total / ngrp, j1 = (grp + 1) * total / ngrp;
        unsigned long long* claim_cnt = p.bar + (17 + 2 * grp + (t & 1)) * BAR_STRIDE;
        // This step's counter was zeroed in the step before (or by the host);
        // the other parity's is zeroed now for the next step, by one block of
        // the group: the barrier at the end of this step orders that store
        // before any claim of the next step.
        if (slot == 0 && threadIdx.x == 0)
            __hip_atomic_store(p.bar + (17 + 2 * grp + ((t + 1) & 1)) * BAR_STRIDE, 0ull, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        const int64_t len = j1 - j0;
        if (threadIdx.x == 0)
            claim[0] = (int64_t)__hip_atomic_fetch_add(claim_cnt, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        int cs = 0;   // claim slot being processed
        int64_t mine = claim[0];
        int s = 0;
        while (mine < len) {
            // The other slot was last read before the previous barrier.
            if (threadIdx.x == 0)
                claim[cs ^ 1] = (int64_t)__hip_atomic_fetch_add(claim_cnt, 1ull, __ATOMIC_RELAXED,
                                                                __HIP_MEMORY_SCOPE_AGENT);
            const int64_t j = j0 + mine;
            while (aprefix[s + 1] <= j) s++;   // uniform per block; a block's claims only grow
            const int64_t chunk = ld_const(p.sample_off + s) / bs + (j - aprefix[s]);
            const int64_t i = chunk * bs + threadIdx.x;
            const bool live = i < ld_const(p.sample_end + s);
            if (live) {
                a.omega = ld_const(p.omega + s);
                a.gx = ld_const(p.gx + s);
                node_any<S, LAYOUT, IDX, true>(a, i, NO_FAULT);
            }
            if (check) {
                const double t_sum = block_sum_fixed(live ? a.macros[a.Npad + i] : 0.0, lds);
                if (threadIdx.x == 0) p.partial[chunk] = t_sum;
            }
            __syncthreads();   // the next claim has landed in LDS
            cs ^= 1;
            mine = claim[cs];
        }
        if (!grid_barrier(p, gen)) return;
        // Density guard: stop after the faulting step.  Only a fault of this
        // step or earlier counts: a faster block may already be in the next
        // step, and every block must leave at the same barrier.
        if (threadIdx.x == 0) {
            const unsigned long long fk = __hip_atomic_load(a.fault, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            stop = fk != NO_FAULT && (int64_t)(fk >> 32) <= t;
        }
        __syncthreads();
        if (stop) return;
        if (!check) continue;
        if (threadIdx.x < 64) {
            for (int64_t q = xcd_block(blockIdx.x, G); q < p.nsamples; q += G) {
                if (aprefix[q + 1] == aprefix[q]) continue;   // not running
                const double sum = wave_sum_chunks(p.partial, p.sample_off[q] / bs, (p.sample_n[q] + bs - 1) / bs);
                if (threadIdx.x == 0) {
                    const double mean = sum / (double)p.sample_n[q];
                    const double scale = fmax(fabs(mean), 1e-3 * fabs(p.gx[q]));
                    const double prev = p.prev[q];
                    p.steps[q] = t + 1;
                    p.cur[q] = par ^ 1;
                    if (!isnan(prev) && fabs(mean - prev) <= p.tol * scale) {
                        p.active[q] = 0;
                        __hip_atomic_fetch_add(p.n_active, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                    p.prev[q] = mean;
                }
            }
        }
        if (!grid_barrier(p, gen)) return;
        if (threadIdx.x == 0) stop = __hip_atomic_load(p.n_active, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
        __syncthreads();
        if (stop) return;
        rebuild();
    }
}

// ---------------------------------------------------------------- init / IO kernels
template <typename S, int LAYOUT>
__global__ void k_init_eq(void* f, int64_t N, int64_t Npad, double rho0)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= Npad) return;
#pragma unroll
    for (int j = 0; j < Q; j++) {
        const int64_t k = fpos<LAYOUT>(j, i, Npad);
        if constexpr (sizeof(S) == 8)
            ((double*)f)[k] = feq_ref(j, rho0, 0.0, 0.0, 0.0);  // init_dist_macro
        else if constexpr (sizeof(S) == 4)
            ((float*)f)[k] = 0.f;
        else
            ((__half*)f)[k] = __float2half(0.f);
    }
}

// AoS [n][19] FP64 in V order  <->  device layout.  `first` = first V-order
// node of the chunk, `n` nodes.
template <typename S, int LAYOUT>
__global__ void k_read_pop(const void* f, int64_t Npad, const uint32_t* inv_perm, int64_t first,
                           int64_t n, double rho0, float inv, double* out)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int64_t g = first + r;
    const int64_t k = inv_perm ? (int64_t)inv_perm[g] : g;
#pragma unroll
    for (int j = 0; j < Q; j++) {
        const int64_t p = fpos<LAYOUT>(j, k, Npad);
        double v;
        if constexpr (sizeof(S) == 8)
            v = ((const double*)f)[p];
        else if constexpr (sizeof(S) == 4)
            v = TP[j] * rho0 + (double)((const float*)f)[p];
        else
            v = TP[j] * rho0 + (double)(__half2float(((const __half*)f)[p]) * inv);
        out[r * Q + j] = v;
    }
}

template <typename S, int LAYOUT>
__global__ void k_write_pop(void* f, int64_t Npad, const uint32_t* inv_perm, int64_t first,
                            int64_t n, double rho0, float sc, const double* in)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int64_t g = first + r;
    const int64_t k = inv_perm ? (int64_t)inv_perm[g] : g;
#pragma unroll
    for (int j = 0; j < Q; j++) {
        const int64_t p = fpos<LAYOUT>(j, k, Npad);
        const double v = in[r * Q + j];
        if constexpr (sizeof(S) == 8)
            ((double*)f)[p] = v;
        else if constexpr (sizeof(S) == 4)
            ((float*)f)[p] = (float)(v - TP[j] * rho0);
        else
            ((__half*)f)[p] = __float2half_rn((float)(v - TP[j] * rho0) * sc);
    }
}

// Stored elements as they are, AoS [n][19] in V order <-> device layout
// (checkpoints: no conversion, so a written-back state is bit-identical).
template <typename S, int LAYOUT>
__global__ void k_copy_state(void* f, int64_t Npad, const uint32_t* inv_perm, int64_t first, int64_t n,
                             void* aos_bytes, int to_device)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int64_t g = first + r;
    const int64_t k = inv_perm ? (int64_t)inv_perm[g] : g;
    S* dev = (S*)f;
    S* aos = (S*)aos_bytes;
#pragma unroll
    for (int j = 0; j < Q; j++) {
        const int64_t p = fpos<LAYOUT>(j, k, Npad);
        if (to_device)
            dev[p] = aos[r * Q + j];
        else
            aos[r * Q + j] = dev[p];
    }
}

// The same three copies for a one-buffer AA lattice: population j of node k
// sits at out_pos<form>(k, j), form 1 or 2 (the step kernels' store map).
template <int LAYOUT, int IDX>
__device__ __forceinline__ void aa_positions(const StepArgs& a, int64_t k, int form, int64_t pos[Q]);

template <typename S, int LAYOUT, int IDX>
__global__ void k_read_pop_aa(const StepArgs a, int form, const uint32_t* inv_perm, int64_t first, int64_t n,
                              double rho0, float inv, double* out)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int64_t g = first + r;
    const int64_t k = inv_perm ? (int64_t)inv_perm[g] : g;
    int64_t pos[Q];
    aa_positions<LAYOUT, IDX>(a, k, form, pos);
#pragma unroll
    for (int j = 0; j < Q; j++) {
        double v;
        if constexpr (sizeof(S) == 8)
            v = ((const double*)a.fin)[pos[j]];
        else if constexpr (sizeof(S) == 4)
            v = TP[j] * rho0 + (double)((const float*)a.fin)[pos[j]];
        else
            v = TP[j] * rho0 + (double)(__half2float(((const __half*)a.fin)[pos[j]]) * inv);
        out[r * Q + j] = v;
    }
}

template <typename S, int LAYOUT, int IDX>
__global__ void k_write_pop_aa(const StepArgs a, int form, const uint32_t* inv_perm, int64_t first, int64_t n,
                               double rho0, float sc, const double* in)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int64_t g = first + r;
    const int64_t k = inv_perm ? (int64_t)inv_perm[g] : g;
    int64_t pos[Q];
    aa_positions<LAYOUT, IDX>(a, k, form, pos);
#pragma unroll
    for (int j = 0; j < Q; j++) {
        const double v = in[r * Q + j];
        if constexpr (sizeof(S) == 8)
            ((double*)a.fout)[pos[j]] = v;
        else if constexpr (sizeof(S) == 4)
            ((float*)a.fout)[pos[j]] = (float)(v - TP[j] * rho0);
        else
            ((__half*)a.fout)[pos[j]] = __float2half_rn((float)(v - TP[j] * rho0) * sc);
    }
}

template <typename S, int LAYOUT, int IDX>
__global__ void k_copy_state_aa(const StepArgs a, int form, const uint32_t* inv_perm, int64_t first, int64_t n,
                                void* aos_bytes, int to_device)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int64_t g = first + r;
    const int64_t k = inv_perm ? (int64_t)inv_perm[g] : g;
    int64_t pos[Q];
    aa_positions<LAYOUT, IDX>(a, k, form, pos);
    S* dev = (S*)a.fout;
    S* aos = (S*)aos_bytes;
#pragma unroll
    for (int j = 0; j < Q; j++) {
        if (to_device)
            dev[pos[j]] = aos[r * Q + j];
        else
            aos[r * Q + j] = dev[pos[j]];
    }
}

// out[q][r] = macro list.comp[q] of V-order node first + r.
__global__ void k_read_macros(const double* __restrict__ macros, int64_t Npad, const uint32_t* __restrict__ inv_perm,
                              int64_t first, int64_t n, MacroList list)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int64_t g = first + r;
    const int64_t k = inv_perm ? (int64_t)inv_perm[g] : g;
    for (int q = 0; q < list.n; q++) list.out[q][r] = macros[list.comp[q] * Npad + k];
}

template <int LAYOUT, int IDX>
__device__ __forceinline__ void aa_positions(const StepArgs& a, int64_t k, int form, int64_t pos[Q])
{
    if (form == 1) {
#pragma unroll
        for (int j = 0; j < Q; j++) pos[j] = out_pos<LAYOUT, 1>(a, k, nullptr, j);
    } else {
        int32_t t[Q];
        t[0] = 0;
        lane_sources<LAYOUT, IDX>(a, k, t);
#pragma unroll
        for (int j = 0; j < Q; j++) pos[j] = out_pos<LAYOUT, 2>(a, k, t, j);
    }
}

template <int LAYOUT, int IDX>
__global__ void k_read_table(const StepArgs a, const uint32_t* inv_perm, const uint32_t* perm,
                             int64_t first, int64_t n, int32_t* out)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int64_t g = first + r;
    const int64_t k = inv_perm ? (int64_t)inv_perm[g] : g;
    int32_t t[Q];
    lane_sources<LAYOUT, IDX>(a, k, t);
    for (int j = 1; j < Q; j++) {
        int32_t v = t[j];
        if (v >= 0 && perm) v = (int32_t)perm[v];
        out[(int64_t)(j - 1) * n + r] = v;
    }
}

// ---------------------------------------------------------------- FP64 reductions
constexpr int RED_T = 256;

// Block partial sums over nodes [first, first+n): mass (sum of the stored
// populations) and ux.
template <typename S, int LAYOUT>
__global__ void __launch_bounds__(RED_T)
k_reduce_partial(const void* f, const double* ux, int64_t first, int64_t n, int64_t Npad,
                 float inv, double* partial)
{
    __shared__ double sm[2][RED_T];
    double m = 0.0, s = 0.0;
    for (int64_t r = (int64_t)blockIdx.x * RED_T + threadIdx.x; r < n;
         r += (int64_t)gridDim.x * RED_T) {
        const int64_t i = first + r;
        double mi = 0.0;
#pragma unroll
        for (int j = 0; j < Q; j++) {
            const int64_t p = fpos<LAYOUT>(j, i, Npad);
            if constexpr (sizeof(S) == 8)
                mi += ((const double*)f)[p];
            else if constexpr (sizeof(S) == 4)
                mi += (double)((const float*)f)[p];
            else
                mi += (double)(__half2float(((const __half*)f)[p]) * inv);
        }
        m += mi;
        s += ux[i];
    }
    sm[0][threadIdx.x] = m;
    sm[1][threadIdx.x] = s;
    __syncthreads();
    for (int off = RED_T / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
            sm[0][threadIdx.x] += sm[0][threadIdx.x + off];
            sm[1][threadIdx.x] += sm[1][threadIdx.x + off];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        partial[2 * blockIdx.x] = sm[0][0];
        partial[2 * blockIdx.x + 1] = sm[1][0];
    }
}

// ---------------------------------------------------------------- per-sample u_x sums (batches)
// A sample's sum of u_x is formed in one fixed order by both batch drivers
// (one launch per step, and the persistent launch): per chunk (one block of
// the batch layout) a fixed tree over its nodes, then per sample the chunk
// partials, lane l of one wave taking chunks l, l+64, ... in turn, and a
// fixed butterfly over the 64 lanes.  Both drivers therefore see the same
// sums bit for bit and stop every sample at the same step.

// partial[chunk] = sum of ux over the chunk's nodes, for the listed chunks.
__global__ void __launch_bounds__(1024)
k_chunk_partials(const double* ux, const int32_t* chunks, const int32_t* chunk_sample,
                 const int64_t* sample_end, double* partial)
{
    __shared__ double lds[16];
    const int64_t chunk = chunks[blockIdx.x];
    const int64_t i = chunk * blockDim.x + threadIdx.x;
    const double v = i < sample_end[chunk_sample[chunk]] ? ux[i] : 0.0;
    const double t = block_sum_fixed(v, lds);
    if (threadIdx.x == 0) partial[chunk] = t;
}

// out[s] = sum of sample s's chunk partials (one wave per sample).
__global__ void __launch_bounds__(64)
k_sample_sums(const double* partial, const int64_t* off, const int64_t* n, int bs, double* out)
{
    const int s = blockIdx.x;
    const double t = wave_sum_chunks(partial, off[s] / bs, (n[s] + bs - 1) / bs);
    if (threadIdx.x == 0) out[s] = t;
}

// The sums, and the fault words when asked, go to page-locked memory: a copy
// back to the host takes 8 us more than the kernel's own stores.
__global__ void __launch_bounds__(RED_T)
k_reduce_final(const double* partial, int nb, double* sums, const unsigned long long* fault, HostWords* words)
{
    __shared__ double sm[2][RED_T];
    double m = 0.0, s = 0.0;
    for (int b = threadIdx.x; b < nb; b += RED_T) {
        m += partial[2 * b];
        s += partial[2 * b + 1];
    }
    sm[0][threadIdx.x] = m;
    sm[1][threadIdx.x] = s;
    __syncthreads();
    for (int off = RED_T / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
            sm[0][threadIdx.x] += sm[0][threadIdx.x + off];
            sm[1][threadIdx.x] += sm[1][threadIdx.x + off];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        sums[0] = sm[0][0];
        sums[1] = sm[1][0];
    }
    if (words && threadIdx.x < 2) words->fault[threadIdx.x] = fault[threadIdx.x];
}

__global__ void k_fault_words(const unsigned long long* fault, HostWords* words)
{
    if (threadIdx.x < 2) words->fault[threadIdx.x] = fault[threadIdx.x];
}

// ---------------------------------------------------------------- launchers
static unsigned nblk(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

#define PLB_DISPATCH(PREC, LAYOUT, KERNEL, ...)                                             \
    do {                                                                                    \
        if ((PREC) == PLB_FP64) {                                                           \
            if ((LAYOUT) == PLB_LAYOUT_SOA) hipLaunchKernelGGL((KERNEL<double, PLB_LAYOUT_SOA>), __VA_ARGS__); \
            else hipLaunchKernelGGL((KERNEL<double, PLB_LAYOUT_AOSOA>), __VA_ARGS__);        \
        } else if ((PREC) == PLB_FP32) {                                                    \
            if ((LAYOUT) == PLB_LAYOUT_SOA) hipLaunchKernelGGL((KERNEL<float, PLB_LAYOUT_SOA>), __VA_ARGS__); \
            else hipLaunchKernelGGL((KERNEL<float, PLB_LAYOUT_AOSOA>), __VA_ARGS__);         \
        } else {                                                                            \
            if ((LAYOUT) == PLB_LAYOUT_SOA) hipLaunchKernelGGL((KERNEL<__half, PLB_LAYOUT_SOA>), __VA_ARGS__); \
            else hipLaunchKernelGGL((KERNEL<__half, PLB_LAYOUT_AOSOA>), __VA_ARGS__);        \
        }                                                                                   \
    } while (0)

#define PLB_DISPATCH_ONE_IDX(PREC, LAYOUT, IDXC, KERNEL, ...)                                  \
    do {                                                                                        \
        if ((PREC) == PLB_FP64) {                                                               \
            if ((LAYOUT) == PLB_LAYOUT_SOA) hipLaunchKernelGGL((KERNEL<double, PLB_LAYOUT_SOA, IDXC>), __VA_ARGS__); \
            else hipLaunchKernelGGL((KERNEL<double, PLB_LAYOUT_AOSOA, IDXC>), __VA_ARGS__);      \
        } else if ((PREC) == PLB_FP32) {                                                        \
            if ((LAYOUT) == PLB_LAYOUT_SOA) hipLaunchKernelGGL((KERNEL<float, PLB_LAYOUT_SOA, IDXC>), __VA_ARGS__); \
            else hipLaunchKernelGGL((KERNEL<float, PLB_LAYOUT_AOSOA, IDXC>), __VA_ARGS__);       \
        } else {                                                                                \
            if ((LAYOUT) == PLB_LAYOUT_SOA) hipLaunchKernelGGL((KERNEL<__half, PLB_LAYOUT_SOA, IDXC>), __VA_ARGS__); \
            else hipLaunchKernelGGL((KERNEL<__half, PLB_LAYOUT_AOSOA, IDXC>), __VA_ARGS__);      \
        }                                                                                       \
    } while (0)

// All three index kinds (single lattice).
#define PLB_DISPATCH3(PREC, LAYOUT, IDX, KERNEL, ...)                                         \
    do {                                                                                      \
        if ((IDX) == PLB_INDEX_I32) PLB_DISPATCH_ONE_IDX(PREC, LAYOUT, PLB_INDEX_I32, KERNEL, __VA_ARGS__); \
        else if ((IDX) == PLB_INDEX_TILE8) PLB_DISPATCH_ONE_IDX(PREC, LAYOUT, PLB_INDEX_TILE8, KERNEL, __VA_ARGS__); \
        else PLB_DISPATCH_ONE_IDX(PREC, LAYOUT, PLB_INDEX_BITMAP, KERNEL, __VA_ARGS__);        \
    } while (0)

// Table index kinds only (batches of samples).
#define PLB_DISPATCH2(PREC, LAYOUT, IDX, KERNEL, ...)                                         \
    do {                                                                                      \
        if ((IDX) == PLB_INDEX_I32) PLB_DISPATCH_ONE_IDX(PREC, LAYOUT, PLB_INDEX_I32, KERNEL, __VA_ARGS__); \
        else PLB_DISPATCH_ONE_IDX(PREC, LAYOUT, PLB_INDEX_TILE8, KERNEL, __VA_ARGS__);         \
    } while (0)

StepArgs make_args(plb_ctx* c, int64_t it, bool write_macros)
{
    StepArgs a;
    a.fin = c->f[c->cur];
    a.fout = c->f[c->cur ^ 1];
    a.tab = c->tab;
    a.tdesc = c->tdesc;
    a.toff = c->toff;
    a.toff16 = c->toff16;
    a.twide = c->twide;
    a.N = c->N;
    a.Npad = c->Npad;
    a.omega = c->omega;
    a.gx = c->cfg.gx;
    a.rho0 = c->cfg.rho0;
    a.it = it;
    a.write_macros = write_macros ? 1 : 0;
    a.macros = c->macros;
    a.fault = c->fault;
    a.perm = c->perm;
    a.scale = c->scale;
    a.inv_scale = c->inv_scale;
    a.bm = c->bm;
    a.vox = c->vox;
    a.nx = (uint32_t)c->nx;
    a.ny = (uint32_t)c->ny;
    a.nz = (uint32_t)c->nz;
    a.py = (uint32_t)(c->py > 0 ? c->py : c->ny);
    a.div_nx = make_fastdiv(a.nx);
    a.div_py = make_fastdiv(a.py);
    a.div_nz = make_fastdiv(a.nz);
    a.it_base = nullptr;
    a.stochastic = c->cfg.precision == PLB_FP16 && c->cfg.fp16_rounding == PLB_ROUND_STOCHASTIC;
    a.key_perm = c->key_perm ? c->key_perm : c->perm;
    a.kseg = c->kseg;
    a.has_const = c->cfg.bb_mode == PLB_BB_REFCOMPAT;
    return a;
}

// Dynamic LDS per block that caps the step kernel at cfg.waves_per_simd waves
// per SIMD (the kernel itself uses no LDS): with w waves on each of a CU's 4
// SIMDs the CU holds 4*w*64/bs blocks, so each block reserves that share of
// the CU's LDS, rounded down to 512 bytes (at most 64 KB).  0 = no cap.
static unsigned step_lds_bytes(const plb_ctx* c, int bs)
{
    const int w = c->cfg.waves_per_simd;
    if (w <= 0 || w >= 8 || c->lds_per_cu <= 0) return 0u;
    const int blocks = std::max(1, 4 * w * 64 / bs);
    const long share = std::min<long>(65536, (long)c->lds_per_cu / blocks);
    return (unsigned)(share / 512 * 512);
}

// Groups of 16 whose stores are plain; 0: k_step.
static int keep_stores(const plb_ctx* c)
{
    const double bytes = (2.0 * Q * c->elem + c->index_bytes) * (double)c->N;
    if (c->cfg.precision == PLB_FP16 || bytes <= KEEP_ABOVE || bytes > KEEP_MOST) return 0;
    return bytes <= KEEP_ALL ? 16 : (int)(16.0 * KEEP_BYTES / bytes + 0.5);
}

static void launch_keep(const plb_ctx* c, const StepArgs& a, int keep, dim3 grid, dim3 block, unsigned lds)
{
    auto run = [&](auto* kern) { hipLaunchKernelGGL(kern, grid, block, lds, c->stream, a, keep); };
    auto with = [&](auto layout, auto idx) {
        constexpr int L = decltype(layout)::value, I = decltype(idx)::value;
        c->cfg.precision == PLB_FP64 ? run(k_step_keep<double, L, I>) : run(k_step_keep<float, L, I>);
    };
    auto with_idx = [&](auto layout) {
        if (c->cfg.index_kind == PLB_INDEX_I32) with(layout, std::integral_constant<int, PLB_INDEX_I32>{});
        else if (c->cfg.index_kind == PLB_INDEX_TILE8) with(layout, std::integral_constant<int, PLB_INDEX_TILE8>{});
        else with(layout, std::integral_constant<int, PLB_INDEX_BITMAP>{});
    };
    if (c->cfg.layout == PLB_LAYOUT_SOA) with_idx(std::integral_constant<int, PLB_LAYOUT_SOA>{});
    else with_idx(std::integral_constant<int, PLB_LAYOUT_AOSOA>{});
}

int launch_step(plb_ctx* c, int64_t it, bool write_macros, const int64_t* it_base)
{
    if (c->N == 0) {  // a mask without pores: nothing to update
        c->cur ^= 1;
        return PLB_OK;
    }
    StepArgs a = make_args(c, it, write_macros);
    a.it_base = it_base;
    const int bs = c->cfg.block_size;
    const unsigned lds = step_lds_bytes(c, bs);
    if (c->cfg.stream_mode == PLB_STREAM_AA) {
        // one buffer: c->cur 1 = local-step store form (a neighbour step
        // next), 0 = neighbour-step store form (a local step next)
        if (c->cur == 0)
            PLB_DISPATCH_ONE_IDX(c->cfg.precision, c->cfg.layout, PLB_INDEX_I32, k_step_aa_even,
                                 dim3(nblk(c->N, bs)), dim3(bs), lds, c->stream, a);
        else
            PLB_DISPATCH3(c->cfg.precision, c->cfg.layout, c->cfg.index_kind, k_step_aa_odd, dim3(nblk(c->N, bs)),
                          dim3(bs), lds, c->stream, a);
    } else if (c->cfg.nodes_per_thread == 2) {
        const int64_t threads = (c->N + 127) / 128 * 64;
        PLB_DISPATCH3(c->cfg.precision, c->cfg.layout, c->cfg.index_kind, k_step2,
                      dim3(nblk(threads, bs)), dim3(bs), lds, c->stream, a);
    } else if (const int keep = keep_stores(c)) {
        launch_keep(c, a, keep, dim3(nblk(c->N, bs)), dim3(bs), lds);
    } else {
        PLB_DISPATCH3(c->cfg.precision, c->cfg.layout, c->cfg.index_kind, k_step, dim3(nblk(c->N, bs)),
                      dim3(bs), lds, c->stream, a);
    }
    PLB_HIP(hipGetLastError());
    c->cur ^= 1;
    return PLB_OK;
}

__global__ void k_set_step(int64_t* it_dev, int64_t it)
{
    if (threadIdx.x == 0) *it_dev = it;
}

// G steps (G even, so the buffers end where they started) from a graph
// captured once per starting buffer.  The step number is not baked into the
// graph: every kernel adds *it_dev, which a plain launch sets before each
// replay.  The graph holds kernel nodes only.
int launch_graph_steps(plb_ctx* c, int64_t it0, int64_t G)
{
    hipStream_t s = c->stream;
    const int p = c->cur;
    if (!c->gexec[p]) {
        PLB_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        int rc = PLB_OK;
        for (int64_t k = 0; k < G && rc == PLB_OK; k++) rc = launch_step(c, k, false, c->it_dev);
        hipGraph_t g = nullptr;
        const hipError_t e = hipStreamEndCapture(s, &g);
        c->cur = p;  // capture does not run anything
        if (rc) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        PLB_HIP(e);
        const hipError_t ei = hipGraphInstantiate(&c->gexec[p], g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        PLB_HIP(ei);
    }
    hipLaunchKernelGGL(k_set_step, dim3(1), dim3(64), 0, s, c->it_dev, it0);
    PLB_HIP(hipGetLastError());
    PLB_HIP(hipGraphLaunch(c->gexec[p], s));
    return PLB_OK;
}

// One step over the active blocks of a batch (the context holds the
// concatenated samples; c->omega / c->cfg.gx are unused).
int launch_step_batch(plb_ctx* c, int64_t it, bool write_macros, const int32_t* active,
                      int n_active, const int32_t* block_sample, const int64_t* sample_end,
                      const double* omega, const double* gx)
{
    if (n_active > 0) {
        const StepArgs a = make_args(c, it, write_macros);
        BatchArgs b;
        b.active = active;
        b.block_sample = block_sample;
        b.sample_end = sample_end;
        b.omega = omega;
        b.gx = gx;
        PLB_DISPATCH2(c->cfg.precision, c->cfg.layout, c->cfg.index_kind, k_step_batch,
                      dim3(n_active), dim3(c->cfg.block_size), step_lds_bytes(c, c->cfg.block_size),
                      c->stream, a, b);
        PLB_HIP(hipGetLastError());
    }
    c->cur ^= 1;
    return PLB_OK;
}


// The persistent batch run as one cooperative launch of as many blocks as can
// be resident at once (at most one per chunk).  *blocks = the grid size.
template <typename S, int LAYOUT, int IDX>
static int launch_persistent_t(plb_ctx* c, const PersistArgs& p, int max_blocks, int* blocks)
{
    auto kern = k_batch_persistent<S, LAYOUT, IDX>;
    const int bs = c->cfg.block_size;
    // The wave cap's LDS share per block, less what the kernel holds itself.
    hipFuncAttributes fa;
    PLB_HIP(hipFuncGetAttributes(&fa, (const void*)kern));
    unsigned lds = step_lds_bytes(c, bs);
    lds = lds > fa.sharedSizeBytes ? (unsigned)((lds - fa.sharedSizeBytes) / 512 * 512) : 0u;
    int per_cu = 0, cus = 0;
    PLB_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, bs, lds));
    PLB_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
    // One block per CU below the computed residency: a grid at exactly the
    // computed limit waited at its first barrier for blocks that never
    // started (the limit is an estimate; the bounded wait reported it).
    if (per_cu > 1) per_cu--;
    int64_t g = std::min<int64_t>((int64_t)per_cu * cus, p.nchunks);
    if (max_blocks > 0) g = std::min<int64_t>(g, max_blocks);
    if (g < 1) return PLB_ERR_INVALID;
    StepArgs a = make_args(c, 0, false);
    PersistArgs pp = p;
    void* args[] = {(void*)&a, (void*)&pp};
    PLB_HIP(hipLaunchCooperativeKernel((const void*)kern, dim3((unsigned)g), dim3(bs), args, lds, c->stream));
    *blocks = (int)g;
    return PLB_OK;
}

int launch_batch_persistent(plb_ctx* c, const PersistArgs& p, int max_blocks, int* blocks)
{
    const int pr = c->cfg.precision, lay = c->cfg.layout, idx = c->cfg.index_kind;
#define PLB_PERSIST(ST, L, I) if (pr == (sizeof(ST) == 8 ? PLB_FP64 : sizeof(ST) == 4 ? PLB_FP32 : PLB_FP16) && lay == L && idx == I) return launch_persistent_t<ST, L, I>(c, p, max_blocks, blocks)
    PLB_PERSIST(double, PLB_LAYOUT_SOA, PLB_INDEX_I32);
    PLB_PERSIST(double, PLB_LAYOUT_SOA, PLB_INDEX_TILE8);
    PLB_PERSIST(double, PLB_LAYOUT_AOSOA, PLB_INDEX_I32);
    PLB_PERSIST(double, PLB_LAYOUT_AOSOA, PLB_INDEX_TILE8);
    PLB_PERSIST(float, PLB_LAYOUT_SOA, PLB_INDEX_I32);
    PLB_PERSIST(float, PLB_LAYOUT_SOA, PLB_INDEX_TILE8);
    PLB_PERSIST(float, PLB_LAYOUT_AOSOA, PLB_INDEX_I32);
    PLB_PERSIST(float, PLB_LAYOUT_AOSOA, PLB_INDEX_TILE8);
    PLB_PERSIST(__half, PLB_LAYOUT_SOA, PLB_INDEX_I32);
    PLB_PERSIST(__half, PLB_LAYOUT_SOA, PLB_INDEX_TILE8);
    PLB_PERSIST(__half, PLB_LAYOUT_AOSOA, PLB_INDEX_I32);
    PLB_PERSIST(__half, PLB_LAYOUT_AOSOA, PLB_INDEX_TILE8);
#undef PLB_PERSIST
    return PLB_ERR_INVALID;
}

int launch_init_eq(plb_ctx* c)
{
    for (int b = 0; b < 2; b++)
        PLB_DISPATCH(c->cfg.precision, c->cfg.layout, k_init_eq, dim3(nblk(c->Npad, 256)), dim3(256),
                     0, c->stream, c->f[b], c->N, c->Npad, c->cfg.rho0);
    PLB_HIP(hipGetLastError());
    return PLB_OK;
}

int launch_read_pop(plb_ctx* c, int64_t first, int64_t n, double* dout)
{
    if (c->cfg.stream_mode == PLB_STREAM_AA) {
        PLB_DISPATCH3(c->cfg.precision, c->cfg.layout, c->cfg.index_kind, k_read_pop_aa, dim3(nblk(n, 256)),
                      dim3(256), 0, c->stream, make_args(c, 0, false), c->cur == 1 ? 1 : 2, c->inv_perm, first, n,
                      c->cfg.rho0, c->inv_scale, dout);
        PLB_HIP(hipGetLastError());
        return PLB_OK;
    }
    PLB_DISPATCH(c->cfg.precision, c->cfg.layout, k_read_pop, dim3(nblk(n, 256)), dim3(256), 0,
                 c->stream, c->f[c->cur], c->Npad, c->inv_perm, first, n, c->cfg.rho0,
                 c->inv_scale, dout);
    PLB_HIP(hipGetLastError());
    return PLB_OK;
}

int launch_write_pop(plb_ctx* c, int64_t first, int64_t n, const double* din)
{
    if (c->cfg.stream_mode == PLB_STREAM_AA) {
        PLB_DISPATCH3(c->cfg.precision, c->cfg.layout, c->cfg.index_kind, k_write_pop_aa, dim3(nblk(n, 256)),
                      dim3(256), 0, c->stream, make_args(c, 0, false), c->cur == 1 ? 1 : 2, c->inv_perm, first, n,
                      c->cfg.rho0, c->scale, din);
        PLB_HIP(hipGetLastError());
        return PLB_OK;
    }
    PLB_DISPATCH(c->cfg.precision, c->cfg.layout, k_write_pop, dim3(nblk(n, 256)), dim3(256), 0,
                 c->stream, c->f[c->cur], c->Npad, c->inv_perm, first, n, c->cfg.rho0, c->scale,
                 din);
    PLB_HIP(hipGetLastError());
    return PLB_OK;
}

int launch_copy_state(plb_ctx* c, int64_t first, int64_t n, void* aos, bool to_device)
{
    if (c->cfg.stream_mode == PLB_STREAM_AA) {
        PLB_DISPATCH3(c->cfg.precision, c->cfg.layout, c->cfg.index_kind, k_copy_state_aa, dim3(nblk(n, 256)),
                      dim3(256), 0, c->stream, make_args(c, 0, false), c->cur == 1 ? 1 : 2, c->inv_perm, first, n,
                      aos, to_device ? 1 : 0);
        PLB_HIP(hipGetLastError());
        return PLB_OK;
    }
    PLB_DISPATCH(c->cfg.precision, c->cfg.layout, k_copy_state, dim3(nblk(n, 256)), dim3(256), 0,
                 c->stream, c->f[c->cur], c->Npad, c->inv_perm, first, n, aos, to_device ? 1 : 0);
    PLB_HIP(hipGetLastError());
    return PLB_OK;
}

int launch_read_macros(plb_ctx* c, const MacroList& list, int64_t first, int64_t n)
{
    hipLaunchKernelGGL(k_read_macros, dim3(nblk(n, 256)), dim3(256), 0, c->stream, c->macros, c->Npad, c->inv_perm,
                       first, n, list);
    PLB_HIP(hipGetLastError());
    return PLB_OK;
}

#define PLB_READ_TABLE(LAYOUT, IDXC)                                                       \
    hipLaunchKernelGGL((k_read_table<LAYOUT, IDXC>), g, b, 0, c->stream, a, c->inv_perm, c->perm, \
                       first, n, dout)

int launch_read_table(plb_ctx* c, int64_t first, int64_t n, int32_t* dout)
{
    const StepArgs a = make_args(c, 0, false);
    const dim3 g(nblk(n, 256)), b(256);
    const int idx = c->cfg.index_kind;
    if (c->cfg.layout == PLB_LAYOUT_SOA) {
        if (idx == PLB_INDEX_TILE8) PLB_READ_TABLE(PLB_LAYOUT_SOA, PLB_INDEX_TILE8);
        else if (idx == PLB_INDEX_BITMAP) PLB_READ_TABLE(PLB_LAYOUT_SOA, PLB_INDEX_BITMAP);
        else PLB_READ_TABLE(PLB_LAYOUT_SOA, PLB_INDEX_I32);
    } else {
        if (idx == PLB_INDEX_TILE8) PLB_READ_TABLE(PLB_LAYOUT_AOSOA, PLB_INDEX_TILE8);
        else if (idx == PLB_INDEX_BITMAP) PLB_READ_TABLE(PLB_LAYOUT_AOSOA, PLB_INDEX_BITMAP);
        else PLB_READ_TABLE(PLB_LAYOUT_AOSOA, PLB_INDEX_I32);
    }
    PLB_HIP(hipGetLastError());
    return PLB_OK;
}

// Enqueues sums[0] = sum of stored populations (raw for FP64, deviations
// otherwise) over nodes [first, first+n) of buffer `buf`, sums[1] = sum of ux
// macros; sums and words (null: none) are page-locked.  Deterministic: fixed
// grid, fixed tree order.
int launch_reduce_range(plb_ctx* c, int buf, int64_t first, int64_t n, double* sums, HostWords* words)
{
    const int nb = std::max(1, std::min<int>(c->red_blocks, (int)((n + RED_T - 1) / RED_T)));
    PLB_DISPATCH(c->cfg.precision, c->cfg.layout, k_reduce_partial, dim3(nb), dim3(RED_T), 0,
                 c->stream, c->f[buf], c->macros + c->Npad, first, n, c->Npad, c->inv_scale, c->red);
    hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(RED_T), 0, c->stream, c->red, nb, sums, c->fault, words);
    PLB_HIP(hipGetLastError());
    return PLB_OK;
}

int launch_reduce(plb_ctx* c)
{
    return launch_reduce_range(c, c->cur, 0, c->N, c->host->sum, c->host);
}

int launch_fault_words(plb_ctx* c)
{
    hipLaunchKernelGGL(k_fault_words, dim3(1), dim3(64), 0, c->stream, c->fault, c->host);
    PLB_HIP(hipGetLastError());
    return PLB_OK;
}

int launch_sample_sums(plb_ctx* c, const int32_t* d_active, int n_active, const int32_t* chunk_sample,
                       const int64_t* sample_end, const int64_t* d_off, const int64_t* d_n, int nsamples,
                       double* d_partial, double* d_out)
{
    if (n_active > 0)
        hipLaunchKernelGGL(k_chunk_partials, dim3(n_active), dim3(c->cfg.block_size), 0, c->stream,
                           c->macros + c->Npad, d_active, chunk_sample, sample_end, d_partial);
    hipLaunchKernelGGL(k_sample_sums, dim3(nsamples), dim3(64), 0, c->stream, d_partial, d_off, d_n,
                       c->cfg.block_size, d_out);
    PLB_HIP(hipGetLastError());
    return PLB_OK;
}

}  // namespace plb
