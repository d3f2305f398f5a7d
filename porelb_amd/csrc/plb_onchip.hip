// plb_onchip.hip -- many time steps of a small lattice in one launch, with the
// populations held in the CUs' LDS.
//
// One launch per step costs a small lattice the launch gap (2.6 us) and one
// load -> gather -> store latency chain per step, whatever its size, and its
// populations cross the L2s every step.  Here every CU keeps one block of
// nodes for the whole run: a step reads and writes LDS, and only the links
// between blocks go through memory.
//
// Blocks.  The pore nodes are cut into slabs, rows and G <= CUs compact blocks of
// equal size, at most NS node slots each.  Inside
// a block, the nodes with a link to another block are dealt out evenly to the
// waves' first groups of 64 slots, and the others fill up; both in V order
// (short runs along x, which keep the LDS gathers nearly free of bank
// conflicts).  LDS holds the post-collision populations as F[slot][j]: the
// row length 19 is odd, so neighbouring slots' populations of one direction lie
// in different banks, and a node's 19 stores share one address register.
//
// Links.  idx holds, per node and direction, the LDS position the population
// is pulled from: the upstream node's row; the node's own cell re[j] for a
// bounce; a constant cell (reference bounce order); and again the node's own
// cell re[j] for a link from another block -- that slot's value has left for the
// other block, and no node of this block reads it, so the incoming value takes
// its place.  An exchange entry therefore is one LDS cell, the place of its
// value in the partner's receive buffer, and its own place in this block's.
// Links between blocks are always exchanged both ways (in the reference bounce
// order one way may be unused and is dropped on arrival), so no block can be
// more than one step ahead of a neighbour and two receive buffers, used by
// turns, are enough.
//
// Exchange.  A value travels with the step's number in one word that is stored
// and loaded as one atomic (FP32: 8 bytes, FP64: two halves of 8 bytes, FP16: 4
// bytes), and the receiver polls that word: no flag, no fence, one trip through
// memory (0.9 us per round between 256 blocks, against 5.1 us for a grid barrier
// with agent fences).  Where a thread has two nodes, the block's shared nodes are
// the first ones if they are no more than the threads, and their values leave
// before the second ones are updated, so the trip overlaps that update.  The
// entries of a wave are ordered by the wave at the other end, the same way on
// both sides, so a row of 64 words leaves as a few stretches and not as 64
// partial cache lines: 4.5 -> 4.0 us a step for 91 750 FP64 nodes, 4.9 -> 4.0 for
// 265 421 FP32 ones, 3.2 -> 2.7 for 8 064 FP64 ones.  (Entry lists of a whole
// block, dealt out to its waves: fewer pieces, but a second block barrier and
// sends that wait for the slowest wave; 2.8, 4.7 and 4.6 us.)
//
// Ends.  Blocks wait for each other, so the launch is cooperative, and every
// wait is bounded: a block that waits too long (50 ms for the first exchange,
// 2 s later) names the run in fault[1], holds all queued work off (HOLD_FAULT) and
// every block leaves.  The state before the run is in the other buffer, and
// plb_sync repeats the run with one launch per step; it does the same after a
// density-guard trip, since blocks far from the tripping node go on.
#include <stdio.h>

#include <algorithm>
#include <cmath>
#include <utility>

#include "plb_device.hpp"

namespace plb {

// One lattice, or one sample of a batch: its nodes and its share of the blocks.
struct OnchipSample {
    int64_t off, n;        // internal ids off .. off + n
    int64_t rank0;         // its nodes' numbers within the plan, rank0 .. rank0 + n
    int64_t word0, words;  // its bitmask
    int32_t d[3];          // voxels along x, y, z
    int32_t block0, nblocks;
    int32_t slabs, rows;   // cuts along z, and of each slab along y
};

struct OnchipPlan {
    int G = 0, NS = 0, T = 0, K = 0;
    bool twice = false;
    int64_t E = 0;
    void* fixed = nullptr;     // arrays whose size is known before the links are counted
    void* exchange = nullptr;  // per-entry arrays and the receive buffers
    uint32_t *node = nullptr, *idx = nullptr, *seg = nullptr, *ent_lds = nullptr, *ent_dst = nullptr;
    int32_t* blk_sample = nullptr;
    void* recv = nullptr;
    size_t recv_bytes = 0;
    std::vector<OnchipSample> samples;
    double* macros_own = nullptr;  // a second macros array; runs write the two by turns
    double* macros_alt = nullptr;  // the one the next run writes
    uint32_t tag = 16;     // step number the next run starts with
    uint32_t serial = 0;   // of the last run
};

constexpr uint32_t EMPTY = 0xffffffffu;
// Cells behind the NS rows of F: the constants of directions 1..6 and 7..18,
// and one that takes what is dropped on arrival.
constexpr int EXTRA = 3, DROP = 2;
// Directions come in pairs: 1, 2 | 3, 4 | ...
__device__ __forceinline__ uint32_t opposite(uint32_t j) { return ((j - 1u) ^ 1u) + 1u; }

// ---------------------------------------------------------------- plan
// The voxels that a slab's, or a row's, nodes span.
struct OnchipBox {
    int32_t lo[3], hi[3];
};

// The plan numbers the nodes of the samples that it holds, one after the other
// ("number" below; for one lattice, its internal ids), so that its scratch, 230
// bytes a node, is not taken for a batch's samples that do not fit the chip.
struct OnchipBuild {
    const OnchipSample* samples;
    int nsamples;
    int64_t Ntot;               // numbers
    const uint64_t* xyz;
    const uint32_t* xyz_of;     // xyz is in V order: V id of an internal id (batches); null: by internal id
    const uint32_t* vid;        // V id of an internal id; null: identity
    const uint32_t* node_of_v;  // its inverse
    unsigned long long* bits;
    uint32_t* wpre;
    uint16_t* group;            // slab, then row, of a number within its sample
    OnchipBox* box;             // [2][G] of the slabs and the rows
    uint32_t* base;             // [2][G] first bit of each
    uint32_t* order;            // rank -> number
    uint16_t* blk;              // number -> block
    uint32_t* slot_of;          // number -> block * NS + slot
    int32_t* T;                 // [18][Ntot] pull sources
    uint32_t* M;                // [18][Ntot] node that pulls population re[j]
    uint32_t* at;               // [18][Ntot] the shared link's entry
    const int32_t* block_sample;
    int* err;                   // the table is not that of a lattice (records that contradict each other)
    uint32_t* cnt;              // entries per group of 64 slots
    uint32_t *node, *idx, *seg, *ent_lds, *ent_dst;
    int G, NS;
};

__device__ __forceinline__ int sample_of(const OnchipBuild& b, int64_t k)
{
    int lo = 0, hi = b.nsamples - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (b.samples[mid].rank0 <= k) lo = mid;
        else hi = mid - 1;
    }
    return lo;   // the last that starts at k or before: those that the plan does not hold are empty
}
__device__ __forceinline__ int64_t id_of(const OnchipSample& s, int64_t k) { return s.off + (k - s.rank0); }
__device__ __forceinline__ int64_t number_of(const OnchipSample& s, int64_t id) { return s.rank0 + (id - s.off); }
__device__ __forceinline__ uint64_t coordinates(const OnchipBuild& b, const OnchipSample& s, int64_t k)
{
    const int64_t id = id_of(s, k);
    return b.xyz[b.xyz_of ? (int64_t)b.xyz_of[id] : id];
}

// Partition.  The nodes are cut by rank, three times: along z into slabs, each
// slab along y into rows, each row along x into blocks, all of equal size and
// nearly cubic.  A rank is the number of pores before a node in a bitmask whose
// order is (z, y, x) for the slabs, (y, z, x) within each slab's box for the
// rows and (x, z, y) within each row's box for the blocks.  (Equal cuts of one
// Morton curve have 13 to 23 percent more links between blocks, and the largest
// block 8 to 19 percent more: 4.0 us a step against 3.6 here for 91 750 FP64 nodes,
// 6.1 against 5.1 for 421 478 FP32 ones of a sphere pack.)
// Bit of node k in the bitmask of LEVEL 0, 1 or 2; -1 outside the lattice's box,
// or the bitmask (where records share a voxel, the ranks do not fit the boxes).
template <int LEVEL>
__device__ __forceinline__ int64_t bit_of(const OnchipBuild& b, const OnchipSample& s, int64_t k)
{
    const uint64_t p = coordinates(b, s, k);
    const int c[3] = {(int)(p & 0xffff), (int)((p >> 16) & 0xffff), (int)((p >> 32) & 0xffff)};
    if (c[0] >= s.d[0] || c[1] >= s.d[1] || c[2] >= s.d[2]) return -1;
    if constexpr (LEVEL == 0) return s.word0 * 64 + ((int64_t)c[2] * s.d[1] + c[1]) * s.d[0] + c[0];
    else {
        constexpr int A = LEVEL == 1 ? 1 : 0, C = LEVEL == 1 ? 0 : 1;   // slowest and fastest axis; z between them
        const int64_t g = (int64_t)(LEVEL - 1) * b.G + s.block0 + b.group[k];
        const OnchipBox& o = b.box[g];
        const int64_t m = (int64_t)b.base[g] +
                          ((int64_t)(c[A] - o.lo[A]) * (o.hi[2] - o.lo[2] + 1) + (c[2] - o.lo[2])) * (o.hi[C] - o.lo[C] + 1) +
                          (c[C] - o.lo[C]);
        return m >= 0 && m < s.words * 64 ? s.word0 * 64 + m : -1;
    }
}

template <int LEVEL>
__global__ void k_onchip_bits(const OnchipBuild b)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= b.Ntot) return;
    const int64_t m = bit_of<LEVEL>(b, b.samples[sample_of(b, k)], k);
    const unsigned long long bit = 1ull << (m & 63);
    // two records with the same coordinates, or some outside the box
    if (m < 0 || (atomicOr(b.bits + (m >> 6), bit) & bit)) *b.err = 1;
}

// Exclusive scan of n values by one block, from `carry` on (out[n] = the total
// when asked): a few thousand to a few hundred thousand values, not worth
// several launches and their allocations.
template <typename In>
__device__ __forceinline__ void block_scan(In in, uint32_t* out, int64_t n, uint32_t carry, bool total_too)
{
    constexpr int PER = 8;
    __shared__ uint32_t wsum[16];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    for (int64_t b = 0; b < n; b += 1024 * PER) {
        uint32_t v[PER], sum = 0;
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int64_t i = b + (int64_t)tid * PER + k;
            v[k] = i < n ? in(i) : 0u;
            sum += v[k];
        }
        uint32_t inc = sum;
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            const uint32_t t = __shfl_up(inc, m, 64);
            if (lane >= m) inc += t;
        }
        if (lane == 63) wsum[w] = inc;
        __syncthreads();
        uint32_t before = 0, total = 0;
        for (int q = 0; q < 16; q++) {
            if (q < w) before += wsum[q];
            total += wsum[q];
        }
        uint32_t e = carry + before + inc - sum;
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int64_t i = b + (int64_t)tid * PER + k;
            if (i < n) out[i] = e;
            e += v[k];
        }
        carry += total;
        __syncthreads();
    }
    if (total_too && tid == 0) out[n] = carry;
}

// Pores before each word of a sample's bitmask, one block per sample.
__global__ void __launch_bounds__(1024) k_onchip_words(const OnchipBuild b)
{
    const OnchipSample s = b.samples[blockIdx.x];
    const unsigned long long* const bits = b.bits + s.word0;
    block_scan([&](int64_t i) { return (uint32_t)__popcll(bits[i]); }, b.wpre + s.word0, s.words, (uint32_t)s.rank0, false);
}

__global__ void __launch_bounds__(1024) k_onchip_segs(const OnchipBuild b, int64_t groups)
{
    block_scan([&](int64_t i) { return b.cnt[i]; }, b.seg, groups, 0u, true);
}

// First bit of the boxes of LEVEL 0's slabs or 1's rows, one block per sample.
template <int LEVEL>
__global__ void __launch_bounds__(1024) k_onchip_boxes(const OnchipBuild b)
{
    const OnchipSample s = b.samples[blockIdx.x];
    const int64_t g0 = (int64_t)LEVEL * b.G + s.block0;
    block_scan(
        [&](int64_t i) {
            const OnchipBox o = b.box[g0 + i];
            uint32_t n = 1;
            for (int d = 0; d < 3; d++) n *= o.hi[d] < o.lo[d] ? 0u : (uint32_t)(o.hi[d] - o.lo[d] + 1);
            return n;
        },
        b.base + g0, s.nblocks ? s.slabs * (LEVEL ? s.rows : 1) : 0, 0u, false);
}

template <int LEVEL>
__global__ void k_onchip_rank(const OnchipBuild b)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= b.Ntot) return;
    const OnchipSample s = b.samples[sample_of(b, k)];
    const int64_t m = bit_of<LEVEL>(b, s, k);
    if (m < 0) return;
    const int64_t r = (int64_t)b.wpre[m >> 6] + __popcll(b.bits[m >> 6] & ((1ull << (m & 63)) - 1ull));
    auto block = [&](int64_t rank) { return (int)((rank - s.rank0) * s.nblocks / s.n); };
    if constexpr (LEVEL == 2) {
        b.order[r] = (uint32_t)k;
        b.blk[k] = (uint16_t)(s.block0 + block(r));
    } else {
        // slab g has the blocks from nblocks * g / slabs on, and so have its rows
        auto group = [&](int64_t rank) {
            const int blk = block(rank), slab = ((blk + 1) * s.slabs - 1) / s.nblocks;
            if constexpr (LEVEL == 0) return slab;
            const int b0 = s.nblocks * slab / s.slabs, n = s.nblocks * (slab + 1) / s.slabs - b0;
            return slab * s.rows + ((blk - b0 + 1) * s.rows - 1) / n;
        };
        const int g = group(r);
        // Its box, from its first and its last node; the slab's along z, all of it along x.
        OnchipBox& o = b.box[(int64_t)LEVEL * b.G + s.block0 + g];
        const OnchipBox& slab = b.box[s.block0 + (LEVEL ? b.group[k] : 0)];
        const uint64_t p = coordinates(b, s, k);
        const int y = (int)((p >> 16) & 0xffff), z = (int)((p >> 32) & 0xffff);
        if (r == s.rank0 || group(r - 1) != g) {
            o.lo[0] = 0;
            o.lo[1] = LEVEL ? y : 0;
            o.lo[2] = LEVEL ? slab.lo[2] : z;
        }
        if (r == s.rank0 + s.n - 1 || group(r + 1) != g) {
            o.hi[0] = s.d[0] - 1;
            o.hi[1] = LEVEL ? y : s.d[1] - 1;
            o.hi[2] = LEVEL ? slab.hi[2] : z;
        }
        b.group[k] = (uint16_t)g;
    }
}

template <int LAYOUT, int IDX>
__global__ void k_onchip_links(const StepArgs a, const OnchipBuild b)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= b.Ntot) return;
    const OnchipSample& s = b.samples[sample_of(b, k)];
    const int32_t shift = (int32_t)(s.rank0 - s.off);
    int32_t t[Q];
    lane_sources<LAYOUT, IDX>(a, id_of(s, k), t);
#pragma unroll
    for (int j = 1; j < Q; j++) {
        if (t[j] >= 0) t[j] += shift;
        b.T[(int64_t)(j - 1) * b.Ntot + k] = t[j];
        if (t[j] >= 0 && atomicExch(b.M + (int64_t)(RE[j] - 1) * b.Ntot + t[j], (uint32_t)k) != EMPTY) *b.err = 1;
    }
}

// Link j of node k: the node of another block it is shared with, or EMPTY.
// The node it pulls from must be the one that pulls re[j] from it, if any:
// the exchange and the reuse of its LDS cell rest on that.  A mask always
// gives such links; V records are taken as they are, so it is checked.
__device__ __forceinline__ uint32_t partner(const OnchipBuild& b, int64_t k, int j, uint16_t mine, int32_t& t)
{
    t = b.T[(int64_t)(j - 1) * b.Ntot + k];
    const uint32_t m = b.M[(int64_t)(j - 1) * b.Ntot + k];
    if (t >= 0 && m != EMPTY && (uint32_t)t != m) *b.err = 1;
    const uint32_t with = t >= 0 ? (uint32_t)t : m;
    return with != EMPTY && b.blk[with] != mine ? with : EMPTY;
}

// Slot order of one block's nodes: key (no shared link, V id), sorted in LDS.
constexpr int SORT_MAX = 4096;
__global__ void __launch_bounds__(1024) k_onchip_slots(const OnchipBuild b, int T)
{
    __shared__ uint32_t key[SORT_MAX];
    const int blk = blockIdx.x;
    const OnchipSample s = b.samples[b.block_sample[blk]];
    const int64_t lb = blk - s.block0;
    const int64_t r0 = (lb * s.n + s.nblocks - 1) / s.nblocks, r1 = ((lb + 1) * s.n + s.nblocks - 1) / s.nblocks;
    const int n = (int)(r1 - r0);
    int P = 64;
    while (P < n) P <<= 1;
    for (int q = threadIdx.x; q < P; q += blockDim.x) {
        uint32_t v = EMPTY;
        if (q < n) {
            const uint32_t k = b.order[s.rank0 + r0 + q];
            if (k != EMPTY) {  // a rank stays empty where two records share a voxel
                bool shared = false;
                int32_t t;
                for (int j = 1; j < Q; j++) shared |= partner(b, k, j, (uint16_t)blk, t) != EMPTY;
                const uint32_t id = (uint32_t)id_of(s, k);
                v = (b.vid ? b.vid[id] : id) | (shared ? 0u : 0x80000000u);
            }
        }
        key[q] = v;
    }
    __syncthreads();
    for (int size = 2; size <= P; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int q = threadIdx.x; q < P / 2; q += blockDim.x) {
                const int lo = 2 * q - (q & (stride - 1)), hi = lo + stride;
                const bool up = (lo & size) == 0;
                const uint32_t x = key[lo], y = key[hi];
                if ((x > y) == up) {
                    key[lo] = y;
                    key[hi] = x;
                }
            }
            __syncthreads();
        }
    // S shared nodes (of n), an equal share of them in each of the nw first groups
    __shared__ int shared_nodes;
    if (threadIdx.x == 0) {
        int lo = 0, hi = n;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (key[mid] & 0x80000000u) hi = mid;
            else lo = mid + 1;
        }
        shared_nodes = lo;
    }
    __syncthreads();
    const int S = shared_nodes, nw = T / 64;
    for (int q = threadIdx.x; q < n; q += blockDim.x) {
        if (key[q] == EMPTY) continue;
        int slot = q;
        if (S < T) {
            if (q < S) {
                const int g = ((q + 1) * nw - 1) / S;
                slot = g * 64 + q - S * g / nw;
            } else {
                const int i = q - S;   // the groups hold 64 - (their shared nodes) others
                int g = 0;
                while (g < nw && i >= 64 * (g + 1) - S * (g + 1) / nw) g++;
                if (g < nw) slot = 64 * g + (S * (g + 1) / nw - S * g / nw) + i - (64 * g - S * g / nw);
                else slot = T + i - (T - S);
            }
        }
        const uint32_t v = key[q] & 0x7fffffffu;
        const uint32_t k = (uint32_t)number_of(s, b.node_of_v ? b.node_of_v[v] : v);
        b.slot_of[k] = (uint32_t)blk * (uint32_t)b.NS + (uint32_t)slot;
        b.node[(int64_t)blk * b.NS + slot] = k;
    }
}

// Entries of each group of 64 slots.  Their order is (block and group at the
// other end, direction and slot as the end with the lower number has them), so
// the links that two groups share have the same order in both lists: what a
// wave sends as one row of 64 words goes to a few stretches of the receive
// buffers.  (In the order (direction, slot) a row went to 18 pieces of 64 bytes
// on average, in this one to 11, 8 being the least.)
// FILL 0: counts them; 1: writes the entries and the index words.
constexpr int GROUP_KEYS = 2048;   // 64 slots x 18 directions
template <int FILL>
__global__ void __launch_bounds__(256) k_onchip_groups(const OnchipBuild b)
{
    __shared__ uint32_t keys[FILL ? 4 : 1][FILL ? GROUP_KEYS : 1];
    const int lane = threadIdx.x & 63;
    const int ng = b.NS / 64;
    const uint32_t NS = (uint32_t)b.NS;
    const int64_t g = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), groups = (int64_t)b.G * ng;
    const bool in = g < groups;
    const int blk = in ? (int)(g / ng) : 0;
    const uint32_t first = in ? (uint32_t)(g % ng) * 64 : 0u, slot = first + lane;
    const uint32_t k = in ? b.node[g * 64 + lane] : EMPTY;
    uint32_t* const key = keys[FILL ? threadIdx.x >> 6 : 0];
    uint32_t n = 0, lo = 0;
#pragma unroll
    for (int j = 1; j < Q; j++) {
        int32_t t = TAB_CONST;
        uint32_t with = EMPTY;
        if (k != EMPTY) with = partner(b, k, j, (uint16_t)blk, t);
        const uint64_t m = __builtin_amdgcn_ballot_w64(with != EMPTY);
        if constexpr (FILL) {
            const bool in_block = t >= 0 && b.blk[t] == (uint16_t)blk;
            uint32_t pos = slot * Q + RE[j];
            if (in_block) pos = b.slot_of[t] % NS * Q + j;
            else if (t == TAB_CONST) pos = NS * Q + (j > 6 ? 1u : 0u);
            if (k == EMPTY) pos = 0;
            // words 0..8 hold directions 1, 2 | 3, 4 | ... | 17, 18
            if (j & 1) lo = pos;
            else if (in) b.idx[((int64_t)blk * 9 + (j / 2 - 1)) * NS + slot] = lo | (pos << 16);
            if (with != EMPTY) {
                const int other = b.blk[with];
                const uint32_t there = b.slot_of[with] % NS;
                const uint32_t block0 = (uint32_t)b.samples[b.block_sample[blk]].block0;
                const uint32_t dir = blk < other ? (uint32_t)j : (uint32_t)RE[j];
                const uint32_t at = blk < other ? slot : there;
                key[n + __popcll(m & ((1ull << lane) - 1ull))] =
                    ((uint32_t)other - block0) << 16 | (there >> 6) << 11 | dir << 6 | (at & 63u);
            }
        }
        n += (uint32_t)__popcll(m);
    }
    if constexpr (FILL == 0) {
        // Whole rows of 64, so that the exchange needs no lane masks: the rest
        // are entries a block sends to itself and drops.
        if (in && lane == 0) b.cnt[g] = (n + 63u) & ~63u;
    } else {
        uint32_t P = 64;
        while (P < n) P <<= 1;
        for (uint32_t q = n + lane; q < P; q += 64) key[q] = EMPTY;
        // one wave sorts its own keys: LDS operations of a wave stay in order
        auto fence = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
        fence();
        for (uint32_t size = 2; n && size <= P; size <<= 1)
            for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                for (uint32_t q = lane; q < P / 2; q += 64) {
                    const uint32_t a = 2 * q - (q & (stride - 1)), c = a + stride;
                    const uint32_t x = key[a], y = key[c];
                    if ((x > y) == ((a & size) == 0)) {
                        key[a] = y;
                        key[c] = x;
                    }
                }
                fence();
            }
        if (!in) return;
        const uint32_t e0 = b.seg[g], e1 = b.seg[g + 1];
        const int block0 = b.samples[b.block_sample[blk]].block0;
        for (uint32_t q = lane; e0 + q < e1; q += 64) {
            const uint32_t e = e0 + q;
            if (q >= n) {
                b.ent_lds[e] = (NS * Q + DROP) * 0x10001u;
                b.ent_dst[e] = e;
                continue;
            }
            const int other = block0 + (int)(key[q] >> 16);
            uint32_t j = (key[q] >> 6) & 31u, mine = first + (key[q] & 63u);
            int32_t t;
            if (other < blk) {   // the key has the other end's direction and slot
                const uint32_t far = ((key[q] >> 11) & 31u) * 64 + (key[q] & 63u);
                mine = b.slot_of[partner(b, b.node[(int64_t)other * NS + far], (int)j, (uint16_t)other, t)] % NS;
                j = opposite(j);
            }
            const uint32_t me = b.node[(int64_t)blk * NS + mine], own = mine * Q + opposite(j);
            const uint32_t with = partner(b, me, (int)j, (uint16_t)blk, t);
            b.ent_lds[e] = own | (t >= 0 ? own : NS * Q + DROP) << 16;
            b.ent_dst[e] = with;                            // the partner node until k_onchip_dst
            b.at[(int64_t)(j - 1) * b.Ntot + me] = e;
        }
    }
}

// The partner's entry is the other end of the same link: direction re[j] at
// the partner node, and re[j] is the direction of the entry's LDS cell.  The
// slots get their nodes' internal ids in place of the numbers.
__global__ void k_onchip_dst(const OnchipBuild b, int64_t E, int64_t slots)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < slots && b.node[e] != EMPTY) b.node[e] = (uint32_t)id_of(b.samples[b.block_sample[e / b.NS]], b.node[e]);
    if (e >= E) return;
    const uint32_t cell = b.ent_lds[e] & 0xffffu;
    if (cell < (uint32_t)b.NS * Q) b.ent_dst[e] = b.at[(int64_t)(cell % Q - 1) * b.Ntot + b.ent_dst[e]];
}

// ---------------------------------------------------------------- exchange words
// A population and the step's number in one word; FP64 takes two words, one
// per half, in two planes of the buffer.
template <typename S>
struct Wire;
template <>
struct Wire<float> {
    using Word = uint64_t;
    static constexpr int WORDS = 1;
    static __device__ __forceinline__ void pack(float v, uint32_t tag, Word w[1])
    {
        w[0] = ((uint64_t)tag << 32) | __float_as_uint(v);
    }
    static __device__ __forceinline__ bool is(Word w, uint32_t tag) { return (uint32_t)(w >> 32) == tag; }
    static __device__ __forceinline__ Word none(uint32_t tag) { return (uint64_t)tag << 32; }
    static __device__ __forceinline__ float unpack(const Word w[1]) { return __uint_as_float((uint32_t)w[0]); }
};
template <>
struct Wire<double> {
    using Word = uint64_t;
    static constexpr int WORDS = 2;
    static __device__ __forceinline__ void pack(double v, uint32_t tag, Word w[2])
    {
        const uint64_t b = (uint64_t)__double_as_longlong(v);
        w[0] = ((uint64_t)tag << 32) | (b & 0xffffffffull);
        w[1] = ((uint64_t)tag << 32) | (b >> 32);
    }
    static __device__ __forceinline__ bool is(Word w, uint32_t tag) { return (uint32_t)(w >> 32) == tag; }
    static __device__ __forceinline__ Word none(uint32_t tag) { return (uint64_t)tag << 32; }
    static __device__ __forceinline__ double unpack(const Word w[2])
    {
        return __longlong_as_double((long long)((w[0] & 0xffffffffull) | (w[1] << 32)));
    }
};
template <>
struct Wire<__half> {
    using Word = uint32_t;
    static constexpr int WORDS = 1;
    static __device__ __forceinline__ void pack(__half v, uint32_t tag, Word w[1])
    {
        w[0] = (tag << 16) | __half_as_ushort(v);
    }
    static __device__ __forceinline__ bool is(Word w, uint32_t tag) { return (w >> 16) == (tag & 0xffffu); }
    static __device__ __forceinline__ Word none(uint32_t tag) { return tag << 16; }
    static __device__ __forceinline__ __half unpack(const Word w[1])
    {
        return __ushort_as_half((unsigned short)(w[0] & 0xffffu));
    }
};

struct OnchipArgs {
    const uint32_t *node, *idx, *seg, *ent_lds, *ent_dst;
    void* recv;
    int64_t E;
    int NS;
    int64_t nstride, dstride;  // element (j, node): AoSoA (node >> 6) * nstride + (node & 63) + j * dstride
    int soa;
    int64_t nsteps;
    uint32_t tag, serial;
    uint64_t first_ticks, wait_ticks;
    // batches: the blocks of this launch, and each block's sample
    const int32_t *list, *blk_sample;
    const double *omega, *gx;
};

// ---------------------------------------------------------------- the run
// K nodes per thread, slots tid, tid + T, ...: the shared nodes, which come
// first, are spread over all waves.
// TWICE: two copies of F, read and written by turns, where they fit the LDS:
// one block barrier per step instead of two, and no values held across it.
template <typename S, int K, bool TWICE, int MAXT>
__global__ void __launch_bounds__(MAXT) k_onchip(StepArgs a, const OnchipArgs p)
{
    using W = Wire<S>;
    using Word = typename W::Word;
    constexpr int RL = MAXT > 512 ? 6 : 10;   // rows of the entry list kept in registers
    extern __shared__ __align__(16) char lds[];
    S* F = (S*)lds;                            // the copy that is read
    __shared__ int bad[2];                     // by step parity: a wave may be one poll ahead of another
    // Queued behind a step that did not complete: nothing to do.  (A key of
    // this run's own steps, set by a block that started earlier, does not count.)
    const unsigned long long fk = *a.fault;
    if (frozen(fk, a.it)) return;

    const int T = blockDim.x, tid = threadIdx.x, lane = tid & 63, NS = p.NS;
    const int copy = NS * Q + EXTRA;
    S* G = TWICE ? F + copy : F;               // the copy that is written
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t blk = p.list ? ld_const(p.list + blockIdx.x) : (int)blockIdx.x;
    if (p.blk_sample) {
        const int s = ld_const(p.blk_sample + blk);
        a.omega = ld_const(p.omega + s);
        a.gx = ld_const(p.gx + s);
    }
    const S* __restrict__ fin = (const S*)a.fin;
    uint32_t node[K], w[K][9], key[K], s0[K], s1[K];
    bool any[K];   // whether the wave has nodes in its k-th group
    const bool sr = sizeof(S) == 2 && a.stochastic;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int slot = k * T + tid;
        node[k] = p.node[blk * NS + slot];
        any[k] = k == 0 || __builtin_amdgcn_ballot_w64(node[k] != EMPTY) != 0;
#pragma unroll
        for (int q = 0; q < 9; q++) w[k][q] = p.idx[(blk * 9 + q) * NS + slot];
        const int64_t g = blk * (NS / 64) + k * (T / 64) + wave;
        s0[k] = p.seg[g];
        s1[k] = p.seg[g + 1];
        key[k] = node[k];
        if (node[k] != EMPTY) {
            if (sr && a.key_perm) key[k] = a.key_perm[node[k]];
            const int64_t at = p.soa ? (int64_t)node[k] : (int64_t)(node[k] >> 6) * p.nstride + (node[k] & 63u);
#pragma unroll
            for (int j = 0; j < Q; j++) F[slot * Q + j] = fin[at + j * p.dstride];
        }
    }
    if (tid < EXTRA) {
        S v = S(0);
        if constexpr (sizeof(S) == 8) v = tid == DROP ? 0.0 : (tid ? TP[7] : TP[1]) * a.rho0 * 1.0;
        F[NS * Q + tid] = v;
        G[NS * Q + tid] = v;
    }
    if (tid < 2) bad[tid] = 0;
    // The first RL rows of the wave's first group's entries stay in registers
    // (read from memory every step, the lists cost more than the exchange);
    // the other groups, which mostly have none, look theirs up.
    uint32_t cell[RL], dst[RL];
#pragma unroll
    for (int r = 0; r < RL; r++) {
        const uint32_t e = s0[0] + r * 64;
        cell[r] = dst[r] = 0;
        if (e < s1[0]) {
            cell[r] = p.ent_lds[e + lane];
            dst[r] = p.ent_dst[e + lane];
        }
    }
    __syncthreads();

    // Cells of a group are written and read by lanes of one wave: LDS
    // operations of a wave stay in order, the fence keeps the compiler to it.
    auto put_word = [&](Word* buf, uint32_t to, S value, uint32_t tag) {
        Word v[W::WORDS];
        W::pack(value, tag, v);
#pragma unroll
        for (int q = 0; q < W::WORDS; q++)
            __hip_atomic_store(buf + to + q * p.E, v[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto send = [&](int k, const S* from, uint32_t tag) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        Word* const buf = (Word*)p.recv + (int64_t)(tag & 1u) * W::WORDS * p.E;
        if (k == 0) {
            // All values first, then all stores: with an LDS read between two
            // stores the compiler may put a wait for the first one, a trip
            // through memory, in front of it (2.5 -> 5 us a step).
            S v[RL];
#pragma unroll
            for (int r = 0; r < RL; r++) {
                if (s0[0] + r * 64 >= s1[0]) break;
                v[r] = from[cell[r] & 0xffffu];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < RL; r++) {
                if (s0[0] + r * 64 >= s1[0]) break;
                put_word(buf, dst[r], v[r], tag);
            }
        }
        for (uint32_t b = s0[k] + (k == 0 ? RL * 64 : 0); b < s1[k]; b += 64 * 4) {
            uint32_t c[4], d[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if (b + r * 64 >= s1[k]) break;
                c[r] = p.ent_lds[b + r * 64 + lane];
                d[r] = p.ent_dst[b + r * 64 + lane];
            }
            S v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if (b + r * 64 >= s1[k]) break;
                v[r] = from[c[r] & 0xffffu];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if (b + r * 64 >= s1[k]) break;
                put_word(buf, d[r], v[r], tag);
            }
        }
    };
    // Up to N rows of entries from e0: all are waited for, then stored to `to`.
    auto receive_rows = [&](auto count, uint32_t e0, uint32_t e1, S* to, uint32_t tag, uint64_t limit, auto cell_of) {
        constexpr int N = decltype(count)::value;
        const int parity = (int)(tag & 1u);
        const Word* const buf = (const Word*)p.recv + (int64_t)(tag & 1u) * W::WORDS * p.E + lane;
        Word v[N][W::WORDS];
        auto load = [&](int r) {
#pragma unroll
            for (int q = 0; q < W::WORDS; q++)
                v[r][q] = __hip_atomic_load(buf + (e0 + r * 64) + q * p.E, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        auto missing = [&](int r) {
            bool ok = true;
#pragma unroll
            for (int q = 0; q < W::WORDS; q++) ok &= W::is(v[r][q], tag);
            return !ok;
        };
#pragma unroll
        for (int r = 0; r < N; r++) {
            if (e0 + r * 64 >= e1) break;
            load(r);
        }
        uint64_t since = 0;
        for (uint32_t spins = 1;; spins++) {
            bool wait = false;
#pragma unroll
            for (int r = 0; r < N; r++) {
                if (e0 + r * 64 >= e1) break;
                wait |= missing(r);
            }
            if (__builtin_amdgcn_ballot_w64(wait) == 0) break;
#pragma unroll
            for (int r = 0; r < N; r++) {
                if (e0 + r * 64 >= e1) break;
                if (missing(r)) load(r);
            }
            if (spins % 256 == 0) {
                const uint64_t now = wall_clock64();
                if (since == 0) since = now;
                const bool late = now - since > limit;
                if (late) {
                    __hip_atomic_store(a.fault + 1, (unsigned long long)p.serial, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_fetch_min(a.fault, HOLD_FAULT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                if (late || __hip_atomic_load(a.fault + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                                (unsigned long long)p.serial) {
                    bad[parity] = 1;
                    return;
                }
            }
        }
#pragma unroll
        for (int r = 0; r < N; r++) {
            if (e0 + r * 64 >= e1) break;
            to[cell_of(r) >> 16] = W::unpack(v[r]);
        }
    };
    auto receive = [&](int k, S* to, uint32_t tag, uint64_t limit) {
        if (k == 0 && s0[0] < s1[0])
            receive_rows(std::integral_constant<int, RL>{}, s0[0], s1[0], to, tag, limit, [&](int r) { return cell[r]; });
        for (uint32_t b = s0[k] + (k == 0 ? RL * 64 : 0); b < s1[k]; b += 64 * 4)
            receive_rows(std::integral_constant<int, 4>{}, b, s1[k], to, tag, limit,
                         [&](int r) { return p.ent_lds[b + r * 64 + lane]; });
    };
    auto cell_at = [&](int k, int j) -> S {
        return j == 0 ? F[(k * T + tid) * Q] : F[(w[k][(j - 1) >> 1] >> (((j - 1) & 1) * 16)) & 0xffffu];
    };
    auto update = [&](int k, auto value) {
        if (node[k] == EMPTY) return;
        S* const own = G + (k * T + tid) * Q;
        auto put = [&](int j, S v) { own[j] = v; };
        if constexpr (sizeof(S) == 8) {
            double f[Q];
#pragma unroll
            for (int j = 0; j < Q; j++) f[j] = value(j);
            relax_f64(a, node[k], f, NO_FAULT, put);
        } else {
            float ds[Q];
#pragma unroll
            for (int j = 0; j < Q; j++) ds[j] = to_float(value(j));
            relax_shift<S>(a, node[k], ds, NO_FAULT, key[k], put);
        }
    };

#pragma unroll
    for (int k = 0; k < K; k++) send(k, F, p.tag);
    const int64_t it0 = a.it;
    for (int64_t t = 0; t < p.nsteps; t++) {
        const uint32_t tag = p.tag + (uint32_t)t;
        const bool last = t + 1 == p.nsteps;
        a.it = it0 + t;
        a.write_macros = last ? 1 : 0;
        if constexpr (MAXT > 512) {
            // Unpacked every step: hoisted out of the loop, the addresses
            // would spill.
#pragma unroll
            for (int k = 0; k < K; k++) {
                asm volatile("" : "+v"(node[k]));
#pragma unroll
                for (int q = 0; q < 9; q++) asm volatile("" : "+v"(w[k][q]));
            }
        }
#pragma unroll
        for (int k = 0; k < K; k++) receive(k, F, tag, t == 0 ? p.first_ticks : p.wait_ticks);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if constexpr (TWICE) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                if (!any[k]) break;
                update(k, [&](int j) { return cell_at(k, j); });
                if (!last) send(k, G, tag + 1);
                if constexpr (K > 1) __builtin_amdgcn_sched_barrier(0);  // one node's values at a time
            }
            S* const r = F;
            F = G;
            G = r;
        } else {
            S raw[K][Q];
#pragma unroll
            for (int k = 0; k < K; k++) {
                if (!any[k]) break;
#pragma unroll
                for (int j = 0; j < Q; j++) raw[k][j] = cell_at(k, j);
            }
            __syncthreads();  // every gather is done
#pragma unroll
            for (int k = 0; k < K; k++) {
                if (!any[k]) break;
                update(k, [&](int j) { return raw[k][j]; });
                if (!last) send(k, G, tag + 1);
                if constexpr (K > 1) __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();  // every population is in place
        if (bad[tag & 1u]) return;  // set before the barrier, the same for all threads
        if constexpr (TWICE) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    S* __restrict__ fout = (S*)a.fout;
#pragma unroll
    for (int k = 0; k < K; k++)
        if (node[k] != EMPTY) {
            const int64_t at = p.soa ? (int64_t)node[k] : (int64_t)(node[k] >> 6) * p.nstride + (node[k] & 63u);
#pragma unroll
            for (int j = 0; j < Q; j++) fout[at + j * p.dstride] = F[(k * T + tid) * Q + j];
        }
}

// ---------------------------------------------------------------- host
static unsigned nblk(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }
void onchip_destroy(plb_ctx* c)
{
    OnchipPlan* p = c->chip;
    if (!p) return;
    (void)hipStreamSynchronize(c->stream);
    for (void* q : {p->fixed, p->exchange, (void*)p->macros_own})
        if (q) dev_free(q);
    delete p;
    c->chip = nullptr;
}

void onchip_restore_macros(plb_ctx* c, double* macros)
{
    if (c->chip && c->chip->macros_alt == macros) std::swap(c->macros, c->chip->macros_alt);
}

// Node slots of a block, and whether two copies of its populations fit the
// LDS.  One copy holds what the registers can carry over the barrier: 1 FP64
// or 2 FP32 nodes per thread.
static size_t lds_bytes(const plb_ctx* c, int NS, bool twice)
{
    return ((size_t)Q * NS + EXTRA) * c->elem * (twice ? 2 : 1);
}
// Two nodes per thread: always 1024 threads, of which the second nodes may keep
// only some waves busy (1 037 nodes: 576 threads took 6.0 to 7.8 us a step, 1024 take 5.0 to 5.5).
static int slots_for(int nodes) { return nodes > 1024 ? 2048 : (nodes + 63) / 64 * 64; }
static bool fits_twice(const plb_ctx* c, int NS) { return lds_bytes(c, NS, true) + 64 <= (size_t)c->lds_per_cu; }
// Slots, nodes per thread, threads and copies of a block of up to `nodes` nodes.
static void shape(const plb_ctx* c, OnchipPlan* p, int nodes)
{
    p->NS = slots_for(nodes);
    p->K = nodes > 1024 ? 2 : 1;
    p->T = p->NS / p->K;
    p->twice = fits_twice(c, p->NS);
}

// f(the kernel of a plan); false where there is none of its shape.
template <typename F>
static bool with_kernel(const plb_ctx* c, const OnchipPlan* p, F f)
{
    const bool small = p->T <= 512, one = p->K == 1, twice = p->twice;
    if (c->cfg.precision == PLB_FP64) {
        if (!one || (twice && !small)) return false;
        twice ? f(k_onchip<double, 1, true, 512>) : f(k_onchip<double, 1, false, 1024>);
    } else if (c->cfg.precision == PLB_FP32) {
        if (one != twice) return false;
        !twice ? f(k_onchip<float, 2, false, 1024>)
               : small ? f(k_onchip<float, 1, true, 512>) : f(k_onchip<float, 1, true, 1024>);
    } else {
        // (Blocks of more than 2048 slots, with 3 nodes per thread and one copy, spill: 22 us a
        // step for 629 146 nodes, against 16.8 us with one launch per step.)
        if (!twice) return false;
        !one ? f(k_onchip<__half, 2, true, 1024>)
             : small ? f(k_onchip<__half, 1, true, 512>) : f(k_onchip<__half, 1, true, 1024>);
    }
    return true;
}

static bool fits(const plb_ctx* c, int nodes)
{
    if (nodes > (c->cfg.precision == PLB_FP64 ? 1024 : 2048)) return false;
    OnchipPlan p;
    shape(c, &p, nodes);
    return with_kernel(c, &p, [](auto*) {}) && lds_bytes(c, p.NS, p.twice) + 64 <= (size_t)c->lds_per_cu;
}

// Slabs and rows of a sample, so that blocks are about as long as wide.
static void cuts(OnchipSample& s)
{
    const double side = std::cbrt((double)s.d[0] * s.d[1] * s.d[2] / std::max(1, s.nblocks));
    s.slabs = std::max(1, std::min(s.nblocks, (int)std::lround(s.d[2] / side)));
    const int per_slab = s.nblocks / s.slabs;
    s.rows = std::max(1, std::min(per_slab, (int)std::lround(std::sqrt((double)per_slab * s.d[1] / s.d[0]))));
}
// Bits that hold any of its bitmasks: neighbouring slabs share a plane at most, neighbouring rows a line of one.
static int64_t box_bits(const OnchipSample& s)
{
    return (int64_t)s.d[0] * (s.d[1] + s.rows) * (s.d[2] + s.slabs);
}
constexpr int64_t BOX_BITS_MAX = (int64_t)1 << 27;   // not for a sparse mask in a huge box

static int build_onchip(plb_ctx* c, std::vector<OnchipSample> samples, int G, int NS)
{
    OnchipPlan* p = new OnchipPlan();
    c->chip = p;
    hipStream_t s = c->stream;
    p->G = G;
    shape(c, p, NS);
    NS = p->NS;
    const int ng = NS / 64;
    int64_t words = 0, rank = 0;
    std::vector<int32_t> block_sample(G);
    for (size_t k = 0; k < samples.size(); k++) {
        OnchipSample& smp = samples[k];
        smp.word0 = words;
        smp.rank0 = rank;
        cuts(smp);
        smp.words = smp.nblocks ? (box_bits(smp) + 63) / 64 : 0;
        words += smp.words;
        if (smp.nblocks) rank += smp.n;
        for (int q = 0; q < smp.nblocks; q++) block_sample[smp.block0 + q] = (int32_t)k;
    }
    p->samples = samples;
    const int64_t Ntot = rank;
    // arrays of the plan
    const int64_t slots = (int64_t)G * NS, groups = (int64_t)G * ng;
    PLB_HIP(dev_alloc(&p->fixed, sizeof(uint32_t) * (slots * 10 + groups + 1 + G)));
    p->node = (uint32_t*)p->fixed;
    p->idx = p->node + slots;
    p->seg = p->idx + 9 * slots;
    p->blk_sample = (int32_t*)(p->seg + groups + 1);
    // scratch of the build
    Arena mem(s);
    DevBuf<char> scratch;
    size_t need = 0;
    auto part = [&](size_t bytes) {
        const size_t at = need;
        need += (bytes + 255) / 256 * 256;
        return at;
    };
    const size_t o_smp = part(sizeof(OnchipSample) * samples.size()), o_bits = part(8 * (size_t)words), o_wpre = part(4 * (size_t)(words + 1)), o_order = part(4 * Ntot),
                 o_blk = part(2 * Ntot), o_group = part(2 * Ntot),
                 o_box = part(sizeof(OnchipBox) * 2 * (size_t)G), o_base = part(4 * 2 * (size_t)G), o_slot = part(4 * Ntot), o_T = part(4 * 18 * Ntot), o_M = part(4 * 18 * Ntot), o_at = part(4 * 18 * Ntot),
                 o_cnt = part(4 * groups), o_err = part(4);
    PLB_HIP(scratch.alloc((int64_t)need, &mem));
    char* const base = scratch.p;
    OnchipBuild b = {};
    b.samples = (const OnchipSample*)(base + o_smp);
    b.nsamples = (int)samples.size();
    b.Ntot = Ntot;
    b.xyz = c->node_xyz;
    const bool batch = c->key_perm != nullptr;
    b.xyz_of = batch ? c->perm : nullptr;  // batches keep coordinates in V order
    b.vid = c->perm;
    b.node_of_v = c->inv_perm;
    b.bits = (unsigned long long*)(base + o_bits);
    b.wpre = (uint32_t*)(base + o_wpre);
    b.order = (uint32_t*)(base + o_order);
    b.group = (uint16_t*)(base + o_group);
    b.box = (OnchipBox*)(base + o_box);
    b.base = (uint32_t*)(base + o_base);
    b.blk = (uint16_t*)(base + o_blk);
    b.slot_of = (uint32_t*)(base + o_slot);
    b.T = (int32_t*)(base + o_T);
    b.M = (uint32_t*)(base + o_M);
    b.at = (uint32_t*)(base + o_at);
    b.block_sample = p->blk_sample;
    b.cnt = (uint32_t*)(base + o_cnt);
    b.err = (int*)(base + o_err);
    b.node = p->node;
    b.idx = p->idx;
    b.seg = p->seg;
    b.G = G;
    b.NS = NS;
    PLB_HIP(hipMemcpyAsync(base + o_smp, samples.data(), sizeof(OnchipSample) * samples.size(), hipMemcpyHostToDevice, s));
    PLB_HIP(hipMemcpyAsync(p->blk_sample, block_sample.data(), sizeof(int32_t) * G, hipMemcpyHostToDevice, s));
    PLB_HIP(hipMemsetAsync(p->node, 0xff, sizeof(uint32_t) * slots, s));
    const std::vector<OnchipBox> none(2 * (size_t)G, OnchipBox{{1 << 30, 1 << 30, 1 << 30}, {-1, -1, -1}});
    PLB_HIP(hipMemcpyAsync(b.box, none.data(), sizeof(OnchipBox) * none.size(), hipMemcpyHostToDevice, s));
    PLB_HIP(hipMemsetAsync(b.group, 0, 2 * (size_t)Ntot, s));
    PLB_HIP(hipMemsetAsync(b.M, 0xff, 4 * 18 * (size_t)Ntot, s));
    PLB_HIP(hipMemsetAsync(b.order, 0xff, 4 * (size_t)Ntot, s));
    PLB_HIP(hipMemsetAsync(b.err, 0, sizeof(int), s));
    const dim3 per_node(nblk(Ntot, 256)), t256(256);
    const dim3 per_sample((unsigned)samples.size()), t1024(1024);
    PLB_HIP(hipMemsetAsync(b.bits, 0, 8 * (size_t)words, s));
    hipLaunchKernelGGL(k_onchip_bits<0>, per_node, t256, 0, s, b);
    hipLaunchKernelGGL(k_onchip_words, per_sample, t1024, 0, s, b);
    hipLaunchKernelGGL(k_onchip_rank<0>, per_node, t256, 0, s, b);
    hipLaunchKernelGGL(k_onchip_boxes<0>, per_sample, t1024, 0, s, b);
    PLB_HIP(hipMemsetAsync(b.bits, 0, 8 * (size_t)words, s));
    hipLaunchKernelGGL(k_onchip_bits<1>, per_node, t256, 0, s, b);
    hipLaunchKernelGGL(k_onchip_words, per_sample, t1024, 0, s, b);
    hipLaunchKernelGGL(k_onchip_rank<1>, per_node, t256, 0, s, b);
    hipLaunchKernelGGL(k_onchip_boxes<1>, per_sample, t1024, 0, s, b);
    PLB_HIP(hipMemsetAsync(b.bits, 0, 8 * (size_t)words, s));
    hipLaunchKernelGGL(k_onchip_bits<2>, per_node, t256, 0, s, b);
    hipLaunchKernelGGL(k_onchip_words, per_sample, t1024, 0, s, b);
    hipLaunchKernelGGL(k_onchip_rank<2>, per_node, t256, 0, s, b);
    const StepArgs a = make_args(c, 0, false);
    const int idx = c->cfg.index_kind;
#define PLB_LINKS(L, I) hipLaunchKernelGGL((k_onchip_links<L, I>), per_node, t256, 0, s, a, b)
    if (c->cfg.layout == PLB_LAYOUT_SOA) {
        if (idx == PLB_INDEX_TILE8) PLB_LINKS(PLB_LAYOUT_SOA, PLB_INDEX_TILE8);
        else if (idx == PLB_INDEX_BITMAP) PLB_LINKS(PLB_LAYOUT_SOA, PLB_INDEX_BITMAP);
        else PLB_LINKS(PLB_LAYOUT_SOA, PLB_INDEX_I32);
    } else {
        if (idx == PLB_INDEX_TILE8) PLB_LINKS(PLB_LAYOUT_AOSOA, PLB_INDEX_TILE8);
        else if (idx == PLB_INDEX_BITMAP) PLB_LINKS(PLB_LAYOUT_AOSOA, PLB_INDEX_BITMAP);
        else PLB_LINKS(PLB_LAYOUT_AOSOA, PLB_INDEX_I32);
    }
#undef PLB_LINKS
    hipLaunchKernelGGL(k_onchip_slots, dim3(G), dim3(std::min(1024, NS)), 0, s, b, p->T);
    hipLaunchKernelGGL(k_onchip_groups<0>, dim3(nblk(groups, 4)), t256, 0, s, b);
    hipLaunchKernelGGL(k_onchip_segs, dim3(1), dim3(1024), 0, s, b, groups);
    PLB_HIP(hipGetLastError());
    uint32_t E = 0;
    int err = 0;
    PLB_HIP(hipMemcpyAsync(&E, b.seg + groups, sizeof E, hipMemcpyDeviceToHost, s));
    PLB_HIP(hipMemcpyAsync(&err, b.err, sizeof err, hipMemcpyDeviceToHost, s));
    PLB_HIP(hipStreamSynchronize(s));
    if (err) return PLB_ERR_INVALID;
    p->E = E;
    if (E) {
        const size_t word = c->cfg.precision == PLB_FP16 ? 4 : c->cfg.precision == PLB_FP32 ? 8 : 16;
        const size_t lists = (8 * (size_t)E + 255) / 256 * 256;
        PLB_HIP(dev_alloc(&p->exchange, lists + 2 * word * E));
        b.ent_lds = p->ent_lds = (uint32_t*)p->exchange;
        b.ent_dst = p->ent_dst = p->ent_lds + E;
        p->recv = (char*)p->exchange + lists;
        // no number a run will wait for
        p->recv_bytes = 2 * word * E;
        PLB_HIP(hipMemsetAsync(p->recv, 0, p->recv_bytes, s));
    }
    hipLaunchKernelGGL(k_onchip_groups<1>, dim3(nblk(groups, 4)), t256, 0, s, b);
    hipLaunchKernelGGL(k_onchip_dst, dim3(nblk(std::max<int64_t>(E, slots), 256)), t256, 0, s, b, (int64_t)E, slots);
    PLB_HIP(hipGetLastError());
    if (!batch) {
        PLB_HIP(dev_alloc((void**)&p->macros_own, sizeof(double) * 4 * c->Npad));
        p->macros_alt = p->macros_own;
        PLB_HIP(hipMemsetAsync(p->macros_alt, 0, sizeof(double) * 4 * c->Npad, s));
    }
    PLB_HIP(hipStreamSynchronize(s));  // the scratch goes back
    int rc = PLB_OK;
    with_kernel(c, p, [&](auto* kern) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes(c, NS, p->twice)) !=
            hipSuccess)
            rc = PLB_ERR_HIP;
    });
    return rc;
}

static int plan_single(plb_ctx* c)
{
    int cus = 0;
    PLB_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
    const int64_t per = std::max<int64_t>(ONCHIP_MIN_SLOTS, (c->N + cus - 1) / cus);
    const int NS = (int)std::min<int64_t>(65536, (per + 63) / 64 * 64);
    if (!fits(c, NS)) return PLB_ERR_RANGE;
    OnchipSample smp = {};
    smp.n = c->N;
    smp.d[0] = c->nx;
    smp.d[1] = c->ny;
    smp.d[2] = c->nz;
    smp.nblocks = (int)((c->N + NS - 1) / NS);
    cuts(smp);
    if (box_bits(smp) > BOX_BITS_MAX) return PLB_ERR_RANGE;
    std::vector<OnchipSample> samples{smp};
    return build_onchip(c, samples, smp.nblocks, NS);
}

// A run gave up: some of its blocks did not start within 50 ms, because other
// work kept the CUs.  Launches per step take over for a while, twice as long after
// each time, so that a busy chip costs a few waits (16 384 steps of a small lattice,
// 70 ms, take about as long as one) and a chip that is free again is used.
int onchip_gave_up(plb_ctx* c)
{
    fprintf(stderr, "libplb: an on-chip run's blocks were not all resident; the next %lld steps go with one launch per step\n",
            (long long)c->chip_pause);
    c->chip_rest = c->chip_pause;
    c->chip_pause *= c->chip_pause < ((int64_t)1 << 60) ? 2 : 1;
    return onchip_clear(c);
}

// Whether a call of nsteps steps falls into such a while.
bool onchip_resting(plb_ctx* c, int64_t nsteps)
{
    if (c->chip_rest <= 0) return false;
    c->chip_rest -= nsteps;
    return true;
}

// Whether this call of nsteps steps runs on chip; builds the plan when it pays.
bool onchip_ready(plb_ctx* c, int64_t nsteps)
{
    if (c->chip_state < 0 || nsteps < 16 || c->N == 0 || c->fault_seen) return false;
    if (c->cfg.stream_mode != PLB_STREAM_PULL || c->cfg.graph_steps != 0) return false;
    if (c->chip_state == 0) {
        c->chip_steps += nsteps;
        if (c->chip_steps < ONCHIP_PLAN_STEPS) return false;
        // a capture of the caller's elsewhere in this thread is none of the plan's business
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        const int rc = guarded([&] { return plan_single(c); });
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        if (rc) {  // too large, or no memory for the plan: one launch per step
            (void)hipGetLastError();
            onchip_destroy(c);
        }
        c->chip_state = rc ? -1 : 1;
    }
    return c->chip_state == 1 && !onchip_resting(c, nsteps);
}

// One launch of `blocks` blocks (list: which) for steps it0 .. it0 + n - 1.
static hipError_t launch(plb_ctx* c, const StepArgs& a0, OnchipArgs o, int64_t n, int blocks)
{
    OnchipPlan* p = c->chip;
    StepArgs a = a0;
    o.node = p->node;
    o.idx = p->idx;
    o.seg = p->seg;
    o.ent_lds = p->ent_lds;
    o.ent_dst = p->ent_dst;
    o.recv = p->recv;
    o.E = p->E;
    o.NS = p->NS;
    o.soa = c->cfg.layout == PLB_LAYOUT_SOA;
    o.nstride = Q * 64;
    o.dstride = o.soa ? c->Npad : 64;
    o.nsteps = n;
    int khz = 0;
    (void)hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, c->device);
    if (khz < 1000) khz = 100000;
    o.first_ticks = (uint64_t)khz * 50;
    o.wait_ticks = (uint64_t)khz * 2000;
    hipError_t e = hipErrorUnknown;
    if (blocks > 1 && c->chip_withhold > 0) {
        c->chip_withhold--;
        blocks--;   // the others wait for it, and give up
    }
    with_kernel(c, p, [&](auto* kern) {
        void* args[] = {(void*)&a, (void*)&o};
        const size_t lds = lds_bytes(c, p->NS, p->twice);
        if (blocks > 1) {
            e = hipLaunchCooperativeKernel((const void*)kern, dim3(blocks), dim3(p->T), args, (unsigned)lds, c->stream);
        } else {
            hipLaunchKernelGGL(kern, dim3(1), dim3(p->T), lds, c->stream, a, o);
            e = hipGetLastError();
        }
    });
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
}

// No step number of an earlier run is left in the buffers.  A run's numbers go on
// from those of the run before it, whose words lie one or two numbers back when
// it has run to its end; a run that was held off by a fault stores none, so the
// numbers (16 bits with FP16 words) may come round to the old words.  A fault ends
// with a new state, and so does a run of a batch begin.
int onchip_clear(plb_ctx* c)
{
    if (c->chip->recv_bytes) PLB_HIP(hipMemsetAsync(c->chip->recv, 0, c->chip->recv_bytes, c->stream));
    c->chip->tag = 16;
    return PLB_OK;
}

// Tests only: launches the next `runs` runs of more than one block without the
// last one, as if it were not resident; returns how many were still to come.
extern "C" int plb_test_withhold_block(plb_ctx* c, int runs) { return std::exchange(c->chip_withhold, runs); }

static uint32_t next_serial(OnchipPlan* p) { return ++p->serial ? p->serial : ++p->serial; }

int launch_onchip(plb_ctx* c, int64_t it0, int64_t n, uint32_t* serial)
{
    OnchipPlan* p = c->chip;
    *serial = 0;
    std::swap(c->macros, p->macros_alt);
    OnchipArgs o = {};
    o.tag = p->tag;
    o.serial = next_serial(p);
    if (launch(c, make_args(c, it0, false), o, n, p->G) != hipSuccess) {
        // refused before anything ran: one launch per step
        std::swap(c->macros, p->macros_alt);
        c->chip_state = -1;
        return PLB_OK;
    }
    p->tag += (uint32_t)n + 2;  // the runs' numbers do not meet
    *serial = o.serial;
    c->cur ^= 1;
    return PLB_OK;
}

// ---------------------------------------------------------------- batches
// Samples that fit share the launches: as many samples as have room on the
// chip at once run to the next check, then the next ones.  First fit, largest
// sample first: launch[k] = the samples of launch k.
void onchip_pack(const std::vector<int>& blocks, int cus, std::vector<std::vector<int>>* launches)
{
    std::vector<int> order, room;
    for (size_t k = 0; k < blocks.size(); k++)
        if (blocks[k] > 0) order.push_back((int)k);
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return blocks[x] > blocks[y]; });
    launches->clear();
    for (int s : order) {
        size_t l = 0;
        while (l < room.size() && room[l] < blocks[s]) l++;
        if (l == room.size()) {
            room.push_back(cus);
            launches->emplace_back();
        }
        room[l] -= blocks[s];
        (*launches)[l].push_back(s);
    }
}

// Time of a step of a launch that fills the chip with blocks of up to NS nodes,
// in ns: fits of 64^3 to 119^3 noise masks and sphere packs (FP32: 2.2 us at 359
// nodes, 3.8 to 4.2 at 1152, 4.9 to 5.5 at 1664, 5.5 to 5.9 at 1975; FP64: 3.6 at 359,
// 5.2 at 600, 6.3 at 1005; FP16: 4.2 to 4.8 at 1152, 6.2 to 7.3 at 2000).  Above 1024
// nodes a thread has two.
static int64_t step_ns(const plb_ctx* c, int NS)
{
    if (c->cfg.precision == PLB_FP64) return 2600 + NS * 37 / 10;
    if (NS <= 1024) return 1900 + NS * 6 / 5;
    return c->cfg.precision == PLB_FP32 ? 1900 + NS * 37 / 20 : 1000 + NS * 14 / 5;
}

bool onchip_batch_ready(plb_ctx* c, const std::vector<int64_t>& off, const std::vector<int64_t>& n,
                        const std::vector<int>& nx, const std::vector<int>& ny, const std::vector<int>& nz,
                        int64_t steps)
{
    if (c->chip_state != 0 || steps < 128) return c->chip_state == 1 && steps >= 16;
    c->chip_state = -1;
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device) != hipSuccess) return false;
    int most = 0;
    for (int q = 64; q <= 4096 && fits(c, q); q += 64) most = q;
    std::vector<OnchipSample> samples(n.size());
    std::vector<int> blocks(n.size());
    std::vector<std::vector<int>> launches;
    int G = 0;
    auto divide = [&](int NS) {
        G = 0;
        for (size_t k = 0; k < n.size(); k++) {
            OnchipSample& s = samples[k];
            s = {};
            s.off = off[k];
            s.n = n[k];
            s.d[0] = nx[k];
            s.d[1] = ny[k];
            s.d[2] = nz[k];
            s.block0 = G;
            s.nblocks = n[k] > 0 && n[k] <= (int64_t)most * cus ? (int)((n[k] + NS - 1) / NS) : 0;
            cuts(s);
            if (box_bits(s) > BOX_BITS_MAX) s.nblocks = 0;
            if (s.nblocks > cus) return false;  // this sample needs larger blocks
            blocks[k] = s.nblocks;
            G += s.nblocks;
        }
        onchip_pack(blocks, cus, &launches);
        return true;
    };
    // larger blocks: fewer launches for a step of the whole batch, each longer
    int NS = 0;
    int64_t cost = 0;
    for (int q = ONCHIP_MIN_SLOTS; q <= most; q += 64) {
        if (!divide(q)) continue;
        const int64_t w = (int64_t)launches.size() * step_ns(c, q);
        if (NS == 0 || w < cost) {
            NS = q;
            cost = w;
        }
    }
    if (NS == 0 || !divide(NS)) return false;
    if (G == 0 || G > 65535) return false;
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    const int rc = guarded([&] { return build_onchip(c, samples, G, NS); });
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (rc) {
        (void)hipGetLastError();
        onchip_destroy(c);
        return false;
    }
    c->chip_state = 1;
    return true;
}

int onchip_blocks(const plb_ctx* c, int sample, int* block0)
{
    const OnchipSample& s = c->chip->samples[sample];
    *block0 = s.block0;
    return s.nblocks;
}

// The samples of `list`, n steps from buffer c->cur to the buffer that n
// single steps end in.  Launches of one interval use the same step numbers.
int launch_onchip_batch(plb_ctx* c, int64_t it0, int64_t n, const int32_t* list, int blocks, const double* omega,
                        const double* gx)
{
    StepArgs a = make_args(c, it0, false);
    a.fout = c->f[c->cur ^ (int)(n & 1)];  // a block reads and writes its own nodes only
    OnchipArgs o = {};
    o.tag = c->chip->tag;
    o.serial = next_serial(c->chip);
    o.list = list;
    o.blk_sample = c->chip->blk_sample;
    o.omega = omega;
    o.gx = gx;
    if (launch(c, a, o, n, blocks) == hipSuccess) return PLB_OK;
    c->chip_state = -1;  // refused before anything ran
    return PLB_ERR_HIP;
}

void onchip_batch_next(plb_ctx* c, int64_t n) { c->chip->tag += (uint32_t)n + 2; }

}  // namespace plb
