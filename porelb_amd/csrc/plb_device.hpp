// plb_device.hpp -- device code of one node update, shared by the kernels that
// advance the lattice: pull-table decoding,
// gathers, and the FP64 and shifted FP32/FP16 collisions.
#pragma once

#include <type_traits>

#include "plb_internal.hpp"

namespace plb {

struct StepArgs;
StepArgs make_args(plb_ctx* c, int64_t it, bool write_macros);

struct StepArgs {
    const void* fin;
    void* fout;
    const int32_t* tab;
    const int32_t* tdesc;
    const uint32_t* toff;
    const uint16_t* toff16;
    const int32_t* twide;
    int64_t N, Npad;
    double omega, gx, rho0;
    int64_t it;
    int write_macros;
    double* macros;  // [4][Npad]
    unsigned long long* fault;
    const uint32_t* perm;
    float scale, inv_scale;
    // BITMAP index: voxel position V = x + nx*(ly + py*(z + nz*yb)), y = yb*py + ly
    const uint2* bm;
    const uint32_t* vox;
    uint32_t nx, ny, nz, py;
    FastDiv div_nx, div_py, div_nz;
    // Graph replays: the step number is it + *it_base (set before each replay).
    const int64_t* it_base;
    int stochastic;  // FP16 stores: stochastic rounding
    int has_const;   // the table may hold constant entries (reference bounce order)
    // Node id that keys the rounding stream: the V-order id of the node
    // (within its sample for batches), so every node order and a batch give
    // the same results as a single lattice in the V order.  Null: identity.
    const uint32_t* key_perm;
    // The same keys as runs per 64-node tile (null: load key_perm per node).
    const uint4* kseg;
};

__device__ __forceinline__ StepArgs with_step(const StepArgs& a)
{
    StepArgs b = a;
    if (a.it_base) b.it += *a.it_base;
    return b;
}

// ---------------------------------------------------------------- FP64, reference order
__device__ __forceinline__ double feq_ref(int k, double rho, double u, double v, double w)
{
    // porelb.c:8-12, same operations in the same order.
    double uv, eu, x;
    eu = EX[k] * u + EY[k] * v + EZ[k] * w;
    uv = u * u + v * v + w * w;
    x = TP[k] * rho * (1.0 + 3 * eu + 4.5 * eu * eu - 1.5 * uv);
    return x;
}

__device__ __forceinline__ void record_fault(const StepArgs& a, int64_t i, double rho)
{
    const uint64_t g = a.perm ? (uint64_t)a.perm[i] : (uint64_t)i;
    const uint64_t key = ((uint64_t)a.it << 32) | g;
    atomicMin(a.fault, (unsigned long long)key);
    a.macros[i] = rho;  // rho of the offending node, read back by plb_last_fault
}

// A step after the first faulting step stores nothing, so the state stays
// that of the faulting step (the reference exits there); nor does any step
// queued behind an on-chip run that gave up (HOLD_FAULT).  The fault word is
// loaded at kernel entry but only consulted before the stores, so it adds no
// latency in front of the table and population loads.
__device__ __forceinline__ bool frozen(unsigned long long fk, int64_t it)
{
    return fk != NO_FAULT && ((int64_t)(fk >> 32) < it || fk == HOLD_FAULT);
}

// ---------------------------------------------------------------- phases of one node
// A node update runs in four phases so a thread can interleave two nodes
// (issue both nodes' index loads, then both nodes' gathers, before waiting):
//   issue_entries  -> index loads (I32: 18 words; TILE8: 4 words + 1 short + 18 scalar
//                     descriptors of the wave's tile)
//   decode_entries -> t[1..18]: >= 0 source node, -1 bounce, -2 constant
//   gather         -> the 19 stored populations
//   collide_*      -> collision and the 19 stores

template <int IDX>
struct Entries {
    int32_t t[Q];                // I32: raw entries; after decode: decoded
    uint32_t w[TILE8_WORDS];     // TILE8: packed offsets of this lane
    int32_t desc[Q];             // TILE8: the tile's descriptors (uniform)
    uint32_t v;                  // BITMAP: the node's voxel position
};

// ---------------------------------------------------------------- BITMAP sources
// Periodic neighbour coordinate c - e (e in {-1, 0, 1}) on [0, n).
__device__ __forceinline__ uint32_t wrap_sub(uint32_t c, int e, uint32_t n)
{
    if (e > 0) return c == 0 ? n - 1 : c - 1;
    if (e < 0) return c + 1 == n ? 0 : c + 1;
    return c;
}

// Voxel position of the pull source x - e_j, for any node.
__device__ __forceinline__ uint32_t bitmap_src_general(const StepArgs& a, int j, uint32_t x, uint32_t y,
                                                       uint32_t z)
{
    const uint32_t xs = wrap_sub(x, EX[j], a.nx);
    const uint32_t ys = wrap_sub(y, EY[j], a.ny);
    const uint32_t zs = wrap_sub(z, EZ[j], a.nz);
    const uint32_t yb = fastdiv(ys, a.div_py);
    const uint32_t ly = ys - yb * a.py;
    return ((yb * a.nz + zs) * a.py + ly) * a.nx + xs;
}

__device__ __forceinline__ void bitmap_coords(const StepArgs& a, uint32_t v, uint32_t& x, uint32_t& y,
                                              uint32_t& z, uint32_t& ly)
{
    const uint32_t r1 = fastdiv(v, a.div_nx);
    x = v - r1 * a.nx;
    const uint32_t r2 = fastdiv(r1, a.div_py);
    ly = r1 - r2 * a.py;
    const uint32_t yb = fastdiv(r2, a.div_nz);
    z = r2 - yb * a.nz;
    y = yb * a.py + ly;
}

// Node id of the pore at voxel position v, or TAB_BOUNCE for a solid voxel
// (half-way bounce-back): the word's pore count plus the pores below v.
__device__ __forceinline__ int32_t bitmap_lookup(uint2 wd, uint32_t v)
{
    const uint32_t b = v & 31u;
    const uint32_t below = __builtin_amdgcn_ubfe(wd.x, 0, b);
    const int32_t id = (int32_t)(wd.y + __builtin_popcount(below));
    return ((wd.x >> b) & 1u) ? id : TAB_BOUNCE;
}

// A read through the constant address space, for data no kernel of the
// launch writes (sample tables, pull-table descriptors): it stays a scalar
// load where the address is uniform, also in kernels that store elsewhere.
template <typename T>
__device__ __forceinline__ T ld_const(const T* q)
{
    return *(const __attribute__((address_space(4))) T*)q;
}

// CONST_DESC: read the TILE8 descriptors through the constant address space
// (for loops that also store; one-node kernels get scalar loads anyway).
template <int LAYOUT, int IDX, bool CONST_DESC = false>
__device__ __forceinline__ void issue_entries(const StepArgs& a, int64_t i, Entries<IDX>& e)
{
    // Index words are read once per step: non-temporal loads keep them from
    // displacing population lines that neighbouring tiles read again.
    if constexpr (IDX == PLB_INDEX_I32) {
#pragma unroll
        for (int j = 1; j < Q; j++) e.t[j] = __builtin_nontemporal_load(a.tab + tpos<LAYOUT>(j - 1, i, a.Npad));
    } else if constexpr (IDX == PLB_INDEX_BITMAP) {
        e.v = __builtin_nontemporal_load(a.vox + i);
    } else {
        // TILE8: the wave is one 64-node tile, so its 18 descriptors are
        // uniform (scalar loads); each lane reads 4 words and a short of packed
        // offsets.
        const int64_t tile = __builtin_amdgcn_readfirstlane((int)(i >> 6));
        const uint32_t* o = a.toff + tile * TILE8_FULL * 64 + (i & 63);
#pragma unroll
        for (int k = 0; k < TILE8_FULL; k++) e.w[k] = __builtin_nontemporal_load(o + k * 64);
        e.w[TILE8_FULL] = __builtin_nontemporal_load(a.toff16 + tile * 64 + (i & 63));
        const int32_t* d = a.tdesc + tile * (Q - 1);
        if constexpr (CONST_DESC) {
            // never written while steps run: scalar loads even in a loop
            // that stores, where the compiler could not prove it otherwise
#pragma unroll
            for (int j = 1; j < Q; j++) e.desc[j] = ld_const(d + j - 1);
        } else {
#pragma unroll
            for (int j = 1; j < Q; j++) e.desc[j] = d[j - 1];
        }
    }
}

template <int IDX>
__device__ __forceinline__ void decode_entries(const StepArgs& a, int64_t i, Entries<IDX>& e)
{
    if constexpr (IDX == PLB_INDEX_BITMAP) {
        const uint32_t v = e.v;
        uint32_t x, y, z, ly;
        bitmap_coords(a, v, x, y, z, ly);
        // Away from pencil edges and the periodic y/z boundary every source is
        // a fixed offset in node order; x wraps are a per-lane correction.
        const bool inner = (int)ly >= 1 && (int)ly <= (int)a.py - 2 && (int)y >= 1 &&
                           (int)y <= (int)a.ny - 2 && (int)z >= 1 && (int)z <= (int)a.nz - 2;
        uint32_t vs[Q];
        if (__builtin_amdgcn_ballot_w64(!inner) == 0) {
            const uint32_t xm = x == 0 ? a.nx : 0u;            // source at x-1 wraps to nx-1
            const uint32_t xp = x + 1 == a.nx ? a.nx : 0u;     // source at x+1 wraps to 0
            const uint32_t row = a.nx, plane = a.nx * a.py;
#pragma unroll
            for (int j = 1; j < Q; j++) {
                uint32_t d = v - (uint32_t)EX[j] - (uint32_t)EY[j] * row - (uint32_t)EZ[j] * plane;
                if (EX[j] > 0) d += xm;
                if (EX[j] < 0) d -= xp;
                vs[j] = d;
            }
        } else {
#pragma unroll
            for (int j = 1; j < Q; j++) vs[j] = bitmap_src_general(a, j, x, y, z);
        }
        uint2 wd[Q];
#pragma unroll
        for (int j = 1; j < Q; j++) wd[j] = a.bm[vs[j] >> 5];
#pragma unroll
        for (int j = 1; j < Q; j++) e.t[j] = bitmap_lookup(wd[j], vs[j]);
    } else if constexpr (IDX == PLB_INDEX_TILE8) {
        int32_t any = 0;
#pragma unroll
        for (int j = 1; j < Q; j++) {
            // one select: 0..253 -> base + v, 254 -> -2 (const), 255 -> -1 (bounce)
            const int32_t v = (int32_t)((e.w[(j - 1) >> 2] >> (8 * ((j - 1) & 3))) & 0xffu);
            e.t[j] = v < 254 ? e.desc[j] + v : v - 256;
            any |= e.desc[j];
        }
        if (any < 0) {  // a (tile, direction) pair of this tile is wide
#pragma unroll
            for (int j = 1; j < Q; j++)
                if (e.desc[j] < 0)
                    e.t[j] = __builtin_nontemporal_load(a.twide + (int64_t)(-e.desc[j] - 1) * 64 + (i & 63));
        }
    }
}

// 19 gathers: rest population of the node, then per direction the source
// node's slot j (stream) or the node's own slot re[j] (bounce; constant
// entries read that slot too and are replaced afterwards).
template <typename S, int LAYOUT>
__device__ __forceinline__ void gather(const StepArgs& a, int64_t i, const int32_t t[Q], S raw[Q])
{
    const S* __restrict__ fin = (const S*)a.fin;
    raw[0] = fin[fpos<LAYOUT>(0, i, a.Npad)];
#pragma unroll
    for (int j = 1; j < Q; j++) {
        const int64_t src = t[j] >= 0 ? fpos<LAYOUT>(j, t[j], a.Npad) : fpos<LAYOUT>(RE[j], i, a.Npad);
        raw[j] = fin[src];
    }
}

// Where the post-collision population j of node i is stored.  MODE 0: the
// other buffer, slot j (pull, two buffers).  One buffer with the AA pattern:
// MODE 1 (local steps) the node's own slot re[j]; MODE 2 (neighbour steps)
// slot j of the node downstream, t[re[j]] (x + e_j), or the node's own slot
// re[j] when that neighbour is solid (half-way bounce-back).  The rest
// population stays in slot 0.
template <int LAYOUT, int MODE>
__device__ __forceinline__ int64_t out_pos(const StepArgs& a, int64_t i, const int32_t t[Q], int j)
{
    if constexpr (MODE == 0) return fpos<LAYOUT>(j, i, a.Npad);
    else if constexpr (MODE == 1) return fpos<LAYOUT>(RE[j], i, a.Npad);
    else {
        if (j == 0) return fpos<LAYOUT>(0, i, a.Npad);
        return t[RE[j]] >= 0 ? fpos<LAYOUT>(j, t[RE[j]], a.Npad) : fpos<LAYOUT>(RE[j], i, a.Npad);
    }
}

// Stores of the step kernels: non-temporal, or (KEEP, and `keep` of the wave)
// plain, where the next step is to find them in the memory-side cache.
template <bool KEEP, typename S>
__device__ __forceinline__ void st_dev(S* p, S v, bool keep)
{
    if (KEEP && keep) {
        asm volatile("");   // or the compiler makes one plain store of the two
        *p = v;
        asm volatile("");
    } else if constexpr (sizeof(S) == 2) {
        __builtin_nontemporal_store(__half_as_ushort(v), (unsigned short*)p);
    } else {
        __builtin_nontemporal_store(v, p);
    }
}

// FP64 collision in the reference's evaluation order (porelb.c:326-362) on
// the streamed populations f of node i; put(j, value) takes the results.
template <typename Put>
__device__ __forceinline__ void relax_f64(const StepArgs& a, int64_t i, const double f[Q], unsigned long long fk,
                                          Put put)
{
    double rho = 0.0, rhou = 0.0, rhov = 0.0, rhow = 0.0;
#pragma unroll
    for (int j = 0; j < Q; j++) {
        rho += f[j];
        rhou += EX[j] * f[j];
        rhov += EY[j] * f[j];
        rhow += EZ[j] * f[j];
    }
    if (frozen(fk, a.it)) return;
    if ((rho > 1.2) | (rho < 0.5)) record_fault(a, i, rho);
    if (a.it > 0) rhou += 0.5 * a.gx;
    const double u = rhou / rho, v = rhov / rho, w = rhow / rho;
    if (a.write_macros) {
        a.macros[i] = rho;
        a.macros[a.Npad + i] = u;
        a.macros[2 * a.Npad + i] = v;
        a.macros[3 * a.Npad + i] = w;
    }
    const double omega = a.omega, Xforce = a.gx;
#pragma unroll
    for (int j = 0; j < Q; j++) {
        const double o = (1.0 - omega) * f[j] +
                         (omega + (1.0 - 0.5 * omega) * 3.0 * (EX[j] - u) * Xforce) *
                             feq_ref(j, rho, u, v, w);
        put(j, o);
    }
}

template <int LAYOUT, int MODE = 0, bool KEEP = false>
__device__ __forceinline__ void collide_f64(const StepArgs& a, int64_t i, const int32_t t[Q],
                                            double f[Q], unsigned long long fk, bool keep)
{
    double* __restrict__ fout = (double*)a.fout;
    if constexpr (MODE == 0) {  // constant entries: reference bounce order, two buffers only
#pragma unroll
        for (int j = 1; j < Q; j++)
            if (t[j] == TAB_CONST) f[j] = TP[j] * a.rho0 * 1.0;  // feq(rho0, u=0) = initial f1
    }
    relax_f64(a, i, f, fk, [&](int j, double o) {
        st_dev<KEEP>(fout + out_pos<LAYOUT, MODE>(a, i, t, j), o, keep);
    });
}

// ---------------------------------------------------------------- shifted FP32 / FP16 storage
// The collision works in the stored scale: ds_j = d_j * sc (sc = 2^k for
// FP16, 1 for FP32).  Scaling by a power of two commutes with every FP32
// rounding, so the moments unscaled once and the stores with the scale
// folded into the collision constants are bit-identical to unscaling each
// population and scaling each store.
__device__ __forceinline__ float to_float(float v) { return v; }
__device__ __forceinline__ float to_float(__half v) { return __half2float(v); }
// The collision's result as stored: FP32 as it is, FP16 rounded to nearest.
template <typename S>
__device__ __forceinline__ S to_stored(float v)
{
    if constexpr (sizeof(S) == 2) return __float2half_rn(v);
    else return v;
}

// Stochastic rounding of FP16 stores.  v_cvt_sr_f16_f32 rounds up with
// probability equal to the dropped fraction of an FP16 ulp, taken from the
// random word r; the expected stored value equals the FP32 value, so the
// sub-ulp increments of a flow near steady state accumulate instead of
// being rounded away.  r for direction j of a node: a 32-bit hash of the
// node id and the step (lowbias32, C. Wellons, "Prospecting for hash
// functions", 2018) plus j times the golden-ratio constant, which keeps every
// direction's word uniformly distributed.
typedef _Float16 plb_half2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t mix32(uint32_t x)
{
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}
template <typename S>
__device__ __forceinline__ S to_stored_sr(float v, uint32_t r)
{
    if constexpr (sizeof(S) == 2) {
        const plb_half2 h = __builtin_amdgcn_cvt_sr_f16_f32(plb_half2{0, 0}, v, r, false);
        return __ushort_as_half(__builtin_bit_cast(unsigned short, h[0]));
    } else {
        return v;
    }
}

// The collision on the streamed deviations ds (in the stored scale) of node
// i; put(j, stored value) takes the results.
template <typename S, typename Put>
__device__ __forceinline__ void relax_shift(const StepArgs& a, int64_t i, const float ds[Q], unsigned long long fk,
                                            uint32_t key, Put put)
{
    constexpr bool scaled = sizeof(S) == 2;
    const float inv = a.inv_scale, sc = a.scale;
    float drho = 0.f, jx = 0.f, jy = 0.f, jz = 0.f;
#pragma unroll
    for (int j = 0; j < Q; j++) {
        drho += ds[j];
        if (EX[j]) jx += EX[j] > 0 ? ds[j] : -ds[j];
        if (EY[j]) jy += EY[j] > 0 ? ds[j] : -ds[j];
        if (EZ[j]) jz += EZ[j] > 0 ? ds[j] : -ds[j];
    }
    if constexpr (scaled) {
        drho *= inv;
        jx *= inv;
        jy *= inv;
        jz *= inv;
    }
    const float rho0 = (float)a.rho0;
    const float rho = rho0 + drho;
    if (frozen(fk, a.it)) return;
    if ((rho > 1.2f) | (rho < 0.5f)) record_fault(a, i, (double)rho);
    const float F = (float)a.gx;
    if (a.it > 0) jx += 0.5f * F;
    const float rinv = 1.0f / rho;
    const float u = jx * rinv, v = jy * rinv, w = jz * rinv;
    if (a.write_macros) {
        a.macros[i] = (double)rho;
        a.macros[a.Npad + i] = (double)u;
        a.macros[2 * a.Npad + i] = (double)v;
        a.macros[3 * a.Npad + i] = (double)w;
    }
    const float omega = (float)a.omega;
    const float c1 = 1.0f - omega;
    const float c2 = (1.0f - 0.5f * omega) * 3.0f * F;
    // Fused multiply-adds are written out (the library is built without
    // contraction for the FP64 path's sake); this path is held to a
    // tolerance against FP64, not to bitwise equality.
    const float usq = 1.5f * fmaf(u, u, fmaf(v, v, w * w));
    const float fu = -c2 * u;  // force term c2 (e_jx - u) for e_jx = 0, then +-c2
    // the store scale folded into the constants of the dfeq and force terms
    const float omega_s = scaled ? omega * sc : omega;
    const float f0s = scaled ? fu * sc : fu, fps = scaled ? (fu + c2) * sc : fu + c2,
                fms = scaled ? (fu - c2) * sc : fu - c2;
    // The rounding mode is uniform: one loop per mode under a scalar branch.
    auto relax = [&](auto stochastic) {
        constexpr bool SR = decltype(stochastic)::value;
        uint32_t rnd = 0;
        if constexpr (SR) rnd = mix32(key ^ mix32((uint32_t)a.it * 0x9e3779b9u + 0x632be5abu));
#pragma unroll
        for (int j = 0; j < Q; j++) {
            float eu = 0.f;
            if (EX[j]) eu = EX[j] > 0 ? u : -u;
            if (EY[j]) eu += EY[j] > 0 ? v : -v;
            if (EZ[j]) eu += EZ[j] > 0 ? w : -w;
            const float P = fmaf(eu, fmaf(4.5f, eu, 3.0f), -usq);
            const float wj = (float)TP[j];
            const float dfeq = wj * fmaf(rho, P, drho);
            const float feq = fmaf(wj, rho0, dfeq);
            const float frc = EX[j] > 0 ? fps : (EX[j] < 0 ? fms : f0s);
            const float o = fmaf(c1, ds[j], fmaf(omega_s, dfeq, frc * feq));
            if constexpr (SR)
                put(j, to_stored_sr<S>(o, rnd + (uint32_t)j * 0x9e3779b9u));
            else
                put(j, to_stored<S>(o));
        }
    };
    if constexpr (scaled) {
        if (__builtin_amdgcn_readfirstlane(a.stochastic))
            relax(std::true_type{});
        else
            relax(std::false_type{});
    } else {
        relax(std::false_type{});
    }
}

template <typename S, int LAYOUT, int MODE = 0, bool KEEP = false>
__device__ __forceinline__ void collide_shift(const StepArgs& a, int64_t i, const int32_t t[Q],
                                              const S raw[Q], unsigned long long fk, uint32_t key, bool keep)
{
    S* __restrict__ fout = (S*)a.fout;
    float ds[Q];
#pragma unroll
    for (int j = 0; j < Q; j++) ds[j] = to_float(raw[j]);
    if constexpr (MODE == 0) {
        if (__builtin_amdgcn_readfirstlane(a.has_const)) {  // constant entries: reference bounce order only
#pragma unroll
            for (int j = 1; j < Q; j++)
                if (t[j] == TAB_CONST) ds[j] = 0.f;
        }
    }
    S* __restrict__ onode = fout + fpos<LAYOUT>(0, i, a.Npad);
    relax_shift<S>(a, i, ds, fk, key, [&](int j, S v) {
        if constexpr (MODE == 0) st_dev<KEEP>(onode + fpos<LAYOUT>(j, 0, a.Npad), v, keep);
        else st_dev<KEEP>(fout + out_pos<LAYOUT, MODE>(a, i, t, j), v, keep);
    });
}

// Key of node i's stochastic-rounding stream (FP16 storage only): from the
// tile's runs of consecutive keys (one scalar load per wave), or per node in
// the tiles marked as not fitting three runs.  Called after the gathers are
// issued, so the scalar load's latency hides behind theirs.
template <typename S>
__device__ __forceinline__ uint32_t sr_key(const StepArgs& a, int64_t i)
{
    if constexpr (sizeof(S) == 2)
        if (a.stochastic && a.key_perm) {
            if (a.kseg) {
                const int64_t tile = __builtin_amdgcn_readfirstlane((int)(i >> 6));
                const uint32_t* d = (const uint32_t*)(a.kseg + tile);
                const uint32_t b0 = ld_const(d), b1 = ld_const(d + 1), b2 = ld_const(d + 2), st = ld_const(d + 3);
                const uint32_t lane = (uint32_t)i & 63u;
                const uint32_t base = lane >= ((st >> 8) & 0xffu) ? b2 : (lane >= (st & 0xffu) ? b1 : b0);
                if (!(st >> 31)) return base + lane;
            }
            return a.key_perm[i];
        }
    return (uint32_t)i;
}

template <typename S, int LAYOUT, int MODE = 0, bool KEEP = false>
__device__ __forceinline__ void collide_any(const StepArgs& a, int64_t i, const int32_t t[Q], S raw[Q],
                                            unsigned long long fk, uint32_t key, bool keep = false)
{
    if constexpr (sizeof(S) == 8)
        collide_f64<LAYOUT, MODE, KEEP>(a, i, t, (double*)raw, fk, keep);
    else
        collide_shift<S, LAYOUT, MODE, KEEP>(a, i, t, raw, fk, key, keep);
}

template <typename S, int LAYOUT, int IDX, bool CONST_DESC = false, bool KEEP = false>
__device__ __forceinline__ void node_any(const StepArgs& a, int64_t i, unsigned long long fk, bool keep = false)
{
    Entries<IDX> e;
    issue_entries<LAYOUT, IDX, CONST_DESC>(a, i, e);
    decode_entries<IDX>(a, i, e);
    S raw[Q];
    gather<S, LAYOUT>(a, i, e.t, raw);
    const uint32_t key = sr_key<S>(a, i);
    collide_any<S, LAYOUT, 0, KEEP>(a, i, e.t, raw, fk, key, keep);
}

// Pull sources t[1..18] of internal node k, decoded by one lane on its own
// (the lanes of a wave may hold unrelated nodes).
template <int LAYOUT, int IDX>
__device__ __forceinline__ void lane_sources(const StepArgs& a, int64_t k, int32_t t[Q])
{
    if constexpr (IDX == PLB_INDEX_I32) {
        Entries<IDX> e;
        issue_entries<LAYOUT, IDX>(a, k, e);
        for (int j = 1; j < Q; j++) t[j] = e.t[j];
    } else if constexpr (IDX == PLB_INDEX_BITMAP) {
        uint32_t x, y, z, ly;
        bitmap_coords(a, a.vox[k], x, y, z, ly);
        for (int j = 1; j < Q; j++) {
            const uint32_t vs = bitmap_src_general(a, j, x, y, z);
            t[j] = bitmap_lookup(a.bm[vs >> 5], vs);
        }
    } else {
        // Lanes of a wave hold unrelated nodes here: decode without the
        // per-wave descriptor shortcut.
        const int64_t tile = k >> 6;
        const int lane = (int)(k & 63);
        for (int j = 1; j < Q; j++) {
            const int32_t desc = a.tdesc[tile * (Q - 1) + j - 1];
            if (desc >= 0) {
                const int wi = (j - 1) >> 2;  // packed word holding direction j
                const uint32_t word = wi < TILE8_FULL ? a.toff[(tile * TILE8_FULL + wi) * 64 + lane]
                                                      : (uint32_t)a.toff16[tile * 64 + lane];
                const int32_t v = (int32_t)((word >> (8 * ((j - 1) & 3))) & 0xffu);
                t[j] = v == 255 ? TAB_BOUNCE : (v == 254 ? TAB_CONST : desc + v);
            } else {
                t[j] = a.twide[(int64_t)(-desc - 1) * 64 + lane];
            }
        }
    }
}

}  // namespace plb
