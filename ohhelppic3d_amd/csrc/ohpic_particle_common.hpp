// ohpic_particle_common.hpp -- device helpers shared by the FP64 and the
// mixed-precision particle kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "ohpic_internal.hpp"

namespace ohpic {
namespace {

// Minimum waves per SIMD the fused kernel is compiled for (register budget).
#ifndef OHPIC_PUSH_MIN_WAVES
#define OHPIC_PUSH_MIN_WAVES 1
#endif

constexpr int kLeaveCap = 32;  // per-wave buffer of particles that left the tile
constexpr int kStash = 64;     // per-wave stash of particles that stayed (below)

// Output of the particles that stay in their tile.  The front run of the new
// bin is written in blocks of 64 slots, each by one wavefront with every lane
// storing its own slot: full 128-byte lines.  (A copy in this kernel's shape
// reaches 5.1 TB/s with such stores and 3.6-4.8 TB/s (FP32) or 4.4-4.9 TB/s
// (FP64) when the wavefronts' 64 slots start anywhere.)  A lane whose particle
// left takes one from the wavefront's stash instead; a wavefront whose stash
// is too small for its holes puts its stayers there and stores nothing, which
// happens once per kStash leavers or so.  The stashes that are left at the end
// follow the last block as one run, or, of a tile split among several work
// items, go to the back run, so the front run has no gap.

// Rank of this lane among the set lanes below it.
__device__ __forceinline__ int lane_rank(unsigned long long m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                          __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// A value every lane holds, in scalar registers.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float uniform(float v)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ int64_t uniform(int64_t v)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double uniform(double v)
{
    return __longlong_as_double(uniform((int64_t)__double_as_longlong(v)));
}

// The value, hidden from the optimizer: what is computed from it is not hoisted
// out of the loop around.
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}
// Element i of an LDS array as the base of reads at constant offsets from it.
// (Opaque, so that every offset goes into the LDS instruction and not into an
// address register of its own.)
template <typename T>
using lds_ptr = const __attribute__((address_space(3))) T *;

template <typename T>
__device__ __forceinline__ lds_ptr<T> lds_base(const T *a, unsigned i)
{
    lds_ptr<T> p = (lds_ptr<T>)a + i;
    asm("" : "+v"(p));
    return p;
}
template <typename T>
__device__ __forceinline__ T lds_read(lds_ptr<T> p, int i)
{
    return p[i];
}
__device__ __forceinline__ float2 lds_read(lds_ptr<float2> p, int i)
{
    typedef float f2v __attribute__((ext_vector_type(2)));
    const f2v v = ((lds_ptr<f2v>)p)[i];
    return make_float2(v.x, v.y);
}

// LDS written by other lanes of this wavefront is visible after this.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int WO>
__device__ __forceinline__ void cic_w(double r, double &w0, double &w1)
{
    // WO 0: lower node gets r (the reference's order); WO 1: lower gets 1-r
    if (WO == 0) {
        w0 = r;
        w1 = 1.0 - r;
    } else {
        w0 = 1.0 - r;
        w1 = r;
    }
}

// periodic_particle_boundary.f90:46-52: the two comparisons in this order
__device__ __forceinline__ double apply_periodic(double p, int n)
{
    const double dn = (double)n;
    if (p < 0) p = dn + p;
    if (p >= dn) p = p - dn;
    return p;
}

__device__ __forceinline__ int lane_id() { return __lane_id(); }

// The value lane `src` holds, for a wave-uniform `src`: v_readlane through a
// scalar register (a shuffle would route all 64 lanes through the LDS unit,
// which the gather and deposit keep busy).
__device__ __forceinline__ int lane_bcast(int v, int src) { return __builtin_amdgcn_readlane(v, src); }
__device__ __forceinline__ unsigned long long lane_bcast(unsigned long long v, int src)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), src);
    return ((unsigned long long)hi << 32) | lo;
}

// Particle state streams through each step once, so its full-line accesses
// carry the non-temporal hint: 256^3 x 32 ppc mixed 11.82 -> 10.91 ms per
// launch, 256^3 x 16 FP64 11.14 -> 10.42 ms, and the field kernels of smaller
// grids find their arrays in the last-level cache (the 32^3 x 16 push loses
// 1 us, its field solve gains 1.5 us).  Partial lines (leavers, the ends of
// runs) are stored without it: they are merged in L2.
template <typename T>
__device__ __forceinline__ T sload(const T *p, int64_t i)
{
    return __builtin_nontemporal_load(&as_global(p)[i]);
}

template <bool NT, typename T>
__device__ __forceinline__ void sstore(T *p, int64_t i, T v)
{
    if (NT)
        __builtin_nontemporal_store(v, &as_global(p)[i]);
    else
        as_global(p)[i] = v;
}

// relaxed device-scope atomic add on global memory (as atomicAdd)
__device__ __forceinline__ unsigned long long gatomic_add(unsigned long long *p,
                                                          unsigned long long v)
{
    return __hip_atomic_fetch_add(as_global(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// *p += 1 for every active lane, by one atomic of the wavefront: flag counters
// are one address that every XCD adds to, and a fast plasma has every lane
// there (64^3 x 32 ppc, thermal speed 3 cells per step, chunks 1: 272 ms per
// step with an atomic per lane, 20.4 with one per wavefront, FP64 and mixed).
__device__ __forceinline__ void count_lanes(unsigned long long *p)
{
    const unsigned long long m = __ballot(1);
    if (lane_rank(m) == 0) gatomic_add(p, (unsigned long long)__popcll(m));
}

// counter[t] += 1 for every active lane with `valid`; returns the lane's
// value of the counter before its own increment.  Lanes of the wavefront
// that share t are served by one atomic (their leader adds the group size and
// each lane takes old + its rank in the group), for the first kAggRounds
// distinct values of t; the remaining lanes add individually.  Particle lists
// written by the step kernels keep each source tile's particles together, so
// a wavefront usually targets one to a few bins.
constexpr int kAggRounds = 4;

__device__ __forceinline__ unsigned long long wave_counter_add(unsigned long long *counter, int t,
                                                               bool valid)
{
    const int lane = __lane_id();
    const unsigned long long lt = (1ull << lane) - 1ull;
    unsigned long long todo = __ballot(valid);
    unsigned long long result = 0ull;
    for (int r = 0; r < kAggRounds && todo; ++r) {
        const int leader = __ffsll((unsigned long long)todo) - 1;
        const int tl = lane_bcast(t, leader);
        const unsigned long long m = __ballot(valid && t == tl) & todo;
        unsigned long long old = 0ull;
        if (lane == leader) old = gatomic_add(&counter[tl], (unsigned long long)__popcll(m));
        old = lane_bcast(old, leader);
        if ((m >> lane) & 1ull) result = old + (unsigned long long)__popcll(m & lt);
        todo &= ~m;
    }
    if ((todo >> lane) & 1ull) result = gatomic_add(&counter[t], 1ull);
    return result;
}

// One species of a work item: its bin's runs, capacity and first slot, and (in
// list mode) the item's reserved range of the species' list.
struct SpecMeta {
    int F, B, cap;
    int64_t base, list;
};

// Slots per chunk of a bin holding cnt particles, a multiple of the 64-slot
// blocks of the front run.
__device__ __forceinline__ int chunk_size(int cnt, int nchunks)
{
    return ((cnt + nchunks - 1) / nchunks + 63) & ~63;
}

// Thread s < ns loads species s.
template <bool LIST>
__device__ __forceinline__ void load_meta(SpecMeta *meta, const InstDev *__restrict__ I,
                                          const WorkItem &it, int par, int tid, int ns)
{
    if (tid >= ns) return;
    const SpecDev &S = I->sp[tid];
    SpecMeta m;
    m.cap = gload(S.bin_cap, it.tile);
    const unsigned long long word = gload(S.count[par], it.tile);
    m.base = gload(S.bin_base, it.tile);
    m.F = min(bin_front(word), m.cap);
    m.B = min(bin_back(word), m.cap - m.F);
    m.list = 0;
    if (LIST) {  // one reservation per item and species
        const int cnt = m.F + m.B;
        const int per = chunk_size(cnt, it.nchunks);
        const int n = min(cnt, (it.chunk + 1) * per) - it.chunk * per;
        if (n > 0)
            m.list = (int64_t)gatomic_add(&S.count[par ^ 1][0], (unsigned long long)n);
    }
    meta[tid] = m;
}

// The front run of a split tile's bin is shared by its items: a wavefront takes
// each of its blocks from a counter of the tile's own, and adds them to the
// bin's word when the species is done.  (Taken from the word itself, which all
// arrivals add to, with the words of 15 other tiles in its cache line: 16^3 x
// 1000 ppc, 12 items per tile, 1285 us per step FP64 and 1465 mixed, against
// 1017 and 1086.  Items with parts of the front run of their own and a launch
// to join them: 1080 and 1188.)  It is called, and its answer waited for, where
// only split tiles come: an answer pending in a register that whole tiles share
// makes them wait for their loads ahead and their stores as well (96^3 x 32 ppc
// FP64 1105 -> 1120 us per launch, 128^3 x 8 mixed in 4^3 tiles 546 -> 582).
__device__ __forceinline__ int claim_block(const InstDev *__restrict__ I, const WorkItem &it, int s)
{
    int32_t *p = &I->claims[(int64_t)(it.slot - it.chunk) * kMaxSpecies + s];
    return uniform(
        __hip_atomic_fetch_add(as_global(p), 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// Adds the m stayers of a tile that is one item.  Arrivals look at the word as
// they add to it (route_back); the runs of a bin that is too full also meet
// where its stayers come last, which the end of the step (k_end_step_b), or
// here the CHECKing item itself, sees: a step is redone only if stayers and
// arrivals together exceed a bin.  (With the whole old count reserved at the
// start of the step, 32^3 x 16 ppc at a thermal speed of 0.3 cells per step
// overflowed every step: 540 us against 121, FP64.)
template <bool CHECK>
__device__ __forceinline__ bool add_front(unsigned long long *word, int m, int cap)
{
    if (CHECK) {
        const unsigned long long old = gatomic_add(word, (unsigned long long)m);
        return (int64_t)bin_front(old) + m + bin_back(old) > cap;
    }
    if (m > 0) gatomic_add(word, (unsigned long long)m);
    return false;
}

// The item's kinetic-energy partials, summed over its W wavefronts in order.
template <int W>
__device__ __forceinline__ void write_ke(const InstDev *__restrict__ I, const WorkItem &it, int tid,
                                         int ns, const double (*ke)[W])
{
    if (tid >= 2 * ns) return;
    const int s = tid >> 1, k = (tid & 1) ? kMaxSpecies + s : s;
    double v = 0.0;
    for (int w = 0; w < W; ++w) v += ke[k][w];
    gstore(I->ke_partial, (int64_t)k * I->nitems + it.slot, 0.5 * I->sp[s].mass * v);
}

// Sum over the wavefront, in lane 0.
__device__ __forceinline__ double wave_total(double v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

}  // namespace
}  // namespace ohpic
