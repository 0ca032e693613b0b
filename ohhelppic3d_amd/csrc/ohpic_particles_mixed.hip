// ohpic_particles_mixed.hip -- mixed-precision particle kernels for gfx950.
//
// Storage per binned particle (24 B): for each axis one 32-bit word holding
// the particle's cell relative to its tile origin in the top 8 bits (signed)
// and its in-cell offset as a 24-bit fixed-point fraction in the low 24 bits,
// and FP32 velocities.  The tile is the bin the particle sits in, so the cell
// index costs no storage; the offset f24 * 2^-24 converts exactly to FP32.
// Contiguous particle lists (host transfers, re-binning input, the overflow
// retry) carry the tile index in a seventh word.
//
// Gather, Boris, drift and the deposit weights run in FP32; the new offset is
// rounded to the 24-bit grid (carry into the cell) and the deposit uses that
// stored position; every deposit contribution is rounded into the same int64
// fixed-point charge grid the FP64 path uses, so rho, the Poisson solve, E
// and the diagnostics stay FP64.  The periodic boundary is an integer wrap of
// the cell index.  Work decomposition, LDS staging, deposit blocks and
// re-binning are those of the FP64 kernel.
//
// What bounds it: 48 B per particle, and the instructions (about 220 VALU and
// 22 LDS per particle) with their latencies.  So the wrap and the new tile are
// found only for particles that leave, when their buffer is routed; the E
// gather reads its eight nodes before it uses one; and no iteration waits for
// its own stores.  With that, the aligned blocks of the front run and the
// larger workgroups below: 256^3 x 32 ppc 12.62 -> 10.4 ms, 128^3 x 64 with a
// density peak 3.93 -> 2.75 ms, 64^3 x 32 313 -> 219 us per launch.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "ohpic_internal.hpp"
#include "ohpic_kernels.hpp"
#include "ohpic_particle_common.hpp"
#include "ohpic_pcg.hpp"

namespace ohpic {

namespace {

#ifndef OHPIC_MX_PREFETCH
#define OHPIC_MX_PREFETCH 1
#endif
// Waves per SIMD the mixed kernel's registers are limited for: 5 (96 VGPRs)
// measured faster than the 4 the compiler picks on its own at 256^3 x 64 ppc
// with workgroups of 256 threads.  (Two workgroups of 512 are resident per CU,
// 4 waves per SIMD.)
#ifndef OHPIC_MX_MIN_WAVES
#define OHPIC_MX_MIN_WAVES 5
#endif
constexpr int kMxPrefetch = OHPIC_MX_PREFETCH;  // particles per lane loaded ahead

constexpr int kFracBits = 24;
constexpr uint32_t kFracOne = 1u << kFracBits;
constexpr uint32_t kFracMask = kFracOne - 1u;
constexpr float kFracScale = 16777216.0f;            // 2^24
constexpr float kFracUnit = 5.9604644775390625e-8f;  // 2^-24
constexpr float kMaxShift = 64.0f * kFracScale;      // largest drift per step: 64 cells

__device__ __forceinline__ uint32_t pos_word(int rel, uint32_t f24)
{
    return ((uint32_t)rel << kFracBits) | f24;
}
__device__ __forceinline__ int pos_rel(uint32_t w) { return (int32_t)w >> kFracBits; }
__device__ __forceinline__ float pos_frac(uint32_t w) { return (float)(w & kFracMask) * kFracUnit; }

struct PMx {
    uint32_t w[3];
    float v[3];
    int64_t id;
};

// binned form: buf[b][1..3] position words, buf[b][4..6] velocities
__device__ __forceinline__ PMx load_pmx(const SpecDev &S, int b, int64_t o, bool ids)
{
    PMx q;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        q.w[a] = gload((const uint32_t *)S.buf[b][1 + a], o);
        q.v[a] = gload((const float *)S.buf[b][4 + a], o);
    }
    q.id = ids ? gload(S.pid[b], o) : 0;
    return q;
}

__device__ __forceinline__ void store_pmx(const SpecDev &S, int b, int64_t o, const PMx &q,
                                          bool ids)
{
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        gstore((uint32_t *)S.buf[b][1 + a], o, q.w[a]);
        gstore((float *)S.buf[b][4 + a], o, q.v[a]);
    }
    if (ids) gstore(S.pid[b], o, q.id);
}

// The bin of one tile in one buffer: array bases offset to the bin's first
// element (uniform per workgroup, so they live in scalar registers) and
// particles addressed by a 32-bit byte offset (a bin holds < 2^30 particles),
// which the global instructions take directly (no 64-bit address arithmetic
// per particle).
struct BinView {
    const char *w[3];
    const char *v[3];
    const int64_t *id;
};

__device__ __forceinline__ BinView bin_view(const SpecDev &S, int b, int64_t base, bool ids)
{
    BinView r;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        r.w[a] = (const char *)((const uint32_t *)S.buf[b][1 + a] + base);
        r.v[a] = (const char *)((const float *)S.buf[b][4 + a] + base);
    }
    r.id = ids ? S.pid[b] + base : nullptr;
    return r;
}

__device__ __forceinline__ PMx load_bin(const BinView &bv, uint32_t slot, bool ids)
{
    const uint32_t off = slot * 4u;
    PMx q;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        q.w[a] = sload((const uint32_t *)(bv.w[a] + off), 0);
        q.v[a] = sload((const float *)(bv.v[a] + off), 0);
    }
    q.id = ids ? gload(bv.id, (int64_t)slot) : 0;
    return q;
}

// FULL: the wavefront stores full lines
template <bool FULL>
__device__ __forceinline__ void store_bin(const BinView &bv, uint32_t slot, const PMx &q, bool ids)
{
    const uint32_t off = slot * 4u;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        sstore<FULL>((uint32_t *)(bv.w[a] + off), 0, q.w[a]);
        sstore<FULL>((float *)(bv.v[a] + off), 0, q.v[a]);
    }
    if (ids) gstore(const_cast<int64_t *>(bv.id), (int64_t)slot, q.id);
}

// The particle's loads have completed from here on.
__device__ __forceinline__ void arrived(PMx &q, bool ids)
{
#pragma unroll
    for (int a = 0; a < 3; ++a) asm volatile("" : "+v"(q.w[a]), "+v"(q.v[a]));
    if (ids) asm volatile("" : "+v"(q.id));
}

// list form: the binned words plus the tile index in buf[b][0]
__device__ __forceinline__ void store_list_mx(const SpecDev &S, int b, int64_t o, const PMx &q,
                                              int tile, bool ids)
{
    gstore((int32_t *)S.buf[b][0], o, (int32_t)tile);
    store_pmx(S, b, o, q, ids);
}

template <int WO>
__device__ __forceinline__ void cic_wf(float r, float &w0, float &w1)
{
    if (WO == 0) {
        w0 = r;
        w1 = 1.0f - r;
    } else {
        w0 = 1.0f - r;
        w1 = r;
    }
}

// g mod n: one add or subtract for a cell within a box length of [0, n)
// (every step of a particle slower than a box length per step), a division
// only beyond that
__device__ __forceinline__ int wrap_cell(int g, int n)
{
    if (g < 0 || g >= n) {
        g += g < 0 ? n : -n;
        if (g < 0 || g >= n) g = ((g % n) + n) % n;
    }
    return g;
}

__device__ __forceinline__ void route_back_mx(const SpecDev &S, int nbuf, int t, const PMx &q,
                                              bool ids, unsigned long long *flags)
{
    const int cap = gload(S.bin_cap, t);
    const int64_t base = gload(S.bin_base, t);
    const unsigned long long old = gatomic_add(&S.count[nbuf][t], 1ull << 32);
    const int f = bin_front(old), b = bin_back(old);
    if (b + f < cap)
        store_pmx(S, nbuf, base + (cap - 1 - b), q, ids);
    else
        count_lanes(&flags[kFlagOverflow]);
}

template <bool IDS, int CAP>
struct BufMx {
    uint32_t w[3][CAP];
    float v[3][CAP];
    int64_t id[IDS ? CAP : 1];

    __device__ __forceinline__ void put(int i, const PMx &q, bool ids)
    {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            w[a][i] = q.w[a];
            v[a][i] = q.v[a];
        }
        if (IDS && ids) id[i] = q.id;
    }
    __device__ __forceinline__ void get(int i, PMx &q, bool ids) const
    {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            q.w[a] = w[a][i];
            q.v[a] = v[a][i];
        }
        if (IDS && ids) q.id = id[i];
    }
};

// The tile a position word triple relative to tile origin (lox, loy, loz)
// falls in after the periodic wrap; w becomes relative to that tile.
template <int TX, int TY, int TZ>
__device__ __forceinline__ int rebase_words(uint32_t w[3], const InstDev *__restrict__ I, int lox,
                                            int loy, int loz)
{
    const int ntx = I->nt[0], nty = I->nt[1];
    const int gx = wrap_cell(lox + pos_rel(w[0]), I->n[0]), gy = wrap_cell(loy + pos_rel(w[1]), I->n[1]),
              gz = wrap_cell(loz + pos_rel(w[2]), I->n[2]);
    const int tx = (int)((unsigned)gx / TX), ty = (int)((unsigned)gy / TY),
              tz = (int)((unsigned)gz / TZ);
    w[0] = pos_word(gx - tx * TX, w[0] & kFracMask);
    w[1] = pos_word(gy - ty * TY, w[1] & kFracMask);
    w[2] = pos_word(gz - tz * TZ, w[2] & kFracMask);
    // tile counts are below 2^24 (axes <= 1024 cells, tiles >= 4)
    return tx + (int)__umul24((unsigned)ty, (unsigned)ntx) +
           (int)__umul24((unsigned)tz, (unsigned)(ntx * nty));
}

// Routes the first `cnt` buffered leavers of this wavefront (lane l takes
// entry l) to the back runs of their new tiles.  The wrap and the new tile are
// found here, for up to kLeaveCap particles at once, and not for every
// particle of the sweep (about 60 of its 254 VALU instructions).
template <int TX, int TY, int TZ, bool IDS>
__device__ __forceinline__ void flush_leavers_mx(const BufMx<IDS, kLeaveCap> &lb, int cnt,
                                                 const InstDev *__restrict__ I, const SpecDev &S,
                                                 int nbuf, bool ids, int lox, int loy, int loz)
{
    wave_sync();
    const int l = lane_id();
    if (l < cnt) {
        PMx q;
        lb.get(l, q, ids);
        const int t = rebase_words<TX, TY, TZ>(q.w, I, lox, loy, loz);
        route_back_mx(S, nbuf, t, q, IDS && ids, I->flags);
    }
    wave_sync();
}

// Threads per workgroup: 512 for tiles of 512 cells, 256 for smaller ones.  Two
// large workgroups per CU share their E tile and charge block among twice the
// wavefronts and end a launch's last tiles sooner (8^3 tiles: 64^3 x 32 ppc
// 247 -> 223 us per launch, 128^3 x 64 with a density peak 3.10 -> 2.76 ms,
// 256^3 x 32 10.91 -> 10.78 ms); a small tile has too little work for them
// (8x8x4 tiles of a group of 32: 12.5 ms per 8 steps with 256, 15.6 with 512).
constexpr int mx_block(int cells) { return cells >= 512 ? 512 : 256; }
// With ids, the workgroups of 512 and the resident grid take the registers that
// 4 waves per SIMD leave them: 5 would need scratch.
constexpr int mx_min_waves(int cells, int mode, bool ids)
{
    return ids && (cells >= 512 || mode == kModeFusedQueue) ? 4 : OHPIC_MX_MIN_WAVES;
}

// IDS: instances may keep particle ids (each instance's track_ids says whether
// it does); without it no register, LDS or branch is spent on them.
template <int TX, int TY, int TZ, int WO, int MODE_, bool IDS>
__global__ void __launch_bounds__(mx_block(TX *TY *TZ))
    __attribute__((amdgpu_waves_per_eu(mx_min_waves(TX *TY *TZ, MODE_, IDS), 8)))
    k_particles_mixed(const InstDev *__restrict__ insts, const WorkItem *__restrict__ items,
                      const int *__restrict__ parity, unsigned int *__restrict__ queue,
                      int nitems)
{
    // kModeFusedQueue: the fused step over a resident grid, each workgroup
    // claiming work items in list order from `queue` until none is left
    constexpr bool QUEUE = (MODE_ == kModeFusedQueue);
    constexpr int MODE = QUEUE ? (int)kModeFused : MODE_;
    constexpr bool LIST = (MODE == kModeFusedList || MODE == kModeBoundaryList);
    constexpr bool PUSH = (MODE == kModeFused || MODE == kModeGatherPush || MODE == kModeFusedList);
    constexpr bool REBIN = (MODE == kModeFused || MODE == kModeBoundary || LIST);
    constexpr bool DEP = (MODE == kModeFused || MODE == kModeDeposit || MODE == kModeFusedList);
    constexpr bool BINS = REBIN && !LIST;
    constexpr int EX = TX + 1, EY = TY + 1, EZ = TZ + 1, NE = EX * EY * EZ;
    constexpr int RX = TX + 3, RY = TY + 3, RZ = TZ + 3, NR = RX * RY * RZ;
    // E tile: (E_x, E_y) of a node side by side and E_z apart, so that the
    // gather reads the two x-neighbours of each (y, z) pair with one 2x64-bit
    // and one 2x32-bit LDS load at constant offsets from the particle's base
    // node (measured 3% faster per step than 16-byte nodes, whose loads share
    // fewer LDS banks, and than three separate arrays)
    constexpr int kThreads = mx_block(TX * TY * TZ), kWaves = kThreads / 64;
    __shared__ float2 sExy[PUSH ? NE : 1];
    __shared__ float sEz[PUSH ? NE : 1];
    __shared__ unsigned long long sR[DEP ? NR : 1];
    __shared__ BufMx<IDS, kLeaveCap> sLeave[BINS ? kWaves : 1];
    __shared__ BufMx<IDS, kStash> sStash[BINS ? kWaves : 1];
    __shared__ double sKe[PUSH ? kKeSlots : 1][kWaves];
    __shared__ SpecMeta sMeta[kMaxSpecies];
    __shared__ int sBlk[BINS ? kMaxSpecies : 1];           // slots of the blocks written
    __shared__ int sLeft[BINS ? kMaxSpecies : 1][kWaves];  // stayers left in each stash
    __shared__ int sItem;

    const int lane = lane_id();
    const int wv = uniform((int)threadIdx.x >> 6);
    for (int iter = 0;; ++iter) {
        // (opaque: index arithmetic hoisted out of the item loop would hold
        // registers through the particle loop)
        const int tid = QUEUE ? opaque((int)threadIdx.x) : (int)threadIdx.x;
        // the first item of a workgroup is its own index; the counter hands out
        // those after gridDim.x, each asked for while the one before is worked on
        // (asked for when needed, the answer was a wait per item: 32 members
        // 1362 -> 1340 us per launch in 8x8x4 tiles, 64 members 1507 -> 1417 in 8^3)
        int item = blockIdx.x;
        unsigned int next = 0u;
        if (QUEUE) {
            if (iter > 0) item = uniform(sItem);
            if (item >= nitems) break;
            if (tid == 0) next = gridDim.x + atomicAdd(queue, 1u);
        } else if (iter > 0) {
            break;
        }
        const WorkItem it = items[item];
        const InstDev *__restrict__ I = insts + it.inst;
        const int par = parity[it.inst];
        const int nx = I->n[0], ny = I->n[1], nz = I->n[2];
        const int ntx = I->nt[0], nty = I->nt[1];
        const int tile = it.tile;
        const int tx = tile % ntx, ty = (tile / ntx) % nty, tz = tile / (ntx * nty);
        const int lox = tx * TX, loy = ty * TY, loz = tz * TZ;
        const bool ids = IDS && I->track_ids != 0;
        const bool excl = it.nchunks == 1;  // this workgroup alone fills the tile's front runs
        const int ns = I->nspecies;
        const int nbuf = par ^ 1;
        const int acc_buf = (MODE == kModeFused || MODE == kModeFusedList) ? nbuf : par;

        // every load of the E tile and of the species' bin words is issued
        // before the first one is used
        constexpr int KE = PUSH ? (NE + kThreads - 1) / kThreads : 1;
        double ev[3][KE];
        if (PUSH) {
#pragma unroll
            for (int k = 0; k < KE; ++k) {
                const int l = min(tid + k * kThreads, NE - 1);
                const int lx = l % EX, ly = (l / EX) % EY, lz = l / (EX * EY);
                const int gx = wrap_near(lox + lx, nx), gy = wrap_near(loy + ly, ny),
                          gz = wrap_near(loz + lz, nz);
                const int64_t g = gx + (int64_t)nx * (gy + (int64_t)ny * gz);
#pragma unroll
                for (int a = 0; a < 3; ++a) ev[a][k] = gload(I->e[a], g);
            }
        }
        load_meta<LIST>(sMeta, I, it, par, tid, ns);
        if (BINS && tid < kMaxSpecies) sBlk[tid] = 0;
        if (DEP)
            for (int l = tid; l < NR; l += kThreads) sR[l] = 0ull;
        if (PUSH) {
#pragma unroll
            for (int k = 0; k < KE; ++k) {
                const int l = tid + k * kThreads;
                if (l < NE) {
                    sExy[l] = make_float2((float)ev[0][k], (float)ev[1][k]);
                    sEz[l] = (float)ev[2][k];
                }
            }
        }
        __syncthreads();
        // (every thread has read sItem)
        if (QUEUE && tid == 0) sItem = (int)next;

        const float dt = (float)I->dt;
        const float dt2 = uniform(0.5f * dt);
        const float dts = uniform(dt * kFracScale);  // cells per unit velocity, in 2^-24 units
        const float bx = (float)I->b0[0], by = (float)I->b0[1], bz = (float)I->b0[2];
        // cells of the tile inside the box; an axis of a single tile can wrap
        // a particle back into its own tile
        const unsigned limx = (unsigned)min(TX, nx - lox), limy = (unsigned)min(TY, ny - loy),
                       limz = (unsigned)min(TZ, nz - loz);
        const bool one_tile = ntx == 1 || nty == 1 || I->nt[2] == 1;

        for (int s = 0; s < ns; ++s) {
            const SpecDev &S = I->sp[s];
            const int F = uniform(sMeta[s].F), B = uniform(sMeta[s].B);
            const int cap = uniform(sMeta[s].cap);
            const int cnt = F + B;
            const int64_t base = uniform(sMeta[s].base);
            const int per = chunk_size(cnt, it.nchunks);
            const int start = it.chunk * per;
            const int end = min(cnt, start + per);
            const int64_t list0 = LIST ? uniform(sMeta[s].list) : 0;
            const float qm = uniform((float)S.qm);
            const double qfix = S.qfix;
            const float t0 = uniform(qm * bx * dt2), t1 = uniform(qm * by * dt2),
                        t2 = uniform(qm * bz * dt2);
            const float tt = t0 * t0 + t1 * t1 + t2 * t2;
            const float s0 = uniform(2.0f * t0 / (1.0f + tt)), s1 = uniform(2.0f * t1 / (1.0f + tt)),
                        s2 = uniform(2.0f * t2 / (1.0f + tt));
            double keo = 0.0, ken = 0.0;
            int taken = 0;       // slots of this wavefront's blocks
            int lc = 0, sc = 0;  // particles in this wavefront's leaver buffer and stash

            // the next kMxPrefetch particles of this lane are loaded ahead, so each
            // lane keeps that many particle reads in flight
            const BinView cur = bin_view(S, par, base, ids);
            const BinView nxt = bin_view(S, nbuf, base, ids);
            PMx ahead[kMxPrefetch];
#pragma unroll
            for (int k = 0; k < kMxPrefetch; ++k) {
                ahead[k] = PMx{{0u, 0u, 0u}, {0.0f, 0.0f, 0.0f}, 0};
                if (start + tid + k * kThreads < end)
                    ahead[k] = load_bin(cur, (uint32_t)bin_slot(start + tid + k * kThreads, F, B, cap),
                                        ids);
            }
            for (int p0 = start; p0 < end; p0 += kThreads) {
                const int p = p0 + tid;
                const bool active = p < end;
                PMx q = ahead[0];
#pragma unroll
                for (int k = 0; k + 1 < kMxPrefetch; ++k) ahead[k] = ahead[k + 1];
                if (p + kMxPrefetch * kThreads < end)
                    ahead[kMxPrefetch - 1] =
                        load_bin(cur, (uint32_t)bin_slot(p + kMxPrefetch * kThreads, F, B, cap), ids);
                // cell relative to this tile's origin and in-cell offset per axis
                int rx = pos_rel(q.w[0]), ry = pos_rel(q.w[1]), rz = pos_rel(q.w[2]);
                float ox = pos_frac(q.w[0]), oy = pos_frac(q.w[1]), oz = pos_frac(q.w[2]);
                if (PUSH && active) {
                    float wx0, wx1, wy0, wy1, wz0, wz1;
                    cic_wf<WO>(ox, wx0, wx1);
                    cic_wf<WO>(oy, wy0, wy1);
                    cic_wf<WO>(oz, wz0, wz1);
                    const int lx = min(max(rx, 0), TX - 1);
                    const int ly = min(max(ry, 0), TY - 1);
                    const int lz = min(max(rz, 0), TZ - 1);
                    // base node with 24-bit multiplies (full rate)
                    const unsigned nb =
                        __umul24((unsigned)lz, EX * EY) + __umul24((unsigned)ly, EX) + (unsigned)lx;
                    const lds_ptr<float2> exy = lds_base(sExy, nb);
                    const lds_ptr<float> ez0 = lds_base(sEz, nb);
                    // all eight nodes are read before the first is used: one
                    // LDS latency instead of eight
                    float2 gxy[2][2][2];
                    float gz_[2][2][2];
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int k = 0; k < 2; ++k)
#pragma unroll
                            for (int i = 0; i < 2; ++i) {
                                gxy[i][j][k] = lds_read(exy, i + EX * (j + EY * k));
                                gz_[i][j][k] = lds_read(ez0, i + EX * (j + EY * k));
                            }
                    __builtin_amdgcn_sched_barrier(0);
                    float e0 = 0.0f, e1 = 0.0f, e2 = 0.0f;
                    const float wx[2] = {wx0, wx1}, wy[2] = {wy0, wy1}, wz[2] = {wz0, wz1};
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
#pragma unroll
                            for (int k = 0; k < 2; ++k) {
                                const float w = wx[i] * wy[j] * wz[k];
                                e0 += gxy[i][j][k].x * w;
                                e1 += gxy[i][j][k].y * w;
                                e2 += gz_[i][j][k] * w;
                            }
                    const float vx = q.v[0], vy = q.v[1], vz = q.v[2];
                    keo += (double)(vx * vx + vy * vy + vz * vz);
                    const float um0 = vx + qm * e0 * dt2;
                    const float um1 = vy + qm * e1 * dt2;
                    const float um2 = vz + qm * e2 * dt2;
                    const float ua0 = um0 + (um1 * t2 - um2 * t1);
                    const float ua1 = um1 + (um2 * t0 - um0 * t2);
                    const float ua2 = um2 + (um0 * t1 - um1 * t0);
                    const float up0 = um0 + (ua1 * s2 - ua2 * s1);
                    const float up1 = um1 + (ua2 * s0 - ua0 * s2);
                    const float up2 = um2 + (ua0 * s1 - ua1 * s0);
                    q.v[0] = up0 + qm * e0 * dt2;
                    q.v[1] = up1 + qm * e1 * dt2;
                    q.v[2] = up2 + qm * e2 * dt2;
                    ken += (double)(q.v[0] * q.v[0] + q.v[1] * q.v[1] + q.v[2] * q.v[2]);
                    // drift in fixed point: the tile-relative position word (8.24)
                    // plus the displacement rounded to 2^-24 of a cell, exact in
                    // int32 while |v dt| < 64 cells (farther is reported)
                    const float sx = q.v[0] * dts, sy = q.v[1] * dts, sz = q.v[2] * dts;
                    const bool ok =
                        fabsf(sx) < kMaxShift && fabsf(sy) < kMaxShift && fabsf(sz) < kMaxShift;
                    if (!ok) {
                        count_lanes(&I->flags[kFlagRange]);
                    } else {
                        q.w[0] = (uint32_t)((int32_t)q.w[0] + (int32_t)rintf(sx));
                        q.w[1] = (uint32_t)((int32_t)q.w[1] + (int32_t)rintf(sy));
                        q.w[2] = (uint32_t)((int32_t)q.w[2] + (int32_t)rintf(sz));
                    }
                    rx = pos_rel(q.w[0]);
                    ry = pos_rel(q.w[1]);
                    rz = pos_rel(q.w[2]);
                    ox = pos_frac(q.w[0]);
                    oy = pos_frac(q.w[1]);
                    oz = pos_frac(q.w[2]);
                    if (MODE == kModeGatherPush) {
                        // not re-binned: the cell stays relative to this tile
                        store_bin<true>(cur, (uint32_t)bin_slot(p, F, B, cap), q, ids);
                    }
                }
                if (MODE == kModeGatherPush) continue;

                bool block = false;  // this wavefront stores a full block
                int blk;             // its first slot (lane 0)
                bool stay = false;
                int nst = 0;
                unsigned long long sm = 0ull;
                PMx fill;            // what the lanes of leavers store
                if (BINS) {
                    stay = active && (unsigned)rx < limx && (unsigned)ry < limy &&
                           (unsigned)rz < limz;
                    if (one_tile && active && !stay) {
                        PMx r = q;
                        if (rebase_words<TX, TY, TZ>(r.w, I, lox, loy, loz) == tile) {
                            q = r;
                            stay = true;
                        }
                    }
                    sm = __ballot(stay);
                    const unsigned long long lm = __ballot(active && !stay);
                    if (lm) {
                        // particles that left: per-wave LDS buffer, routed in batches
                        const int nl = (int)__popcll(lm);
                        const bool leave = active && !stay;
                        if (lc + nl > kLeaveCap) {
                            flush_leavers_mx<TX, TY, TZ, IDS>(sLeave[wv], lc, I, S, nbuf,
                                                              ids, lox, loy, loz);
                            lc = 0;
                        }
                        if (nl <= kLeaveCap) {
                            if (leave) sLeave[wv].put(lc + lane_rank(lm), q, ids);
                            lc += nl;
                        } else if (leave) {
                            PMx r = q;
                            const int t = rebase_words<TX, TY, TZ>(r.w, I, lox, loy, loz);
                            route_back_mx(S, nbuf, t, r, ids, I->flags);
                        }
                    }
                    nst = (int)__popcll(sm);
                    const int holes = 64 - nst;
                    block = holes <= sc;
                    if (block) {
                        // both arrive while the charge is deposited
                        if (excl && lane == 0) blk = atomicAdd(&sBlk[s], 64);
                        sc -= holes;
                        taken += 64;
                        wave_sync();
                        if (!stay) sStash[wv].get(sc + lane_rank(~sm), fill, ids);
                    }
                }
                if (DEP && active) {
                    float wx0, wx1, wy0, wy1, wz0, wz1;
                    cic_wf<WO>(ox, wx0, wx1);
                    cic_wf<WO>(oy, wy0, wy1);
                    cic_wf<WO>(oz, wz0, wz1);
                    const float wx[2] = {wx0, wx1}, wy[2] = {wy0, wy1}, wz[2] = {wz0, wz1};
                    // node (x, y, z) of the deposit block is cell lo - 1 + (x, y, z)
                    // taken periodically, so the particle's cell relative to the
                    // tile plus one indexes it, wrapped or not
                    const unsigned dx = (unsigned)(rx + 1), dy = (unsigned)(ry + 1),
                                   dz = (unsigned)(rz + 1);
                    if (dx <= TX + 1 && dy <= TY + 1 && dz <= TZ + 1) {
                        unsigned long long *__restrict__ r0 = (unsigned long long *)(
                            (char *)sR + (__umul24(dz, RX * RY * 8u) + __umul24(dy, RX * 8u) +
                                          dx * 8u));
                        // the fixed-point charge of node (i, j, k) is
                        // round(qfix * (wx wy) * wz) with wx wy rounded to FP32 and
                        // the rest exact in FP64 (FP32 products of 24-bit
                        // mantissas, one rounding in the FMA)
                        const double wzd[2] = {(double)wz0, (double)wz1};
#pragma unroll
                        for (int i = 0; i < 2; ++i)
#pragma unroll
                            for (int j = 0; j < 2; ++j) {
                                const double qxy = (double)(wx[i] * wy[j]) * qfix;
#pragma unroll
                                for (int k = 0; k < 2; ++k)
                                    atomicAdd(&r0[i + RX * (j + RY * k)],
                                              (unsigned long long)fix_round(wzd[k], qxy));
                            }
                    } else {
                        unsigned long long *__restrict__ racc = I->rho_acc[acc_buf];
                        count_lanes(&I->flags[kFlagFast]);
                        const int gx = wrap_cell(lox + rx, nx), gy = wrap_cell(loy + ry, ny),
                                  gz = wrap_cell(loz + rz, nz);
#pragma unroll
                        for (int i = 0; i < 2; ++i)
#pragma unroll
                            for (int j = 0; j < 2; ++j) {
                                const double qxy = (double)(wx[i] * wy[j]) * qfix;
#pragma unroll
                                for (int k = 0; k < 2; ++k) {
                                    const int hx = (gx + i) % nx, hy = (gy + j) % ny,
                                              hz = (gz + k) % nz;
                                    const long long v = fix_round((double)wz[k], qxy);
                                    gatomic_add(&racc[hx + (int64_t)nx * (hy + (int64_t)ny * hz)],
                                                (unsigned long long)v);
                                }
                            }
                    }
                }
                // the loads ahead arrive before the stores are issued: memory
                // operations complete in order, so a wait for them at the top
                // of the next iteration would be one for these stores as well
#pragma unroll
                for (int k = 0; BINS && k < kMxPrefetch; ++k) arrived(ahead[k], ids);
                if (LIST) {
                    // retry path: every particle to the species' contiguous
                    // list, in bin order inside this item's reserved range
                    if (active) {
                        const int t = rebase_words<TX, TY, TZ>(q.w, I, lox, loy, loz);
                        store_list_mx(S, nbuf, list0 + (p - start), q, t, ids);
                    }
                } else if (block) {
                    if (!stay) q = fill;
                    if (!excl && lane == 0) blk = claim_block(I, it, s);
                    store_bin<true>(nxt, (uint32_t)(lane_bcast(blk, 0) + lane), q, ids);
                } else if (nst > 0) {
                    wave_sync();
                    if (stay) sStash[wv].put(sc + lane_rank(sm), q, ids);
                    sc += nst;
                }
            }
            if (BINS) {
                flush_leavers_mx<TX, TY, TZ, IDS>(sLeave[wv], lc, I, S, nbuf, ids, lox, loy, loz);
                // the stayers left in the stashes: behind the blocks, or in the
                // back run of a split tile
                if (excl) {
                    if (lane == 0) sLeft[s][wv] = sc;
                    __syncthreads();
                    int o = sBlk[s], m = o;
#pragma unroll
                    for (int w = 0; w < kWaves; ++w) {
                        const int r = sLeft[s][w];
                        if (w < wv) o += r;
                        m += r;
                    }
                    if (lane < sc) {
                        PMx q;
                        sStash[wv].get(lane, q, ids);
                        store_bin<false>(nxt, (uint32_t)(o + lane), q, ids);
                    }
                    if (tid == 0 && add_front<MODE == kModeBoundary>(&S.count[nbuf][tile], m, cap))
                        count_lanes(&I->flags[kFlagOverflow]);
                } else if (taken + sc > 0) {
                    unsigned long long old = 0ull;
                    if (lane == 0)
                        old = gatomic_add(&S.count[nbuf][tile],
                                          (unsigned long long)taken | (unsigned long long)sc << 32);
                    old = lane_bcast(old, 0);
                    const int front = bin_front(old) + taken, back = bin_back(old);
                    if (front + back + sc > cap) {
                        if (lane == 0) gatomic_add(&I->flags[kFlagOverflow], 1ull);
                    } else if (lane < sc) {
                        PMx q;
                        sStash[wv].get(lane, q, ids);
                        store_bin<false>(nxt, (uint32_t)(cap - 1 - back - lane), q, ids);
                    }
                }
                wave_sync();
            }
            if (PUSH) {
                keo = wave_total(keo);
                ken = wave_total(ken);
                if (lane == 0) {
                    sKe[s][wv] = keo;
                    sKe[kMaxSpecies + s][wv] = ken;
                }
            }
        }

        __syncthreads();
        if (PUSH) write_ke<kWaves>(I, it, tid, ns, sKe);
        if (DEP) {
            unsigned long long *__restrict__ racc = I->rho_acc[acc_buf];
            for (int l = tid; l < NR; l += kThreads) {
                const unsigned long long v = sR[l];
                if (v == 0ull) continue;
                const int lx = l % RX, ly = (l / RX) % RY, lz = l / (RX * RY);
                const int gx = wrap_near(lox - 1 + lx, nx);
                const int gy = wrap_near(loy - 1 + ly, ny);
                const int gz = wrap_near(loz - 1 + lz, nz);
                gatomic_add(&racc[gx + (int64_t)nx * (gy + (int64_t)ny * gz)], v);
            }
        }
        // the next item reuses the LDS blocks and sItem
        if (QUEUE) __syncthreads();
    }
}

// ---------------------------------------------------------------- binning
// A list entry (tile, words) names a cell inside the box: tile in range, the
// relative cell inside the tile, the global cell inside the (possibly partly
// covered) last tile, the fraction below 1 by construction.
__device__ __forceinline__ bool list_valid(const InstDev *I, int tile, const PMx &q, int tx_,
                                           int ty_, int tz_)
{
    if (tile < 0 || tile >= I->ntiles) return false;
    const int t3[3] = {tile % I->nt[0], (tile / I->nt[0]) % I->nt[1], tile / (I->nt[0] * I->nt[1])};
    const int T3[3] = {tx_, ty_, tz_};
    for (int a = 0; a < 3; ++a) {
        const int r = pos_rel(q.w[a]);
        if (r < 0 || r >= T3[a] || t3[a] * T3[a] + r >= I->n[a]) return false;
    }
    return true;
}

__global__ void k_bin_count_mx(const InstDev *__restrict__ insts, int inst, int s, int lbuf,
                               int64_t n, int tx_, int ty_, int tz_)
{
    const InstDev *I = insts + inst;
    const SpecDev &S = I->sp[s];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < n;
    PMx q{{0u, 0u, 0u}, {0.0f, 0.0f, 0.0f}, 0};
    int t = 0;
    if (live) {
        q = load_pmx(S, lbuf, i, false);
        t = gload((const int32_t *)S.buf[lbuf][0], i);
    }
    const bool ok = live && list_valid(I, t, q, tx_, ty_, tz_);
    if (live && !ok) count_lanes(&I->flags[kFlagRange]);
    (void)wave_counter_add(S.count[lbuf ^ 1], ok ? t : 0, ok);
}

__global__ void k_bin_scatter_mx(const InstDev *__restrict__ insts, int inst, int s, int lbuf,
                                 int64_t n, int tx_, int ty_, int tz_)
{
    const InstDev *I = insts + inst;
    const SpecDev &S = I->sp[s];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < n;
    const bool ids = I->track_ids != 0;
    PMx q{{0u, 0u, 0u}, {0.0f, 0.0f, 0.0f}, 0};
    int t = 0;
    if (live) {
        q = load_pmx(S, lbuf, i, ids);
        t = gload((const int32_t *)S.buf[lbuf][0], i);
    }
    const bool ok = live && list_valid(I, t, q, tx_, ty_, tz_);
    const unsigned long long old = wave_counter_add(S.count[lbuf ^ 1], ok ? t : 0, ok);
    if (!ok) return;
    const int slot = bin_front(old);
    if (slot < gload(S.bin_cap, t))
        store_pmx(S, lbuf ^ 1, gload(S.bin_base, t) + slot, q, ids);
    else
        count_lanes(&I->flags[kFlagOverflow]);
}

__global__ void k_bins_to_list_mx(const InstDev *__restrict__ insts, int inst, int s, int src,
                                  int dst, const int *__restrict__ tiles, int t0,
                  const int64_t *__restrict__ list_off)
{
    const InstDev *I = insts + inst;
    const SpecDev &S = I->sp[s];
    const int t = tiles ? tiles[blockIdx.x] : t0 + (int)blockIdx.x;
    const unsigned long long w = S.count[src][t];
    const int cap = S.bin_cap[t];
    const int F = min(bin_front(w), cap);
    const int B = min(bin_back(w), cap - F);
    const int64_t ib = S.bin_base[t];
    const int64_t ob = list_off[blockIdx.x];
    const bool ids = I->track_ids != 0;
    for (int v = threadIdx.x; v < F + B; v += blockDim.x) {
        const PMx q = load_pmx(S, src, ib + bin_slot(v, F, B, cap), ids);
        store_list_mx(S, dst, ob + v, q, t, ids);
    }
}

__global__ void k_cell_counts_mx(const InstDev *__restrict__ insts, int inst, int s, int par,
                                 int32_t *__restrict__ counts, int tx_, int ty_, int tz_)
{
    const InstDev *I = insts + inst;
    const SpecDev &S = I->sp[s];
    const int t = blockIdx.x;
    const unsigned long long w = S.count[par][t];
    const int cap = S.bin_cap[t];
    const int F = min(bin_front(w), cap);
    const int B = min(bin_back(w), cap - F);
    const int64_t b = S.bin_base[t];
    const int nx = I->n[0], ny = I->n[1];
    const int ox = (t % I->nt[0]) * tx_, oy = ((t / I->nt[0]) % I->nt[1]) * ty_,
              oz = (t / (I->nt[0] * I->nt[1])) * tz_;
    for (int v = threadIdx.x; v < F + B; v += blockDim.x) {
        const int64_t o = b + bin_slot(v, F, B, cap);
        const int cx = ox + pos_rel(((const uint32_t *)S.buf[par][1])[o]);
        const int cy = oy + pos_rel(((const uint32_t *)S.buf[par][2])[o]);
        const int cz = oz + pos_rel(((const uint32_t *)S.buf[par][3])[o]);
        atomicAdd(&counts[cx + (int64_t)nx * (cy + (int64_t)ny * cz)], 1);
    }
}

// ---------------------------------------------------------------- loaders
// FP64 position -> list entry.  The cell is the FP64 int() truncation; an
// offset that rounds up to 1 on the 24-bit grid is clamped below it, so the
// particle stays on the same side of the cell face as in FP64 (the mirrored
// CIC weights jump there).
__device__ __forceinline__ void store_loaded_mx(const InstDev *I, const SpecDev &S, int b,
                                                int64_t i, double x, double y, double z,
                                                double vx, double vy, double vz, int64_t id,
                                                bool ids, int tx_, int ty_, int tz_)
{
    const double p[3] = {x, y, z};
    const int T3[3] = {tx_, ty_, tz_};
    int tc[3];
    PMx q;
    for (int a = 0; a < 3; ++a) {
        const int c = (int)p[a];
        double f = rint((p[a] - (double)c) * 16777216.0);
        if (f > 16777215.0) f = 16777215.0;
        tc[a] = c / T3[a];
        q.w[a] = pos_word(c - tc[a] * T3[a], (uint32_t)f);
    }
    q.v[0] = (float)vx;
    q.v[1] = (float)vy;
    q.v[2] = (float)vz;
    q.id = id;
    store_list_mx(S, b, i, q, tc[0] + I->nt[0] * (tc[1] + I->nt[1] * tc[2]), ids);
}

__global__ void k_load_uniform_mx(const InstDev *__restrict__ insts, int inst, int s, int b,
                                  Pcg32Dev rng0, uint64_t offset, int64_t np, double vth,
                                  int tx_, int ty_, int tz_)
{
    const InstDev *I = insts + inst;
    const SpecDev &S = I->sp[s];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    Pcg32Dev r = rng0;
    pcg_advance(r, offset + 7u * (uint64_t)i);
    const double x = pcg_double(r) * (double)I->n[0] + 0.0;
    const double y = pcg_double(r) * (double)I->n[1] + 0.0;
    const double z = pcg_double(r) * (double)I->n[2] + 0.0;
    double vx, vy, vz;
    maxwell3(r, vth, vx, vy, vz);
    store_loaded_mx(I, S, b, i, x, y, z, vx, vy, vz, i, I->track_ids != 0, tx_, ty_, tz_);
}

__global__ void k_load_hump_mx(const InstDev *__restrict__ insts, int inst, int s, int b,
                               Pcg32Dev rng0, uint64_t offset, uint64_t budget, int64_t np,
                               double amp, double sigma, double vth,
                               unsigned long long *__restrict__ fail, int tx_, int ty_, int tz_)
{
    const InstDev *I = insts + inst;
    const SpecDev &S = I->sp[s];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const int nx = I->n[0], ny = I->n[1], nz = I->n[2];
    Pcg32Dev r = rng0;
    pcg_advance(r, offset + (uint64_t)i * budget);
    const double cx = 0.5 * nx, cy = 0.5 * ny, cz = 0.5 * nz;
    const double inv2s2 = 1.0 / (2.0 * sigma * sigma);
    const uint64_t maxc = (budget - 4u) / 4u;
    double x = cx, y = cy, z = cz;
    bool ok = false;
    for (uint64_t c = 0; c < maxc; ++c) {
        const double px = pcg_double(r) * (double)nx;
        const double py = pcg_double(r) * (double)ny;
        const double pz = pcg_double(r) * (double)nz;
        const double u = pcg_double(r);
        const double dx = px - cx, dy = py - cy, dz = pz - cz;
        const double f = (1.0 + amp * exp(-(dx * dx + dy * dy + dz * dz) * inv2s2)) / (1.0 + amp);
        if (u < f) {
            x = px;
            y = py;
            z = pz;
            ok = true;
            break;
        }
    }
    if (!ok) count_lanes(fail);
    double vx, vy, vz;
    maxwell3(r, vth, vx, vy, vz);
    store_loaded_mx(I, S, b, i, x, y, z, vx, vy, vz, i, I->track_ids != 0, tx_, ty_, tz_);
}

}  // namespace

// ---------------------------------------------------------------- launchers
// List mode always handles ids (it is the rare retry); a deposit reads none.
template <int TX, int TY, int TZ, int WO>
static hipError_t launch_tile_mx(int mode, bool ids, const InstDev *insts, const WorkItem *items,
                              int nitems, const int *parity, hipStream_t st)
{
    dim3 g(nitems), b(mx_block(TX * TY * TZ));
#define OHPIC_MX_CASE(M, IDS)                                                                     \
    hipLaunchKernelGGL((k_particles_mixed<TX, TY, TZ, WO, M, IDS>), g, b, 0, st, insts, items, parity, \
                       nullptr, nitems)
    switch (mode) {
    case kModeFused:
        if (ids)
            OHPIC_MX_CASE(kModeFused, true);
        else
            OHPIC_MX_CASE(kModeFused, false);
        break;
    case kModeGatherPush:
        if (ids)
            OHPIC_MX_CASE(kModeGatherPush, true);
        else
            OHPIC_MX_CASE(kModeGatherPush, false);
        break;
    case kModeBoundary:
        if (ids)
            OHPIC_MX_CASE(kModeBoundary, true);
        else
            OHPIC_MX_CASE(kModeBoundary, false);
        break;
    case kModeDeposit: OHPIC_MX_CASE(kModeDeposit, false); break;
    case kModeFusedList: OHPIC_MX_CASE(kModeFusedList, true); break;
    case kModeBoundaryList: OHPIC_MX_CASE(kModeBoundaryList, true); break;
    default:
        return hipErrorInvalidValue;
    }
#undef OHPIC_MX_CASE
    return hipGetLastError();
}

template <int TX, int TY, int TZ, int WO>
static hipError_t launch_tile_mx_queue(bool ids, const InstDev *insts, const WorkItem *items,
                                    int nitems, const int *parity, unsigned int *queue, int blocks,
                                    hipStream_t st)
{
    if (ids)
        hipLaunchKernelGGL((k_particles_mixed<TX, TY, TZ, WO, kModeFusedQueue, true>), dim3(blocks),
                           dim3(mx_block(TX * TY * TZ)), 0, st, insts, items, parity, queue, nitems);
    else
        hipLaunchKernelGGL((k_particles_mixed<TX, TY, TZ, WO, kModeFusedQueue, false>), dim3(blocks),
                           dim3(mx_block(TX * TY * TZ)), 0, st, insts, items, parity, queue, nitems);
    return hipGetLastError();
}

template <int TX, int TY, int TZ, int WO>
static int queue_blocks_per_cu_mx(bool ids)
{
    int nb = 0;
    const void *f = ids ? reinterpret_cast<const void *>(
                              &k_particles_mixed<TX, TY, TZ, WO, kModeFusedQueue, true>)
                        : reinterpret_cast<const void *>(
                              &k_particles_mixed<TX, TY, TZ, WO, kModeFusedQueue, false>);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, mx_block(TX * TY * TZ), 0) != hipSuccess) {
        (void)hipGetLastError();
        nb = 1;
    }
    return nb > 0 ? nb : 1;
}

hipError_t launch_particles_mixed(int mode, int weight_order, const int T[3], bool ids,
                                  const InstDev *insts, const WorkItem *items, int nitems,
                                  const int *parity, hipStream_t st)
{
#define OHPIC_TILE(A, B, C)                                                                  \
    if (T[0] == A && T[1] == B && T[2] == C)                                                 \
        return weight_order == 0                                                             \
                   ? launch_tile_mx<A, B, C, 0>(mode, ids, insts, items, nitems, parity, st) \
                   : launch_tile_mx<A, B, C, 1>(mode, ids, insts, items, nitems, parity, st);
    OHPIC_TILE(4, 4, 4)
    OHPIC_TILE(8, 8, 8)
    OHPIC_TILE(8, 8, 4)
    OHPIC_TILE(16, 8, 4)
#undef OHPIC_TILE
    return hipErrorInvalidValue;
}

hipError_t launch_particles_mixed_queue(int weight_order, const int T[3], bool ids,
                                        const InstDev *insts, const WorkItem *items, int nitems,
                                        const int *parity, unsigned int *queue, int blocks,
                                        hipStream_t st)
{
#define OHPIC_TILE(A, B, C)                                                                       \
    if (T[0] == A && T[1] == B && T[2] == C)                                                      \
        return weight_order == 0 ? launch_tile_mx_queue<A, B, C, 0>(ids, insts, items, nitems,    \
                                                                    parity, queue, blocks, st)    \
                                 : launch_tile_mx_queue<A, B, C, 1>(ids, insts, items, nitems,    \
                                                                    parity, queue, blocks, st);
    OHPIC_TILE(4, 4, 4)
    OHPIC_TILE(8, 8, 8)
    OHPIC_TILE(8, 8, 4)
    OHPIC_TILE(16, 8, 4)
#undef OHPIC_TILE
    return hipErrorInvalidValue;
}

int particles_mixed_queue_blocks(int weight_order, const int T[3], bool ids)
{
#define OHPIC_TILE(A, B, C)                                                      \
    if (T[0] == A && T[1] == B && T[2] == C)                                     \
        return weight_order == 0 ? queue_blocks_per_cu_mx<A, B, C, 0>(ids)       \
                                 : queue_blocks_per_cu_mx<A, B, C, 1>(ids);
    OHPIC_TILE(4, 4, 4)
    OHPIC_TILE(8, 8, 8)
    OHPIC_TILE(8, 8, 4)
    OHPIC_TILE(16, 8, 4)
#undef OHPIC_TILE
    return 1;
}

hipError_t launch_bin_count_mx(const InstDev *insts, int inst, int s, int lbuf, int64_t n,
                               const int T[3], hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_bin_count_mx, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                       insts, inst, s, lbuf, n, T[0], T[1], T[2]);
    return hipGetLastError();
}

hipError_t launch_bin_scatter_mx(const InstDev *insts, int inst, int s, int lbuf, int64_t n,
                                 const int T[3], hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_bin_scatter_mx, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                       insts, inst, s, lbuf, n, T[0], T[1], T[2]);
    return hipGetLastError();
}

hipError_t launch_bins_to_list_mx(const InstDev *insts, int inst, int s, int src, int dst,
                                  const int *tiles, int t0, int ntiles, const int64_t *list_off,
                                  hipStream_t st)
{
    if (ntiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_bins_to_list_mx, dim3(ntiles), dim3(256), 0, st, insts, inst, s, src,
                       dst, tiles, t0, list_off);
    return hipGetLastError();
}

hipError_t launch_cell_counts_mx(const InstDev *insts, int inst, int s, int par, int ntiles,
                                 int32_t *counts, const int T[3], hipStream_t st)
{
    if (ntiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_cell_counts_mx, dim3(ntiles), dim3(256), 0, st, insts, inst, s, par,
                       counts, T[0], T[1], T[2]);
    return hipGetLastError();
}

hipError_t launch_load_uniform_mx(const InstDev *insts, int inst, int s, int b, Pcg32Dev rng0,
                                  uint64_t offset, int64_t np, double vth, const int T[3],
                                  hipStream_t st)
{
    if (np <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_load_uniform_mx, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, st,
                       insts, inst, s, b, rng0, offset, np, vth, T[0], T[1], T[2]);
    return hipGetLastError();
}

hipError_t launch_load_hump_mx(const InstDev *insts, int inst, int s, int b, Pcg32Dev rng0,
                               uint64_t offset, uint64_t budget, int64_t np, double amp,
                               double sigma, double vth, unsigned long long *fail,
                               const int T[3], hipStream_t st)
{
    if (np <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_load_hump_mx, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, st,
                       insts, inst, s, b, rng0, offset, budget, np, amp, sigma, vth, fail, T[0],
                       T[1], T[2]);
    return hipGetLastError();
}

}  // namespace ohpic
