// ohpic_particles.hip -- particle kernels for gfx950 (FP64 storage).
//
// One workgroup processes one work item = (instance, tile, chunk): it stages
// the node-centred E of the tile plus a one-node halo in LDS, walks its slice
// of every species' bin, and for each particle
//   gathers E with CIC weights   (linear_interpolator.f90:22-69),
//   runs the Boris rotation + drift (particle_mover_boris.f90:21-64),
//   applies the periodic wrap twice (periodic_particle_boundary.f90:42-53,
//                                    ohhelppic3d.f90:353-355),
//   deposits q*W(x_new) into an int64 fixed-point LDS copy of the tile's
//   nodes plus halo (linear_scatter.f90:22-55), and
//   re-bins it (the replacement of OhHelp's correct_particle/transbound):
//   a particle that stays in its tile goes to the front run of the tile's
//   bin in the other buffer (64-slot blocks, ohpic_particle_common.hpp), a
//   particle that left goes through a per-wave LDS buffer to the back run of
//   its new tile's bin (batched 64-bit atomics on the bin's front|back word).
// The LDS charge block is flushed with one global 64-bit atomic per node.
// Integer accumulation makes rho independent of particle order and timing.
//
// What bounds it: large grids stream 96 B per particle, at 6.1 TB/s or 0.76 of
// the 8 TB/s peak (256^3 x 64 ppc, 33.9 ms per launch); the rest is per tile (E
// tile, charge flush, the leavers' atomics).  Small grids wait: so every load
// of an item's start is issued before the first is used, nothing in a whole
// tile's particle loop waits for a store, a block's number or the stash, and a
// species ends with one barrier.  Against slots from an LDS counter at any
// alignment, a store wait per iteration and the wrap and tile index of every
// particle: 256^3 x 16 ppc 12.16 -> 9.3-10.4 ms (the same build differs that
// much between runs), 96^3 x 32 1.35 -> 1.11 ms, 32^3 x 16 51 -> 38 us per
// launch.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "ohpic_internal.hpp"
#include "ohpic_kernels.hpp"
#include "ohpic_particle_common.hpp"

namespace ohpic {

namespace {

struct P64 {
    double x, y, z, vx, vy, vz;
    int64_t id;
};

__device__ __forceinline__ void store_p64(const SpecDev &S, int nbuf, int64_t o, const P64 &p,
                                          bool ids)
{
    gstore((double *)S.buf[nbuf][0], o, p.x);
    gstore((double *)S.buf[nbuf][1], o, p.y);
    gstore((double *)S.buf[nbuf][2], o, p.z);
    gstore((double *)S.buf[nbuf][3], o, p.vx);
    gstore((double *)S.buf[nbuf][4], o, p.vy);
    gstore((double *)S.buf[nbuf][5], o, p.vz);
    if (ids) gstore(S.pid[nbuf], o, p.id);
}

__device__ __forceinline__ P64 load_p64(const SpecDev &S, int b, int64_t o, bool ids)
{
    P64 q;
    q.x = sload((const double *)S.buf[b][0], o);
    q.y = sload((const double *)S.buf[b][1], o);
    q.z = sload((const double *)S.buf[b][2], o);
    q.vx = sload((const double *)S.buf[b][3], o);
    q.vy = sload((const double *)S.buf[b][4], o);
    q.vz = sload((const double *)S.buf[b][5], o);
    q.id = ids ? gload(S.pid[b], o) : 0;
    return q;
}

// The bin of one tile in one buffer: array bases offset to the bin's first
// element (uniform per workgroup: scalar registers) and particles addressed
// by a 32-bit byte offset (bins hold < 2^29 particles), so per-particle loads
// and stores need no 64-bit address arithmetic.
struct BinView64 {
    const char *c[6];
    const int64_t *id;
};

__device__ __forceinline__ BinView64 bin_view64(const SpecDev &S, int b, int64_t base, bool ids)
{
    BinView64 r;
#pragma unroll
    for (int k = 0; k < 6; ++k) r.c[k] = (const char *)((const double *)S.buf[b][k] + base);
    r.id = ids ? S.pid[b] + base : nullptr;
    return r;
}

__device__ __forceinline__ P64 load_bin64(const BinView64 &bv, uint32_t slot, bool ids)
{
    const uint32_t off = slot * 8u;
    P64 q;
    q.x = sload((const double *)(bv.c[0] + off), 0);
    q.y = sload((const double *)(bv.c[1] + off), 0);
    q.z = sload((const double *)(bv.c[2] + off), 0);
    q.vx = sload((const double *)(bv.c[3] + off), 0);
    q.vy = sload((const double *)(bv.c[4] + off), 0);
    q.vz = sload((const double *)(bv.c[5] + off), 0);
    q.id = ids ? gload(bv.id, (int64_t)slot) : 0;
    return q;
}

// FULL: the wavefront stores full lines
template <bool FULL>
__device__ __forceinline__ void store_bin64(const BinView64 &bv, uint32_t slot, const P64 &q,
                                            bool ids)
{
    const uint32_t off = slot * 8u;
    sstore<FULL>((double *)(bv.c[0] + off), 0, q.x);
    sstore<FULL>((double *)(bv.c[1] + off), 0, q.y);
    sstore<FULL>((double *)(bv.c[2] + off), 0, q.z);
    sstore<FULL>((double *)(bv.c[3] + off), 0, q.vx);
    sstore<FULL>((double *)(bv.c[4] + off), 0, q.vy);
    sstore<FULL>((double *)(bv.c[5] + off), 0, q.vz);
    if (ids) gstore(const_cast<int64_t *>(bv.id), (int64_t)slot, q.id);
}

// The particle's loads have completed from here on.
__device__ __forceinline__ void arrived(P64 &q, bool ids)
{
    asm volatile("" : "+v"(q.x), "+v"(q.y), "+v"(q.z), "+v"(q.vx), "+v"(q.vy), "+v"(q.vz));
    if (ids) asm volatile("" : "+v"(q.id));
}

// Append one particle to the back run of bin t (slot from the packed word).
__device__ __forceinline__ void route_back(const SpecDev &S, int nbuf, int t, const P64 &q,
                                           bool ids, unsigned long long *flags)
{
    const int cap = gload(S.bin_cap, t);
    const int64_t base = gload(S.bin_base, t);
    const unsigned long long old = gatomic_add(&S.count[nbuf][t], 1ull << 32);
    const int f = bin_front(old), b = bin_back(old);
    if (b + f < cap)
        store_p64(S, nbuf, base + (cap - 1 - b), q, ids);
    else
        count_lanes(&flags[kFlagOverflow]);
}

template <bool IDS, int CAP>
struct Buf64 {
    double c[6][CAP];
    int64_t id[IDS ? CAP : 1];

    __device__ __forceinline__ void put(int i, const P64 &q, bool ids)
    {
        c[0][i] = q.x;
        c[1][i] = q.y;
        c[2][i] = q.z;
        c[3][i] = q.vx;
        c[4][i] = q.vy;
        c[5][i] = q.vz;
        if (IDS && ids) id[i] = q.id;
    }
    __device__ __forceinline__ void get(int i, P64 &q, bool ids) const
    {
        q.x = c[0][i];
        q.y = c[1][i];
        q.z = c[2][i];
        q.vx = c[3][i];
        q.vy = c[4][i];
        q.vz = c[5][i];
        if (IDS && ids) q.id = id[i];
    }
};

// The tile of a particle inside the box.
template <int TX, int TY, int TZ>
__device__ __forceinline__ int tile_of(const P64 &q, int ntx, int nty)
{
    return (int)q.x / TX + ntx * ((int)q.y / TY + nty * ((int)q.z / TZ));
}

// Routes the first `cnt` buffered leavers of this wavefront (lane l takes
// entry l) to the back runs of their new tiles.
template <int TX, int TY, int TZ, bool IDS>
__device__ __forceinline__ void flush_leavers(const Buf64<IDS, kLeaveCap> &lb, int cnt,
                                              const InstDev *__restrict__ I, const SpecDev &S,
                                              int nbuf, bool ids)
{
    wave_sync();
    const int l = lane_id();
    if (l < cnt) {
        P64 q;
        lb.get(l, q, ids);
        route_back(S, nbuf, tile_of<TX, TY, TZ>(q, I->nt[0], I->nt[1]), q, IDS && ids, I->flags);
    }
    wave_sync();
}

// Threads per workgroup, for every tile shape (kept beside mx_block: 512 for
// 512-cell tiles measured 1.20 against 1.15 ms at 96^3 x 32 ppc).
constexpr int fp_block(int) { return kBlock; }

// IDS: instances may keep particle ids (each instance's track_ids says whether
// it does); without it no register, LDS or branch is spent on them.
template <int TX, int TY, int TZ, int WO, int MODE_, bool IDS>
__global__ void __launch_bounds__(fp_block(TX *TY *TZ))
    __attribute__((amdgpu_waves_per_eu(OHPIC_PUSH_MIN_WAVES, 8)))
    k_particles_fp64(const InstDev *__restrict__ insts, const WorkItem *__restrict__ items,
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
    constexpr int kThreads = fp_block(TX * TY * TZ), kWaves = kThreads / 64;
    __shared__ double sE[PUSH ? 3 * NE : 1];
    __shared__ unsigned long long sR[DEP ? NR : 1];
    __shared__ Buf64<IDS, kLeaveCap> sLeave[BINS ? kWaves : 1];
    __shared__ Buf64<IDS, kStash> sStash[BINS ? kWaves : 1];
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
        // (asked for when needed, the answer was a wait per item: eight small
        // instances 76.7 -> 76.0 us per launch)
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
#pragma unroll
                    for (int a = 0; a < 3; ++a) sE[a * NE + l] = ev[a][k];
                }
            }
        }
        __syncthreads();
        // (every thread has read sItem)
        if (QUEUE && tid == 0) sItem = (int)next;

        const double dt = I->dt;
        const double dt2 = dt * 0.5;
        const double bx = I->b0[0], by = I->b0[1], bz = I->b0[2];
        // the tile's part of the box
        const double tlx = uniform((double)lox), tly = uniform((double)loy),
                     tlz = uniform((double)loz);
        const double thx = uniform((double)min(lox + TX, nx)), thy = uniform((double)min(loy + TY, ny)),
                     thz = uniform((double)min(loz + TZ, nz));
        auto in_tile = [&](const P64 &q) {
            return q.x >= tlx && q.x < thx && q.y >= tly && q.y < thy && q.z >= tlz && q.z < thz;
        };

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
            const double qm = S.qm;
            const double qfix = S.qfix;
            // Boris constants for the uniform B (t = qm B dt/2, s = 2t/(1+|t|^2))
            const double t0 = uniform(qm * bx * dt2), t1 = uniform(qm * by * dt2),
                         t2 = uniform(qm * bz * dt2);
            const double tt = t0 * t0 + t1 * t1 + t2 * t2;
            const double s0 = uniform(2 * t0 / (1 + tt)), s1 = uniform(2 * t1 / (1 + tt)),
                         s2 = uniform(2 * t2 / (1 + tt));
            double keo = 0.0, ken = 0.0;
            int taken = 0;       // slots of this wavefront's blocks
            int lc = 0, sc = 0;  // particles in this wavefront's leaver buffer and stash

            const BinView64 cur = bin_view64(S, par, base, ids);
            const BinView64 nxt = bin_view64(S, nbuf, base, ids);
            P64 nextq{0, 0, 0, 0, 0, 0, 0};
            if (start + tid < end)
                nextq = load_bin64(cur, (uint32_t)bin_slot(start + tid, F, B, cap), ids);
            for (int p0 = start; p0 < end; p0 += kThreads) {
                const int p = p0 + tid;
                const bool active = p < end;
                P64 q = nextq;
                // prefetch the next iteration's particle while this one is processed
                if (p + kThreads < end)
                    nextq = load_bin64(cur, (uint32_t)bin_slot(p + kThreads, F, B, cap), ids);
                if (PUSH && active) {
                    const int ix = (int)q.x, iy = (int)q.y, iz = (int)q.z;
                    double wx0, wx1, wy0, wy1, wz0, wz1;
                    cic_w<WO>(q.x - (double)ix, wx0, wx1);
                    cic_w<WO>(q.y - (double)iy, wy0, wy1);
                    cic_w<WO>(q.z - (double)iz, wz0, wz1);
                    // binned particles lie in the tile; the clamp only guards LDS
                    const int lx = min(max(ix - lox, 0), TX - 1);
                    const int ly = min(max(iy - loy, 0), TY - 1);
                    const int lz = min(max(iz - loz, 0), TZ - 1);
                    const unsigned l0 = (unsigned)(lx + EX * (ly + EY * lz));
                    const lds_ptr<double> ex0 = lds_base(sE, l0), ey0 = lds_base(sE + NE, l0),
                                          ez0 = lds_base(sE + 2 * NE, l0);
                    double e0 = 0.0, e1 = 0.0, e2 = 0.0;
                    const double wx[2] = {wx0, wx1}, wy[2] = {wy0, wy1}, wz[2] = {wz0, wz1};
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
#pragma unroll
                            for (int k = 0; k < 2; ++k) {
                                const int l = i + EX * (j + EY * k);
                                const double w = wx[i] * wy[j] * wz[k];
                                e0 += lds_read(ex0, l) * w;
                                e1 += lds_read(ey0, l) * w;
                                e2 += lds_read(ez0, l) * w;
                            }
                    keo += q.vx * q.vx + q.vy * q.vy + q.vz * q.vz;
                    // Boris (particle_mover_boris.f90:42-62)
                    const double um0 = q.vx + qm * e0 * dt2;
                    const double um1 = q.vy + qm * e1 * dt2;
                    const double um2 = q.vz + qm * e2 * dt2;
                    const double ua0 = um0 + (um1 * t2 - um2 * t1);
                    const double ua1 = um1 + (um2 * t0 - um0 * t2);
                    const double ua2 = um2 + (um0 * t1 - um1 * t0);
                    const double up0 = um0 + (ua1 * s2 - ua2 * s1);
                    const double up1 = um1 + (ua2 * s0 - ua0 * s2);
                    const double up2 = um2 + (ua0 * s1 - ua1 * s0);
                    q.vx = up0 + qm * e0 * dt2;
                    q.vy = up1 + qm * e1 * dt2;
                    q.vz = up2 + qm * e2 * dt2;
                    ken += q.vx * q.vx + q.vy * q.vy + q.vz * q.vz;
                    q.x = q.x + q.vx * dt;
                    q.y = q.y + q.vy * dt;
                    q.z = q.z + q.vz * dt;
                }
                if (MODE == kModeGatherPush) {
                    if (active) store_bin64<true>(cur, (uint32_t)bin_slot(p, F, B, cap), q, ids);
                    continue;
                }
                // a particle still in its tile needs no wrap and no new tile
                bool stay = active && in_tile(q);
                if (REBIN && active && !stay) {
                    if (!(q.x >= 0.0 && q.x < nx && q.y >= 0.0 && q.y < ny && q.z >= 0.0 &&
                          q.z < nz)) {
                        q.x = apply_periodic(apply_periodic(q.x, nx), nx);
                        q.y = apply_periodic(apply_periodic(q.y, ny), ny);
                        q.z = apply_periodic(apply_periodic(q.z, nz), nz);
                        if (!(q.x >= 0.0 && q.x < nx && q.y >= 0.0 && q.y < ny && q.z >= 0.0 &&
                              q.z < nz)) {
                            count_lanes(&I->flags[kFlagRange]);
                            q.x = fmin(fmax(q.x - floor(q.x / nx) * nx, 0.0), nx - 1e-9);
                            q.y = fmin(fmax(q.y - floor(q.y / ny) * ny, 0.0), ny - 1e-9);
                            q.z = fmin(fmax(q.z - floor(q.z / nz) * nz, 0.0), nz - 1e-9);
                        }
                        stay = in_tile(q);
                    }
                }
                bool block = false;  // this wavefront stores a full block
                int blk;             // its first slot (lane 0)
                int nst = 0;
                unsigned long long sm = 0ull;
                if (BINS) {
                    sm = __ballot(stay);
                    const unsigned long long lm = __ballot(active && !stay);
                    if (lm) {
                        // particles that left: per-wave LDS buffer, routed in batches
                        const int nl = (int)__popcll(lm);
                        const bool leave = active && !stay;
                        if (lc + nl > kLeaveCap) {
                            flush_leavers<TX, TY, TZ, IDS>(sLeave[wv], lc, I, S, nbuf, ids);
                            lc = 0;
                        }
                        if (nl <= kLeaveCap) {
                            if (leave) sLeave[wv].put(lc + lane_rank(lm), q, ids);
                            lc += nl;
                        } else if (leave) {
                            route_back(S, nbuf, tile_of<TX, TY, TZ>(q, ntx, nty), q, ids, I->flags);
                        }
                    }
                    nst = (int)__popcll(sm);
                    const int holes = 64 - nst;
                    block = holes <= sc;
                    if (block) {
                        // (arrives while the charge is deposited)
                        if (excl && lane == 0) blk = atomicAdd(&sBlk[s], 64);
                        sc -= holes;
                        taken += 64;
                    }
                }
                if (DEP && active) {
                    const int ix = (int)q.x, iy = (int)q.y, iz = (int)q.z;
                    double wx0, wx1, wy0, wy1, wz0, wz1;
                    cic_w<WO>(q.x - (double)ix, wx0, wx1);
                    cic_w<WO>(q.y - (double)iy, wy0, wy1);
                    cic_w<WO>(q.z - (double)iz, wz0, wz1);
                    const double wx[2] = {wx0, wx1}, wy[2] = {wy0, wy1}, wz[2] = {wz0, wz1};
                    int dx = ix - lox + 1, dy = iy - loy + 1, dz = iz - loz + 1;
                    if (!stay) {
                        dx = wrap_index(dx, nx);
                        dy = wrap_index(dy, ny);
                        dz = wrap_index(dz, nz);
                    }
                    if (dx <= TX + 1 && dy <= TY + 1 && dz <= TZ + 1) {
                        const int l0 = dx + RX * (dy + RY * dz);
#pragma unroll
                        for (int i = 0; i < 2; ++i)
#pragma unroll
                            for (int j = 0; j < 2; ++j)
#pragma unroll
                                for (int k = 0; k < 2; ++k) {
                                    const long long v = fix_round(wx[i] * wy[j] * wz[k], qfix);
                                    atomicAdd(&sR[l0 + i + RX * (j + RY * k)],
                                              (unsigned long long)v);
                                }
                    } else {
                        unsigned long long *__restrict__ racc = I->rho_acc[acc_buf];
                        count_lanes(&I->flags[kFlagFast]);
#pragma unroll
                        for (int i = 0; i < 2; ++i)
#pragma unroll
                            for (int j = 0; j < 2; ++j)
#pragma unroll
                                for (int k = 0; k < 2; ++k) {
                                    const int gx = (ix + i) % nx, gy = (iy + j) % ny,
                                              gz = (iz + k) % nz;
                                    const long long v = fix_round(wx[i] * wy[j] * wz[k], qfix);
                                    gatomic_add(&racc[gx + (int64_t)nx * (gy + (int64_t)ny * gz)],
                                                (unsigned long long)v);
                                }
                    }
                }
                // the particle loaded ahead arrives before the stores are issued:
                // memory operations complete in order, so a wait for it at the
                // top of the next iteration would be one for these stores as well
                if (BINS) arrived(nextq, ids);
                if (LIST) {
                    // retry path: every particle to the species' contiguous
                    // list, in bin order inside this item's reserved range
                    if (active) store_p64(S, nbuf, list0 + (p - start), q, ids);
                } else if (block) {
                    wave_sync();
                    if (!stay) sStash[wv].get(sc + lane_rank(~sm), q, ids);
                    if (!excl && lane == 0) blk = claim_block(I, it, s);
                    store_bin64<true>(nxt, (uint32_t)(lane_bcast(blk, 0) + lane), q, ids);
                } else if (nst > 0) {
                    wave_sync();
                    if (stay) sStash[wv].put(sc + lane_rank(sm), q, ids);
                    sc += nst;
                }
            }
            if (BINS) {
                flush_leavers<TX, TY, TZ, IDS>(sLeave[wv], lc, I, S, nbuf, ids);
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
                        P64 q;
                        sStash[wv].get(lane, q, ids);
                        store_bin64<false>(nxt, (uint32_t)(o + lane), q, ids);
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
                        P64 q;
                        sStash[wv].get(lane, q, ids);
                        store_bin64<false>(nxt, (uint32_t)(cap - 1 - back - lane), q, ids);
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
__device__ __forceinline__ bool in_box(const InstDev *I, double x, double y, double z)
{
    return x >= 0.0 && x < I->n[0] && y >= 0.0 && y < I->n[1] && z >= 0.0 && z < I->n[2];
}

// Count a contiguous list [0, n) of buffer lbuf into the bin words of buffer
// lbuf^1 (front runs).  wrap != 0 applies the periodic wrap twice first.
__global__ void k_bin_count(const InstDev *__restrict__ insts, int inst, int s, int lbuf,
                            int64_t n, int tx_, int ty_, int tz_, int wrap)
{
    const InstDev *I = insts + inst;
    const SpecDev &S = I->sp[s];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < n;
    double x = 0.0, y = 0.0, z = 0.0;
    if (live) {
        x = gload((const double *)S.buf[lbuf][0], i);
        y = gload((const double *)S.buf[lbuf][1], i);
        z = gload((const double *)S.buf[lbuf][2], i);
        if (wrap) {
            x = apply_periodic(apply_periodic(x, I->n[0]), I->n[0]);
            y = apply_periodic(apply_periodic(y, I->n[1]), I->n[1]);
            z = apply_periodic(apply_periodic(z, I->n[2]), I->n[2]);
        }
    }
    const bool inb = live && in_box(I, x, y, z);
    if (live && !inb) count_lanes(&I->flags[kFlagRange]);
    const int t =
        inb ? ((int)x) / tx_ + I->nt[0] * (((int)y) / ty_ + I->nt[1] * (((int)z) / tz_)) : 0;
    (void)wave_counter_add(S.count[lbuf ^ 1], t, inb);
}

// Scatter the list into the front runs of buffer lbuf^1 (words zeroed on
// entry; caps already sized from k_bin_count).
__global__ void k_bin_scatter(const InstDev *__restrict__ insts, int inst, int s, int lbuf,
                              int64_t n, int tx_, int ty_, int tz_, int wrap)
{
    const InstDev *I = insts + inst;
    const SpecDev &S = I->sp[s];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < n;
    const bool ids = I->track_ids != 0;
    P64 q{0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0};
    if (live) {
        q = load_p64(S, lbuf, i, ids);
        if (wrap) {
            q.x = apply_periodic(apply_periodic(q.x, I->n[0]), I->n[0]);
            q.y = apply_periodic(apply_periodic(q.y, I->n[1]), I->n[1]);
            q.z = apply_periodic(apply_periodic(q.z, I->n[2]), I->n[2]);
        }
    }
    const bool inb = live && in_box(I, q.x, q.y, q.z);
    const int t = inb ? ((int)q.x) / tx_ + I->nt[0] * (((int)q.y) / ty_ + I->nt[1] * (((int)q.z) / tz_))
                      : 0;
    const unsigned long long old = wave_counter_add(S.count[lbuf ^ 1], t, inb);
    if (!inb) return;
    const int slot = bin_front(old);
    if (slot < gload(S.bin_cap, t))
        store_p64(S, lbuf ^ 1, gload(S.bin_base, t) + slot, q, ids);
    else
        count_lanes(&I->flags[kFlagOverflow]);
}

// Compact both runs of bins tiles[i] (tiles null: t0 + i) of buffer src into
// contiguous lists of buffer dst at list_off[i].  One workgroup per bin.  With
// src == dst each list must lie outside every bin's current slots.
__global__ void k_bins_to_list(const InstDev *__restrict__ insts, int inst, int s, int src,
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
        const int64_t o = ib + bin_slot(v, F, B, cap);
#pragma unroll
        for (int c = 0; c < 6; ++c)
            ((double *)S.buf[dst][c])[ob + v] = ((const double *)S.buf[src][c])[o];
        if (ids) S.pid[dst][ob + v] = S.pid[src][o];
    }
}

__global__ void k_cell_counts(const InstDev *__restrict__ insts, int inst, int s, int par,
                              int32_t *__restrict__ counts)
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
    for (int v = threadIdx.x; v < F + B; v += blockDim.x) {
        const int64_t o = b + bin_slot(v, F, B, cap);
        const double x = ((const double *)S.buf[par][0])[o];
        const double y = ((const double *)S.buf[par][1])[o];
        const double z = ((const double *)S.buf[par][2])[o];
        const int64_t c = (int)x + (int64_t)nx * ((int)y + (int64_t)ny * (int)z);
        atomicAdd(&counts[c], 1);
    }
}

}  // namespace

// ---------------------------------------------------------------- launchers
// List mode always handles ids (it is the rare retry); a deposit reads none.
template <int TX, int TY, int TZ, int WO>
static hipError_t launch_tile(int mode, bool ids, const InstDev *insts, const WorkItem *items,
                              int nitems, const int *parity, hipStream_t st)
{
    dim3 g(nitems), b(fp_block(TX * TY * TZ));
#define OHPIC_FP_CASE(M, IDS)                                                                     \
    hipLaunchKernelGGL((k_particles_fp64<TX, TY, TZ, WO, M, IDS>), g, b, 0, st, insts, items, parity, \
                       nullptr, nitems)
    switch (mode) {
    case kModeFused:
        if (ids)
            OHPIC_FP_CASE(kModeFused, true);
        else
            OHPIC_FP_CASE(kModeFused, false);
        break;
    case kModeGatherPush:
        if (ids)
            OHPIC_FP_CASE(kModeGatherPush, true);
        else
            OHPIC_FP_CASE(kModeGatherPush, false);
        break;
    case kModeBoundary:
        if (ids)
            OHPIC_FP_CASE(kModeBoundary, true);
        else
            OHPIC_FP_CASE(kModeBoundary, false);
        break;
    case kModeDeposit: OHPIC_FP_CASE(kModeDeposit, false); break;
    case kModeFusedList: OHPIC_FP_CASE(kModeFusedList, true); break;
    case kModeBoundaryList: OHPIC_FP_CASE(kModeBoundaryList, true); break;
    default:
        return hipErrorInvalidValue;
    }
#undef OHPIC_FP_CASE
    return hipGetLastError();
}

template <int TX, int TY, int TZ, int WO>
static hipError_t launch_tile_queue(bool ids, const InstDev *insts, const WorkItem *items,
                                    int nitems, const int *parity, unsigned int *queue, int blocks,
                                    hipStream_t st)
{
    if (ids)
        hipLaunchKernelGGL((k_particles_fp64<TX, TY, TZ, WO, kModeFusedQueue, true>), dim3(blocks),
                           dim3(fp_block(TX * TY * TZ)), 0, st, insts, items, parity, queue, nitems);
    else
        hipLaunchKernelGGL((k_particles_fp64<TX, TY, TZ, WO, kModeFusedQueue, false>), dim3(blocks),
                           dim3(fp_block(TX * TY * TZ)), 0, st, insts, items, parity, queue, nitems);
    return hipGetLastError();
}

template <int TX, int TY, int TZ, int WO>
static int queue_blocks_per_cu(bool ids)
{
    int nb = 0;
    const void *f = ids ? reinterpret_cast<const void *>(
                              &k_particles_fp64<TX, TY, TZ, WO, kModeFusedQueue, true>)
                        : reinterpret_cast<const void *>(
                              &k_particles_fp64<TX, TY, TZ, WO, kModeFusedQueue, false>);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, fp_block(TX * TY * TZ), 0) != hipSuccess) {
        (void)hipGetLastError();
        nb = 1;
    }
    return nb > 0 ? nb : 1;
}

bool tile_supported(int tx, int ty, int tz)
{
    return (tx == ty && ty == tz && (tx == 4 || tx == 8)) || (tx == 8 && ty == 8 && tz == 4) ||
           (tx == 16 && ty == 8 && tz == 4);
}

hipError_t launch_particles(int mode, int precision, int weight_order, const int T[3], bool ids,
                            const InstDev *insts, const WorkItem *items, int nitems,
                            const int *parity, hipStream_t st)
{
    if (nitems <= 0) return hipSuccess;
    if (precision == 1)
        return launch_particles_mixed(mode, weight_order, T, ids, insts, items, nitems, parity, st);
    if (precision != 0) return hipErrorInvalidValue;
#define OHPIC_TILE(A, B, C)                                                               \
    if (T[0] == A && T[1] == B && T[2] == C)                                              \
        return weight_order == 0                                                          \
                   ? launch_tile<A, B, C, 0>(mode, ids, insts, items, nitems, parity, st) \
                   : launch_tile<A, B, C, 1>(mode, ids, insts, items, nitems, parity, st);
    OHPIC_TILE(4, 4, 4)
    OHPIC_TILE(8, 8, 8)
    OHPIC_TILE(8, 8, 4)
    OHPIC_TILE(16, 8, 4)
#undef OHPIC_TILE
    return hipErrorInvalidValue;
}

hipError_t launch_particles_queue(int precision, int weight_order, const int T[3], bool ids,
                                  const InstDev *insts, const WorkItem *items, int nitems,
                                  const int *parity, unsigned int *queue, int blocks,
                                  hipStream_t st)
{
    if (nitems <= 0) return hipSuccess;
    if (blocks > nitems) blocks = nitems;
    if (blocks < 1) blocks = 1;
    if (precision == 1)
        return launch_particles_mixed_queue(weight_order, T, ids, insts, items, nitems, parity,
                                            queue, blocks, st);
    if (precision != 0) return hipErrorInvalidValue;
#define OHPIC_TILE(A, B, C)                                                                       \
    if (T[0] == A && T[1] == B && T[2] == C)                                                      \
        return weight_order == 0 ? launch_tile_queue<A, B, C, 0>(ids, insts, items, nitems,       \
                                                                 parity, queue, blocks, st)       \
                                 : launch_tile_queue<A, B, C, 1>(ids, insts, items, nitems,       \
                                                                 parity, queue, blocks, st);
    OHPIC_TILE(4, 4, 4)
    OHPIC_TILE(8, 8, 8)
    OHPIC_TILE(8, 8, 4)
    OHPIC_TILE(16, 8, 4)
#undef OHPIC_TILE
    return hipErrorInvalidValue;
}

int particles_queue_blocks(int precision, int weight_order, const int T[3], bool ids, int cus)
{
    int per = 1;
    if (precision == 1) {
        per = particles_mixed_queue_blocks(weight_order, T, ids);
    } else {
#define OHPIC_TILE(A, B, C)                                                  \
    if (T[0] == A && T[1] == B && T[2] == C)                                 \
        per = weight_order == 0 ? queue_blocks_per_cu<A, B, C, 0>(ids)       \
                                : queue_blocks_per_cu<A, B, C, 1>(ids);
    OHPIC_TILE(4, 4, 4)
    OHPIC_TILE(8, 8, 8)
    OHPIC_TILE(8, 8, 4)
    OHPIC_TILE(16, 8, 4)
#undef OHPIC_TILE
    }
    return per * cus;
}

hipError_t launch_bin_count(const InstDev *insts, int inst, int s, int lbuf, int64_t n,
                            const int T[3], int wrap, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const int64_t blocks = (n + 255) / 256;
    hipLaunchKernelGGL(k_bin_count, dim3((unsigned)blocks), dim3(256), 0, st, insts, inst, s,
                       lbuf, n, T[0], T[1], T[2], wrap);
    return hipGetLastError();
}

hipError_t launch_bin_scatter(const InstDev *insts, int inst, int s, int lbuf, int64_t n,
                              const int T[3], int wrap, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const int64_t blocks = (n + 255) / 256;
    hipLaunchKernelGGL(k_bin_scatter, dim3((unsigned)blocks), dim3(256), 0, st, insts, inst, s,
                       lbuf, n, T[0], T[1], T[2], wrap);
    return hipGetLastError();
}

// Bins tiles[i] of species s take base[i] and cap[i], and used[i] particles
// as one front run of buffer par (after their particles moved there).
__global__ void k_set_bins(const InstDev *__restrict__ insts, int inst, int s, int par,
                           const int *__restrict__ tiles, const int64_t *__restrict__ base,
                           const int32_t *__restrict__ cap, const int64_t *__restrict__ used,
                           int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const SpecDev &S = insts[inst].sp[s];
    const int t = tiles[i];
    S.bin_base[t] = base[i];
    S.bin_cap[t] = cap[i];
    S.count[par][t] = (unsigned long long)used[i];
}

hipError_t launch_set_bins(const InstDev *insts, int inst, int s, int par, const int *tiles,
                           const int64_t *base, const int32_t *cap, const int64_t *used, int n,
                           hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_set_bins, dim3((n + 255) / 256), dim3(256), 0, st, insts, inst, s, par,
                       tiles, base, cap, used, n);
    return hipGetLastError();
}

hipError_t launch_bins_to_list(const InstDev *insts, int inst, int s, int src, int dst,
                               const int *tiles, int t0, int ntiles, const int64_t *list_off,
                               hipStream_t st)
{
    if (ntiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_bins_to_list, dim3(ntiles), dim3(256), 0, st, insts, inst, s, src, dst,
                       tiles, t0, list_off);
    return hipGetLastError();
}

hipError_t launch_cell_counts(const InstDev *insts, int inst, int s, int par, int ntiles,
                              int32_t *counts, hipStream_t st)
{
    if (ntiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_cell_counts, dim3(ntiles), dim3(256), 0, st, insts, inst, s, par,
                       counts);
    return hipGetLastError();
}

}  // namespace ohpic
