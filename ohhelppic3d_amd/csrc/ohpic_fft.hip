// ohpic_fft.hip -- separable real-to-real 3-D FFT (FFTW R2HC / HC2R
// semantics) and the periodic spectral Poisson solve for gfx950.
//
// Replaces the FFTW-MPI backend (mpi_fftw3_solver.f90:39-236) and
// poissonSolver3d_solve (poisson_solver3d.f90:134-207) on one device.
//
// Each launch transforms every line of one axis of an nx*ny*nz array (x
// fastest).  Lines of n = A B points with A, B <= 16 take k_fft_two_step; for
// the others (longer lines, and lengths without such factors) a workgroup of
// k_fft_pass loads G real lines of that axis with coalesced
// reads (G consecutive rows for x; G consecutive x positions for y and z),
// packs line pairs into complex lines z = a + i b in LDS, runs a mixed-radix
// Stockham FFT in LDS (radix 4/2/3/5 and a generic small-prime stage), and
// unpacks the two real spectra into FFTW's halfcomplex order
// r0, r1, ..., r_{n/2}, i_{(n+1)/2-1}, ..., i1.  The inverse runs the same
// steps backwards.  The z pass of the Poisson solve is fused: forward along
// z, divide by the modified wave number sum (DC := 0), inverse along z, in one
// LDS-resident visit of each z line.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "ohpic_dft.hpp"
#include "ohpic_fft.hpp"
#include "ohpic_internal.hpp"

namespace ohpic {

namespace {

__device__ __forceinline__ int fastdiv(int t, uint32_t m)
{
    return m ? (int)__umulhi((uint32_t)t, m) : t;
}

// One Stockham radix-P stage, in place over `nlines` complex lines of length
// n held in LDS.  Task (line, row, f): inputs y[(row + q*r)*Ls + f] times
// w_L^{f q}, outputs y[row*L + f + Ls*u] = sum_q (...) w_p^{u q}.  Every
// thread reads the inputs of all its tasks into registers, the block
// synchronises, then the outputs are written back over the same buffer.
// Twiddle tables live in global memory, or (TL) in the workgroup's LDS copy
// for lengths up to kTwLds: staged once per workgroup (4 KiB at n = 256, so
// 8 workgroups still fit a CU), they cut a single-transform pass of 256-point
// lines at 256^3 from 60-62 us to 56-59 us.
constexpr int kTwLds = 256;
typedef double d2v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) d2v lds_d2v;

template <int SIGN, bool TL>
__device__ __forceinline__ cplx twiddle(const double2 *__restrict__ tw, int k)
{
    // one 16-byte load (a native vector type: HIP's double2 class does not
    // bind to an address-space-qualified reference)
    d2v w;
    if (TL)
        w = ((const lds_d2v *)tw)[k];
    else
        w = gload(reinterpret_cast<const d2v *>(tw), k);
    return cplx{w.x, SIGN < 0 ? w.y : -w.y};
}

template <int SIGN, int P, bool TL>
__device__ __forceinline__ void fft_stage(cplx *__restrict__ buf, int n, int nlines, int Ls,
                                          const double2 *__restrict__ tw, uint32_t mg_tpl,
                                          uint32_t mg_Ls)
{
    constexpr int KMAX = (kFftLdsCplx / kFftBlock + P - 1) / P;  // tasks per thread
    const int L = Ls * P;
    const int r = n / L;
    const int tpl = n / P;
    const int total = tpl * nlines;
    cplx a[KMAX][P];
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
        const int t = threadIdx.x + k * kFftBlock;
        if (t < total) {
            const int line = fastdiv(t, mg_tpl);
            const int i = t - line * tpl;
            const int row = fastdiv(i, mg_Ls);
            const int f = i - row * Ls;
            const cplx *s = buf + line * n;
#pragma unroll
            for (int q = 0; q < P; ++q) {
                cplx v = s[(row + q * r) * Ls + f];
                if (q > 0 && f > 0) v = cmul(v, twiddle<SIGN, TL>(tw, f * q * r));
                a[k][q] = v;
            }
            Dft<SIGN, P>::run(a[k]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
        const int t = threadIdx.x + k * kFftBlock;
        if (t < total) {
            const int line = fastdiv(t, mg_tpl);
            const int i = t - line * tpl;
            const int row = fastdiv(i, mg_Ls);
            const int f = i - row * Ls;
            cplx *d = buf + line * n + row * L + f;
#pragma unroll
            for (int u = 0; u < P; ++u) d[Ls * u] = a[k][u];
        }
    }
    __syncthreads();
}

// Runs all stages in place.  RS selects the compiled radix set (0: 4 and 2;
// 1: 4, 2 and 3; 2: every prime up to kMaxRadix) so power-of-two lengths do
// not pay the register cost of the large generic stages.
template <int SIGN, int RS, bool TL>
__device__ __forceinline__ void fft_lds_t(cplx *buf, int n, int nlines, const FftAxisDev &ax,
                                          const double2 *tw)
{
    int Ls = 1;
    for (int s = 0; s < ax.nfac; ++s) {
        const int p = ax.fac[s];
        const uint32_t mt = ax.mg_tpl[s], ml = ax.mg_Ls[s];
        if (p == 4) {
            fft_stage<SIGN, 4, TL>(buf, n, nlines, Ls, tw, mt, ml);
        } else if (p == 2) {
            fft_stage<SIGN, 2, TL>(buf, n, nlines, Ls, tw, mt, ml);
        } else if (RS >= 1 && p == 3) {
            fft_stage<SIGN, 3, TL>(buf, n, nlines, Ls, tw, mt, ml);
        } else if (RS >= 2) {
            switch (p) {
            case 5: fft_stage<SIGN, 5, TL>(buf, n, nlines, Ls, tw, mt, ml); break;
            case 7: fft_stage<SIGN, 7, TL>(buf, n, nlines, Ls, tw, mt, ml); break;
            case 11: fft_stage<SIGN, 11, TL>(buf, n, nlines, Ls, tw, mt, ml); break;
            default: fft_stage<SIGN, 13, TL>(buf, n, nlines, Ls, tw, mt, ml); break;
            }
        }
        Ls *= p;
    }
}

// All stages, twiddles from the LDS copy stw when the kernel staged them
// (lengths up to kTwLds), else from the global table.
template <int SIGN, int RS>
__device__ __forceinline__ void fft_lds(cplx *buf, int n, int nlines, const FftAxisDev &ax,
                                        const double2 *stw)
{
    if (n <= kTwLds)
        fft_lds_t<SIGN, RS, true>(buf, n, nlines, ax, stw);
    else
        fft_lds_t<SIGN, RS, false>(buf, n, nlines, ax, ax.tw);
}

// The G lines of one workgroup: line g (< nvalid) starts at element
// base + g * gstride and its elements are estride apart.  x: G consecutive
// rows; y: G consecutive x positions of one z plane; z: G consecutive (x, y)
// positions.
struct LineBlock {
    int64_t base;
    int64_t estride;
    int gstride;
    int nvalid;
};

template <int AXIS>
__device__ __forceinline__ LineBlock line_block(int grp, int G, int nx, int ny, int nz)
{
    LineBlock b;
    if (AXIS == 0) {
        const int64_t row0 = (int64_t)grp * G;
        b.base = row0 * nx;
        b.gstride = nx;
        b.estride = 1;
        b.nvalid = (int)min<int64_t>(G, (int64_t)ny * nz - row0);
    } else if (AXIS == 1) {
        const int gpp = (nx + G - 1) / G;
        const int iz = grp / gpp;
        const int ix0 = (grp - iz * gpp) * G;
        b.base = ix0 + (int64_t)nx * ny * iz;
        b.gstride = 1;
        b.estride = nx;
        b.nvalid = min(G, nx - ix0);
    } else {
        const int64_t l0 = (int64_t)grp * G;
        b.base = l0;
        b.gstride = 1;
        b.estride = (int64_t)nx * ny;
        b.nvalid = (int)min<int64_t>(G, (int64_t)nx * ny - l0);
    }
    return b;
}

// element e of the group -> (line g, position j): x lines are read row by
// row (g = e / n), y and z lines across the G lines first (j = e / G) so a
// wavefront touches G consecutive doubles per position
template <int AXIS>
__device__ __forceinline__ void elem_of(int e, int n, int G, const FftAxisDev &ax, int &g, int &j)
{
    if (AXIS == 0) {
        g = fastdiv(e, ax.mg_n);
        j = e - g * n;
    } else {
        j = fastdiv(e, ax.mg_G);
        g = e - j * G;
    }
}

constexpr int kLineElems = 2 * kFftLdsCplx / kFftBlock;  // real elements per thread

// Load G real lines into LDS packed as complex (line pair -> re/im).  Every
// thread issues all of its (up to kLineElems) global loads before the first
// LDS write, so each lane keeps that many reads in flight.
template <int AXIS>
__device__ void load_lines(const gmem_t<double> *__restrict__ src, cplx *buf, const LineBlock &lb,
                           int G, int n, const FftAxisDev &ax)
{
    double *bd = reinterpret_cast<double *>(buf);
    const int total = G * n;
    double v[kLineElems];
    int at[kLineElems];
#pragma unroll
    for (int k = 0; k < kLineElems; ++k) {
        const int e = threadIdx.x + k * kFftBlock;
        v[k] = 0.0;
        at[k] = -1;
        if (e < total) {
            int g, j;
            elem_of<AXIS>(e, n, G, ax, g, j);
            if (g < lb.nvalid)
                v[k] = src[lb.base + (int64_t)g * lb.gstride + (int64_t)j * lb.estride];
            at[k] = ((g >> 1) * n + j) * 2 + (g & 1);
        }
    }
#pragma unroll
    for (int k = 0; k < kLineElems; ++k)
        if (at[k] >= 0) bd[at[k]] = v[k];
}


// Task t of a (line pair c, position k < per_c) sweep: x lines take
// consecutive positions of one pair per wavefront (rows stay contiguous), y
// and z lines consecutive pairs at one position (the G lines of a position are
// adjacent in memory).
template <int AXIS>
__device__ __forceinline__ void pair_task(int t, int per_c, uint32_t mg_per, int nlines,
                                          uint32_t mg_nl, int &c, int &k)
{
    if (AXIS == 0) {
        c = fastdiv(t, mg_per);
        k = t - c * per_c;
    } else {
        k = fastdiv(t, mg_nl);
        c = t - k * nlines;
    }
}

// R2HC output: the task (c, k <= n/2) reads Z_k and Z_{n-k} once and writes
// r_k (position k) and i_k (position n - k) of both lines of the pair, with
// A_k = (Z_k + conj Z_{n-k}) / 2 and B_k = (Z_k - conj Z_{n-k}) / 2i.
template <int AXIS>
__device__ __forceinline__ void store_r2hc_pairs(const cplx *buf, gmem_t<double> *__restrict__ dst,
                                                 const LineBlock &lb, int n, int nlines,
                                                 const FftAxisDev &ax)
{
    const int half = n / 2 + 1;
    const int total = half * nlines;
    for (int t = threadIdx.x; t < total; t += kFftBlock) {
        int c, k;
        pair_task<AXIS>(t, half, ax.mg_half, nlines, ax.mg_nl, c, k);
        const int km = k == 0 ? 0 : n - k;
        const cplx zk = buf[c * n + k], zm = buf[c * n + km];
        const double ar = 0.5 * (zk.re + zm.re), ai = 0.5 * (zk.im - zm.im);
        const double br = 0.5 * (zk.im + zm.im), bi = 0.5 * (zm.re - zk.re);
        const int64_t la = lb.base + (int64_t)(2 * c) * lb.gstride;
        if (2 * c < lb.nvalid) {
            dst[la + (int64_t)k * lb.estride] = ar;
            if (km != k) dst[la + (int64_t)km * lb.estride] = ai;
        }
        if (2 * c + 1 < lb.nvalid) {
            const int64_t lbb = la + lb.gstride;
            dst[lbb + (int64_t)k * lb.estride] = br;
            if (km != k) dst[lbb + (int64_t)km * lb.estride] = bi;
        }
    }
}

// HC2R input: the task (c, k <= n/2) loads positions k and n - k of both
// halfcomplex lines and writes the packed spectrum Z = A + i B at k and n - k
// (A_k = r_k + i i_k from line a, B_k likewise from line b).
template <int AXIS>
__device__ __forceinline__ void load_hc_packed(const gmem_t<double> *__restrict__ src, cplx *buf,
                                               const LineBlock &lb, int n, int nlines,
                                               const FftAxisDev &ax)
{
    const int half = n / 2 + 1;
    const int total = half * nlines;
    for (int t = threadIdx.x; t < total; t += kFftBlock) {
        int c, k;
        pair_task<AXIS>(t, half, ax.mg_half, nlines, ax.mg_nl, c, k);
        const int km = k == 0 ? 0 : n - k;
        const int64_t la = lb.base + (int64_t)(2 * c) * lb.gstride;
        double ak = 0.0, am = 0.0, bk = 0.0, bm = 0.0;
        if (2 * c < lb.nvalid) {
            ak = src[la + (int64_t)k * lb.estride];
            am = src[la + (int64_t)km * lb.estride];
        }
        if (2 * c + 1 < lb.nvalid) {
            bk = src[la + lb.gstride + (int64_t)k * lb.estride];
            bm = src[la + lb.gstride + (int64_t)km * lb.estride];
        }
        if (km == k) {  // k = 0 and k = n/2: real r_k of both lines
            buf[c * n + k] = cplx{ak, bk};
        } else {
            buf[c * n + k] = cplx{ak - bm, am + bk};
            buf[c * n + km] = cplx{ak + bm, bk - am};
        }
    }
}

// Complex output (HC2R and the Poisson pass): position m of the pair's
// spectrum holds (line a, line b) = (re, im).
template <int AXIS>
__device__ __forceinline__ void store_complex_pairs(const cplx *buf, gmem_t<double> *__restrict__ dst,
                                                    const LineBlock &lb, int n, int nlines,
                                                    const FftAxisDev &ax, double scale)
{
    const int total = n * nlines;
    for (int t = threadIdx.x; t < total; t += kFftBlock) {
        int c, m;
        pair_task<AXIS>(t, n, ax.mg_n, nlines, ax.mg_nl, c, m);
        const cplx z = buf[c * n + m];
        const int64_t la = lb.base + (int64_t)(2 * c) * lb.gstride + (int64_t)m * lb.estride;
        if (2 * c < lb.nvalid) dst[la] = z.re * scale;
        if (2 * c + 1 < lb.nvalid) dst[la + lb.gstride] = z.im * scale;
    }
}

// One axis pass for every job of the table (blockIdx.y = job, blockIdx.x =
// line group; groups beyond a job's count exit).  FROM_SRC reads job.src
// (rho) instead of transforming job.data in place; SCALE multiplies the
// output by job.inv_n (the final HC2R pass).
#ifndef OHPIC_FFT_MIN_WAVES
#define OHPIC_FFT_MIN_WAVES 8
#endif

template <int KIND, int AXIS, int RS, bool FROM_SRC, bool SCALE>
__global__ void __launch_bounds__(kFftBlock)
    __attribute__((amdgpu_waves_per_eu(OHPIC_FFT_MIN_WAVES, 8)))
    k_fft_pass(const FftJob *__restrict__ jobs)
{
    __shared__ cplx buf[kFftLdsCplx];
    __shared__ double sLamXY[KIND == kFftPoisson ? 64 : 1];
    __shared__ double2 sTw[kTwLds];
    const FftJob &J = jobs[blockIdx.y];
    const int nx = J.n[0], ny = J.n[1], nz = J.n[2];
    const FftAxisDev &ax = J.ax[AXIS];
    const int n = ax.n;
    if (ax.A) return;  // k_fft_two_step's
    const int G = fft_group_lines(n);
    const int64_t ngroups = fft_groups(AXIS, G, nx, ny, nz);
    if ((int64_t)blockIdx.x >= ngroups) return;
    // neighbouring line groups read the two halves of the same 128-byte
    // lines (y and z passes): keep them on one XCD
    const int grp = xcd_remap((int)blockIdx.x, (int)ngroups);
    const gmem_t<double> *__restrict__ src = as_global(FROM_SRC ? J.src : J.data);
    gmem_t<double> *__restrict__ dst = as_global(J.data);
    const double out_scale = SCALE ? J.inv_n : 1.0;
    const int nlines = (G + 1) / 2;
    const LineBlock lb = line_block<AXIS>(grp, G, nx, ny, nz);

    if (KIND == kFftPoisson && (int)threadIdx.x < G) {
        // lam_x(ix) + lam_y(iy) of z line g; the DC line (ix = iy = 0) is marked
        // by -1 (its k_z = 0 mode is set to zero)
        const int g = threadIdx.x;
        double v = 0.0;
        if (g < lb.nvalid) {
            const int l = (int)lb.base + g;
            const int iy = l / nx;
            const int ix = l - iy * nx;
            v = (l == 0) ? -1.0 : gload(J.lam[0], ix) + gload(J.lam[1], iy);
        }
        sLamXY[g] = v;
    }
    if (n <= kTwLds)
        for (int i = threadIdx.x; i < n; i += kFftBlock) {
            const d2v w = gload(reinterpret_cast<const d2v *>(ax.tw), i);
            sTw[i] = make_double2(w.x, w.y);
        }
    if (KIND == kFftHC2R)
        load_hc_packed<AXIS>(src, buf, lb, n, nlines, ax);
    else
        load_lines<AXIS>(src, buf, lb, G, n, ax);
    __syncthreads();

    if (KIND == kFftR2HC || KIND == kFftPoisson) {
        fft_lds<-1, RS>(buf, n, nlines, ax, sTw);
        if (KIND == kFftPoisson) {
            // Green's-function division on the packed spectra: with
            // Z = FFT(a + i b), A_k = (Z_k + conj Z_{n-k}) / 2 and
            // B_k = (Z_k - conj Z_{n-k}) / 2i; A and B are divided by their
            // lines' denominators (DC := 0) and repacked as A' + i B', whose
            // inverse transform is (n a', n b') as HC2R of the halfcomplex
            // quotients gives.  One task per (pair, k <= n/2) owns slots k and
            // n - k, so the update needs no barrier of its own; one reciprocal
            // per denominator (within an ulp of the quotient).
            const gmem_t<double> *__restrict__ lamz = as_global(J.lam[2]);
            const int half = n / 2 + 1;
            const int total = half * nlines;
            constexpr int kTasks = (kFftLdsCplx / 2 + kFftLdsCplx / 16 + kFftBlock - 1) / kFftBlock + 1;
            const uint32_t mg_half = ax.mg_half;
#pragma unroll
            for (int q = 0; q < kTasks; ++q) {
                const int t = threadIdx.x + q * kFftBlock;
                if (t >= total) break;
                const int c = fastdiv(t, mg_half);
                const int k = t - c * half;
                const int km = k == 0 ? 0 : n - k;
                const cplx zk = buf[c * n + k], zm = buf[c * n + km];
                cplx A = {0.5 * (zk.re + zm.re), 0.5 * (zk.im - zm.im)};
                cplx B = {0.5 * (zk.im + zm.im), -0.5 * (zk.re - zm.re)};
                const double la = sLamXY[2 * c], lbv = sLamXY[2 * c + 1];
                const double lz = lamz[k];
                if (2 * c < lb.nvalid) {
                    if (la < 0.0 && k == 0) {
                        A = {0.0, 0.0};
                    } else {
                        const double d = (la < 0.0 ? 0.0 : la) + lz;
                        const double rd = 1.0 / d;
                        A = {A.re * rd, A.im * rd};
                    }
                }
                if (2 * c + 1 < lb.nvalid) {
                    if (lbv < 0.0 && k == 0) {
                        B = {0.0, 0.0};
                    } else {
                        const double d = (lbv < 0.0 ? 0.0 : lbv) + lz;
                        const double rd = 1.0 / d;
                        B = {B.re * rd, B.im * rd};
                    }
                }
                buf[c * n + k] = cplx{A.re - B.im, A.im + B.re};
                if (km != k) buf[c * n + km] = cplx{A.re + B.im, B.re - A.im};
            }
            __syncthreads();
            fft_lds<+1, RS>(buf, n, nlines, ax, sTw);
        }
    } else {
        fft_lds<+1, RS>(buf, n, nlines, ax, sTw);
    }

    if (KIND == kFftR2HC)
        store_r2hc_pairs<AXIS>(buf, dst, lb, n, nlines, ax);
    else
        store_complex_pairs<AXIS>(buf, dst, lb, n, nlines, ax, out_scale);
}

// ------------------------------------------------ axis passes of n = A B points
// For n = A B with A, B <= 16 (fft_two_step): the transform as two steps of
// DFTs held in registers.  With positions p = j + B m and modes k = k1 + A k2,
//   X[k] = sum_j w_n^{j k1} w_B^{j k2} sum_m w_A^{m k1} x[j + B m]:
// thread j of a line loads its A points, DFT of A points, twiddles, transpose
// through LDS, and thread k1 takes the DFT of B points and holds X[k1 + A k2].
// A workgroup is one wavefront of 64 / max(A, B) complex lines (pairs of real
// lines), so its LDS exchanges need no barrier; every global access of a pass
// goes straight to or from registers.  A mode and its conjugate partner n - k
// meet through one more LDS exchange: unpacking R2HC output, packing HC2R
// input, and the Green's-function division of the fused Poisson z pass, whose
// inverse runs the same steps backwards.
//
// What bounds it: at 256^3 (16 x 16) a pass moves 16 B per node in 44 to 46 us,
// 5.9 TB/s (52 to 63 us with radix-4 stages in LDS; the fused z pass takes 56,
// its division included).  The passes of a small grid are one wavefront's
// chain of a load, two or three exchanges and a store: at 32^3 4.2 to 6.9 us
// each, where the LDS stages (2 to 5 round trips, twice the barriers) took 6.3
// to 12.3.  Solves, stages -> two steps: 64^3 59 -> 48 us, 90x126x75 115 -> 82,
// 128^3 113 -> 105, 169^3 1512 -> 196 (radix 13), 256^3 426 -> 406, and no
// length of 4 to 256 measured slower.  The step functions are compiled for
// each number of points and chosen once per step: with loops over 16 guarded
// points the passes at 32^3 took 5.3 to 9.3 us.
constexpr int kAbThreads = 64;
constexpr int kPlaneWaves = 4;          // most wavefronts of k_fft_planes
constexpr int64_t kPlaneLds = 64 << 10;  // and its LDS
constexpr int64_t kMaxPlanes = 512;      // planes of a launch (fft_by_planes)

// 1/d for 0 < d < 2^1000 (d = 0 gives inf, which the caller discards): the
// hardware estimate (about 23 correct bits) refined by two Newton steps, so
// the error is that of the final rounding.  Replacing correctly rounded
// divisions (and their branches) took the 256-point z pass from 82 to 67 us at
// 256^3.
__device__ __forceinline__ double fast_recip(double d)
{
    double r = __builtin_amdgcn_rcp(d);
    r = __fma_rn(__fma_rn(-d, r, 1.0), r, r);
    return __fma_rn(__fma_rn(-d, r, 1.0), r, r);
}

__device__ __forceinline__ void wave_exchange()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// f(P) with P as a constant; the same P in every lane.
template <int FIXED, class F>
__device__ __forceinline__ void with_points(int P, F &f)
{
#define OHPIC_POINTS(N) \
    case N: f(std::integral_constant<int, N>()); break
    if (FIXED) {
        f(std::integral_constant<int, FIXED ? FIXED : 2>());
        return;
    }
    switch (P) {
        OHPIC_POINTS(2);
        OHPIC_POINTS(3);
        OHPIC_POINTS(4);
        OHPIC_POINTS(5);
        OHPIC_POINTS(6);
        OHPIC_POINTS(7);
        OHPIC_POINTS(8);
        OHPIC_POINTS(9);
        OHPIC_POINTS(10);
        OHPIC_POINTS(11);
        OHPIC_POINTS(12);
        OHPIC_POINTS(13);
        OHPIC_POINTS(14);
        OHPIC_POINTS(15);
        OHPIC_POINTS(16);
    }
#undef OHPIC_POINTS
}

// One thread's place in a wavefront's complex lines of n = A B points: thread t
// of line c, taking part in step 1 (as j = t) and step 2 (as k1 = t).
struct TwoStep {
    int A, B, n, L, c, t;
    bool live, one, two;
    int RA, RB;         // odd rows of the LDS exchanges
    const cplx *tw;     // twiddles (LDS)
    cplx *xl;           // the line's exchange buffer (LDS)
    const double *lam;  // Poisson: lam_x + lam_y of the wavefront's real lines,
    const double *lz;   // and lam_z of the modes (LDS)
};

__host__ __device__ inline int two_step_row(int A, int B)  // complex values per line
{
    const int ra = B * (A | 1), rb = A * (B | 1);
    return ra > rb ? ra : rb;
}

// The 16 x 16 z pass exchanges real and imaginary parts one after the other,
// in half the LDS: with more registers and work per line than the other passes
// it is short of wavefronts in flight (6 per CU, with the split 10):
// 68 -> 56 us at 256^3.
__host__ __device__ constexpr bool two_step_split(int kind, int fixed)
{
    return kind == kFftPoisson && fixed == 16;
}

__device__ __forceinline__ TwoStep two_step_of(int A, int B, int L, uint32_t mg_M, int lane,
                                               const cplx *tw, cplx *xbuf)
{
    TwoStep w;
    w.A = A;
    w.B = B;
    w.n = A * B;
    w.L = L;
    const int M = max(A, B);
    w.c = fastdiv(lane, mg_M);
    w.t = lane - w.c * M;
    w.live = w.c < L;
    w.one = w.live && w.t < B;
    w.two = w.live && w.t < A;
    w.RA = A | 1;
    w.RB = B | 1;
    w.tw = tw;
    w.xl = xbuf + (w.live ? w.c : 0) * two_step_row(A, B);
    return w;
}

// Transforms the wavefront's lines in `a`.  load(count, step) fills a[m] with
// point t + step m of the thread's line, m < count; stage() makes the LDS
// tables ready; store(count, step) takes a[m] as point t + step m.
template <int KIND, int FIXED, class Load, class Stage, class Store>
__device__ __forceinline__ void two_step_lines(const TwoStep &W, cplx (&a)[16], Load &&load,
                                               Stage &&stage, Store &&store)
{
    constexpr int SIGN = KIND == kFftHC2R ? +1 : -1;
    using Sign = std::integral_constant<int, SIGN>;
    using Back = std::integral_constant<int, +1>;
    const int A = FIXED ? FIXED : W.A, B = FIXED ? FIXED : W.B, n = A * B;
    const int RA = FIXED ? (FIXED | 1) : W.RA, RB = FIXED ? (FIXED | 1) : W.RB;
    const int t = W.t;
    const bool one = W.one, two = W.two;
    cplx *xl = W.xl;

    // a[k] *= exp(SIGN 2 pi i t k / n)
    auto twiddles = [&](auto sign, auto count) __attribute__((always_inline))
    {
#pragma unroll
        for (int k = 1; k < decltype(count)::value; ++k) {
            const cplx w = W.tw[t * k];
            a[k] = cmul(a[k], cplx{w.re, decltype(sign)::value < 0 ? w.im : -w.im});
        }
    };
    // SPLIT: a[k] goes to place put(k) of the line's buffer and b[k] is read from
    // place get(k), real parts first and then the imaginary ones, so the buffer
    // holds doubles
    constexpr bool SPLIT = two_step_split(KIND, FIXED);
    auto exchange = [&](cplx (&b)[16], auto put, auto get) __attribute__((always_inline))
    {
        double *x = reinterpret_cast<double *>(xl), re[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) x[put(k)] = a[k].re;
        wave_exchange();
#pragma unroll
        for (int k = 0; k < 16; ++k) re[k] = x[get(k)];
        wave_exchange();
#pragma unroll
        for (int k = 0; k < 16; ++k) x[put(k)] = a[k].im;
        wave_exchange();
#pragma unroll
        for (int k = 0; k < 16; ++k) b[k] = cplx{re[k], x[get(k)]};
        wave_exchange();
    };
    auto by_row = [&](int k) __attribute__((always_inline)) { return t * 17 + k; };
    auto by_column = [&](int k) __attribute__((always_inline)) { return k * 17 + t; };
    // step 1 (thread j = t), twiddles, transpose
    auto first = [&](auto count) __attribute__((always_inline))
    {
        constexpr int P = decltype(count)::value;  // A
        constexpr int RP = P | 1;
        if (one) load(count, B);
        stage();
        wave_exchange();
        if (KIND == kFftHC2R) {
            // halfcomplex values V_p of both lines -> packed spectrum Z = A + i B
            if (one) {
#pragma unroll
                for (int m = 0; m < P; ++m) xl[m * RB + t] = a[m];
            }
            wave_exchange();
            if (one) {
                // position n - p: row P - 1 - m, or P - m (mod P) for t = 0
                const cplx *x = t == 0 ? xl + RB : xl + B - t;
#pragma unroll
                for (int m = 0; m < P; ++m) {
                    const int p = t + B * m;
                    const cplx v = a[m];
                    const cplx w = m == 0 && t == 0 ? xl[0] : x[(P - 1 - m) * RB];
                    const cplx lo = {v.re - w.im, w.re + v.im}, hi = {w.re + v.im, w.im - v.re};
                    // below n/2 up to m = P/2 - 1, above it from m = P/2 + 1
                    if (m == 0)
                        a[m] = t == 0 ? v : lo;
                    else if (2 * m + 2 <= P)
                        a[m] = lo;
                    else if (2 * m > P)
                        a[m] = hi;
                    else
                        a[m] = 2 * p == n ? v : (2 * p < n ? lo : hi);
                }
            }
            wave_exchange();  // reads done before the buffer is reused
        }
        if (one) {
            Dft<SIGN, P>::run(a);
            twiddles(Sign(), count);
            if (SPLIT) {
                exchange(a, by_row, by_column);
                return;
            }
#pragma unroll
            for (int k1 = 0; k1 < P; ++k1) xl[t * RP + k1] = a[k1];
        }
        wave_exchange();
    };
    // step 2 (thread k1 = t): a[k2] = X[t + A k2], and what follows on modes
    auto second = [&](auto count) __attribute__((always_inline))
    {
        constexpr int P = decltype(count)::value;  // B
        constexpr int RP = P | 1;
        if (two) {
            if (!SPLIT)
#pragma unroll
                for (int j = 0; j < P; ++j) a[j] = xl[j * RA + t];
            Dft<SIGN, P>::run(a);
        }
        if (KIND == kFftHC2R) {
            if (two) store(count, A);
            return;
        }
        // each mode meets its partner n - k
        cplx z[16];
        if (SPLIT) {
            exchange(z, by_column, [&](int k2) __attribute__((always_inline)) {
                return t == 0 ? (k2 == 0 ? 0 : (16 - k2) * 17) : (15 - k2) * 17 + 16 - t;
            });
        } else {
            wave_exchange();  // transpose reads done
            if (two) {
#pragma unroll
                for (int k2 = 0; k2 < P; ++k2) xl[k2 * RA + t] = a[k2];
            }
            wave_exchange();
        }
        if (two) {
            // mode n - k: row P - 1 - k2, or P - k2 (mod P) for t = 0
            const cplx *x = t == 0 ? xl + RA : xl + A - t;
            const double lam_a = KIND == kFftPoisson ? W.lam[2 * W.c] : 0.0;
            const double lam_b = KIND == kFftPoisson ? W.lam[2 * W.c + 1] : 0.0;
            const double lxa = lam_a < 0.0 ? 0.0 : lam_a, lxb = lam_b < 0.0 ? 0.0 : lam_b;
#pragma unroll
            for (int k2 = 0; k2 < P; ++k2) {
                const int k = t + A * k2;
                const cplx zk = a[k2];
                const cplx zm = SPLIT ? z[k2] : k2 == 0 && t == 0 ? xl[0] : x[(P - 1 - k2) * RA];
                if (KIND == kFftR2HC) {
                    // position k of the halfcomplex lines: of A_k = (Z_k +
                    // conj Z_{n-k}) / 2 and B_k = (Z_k - conj Z_{n-k}) / 2i the
                    // real parts up to n/2, then the imaginary parts of mode
                    // n - k
                    // (k2 from P/2 + 1; up to P/2 - 1 real)
                    const bool im = 2 * k2 + 2 > P && (2 * k2 > P || 2 * k > n);
                    a[k2] = im ? cplx{0.5 * (zm.im - zk.im), 0.5 * (zk.re - zm.re)}
                               : cplx{0.5 * (zk.re + zm.re), 0.5 * (zk.im + zm.im)};
                } else {
                    // A_k and B_k divided by their lines' denominators (the DC
                    // line's k = 0 mode, whose denominator is 0, set to zero),
                    // repacked as A' + i B'
                    const double ra = fast_recip(lxa + W.lz[k]), rb = fast_recip(lxb + W.lz[k]);
                    const double sa = (lam_a < 0.0 && k == 0) ? 0.0 : 0.5 * ra;
                    const double sb = (lam_b < 0.0 && k == 0) ? 0.0 : 0.5 * rb;
                    const cplx U = {sa * (zk.re + zm.re), sa * (zk.im - zm.im)};
                    const cplx V = {sb * (zk.im + zm.im), -sb * (zk.re - zm.re)};
                    a[k2] = cplx{U.re - V.im, U.im + V.re};
                }
            }
        }
        if (KIND == kFftR2HC) {
            if (two) store(count, A);
            return;
        }
        // inverse: DFT over k2 (thread k1 = t), twiddles, transpose
        if (!SPLIT) wave_exchange();  // partner reads done before the buffer is reused
        if (two) {
            Dft<+1, P>::run(a);
            twiddles(Back(), count);
            if (SPLIT) {
                exchange(a, by_row, by_column);
                return;
            }
#pragma unroll
            for (int j = 0; j < P; ++j) xl[t * RP + j] = a[j];
        }
        wave_exchange();
    };
    // ... and over k1 (thread j = t)
    auto third = [&](auto count) __attribute__((always_inline))
    {
        constexpr int P = decltype(count)::value;  // A
        if (one) {
#pragma unroll
            for (int k1 = 0; k1 < P; ++k1)
                if (!SPLIT) a[k1] = xl[k1 * RB + t];
            Dft<+1, P>::run(a);
            store(count, B);
        }
    };
    with_points<FIXED>(A, first);
    with_points<FIXED>(B, second);
    if (KIND == kFftPoisson) with_points<FIXED>(A, third);
}

// Line access of a group of 2 L real lines in global memory: complex line c is
// real lines 2c (re) and 2c + 1 (im).  y and z lines are adjacent: one 16-byte
// access per point when every pair is aligned (an even stride; the number of
// lines is then even too).
template <int AXIS>
struct LineAccess {
    int64_t estride;
    uint32_t g1, lane0;  // offsets of the second line and of the thread's first point
    bool v16, va, vb;    // pair access; the two lines are there
    __device__ __forceinline__ LineAccess(const LineBlock &lb, const TwoStep &W)
    {
        estride = lb.estride;
        g1 = (uint32_t)lb.gstride;
        lane0 = (uint32_t)(2 * W.c) * g1 + (uint32_t)W.t * (uint32_t)lb.estride;
        v16 = AXIS != 0 && (lb.estride & 1) == 0;
        va = W.live && 2 * W.c < lb.nvalid;
        vb = W.live && 2 * W.c + 1 < lb.nvalid;
    }
    template <int P>
    __device__ __forceinline__ void load(cplx (&a)[16], const double *p, int step) const
    {
        const gmem_t<double> *s = as_global(p);
        const int64_t inc = step * estride;
#pragma unroll
        for (int m = 0; m < P; ++m) a[m] = cplx{0.0, 0.0};
        if (AXIS != 0 && v16) {
            if (va)
#pragma unroll
                for (int m = 0; m < P; ++m) {
                    const d2v v = ((const gmem_t<d2v> *)(s + m * inc))[lane0 >> 1];
                    a[m] = cplx{v.x, v.y};
                }
        } else {
            if (va)
#pragma unroll
                for (int m = 0; m < P; ++m) a[m].re = (s + m * inc)[lane0];
            if (vb)
#pragma unroll
                for (int m = 0; m < P; ++m) a[m].im = (s + m * inc)[lane0 + g1];
        }
    }
    template <int P>
    __device__ __forceinline__ void store(const cplx (&a)[16], double *p, int step) const
    {
        gmem_t<double> *d = as_global(p);
        const int64_t inc = step * estride;
        if (AXIS != 0 && v16) {
            if (va)
#pragma unroll
                for (int m = 0; m < P; ++m) {
                    d2v w;
                    w.x = a[m].re;
                    w.y = a[m].im;
                    ((gmem_t<d2v> *)(d + m * inc))[lane0 >> 1] = w;
                }
        } else {
            if (va)
#pragma unroll
                for (int m = 0; m < P; ++m) (d + m * inc)[lane0] = a[m].re;
            if (vb)
#pragma unroll
                for (int m = 0; m < P; ++m) (d + m * inc)[lane0 + g1] = a[m].im;
        }
    }
};

// Groups of `lines` real lines of an axis pass; x lines of a job whose planes
// can go by k_fft_planes (plane != 0) are grouped plane by plane.
__host__ __device__ inline int64_t two_step_groups(int axis, int lines, int nx, int ny, int nz,
                                                   int plane)
{
    if (axis == 0 && plane) return (int64_t)((ny + lines - 1) / lines) * nz;
    return fft_groups(axis, lines, nx, ny, nz);
}

// FIXED: A and B when known at compile time (16 x 16), else 0.
template <int KIND, int AXIS, bool FROM_SRC, bool SCALE, int FIXED>
__global__ void __launch_bounds__(kAbThreads) k_fft_two_step(const FftJob *__restrict__ jobs)
{
    extern __shared__ cplx ab_lds[];
    const FftJob &J = jobs[blockIdx.y];
    const int nx = J.n[0], ny = J.n[1], nz = J.n[2];
    const FftAxisDev &ax = J.ax[AXIS];
    // this launch's jobs: 16 x 16 or any other pair
    if (ax.A == 0 || (FIXED == 16) != (ax.A == 16 && ax.B == 16)) return;
    const int A = FIXED ? FIXED : ax.A, B = FIXED ? FIXED : ax.B, n = A * B;
    const int L = FIXED ? kAbThreads / FIXED : ax.ab_lines;
    const int64_t ngroups = two_step_groups(AXIS, 2 * L, nx, ny, nz, J.plane);
    if ((int64_t)blockIdx.x >= ngroups) return;
    // neighbouring groups read the parts of the same 128-byte lines (y and z
    // passes): keep them on one XCD
    const int grp = xcd_remap((int)blockIdx.x, (int)ngroups);
    LineBlock lb;
    if (AXIS == 0 && J.plane) {
        // rows pair up within their plane, as in k_fft_planes
        const int gpp = (int)(ngroups / nz), iz = grp / gpp, row = (grp - iz * gpp) * 2 * L;
        lb.base = (int64_t)nx * ((int64_t)ny * iz + row);
        lb.gstride = nx;
        lb.estride = 1;
        lb.nvalid = min(2 * L, ny - row);
    } else {
        lb = line_block<AXIS>(grp, 2 * L, nx, ny, nz);
    }
    const int tid = threadIdx.x;
    cplx *tw = ab_lds;  // twiddles, then the exchange buffers
    TwoStep W = two_step_of(A, B, L, FIXED ? fastdiv_magic(FIXED) : ax.mg_M, tid, tw, ab_lds + n);
    constexpr bool SPLIT = two_step_split(KIND, FIXED);
    if (SPLIT) W.xl = reinterpret_cast<cplx *>(reinterpret_cast<double *>(ab_lds + n) +
                                               W.c * two_step_row(A, B));
    double *lam = reinterpret_cast<double *>(ab_lds + n) +
                  (SPLIT ? 1 : 2) * L * two_step_row(A, B);  // 2 L
    double *lz = lam + 2 * L;                                                       // n
    W.lam = lam;
    W.lz = lz;

    // twiddles and z denominators on their way before the lines
    constexpr int TQ = 256 / kAbThreads;
    d2v wq[TQ];
    double zq[TQ];
#pragma unroll
    for (int q = 0; q < TQ; ++q) {
        const int i = min(tid + q * kAbThreads, n - 1);
        wq[q] = gload(reinterpret_cast<const d2v *>(ax.tw), i);
        if (KIND == kFftPoisson) zq[q] = gload(J.lam[2], i);
    }
    auto stage = [&]() __attribute__((always_inline))
    {
#pragma unroll
        for (int q = 0; q < TQ; ++q) {
            const int i = tid + q * kAbThreads;
            if (i < n) {
                tw[i] = cplx{wq[q].x, wq[q].y};
                if (KIND == kFftPoisson) lz[i] = zq[q];
            }
        }
        if (KIND == kFftPoisson && tid < 2 * L) {
            // lam_x + lam_y of real line tid; -1 marks the DC line (ix = iy = 0);
            // lines past the grid's end get 1 (they hold zeros; no 0/0)
            double v = 1.0;
            if (tid < lb.nvalid) {
                const int l = (int)lb.base + tid;  // < nx ny <= 2^20
                const int iy = l / nx, ix = l - iy * nx;
                v = (l == 0) ? -1.0 : gload(J.lam[0], ix) + gload(J.lam[1], iy);
            }
            lam[tid] = v;
        }
    };
    const LineAccess<AXIS> acc(lb, W);
    cplx a[16];
    auto load = [&](auto count, int step) __attribute__((always_inline))
    {
        acc.template load<decltype(count)::value>(a, (FROM_SRC ? J.src : J.data) + lb.base, step);
    };
    auto store = [&](auto count, int step) __attribute__((always_inline))
    {
        constexpr int P = decltype(count)::value;
        if (SCALE) {
            const double scale = J.inv_n;
#pragma unroll
            for (int m = 0; m < P; ++m) a[m] = cplx{a[m].re * scale, a[m].im * scale};
        }
        acc.template store<P>(a, J.data + lb.base, step);
    };
    two_step_lines<KIND, FIXED>(W, a, load, stage, store);
}

// ------------------------------------------------ x and y passes by planes
// Where the x and y lengths of every job take the two steps, a z plane fits in
// LDS with at most kPlaneWaves wavefronts of lines (fft_plan_planes) and there
// are few planes (fft_by_planes), one launch does both passes, a workgroup per
// plane: x then y (FWD) or y then x, the plane in LDS in between.  At such
// sizes a pass is latency; this saves the second one's launch, its trip through
// memory and the gap between the two: at 32^3 7.8 and 7.0 us against 4.5 + 4.6
// and 4.7 + 4.3 and the gaps.  STEP: at the start of a step rho comes from the
// charge grid on the way, and a wavefront of its own does the rest of
// launch_begin_step_b (9.7 us; k_begin_step_b and its gap took 4).  Steps:
// 32^3 92.1 -> 85.7 us, 45x50x63 147.0 -> 140.6, eight small instances 945 ->
// 895 per 8 steps.
// The limits: with 1280 planes (a group of 32 members of 16 to 64 cells) the
// pair took 25 us each way for the members that could, 21 to 24 by axis for all
// of them, since 200 registers and the planes' LDS leave few wavefronts per CU;
// 40x40x500 and 48x48x512 solve in 71 and 82 us against 77 and 89.
template <bool FWD, bool STEP>
__global__ void __launch_bounds__((kPlaneWaves + 1) * 64)
    k_fft_planes(const FftJob *__restrict__ jobs, FftStep step0)
{
    extern __shared__ cplx ab_lds[];
    const FftJob &J = jobs[blockIdx.y];
    const int nx = J.n[0], ny = J.n[1], nz = J.n[2];
    const int waves = J.plane;  // wavefronts at work
    if ((int)blockIdx.x >= nz) return;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const InstDev *I = STEP ? step0.insts + blockIdx.y : nullptr;
    const int par = STEP ? step0.parity[blockIdx.y] : 0;
    const FftAxisDev &ax = J.ax[0], &ay = J.ax[1];
    const int ps = nx | 1;  // row of the plane: odd, so columns and rows spread over the banks
    cplx *twx = ab_lds, *twy = twx + nx, *xbuf = twy + ny;
    const int row = max(ax.ab_lines * two_step_row(ax.A, ax.B), ay.ab_lines * two_step_row(ay.A, ay.B));
    double *plane = reinterpret_cast<double *>(xbuf + waves * row);
    xbuf += min(wave, waves - 1) * row;
    const int64_t base = (int64_t)nx * ny * blockIdx.x;
    auto stage = [&]() __attribute__((always_inline))
    {
        for (int i = tid; i < nx; i += (int)blockDim.x) {
            const d2v w = gload(reinterpret_cast<const d2v *>(ax.tw), i);
            twx[i] = cplx{w.x, w.y};
        }
        for (int i = tid; i < ny; i += (int)blockDim.x) {
            const d2v w = gload(reinterpret_cast<const d2v *>(ay.tw), i);
            twy[i] = cplx{w.x, w.y};
        }
        __syncthreads();
    };
    auto staged = []() {};
    cplx a[16];
    constexpr int KIND = FWD ? kFftR2HC : kFftHC2R;
    auto x_lines = [&](int g, auto &stage) __attribute__((always_inline))
    {
        const TwoStep W = two_step_of(ax.A, ax.B, ax.ab_lines, ax.mg_M, lane, twx, xbuf);
        LineBlock lb;
        lb.base = base + (int64_t)(g * 2 * W.L) * nx;
        lb.gstride = nx;
        lb.estride = 1;
        lb.nvalid = min(2 * W.L, ny - g * 2 * W.L);
        const LineAccess<0> acc(lb, W);
        double *p0 = plane + (g * 2 * W.L + 2 * W.c) * ps + W.t;
        auto load = [&](auto count, int step) __attribute__((always_inline))
        {
            constexpr int P = decltype(count)::value;
            if (FWD && STEP) {
                acc.template load<P>(a, (const double *)I->rho_acc[par] + lb.base, step);
                const double scale = I->fix_inv;
                cplx z[16];
#pragma unroll
                for (int m = 0; m < P; ++m) {
                    a[m].re = (double)__double_as_longlong(a[m].re) * scale;
                    a[m].im = (double)__double_as_longlong(a[m].im) * scale;
                    z[m] = cplx{0.0, 0.0};
                }
                acc.template store<P>(a, I->rho + lb.base, step);
                acc.template store<P>(z, (double *)I->rho_acc[par ^ 1] + lb.base, step);
            } else if (FWD) {
                acc.template load<P>(a, J.src + lb.base, step);
            } else {
#pragma unroll
                for (int m = 0; m < P; ++m)
                    a[m] = cplx{acc.va ? p0[m * step] : 0.0, acc.vb ? p0[m * step + ps] : 0.0};
            }
        };
        auto store = [&](auto count, int step) __attribute__((always_inline))
        {
            constexpr int P = decltype(count)::value;
            if (FWD) {
#pragma unroll
                for (int m = 0; m < P; ++m) {
                    if (acc.va) p0[m * step] = a[m].re;
                    if (acc.vb) p0[m * step + ps] = a[m].im;
                }
            } else {
                const double scale = J.inv_n;
#pragma unroll
                for (int m = 0; m < P; ++m) a[m] = cplx{a[m].re * scale, a[m].im * scale};
                acc.template store<P>(a, J.data + lb.base, step);
            }
        };
        two_step_lines<KIND, 0>(W, a, load, stage, store);
    };
    auto y_lines = [&](int g, auto &stage) __attribute__((always_inline))
    {
        const TwoStep W = two_step_of(ay.A, ay.B, ay.ab_lines, ay.mg_M, lane, twy, xbuf);
        LineBlock lb;
        lb.base = base + g * 2 * W.L;
        lb.gstride = 1;
        lb.estride = nx;
        lb.nvalid = min(2 * W.L, nx - g * 2 * W.L);
        const LineAccess<1> acc(lb, W);
        double *p0 = plane + W.t * ps + g * 2 * W.L + 2 * W.c;
        auto load = [&](auto count, int step) __attribute__((always_inline))
        {
            constexpr int P = decltype(count)::value;
            if (!FWD) {
                acc.template load<P>(a, J.data + lb.base, step);
            } else {
#pragma unroll
                for (int m = 0; m < P; ++m)
                    a[m] = cplx{acc.va ? p0[m * step * ps] : 0.0,
                                acc.vb ? p0[m * step * ps + 1] : 0.0};
            }
        };
        auto store = [&](auto count, int step) __attribute__((always_inline))
        {
            constexpr int P = decltype(count)::value;
            if (!FWD) {
#pragma unroll
                for (int m = 0; m < P; ++m) {
                    if (acc.va) p0[m * step * ps] = a[m].re;
                    if (acc.vb) p0[m * step * ps + 1] = a[m].im;
                }
            } else {
                acc.template store<P>(a, J.data + lb.base, step);
            }
        };
        two_step_lines<KIND, 0>(W, a, load, stage, store);
    };
    const int gx = (ny + 2 * ax.ab_lines - 1) / (2 * ax.ab_lines);
    const int gy = (nx + 2 * ay.ab_lines - 1) / (2 * ay.ab_lines);
    // one group of lines per wavefront and axis (waves is the larger number of
    // groups); every wavefront passes the barrier of stage() once
    if (FWD) {
        if (wave < gx)
            x_lines(wave, stage);
        else
            stage();
        if (STEP && wave == waves) {
            // the wavefront beyond those of the lines
            if (step0.queue && blockIdx.x == 0 && blockIdx.y == 0 && lane == 0) *step0.queue = 0u;
            if (blockIdx.x == 0 && lane < kFlagWords) I->flags[lane] = 0ull;
            clear_next(I, par, (int64_t)blockIdx.x * 64 + lane, (int64_t)nz * 64);
        }
        __syncthreads();
        if (wave < gy) y_lines(wave, staged);
    } else {
        if (wave < gy)
            y_lines(wave, stage);
        else
            stage();
        __syncthreads();
        if (wave < gx) x_lines(wave, staged);
    }
}

}  // namespace

void fft_plan_divisors(FftAxisDev &ax)
{
    ax.mg_n = fastdiv_magic((uint32_t)ax.n);
    ax.mg_G = fastdiv_magic((uint32_t)fft_group_lines(ax.n));
    ax.mg_half = fastdiv_magic((uint32_t)(ax.n / 2 + 1));
    ax.mg_nl = fastdiv_magic((uint32_t)(fft_group_lines(ax.n) / 2));
    fft_two_step(ax.n, &ax.A, &ax.B);
    ax.ab_lines = ax.A ? kAbThreads / (ax.A > ax.B ? ax.A : ax.B) : 0;
    ax.mg_M = fastdiv_magic((uint32_t)(ax.A > ax.B ? ax.A : ax.B));
    int Ls = 1;
    for (int s = 0; s < kMaxFactors; ++s) {
        const int p = s < ax.nfac ? ax.fac[s] : 1;
        ax.mg_tpl[s] = fastdiv_magic((uint32_t)(ax.n / p));
        ax.mg_Ls[s] = fastdiv_magic((uint32_t)Ls);
        Ls *= p;
    }
}

void fft_two_step(int n, int *A, int *B)
{
    *A = *B = 0;
    for (int a = 2; a <= 16 && a * a <= n; ++a)
        if (n % a == 0 && n / a <= 16) {
            *A = a;
            *B = n / a;
        }
}

int64_t fft_two_step_lds(int A, int B)
{
    const int L = kAbThreads / (A > B ? A : B);
    return (int64_t)(A * B + L * two_step_row(A, B)) * (int64_t)sizeof(double2) +
           (2 * L + A * B) * (int64_t)sizeof(double);
}

static int64_t two_step_split_lds()
{
    return fft_two_step_lds(16, 16) - 4 * two_step_row(16, 16) * (int64_t)sizeof(double);
}

// LDS bytes of k_fft_planes with `waves` wavefronts
static int64_t plane_lds(const FftJob &J, int waves)
{
    const FftAxisDev &ax = J.ax[0], &ay = J.ax[1];
    const int row = std::max(ax.ab_lines * two_step_row(ax.A, ax.B),
                             ay.ab_lines * two_step_row(ay.A, ay.B));
    return (int64_t)(ax.n + ay.n + waves * row) * (int64_t)sizeof(double2) +
           (int64_t)(ax.n | 1) * ay.n * (int64_t)sizeof(double);
}

void fft_plan_planes(FftJob &J)
{
    J.plane = 0;
    const FftAxisDev &ax = J.ax[0], &ay = J.ax[1];
    if (ax.A == 0 || ay.A == 0) return;
    const int gx = (ay.n + 2 * ax.ab_lines - 1) / (2 * ax.ab_lines);
    const int gy = (ax.n + 2 * ay.ab_lines - 1) / (2 * ay.ab_lines);
    const int waves = std::max(gx, gy);
    if (waves > kPlaneWaves || plane_lds(J, waves) > kPlaneLds) return;
    J.plane = waves;
}

void fft_solve_add(FftSolve &l, const FftJob &J)
{
    for (int a = 0; a < 3; ++a) fft_add(l.ax[a], J.ax[a], a, J.n[0], J.n[1], J.n[2], J.plane);
    if (J.plane == 0) {
        l.all_planes = false;
        return;
    }
    l.planes = std::max(l.planes, J.n[2]);
    l.total_planes += J.n[2];
    l.plane_waves = std::max(l.plane_waves, J.plane);
    l.lds = std::max(l.lds, plane_lds(J, J.plane));
}

bool fft_by_planes(const FftSolve &l)
{
    return l.all_planes && l.total_planes > 0 && l.total_planes <= kMaxPlanes;
}

void fft_add(FftLaunch &l, const FftAxisDev &ax, int axis, int nx, int ny, int nz, int plane)
{
    if (ax.A == 0) {
        l.groups = std::max(l.groups, fft_groups(axis, fft_group_lines(ax.n), nx, ny, nz));
        l.rs = std::max(l.rs, fft_radix_set(ax));
        return;
    }
    const int64_t g = two_step_groups(axis, 2 * ax.ab_lines, nx, ny, nz, plane);
    if (ax.A == 16 && ax.B == 16) {
        l.groups16 = std::max(l.groups16, g);
    } else {
        l.groups_ab = std::max(l.groups_ab, g);
        l.lds_ab = std::max(l.lds_ab, fft_two_step_lds(ax.A, ax.B));
    }
}

int fft_radix_set(const FftAxisDev &ax)
{
    int rs = 0;
    for (int i = 0; i < ax.nfac; ++i) {
        if (ax.fac[i] == 3 && rs < 1) rs = 1;
        if (ax.fac[i] > 4 && ax.fac[i] != 3) rs = 2;
    }
    return rs;
}

template <int KIND, int AXIS, bool FROM_SRC, bool SCALE>
static hipError_t launch_pass(const FftJob *jobs, int njobs, const FftLaunch &l, hipStream_t st)
{
    if (njobs <= 0) return hipSuccess;
    if (l.groups > 0) {
        const dim3 g((unsigned)round_up_xcds(l.groups), (unsigned)njobs), b(kFftBlock);
        if (l.rs == 0)
            hipLaunchKernelGGL((k_fft_pass<KIND, AXIS, 0, FROM_SRC, SCALE>), g, b, 0, st, jobs);
        else if (l.rs == 1)
            hipLaunchKernelGGL((k_fft_pass<KIND, AXIS, 1, FROM_SRC, SCALE>), g, b, 0, st, jobs);
        else
            hipLaunchKernelGGL((k_fft_pass<KIND, AXIS, 2, FROM_SRC, SCALE>), g, b, 0, st, jobs);
    }
    if (l.groups16 > 0) {
        const dim3 g((unsigned)round_up_xcds(l.groups16), (unsigned)njobs), b(kAbThreads);
        hipLaunchKernelGGL((k_fft_two_step<KIND, AXIS, FROM_SRC, SCALE, 16>), g, b,
                           (unsigned)(two_step_split(KIND, 16) ? two_step_split_lds()
                                                               : fft_two_step_lds(16, 16)),
                           st, jobs);
    }
    if (l.groups_ab > 0) {
        const dim3 g((unsigned)round_up_xcds(l.groups_ab), (unsigned)njobs), b(kAbThreads);
        hipLaunchKernelGGL((k_fft_two_step<KIND, AXIS, FROM_SRC, SCALE, 0>), g, b,
                           (unsigned)l.lds_ab, st, jobs);
    }
    return hipGetLastError();
}

hipError_t fft_poisson(const FftJob *jobs, int njobs, const FftSolve &l, const FftStep *step,
                       hipStream_t st)
{
    if (njobs <= 0) return hipSuccess;
    const bool planes = fft_by_planes(l);
    const dim3 g((unsigned)l.planes, (unsigned)njobs), b((unsigned)(64 * l.plane_waves)),
        b1((unsigned)(64 * (l.plane_waves + 1)));
    hipError_t e = hipSuccess;
    if (planes && step)
        hipLaunchKernelGGL((k_fft_planes<true, true>), g, b1, (unsigned)l.lds, st, jobs, *step);
    else if (planes)
        hipLaunchKernelGGL((k_fft_planes<true, false>), g, b, (unsigned)l.lds, st, jobs, FftStep{});
    else {
        e = fft_pass(kPassR2hcXFromSrc, jobs, njobs, l.ax[0], st);
        if (e == hipSuccess) e = fft_pass(kPassR2hcY, jobs, njobs, l.ax[1], st);
    }
    if (e == hipSuccess) e = fft_pass(kPassPoissonZ, jobs, njobs, l.ax[2], st);
    if (e == hipSuccess && planes)
        hipLaunchKernelGGL((k_fft_planes<false, false>), g, b, (unsigned)l.lds, st, jobs, FftStep{});
    else {
        if (e == hipSuccess) e = fft_pass(kPassHc2rY, jobs, njobs, l.ax[1], st);
        if (e == hipSuccess) e = fft_pass(kPassHc2rXScaled, jobs, njobs, l.ax[0], st);
    }
    return e == hipSuccess ? hipGetLastError() : e;
}

hipError_t fft_pass(FftPass pass, const FftJob *jobs, int njobs, const FftLaunch &l,
                    hipStream_t st)
{
    switch (pass) {
    case kPassR2hcXFromSrc: return launch_pass<kFftR2HC, 0, true, false>(jobs, njobs, l, st);
    case kPassR2hcX: return launch_pass<kFftR2HC, 0, false, false>(jobs, njobs, l, st);
    case kPassR2hcY: return launch_pass<kFftR2HC, 1, false, false>(jobs, njobs, l, st);
    case kPassR2hcZ: return launch_pass<kFftR2HC, 2, false, false>(jobs, njobs, l, st);
    case kPassPoissonZ: return launch_pass<kFftPoisson, 2, false, false>(jobs, njobs, l, st);
    case kPassHc2rZ: return launch_pass<kFftHC2R, 2, false, false>(jobs, njobs, l, st);
    case kPassHc2rY: return launch_pass<kFftHC2R, 1, false, false>(jobs, njobs, l, st);
    case kPassHc2rXScaled: return launch_pass<kFftHC2R, 0, false, true>(jobs, njobs, l, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace ohpic
