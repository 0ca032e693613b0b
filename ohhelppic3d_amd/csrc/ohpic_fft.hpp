// ohpic_fft.hpp -- axis-pass FFT launchers (FFTW R2HC/HC2R semantics) and
// the per-length plan (radix factors + twiddle table in device memory).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace ohpic {

constexpr int kMaxRadix = 13;   // largest prime factor an axis length may have
constexpr int kMaxFactors = 24;
#ifndef OHPIC_FFT_BLOCK
#define OHPIC_FFT_BLOCK 256
#endif
constexpr int kFftBlock = OHPIC_FFT_BLOCK;  // threads per FFT workgroup
// 1024 complex values (16 KiB) per workgroup: ten workgroups fit a CU's LDS
// and the passes run at 8 waves per SIMD (34-46 VGPRs); measured 28% faster
// per pass at 256^3 than 32 KiB at 4 waves.  Axis lengths up to 1024.
#ifndef OHPIC_FFT_LDS_CPLX
#define OHPIC_FFT_LDS_CPLX 1024
#endif
constexpr int kFftLdsCplx = OHPIC_FFT_LDS_CPLX;  // complex values per workgroup (16 B each)
constexpr int kMaxFftLen = kFftLdsCplx;  // one complex line must fit a workgroup's LDS

enum FftKind : int { kFftR2HC = 0, kFftHC2R = 1, kFftPoisson = 2 };

// q = t / d for 0 <= t < 2^16 and 1 <= d <= 2^16 as one high multiply by
// m = ceil(2^32 / d) (m = 0 encodes d = 1): with t = q d + r, t m / 2^32 =
// q + r/d + t e/(d 2^32) where m d = 2^32 + e, e < d, and t d < 2^32 keeps the
// last term below 1/d, so the floor is exact.
__host__ __device__ inline uint32_t fastdiv_magic(uint32_t d)
{
    return d <= 1 ? 0u : (uint32_t)((0x100000000ull + d - 1) / d);
}

struct InstDev;

struct FftAxisDev {
    int n;
    int nfac;
    int fac[kMaxFactors];
    const double2 *tw;  // tw[k] = exp(-2 pi i k / n), k in [0, n)
    // divisors of the LDS passes as fastdiv multipliers (fft_plan_divisors)
    uint32_t mg_n;                 // n
    uint32_t mg_G;                 // fft_group_lines(n)
    uint32_t mg_half;              // n / 2 + 1
    uint32_t mg_nl;                // fft_group_lines(n) / 2: line pairs per group
    uint32_t mg_tpl[kMaxFactors];  // n / fac[s]: butterflies per line in stage s
    uint32_t mg_Ls[kMaxFactors];   // fac[0] * ... * fac[s-1]
    int A, B;                      // n = A B of the two-step form, or 0
    int ab_lines;                  // its complex lines per workgroup
    uint32_t mg_M;                 // max(A, B)
};

// n = A B with 2 <= A <= B <= 16 as close as possible (the two-step register
// form), or A = B = 0.  Every length up to 256 of a grid that is not a prime
// and has such factors takes it; the others run the LDS stages.
void fft_two_step(int n, int *A, int *B);
int64_t fft_two_step_lds(int A, int B);  // its LDS bytes per workgroup

// Workgroups of one axis pass over a table of jobs: largest counts over the
// jobs of each form (0: no job of it).
struct FftLaunch {
    int64_t groups = 0;     // LDS stages
    int rs = 0;             // their radix set
    int64_t groups16 = 0;   // two-step form, 16 x 16
    int64_t groups_ab = 0;  // two-step form, other A x B
    int64_t lds_ab = 0;     // its largest LDS bytes
};

// Factorises n (radix 4 first, then 2, 3, 5, ...); false if a prime factor
// exceeds kMaxRadix or n is out of range.
bool fft_factorize(int n, int *fac, int *nfac);

// Fills the fastdiv multipliers of a factorised axis plan.
void fft_plan_divisors(FftAxisDev &ax);

// Host-side twiddle table exp(-2 pi i k/n) in long double, rounded to double.
void fft_twiddles(int n, double2 *tw);

// real lines per workgroup: G/2 complex lines of n fill at most kFftLdsCplx
// complex values (32 KiB); at least 2 lines, at most 64
__host__ __device__ inline int fft_group_lines(int n)
{
    int g = 2 * (kFftLdsCplx / (n > 0 ? n : 1));
    if (g > 64) g = 64;
    if (g < 2) g = 2;
    return g & ~1;
}

// workgroups of one axis pass (G real lines each)
__host__ __device__ inline int64_t fft_groups(int axis, int G, int nx, int ny, int nz)
{
    if (axis == 0) return ((int64_t)ny * nz + G - 1) / G;
    if (axis == 1) return (int64_t)((nx + G - 1) / G) * nz;
    return ((int64_t)nx * ny + G - 1) / G;
}

// One transform job: an nx*ny*nz array with its per-axis plans and (for the
// Poisson pass) the Green's-function denominators per axis.
struct FftJob {
    const double *src;     // source of the first Poisson pass (rho)
    double *data;          // array transformed in place (phi)
    int n[3];
    FftAxisDev ax[3];
    const double *lam[3];  // (2 sin(pi k/n))^2 per axis
    double inv_n;          // 1 / (nx ny nz)
    int plane;             // wavefronts per plane when the x and y passes can go
                           // by planes (fft_plan_planes), or 0
};

// Launches of a Poisson solve over a table of jobs.
struct FftSolve {
    FftLaunch ax[3];          // the axis passes
    bool all_planes = true;   // every job's x and y passes can go by planes:
    int planes = 0;           // most planes of a job,
    int64_t total_planes = 0; // planes of all jobs,
    int plane_waves = 0;      // most wavefronts and LDS bytes
    int64_t lds = 0;
};

// Start of a step whose x and y passes go by planes: rho comes from the charge
// grids of insts[job], and what launch_begin_step_b does is done on the way.
struct FftStep {
    const InstDev *insts;
    const int *parity;
    unsigned int *queue;
};

enum FftPass : int {
    kPassR2hcXFromSrc = 0,  // R2HC along x, src -> data
    kPassR2hcX,             // R2HC along x in place
    kPassR2hcY,
    kPassR2hcZ,
    kPassPoissonZ,          // R2HC z, divide by lam sum (DC := 0), HC2R z
    kPassHc2rZ,
    kPassHc2rY,
    kPassHc2rXScaled        // HC2R along x, times inv_n
};

int fft_radix_set(const FftAxisDev &ax);

// Adds a job's axis to the launch of that axis' passes.
void fft_add(FftLaunch &l, const FftAxisDev &ax, int axis, int nx, int ny, int nz, int plane = 0);

// One axis pass for every job of the device table `jobs`.  Each job's form
// depends on its axis length alone, so it computes the same in every table.
hipError_t fft_pass(FftPass pass, const FftJob *jobs, int njobs, const FftLaunch &l,
                    hipStream_t st);

// Sets J.plane from J.n and J.ax.
void fft_plan_planes(FftJob &J);

// Adds a job to a solve's launches.
void fft_solve_add(FftSolve &l, const FftJob &J);

// The solve's x and y passes go by planes.
bool fft_by_planes(const FftSolve &l);

// Forward x and y from src to data, the fused Poisson z pass, inverse y and x.
// step (only when fft_by_planes): start the step too and take rho from there.
hipError_t fft_poisson(const FftJob *jobs, int njobs, const FftSolve &l, const FftStep *step,
                       hipStream_t st);

}  // namespace ohpic
