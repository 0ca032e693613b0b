// ohpic_dft.hpp -- complex DFTs of 2 to 16 points in registers.
#pragma once

#include <hip/hip_runtime.h>

// Products and sums contract within one statement only, so that the same code
// rounds the same in every kernel it is part of (an instance's transform may
// run in either of two kernels, alone or in a group).
#pragma clang fp contract(on)

namespace ohpic {
namespace {

struct cplx {
    double re, im;
};

__device__ __forceinline__ cplx cmul(cplx a, cplx b)
{
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

// cos and sin of 2 pi k / P in row P
__device__ constexpr double kCos[17][16] = {
        {0},
        {1},
        {1, -1},
        {1, -0.5, -0.5},
        {1, 0, -1, 0},
        {1, 0.30901699437494745, -0.8090169943749475, -0.8090169943749475, 0.30901699437494745},
        {1, 0.5, -0.5, -1, -0.5, 0.5},
        {1, 0.6234898018587335, -0.2225209339563144, -0.9009688679024191, -0.9009688679024191,
     -0.2225209339563144, 0.6234898018587335},
        {1, 0.7071067811865476, 0, -0.7071067811865476, -1, -0.7071067811865476, 0,
     0.7071067811865476},
        {1, 0.766044443118978, 0.17364817766693036, -0.5, -0.9396926207859084,
     -0.9396926207859084, -0.5, 0.17364817766693036, 0.766044443118978},
        {1, 0.8090169943749475, 0.30901699437494745, -0.30901699437494745, -0.8090169943749475,
     -1, -0.8090169943749475, -0.30901699437494745, 0.30901699437494745, 0.8090169943749475},
        {1, 0.8412535328311812, 0.41541501300188644, -0.14231483827328514, -0.6548607339452851,
     -0.9594929736144974, -0.9594929736144974, -0.6548607339452851, -0.14231483827328514,
     0.41541501300188644, 0.8412535328311812},
        {1, 0.8660254037844386, 0.5, 0, -0.5, -0.8660254037844386, -1, -0.8660254037844386,
     -0.5, 0, 0.5, 0.8660254037844386},
        {1, 0.8854560256532099, 0.5680647467311558, 0.12053668025532305, -0.3546048870425356,
     -0.7485107481711011, -0.970941817426052, -0.970941817426052, -0.7485107481711011,
     -0.3546048870425356, 0.12053668025532305, 0.5680647467311558, 0.8854560256532099},
        {1, 0.9009688679024191, 0.6234898018587335, 0.2225209339563144, -0.2225209339563144,
     -0.6234898018587335, -0.9009688679024191, -1, -0.9009688679024191, -0.6234898018587335,
     -0.2225209339563144, 0.2225209339563144, 0.6234898018587335, 0.9009688679024191},
        {1, 0.9135454576426009, 0.6691306063588582, 0.30901699437494745, -0.10452846326765347,
     -0.5, -0.8090169943749475, -0.9781476007338057, -0.9781476007338057, -0.8090169943749475,
     -0.5, -0.10452846326765347, 0.30901699437494745, 0.6691306063588582, 0.9135454576426009},
        {1, 0.9238795325112867, 0.7071067811865476, 0.3826834323650898, 0, -0.3826834323650898,
     -0.7071067811865476, -0.9238795325112867, -1, -0.9238795325112867, -0.7071067811865476,
     -0.3826834323650898, 0, 0.3826834323650898, 0.7071067811865476, 0.9238795325112867},
};
__device__ constexpr double kSin[17][16] = {
        {0},
        {0},
        {0, 0},
        {0, 0.8660254037844386, -0.8660254037844386},
        {0, 1, 0, -1},
        {0, 0.9510565162951535, 0.5877852522924731, -0.5877852522924731, -0.9510565162951535},
        {0, 0.8660254037844386, 0.8660254037844386, 0, -0.8660254037844386,
     -0.8660254037844386},
        {0, 0.7818314824680298, 0.9749279121818236, 0.4338837391175581, -0.4338837391175581,
     -0.9749279121818236, -0.7818314824680298},
        {0, 0.7071067811865476, 1, 0.7071067811865476, 0, -0.7071067811865476, -1,
     -0.7071067811865476},
        {0, 0.6427876096865394, 0.984807753012208, 0.8660254037844386, 0.3420201433256687,
     -0.3420201433256687, -0.8660254037844386, -0.984807753012208, -0.6427876096865394},
        {0, 0.5877852522924731, 0.9510565162951535, 0.9510565162951535, 0.5877852522924731, 0,
     -0.5877852522924731, -0.9510565162951535, -0.9510565162951535, -0.5877852522924731},
        {0, 0.5406408174555976, 0.9096319953545183, 0.9898214418809327, 0.7557495743542583,
     0.28173255684142967, -0.28173255684142967, -0.7557495743542583, -0.9898214418809327,
     -0.9096319953545183, -0.5406408174555976},
        {0, 0.5, 0.8660254037844386, 1, 0.8660254037844386, 0.5, 0, -0.5, -0.8660254037844386,
     -1, -0.8660254037844386, -0.5},
        {0, 0.46472317204376856, 0.8229838658936564, 0.992708874098054, 0.9350162426854148,
     0.6631226582407952, 0.23931566428755777, -0.23931566428755777, -0.6631226582407952,
     -0.9350162426854148, -0.992708874098054, -0.8229838658936564, -0.46472317204376856},
        {0, 0.4338837391175581, 0.7818314824680298, 0.9749279121818236, 0.9749279121818236,
     0.7818314824680298, 0.4338837391175581, 0, -0.4338837391175581, -0.7818314824680298,
     -0.9749279121818236, -0.9749279121818236, -0.7818314824680298, -0.4338837391175581},
        {0, 0.4067366430758002, 0.7431448254773942, 0.9510565162951535, 0.9945218953682733,
     0.8660254037844386, 0.5877852522924731, 0.20791169081775934, -0.20791169081775934,
     -0.5877852522924731, -0.8660254037844386, -0.9945218953682733, -0.9510565162951535,
     -0.7431448254773942, -0.4067366430758002},
        {0, 0.3826834323650898, 0.7071067811865476, 0.9238795325112867, 1, 0.9238795325112867,
     0.7071067811865476, 0.3826834323650898, 0, -0.3826834323650898, -0.7071067811865476,
     -0.9238795325112867, -1, -0.9238795325112867, -0.7071067811865476, -0.3826834323650898},
};

// v * exp(SIGN 2 pi i K / P)
template <int SIGN, int P, int K>
__device__ __forceinline__ cplx twist(cplx v)
{
    constexpr int k = K % P;
    constexpr double c = kCos[P][k], s = SIGN < 0 ? -kSin[P][k] : kSin[P][k];
    if constexpr (k == 0)
        return v;
    else if constexpr (c == 0.0)
        return s > 0.0 ? cplx{-v.im, v.re} : cplx{v.im, -v.re};
    else if constexpr (s == 0.0)
        return cplx{-v.re, -v.im};
    else
        return cmul(v, cplx{c, s});
}

template <int SIGN, int P>
struct Dft;

template <int SIGN>
struct Dft<SIGN, 1> {
    static __device__ __forceinline__ void run(cplx *) {}
};

template <int SIGN>
struct Dft<SIGN, 2> {
    static __device__ __forceinline__ void run(cplx *a)
    {
        const cplx t = a[1];
        a[1] = {a[0].re - t.re, a[0].im - t.im};
        a[0] = {a[0].re + t.re, a[0].im + t.im};
    }
};

template <int SIGN>
struct Dft<SIGN, 4> {
    static __device__ __forceinline__ void run(cplx *a)
    {
        const cplx t0 = {a[0].re + a[2].re, a[0].im + a[2].im};
        const cplx t1 = {a[0].re - a[2].re, a[0].im - a[2].im};
        const cplx t2 = {a[1].re + a[3].re, a[1].im + a[3].im};
        const cplx t3 = {a[1].re - a[3].re, a[1].im - a[3].im};
        const cplx wt3 = {-SIGN * t3.im, SIGN * t3.re};  // (SIGN i) * t3
        a[0] = {t0.re + t2.re, t0.im + t2.im};
        a[1] = {t1.re + wt3.re, t1.im + wt3.im};
        a[2] = {t0.re - t2.re, t0.im - t2.im};
        a[3] = {t1.re - wt3.re, t1.im - wt3.im};
    }
};

// Odd primes: with t_k = a_k + a_{P-k} and d_k = a_k - a_{P-k} (0 < k < P/2),
// outputs u and P - u are a_0 + sum cos(2 pi u k / P) t_k +- SIGN i sum
// sin(2 pi u k / P) d_k: a quarter of the products of the plain sum.
template <int SIGN, int P>
struct DftOdd {
    static __device__ __forceinline__ void run(cplx *a)
    {
        constexpr int H = (P - 1) / 2;
        cplx t[H], d[H];
#pragma unroll
        for (int k = 0; k < H; ++k) {
            const cplx x = a[k + 1], y = a[P - 1 - k];
            t[k] = {x.re + y.re, x.im + y.im};
            d[k] = {x.re - y.re, x.im - y.im};
        }
        cplx sum = a[0];
#pragma unroll
        for (int k = 0; k < H; ++k) {
            sum.re += t[k].re;
            sum.im += t[k].im;
        }
#pragma unroll
        for (int u = 1; u <= H; ++u) {
            cplx m = a[0], j = {0.0, 0.0};
#pragma unroll
            for (int k = 0; k < H; ++k) {
                const int w = u * (k + 1) % P;
                m.re += kCos[P][w] * t[k].re;
                m.im += kCos[P][w] * t[k].im;
                j.re += kSin[P][w] * d[k].re;
                j.im += kSin[P][w] * d[k].im;
            }
            a[u] = {m.re - SIGN * j.im, m.im + SIGN * j.re};
            a[P - u] = {m.re + SIGN * j.im, m.im - SIGN * j.re};
        }
        a[0] = sum;
    }
};

// P = R Q: Q transforms of R points over a[j + Q m], twiddles, R of Q points.
template <int SIGN, int R, int Q>
struct DftProduct {
    template <int J, int K>
    static __device__ __forceinline__ void twiddles(cplx (*t)[R], const cplx *v)
    {
        t[J][K] = twist<SIGN, R * Q, J * K>(v[K]);
        if constexpr (K + 1 < R) twiddles<J, K + 1>(t, v);
    }
    template <int J>
    static __device__ __forceinline__ void first(cplx (*t)[R], const cplx *a)
    {
        cplx v[R];
#pragma unroll
        for (int m = 0; m < R; ++m) v[m] = a[J + Q * m];
        Dft<SIGN, R>::run(v);
        twiddles<J, 0>(t, v);
        if constexpr (J + 1 < Q) first<J + 1>(t, a);
    }
    static __device__ __forceinline__ void run(cplx *a)
    {
        cplx t[Q][R];
        first<0>(t, a);
#pragma unroll
        for (int k = 0; k < R; ++k) {
            cplx u[Q];
#pragma unroll
            for (int j = 0; j < Q; ++j) u[j] = t[j][k];
            Dft<SIGN, Q>::run(u);
#pragma unroll
            for (int j = 0; j < Q; ++j) a[k + R * j] = u[j];
        }
    }
};

template <int SIGN>
struct Dft<SIGN, 3> : DftOdd<SIGN, 3> {};
template <int SIGN>
struct Dft<SIGN, 5> : DftOdd<SIGN, 5> {};
template <int SIGN>
struct Dft<SIGN, 7> : DftOdd<SIGN, 7> {};
template <int SIGN>
struct Dft<SIGN, 11> : DftOdd<SIGN, 11> {};
template <int SIGN>
struct Dft<SIGN, 13> : DftOdd<SIGN, 13> {};
template <int SIGN>
struct Dft<SIGN, 6> : DftProduct<SIGN, 3, 2> {};
template <int SIGN>
struct Dft<SIGN, 8> : DftProduct<SIGN, 4, 2> {};
template <int SIGN>
struct Dft<SIGN, 9> : DftProduct<SIGN, 3, 3> {};
template <int SIGN>
struct Dft<SIGN, 10> : DftProduct<SIGN, 5, 2> {};
template <int SIGN>
struct Dft<SIGN, 12> : DftProduct<SIGN, 4, 3> {};
template <int SIGN>
struct Dft<SIGN, 14> : DftProduct<SIGN, 7, 2> {};
template <int SIGN>
struct Dft<SIGN, 15> : DftProduct<SIGN, 5, 3> {};
template <int SIGN>
struct Dft<SIGN, 16> : DftProduct<SIGN, 4, 4> {};

}  // namespace
}  // namespace ohpic
