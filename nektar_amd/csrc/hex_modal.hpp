// Fused hex Helmholtz operator on affine elements, in Legendre space, for
// gfx950 (Helmholtz.h:549-599, HelmholtzKernels.hpp:389-696).
//
// With one Jacobian and metric per element nothing in the operator depends
// on the point, so the quadrature sums can be taken once, in 1-D.  A mode of
// the Modified_A basis has few Legendre coefficients,
//   phi_0, phi_1 = (P_0 -+ P_1) / 2
//   phi_p        = a_p (P_{p-2} - P_p),  a_p = (p - 1) / (2 (2p - 1)),  p >= 2
// and its derivative only one,
//   phi_0', phi_1' = -+ P_0 / 2,  phi_p' = -(p - 1)/2 P_{p-1},
// while GLL quadrature with Q >= NM points makes the Legendre polynomials up
// to degree NM - 1 orthogonal, P_n having the discrete norm g_n = 2/(2n + 1)
// (2/(Q - 1) at n = Q - 1).  So B^T W B, D^T W D and the mixed products that
// the reference sums over the points are S^T G S, R^T G R, S^T G R with S
// (values) and R (derivatives) the two-banded maps above and G = diag(g_n):
// the same numbers up to rounding, at 2 and 0 products per value instead of
// NQ.  The functions are scaled, psi_n = s_n P_n with s_0 = 1, s_n = -n/2, so
// that the derivative of an interior mode has the coefficient 1.
//
// Work decomposition: NM*NM work-items per element, one per 1-D line; the
// three directions exchange lines through three LDS slabs per element, every
// pass in place on lines of one work-item (one barrier per pass):
//   along p: S, R           -> 2 slabs
//   along q: S S, S R, R S  -> 3 slabs
//   along r: u, d0, d1, d2 in registers, the metric, and the transposes back.
// About 40 operations per coefficient against 183 with the contractions over
// NQ points, and 20 LDS accesses against 33: bound by LDS (its pipe is busy
// 84 % of the cycles at NM = 7, a quarter of it bank conflicts), then HBM.
// Measured against the contractions over the points: 32,768 elements at NM = 7,
// NQ = 8, FP64 90.4 -> 52.5 us (3.5 TB/s of the coefficients and geometry),
// 50,021 elements at NM = 4, NQ = 6, FP32 29.3 -> 8.3 us.  Rounding error
// against extended precision 1.8e-16 at NM = 3, 5, 7 and 10 (relative, 2-norm),
// the sums over the points 5.6, 5.3, 6.7 and 33e-16.
#pragma once

#include <hip/hip_runtime.h>

#include "hex_kernels.hpp"

namespace nektar_amd {
namespace hexmodal {

// Coefficients of the 1-D maps; every argument is a constant after unrolling.
template <int NM, int NQ>
struct Map {
    static constexpr double a(int p) { return (p - 1) / (2.0 * (2 * p - 1)); }
    static constexpr double s(int n) { return n == 0 ? 1.0 : -0.5 * n; }
    // norm of psi_n under the NQ-point GLL rule
    static constexpr double g(int n) { return (n == NQ - 1 ? 2.0 / (NQ - 1) : 2.0 / (2 * n + 1)) * s(n) * s(n); }
    // coefficient of psi_n in modes n and n + 2
    static constexpr double lo(int n) { return -a(n) / s(n); }
    static constexpr double hi(int n) { return a(n + 2) / s(n); }
};

// u = S x: the values' coefficients in psi_n
template <int NM, int NQ, typename T>
__device__ __forceinline__ void values(const T (&x)[NM], T (&u)[NM])
{
    using M = Map<NM, NQ>;
    u[0] = T(0.5) * (x[0] + x[1]);
    if constexpr (NM > 2) u[0] = fma(T(M::hi(0)), x[2], u[0]);
    u[1] = x[0] - x[1];
    if constexpr (NM > 3) u[1] = fma(T(M::hi(1)), x[3], u[1]);
#pragma unroll
    for (int n = 2; n < NM; ++n) {
        u[n] = T(M::lo(n)) * x[n];
        if (n + 2 < NM) u[n] = fma(T(M::hi(n)), x[n + 2], u[n]);
    }
}

// d = R x: the derivative's (the last one is zero)
template <int NM, typename T>
__device__ __forceinline__ void derivs(const T (&x)[NM], T (&d)[NM])
{
    d[0] = T(0.5) * (x[1] - x[0]);
#pragma unroll
    for (int n = 1; n + 1 < NM; ++n) d[n] = x[n + 1];
    d[NM - 1] = T(0);
}

// y = S^T G v (+ R^T G w with DERIV): back to the modes, with the norms
template <int NM, int NQ, bool DERIV, typename T>
__device__ __forceinline__ void transposed(const T (&v)[NM], const T (&w)[NM], T (&y)[NM])
{
    using M = Map<NM, NQ>;
    const T v0 = T(0.5 * M::g(0)) * v[0];
    const T w0 = DERIV ? T(0.5 * M::g(0)) * w[0] : T(0);
    y[0] = fma(T(M::g(1)), v[1], DERIV ? v0 - w0 : v0);
    y[1] = fma(T(-M::g(1)), v[1], DERIV ? v0 + w0 : v0);
#pragma unroll
    for (int p = 2; p < NM; ++p) {
        y[p] = T(M::lo(p) * M::g(p)) * v[p];
        y[p] = fma(T(M::hi(p - 2) * M::g(p - 2)), v[p - 2], y[p]);
        if (DERIV) y[p] = fma(T(M::g(p - 1)), w[p - 1], y[p]);
    }
}

// LDS strides of a slab, value (p, q, r) at p + q*Q + r*R.  The three passes
// walk lines along p, q and r; a 64-lane access is served in groups of 128
// bytes (16 doubles), and the strides are those whose groups meet the fewest
// equal banks over the accesses of all passes (NM = 7, FP64: 1.36 cycles per
// group against 1.71 unpadded and 13 % of the slab for it).
template <typename T, int NM>
struct Strides {
    static constexpr bool D = sizeof(T) == 8;
    static constexpr int Q = NM == 6 ? (D ? 9 : 7) : NM == 10 ? (D ? 10 : 11) : NM % 2 == 0 ? NM + 1 : NM;
    static constexpr int PAD = D ? (NM == 3 ? 3 : NM == 5 ? 4 : NM == 7 ? 6 : NM == 9 ? 8 : NM == 10 ? 6 : 0)
                                 : (NM == 5 ? 1 : NM == 7 ? 3 : NM == 9 ? 8 : 0);
    static constexpr int R = NM * Q + PAD, SLAB = NM * R;
};

// Results go out line by line from the registers, except in FP64 from NM = 9
// on, through LDS so that a wave's stores are contiguous (NM = 9: 54 against
// 61 us; NM = 4: 44 against 41, FP32 NM = 8: 26 against 23).
template <typename T, int NM>
constexpr bool kStaged = sizeof(T) == 8 && NM >= 9;

// One element: work-item t of NM*NM, L its three slabs, g its 7 geometry
// values {J m_00, 01, 02, 11, 12, 22, J}.  DOT: *edot = x . y of the element,
// its lines' sums added in the order of their indices.
template <typename T, int NM, int NQ, bool DOT = false, typename Fetch>
__device__ __forceinline__ void element(const Fetch &fetch, bool valid, int t, const T *__restrict__ g, T lambda,
                                        T *L, T *__restrict__ xout, double *__restrict__ edot = nullptr)
{
    using S = Strides<T, NM>;
    constexpr int Q = S::Q, R = S::R, SL = S::SLAB;
    const int a = t % NM, b = t / NM;
    T *row = L + b * R + a * Q;  // line along direction 0: (q, r) = (a, b)
    T *mid = L + b * R + a;      // along direction 1: (n0, r) = (a, b)
    T *col = L + b * Q + a;      // along direction 2: (n0, n1) = (a, b)
    T xl[NM];  // this work-item's line of the input
    {
        T(&x)[NM] = xl;
        T u[NM], d[NM];
        if constexpr (hex::HasLine<Fetch>::value) {
            if (valid) {
                fetch.line(a, b, x);
            } else {
#pragma unroll
                for (int p = 0; p < NM; ++p) x[p] = T(0);
            }
        } else {
#pragma unroll
            for (int p = 0; p < NM; ++p) x[p] = valid ? fetch(p, a, b) : T(0);
        }
        values<NM, NQ>(x, u);
        derivs(x, d);
#pragma unroll
        for (int p = 0; p < NM; ++p) row[p] = u[p];
#pragma unroll
        for (int p = 0; p < NM; ++p) row[SL + p] = d[p];
    }
    __syncthreads();
    {
        T x[NM], u[NM], d[NM];
#pragma unroll
        for (int q = 0; q < NM; ++q) x[q] = mid[q * Q];
        values<NM, NQ>(x, u);
        derivs(x, d);
#pragma unroll
        for (int q = 0; q < NM; ++q) mid[q * Q] = u[q];
#pragma unroll
        for (int q = 0; q < NM; ++q) mid[2 * SL + q * Q] = d[q];
#pragma unroll
        for (int q = 0; q < NM; ++q) x[q] = mid[SL + q * Q];
        values<NM, NQ>(x, u);
#pragma unroll
        for (int q = 0; q < NM; ++q) mid[SL + q * Q] = u[q];
    }
    T gm[7];
#pragma unroll
    for (int c = 0; c < 7; ++c) gm[c] = valid ? g[c] : T(0);
    __syncthreads();
    {
        T x[NM], u[NM], d0[NM], d1[NM], d2[NM];
#pragma unroll
        for (int r = 0; r < NM; ++r) x[r] = col[r * R];
        values<NM, NQ>(x, u);
        derivs(x, d2);
#pragma unroll
        for (int r = 0; r < NM; ++r) x[r] = col[SL + r * R];
        values<NM, NQ>(x, d0);
#pragma unroll
        for (int r = 0; r < NM; ++r) x[r] = col[2 * SL + r * R];
        values<NM, NQ>(x, d1);
        const T lj = lambda * gm[6];
#pragma unroll
        for (int r = 0; r < NM; ++r) {
            const T e0 = d0[r], e1 = d1[r], e2 = d2[r];
            d0[r] = fma(gm[2], e2, fma(gm[1], e1, gm[0] * e0));
            d1[r] = fma(gm[4], e2, fma(gm[3], e1, gm[1] * e0));
            d2[r] = fma(gm[5], e2, fma(gm[4], e1, gm[2] * e0));
            u[r] *= lj;
        }
        T y[NM];
        transposed<NM, NQ, true>(u, d2, y);
#pragma unroll
        for (int r = 0; r < NM; ++r) col[r * R] = y[r];
        transposed<NM, NQ, false>(d0, d0, y);
#pragma unroll
        for (int r = 0; r < NM; ++r) col[SL + r * R] = y[r];
        transposed<NM, NQ, false>(d1, d1, y);
#pragma unroll
        for (int r = 0; r < NM; ++r) col[2 * SL + r * R] = y[r];
    }
    __syncthreads();
    {
        T v[NM], w[NM], y[NM];
#pragma unroll
        for (int q = 0; q < NM; ++q) v[q] = mid[q * Q];
#pragma unroll
        for (int q = 0; q < NM; ++q) w[q] = mid[2 * SL + q * Q];
        transposed<NM, NQ, true>(v, w, y);
#pragma unroll
        for (int q = 0; q < NM; ++q) mid[q * Q] = y[q];
#pragma unroll
        for (int q = 0; q < NM; ++q) v[q] = mid[SL + q * Q];
        transposed<NM, NQ, false>(v, v, y);
#pragma unroll
        for (int q = 0; q < NM; ++q) mid[SL + q * Q] = y[q];
    }
    __syncthreads();
    {
        T v[NM], w[NM], y[NM];
#pragma unroll
        for (int p = 0; p < NM; ++p) v[p] = row[p];
#pragma unroll
        for (int p = 0; p < NM; ++p) w[p] = row[SL + p];
        transposed<NM, NQ, true>(v, w, y);
        if constexpr (DOT) {
            double s = 0.0;
#pragma unroll
            for (int p = 0; p < NM; ++p) s = fma((double)xl[p], (double)y[p], s);
            row[SL] = T(s);
        }
        if constexpr (kStaged<T, NM>) {
#pragma unroll
            for (int p = 0; p < NM; ++p) row[p] = y[p];
        } else if (valid) {
#pragma unroll
            for (int p = 0; p < NM; ++p) xout[t * NM + p] = y[p];
        }
    }
    if constexpr (kStaged<T, NM> || DOT) __syncthreads();
    if constexpr (kStaged<T, NM>) {
        if (valid) {
#pragma unroll
            for (int r = 0; r < NM; ++r) xout[r * NM * NM + t] = col[r * R];
        }
    }
    if constexpr (DOT) {
        if (t < NM) {
            double s = 0.0;
#pragma unroll
            for (int r = 0; r < NM; ++r) s += (double)L[SL + r * R + t * Q];
            L[SL + t * Q] = T(s);
        }
        __syncthreads();
        if (t == 0 && valid) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < NM; ++q) s += (double)L[SL + q * Q];
            *edot = s;
        }
    }
}

// E elements per workgroup of E*NM*NM work-items
template <typename T, int NM, int E>
constexpr bool fits()
{
    return E * NM * NM <= 1024 && E * 3 * Strides<T, NM>::SLAB * (int)sizeof(T) <= 65536;
}

// Collections form: element-local coefficients
template <typename T, int NM, int NQ, int E>
__global__ __launch_bounds__(E * NM * NM) void helmholtz_kernel(int nelmt, const T *__restrict__ geo, T lambda,
                                                                const T *__restrict__ in, T *__restrict__ out)
{
    constexpr int TPE = NM * NM, NC = NM * NM * NM;
    __shared__ T lds[E][3 * Strides<T, NM>::SLAB];
    const int le = threadIdx.x / TPE, t = threadIdx.x % TPE;
    const int e = blockIdx.x * E + le;
    const bool valid = e < nelmt;
    element<T, NM, NQ>(hex::LocalFetch<T, NM>{in + (size_t)e * NC}, valid, t, geo + (size_t)e * 7, lambda, lds[le],
                       out + (size_t)e * NC);
}

// General solver form: coefficients through the signed local-to-global map
template <typename T, int NM, int NQ, int E>
__global__ __launch_bounds__(E * NM * NM) void helmholtz_mapped_kernel(int nelmt, const T *__restrict__ geo, T lambda,
                                                                       const T *__restrict__ xg,
                                                                       const int *__restrict__ menc,
                                                                       T *__restrict__ out)
{
    constexpr int TPE = NM * NM, NC = NM * NM * NM;
    __shared__ T lds[E][3 * Strides<T, NM>::SLAB];
    const int le = threadIdx.x / TPE, t = threadIdx.x % TPE;
    const int e = blockIdx.x * E + le;
    const bool valid = e < nelmt;
    const hex::MappedFetch<T, NM> f{xg, menc + (size_t)(valid ? e : 0) * NC};
    element<T, NM, NQ>(f, valid, t, geo + (size_t)e * 7, lambda, lds[le], out + (size_t)e * NC);
}

// Grouped form: several operators of one kind; block b belongs to the item
// whose [block0, next block0) range holds it
template <typename T, int NM, int NQ, int E>
__global__ __launch_bounds__(E * NM * NM) void helmholtz_grouped_kernel(int count,
                                                                        const GroupItem<T> *__restrict__ items)
{
    constexpr int TPE = NM * NM, NC = NM * NM * NM;
    __shared__ T lds[E][3 * Strides<T, NM>::SLAB];
    const int blk = blockIdx.x;
    int it = 0;
    while (it + 1 < count && blk >= items[it + 1].block0) ++it;
    const GroupItem<T> I = items[it];
    const int le = threadIdx.x / TPE, t = threadIdx.x % TPE;
    const int e = (blk - I.block0) * E + le;
    const bool valid = e < I.nelmt;
    element<T, NM, NQ>(hex::LocalFetch<T, NM>{I.in + (size_t)e * NC}, valid, t, I.geo + (size_t)e * 7, I.lambda,
                       lds[le], I.out + (size_t)e * NC);
}

// Structured solver form: coefficients gathered from the global C0 vector
// of the n^3 box; FP64: edot[e] = x_e . y_e, whose sum is the CG's s . w
template <typename T, int NM, int NQ, int E>
__global__ __launch_bounds__(E * NM * NM) void helmholtz_gather_kernel(int n, int N, const T *__restrict__ geo,
                                                                       T lambda, const T *__restrict__ xg,
                                                                       T *__restrict__ out,
                                                                       const int *__restrict__ done,
                                                                       double *__restrict__ edot)
{
    if (done && *done) return;
    constexpr int TPE = NM * NM, NC = NM * NM * NM;
    __shared__ T lds[E][3 * Strides<T, NM>::SLAB];
    const int le = threadIdx.x / TPE, t = threadIdx.x % TPE;
    const int nelmt = n * n * n;
    const int e = xcd_work(blockIdx.x, (nelmt + E - 1) / E) * E + le;
    const bool valid = e < nelmt;
    const int ex = e % n, ey = (e / n) % n, ez = e / (n * n);
    const hex::StructuredFetch<T, NM> f{xg, N, ex * (NM - 1), ey * (NM - 1), ez * (NM - 1)};
    if constexpr (sizeof(T) == 8)
        element<T, NM, NQ, true>(f, valid, t, geo + (size_t)e * 7, lambda, lds[le], out + (size_t)e * NC, edot + e);
    else
        element<T, NM, NQ>(f, valid, t, geo + (size_t)e * 7, lambda, lds[le], out + (size_t)e * NC);
}

}  // namespace hexmodal
}  // namespace nektar_amd
