// Fused tet Helmholtz operator on affine elements, in an orthogonal polynomial
// space on the matrix cores of gfx950 (Helmholtz.h:549-599,
// HelmholtzKernels.hpp:700-913).
//
// With one Jacobian and metric per element the operator is
//   y = lambda J M x + sum_de J m_de G_d^T (G_e x),
// M the reference mass matrix and G_d the gradient of the modes in the
// orthonormal polynomials of degree NM - 2 (the metric m_de is constant, so
// it acts on the coefficients as it acts on the points).  The quadrature
// sums of the reference are exact for these products, so both give the same
// numbers up to rounding.  Two things keep the matrices small:
//  * parity: the reflection a -> -a of the first collapsed direction
//    exchanges the modes (0, ...) and (1, ...) and multiplies the others by
//    (-1)^p, so sums and differences of the exchanged pairs split the modes
//    and the polynomials into halves that do not mix; with the directions
//    d_0, d_1 - d_0/2, d_2 - d_0/2 the gradients map halves to halves;
//  * the modes are built on integrated Jacobi polynomials, so a derivative
//    reaches few polynomials: two thirds of the 16x4 blocks are zero.
//
// A wave holds 16 elements: column n = lane % 16 of every product is one
// element, and the lane group g = lane / 16 holds the entries 4s + g (s = 0,
// 1, ...) of its vectors, in registers from the load to the store.  The output
// layout of a 16x16x4 product is the input layout of the next one, so the
// vectors never leave the registers.  The matrices come as a stream of 16x4
// blocks in the order of use.
//
// Bound: the matrix cores (64 cycles a block in FP64, 32 in FP32; busy 55 % and
// 46 % of the cycles at NM = 7) and, in front and behind, the scattered
// coefficient accesses of a wave, which nothing hides.  Measured against sum
// factorisation on the vector units, 32,768 elements at NM = 7, FP64: 125.7 ->
// 27 us; 4,001 elements at NM = 10, FP32: 32.9 -> 13.6 us.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "hex_mfma_block.hpp"
#include "launch.hpp"
#include "tet_modal_layout.hpp"

namespace nektar_amd {
namespace tetmodal {

// f(integral_constant<int, i>) for i = B .. E-1
template <int B, int E, typename F>
__device__ __forceinline__ void for_range(F &&f)
{
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        for_range<B + 1, E>(static_cast<F &&>(f));
    }
}

constexpr int kWaves = 4, kBlock = 64 * kWaves;

// The blocks of the stream that one wave uses alone, positions [P0, P1) of a
// part: from global memory, DEPTH loads ahead (6 to 20 measured the same).
template <typename T, int P0, int P1>
struct OwnStream {
    static constexpr int VW = 16 / sizeof(T), DEPTH = 6;
    static_assert(P0 % VW == 0, "parts start on whole loads");
    using V = T __attribute__((ext_vector_type(VW)));
    const V *p;  // lane's values of load 0 of the stream
    V ring[DEPTH];
    static constexpr int L0 = P0 / VW, L1 = (P1 + VW - 1) / VW;
    __device__ __forceinline__ OwnStream(const T *tab, int lane) : p(reinterpret_cast<const V *>(tab) + lane)
    {
#pragma unroll
        for (int i = 0; i < DEPTH; ++i)
            if (L0 + i < L1) ring[(L0 + i) % DEPTH] = p[(L0 + i) * 64];
    }
    template <int POS>
    __device__ __forceinline__ T get()
    {
        static_assert(POS >= P0 && POS < P1, "block outside this part");
        constexpr int l = POS / VW;
        const T a = ring[l % DEPTH][POS % VW];
        if constexpr (POS % VW == VW - 1 && l + DEPTH < L1) ring[l % DEPTH] = p[(l + DEPTH) * 64];
        return a;
    }
};

// The whole stream, used by the four waves of a workgroup at the same pace:
// chunks of CL loads through two LDS buffers, the next chunk on its way to
// registers while this one is used.  (Each wave loading the stream by itself:
// the same time in FP64, 32,768 elements at NM = 10 in FP32 56 against 51 us.)
template <typename T, int NM>
struct SharedStream {
    using L = Layout<NM>;
    static constexpr int VW = 16 / sizeof(T), CL = 16, NL = L::plan.total / VW, NCH = (NL + CL - 1) / CL, RING = 3;
    using V = T __attribute__((ext_vector_type(VW)));
    using Buffer = V[CL * 64];
    static constexpr int PER = CL * 64 / kBlock;  // vectors of a chunk per work-item
    const V *src;
    Buffer *buf;
    int tid, lane;
    V next[PER], ring[RING];
    static constexpr int loads(int c) { return NL - c * CL < CL ? NL - c * CL : CL; }

    template <int c>
    __device__ __forceinline__ void fetch()
    {
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (i * kBlock < loads(c) * 64) next[i] = src[c * CL * 64 + min(i * kBlock + tid, loads(c) * 64 - 1)];
    }
    // chunk c into its buffer and the next one on its way; the buffer was
    // last read two chunks ago, before the barrier that opened chunk c - 1
    template <int c>
    __device__ __forceinline__ void open()
    {
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (i * kBlock < loads(c) * 64) buf[c % 2][i * kBlock + tid] = next[i];
        if constexpr (c + 1 < NCH) fetch<c + 1>();
        __syncthreads();
#pragma unroll
        for (int i = 0; i < RING; ++i)
            if (i < loads(c)) ring[i] = buf[c % 2][i * 64 + lane];
    }
    __device__ __forceinline__ SharedStream(const T *tab, Buffer *b)
        : src(reinterpret_cast<const V *>(tab)), buf(b), tid(threadIdx.x), lane(threadIdx.x % 64)
    {
        fetch<0>();
    }
    template <int POS>
    __device__ __forceinline__ T get()
    {
        constexpr int l = POS / VW, c = l / CL, prev = L::previous(POS), lp = prev < 0 ? -1 : prev / VW;
        if constexpr (prev < 0 || lp / CL != c) {
            open<c>();
        } else if constexpr (lp != l) {
            // loads lp .. l - 1 are done with (l - lp > 1: padding)
#pragma unroll
            for (int i = lp; i < l; ++i)
                if (i % CL + RING < loads(c)) ring[(i % CL) % RING] = buf[c % 2][(i % CL + RING) * 64 + lane];
        }
        return ring[(l % CL) % RING][POS % VW];
    }
};

template <typename T, int NM>
struct Regs {
    using L = Layout<NM>;
    T xe[L::SE], xo[L::SO];
    typename hexmf::Mma<T>::v4 ye[L::TE], yo[L::TO];
};

// Entry s of a parity's vector
template <bool ODD, int s, typename T, int NM>
__device__ __forceinline__ T entry(const Regs<T, NM> &R)
{
    if constexpr (ODD) return R.xo[s];
    else return R.xe[s];
}
// Its output tile t
template <bool ODD, int t, typename T, int NM>
__device__ __forceinline__ typename hexmf::Mma<T>::v4 &tile(Regs<T, NM> &R)
{
    if constexpr (ODD) return R.yo[t];
    else return R.ye[t];
}

// Coefficient index of entry i of a parity's vector (PARTNER: of the other
// one of its pair), -1 where there is none
template <int NM>
constexpr int column_of(bool odd, bool partner, int i)
{
    using L = Layout<NM>;
    return i >= L::ncols(odd) ? -1 : partner ? L::cols(odd)[i].b : L::cols(odd)[i].a;
}
// of entry 4s + g: constants chosen by lane group, without a table read
template <int NM, bool ODD, bool PARTNER, int s>
__device__ __forceinline__ int column_index(int g)
{
    constexpr int o0 = column_of<NM>(ODD, PARTNER, 4 * s), o1 = column_of<NM>(ODD, PARTNER, 4 * s + 1);
    constexpr int o2 = column_of<NM>(ODD, PARTNER, 4 * s + 2), o3 = column_of<NM>(ODD, PARTNER, 4 * s + 3);
    // mostly four neighbours
    if constexpr (o0 >= 0 && o1 == o0 + 1 && o2 == o0 + 2 && o3 == o0 + 3) return o0 + g;
    int i = o0;
    i = g == 1 ? o1 : i;
    i = g == 2 ? o2 : i;
    return g == 3 ? o3 : i;
}
// its coefficient, 0 where there is none; no branch, so that the loads of all
// entries are in flight together
template <int NM, bool ODD, bool PARTNER, int s, typename T>
__device__ __forceinline__ T load_entry(const T *__restrict__ x, int g)
{
    const int i = column_index<NM, ODD, PARTNER, s>(g);
    constexpr bool all = column_of<NM>(ODD, PARTNER, 4 * s) >= 0 && column_of<NM>(ODD, PARTNER, 4 * s + 1) >= 0 &&
                         column_of<NM>(ODD, PARTNER, 4 * s + 2) >= 0 && column_of<NM>(ODD, PARTNER, 4 * s + 3) >= 0;
    if constexpr (all) return x[i];
    const T v = x[max(i, 0)];
    return i < 0 ? T(0) : v;
}

// Gradient tile t of one row parity (ODD) and its way back
template <typename T, int NM, bool ODD, int t, typename S>
__device__ __forceinline__ void grad_item(Regs<T, NM> &R, S &st, const T (&m)[6])
{
    using L = Layout<NM>;
    using M = hexmf::Mma<T>;
    constexpr auto &B = L::plan.b;
    constexpr int m0 = ODD ? G0O : G0E;
    typename M::v4 g[3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int v = 0; v < 4; ++v) g[d][v] = T(0);
    // direction 0 changes the parity
    constexpr int S0 = ODD ? L::SE : L::SO, S1 = ODD ? L::SO : L::SE;
    for_range<0, (S0 > S1 ? S0 : S1)>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        if constexpr (s < S0) {
            constexpr int pos = B.fwd[m0][t][s];
            if constexpr (pos >= 0) g[0] = M::op(st.template get<pos>(), entry<!ODD, s>(R), g[0]);
        }
        if constexpr (s < S1) {
            constexpr int p1 = B.fwd[m0 + 1][t][s], p2 = B.fwd[m0 + 2][t][s];
            if constexpr (p1 >= 0) g[1] = M::op(st.template get<p1>(), entry<ODD, s>(R), g[1]);
            if constexpr (p2 >= 0) g[2] = M::op(st.template get<p2>(), entry<ODD, s>(R), g[2]);
        }
    });
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const T a0 = g[0][v], a1 = g[1][v], a2 = g[2][v];
        g[0][v] = fma(m[2], a2, fma(m[1], a1, m[0] * a0));
        g[1][v] = fma(m[4], a2, fma(m[3], a1, m[1] * a0));
        g[2][v] = fma(m[5], a2, fma(m[4], a1, m[2] * a0));
    }
    constexpr int T0 = ODD ? L::TE : L::TO, T1 = ODD ? L::TO : L::TE;
    for_range<0, 4>([&](auto vc) {
        constexpr int v = decltype(vc)::value;
        if constexpr (4 * t + v < L::MAXS) {
            for_range<0, (T0 > T1 ? T0 : T1)>([&](auto yc) {
                constexpr int y = decltype(yc)::value;
                if constexpr (y < T0) {
                    constexpr int pos = B.bwd[m0][y][4 * t + v];
                    if constexpr (pos >= 0) {
                        auto &acc = tile<!ODD, y>(R);
                        acc = M::op(st.template get<pos>(), g[0][v], acc);
                    }
                }
                if constexpr (y < T1) {
                    auto &acc = tile<ODD, y>(R);
                    constexpr int p1 = B.bwd[m0 + 1][y][4 * t + v], p2 = B.bwd[m0 + 2][y][4 * t + v];
                    if constexpr (p1 >= 0) acc = M::op(st.template get<p1>(), g[1][v], acc);
                    if constexpr (p2 >= 0) acc = M::op(st.template get<p2>(), g[2][v], acc);
                }
            });
        }
    });
}

template <typename T, int NM, bool ODD, typename S>
__device__ __forceinline__ void mass_item(Regs<T, NM> &R, S &st, T lj)
{
    using L = Layout<NM>;
    using M = hexmf::Mma<T>;
    constexpr auto &B = L::plan.b;
    for_range<0, (ODD ? L::SO : L::SE)>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        const T x = lj * entry<ODD, s>(R);
        for_range<0, (ODD ? L::TO : L::TE)>([&](auto yc) {
            constexpr int y = decltype(yc)::value, pos = B.mass[ODD][y][s];
            if constexpr (pos >= 0) {
                auto &acc = tile<ODD, y>(R);
                acc = M::op(st.template get<pos>(), x, acc);
            }
        });
    });
}

// Items order[F0 .. F1) of the plan
template <typename T, int NM, int F0, int F1, typename S>
__device__ __forceinline__ void items(Regs<T, NM> &R, S &st, const T (&m)[6], T lj)
{
    using L = Layout<NM>;
    for_range<F0, F1>([&](auto kc) {
        constexpr int it = L::plan.order[decltype(kc)::value];
        if constexpr (it < L::GE)
            grad_item<T, NM, false, it>(R, st, m);
        else if constexpr (it < L::GE + L::GO)
            grad_item<T, NM, true, it - L::GE>(R, st, m);
        else
            mass_item<T, NM, (it > L::GE + L::GO)>(R, st, lj);
    });
}

// Part w of the plan for this wave
template <typename T, int NM, int w>
__device__ __forceinline__ void part(Regs<T, NM> &R, const T *__restrict__ tab, int lane, const T (&m)[6], T lj)
{
    using L = Layout<NM>;
    if constexpr (L::plan.start[w] < L::plan.start[w + 1]) {
        OwnStream<T, L::plan.start[w], L::plan.start[w + 1]> st(tab, lane);
        items<T, NM, L::plan.first[w], L::plan.first[w + 1]>(R, st, m, lj);
    }
}

// One workgroup of four waves.  SPLIT: the waves share one tile of 16
// elements, a part of the plan each, and add their results through LDS;
// otherwise each wave has a tile of its own.
template <typename T, int NM, bool SPLIT>
__device__ __forceinline__ void helmholtz_block(int blk, int nelmt, const T *__restrict__ tab,
                                                const T *__restrict__ geo, T lambda, const T *__restrict__ in,
                                                T *__restrict__ out)
{
    using L = Layout<NM>;
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, n = lane % 16, g = lane / 16;
    const int e = (SPLIT ? blk : blk * kWaves + wave) * 16 + n;
    // lanes past the last element repeat it and store nothing
    const bool valid = e < nelmt;
    const size_t ec = valid ? e : nelmt - 1;
    const T *x = in + ec * L::NC;
    Regs<T, NM> R;
    // every load of the element is issued before the first is waited for
    T f[10];
    T xb[(L::NH + 3) / 4], xd[L::SO];
    for_range<0, L::SE>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        R.xe[s] = load_entry<NM, false, false, s>(x, g);
        if constexpr (4 * s < L::NH) xb[s] = load_entry<NM, false, true, s>(x, g);
        if constexpr (s < L::SO && 4 * s + 4 > L::NH) xd[s] = load_entry<NM, true, false, s>(x, g);
    });
#pragma unroll
    for (int c = 0; c < 10; ++c) f[c] = geo[ec * 10 + c];
    __builtin_amdgcn_sched_barrier(0);
    // sums and differences of the exchanged pairs
    for_range<0, L::SO>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        if constexpr (4 * s >= L::NH) R.xo[s] = xd[s];
        else if constexpr (4 * s + 4 <= L::NH) R.xo[s] = xb[s] - R.xe[s];
        else R.xo[s] = 4 * s + g < L::NH ? xb[s] - R.xe[s] : xd[s];
    });
    for_range<0, (L::NH + 3) / 4>([&](auto sc) { R.xe[decltype(sc)::value] += xb[decltype(sc)::value]; });
    // metric of the directions d_0, d_1 - d_0/2, d_2 - d_0/2
    T m[6], lj;
    {
#pragma unroll
        for (int c = 0; c < 6; ++c) m[c] = T(0);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const T f1 = f[3 * j + 1], f2 = f[3 * j + 2], f0 = fma(T(0.5), f1 + f2, f[3 * j]);
            m[0] = fma(f0, f0, m[0]);
            m[1] = fma(f0, f1, m[1]);
            m[2] = fma(f0, f2, m[2]);
            m[3] = fma(f1, f1, m[3]);
            m[4] = fma(f1, f2, m[4]);
            m[5] = fma(f2, f2, m[5]);
        }
#pragma unroll
        for (int c = 0; c < 6; ++c) m[c] *= f[9];
        lj = lambda * f[9];
    }
#pragma unroll
    for (int t = 0; t < L::TE; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) R.ye[t][v] = T(0);
#pragma unroll
    for (int t = 0; t < L::TO; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) R.yo[t][v] = T(0);

    T *y = out + ec * L::NC;
    // entries 4s + g of both parities back to the coefficients
    const auto store = [&](auto sc, T ve, T vo) {
        constexpr int s = decltype(sc)::value;
        constexpr bool pairs = 4 * s < L::NH;
        if constexpr (s < L::SE) {
            const int a = column_index<NM, false, false, s>(g);
            T v = ve;
            if constexpr (pairs) {
                const int b = column_index<NM, false, true, s>(g);
                if (valid && b >= 0) y[b] = ve + vo;
                v = b >= 0 ? ve - vo : ve;
            }
            if (valid && a >= 0) y[a] = v;
        }
        if constexpr (s < L::SO && 4 * s + 4 > L::NH) {
            const int a = column_index<NM, true, false, s>(g);
            if (valid && a >= 0 && 4 * s + g >= L::NH) y[a] = vo;
        }
    };
    constexpr int NS = L::SE > L::SO ? L::SE : L::SO;
    if constexpr (!SPLIT) {
        __shared__ typename SharedStream<T, NM>::Buffer buf[2];
        SharedStream<T, NM> st(tab, buf);
        items<T, NM, 0, L::NITEM>(R, st, m, lj);
        for_range<0, NS>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            store(sc, s < L::SE ? R.ye[s < L::SE ? s / 4 : 0][s % 4] : T(0),
                  s < L::SO ? R.yo[s < L::SO ? s / 4 : 0][s % 4] : T(0));
        });
    } else {
        if (wave == 0) part<T, NM, 0>(R, tab, lane, m, lj);
        else if (wave == 1) part<T, NM, 1>(R, tab, lane, m, lj);
        else if (wave == 2) part<T, NM, 2>(R, tab, lane, m, lj);
        else part<T, NM, 3>(R, tab, lane, m, lj);
        // a quarter of the steps at a time through LDS; wave q adds and
        // stores quarter q
        constexpr int NQ = (NS + 3) / 4;
        __shared__ T red[kWaves][2 * NQ][64];
        for_range<0, 4>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            if constexpr (q > 0) __syncthreads();
            for_range<0, NQ>([&](auto kc) {
                constexpr int k = decltype(kc)::value, s = q * NQ + k;
                if constexpr (s < L::SE) red[wave][2 * k][lane] = R.ye[s < L::SE ? s / 4 : 0][s % 4];
                if constexpr (s < L::SO) red[wave][2 * k + 1][lane] = R.yo[s < L::SO ? s / 4 : 0][s % 4];
            });
            __syncthreads();
            if (wave == q) {
                for_range<0, NQ>([&](auto kc) {
                    constexpr int k = decltype(kc)::value, s = q * NQ + k;
                    T ve = T(0), vo = T(0);
                    if constexpr (s < L::SE)
                        ve = ((red[0][2 * k][lane] + red[1][2 * k][lane]) + red[2][2 * k][lane]) + red[3][2 * k][lane];
                    if constexpr (s < L::SO)
                        vo = ((red[0][2 * k + 1][lane] + red[1][2 * k + 1][lane]) + red[2][2 * k + 1][lane]) +
                             red[3][2 * k + 1][lane];
                    if constexpr (s < NS) store(std::integral_constant<int, s>{}, ve, vo);
                });
            }
        });
    }
}

template <typename T, int NM, bool SPLIT>
__global__ __launch_bounds__(kBlock) void helmholtz_kernel(int nelmt, const T *__restrict__ tab,
                                                           const T *__restrict__ geo, T lambda,
                                                           const T *__restrict__ in, T *__restrict__ out)
{
    helmholtz_block<T, NM, SPLIT>(blockIdx.x, nelmt, tab, geo, lambda, in, out);
}

// Grouped form: several operators of one kind; block b belongs to the item
// whose [block0, next block0) range holds it
template <typename T, int NM>
__global__ __launch_bounds__(kBlock) void helmholtz_grouped_kernel(int count, const GroupItem<T> *__restrict__ items,
                                                                   const T *__restrict__ tab)
{
    const int b = blockIdx.x;
    int it = 0;
    while (it + 1 < count && b >= items[it + 1].block0) ++it;
    const GroupItem<T> I = items[it];
    if (tet_modal_split(I.nelmt))
        helmholtz_block<T, NM, true>(b - I.block0, I.nelmt, tab, I.geo, I.lambda, I.in, I.out);
    else
        helmholtz_block<T, NM, false>(b - I.block0, I.nelmt, tab, I.geo, I.lambda, I.in, I.out);
}

}  // namespace tetmodal
}  // namespace nektar_amd
