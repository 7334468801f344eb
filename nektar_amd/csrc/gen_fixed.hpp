// Prism and pyramid operators with compile-time sizes: the stages of
// generic_kernels.hpp, instantiated for equal modes in the three directions and
// the shape's default points, Q = NM + 1 and NM + 2.
//
// The runtime-size kernels spend their time around the products: trip counts
// and index divisions at run time, every table value a global load of its own,
// all operators in one kernel.  Here the sizes and the operator are constants
// (set in the kernel's copy of the arguments, from where they propagate), and
// every workgroup stages the tables and index tables in LDS (for one element up
// to kFixedGroups elements, for several above).  4,096 prisms at NM = 5, NQ = 6: FP64 45.5 -> 19.9 us,
// FP32 38.0 -> 14.8; bound by LDS, which serves every value of a product (a
// register budget for 6 or 8 waves per SIMD instead of 5 changes nothing, and
// derivatives line by line, one direction per wave with its matrix in scalar
// registers, were slower: 27.5 us).
#pragma once

#include <hip/hip_runtime.h>

#include "generic_kernels.hpp"

namespace nektar_amd {
namespace gen {

// workgroups of the walking grid: at least as many as the LDS and waves of the
// 256 CUs hold
constexpr int kFixedGroups = 256 * 16;

template <int SH, int NM, int NQ>
struct Fixed {
    static constexpr int N0 = NQ, N1 = NQ, N2 = NQ - 1;
    static constexpr int NQT = N0 * N1 * N2, NPQ = NM * NM;
    static constexpr int coeffs()
    {
        int n = 0;
        for (int p = 0; p < NM; ++p)
            for (int q = 0; q < NM; ++q) n += SH == SH_PRISM ? NM - p : NM - (p > q ? p : q);
        return n;
    }
    static constexpr int NC = coeffs();
    // work-items: about one per point, whole waves, at most 256
    static constexpr int THREADS = NQT >= 192 ? 256 : NQT >= 128 ? 192 : NQT > 64 ? 128 : 64;
};

template <typename T, int SH, int NM, int NQ, OpType OP>
__global__ __launch_bounds__((Fixed<SH, NM, NQ>::THREADS)) void fixed_kernel(GenArgs a0)
{
    using F = Fixed<SH, NM, NQ>;
    extern __shared__ __align__(16) unsigned char smem[];
    T *X = reinterpret_cast<T *>(smem);
    T *tab = X + 4 * a0.buf;
    int *itab = reinterpret_cast<int *>(tab + a0.ntab);
    for (int i = threadIdx.x; i < a0.ntab; i += blockDim.x) tab[i] = static_cast<const T *>(a0.tab)[i];
    for (int i = threadIdx.x; i < a0.nitab; i += blockDim.x) itab[i] = a0.itab[i];
    __syncthreads();
    GenArgs a = a0;
    a.op = OP;
    for (int d = 0; d < 3; ++d) a.nm[d] = NM;
    a.nq[0] = F::N0;
    a.nq[1] = F::N1;
    a.nq[2] = F::N2;
    a.nqtot = F::NQT;
    a.ncoeff = F::NC;
    a.npq = F::NPQ;
    a.tab = tab;
    a.itab = itab;
    for (int e = blockIdx.x; e < a.nelmt; e += gridDim.x) {
        element<T, SH>(a, e, X, X + a0.buf, X + 2 * a0.buf, X + 3 * a0.buf);
        __syncthreads();  // the buffers are reused by the next element
    }
}

template <typename T, int SH, int NM, int NQ>
hipError_t launch_fixed(const GenArgs &a)
{
    using F = Fixed<SH, NM, NQ>;
    if (a.nelmt == 0) return hipSuccess;
    const size_t lds = ((size_t)4 * a.buf + a.ntab) * sizeof(T) + (size_t)a.nitab * sizeof(int);
    if (lds > kMaxLds || a.nqtot != F::NQT || a.ncoeff != F::NC || a.npq != F::NPQ) return hipErrorInvalidValue;
    const dim3 grid(a.nelmt < kFixedGroups ? a.nelmt : kFixedGroups), block(F::THREADS);
#define NMF_FIXED(OP)                                                                                               \
    case OP:                                                                                                        \
        hipLaunchKernelGGL((fixed_kernel<T, SH, NM, NQ, OP>), grid, block, (unsigned)lds, a.stream, a);              \
        break;
    switch (a.op) {
        NMF_FIXED(OpType::BwdTrans)
        NMF_FIXED(OpType::IProduct)
        NMF_FIXED(OpType::PhysDeriv)
        NMF_FIXED(OpType::Helmholtz)
        NMF_FIXED(OpType::IProductDeriv)
        NMF_FIXED(OpType::AdvDiffReact)
    default: return hipErrorInvalidValue;
    }
#undef NMF_FIXED
    return hipGetLastError();
}

// (modes, points, precision) of the arguments, which fixed_sizes() accepted
template <int SH>
hipError_t launch_fixed_shape(const GenArgs &a)
{
    const int d = a.nq[0] - a.nm[0];
    switch (a.nm[0]) {
#define NMF_FIXED(N)                                                                                      \
    case N:                                                                                               \
        return d == 1 ? (a.fp32 ? launch_fixed<float, SH, N, N + 1>(a) : launch_fixed<double, SH, N, N + 1>(a)) \
                      : (a.fp32 ? launch_fixed<float, SH, N, N + 2>(a) : launch_fixed<double, SH, N, N + 2>(a));
        NMF_FIXED(3) NMF_FIXED(4) NMF_FIXED(5) NMF_FIXED(6) NMF_FIXED(7)
#undef NMF_FIXED
    default: return hipErrorInvalidValue;
    }
}

}  // namespace gen
}  // namespace nektar_amd
