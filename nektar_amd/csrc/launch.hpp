// Kernel launch dispatch for the matrix-free operators.  Each (shape, NM)
// pair is instantiated in its own translation unit (ops_<shape>_nm<NM>.hip)
// for NQ = NM+1 (the MODIFIED default Q = P+2) and NQ = NM+2.
#pragma once

#include <hip/hip_runtime.h>

namespace nektar_amd {

enum class OpType {
    BwdTrans = 0,
    IProduct = 1,
    PhysDeriv = 2,
    Helmholtz = 3,
    IProductDeriv = 4,
    AdvDiffReact = 5,
    PhysInterp = 6
};

struct KernelArgs {
    OpType op;
    bool fp32;
    bool deformed;
    int nelmt;
    const void *tab;
    const void *geo;
    double lambda;
    const void *in;
    void *out0, *out1, *out2;
    hipStream_t stream;
    int tile = 0;  // Helmholtz: elements per workgroup (0 = default)
    const void *in1 = nullptr, *in2 = nullptr;  // IProductDeriv: inputs 1, 2 (in = input 0)
    const void *adv = nullptr;  // AdvDiffReact: advection coefficients per point
    const int *menc = nullptr;  // hex Helmholtz: signed local-to-global map; `in` is then the global vector
};

// Order-templated kernels of the structured-hex C0 solver.
enum class SolverKernel { Apply = 0, Diag = 1, Rhs = 2, BwdGather = 3 };

struct SolverArgs {
    SolverKernel kind;
    bool fp32;      // Apply only: FP32 operator (vectors, tables, geometry)
    bool deformed;
    int n, N;       // elements and global nodes per direction
    const void *tab;
    const void *dtab;  // Diag: {B^2, B B', B'^2} (FP64)
    const void *geo;
    double lambda;
    const void *in;
    void *out;
    const int *done;   // Apply: early exit flag (NULL = always run)
    hipStream_t stream;
    int tile = 0;      // Apply: elements per workgroup (0 = default)
    double *edot = nullptr;  // FP64 Apply: in_e . out_e per element (required)
};

// Tile shapes (elements per workgroup) available for the hex Helmholtz
// kernels of a given order, in the order the autotuner tries them.
int hex_tile_candidates(int nm, int nq, bool fp32, bool deformed, int *out, int max);

// Grouped Helmholtz: several operators of one kind (shape, modes, points,
// precision, geometry type) in one launch.  Items are ordered with
// block0 ascending from 0; item i owns workgroups [block0_i, block0_{i+1}).
template <typename T>
struct GroupItem {
    const T *geo;
    const T *in;
    T *out;
    T lambda;
    int nelmt;
    int block0;
};

struct GroupArgs {
    bool fp32;
    bool deformed;
    int count;          // items
    const void *items;  // device array of GroupItem<float|double>
    int nblocks;        // total workgroups of the launch
    const void *tab;    // tables shared by every item of the kind
    hipStream_t stream;
    int tile = 0;       // hex: elements per workgroup (0 = default, affine elements only)
};

// Workgroups go to the 8 XCDs in turn, and each XCD has an L2 of its own.
// Kernels whose neighbouring workgroups share cache lines (solver forms: the
// nodes of neighbouring elements, the rows of one) give every XCD one
// contiguous part: work b of n on a grid of xcd_grid(n) workgroups (the last
// ones have none: >= n).
constexpr int kXcds = 8;
constexpr int xcd_grid(int n) { return (n + kXcds - 1) / kXcds * kXcds; }
__host__ __device__ inline int xcd_work(int block, int n)
{
    return (block % kXcds) * ((n + kXcds - 1) / kXcds) + block / kXcds;
}

// Elements per workgroup: hex default fill (tile 0) or the given tile.
// A tet tile is the number of work-items per element: packed
// (nq0*(nq0-1), elements share waves) or wave-aligned (rounded up to a
// multiple of 64); workgroups hold 256/tile elements (at least one).  The
// kernels assert they use the same numbers.
constexpr int hex_fill_elems(int nq) { return 256 / (nq * nq) > 0 ? 256 / (nq * nq) : 1; }
// Hex Helmholtz tiles kMfmaTile + E select the matrix-core kernels with E
// elements per 256-work-item workgroup; they are compiled for NUMMODES >=
// kMfmaMinModes (where the per-direction products are dense enough).
constexpr int kMfmaTile = 1024, kMfmaMinModes = 5;
// Default of the Legendre-space kernels of affine elements (hex_modal.hpp,
// NM^2 work-items per element): whole waves of one element (NM = 7, 8, 10)
// or of as many as one wave or a few waves hold.  Measured in FP64 on 11.2 M
// coefficients, best of 1, 2, 3, 4, 5, 7, 10 and 14 elements: NM = 3: 56 us
// (1 element: 205), 4: 40 (118), 5: 49 (85), 6: 47 (59), 7: 49, 8: 42, 9: 51
// (58), 10: 49; the same ones are best or within 3 % in FP32.
constexpr int hex_modal_elems(int nm)
{
    return nm <= 4 ? 64 / (nm * nm) : nm <= 6 ? 5 : nm == 9 ? 2 : 1;
}
// Default tile of the kernels with per-point geometry: the matrix-core tile
// of one element where its 16-row products are well filled and the vector
// kernel's are not bound by memory yet.  Measured vector / matrix cores, us on
// 1.6 M points: FP64 NM, NQ = 6, 8 35.5/23.2; 7, 8 37/25; 8, 9 28/39; 8, 10
// 41/32; 9, 10 42/37; 10, 11 47/34; 10, 12 47/38; 8, 8 40/26; 10, 10 44/39;
// 6, 7 27/27; 5, 7 26/26; FP32 7, 8 16.8/15.8; 8, 8 17.5/14.8; 8, 10 21/22;
// 10, 11 23/19; 10, 12 25/20.  The mapped form of the general solver gains as
// much (apply and assembly, FP64, 7, 8 at 512 / 4,096 elements 18.7/14.0,
// 52.4/46.3; 10, 11 at 512 / 1,000 34.5/26.2, 43/39.9).  In FP32 at NQ = 11
// the card holds 1,536 elements at once on the matrix cores and 2,048 on the
// vector units: the former are faster while they need no more rounds (10, 11,
// vector / matrix cores at 1,536, 1,552, 2,048, 2,064, 3,072, 4,096, 4,112 and
// 6,144 elements: 1.07, 0.93, 0.89, 1.22, 1.07, 0.97, 1.14, 0.93).
constexpr int hex_deformed_tile(int nm, int nq, bool fp32, int nelmt)
{
    const auto rounds = [&](int held) { return (nelmt + held - 1) / held; };
    const bool mfma = nm >= 6 && (fp32 ? nq == 8 || nq == 12 || (nq == 11 && rounds(1536) == rounds(2048))
                                       : nq == 8 || nq >= 10);
    return mfma ? kMfmaTile + 1 : hex_fill_elems(nq);
}
// elements per workgroup of a tile of a hex Helmholtz kind (0, the default,
// with affine elements only)
inline int hex_tile_elems(int nm, int tile)
{
    if (tile <= 0) return hex_modal_elems(nm);
    return tile >= kMfmaTile ? tile - kMfmaTile : tile;
}
constexpr int tet_packed_tpe(int nq0) { return nq0 * (nq0 - 1); }
constexpr int tet_wave_tpe(int nq0) { return (nq0 * (nq0 - 1) + 63) / 64 * 64; }
// default: wave-aligned where one element fills most of a wave (Q = 8:
// 56 of 64 work-items), packed otherwise (measured, FP64 and FP32 apply)
constexpr int tet_default_tpe(int nq0) { return nq0 == 8 ? tet_wave_tpe(nq0) : tet_packed_tpe(nq0); }
constexpr int tet_tile_elems(int nq0, int tile)
{
    return 256 / (tile > 0 ? tile : tet_default_tpe(nq0)) > 0 ? 256 / (tile > 0 ? tile : tet_default_tpe(nq0)) : 1;
}
// Affine tets run the matrix-core kernel (tet_modal.hpp) whatever the tile:
// 16 elements per wave, four waves per workgroup.  With `split` the four waves
// share 16 elements: shorter, but more of it (each wave loads the 16 elements,
// and the results are added through LDS).  Measured whole against split, FP64
// us at 4,096 / 8,192 / 16,384 elements: NM = 4 4.0/3.4, 4.2/4.2, 4.8/5.9;
// NM = 7 13/7.1, 14/11, 16/20; NM = 10 40/18, 42/32, 47/61; FP32 alike.  The
// line lies where whole waves would fill five eighths of the 1024 SIMDs.
constexpr bool tet_modal_split(int nelmt) { return nelmt <= 640 * 16; }
constexpr int tet_modal_blocks(int nelmt)
{
    return tet_modal_split(nelmt) ? (nelmt + 15) / 16 : (nelmt + 63) / 64;
}
// tet tile candidates (work-items per element) in the order the autotuner
// tries them
int tet_tile_candidates(int nq0, int *out, int max);

hipError_t launch_hex_grouped(int nm, int nq, const GroupArgs &a);

// PhysInterp1DScaled: ni / no points per direction in and out, tables
// IT0 | IT1 | IT2 with ITd[i*ni[d] + p] = weight of input point p for
// output point i (k_interp.hip).
struct InterpArgs {
    bool fp32;
    int nelmt;
    int ni[3], no[3];
    const void *tab;
    const void *in;
    void *out;
    hipStream_t stream;
};
constexpr size_t kInterpMaxLds = 65536;  // dynamic LDS of one workgroup
size_t interp_lds_bytes(const int ni[3], const int no[3], bool fp32);
hipError_t launch_phys_interp(const InterpArgs &a);
hipError_t launch_tet_grouped(int nm, int nq0, const GroupArgs &a);

constexpr int kMinModes = 2, kMaxModes = 10;

bool hex_supported(int nm, int nq);
bool hex_op_supported(int nm, int nq);  // Collections operators: also Q = NUMMODES
bool tet_supported(int nm, int nq0);
hipError_t launch_hex(int nm, int nq, const KernelArgs &a);
hipError_t launch_tet(int nm, int nq0, const KernelArgs &a);
hipError_t launch_hex_solver(int nm, int nq, const SolverArgs &a);

}  // namespace nektar_amd
