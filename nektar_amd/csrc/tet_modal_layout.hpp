// Compile-time layout of the affine-tet Helmholtz operator in an orthogonal
// polynomial space (tet_modal.hpp): orders the modes and the gradient's
// polynomials by their parity in the first collapsed direction, says which
// 16x4 blocks of the operator's matrices are not zero, and numbers those
// blocks in the order in which the kernel uses them.  Shared by the kernel and
// by the host code that fills the blocks (tet_modal.cpp).
#pragma once

#include <vector>

namespace nektar_amd {
namespace tetmodal {

// A column: mode (p, q, r) of the Modified tet basis, or, with at >= 0 in
// `b`, the sum (p = 0) or difference (p = 1) of the two modes a and b that
// the reflection a -> -a of the first collapsed direction exchanges, (0, ...)
// and (1, ...).  a, b: coefficient indices.  Sums and differences are of the
// coefficients; the functions they multiply are half the sum and half the
// difference of the modes.
struct Col {
    short p, q, r, a, b;
};
// A row: orthogonal polynomial (p, q, r), p + q + r <= nm - 2
struct Row {
    short p, q, r;
};

constexpr int coeffs(int nm) { return nm * (nm + 1) * (nm + 2) / 6; }
// coefficient index of mode (p, q, r): p-major, then q, r fastest
constexpr int mode_index(int nm, int p, int q, int r)
{
    int i = 0;
    for (int pp = 0; pp < p; ++pp) i += (nm - pp) * (nm - pp + 1) / 2;
    for (int qq = 0; qq < q; ++qq) i += nm - p - qq;
    return i + r;
}

// The matrices: gradients of even columns into odd rows ... (direction 0 is
// odd under the reflection, the combined directions 1 and 2 are even), and
// the two parities of the mass matrix.
enum Mat { G0E = 0, G1E, G2E, G0O, G1O, G2O, MASS_E, MASS_O };

template <int NM>
struct Layout {
    static constexpr int NC = coeffs(NM), NR = coeffs(NM - 1);
    static constexpr int NH = NM * (NM - 1) / 2;  // exchanged pairs

    struct Lists {
        Col e[NC + 1] = {}, o[NC + 1] = {};
        Row re[NR + 1] = {}, ro[NR + 1] = {};
        int ne = 0, no = 0, nre = 0, nro = 0;
    };
    static constexpr Lists make_lists()
    {
        Lists L{};
        // pairs first, so that entry i of both lists is pair i
        for (int q = 0; q < NM - 1; ++q)
            for (int r = 0; r < NM - 1 - q; ++r) {
                // mode (1, q, r) and its image: (0, 0, 0), (0, 0, r+1), (0, q+1, r)
                const int b = mode_index(NM, 1, q, r);
                const int q0 = q == 0 ? 0 : q + 1, r0 = q == 0 ? (r == 0 ? 0 : r + 1) : r;
                const int a = mode_index(NM, 0, q0, r0);
                L.e[L.ne++] = Col{0, (short)q0, (short)r0, (short)a, (short)b};
                L.o[L.no++] = Col{1, (short)q, (short)r, (short)a, (short)b};
            }
        // modes that are their own image: the top vertex, the collapsed
        // vertex and edge (0, 1, r), and the modes p >= 2 of either parity
        L.e[L.ne++] = Col{0, 0, 1, (short)mode_index(NM, 0, 0, 1), -1};
        for (int r = 0; r < NM - 1; ++r) L.e[L.ne++] = Col{0, 1, (short)r, (short)mode_index(NM, 0, 1, r), -1};
        for (int p = 2; p < NM; ++p)
            for (int q = 0; q < NM - p; ++q)
                for (int r = 0; r < NM - p - q; ++r) {
                    const Col c{(short)p, (short)q, (short)r, (short)mode_index(NM, p, q, r), -1};
                    if (p % 2 == 0) L.e[L.ne++] = c;
                    else L.o[L.no++] = c;
                }
        for (int p = 0; p < NM - 1; ++p)
            for (int q = 0; q < NM - 1 - p; ++q)
                for (int r = 0; r < NM - 1 - p - q; ++r) {
                    const Row w{(short)p, (short)q, (short)r};
                    if (p % 2 == 0) L.re[L.nre++] = w;
                    else L.ro[L.nro++] = w;
                }
        return L;
    }
    static constexpr Lists L = make_lists();
    static constexpr int NE = L.ne, NO = L.no, NRE = L.nre, NRO = L.nro;
    // steps of 4 columns, tiles of 16 columns and rows
    static constexpr int SE = (NE + 3) / 4, SO = (NO + 3) / 4, TE = (NE + 15) / 16, TO = (NO + 15) / 16;
    static constexpr int GE = (NRE + 15) / 16, GO = (NRO + 15) / 16;
    static constexpr int MAXT = TE > 0 ? TE : 1, MAXS = 4 * MAXT;

    static constexpr const Col *cols(bool odd) { return odd ? L.o : L.e; }
    static constexpr const Row *rows(bool odd) { return odd ? L.ro : L.re; }
    static constexpr int ncols(bool odd) { return odd ? NO : NE; }
    static constexpr int nrows(bool odd) { return odd ? NRO : NRE; }
    // parity of a matrix's rows and columns
    static constexpr bool row_odd(int m) { return m == G0O || m == G1O || m == G2O; }
    static constexpr bool col_odd(int m) { return m == G0E || m == G1O || m == G2O || m == MASS_O; }

    // Entries that can be other than zero.  The modes are built on integrated
    // Jacobi polynomials, so a derivative reaches one row degree P in the
    // first collapsed direction (direction 0) or two, a few Q and three R.
    static constexpr bool grad_entry(int m, const Row &w, const Col &c)
    {
        const int dp = w.p - c.p, dq = w.q - c.q, d = dp + dq, dr = w.r - c.r;
        if (dr < -3 - d || dr > -1 - d + (c.p == 0)) return false;
        if (m == G0E || m == G0O) return dp == -1 && dq >= -1 && dq <= 0;
        const bool two = c.p >= 2 && dp == -2;  // P = p - 2
        if (!two && dp != 0) return false;
        if (m == G1E || m == G1O) return two ? (dq >= 0 && dq <= 1) : (dq >= -2 && dq <= (c.p == 0 ? 0 : -1));
        return two ? (dq >= -1 && dq <= 2) : (dq >= -3 && dq <= (c.p == 0 ? 1 : 0));
    }
    static constexpr bool mass_entry(const Col &x, const Col &y)
    {
        const int dp = x.p - y.p, dq = x.q - y.q, d = dp + dq + (x.r - y.r);
        if (d < -5 || d > 5) return false;
        if (dp == 0) return dq >= -4 && dq <= 4;
        if (dp == 2) return dq >= -6 && dq <= 2;
        return dp == -2 && dq >= -2 && dq <= 6;
    }
    // block of 16 rows (tile t) and 4 columns (step s); `tr`: of the
    // transposed gradient, 16 columns by 4 rows
    static constexpr bool grad_block(int m, bool tr, int t, int s)
    {
        const bool ro = row_odd(m), co = col_odd(m);
        const int r0 = tr ? 4 * s : 16 * t, r1 = r0 + (tr ? 4 : 16), c0 = tr ? 16 * t : 4 * s, c1 = c0 + (tr ? 16 : 4);
        for (int r = r0; r < r1 && r < nrows(ro); ++r)
            for (int c = c0; c < c1 && c < ncols(co); ++c)
                if (grad_entry(m, rows(ro)[r], cols(co)[c])) return true;
        return false;
    }
    static constexpr bool mass_block(int m, int t, int s)
    {
        const bool co = col_odd(m);
        for (int r = 16 * t; r < 16 * t + 16 && r < ncols(co); ++r)
            for (int c = 4 * s; c < 4 * s + 4 && c < ncols(co); ++c)
                if (mass_entry(cols(co)[r], cols(co)[c])) return true;
        return false;
    }

    // Work items: one 16-row tile of the gradient (even ones first) with its
    // way back, and the two mass matrices.  PARTS waves share an element
    // tile; the longest remaining item goes to the part with the least.
    static constexpr int NITEM = GE + GO + 2, PARTS = 4;
    // position of every block in the stream (-1: zero), [tile][step]
    struct Blocks {
        short fwd[6][MAXT][MAXS] = {}, bwd[6][MAXT][MAXS] = {}, mass[2][MAXT][MAXS] = {};
        short cost[NITEM] = {};
    };
    // Block present flags first (numbered below).
    static constexpr Blocks present()
    {
        Blocks b{};
        for (int m = 0; m < 6; ++m)
            for (int t = 0; t < MAXT; ++t)
                for (int s = 0; s < MAXS; ++s) {
                    b.fwd[m][t][s] = grad_block(m, false, t, s) ? 0 : -1;
                    b.bwd[m][t][s] = grad_block(m, true, t, s) ? 0 : -1;
                }
        for (int m = 0; m < 2; ++m)
            for (int t = 0; t < MAXT; ++t)
                for (int s = 0; s < MAXS; ++s) b.mass[m][t][s] = mass_block(MASS_E + m, t, s) ? 0 : -1;
        return b;
    }
    static constexpr Blocks P = present();
    static constexpr int item_cost(int it)
    {
        int n = 0;
        if (it >= GE + GO) {
            for (int t = 0; t < MAXT; ++t)
                for (int s = 0; s < MAXS; ++s) n += P.mass[it - GE - GO][t][s] >= 0;
            return n;
        }
        const bool odd = it >= GE;
        const int t = odd ? it - GE : it;
        for (int d = 0; d < 3; ++d) {
            const int m = (odd ? G0O : G0E) + d;
            for (int s = 0; s < MAXS; ++s) n += P.fwd[m][t][s] >= 0;
            for (int v = 0; v < 4; ++v)
                for (int y = 0; y < MAXT; ++y)
                    if (4 * t + v < MAXS) n += P.bwd[m][y][4 * t + v] >= 0;
        }
        return n;
    }
    struct Plan {
        int order[NITEM] = {};           // items, part by part
        int first[PARTS + 1] = {};       // index into order
        int start[PARTS + 1] = {};       // block positions, multiples of 4
        int end[PARTS] = {};             // last block + 1 of each part
        int total = 0;
        Blocks b{};
    };
    static constexpr Plan make_plan()
    {
        Plan pl{};
        int cost[NITEM] = {}, owner[NITEM] = {}, load[PARTS] = {};
        bool done[NITEM] = {};
        for (int i = 0; i < NITEM; ++i) cost[i] = item_cost(i);
        for (int k = 0; k < NITEM; ++k) {
            int best = -1, part = 0;
            for (int i = 0; i < NITEM; ++i)
                if (!done[i] && (best < 0 || cost[i] > cost[best])) best = i;
            for (int p = 1; p < PARTS; ++p)
                if (load[p] < load[part]) part = p;
            done[best] = true;
            owner[best] = part;
            load[part] += cost[best];
        }
        pl.b = P;
        int pos = 0, idx = 0;
        for (int p = 0; p < PARTS; ++p) {
            pl.first[p] = idx;
            pl.start[p] = pos;
            for (int i = 0; i < NITEM; ++i)
                if (owner[i] == p) {
                    pl.order[idx++] = i;
                    number_item(pl.b, i, pos);
                }
            pl.end[p] = pos;
            pos = (pos + 3) / 4 * 4;
        }
        pl.first[PARTS] = idx;
        pl.start[PARTS] = pl.total = pos;
        return pl;
    }
    // The order in which the kernel walks an item's blocks.
    static constexpr void number_item(Blocks &b, int it, int &pos)
    {
        if (it >= GE + GO) {
            const int m = it - GE - GO;
            for (int s = 0; s < MAXS; ++s)
                for (int t = 0; t < MAXT; ++t)
                    if (b.mass[m][t][s] >= 0) b.mass[m][t][s] = (short)pos++;
            return;
        }
        const bool odd = it >= GE;
        const int t = odd ? it - GE : it, m0 = odd ? G0O : G0E;
        for (int s = 0; s < MAXS; ++s)
            for (int d = 0; d < 3; ++d)
                if (b.fwd[m0 + d][t][s] >= 0) b.fwd[m0 + d][t][s] = (short)pos++;
        for (int v = 0; v < 4; ++v)
            for (int y = 0; y < MAXT; ++y)
                for (int d = 0; d < 3; ++d)
                    if (4 * t + v < MAXS && b.bwd[m0 + d][y][4 * t + v] >= 0)
                        b.bwd[m0 + d][y][4 * t + v] = (short)pos++;
    }
    static constexpr Plan plan = make_plan();
    // block used before block pos (-1: none); parts end in padding
    static constexpr int previous(int pos)
    {
        for (int p = 0; p < PARTS; ++p)
            if (pos == plan.start[p] && plan.start[p] < plan.end[p]) {
                for (int q = p - 1; q >= 0; --q)
                    if (plan.start[q] < plan.end[q]) return plan.end[q] - 1;
                return -1;
            }
        return pos - 1;
    }
};

// The stream of an operator's kernel: block after block as the lanes of a
// wave read them (16 bytes per lane: two FP64 or four FP32 blocks)
const std::vector<double> &build_tables(int nm, bool fp32);

}  // namespace tetmodal
}  // namespace nektar_amd
