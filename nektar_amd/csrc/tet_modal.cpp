// Host side of the affine-tet Helmholtz operator in an orthogonal polynomial
// space (tet_modal.hpp): fills the 16x4 blocks of its matrices.
//
// Modes and polynomials are products of functions of the three collapsed
// coordinates, so every entry is a sum of at most three products of 1-D
// integrals; these are taken in extended precision with Gauss-Legendre points
// enough for their degree.
#include "tet_modal_layout.hpp"

#include <array>
#include <cmath>
#include <memory>

#include "common.hpp"

namespace nektar_amd {
namespace tetmodal {

namespace {

using Real = long double;

// P_0^{a,b}(x) .. P_{n-1}^{a,b}(x) by the three-term recurrence
void jacobi_sweep(int n, int a, int b, Real x, Real *p)
{
    if (n > 0) p[0] = 1;
    if (n > 1) p[1] = (a - b + (a + b + 2) * x) / 2;
    for (int k = 1; k + 1 < n; ++k) {
        const Real c = 2 * k + a + b;
        p[k + 1] = ((c + 1) * (c * (c + 2) * x + (Real)a * a - (Real)b * b) * p[k] -
                    2 * (Real)(k + a) * (k + b) * (c + 2) * p[k - 1]) /
                   (2 * (Real)(k + 1) * (k + a + b + 1) * c);
    }
}

Real ipow(Real x, int n)
{
    Real r = 1;
    for (int i = 0; i < n; ++i) r *= x;
    return r;
}

struct Val {
    Real v, d;  // value and derivative
};
Val mul(Val a, Val b) { return {a.v * b.v, a.d * b.v + a.v * b.d}; }
Val low(Real x) { return {(1 - x) / 2, -Real(0.5)}; }
Val high(Real x) { return {(1 + x) / 2, Real(0.5)}; }
Val low_pow(int n, Real x)
{
    if (n == 0) return {1, 0};
    return {ipow((1 - x) / 2, n), -Real(n) / 2 * ipow((1 - x) / 2, n - 1)};
}

// Modified_A (p = 0) and Modified_B (p, 0 .. n-1) at x (Basis.cpp:452-589)
void mod_b(int p, int n, Real x, Val *out)
{
    Real v[16], d[16];
    const int a = p == 0 ? 1 : 2 * p - 1;  // P_k^{a,1} and its derivative
    jacobi_sweep(n, a, 1, x, v);
    d[0] = 0;
    jacobi_sweep(n - 1, a + 1, 2, x, d + 1);
    const Val shape = p == 0 ? mul(low(x), high(x)) : mul(low_pow(p, x), high(x));
    const int first = p == 0 ? 2 : 1;
    for (int q = first; q < n; ++q) {
        const int k = q - first;
        out[q] = mul(shape, Val{v[k], (Real)(k + a + 2) / 2 * d[k]});
    }
    out[0] = p == 0 ? low(x) : low_pow(p, x);
    if (p == 0 && n > 1) out[1] = high(x);
}

// The three 1-D factors of a column's function, by class: many columns share
// one.  Direction 1: Modified_B (p, q), or 1 (top vertex); direction 2:
// Modified_B (p + q, r), which holds the top vertex's (1 + c)/2 as (0, 1).
int class_a(int nm, const Col &m) { return m.p >= 2 || m.b >= 0 ? m.p : nm; }
int class_b(int nm, const Col &m) { return m.b < 0 && m.p == 0 && m.q == 0 ? nm * nm : m.p * nm + m.q; }
int class_c(int nm, const Col &m) { return (m.p + m.q) * nm + m.r; }
// Gauss-Legendre points and weights
void legendre_rule(int n, std::vector<Real> &z, std::vector<Real> &w)
{
    z.resize(n);
    w.resize(n);
    for (int i = 0; i < n; ++i) {
        Real x = -std::cos(3.14159265358979323846264338327950288L * (i + Real(0.75)) / (n + Real(0.5)));
        Real p[32], d = 1;
        for (int it = 0; it < 50; ++it) {
            jacobi_sweep(n + 1, 0, 0, x, p);
            d = n * (p[n - 1] - x * p[n]) / (1 - x * x);
            x -= p[n] / d;
            if (std::fabs(p[n] / d) < 1e-18L) break;
        }
        z[i] = x;
        w[i] = 2 / ((1 - x * x) * d * d);
    }
}

// 1-D integrals of a pair of classes, each taken once
template <int W>
struct Memo {
    int cols;
    std::vector<char> have;
    std::unique_ptr<std::array<Real, W>[]> val;  // left as allocated: few pairs are asked for
    Memo(int rows, int c) : cols(c), have((size_t)rows * c, 0), val(new std::array<Real, W>[(size_t)rows * c]) {}
    template <typename F>
    const std::array<Real, W> &get(int r, int c, F &&f)
    {
        const size_t i = (size_t)r * cols + c;
        if (!have[i]) {
            val[i] = f();
            have[i] = 1;
        }
        return val[i];
    }
};

template <int NM>
struct Entries {
    using L = Layout<NM>;
    static constexpr int N = NM + 3, NN = NM * NM;  // exact to degree 2 NM + 5
    std::vector<Real> z, w;
    // columns' factors of direction 0 and of directions 1 and 2 [class * N + point]
    std::vector<Val> fa, fb;
    // rows' factors with the collapse's weights h_b h_c^2, of which one power
    // of each is left to the integrals: [class * N + point], classes P,
    // (P, Q) and (P + Q, R) of the orthogonal polynomials
    std::vector<Real> ra, rb, rc;
    std::vector<Real> scale[2];  // 1 / norm of the even and odd rows
    // columns' factors with the weights of directions 0, 1 (h_b) and 2 (h_c^2)
    std::vector<Real> wa, wb, wc;
    Memo<3> ga{NM, NM + 1};
    Memo<4> gb{NN, NN + 1};
    Memo<2> gc{NN, NN};
    Memo<1> ma{NM + 1, NM + 1}, mb{NN + 1, NN + 1}, mc{NN, NN};
    Entries() : fa((NM + 1) * N), fb((NN + 1) * N), ra(NM * N), rb(NN * N), rc(NN * N)
    {
        legendre_rule(N, z, w);
        for (int odd = 0; odd < 2; ++odd)
            for (int r = 0; r < L::nrows(odd); ++r) {
                const Row &R = L::rows(odd)[r];
                scale[odd].push_back(1 / std::sqrt(2 / Real(2 * R.p + 1) * (2 / Real(2 * (R.p + R.q) + 2)) *
                                                   (2 / Real(2 * (R.p + R.q + R.r) + 3))));
            }
        for (int i = 0; i < N; ++i) {
            const Real x = z[i], h = (1 - x) / 2;
            Val m[NM];
            Real p[NM + 1];
            mod_b(0, NM, x, m);
            for (int c = 2; c < NM; ++c) fa[c * N + i] = m[c];
            fa[i] = {Real(0.5), 0};           // half the sum of (1 -+ a)/2
            fa[N + i] = {x / 2, Real(0.5)};   // half the difference
            fa[NM * N + i] = {1, 0};
            fb[NN * N + i] = {1, 0};
            jacobi_sweep(NM, 0, 0, x, p);
            for (int c = 0; c < NM; ++c) ra[c * N + i] = w[i] * p[c];
            for (int c = 0; c < NM; ++c) {
                // entries c, k with c + k < NM are the ones there are
                mod_b(c, NM - c, x, m);
                for (int k = 0; k < NM - c; ++k) fb[(c * NM + k) * N + i] = m[k];
                jacobi_sweep(NM - c, 2 * c + 1, 0, x, p);
                for (int k = 0; k < NM - c; ++k) rb[(c * NM + k) * N + i] = w[i] * ipow(h, c) * p[k];
                jacobi_sweep(NM - c, 2 * c + 2, 0, x, p);
                for (int k = 0; k < NM - c; ++k) rc[(c * NM + k) * N + i] = w[i] * ipow(h, c + 1) * p[k];
            }
        }
        for (size_t k = 0; k < fa.size(); ++k) wa.push_back(w[k % N] * fa[k].v);
        for (size_t k = 0; k < fb.size(); ++k) {
            const Real h = (1 - z[k % N]) / 2;
            wb.push_back(w[k % N] * h * fb[k].v);
            wc.push_back(w[k % N] * h * h * fb[k].v);
        }
    }
    // <row, d_0 col>, <row, (d_1 - d_0/2) col>, <row, (d_2 - d_0/2) col> with
    //   d_0 = A' B/h_b C/h_c,  d_1 - d_0/2 = a/2 d_0 + A B' C/h_c,
    //   d_2 - d_0/2 = a/2 d_0 + (1 + b)/2 A B' C/h_c + A B C'
    double grad(int m, int r, int c)
    {
        const Row &R = L::rows(L::row_odd(m))[r];
        const Col &C = L::cols(L::col_odd(m))[c];
        const int pq = R.p + R.q, ca = class_a(NM, C), cb = class_b(NM, C), cc = class_c(NM, C);
        const auto &A = ga.get(R.p, ca, [&] {  // A, A', a/2 A'
            std::array<Real, 3> s{};
            for (int i = 0; i < N; ++i) {
                const Real q = ra[R.p * N + i];
                const Val f = fa[ca * N + i];
                s[0] += q * f.v;
                s[1] += q * f.d;
                s[2] += q * z[i] / 2 * f.d;
            }
            return s;
        });
        const int kb = R.p * NM + R.q;
        const auto &B = gb.get(kb, cb, [&] {  // B/h_b, B', (1 + b)/2 B', B
            std::array<Real, 4> s{};
            for (int i = 0; i < N; ++i) {
                const Real q = rb[kb * N + i], h = (1 - z[i]) / 2;
                const Val f = fb[cb * N + i];
                s[0] += q * f.v;
                s[1] += q * h * f.d;
                s[2] += q * h * (1 + z[i]) / 2 * f.d;
                s[3] += q * h * f.v;
            }
            return s;
        });
        const int kc = pq * NM + R.r;
        const auto &G = gc.get(kc, cc, [&] {  // C/h_c, C'
            std::array<Real, 2> s{};
            for (int i = 0; i < N; ++i) {
                const Real q = rc[kc * N + i];
                const Val f = fb[cc * N + i];
                s[0] += q * f.v;
                s[1] += q * (1 - z[i]) / 2 * f.d;
            }
            return s;
        });
        const Real s = scale[L::row_odd(m)][r];
        if (m == G0E || m == G0O) return (double)(A[1] * B[0] * G[0] * s);
        if (m == G1E || m == G1O) return (double)((A[2] * B[0] + A[0] * B[1]) * G[0] * s);
        return (double)(((A[2] * B[0] + A[0] * B[2]) * G[0] + A[0] * B[3] * G[1]) * s);
    }
    double mass(bool odd, int r, int c)
    {
        const Col &X = L::cols(odd)[r], &Y = L::cols(odd)[c];
        const auto product = [&](Memo<1> &memo, const std::vector<Real> &fw, const std::vector<Val> &f, int x, int y) {
            return memo.get(x, y, [&] {
                std::array<Real, 1> s{};
                for (int i = 0; i < N; ++i) s[0] += fw[x * N + i] * f[y * N + i].v;
                return s;
            })[0];
        };
        return (double)(product(ma, wa, fa, class_a(NM, X), class_a(NM, Y)) *
                        product(mb, wb, fb, class_b(NM, X), class_b(NM, Y)) *
                        product(mc, wc, fb, class_c(NM, X), class_c(NM, Y)));
    }
};

template <int NM>
std::vector<double> build(bool fp32)
{
    using L = Layout<NM>;
    constexpr auto &plan = L::plan;
    Entries<NM> E;
    std::vector<double> gm[6], mm[2];
    for (int m = 0; m < 6; ++m) {
        const int nr = L::nrows(L::row_odd(m)), nc = L::ncols(L::col_odd(m));
        gm[m].assign((size_t)nr * nc, 0.0);
        for (int r = 0; r < nr; ++r)
            for (int c = 0; c < nc; ++c)
                if (L::grad_entry(m, L::rows(L::row_odd(m))[r], L::cols(L::col_odd(m))[c]))
                    gm[m][(size_t)r * nc + c] = E.grad(m, r, c);
    }
    for (int m = 0; m < 2; ++m) {
        const int nc = L::ncols(m);
        mm[m].assign((size_t)nc * nc, 0.0);
        for (int r = 0; r < nc; ++r)
            for (int c = 0; c <= r; ++c)
                if (L::mass_entry(L::cols(m)[r], L::cols(m)[c]))
                    mm[m][(size_t)r * nc + c] = mm[m][(size_t)c * nc + r] = E.mass(m, r, c);
    }
    const int vw = fp32 ? 4 : 2;
    std::vector<double> tab((size_t)plan.total * 64, 0.0);
    // lane l of block pos: row slot l % 16, column l / 16 of the block
    const auto put = [&](int pos, auto entry) {
        for (int l = 0; l < 64; ++l) {
            // (Mma::slot: register r of lane group g of a product holds row 4r + g)
            const int row = fp32 ? 4 * (l % 4) + l % 16 / 4 : l % 16;
            tab[((size_t)(pos / vw) * 64 + l) * vw + pos % vw] = entry(row, l / 16);
        }
    };
    for (int m = 0; m < 6; ++m) {
        const int nr = L::nrows(L::row_odd(m)), nc = L::ncols(L::col_odd(m));
        const auto at = [&](int r, int c) { return r < nr && c < nc ? gm[m][(size_t)r * nc + c] : 0.0; };
        for (int t = 0; t < L::MAXT; ++t)
            for (int s = 0; s < L::MAXS; ++s) {
                if (plan.b.fwd[m][t][s] >= 0)
                    put(plan.b.fwd[m][t][s], [&](int i, int k) { return at(16 * t + i, 4 * s + k); });
                if (plan.b.bwd[m][t][s] >= 0)
                    put(plan.b.bwd[m][t][s], [&](int i, int k) { return at(4 * s + k, 16 * t + i); });
            }
    }
    for (int m = 0; m < 2; ++m) {
        const int nc = L::ncols(m);
        for (int t = 0; t < L::MAXT; ++t)
            for (int s = 0; s < L::MAXS; ++s)
                if (plan.b.mass[m][t][s] >= 0)
                    put(plan.b.mass[m][t][s], [&](int i, int k) {
                        const int r = 16 * t + i, c = 4 * s + k;
                        return r < nc && c < nc ? mm[m][(size_t)r * nc + c] : 0.0;
                    });
    }
    return tab;
}

// Constant tables of the element type: built at the first operator of the
// kind (0.3 ms at NM = 7, 1.3 at 10), kept for the process (2.5 MB for all)
template <int NM, bool FP32>
const std::vector<double> &table()
{
    static const std::vector<double> t = build<NM>(FP32);
    return t;
}
template <int NM>
const std::vector<double> &table(bool fp32)
{
    return fp32 ? table<NM, true>() : table<NM, false>();
}

}  // namespace

const std::vector<double> &build_tables(int nm, bool fp32)
{
    switch (nm) {
    case 2: return table<2>(fp32);
    case 3: return table<3>(fp32);
    case 4: return table<4>(fp32);
    case 5: return table<5>(fp32);
    case 6: return table<6>(fp32);
    case 7: return table<7>(fp32);
    case 8: return table<8>(fp32);
    case 9: return table<9>(fp32);
    case 10: return table<10>(fp32);
    default: throw Error(NMF_ERR_UNSUPPORTED, "affine tet tables: modes out of range");
    }
}

}  // namespace tetmodal
}  // namespace nektar_amd
