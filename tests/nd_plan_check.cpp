// CPU check of the nested-dissection plan (nd_plan.h): the tree is executed
// with dense complex<double> fronts, following the gather semantics of the
// device kernels, on random complex symmetric periodic 5-point operators.
// Prints one line per grid: every cell is eliminated exactly once, every
// child boundary cell appears in its parent's front, and the solve of
// A x = b reaches a relative residual below 1e-10 (a dropped, doubled or
// misplaced coupling fails by orders of magnitude).
#include <cmath>
#include <complex>
#include <cstdio>
#include <random>
#include <vector>

#include "nd_plan.h"

using namespace fdfd::nd;
using cd = std::complex<double>;

static bool run(int Nx, int Ny) {
    const int N = Nx * Ny;
    std::mt19937_64 rng(17 * Nx + Ny);
    std::uniform_real_distribution<double> u(-1, 1);
    std::vector<cd> C(N), E(N), T(N), rhs(N);  // diagonal, coupling to x + 1, to y + 1
    for (int k = 0; k < N; ++k) {
        C[k] = cd(-3.6 + 0.4 * u(rng), 0.3 * u(rng));
        E[k] = cd(1 + 0.2 * u(rng), 0.2 * u(rng));
        T[k] = cd(1 + 0.2 * u(rng), 0.2 * u(rng));
        rhs[k] = cd(u(rng), u(rng));
    }
    auto east = [&](int k) { return k % Nx + 1 == Nx ? k - Nx + 1 : k + 1; };
    auto north = [&](int k) { return k / Nx + 1 == Ny ? k % Nx : k + Nx; };
    auto orig = [&](int k, int l) {
        cd v = 0;
        if (k == l) v += C[k];
        if (l == east(k)) v += E[k];
        if (k == east(l)) v += E[l];
        if (l == north(k)) v += T[k];
        if (k == north(l)) v += T[l];
        return v;
    };
    const std::vector<Level> L = make_plan(Nx, Ny);
    const int nl = (int)L.size();
    std::vector<int> seen(N, 0);
    bool ok = true;
    struct Front {
        std::vector<cd> X, Q, S;  // p x p, p x b, b x b
        std::vector<cd> v, u;     // solve: separator values, boundary updates
    };
    std::vector<std::vector<Front>> F(nl);
    auto node = [&](const Level& l, const Box& b, int i) {
        return i < l.p ? sep_node(l.kind, b, i, Nx) : bnd_node(b, l.wrapx, l.wrapy, i - l.p, Nx, Ny);
    };
    for (int li = nl - 1; li >= 0; --li) {
        const Level& l = L[li];
        const int p = l.p, b = l.b, f = p + b;
        F[li].resize(l.box.size());
        for (size_t fi = 0; fi < l.box.size(); ++fi) {
            Front& fr = F[li][fi];
            std::vector<int> nd(f);
            for (int i = 0; i < f; ++i) nd[i] = node(l, l.box[fi], i);
            for (int i = 0; i < p; ++i)
                if (nd[i] >= 0) ++seen[nd[i]];
            std::vector<cd> A((size_t)f * f, 0.0);
            std::vector<int> m[2];
            for (int c = 0; c < l.nch; ++c) {
                const Level& lc = L[li + 1];
                const Box& cb = lc.box[l.nch * fi + c];
                m[c].resize(f);
                int hits = 0;
                for (int i = 0; i < f; ++i) {
                    m[c][i] = bnd_pos(cb, lc.wrapx, lc.wrapy, nd[i], Nx, Ny);
                    if (m[c][i] >= 0) {
                        ++hits;
                        if (bnd_node(cb, lc.wrapx, lc.wrapy, m[c][i], Nx, Ny) != nd[i]) ok = false;
                    }
                }
                if (hits != bnd_count(cb, lc.wrapx, lc.wrapy, Nx, Ny)) ok = false;
            }
            for (int i = 0; i < f; ++i)
                for (int j = 0; j < f; ++j) {
                    cd v = 0;
                    if (nd[i] < 0 || nd[j] < 0) v = i == j && i < p ? 1.0 : 0.0;
                    else {
                        if (i < p || j < p) v = orig(nd[i], nd[j]);
                        for (int c = 0; c < l.nch; ++c)
                            if (m[c][i] >= 0 && m[c][j] >= 0)
                                v += F[li + 1][l.nch * fi + c].S[(size_t)m[c][i] * L[li + 1].b + m[c][j]];
                    }
                    A[(size_t)i * f + j] = v;
                }
            // in-place sweep of the separator
            for (int k = 0; k < p; ++k) {
                const cd r = 1.0 / A[(size_t)k * f + k];
                for (int i = 0; i < f; ++i)
                    if (i != k)
                        for (int j = 0; j < f; ++j)
                            if (j != k) A[(size_t)i * f + j] -= A[(size_t)i * f + k] * r * A[(size_t)k * f + j];
                for (int j = 0; j < f; ++j)
                    if (j != k) {
                        A[(size_t)k * f + j] *= r;
                        A[(size_t)j * f + k] *= -r;
                    }
                A[(size_t)k * f + k] = r;
            }
            fr.X.resize((size_t)p * p);
            fr.Q.resize((size_t)p * b);
            fr.S.resize((size_t)b * b);
            for (int i = 0; i < f; ++i)
                for (int j = 0; j < f; ++j) {
                    if (i < p && j < p) fr.X[(size_t)i * p + j] = A[(size_t)i * f + j];
                    if (i < p && j >= p) fr.Q[(size_t)i * b + j - p] = A[(size_t)i * f + j];
                    if (i >= p && j >= p) fr.S[(size_t)(i - p) * b + j - p] = A[(size_t)i * f + j];
                }
        }
    }
    for (int k = 0; k < N; ++k)
        if (seen[k] != 1) ok = false;
    // solve: child updates gathered up the tree, then down
    std::vector<cd> x(N, 0.0);
    for (int li = nl - 1; li >= 0; --li) {
        const Level& l = L[li];
        for (size_t fi = 0; fi < l.box.size(); ++fi) {
            Front& fr = F[li][fi];
            fr.v.assign(l.p, 0.0);
            fr.u.assign(l.b, 0.0);
            for (int i = 0; i < l.p + l.b; ++i) {
                const int k = node(l, l.box[fi], i);
                if (k < 0) continue;
                cd v = i < l.p ? rhs[k] : cd(0);
                for (int c = 0; c < l.nch; ++c) {
                    const Level& lc = L[li + 1];
                    const int mm = bnd_pos(lc.box[l.nch * fi + c], lc.wrapx, lc.wrapy, k, Nx, Ny);
                    if (mm >= 0) v += F[li + 1][l.nch * fi + c].u[mm];
                }
                (i < l.p ? fr.v[i] : fr.u[i - l.p]) = v;
            }
            for (int j = 0; j < l.b; ++j)
                for (int i = 0; i < l.p; ++i) fr.u[j] -= fr.Q[(size_t)i * l.b + j] * fr.v[i];
        }
    }
    for (int li = 0; li < nl; ++li) {
        const Level& l = L[li];
        for (size_t fi = 0; fi < l.box.size(); ++fi) {
            const Front& fr = F[li][fi];
            for (int i = 0; i < l.p; ++i) {
                cd v = 0;
                for (int k = 0; k < l.p; ++k) v += fr.X[(size_t)i * l.p + k] * fr.v[k];
                for (int j = 0; j < l.b; ++j) {
                    const int k = node(l, l.box[fi], l.p + j);
                    if (k >= 0) v -= fr.Q[(size_t)i * l.b + j] * x[k];
                }
                const int k = node(l, l.box[fi], i);
                if (k >= 0) x[k] = v;
            }
        }
    }
    double rn = 0, bn = 0;
    for (int k = 0; k < N; ++k) {
        cd r = rhs[k] - C[k] * x[k] - E[k] * x[east(k)] - T[k] * x[north(k)];
        const int w = k % Nx == 0 ? k + Nx - 1 : k - 1, s = k < Nx ? k + N - Nx : k - Nx;
        r -= E[w] * x[w] + T[s] * x[s];
        rn += std::norm(r);
        bn += std::norm(rhs[k]);
    }
    const double rel = std::sqrt(rn / bn);
    ok = ok && rel < 1e-10;
    printf("%s %d x %d: levels %d, residual %.2e\n", ok ? "OK" : "FAIL", Nx, Ny, nl, rel);
    return ok;
}

int main() {
    const int s[][2] = {{4, 4},   {5, 4},   {4, 7},   {8, 8},   {16, 16}, {17, 16}, {13, 29}, {24, 20},
                        {37, 41}, {40, 16}, {16, 90}, {64, 48}, {45, 61}, {23, 100}, {70, 33}, {18, 18}};
    bool ok = true;
    for (auto& q : s) ok = run(q[0], q[1]) && ok;
    return ok ? 0 : 1;
}
