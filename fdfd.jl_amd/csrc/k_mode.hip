// Batched 1-D eigenmodes for mode sources: eigenmode(d::Device{1}, pol,
// neff, nev) of src/solver/eigen.jl:6-29, called by get_modes / setup_mode!
// (src/device.jl:118-149) on a slice of eps.
//
// Operator of a slice of n cells (periodic, no PML; grid.jl:138,141):
//   TM: A = k0^2 diag(eps) + dxf dxb
//       A[i][i +- 1] = 1/dx^2, A[i][i] = k0^2 eps_i - 2/dx^2
//   TE: A = k0^2 diag(eps) + diag(eps) dxf diag(1/avg eps) dxb
//       A[i][i+1] = eps_i / (dx^2 a_{i+1}), A[i][i-1] = eps_i / (dx^2 a_i),
//       A[i][i] = k0^2 eps_i - A[i][i+1] - A[i][i-1],  a_i = (eps_i + eps_{i-1})/2
// (grid_average, grid.jl:157-158), k0^2 = omega^2 mu0' eps0'.
//
// Eigs with sigma (eigen.jl:26) is shift-invert Arnoldi on
// OP = (A - sigma I)^-1 keeping the nev Ritz values of largest magnitude,
// i.e. the eigenvalues nearest sigma.  One workgroup per problem:
//   * A - sigma I is factored once by Givens QR (tri_qr.h, one lane; the
//     operator is periodic tridiagonal, O(n)), and every OP application is
//     one O(n) solve on one wave (tri_solve);
//   * Arnoldi vectors live in global memory; CGS2 dot products (a wave takes
//     every fourth vector), updates and norms use the whole workgroup;
//   * the projected (ncv x ncv) eigenproblem runs on one wave from LDS
//     (wave_eig, the algorithm of small_eig.h);
//   * thick restart keeps the span of the `keep` wanted Ritz vectors.
// Slices are few and short, so the chain of one workgroup is the whole time: the
// recurrences take their operands from LDS and leave everything that is not a
// recurrence to the lanes.  64 slices of 51 cells, 20 applications: 0.65 ms
// (factorization 70 us, Gram-Schmidt 110, the rest applications and, the larger part,
// the eigenproblem), against 4.9 ms with recurrences and eigenproblem on one lane.
// Output: beta = sqrt(sigma + 1/theta) (principal branch, eigen.jl:28) nearest
// first, eigenvectors of unit 2-norm with their largest entry real > 0.
#include "fdfd_common.h"
#include "small_eig.h"
#include "tri_qr.h"

namespace fdfd {

namespace {

constexpr int MT = 256;       // threads per workgroup
constexpr int MW = MT / 64;   // waves per workgroup

using eig::cz;
using eig::mkz;

__device__ inline cz ld(const double2* p) {
    const double2 v = *p;
    return mkz(v.x, v.y);
}
__device__ inline void st(double2* p, cz v) { *p = make_double2(v.re, v.im); }

__device__ inline double wsum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// LDS written by lanes of this wave before is visible to its lanes after
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
__device__ inline double cabs1(cz a) { return fabs(a.re) + fabs(a.im); }
// lane l's value (l the same on every lane)
__device__ inline cz from_lane(cz a, int l) {
    auto get = [l](double v) {
        const long long b = __double_as_longlong(v);
        const unsigned lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
        return __longlong_as_double(((long long)hi << 32) | lo);
    };
    return mkz(get(a.re), get(a.im));
}
__device__ inline cz pick(bool c, cz a, cz b) { return mkz(c ? a.re : b.re, c ? a.im : b.im); }

// Rows of the factors for 64 steps of a recurrence
struct TriBuf {
    cz a[64][4];
};

// w = (R^-1 Q) v by one wave.  All lanes run the recurrences alike; lane r of a
// chunk of 64 rows loads row r, does its share that is no recurrence, and keeps
// its result.
__device__ inline void tri_solve(int n, const double* trw, const double2* v, double2* w, TriBuf& tb) {
    const int lane = threadIdx.x & 63;
    // y = Q v
    cz carry = ld(v), tail = ld(v + n - 1);
    for (int base = 0; base < n; base += 64) {
        const int cnt = min(64, n - base), k = base + min(lane, cnt - 1);
        double c1, c2;
        cz s1, s2, y = mkz(0, 0);
        tri::get_rot(trw, k, 0, c1, s1);
        tri::get_rot(trw, k, 1, c2, s2);
        const cz nx = ld(v + min(k + 1, n - 1));
        wave_sync();
        tb.a[lane][0] = s1;
        tb.a[lane][1] = s2;
        tb.a[lane][2] = mkz(c1, c2);
        tb.a[lane][3] = nx;
        wave_sync();
        const int main = min(cnt, n - 2 - base);
#pragma unroll 4
        for (int r = 0; r < main; ++r) {
            const cz f0 = tb.a[r][0], f1 = tb.a[r][1], f2 = tb.a[r][2];
            cz nxt = tb.a[r][3];
            tri::rot(f2.re, f0, carry, nxt);
            tri::rot(f2.im, f1, carry, tail);
            y = pick(lane == r, carry, y);
            carry = nxt;
        }
        for (int r = max(main, 0); r < cnt; ++r) {  // rows n - 2 and n - 1
            if (base + r + 2 == n) {
                tri::rot(tb.a[r][2].re, tb.a[r][0], carry, tail);
                y = pick(lane == r, carry, y);
            } else {
                y = pick(lane == r, tail, y);
            }
        }
        if (lane < cnt) st(w + base + lane, y);
    }
    __threadfence_block();
    // x = R^-1 y:  x_k = t_k - a1_k x_{k+1} - a2_k x_{k+2}, with
    // t = (y - r3 x_{n-2} - r4 x_{n-1}) / r0 and a = (r1, r2) / r0 by the lanes
    const cz xB = eig::zmul(ld(w + n - 1), tri::get_r(trw, n, n - 1, 0));
    const cz xA = eig::zmul(eig::zsub(ld(w + n - 2), eig::zmul(tri::get_r(trw, n, n - 2, 4), xB)),
                            tri::get_r(trw, n, n - 2, 0));
    cz x1 = xA, x2 = xB;
    for (int base = ((n - 1) / 64) * 64; base >= 0; base -= 64) {
        const int cnt = min(64, n - base), k = base + min(lane, cnt - 1);
        const cz ri = tri::get_r(trw, n, k, 0);
        cz y = eig::zsub(ld(w + k), eig::zmul(tri::get_r(trw, n, k, 3), xA));
        y = eig::zmul(eig::zsub(y, eig::zmul(tri::get_r(trw, n, k, 4), xB)), ri);
        cz x = pick(k == n - 1, xB, xA);
        wave_sync();
        tb.a[lane][0] = y;
        tb.a[lane][1] = eig::zmul(tri::get_r(trw, n, k, 1), ri);
        tb.a[lane][2] = eig::zmul(tri::get_r(trw, n, k, 2), ri);
        wave_sync();
        const int top = min(cnt - 1, n - 3 - base);
#pragma unroll 4
        for (int r = top; r >= 0; --r) {
            const cz xk = eig::zsub(eig::zsub(tb.a[r][0], eig::zmul(tb.a[r][2], x2)), eig::zmul(tb.a[r][1], x1));
            x = pick(lane == r, xk, x);
            x2 = x1;
            x1 = xk;
        }
        if (lane < cnt) st(w + base + lane, x);
    }
}

constexpr int LD = MODE_NCV + 1;  // row stride of the small matrices (no two rows share a bank)

// Givens rotation from squared magnitudes (hypot, for the ranges where these
// could leave the exponent's, in tri_qr.h)
__device__ inline void wave_givens(cz x, cz y, double& c, cz& s) {
    const double nx = eig::znorm2(x), ny = eig::znorm2(y), t = nx + ny;
    if (nx > 1e-140 && t < 1e140) {
        const double rx = rsqrt(nx), rt = rsqrt(t), q = rx * rt;
        c = nx * q;
        s = eig::zscale(eig::zmul(x, eig::zconj(y)), q);
        return;
    }
    cz r;
    eig::qr_givens(x, y, c, s, r);
}

// small_eig (small_eig.h) by one wave: A (destroyed), Q and Y are n x n with row
// stride LD, v holds n.  Lane j takes column j of a row operation; lanes 0 .. 31 take
// row i of A and lanes 32 .. 63 row i of Q of a column operation; each lane
// back-substitutes its own eigenvector.  Control flow is the same on every lane.
__device__ inline int wave_eig(int n, cz* A, cz* Q, cz* evals, cz* Y, cz* v) {
    const int lane = threadIdx.x & 63, row = lane & 31;
    const bool on = row < n;
    cz* M = (lane < 32 ? A : Q) + min(row, n - 1) * LD;  // this lane's row of A or Q
    auto a = [&](int i, int j) -> cz& { return A[i * LD + j]; };
    for (int e = lane; e < n * n; e += 64) Q[(e / n) * LD + e % n] = mkz(e / n == e % n ? 1.0 : 0.0, 0);
    wave_sync();
    // Hessenberg reduction
    for (int k = 0; k + 2 < n; ++k) {
        const bool in = lane > k && lane < n;
        cz x = in ? a(lane, k) : mkz(0, 0);
        const double nx = sqrt(wsum(eig::znorm2(x)));
        if (nx == 0) continue;
        const cz x0 = a(k + 1, k);
        const double a0 = eig::zmag(x0);
        const cz alpha = a0 > 0 ? eig::zscale(x0, -nx / a0) : mkz(-nx, 0);
        if (lane == k + 1) x = eig::zsub(x, alpha);
        const double vn = sqrt(wsum(eig::znorm2(x)));
        if (vn == 0) continue;
        if (lane < n) v[lane] = eig::zscale(x, 1.0 / vn);
        wave_sync();
        if (lane < n) {
            cz s = mkz(0, 0);
            for (int i = k + 1; i < n; ++i) s = eig::zadd(s, eig::zmul(eig::zconj(v[i]), a(i, lane)));
            for (int i = k + 1; i < n; ++i) a(i, lane) = eig::zsub(a(i, lane), eig::zscale(eig::zmul(v[i], s), 2.0));
        }
        wave_sync();
        if (on) {
            cz s = mkz(0, 0);
            for (int j = k + 1; j < n; ++j) s = eig::zadd(s, eig::zmul(M[j], v[j]));
            for (int j = k + 1; j < n; ++j) M[j] = eig::zsub(M[j], eig::zscale(eig::zmul(s, eig::zconj(v[j])), 2.0));
        }
        wave_sync();
        if (lane > k + 1 && lane < n) a(lane, k) = mkz(0, 0);
        wave_sync();
    }
    // shifted QR iterations
    const double eps = 2.220446049250313e-16;
    int hi = n - 1, iter = 0, total = 0;
    while (hi > 0) {
        bool small = lane == 0;
        if (lane > 0 && lane <= hi) {
            double s = cabs1(a(lane - 1, lane - 1)) + cabs1(a(lane, lane));
            if (s == 0) s = 1;
            small = cabs1(a(lane, lane - 1)) <= eps * s;
        }
        const int l = 63 - __builtin_clzll(__ballot(small));
        if (l > 0 && lane == 0) a(l, l - 1) = mkz(0, 0);
        wave_sync();
        if (l == hi) {
            --hi;
            iter = 0;
            continue;
        }
        if (++total > 100 * n) return -1;
        const cz p = a(hi - 1, hi - 1), b = a(hi - 1, hi), c = a(hi, hi - 1), d = a(hi, hi);
        cz mu;
        if (iter > 0 && iter % 11 == 0) {
            mu = eig::zadd(d, mkz(eig::zmag(c), 0));  // exceptional shift
        } else {
            const cz pmd = eig::zsub(p, d);
            const cz disc = eig::zsqrt(eig::zadd(eig::zscale(eig::zmul(pmd, pmd), 0.25), eig::zmul(b, c)));
            const cz half = eig::zscale(eig::zadd(p, d), 0.5);
            const cz m1 = eig::zadd(half, disc), m2 = eig::zsub(half, disc);
            mu = eig::znorm2(eig::zsub(m1, d)) < eig::znorm2(eig::zsub(m2, d)) ? m1 : m2;
        }
        ++iter;
        cz x = eig::zsub(a(l, l), mu), y = a(l + 1, l);
        for (int k = l; k < hi; ++k) {
            double cs;
            cz sn;
            wave_givens(x, y, cs, sn);
            if (lane >= (k == l ? l : k - 1) && lane < n) {
                const cz e = a(k, lane), f = a(k + 1, lane);
                a(k, lane) = eig::zadd(eig::zscale(e, cs), eig::zmul(sn, f));
                a(k + 1, lane) = (k > l && lane == k - 1) ? mkz(0, 0)
                                                          : eig::zsub(eig::zscale(f, cs), eig::zmul(eig::zconj(sn), e));
            }
            wave_sync();
            cz e = mkz(0, 0);
            if (on && (lane >= 32 || row <= min(k + 2, hi))) {
                e = M[k];
                const cz f = M[k + 1], g = e;
                e = eig::zadd(eig::zscale(e, cs), eig::zmul(f, eig::zconj(sn)));
                M[k] = e;
                M[k + 1] = eig::zsub(eig::zscale(f, cs), eig::zmul(g, sn));
            }
            wave_sync();
            // the bulge for the next step: entries (k + 1, k) and (k + 2, k)
            x = from_lane(e, k + 1);
            y = from_lane(e, min(k + 2, hi));
        }
    }
    if (lane < n) evals[lane] = a(lane, lane);
    // eigenvectors of T, lane k the one of T[k][k], then Q z
    double tn = 0;
    if (lane < n)
        for (int i = 0; i <= lane; ++i) tn = fmax(tn, eig::zmag(a(i, lane)));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) tn = fmax(tn, __shfl_xor(tn, o, 64));
    const double tiny = eps * (tn > 1e-300 ? tn : 1e-300);
    wave_sync();
    if (lane < n) {
        const cz ev = evals[lane];
        Y[lane * LD + lane] = mkz(1, 0);
        for (int i = lane - 1; i >= 0; --i) {
            cz s = mkz(0, 0);
            for (int j = i + 1; j <= lane; ++j) s = eig::zadd(s, eig::zmul(a(i, j), Y[j * LD + lane]));
            cz den = eig::zsub(a(i, i), ev);
            if (eig::zmag(den) < tiny) den = mkz(tiny, 0);
            Y[i * LD + lane] = eig::zscale(eig::zdiv(s, den), -1.0);
        }
    }
    wave_sync();  // T is read; its column takes the product
    if (lane < n) {
        double nz = 0;
        for (int i = 0; i < n; ++i) {
            cz s = mkz(0, 0);
            for (int j = 0; j <= lane; ++j) s = eig::zadd(s, eig::zmul(Q[i * LD + j], Y[j * LD + lane]));
            a(i, lane) = s;
            nz += eig::znorm2(s);
        }
        nz = 1.0 / sqrt(nz);
        for (int i = 0; i < n; ++i) Y[i * LD + lane] = eig::zscale(a(i, lane), nz);
    }
    wave_sync();
    return 0;
}

}  // namespace

__global__ __launch_bounds__(MT) void k_mode(const ModeJob* jobs, int nev, double tol,
                                             int maxiter) {
    const ModeJob J = jobs[blockIdx.x];
    const int n = J.n, t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int m = J.ncv;
    __shared__ cz H[(MODE_NCV + 1) * MODE_NCV];  // (m + 1) x m, row-major
    // row stride LD: wave_eig's input, then Qk (m x keep); its Q, then H Qk; Ritz
    // vectors of the projected matrix.  The factorization's coefficients before.
    __shared__ cz S[3][MODE_NCV * LD];
    cz *S0 = S[0], *S1 = S[1], *Y = S[2];
    __shared__ cz theta[MODE_NCV], vs[MODE_NCV + 1];
    __shared__ TriBuf tb;
    __shared__ cz hc[MODE_NCV + 1];
    __shared__ double rre[MW];
    __shared__ double rmag[MW];
    __shared__ int ridx[MW];
    __shared__ int order[MODE_NCV];
    __shared__ int flag[4];  // status, nconv, done, restarts
    const int keep = min(m - 1, nev + max(2, (m - nev) / 2));
    auto vp = [&](int q) { return J.V + (size_t)q * n; };

    // out[q] = V_q^H w for q < cnt (all threads; out valid after return)
    auto dots = [&](int cnt, const double2* w, cz* out) {
        constexpr int QW = (MODE_NCV + MW - 1) / MW;  // vectors of a wave: wv, wv + MW, ..
        double sr[QW], si[QW];
#pragma unroll
        for (int u = 0; u < QW; ++u) sr[u] = si[u] = 0;
        for (int i = lane; i < n; i += 64) {
            const double2 b = w[i];
#pragma unroll
            for (int u = 0; u < QW; ++u) {
                if (wv + MW * u < cnt) {
                    const double2 a = vp(wv + MW * u)[i];
                    sr[u] += a.x * b.x + a.y * b.y;
                    si[u] += a.x * b.y - a.y * b.x;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < QW; ++u) {
            if (wv + MW * u < cnt) {
                const double re = wsum(sr[u]), im = wsum(si[u]);
                if (lane == 0) out[wv + MW * u] = mkz(re, im);
            }
        }
        __syncthreads();
    };
    // w -= sum_q V_q c[q]
    auto update = [&](int cnt, double2* w, const cz* c) {
        for (int i = t; i < n; i += MT) {
            double xr = w[i].x, xi = w[i].y;
            for (int q = 0; q < cnt; ++q) {
                const double2 a = vp(q)[i];
                xr -= a.x * c[q].re - a.y * c[q].im;
                xi -= a.x * c[q].im + a.y * c[q].re;
            }
            w[i] = make_double2(xr, xi);
        }
        __syncthreads();
    };
    auto norm = [&](const double2* w) -> double {
        double s = 0;
        for (int i = t; i < n; i += MT) s += w[i].x * w[i].x + w[i].y * w[i].y;
        s = wsum(s);
        if (lane == 0) rre[wv] = s;
        __syncthreads();
        double tot = 0;
        for (int k = 0; k < MW; ++k) tot += rre[k];
        __syncthreads();
        return sqrt(tot);
    };
    auto scale = [&](double2* w, cz a) {
        for (int i = t; i < n; i += MT) {
            const double2 x = w[i];
            w[i] = make_double2(x.x * a.re - x.y * a.im, x.x * a.im + x.y * a.re);
        }
        __syncthreads();
    };
    int applies = 0;
    // w = OP v
    auto op = [&](const double2* v, double2* w) {
        if (wv == 0) tri_solve(n, J.trw, v, w, tb);
        ++applies;
        __syncthreads();
    };

    // ---- factor A - sigma I (one lane) and the start vector --------------
    {
        const cz sg = mkz(J.sigma.x, J.sigma.y);
        auto row = [&](int i, cz& d, cz& e, cz& f) {
            const cz ei = ld(J.eps + i);
            const cz k2e = eig::zscale(ei, J.k0sq);
            if (J.pol == 1) {
                e = mkz(J.idx2, 0);
                f = mkz(J.idx2, 0);
            } else {
                const cz em = ld(J.eps + (i + n - 1) % n), ep = ld(J.eps + (i + 1) % n);
                const cz a_i = eig::zscale(eig::zadd(ei, em), 0.5);
                const cz a_ip = eig::zscale(eig::zadd(ep, ei), 0.5);
                e = eig::zscale(eig::zdiv(ei, a_ip), J.idx2);
                f = eig::zscale(eig::zdiv(ei, a_i), J.idx2);
            }
            d = eig::zsub(eig::zsub(eig::zsub(k2e, e), f), sg);
        };
        // the rows of a slice that fits the small matrices are formed by all lanes
        cz* rows = &S[0][0];
        const bool fits = 3 * n <= 3 * MODE_NCV * LD;
        if (fits) {
            for (int i = t; i < n; i += MT) row(i, rows[3 * i], rows[3 * i + 1], rows[3 * i + 2]);
            __syncthreads();
        }
        auto coef = [&](int i, cz& d, cz& e, cz& f) {
            if (fits) {
                d = rows[3 * i];
                e = rows[3 * i + 1];
                f = rows[3 * i + 2];
            } else {
                row(i, d, e, f);
            }
        };
        if (t == 0) {
            double pmin, pmax;
            const int rc = tri::factor(n, coef, J.trw, pmin, pmax);
            flag[0] = rc ? MODE_SINGULAR : MODE_OK;
            flag[1] = 0;
            flag[2] = 0;
            flag[3] = 0;
            // deterministic start vector (xorshift64)
            unsigned long long s = 0x9e3779b97f4a7c15ULL;
            double2* v0 = vp(0);
            for (int i = 0; i < n; ++i) {
                s ^= s << 13; s ^= s >> 7; s ^= s << 17;
                const double a = (double)(s >> 11) / 9007199254740992.0 - 0.5;
                s ^= s << 13; s ^= s >> 7; s ^= s << 17;
                const double b = (double)(s >> 11) / 9007199254740992.0 - 0.5;
                v0[i] = make_double2(a, b);
            }
        }
    }
    __syncthreads();
    if (flag[0] != MODE_OK) {
        if (t == 0) {
            J.info[0] = flag[0];
            J.info[1] = 0;
            J.info[2] = 0;
            J.info[3] = 0;
        }
        return;  // uniform: every thread read the same flag
    }
    {
        const double nv = norm(vp(0));
        scale(vp(0), mkz(1.0 / nv, 0));
    }
    for (int i = t; i < (m + 1) * m; i += MT) H[i] = mkz(0, 0);
    __syncthreads();

    // ---- thick-restart Arnoldi -------------------------------------------
    int start = 0;
    for (;;) {
        for (int j = start; j < m; ++j) {
            double2* w = vp(j + 1);
            op(vp(j), w);
            dots(j + 1, w, hc);
            if (t <= j) H[t * m + j] = hc[t];
            __syncthreads();
            update(j + 1, w, hc);
            dots(j + 1, w, hc);
            if (t <= j) H[t * m + j] = eig::zadd(H[t * m + j], hc[t]);
            __syncthreads();
            update(j + 1, w, hc);
            const double hn = norm(w);
            if (t == 0) H[(j + 1) * m + j] = mkz(hn, 0);
            if (hn > 0) scale(w, mkz(1.0 / hn, 0));
            __syncthreads();
        }
        for (int e = t; e < m * m; e += MT) S0[(e / m) * LD + e % m] = H[e];
        __syncthreads();
        if (wv == 0) {
            if (wave_eig(m, S0, S1, theta, Y, vs)) {
                if (lane == 0) {
                    flag[0] = MODE_EIG_FAIL;
                    flag[2] = 1;
                }
            } else {
                // order by |theta| descending, equal ones as they come
                if (lane < m) order[lane] = lane;
                wave_sync();
                if (lane < m) {
                    const double ai = eig::zmag(theta[lane]);
                    int rank = 0;
                    for (int k = 0; k < m; ++k) {
                        const double ak = eig::zmag(theta[k]);
                        rank += ak > ai || (ak == ai && k < lane);
                    }
                    if (ai == ai) order[rank] = lane;
                }
                wave_sync();
                // residual of Ritz pair i: |H[m, :] y_i|
                bool conv = false;
                if (lane < nev) {
                    const int i = order[lane];
                    cz r = mkz(0, 0);
                    for (int k = 0; k < m; ++k) r = eig::zadd(r, eig::zmul(H[m * m + k], Y[k * LD + i]));
                    conv = eig::zmag(r) <= tol * eig::zmag(theta[i]);
                }
                const int nc = __popcll(__ballot(conv));
                if (lane == 0) {
                    flag[1] = nc;
                    flag[2] = (nc >= nev || flag[3] >= maxiter) ? 1 : 0;
                }
            }
        }
        __syncthreads();
        if (flag[2]) break;
        // restart: Qk = orthonormal basis of the keep wanted Ritz vectors
        if (wv == 0) {
            if (lane == 0) flag[3] += 1;
            for (int q = 0; q < keep; ++q) {
                cz x = lane < m ? Y[lane * LD + order[q]] : mkz(0, 0);
                for (int pass = 0; pass < 2; ++pass)
                    for (int p = 0; p < q; ++p) {
                        const cz b = lane < m ? S0[lane * LD + p] : mkz(0, 0);
                        const cz g = eig::zmul(eig::zconj(b), x);
                        x = eig::zsub(x, eig::zmul(mkz(wsum(g.re), wsum(g.im)), b));
                    }
                const double nq = sqrt(wsum(eig::znorm2(x)));
                if (lane < m) S0[lane * LD + q] = eig::zscale(x, 1.0 / nq);
                wave_sync();
            }
        }
        __syncthreads();
        // W[:, q] = V_m Qk[:, q]
        for (int q = wv; q < keep; q += MW)
            for (int i = lane; i < n; i += 64) {
                double xr = 0, xi = 0;
                for (int k = 0; k < m; ++k) {
                    const double2 a = vp(k)[i];
                    const cz c = S0[k * LD + q];
                    xr += a.x * c.re - a.y * c.im;
                    xi += a.x * c.im + a.y * c.re;
                }
                J.W[(size_t)q * n + i] = make_double2(xr, xi);
            }
        __syncthreads();
        // v_keep = v_m, then V[:, 0:keep] = W
        for (int i = t; i < n; i += MT) vp(keep)[i] = vp(m)[i];
        __syncthreads();
        for (int i = t; i < n; i += MT)
            for (int q = 0; q < keep; ++q) vp(q)[i] = J.W[(size_t)q * n + i];
        // H_new = Qk^H H_m Qk, row keep = H[m, :] Qk
        for (int e = t; e < (m + 1) * keep; e += MT) {
            const int i = e / keep, q = e % keep;
            cz s = mkz(0, 0);
            for (int k = 0; k < m; ++k) s = eig::zadd(s, eig::zmul(H[i * m + k], S0[k * LD + q]));
            if (i < m) S1[i * LD + q] = s;
            else vs[q] = s;
        }
        __syncthreads();
        for (int e = t; e < (m + 1) * m; e += MT) {
            const int p = e / m, q = e % m;
            cz s = mkz(0, 0);
            if (p < keep && q < keep)
                for (int i = 0; i < m; ++i)
                    s = eig::zadd(s, eig::zmul(eig::zconj(S0[i * LD + p]), S1[i * LD + q]));
            else if (p == keep && q < keep)
                s = vs[q];
            H[e] = s;
        }
        __syncthreads();
        start = keep;
    }

    // ---- outputs ------------------------------------------------------------
    const bool ok = flag[0] == MODE_OK;
    if (ok) {
        for (int q = 0; q < nev; ++q) {
            const int sel = order[q];
            double2* x = J.vec + (size_t)q * n;
            for (int i = t; i < n; i += MT) {
                double xr = 0, xi = 0;
                for (int k = 0; k < m; ++k) {
                    const double2 a = vp(k)[i];
                    const cz c = Y[k * LD + sel];
                    xr += a.x * c.re - a.y * c.im;
                    xi += a.x * c.im + a.y * c.re;
                }
                x[i] = make_double2(xr, xi);
            }
            __syncthreads();
            // largest entry (lowest index among equals) and the 2-norm
            double best = -1, s2 = 0;
            int bi = 0;
            for (int i = t; i < n; i += MT) {
                const double a2 = x[i].x * x[i].x + x[i].y * x[i].y;
                s2 += a2;
                if (a2 > best) {
                    best = a2;
                    bi = i;
                }
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                const double ob = __shfl_xor(best, o, 64);
                const int oi = __shfl_xor(bi, o, 64);
                if (ob > best || (ob == best && oi < bi)) {
                    best = ob;
                    bi = oi;
                }
            }
            s2 = wsum(s2);
            if (lane == 0) {
                rmag[wv] = best;
                ridx[wv] = bi;
                rre[wv] = s2;
            }
            __syncthreads();
            double gb = rmag[0], tot = 0;
            int gi = ridx[0];
            for (int k = 0; k < MW; ++k) {
                tot += rre[k];
                if (rmag[k] > gb || (rmag[k] == gb && ridx[k] < gi)) {
                    gb = rmag[k];
                    gi = ridx[k];
                }
            }
            const cz ph = ld(x + gi);
            const double pm = eig::zmag(ph);
            __syncthreads();
            const cz a = eig::zscale(eig::zconj(ph), 1.0 / (pm * sqrt(tot)));
            scale(x, a);
            if (t == 0) {
                const cz lam = eig::zadd(mkz(J.sigma.x, J.sigma.y), tri::zinv(theta[sel]));
                st(J.beta + q, eig::zsqrt(lam));
            }
        }
    }
    if (t == 0) {
        J.info[0] = flag[0];
        J.info[1] = ok ? flag[1] : 0;
        J.info[2] = flag[3];
        J.info[3] = applies;
    }
}

void launch_mode(hipStream_t s, const ModeJob* jobs_d, int njobs, int nev, double tol,
                 int maxiter) {
    k_mode<<<njobs, MT, 0, s>>>(jobs_d, nev, tol, maxiter);
}

}  // namespace fdfd
