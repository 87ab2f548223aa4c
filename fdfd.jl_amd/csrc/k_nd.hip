// Nested-dissection kernels of libfdfd (gfx950).
//
// The fronts of a tree level (nd_plan.h) form one batch: front f of factor q
// has a separator of p cells and a boundary of b cells (padded sizes of the
// level).  With the operator symmetrised (S = U^-1 A' U, see k_nd_coef), a
// front is F = [F11 F12; F12^T F22]; eliminating the separator leaves
//   X = F11^-1,   Q = X F12,   F22 - F12^T Q
// and the last block is gathered into the parent's front.  X and Q are the
// factor; the reduced solve sends boundary updates up the tree
// (u = u_children - Q^T v) and values down (x = X v - Q x_boundary).
// Every gather follows index maps, so no atomics are needed and results do
// not depend on scheduling.
#include "fdfd_common.h"
#include "k_device.h"
#include "nd_dev.h"

#include <algorithm>

namespace fdfd {

using namespace nd;

// Factors are complex128 for both precision options of the interface: the
// boxes of a tree come close to resonance here and there, and where the
// eigenvalue gap of a box is delta, its Schur complement grows by about
// 1 / delta and loses as many digits.  Over the million cells of a 1024^2
// grid growths of 1e4 .. 1e5 are ordinary, which FP64 carries (one or two
// refinement steps) and FP32 does not: with complex64 fronts the factorization
// took 14 instead of 22 ms at 1024^2, but the refinement 5 to 16 iterations
// (7 .. 21 ms) instead of 2 (3 ms), and some wavelengths of a sweep did not
// converge.
using R = double;
using C = cplx<R>;

// ---------------------------------------------------------------------------
// Index maps of a level: the cell of every front index and its position in
// the boundary of each child (-1: none).
// ---------------------------------------------------------------------------
__global__ void k_nd_maps(NdMapArgs a, int* node, short* cm) {
    const int f = a.p + a.b;
    const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (e >= (long)a.cnt * f) return;
    const int fr = (int)(e / f), i = (int)(e % f);
    const Box bx = a.box[fr];
    const int k = i < a.p ? sep_node(a.kind, bx, i, a.Nx)
                          : bnd_node(bx, a.wrapx, a.wrapy, i - a.p, a.Nx, a.Ny);
    node[e] = k;
    for (int c = 0; c < 2; ++c) {
        int m = -1;
        if (c < a.nch) m = bnd_pos(a.cbox[(long)a.nch * fr + c], a.cwrapx, a.cwrapy, k, a.Nx, a.Ny);
        cm[((long)fr * 2 + c) * f + i] = (short)m;
    }
}

void launch_nd_maps(hipStream_t s, const NdMapArgs& a, int* node, short* cm) {
    const long n = (long)a.cnt * (a.p + a.b);
    k_nd_maps<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(a, node, cm);
}

// ---------------------------------------------------------------------------
// Symmetrisation.  With the periodic differences A'^T = W^-1 A' W for the
// diagonal W = wx (x) wy, so S = U^-1 A' U with U = W^(1/2) is symmetric.
// k_nd_u stores ux = sqrt(wx), 1 / ux, uy, 1 / uy; k_nd_coef scales the
// couplings to x + 1 and y + 1 in place: S[k, l] = A'[k, l] u_l / u_k.
// ---------------------------------------------------------------------------
__device__ inline double2 csqrt_d(double2 z) {
    const double r = hypot(z.x, z.y);
    double a = sqrt(0.5 * (r + fabs(z.x)));
    if (a == 0.0) return make_double2(0, 0);
    const double b = 0.5 * z.y / a;
    return z.x >= 0 ? make_double2(a, b) : make_double2(fabs(b), z.y >= 0 ? a : -a);
}

__global__ void k_nd_u(double2* us, const double2* wx, const double2* wy, int Nx, int Ny) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < Nx) {
        const double2 u = csqrt_d(wx[t]);
        us[t] = u;
        us[Nx + t] = crcp(u);
    } else if (t < Nx + Ny) {
        const double2 u = csqrt_d(wy[t - Nx]);
        us[2 * Nx + t - Nx] = u;
        us[2 * Nx + Ny + t - Nx] = crcp(u);
    }
}

__global__ void k_nd_coef(double2* coef, const double2* us, int Nx, int Ny) {
    const long N = (long)Nx * Ny, k = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (k >= N) return;
    const int x = (int)(k % Nx), y = (int)(k / Nx);
    const double2 *ux = us, *uxi = us + Nx, *uy = us + 2 * Nx, *uyi = uy + Ny;
    const int xe = x + 1 == Nx ? 0 : x + 1, yn = y + 1 == Ny ? 0 : y + 1;
    double2* e = coef + (long)CE * N + k;
    double2* t = coef + (long)CN * N + k;
    *e = cmul(*e, cmul(ux[xe], uxi[x]));
    *t = cmul(*t, cmul(uy[yn], uyi[y]));
}

void launch_nd_symmetrise(hipStream_t s, double2* coef, double2* us, const double2* wx,
                          const double2* wy, int Nx, int Ny) {
    k_nd_u<<<(Nx + Ny + 255) / 256, 256, 0, s>>>(us, wx, wy, Nx, Ny);
    k_nd_coef<<<(unsigned)(((long)Nx * Ny + 255) / 256), 256, 0, s>>>(coef, us, Nx, Ny);
}

// entry (k, l) of the symmetrised operator (coupling planes of k_nd_coef)
__device__ inline double2 nd_entry(const double2* coef, long N, int Nx, int Ny, int k, int l) {
    double2 v = make_double2(0, 0);
    const int xk = k % Nx, yk = k / Nx, xl = l % Nx, yl = l / Nx;
    const int xke = xk + 1 == Nx ? 0 : xk + 1, xle = xl + 1 == Nx ? 0 : xl + 1;
    const int ykn = yk + 1 == Ny ? 0 : yk + 1, yln = yl + 1 == Ny ? 0 : yl + 1;
    if (yk == yl) {
        if (xk == xl) v = cadd(v, gload(coef + (long)CC * N + k));
        if (xl == xke) v = cadd(v, gload(coef + (long)CE * N + k));
        if (xk == xle) v = cadd(v, gload(coef + (long)CE * N + l));
    }
    if (xk == xl) {
        if (yl == ykn) v = cadd(v, gload(coef + (long)CN * N + k));
        if (yk == yln) v = cadd(v, gload(coef + (long)CN * N + l));
    }
    return v;
}

// ---------------------------------------------------------------------------
// Leaves: one workgroup per leaf, the whole front (p + b <= 16 T) in
// registers as a 16 x 16 cyclic distribution (thread (ti, tj) holds entries
// (ti + 16 a, tj + 16 c)), eliminated cell by cell in place (a sweep): the
// pivot row goes through LDS, double-buffered, one barrier per cell.  By
// symmetry the pivot column is the pivot row with the sign of the already
// swept rows flipped.
// ---------------------------------------------------------------------------
template <int T>
__global__ __launch_bounds__(256) void k_nd_leaf(NdLev lv, const NdFac* fac, int Nx, int Ny, void* Sv) {
    const NdFac F = fac[blockIdx.y];
    const int p = lv.p, b = lv.b, f = p + b, fr = blockIdx.x;
    const long N = (long)Nx * Ny;
    __shared__ int nd[16 * T];
    __shared__ C row[2][16 * T];
    const int t = threadIdx.x, ti = t >> 4, tj = t & 15;
    for (int i = t; i < 16 * T; i += 256) nd[i] = i < f ? lv.node[(long)fr * f + i] : -1;
    __syncthreads();
    C A[T][T];
#pragma unroll
    for (int a = 0; a < T; ++a)
#pragma unroll
        for (int c = 0; c < T; ++c) {
            const int i = ti + 16 * a, j = tj + 16 * c;
            const int ki = nd[i], kj = nd[j];
            A[a][c] = mk<C>(R(0), R(0));
            if (i < p || j < p) {
                if (ki >= 0 && kj >= 0) A[a][c] = (nd_entry(F.coef, N, Nx, Ny, ki, kj));
                else if (i == j) A[a][c] = mk<C>(R(1), R(0));
            }
        }
    R mn = R(1e30), mx = R(0);
    bool zero = false;
    static_for<0, T>([&](auto ac) {
        constexpr int ka = decltype(ac)::value;
        for (int kk = 0; kk < 16; ++kk) {
            const int k = 16 * ka + kk;
            if (k >= p) break;  // uniform
            C* rb = row[kk & 1];
            if (ti == kk) {
#pragma unroll
                for (int c = 0; c < T; ++c) rb[tj + 16 * c] = A[ka][c];
            }
            __syncthreads();
            const C d = rb[k];
            const C r = crcp_scaled(d);
            if (nd[k] >= 0) {
                const R m = cabs1(d);
                mn = m < mn ? m : mn;
                mx = m > mx ? m : mx;
                if (!(m > R(0))) zero = true;
            }
            C ci[T], rj[T];
#pragma unroll
            for (int a = 0; a < T; ++a) {
                const int i = ti + 16 * a;
                const C v = cmul(rb[i], r);           // F[k][i] / d
                ci[a] = i < k ? v : cneg(v);          // -F[i][k] / d
                rj[a] = rb[tj + 16 * a];
            }
#pragma unroll
            for (int a = 0; a < T; ++a)
#pragma unroll
                for (int c = 0; c < T; ++c) A[a][c] = cadd(A[a][c], cmul(ci[a], rj[c]));
            // pivot column and row (overwrite the update of their entries)
            if (tj == kk) {
#pragma unroll
                for (int a = 0; a < T; ++a) A[a][ka] = ci[a];
            }
            if (ti == kk) {
#pragma unroll
                for (int c = 0; c < T; ++c) A[ka][c] = cmul(rj[c], r);
                if (tj == kk) A[ka][ka] = r;
            }
        }
    });
    C* X = (C*)F.arena + lv.offX + (long)fr * p * p;
    C* Q = (C*)F.arena + lv.offQ + (long)fr * p * b;
    C* S = (C*)Sv + ((long)blockIdx.y * lv.cnt + fr) * b * b;
#pragma unroll
    for (int a = 0; a < T; ++a)
#pragma unroll
        for (int c = 0; c < T; ++c) {
            const int i = ti + 16 * a, j = tj + 16 * c;
            if (i < p && j < p) gstore(X + i * p + j, A[a][c]);
            else if (i < p && j < f) gstore(Q + i * b + (j - p), A[a][c]);
            else if (i >= p && i < f && j >= p && j < f) gstore(S + (i - p) * b + (j - p), A[a][c]);
        }
    if (t == 0) {
        double* ps = F.pivstat + 3 * (long)(lv.stat + fr);
        ps[0] = (double)mn;
        ps[1] = (double)mx;
        ps[2] = zero ? 1.0 : 0.0;
    }
}

void launch_nd_leaf(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, int Nx, int Ny, void* S) {
    const int f = lv.p + lv.b;
    const dim3 g(lv.cnt, B);
    if (f <= 32) k_nd_leaf<2><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, S);
    else if (f <= 48) k_nd_leaf<3><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, S);
    else if (f <= 64) k_nd_leaf<4><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, S);
    else k_nd_leaf<5><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, S);
}

// children's contribution to entry (i, j) of a front, i, j front indices
__device__ inline C nd_gather(const NdLev& lv, const C* Sc, const short* cm, int i, int j) {
    const int f = lv.p + lv.b;
    C v = mk<C>(0, 0);
    const int i0 = cm[i], j0 = cm[j];
    if (i0 >= 0 && j0 >= 0) v = gload(Sc + (long)i0 * lv.cb + j0);
    if (lv.nch > 1) {
        const int i1 = cm[f + i], j1 = cm[f + j];
        if (i1 >= 0 && j1 >= 0) v = cadd(v, gload(Sc + (long)lv.cb * lv.cb + (long)i1 * lv.cb + j1));
    }
    return v;
}

// ---------------------------------------------------------------------------
// Assembly of [F11 | F12] of a level: operator entries plus the children's
// Schur complements, padded separator cells as unit rows.  The first
// workgroup of a front also writes its Gauss-Jordan job and start state.
// ---------------------------------------------------------------------------
constexpr int ASM_ROWS = 8;

__global__ __launch_bounds__(256) void k_nd_asm(NdLev lv, const NdFac* fac, int Nx, int Ny,
                                                const void* Scv, NdGj w, int nchunk) {
    const int fr = blockIdx.x / nchunk, ch = blockIdx.x % nchunk, q = blockIdx.y;
    const NdFac F = fac[q];
    const int p = lv.p, b = lv.b, f = p + b;
    const long N = (long)Nx * Ny, job = (long)q * lv.cnt + fr;
    const int* node = lv.node + (long)fr * f;
    const short* cm = lv.cm + (long)fr * 2 * f;
    const C* Sc = (const C*)Scv + ((long)q * lv.cnt * lv.nch + (long)fr * lv.nch) * lv.cb * lv.cb;
    C* Y = (C*)w.Y + job * p * p;
    C* G = (C*)w.F12 + job * p * b;
    const int t = threadIdx.x;
    for (int r = 0; r < ASM_ROWS; ++r) {
        const int i = ch * ASM_ROWS + r;
        if (i >= p) break;
        const int ki = node[i];
        for (int j = t; j < f; j += 256) {
            const int kj = node[j];
            C v = mk<C>(R(0), R(0));
            if (ki >= 0 && kj >= 0) {
                v = (nd_entry(F.coef, N, Nx, Ny, ki, kj));
                v = cadd(v, nd_gather(lv, Sc, cm, i, j));
            } else if (i == j) {
                v = mk<C>(R(1), R(0));
            }
            if (j < p) gstore(Y + (long)i * p + j, v);
            else gstore(G + (long)i * b + (j - p), v);
        }
    }
    if (ch != 0) return;
    for (int i = t; i < p; i += 256) {
        w.used[job * p + i] = 0;
        w.iprow[job * p + i] = -1;
    }
    for (int i = t; i < 64; i += 256) w.win[job * 64 + i] = i < p ? i : -1;
    if (t == 0) {
        LineJob J;
        J.Y = Y;
        J.used = w.used + job * p;
        J.prow = w.prow + job * p;
        J.iprow = w.iprow + job * p;
        J.Vbuf = (C*)w.Vbuf + job * p * VMAX;
        J.LU = (C*)w.LU + job * 2 * PMAX * PMAX;
        J.piv = w.piv + job * VMAX;
        J.Z = (C*)w.Z + job * VMAX * p;
        J.win = w.win + job * 64;
        J.verr = w.verr + q;
        J.pivstat = F.pivstat + 3 * (long)(lv.stat + fr);
        J.n = p;
        J.pivstat[0] = __builtin_huge_val();
        J.pivstat[1] = 0;
        J.pivstat[2] = 0;
        w.jobs[job] = J;
    }
}

void launch_nd_asm(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, int Nx, int Ny,
                   const void* Sc, const NdGj& w) {
    const int nch = (lv.p + ASM_ROWS - 1) / ASM_ROWS;
    k_nd_asm<<<dim3(lv.cnt * nch, B), 256, 0, s>>>(lv, fac, Nx, Ny, Sc, w, nch);
}

// X[a][c] = Y[prow[a]][iprow[c]] (natural order) into the factor's arena
__global__ __launch_bounds__(256) void k_nd_unperm(NdLev lv, const NdFac* fac, NdGj w, int nchunk) {
    const int fr = blockIdx.x / nchunk, ch = blockIdx.x % nchunk, q = blockIdx.y;
    const int p = lv.p;
    const long job = (long)q * lv.cnt + fr;
    const C* Y = (const C*)w.Y + job * p * p;
    const int *pr = w.prow + job * p, *ip = w.iprow + job * p;
    C* X = (C*)fac[q].arena + lv.offX + (long)fr * p * p;
    for (int r = 0; r < ASM_ROWS; ++r) {
        const int a = ch * ASM_ROWS + r;
        if (a >= p) break;
        const C* y = Y + (long)pr[a] * p;
        for (int c = threadIdx.x; c < p; c += 256) gstore(X + (long)a * p + c, gload(y + ip[c]));
    }
}

void launch_nd_unperm(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, const NdGj& w) {
    const int nch = (lv.p + ASM_ROWS - 1) / ASM_ROWS;
    k_nd_unperm<<<dim3(lv.cnt * nch, B), 256, 0, s>>>(lv, fac, w, nch);
}

// ---------------------------------------------------------------------------
// Batched complex products of a level on MFMA, complex values as three real
// products (Gauss):
//   SCHUR = false:  Q = X F12                          (p x b, K = p)
//   SCHUR = true:   S = gather(children) - F12^T Q     (b x b, K = p),
// the latter only on tiles that meet the lower triangle; entries below the
// diagonal are written to both halves.  Operands are staged KT rows of K at a
// time through LDS, the next stage loading into registers meanwhile.
// ---------------------------------------------------------------------------
template <int TM, int TN, int KT, int WR, int WC, bool SCHUR>
__global__ __launch_bounds__(64 * WR * WC) void k_nd_gemm(NdLev lv, const NdFac* fac, const void* F12v,
                                                        const void* Scv, void* Sv, int ntm, int ntn) {
    using M = mfma_t<R>;
    using acc_t = typename M::acc;
    constexpr int NT = 64 * WR * WC;
    constexpr int WM = TM / WR, WN = TN / WC, BM = WM / 16, BN = WN / 16;
    constexpr int PA = TM + 16, PB = TN + 16;
    constexpr int AE = TM * KT / NT, BE = TN * KT / NT;
    static_assert(AE >= 1 && BE >= 1 && BM >= 1 && BN >= 1, "tile shape");
    __shared__ R sAr[KT][PA], sAi[KT][PA], sBr[KT][PB], sBi[KT][PB];
    const int q = blockIdx.y, tiles = ntm * ntn;
    const int fr = blockIdx.x / tiles, tile = blockIdx.x % tiles;
    const int i0 = (tile / ntn) * TM, j0 = (tile % ntn) * TN;
    if (SCHUR && i0 + TM <= j0) return;  // strictly upper tile
    const int p = lv.p, b = lv.b;
    const long job = (long)q * lv.cnt + fr;
    const C* F12 = (const C*)F12v + job * p * b;
    const C* X = (const C*)fac[q].arena + lv.offX + (long)fr * p * p;
    C* Q = (C*)fac[q].arena + lv.offQ + (long)fr * p * b;
    const int Mr = SCHUR ? b : p;  // rows of the product
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int wr = wv / WC, wc = wv % WC, lr = lane & 15, lk = lane >> 4;
    const C* Bg = SCHUR ? Q : F12;
    C ra[AE], rb[BE];
    const C zero = mk<C>(R(0), R(0));
    auto load = [&](int kb) {
#pragma unroll
        for (int e = 0; e < AE; ++e) {
            const int id = t + NT * e;
            if (SCHUR) {
                const int k = kb + id / TM, i = i0 + id % TM;
                const bool ok = k < p && i < b;
                ra[e] = gload(F12 + (ok ? (long)k * b + i : 0));
                if (!ok) ra[e] = zero;
            } else {
                const int i = i0 + id / KT, k = kb + id % KT;
                const bool ok = k < p && i < p;
                ra[e] = gload(X + (ok ? (long)i * p + k : 0));
                if (!ok) ra[e] = zero;
            }
        }
#pragma unroll
        for (int e = 0; e < BE; ++e) {
            const int id = t + NT * e;
            const int k = kb + id / TN, j = j0 + id % TN;
            const bool ok = k < p && j < b;
            rb[e] = gload(Bg + (ok ? (long)k * b + j : 0));
            if (!ok) rb[e] = zero;
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int e = 0; e < AE; ++e) {
            const int id = t + NT * e;
            const int k = SCHUR ? id / TM : id % KT, i = SCHUR ? id % TM : id / KT;
            sAr[k][i] = ra[e].x;
            sAi[k][i] = ra[e].y;
        }
#pragma unroll
        for (int e = 0; e < BE; ++e) {
            const int id = t + NT * e;
            sBr[id / TN][id % TN] = rb[e].x;
            sBi[id / TN][id % TN] = rb[e].y;
        }
    };
    acc_t c1[BM][BN], c2[BM][BN], c3[BM][BN];
#pragma unroll
    for (int x = 0; x < BM; ++x)
#pragma unroll
        for (int y = 0; y < BN; ++y) {
            c1[x][y] = acc_t{0, 0, 0, 0};
            c2[x][y] = acc_t{0, 0, 0, 0};
            c3[x][y] = acc_t{0, 0, 0, 0};
        }
    load(0);
    for (int kb = 0; kb < p; kb += KT) {
        store();
        __syncthreads();
        if (kb + KT < p) load(kb + KT);
#pragma unroll
        for (int kk = 0; kk < KT; kk += 4) {
            R ar[BM], ai[BM], as[BM], br[BN], bi[BN], bs[BN];
#pragma unroll
            for (int x = 0; x < BM; ++x) {
                ar[x] = sAr[kk + lk][wr * WM + x * 16 + lr];
                ai[x] = sAi[kk + lk][wr * WM + x * 16 + lr];
                as[x] = ar[x] + ai[x];
            }
#pragma unroll
            for (int y = 0; y < BN; ++y) {
                br[y] = sBr[kk + lk][wc * WN + y * 16 + lr];
                bi[y] = sBi[kk + lk][wc * WN + y * 16 + lr];
                bs[y] = br[y] + bi[y];
            }
#pragma unroll
            for (int x = 0; x < BM; ++x)
#pragma unroll
                for (int y = 0; y < BN; ++y) c1[x][y] = M::run(ar[x], br[y], c1[x][y]);
#pragma unroll
            for (int x = 0; x < BM; ++x)
#pragma unroll
                for (int y = 0; y < BN; ++y) c2[x][y] = M::run(ai[x], bi[y], c2[x][y]);
#pragma unroll
            for (int x = 0; x < BM; ++x)
#pragma unroll
                for (int y = 0; y < BN; ++y) c3[x][y] = M::run(as[x], bs[y], c3[x][y]);
        }
        __syncthreads();
    }
    const short* cm = lv.cm + (long)fr * 2 * (p + b);
    const C* Sc = SCHUR ? (const C*)Scv + ((long)q * lv.cnt * lv.nch + (long)fr * lv.nch) * lv.cb * lv.cb
                        : nullptr;
    C* S = SCHUR ? (C*)Sv + job * b * b : nullptr;
#pragma unroll
    for (int x = 0; x < BM; ++x)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = i0 + wr * WM + x * 16 + M::row(lane, v);
            if (i >= Mr) continue;
#pragma unroll
            for (int y = 0; y < BN; ++y) {
                const int j = j0 + wc * WN + y * 16 + lr;
                if (j >= b) continue;
                const R re = c1[x][y][v] - c2[x][y][v];
                const R im = c3[x][y][v] - c1[x][y][v] - c2[x][y][v];
                if (!SCHUR) {
                    gstore(Q + (long)i * b + j, mk<C>(re, im));
                } else if (i >= j) {
                    const C o = nd_gather(lv, Sc, cm, p + i, p + j);
                    const C z = mk<C>(o.x - re, o.y - im);
                    gstore(S + (long)i * b + j, z);
                    if (i > j) gstore(S + (long)j * b + i, z);
                }
            }
        }
}

void launch_nd_gemm(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, const void* F12,
                    const void* Sc, void* S, bool schur) {
    auto go = [&](auto kern, int TM, int TN, int NT) {
        const int ntm = ((schur ? lv.b : lv.p) + TM - 1) / TM, ntn = (lv.b + TN - 1) / TN;
        kern<<<dim3(lv.cnt * ntm * ntn, B), NT, 0, s>>>(lv, fac, F12, Sc, S, ntm, ntn);
    };
    constexpr int TN = 64;
    if (lv.b >= 256 && lv.p >= 96) {
        if (schur) go(k_nd_gemm<128, TN, 16, 4, 2, true>, 128, TN, 512);
        else go(k_nd_gemm<128, TN, 16, 4, 2, false>, 128, TN, 512);
    } else {
        if (schur) go(k_nd_gemm<64, 64, 8, 2, 2, true>, 64, 64, 256);
        else go(k_nd_gemm<64, 64, 8, 2, 2, false>, 64, 64, 256);
    }
}

// smallest and largest pivot and zero-pivot flag of each factor's fronts
__global__ __launch_bounds__(256) void k_nd_stat(const NdFac* fac, int nfronts, double* out) {
    const double* ps = fac[blockIdx.x].pivstat;
    double mn = __builtin_huge_val(), mx = 0, z = 0;
    for (int i = threadIdx.x; i < nfronts; i += 256) {
        mn = fmin(mn, ps[3 * i]);
        mx = fmax(mx, ps[3 * i + 1]);
        z = fmax(z, ps[3 * i + 2]);
    }
    __shared__ double r[3][256];
    r[0][threadIdx.x] = mn;
    r[1][threadIdx.x] = mx;
    r[2][threadIdx.x] = z;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            r[0][threadIdx.x] = fmin(r[0][threadIdx.x], r[0][threadIdx.x + o]);
            r[1][threadIdx.x] = fmax(r[1][threadIdx.x], r[1][threadIdx.x + o]);
            r[2][threadIdx.x] = fmax(r[2][threadIdx.x], r[2][threadIdx.x + o]);
        }
        __syncthreads();
    }
    if (threadIdx.x < 3) out[3 * blockIdx.x + threadIdx.x] = r[threadIdx.x][0];
}
void launch_nd_stat(hipStream_t s, const NdFac* fac, int B, int nfronts, double* out) {
    k_nd_stat<<<B, 256, 0, s>>>(fac, nfronts, out);
}

// ---------------------------------------------------------------------------
// Reduced solve.  Upward step of a level: the separator values
//   v = scaled right-hand side + children's updates
// and the boundary update u = children's updates - Q^T v.  A workgroup takes
// CW boundary columns; 256 / CW row groups split the separator.
// ---------------------------------------------------------------------------
template <int CW>
__global__ __launch_bounds__(256) void k_nd_up(NdLev lv, const void* arena, NdVec z, int Nx, int nchunk) {
    constexpr int RG = 256 / CW;
    extern __shared__ char nd_lds[];
    C* vs = (C*)nd_lds;
    __shared__ C red[RG][CW];
    const int fr = blockIdx.x / nchunk, ch = blockIdx.x % nchunk;
    const int p = lv.p, b = lv.b, f = p + b;
    const int src = z.ridx ? z.ridx[0] : 0;
    const double2* in = z.in + (long)src * z.rs;
    double2* vb = z.v + lv.offV + (long)fr * p;
    double2* ub = z.u + lv.offU + (long)fr * b;
    const double2* uc = z.u + lv.offUc + (long)fr * lv.nch * lv.cb;
    const int* node = lv.node + (long)fr * f;
    const short* cm = lv.cm + (long)fr * 2 * f;
    const int t = threadIdx.x;
    auto kids = [&](int i) {
        double2 a = make_double2(0, 0);
        if (lv.nch > 0) {
            const int m0 = cm[i];
            if (m0 >= 0) a = uc[m0];
            if (lv.nch > 1) {
                const int m1 = cm[f + i];
                if (m1 >= 0) a = cadd(a, uc[lv.cb + m1]);
            }
        }
        return a;
    };
    for (int i = t; i < p; i += 256) {
        const int k = node[i];
        double2 v = make_double2(0, 0);
        if (k >= 0) {
            v = cmul(in[k], cmul(z.six[k % Nx], z.siy[k / Nx]));
            v = cadd(v, kids(i));
        }
        vs[i] = (v);
        if (ch == 0) vb[i] = v;
    }
    if (b == 0) return;
    __syncthreads();
    const int c = t % CW, rg = t / CW, j = ch * CW + c;
    C acc = mk<C>(R(0), R(0));
    if (j < b) {
        const C* Q = (const C*)arena + lv.offQ + (long)fr * p * b + j;
        int i = rg;
        for (; i + 3 * RG < p; i += 4 * RG) {
            const C q0 = gload(Q + (long)i * b), q1 = gload(Q + (long)(i + RG) * b),
                    q2 = gload(Q + (long)(i + 2 * RG) * b), q3 = gload(Q + (long)(i + 3 * RG) * b);
            acc = cadd(acc, cmul(q0, vs[i]));
            acc = cadd(acc, cmul(q1, vs[i + RG]));
            acc = cadd(acc, cmul(q2, vs[i + 2 * RG]));
            acc = cadd(acc, cmul(q3, vs[i + 3 * RG]));
        }
        for (; i < p; i += RG) acc = cadd(acc, cmul(gload(Q + (long)i * b), vs[i]));
    }
    red[rg][c] = acc;
    __syncthreads();
    if (t < CW && j < b) {
#pragma unroll 4
        for (int r = 1; r < RG; ++r) acc = cadd(acc, red[r][c]);
        ub[j] = csub(kids(p + j), (acc));
    }
}

// Downward step: x = X v - Q x_boundary, one wave per row (RPW rows at a
// time), the vector staged through LDS in pieces.
constexpr int DN_PIECE = 512;

template <int RPW>
__global__ __launch_bounds__(256) void k_nd_down(NdLev lv, const void* arena, NdVec z, int Nx, int nchunk) {
    __shared__ C xs[DN_PIECE];
    const int fr = blockIdx.x / nchunk, ch = blockIdx.x % nchunk;
    const int p = lv.p, b = lv.b, f = p + b;
    const int src = z.ridx ? z.ridx[0] : 0;
    double2* out = z.out + (long)src * z.rs;
    double2* xg = z.x;
    const double2* vb = z.v + lv.offV + (long)fr * p;
    const int* node = lv.node + (long)fr * f;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const C* X = (const C*)arena + lv.offX + (long)fr * p * p;
    const C* Q = (const C*)arena + lv.offQ + (long)fr * p * b;
    const int r0 = (ch * 4 + wv) * RPW;
    C acc[RPW];
#pragma unroll
    for (int r = 0; r < RPW; ++r) acc[r] = mk<C>(R(0), R(0));
    for (int part = 0; part < 2; ++part) {
        const int len = part ? b : p;
        const C* Mt = part ? Q : X;
        for (int k0 = 0; k0 < len; k0 += DN_PIECE) {
            const int n = min(DN_PIECE, len - k0);
            __syncthreads();
            for (int k = t; k < n; k += 256) {
                if (part) {
                    const int kk = node[p + k0 + k];
                    xs[k] = kk >= 0 ? (cneg(xg[kk])) : mk<C>(R(0), R(0));
                } else {
                    xs[k] = (vb[k0 + k]);
                }
            }
            __syncthreads();
            for (int k = lane; k < n; k += 64) {
                const C x = xs[k];
#pragma unroll
                for (int r = 0; r < RPW; ++r) {
                    const int i = min(r0 + r, p - 1);
                    acc[r] = cadd(acc[r], cmul(gload(Mt + (long)i * len + k0 + k), x));
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        for (int o = 32; o > 0; o >>= 1) {
            acc[r].x += shfl_x(acc[r].x, o);
            acc[r].y += shfl_x(acc[r].y, o);
        }
        const int i = r0 + r;
        if (lane == 0 && i < p) {
            const int k = node[i];
            if (k >= 0) {
                const double2 x = (acc[r]);
                xg[k] = x;
                out[k] = cmul(x, cmul(z.sox[k % Nx], z.soy[k / Nx]));
            }
        }
    }
}

void launch_nd_up(hipStream_t s, const NdLev& lv, const void* arena, const NdVec& z, int Nx) {
    const size_t lds = sizeof(C) * lv.p;
    auto go = [&](auto kern, int CW) {
        const int nch = std::max(1, (lv.b + CW - 1) / CW);
        kern<<<dim3(lv.cnt * nch), 256, lds, s>>>(lv, arena, z, Nx, nch);
    };
    // few fronts: narrow column groups, so that more workgroups share a front
    if ((long)lv.cnt * lv.b < 64 * 512) go(k_nd_up<4>, 4);
    else if (lv.b <= 32 || (long)lv.cnt * lv.b < 64 * 2048) go(k_nd_up<16>, 16);
    else go(k_nd_up<64>, 64);
}
void launch_nd_down(hipStream_t s, const NdLev& lv, const void* arena, const NdVec& z, int Nx) {
    auto go = [&](auto kern, int RPW) {
        const int nch = (lv.p + 4 * RPW - 1) / (4 * RPW);
        kern<<<dim3(lv.cnt * nch), 256, 0, s>>>(lv, arena, z, Nx, nch);
    };
    if ((long)lv.cnt * lv.p < 4096) go(k_nd_down<1>, 1);
    else go(k_nd_down<4>, 4);
}

// ---------------------------------------------------------------------------
// The reduced solve for 2 .. 16 sources on MFMA (16 x 16 x 4).  Work vectors
// keep the sources innermost (entry (i, s) at 16 i + s, zero past the active
// ones), so a row of 16 sources is one contiguous piece of every gather and
// the product's B operand; the factor streams straight into the A operand, so
// it is read once for all sources.  With one wave a tile of 16 outputs, a
// CU's four SIMDs consume about 16 B of factor a clock in FP32 and FP64
// alike, above its share of the memory rate, so the products cost no more than
// the stream.  Levels with few tiles split K over KS waves of a workgroup.
// ---------------------------------------------------------------------------
// x[k][s] = scale_k in_s[k] (PACK), or out_s[k] = scale_k x[k][s]
template <bool PACK>
__global__ __launch_bounds__(256) void k_ndm_io(NdVec z, C* x, long N, int Nx, int na) {
    __shared__ double2 tile[16][65];
    const long k0 = blockIdx.x * 64L;
    const int t = threadIdx.x;
    const double2 *sx = PACK ? z.six : z.sox, *sy = PACK ? z.siy : z.soy;
    if (PACK) {
        for (int e = t; e < 1024; e += 256) {
            const int s = e >> 6, c = e & 63;
            const long k = k0 + c;
            double2 v = make_double2(0, 0);
            if (s < na && k < N) v = cmul(z.in[(long)z.ridx[s] * z.rs + k], cmul(sx[k % Nx], sy[k / Nx]));
            tile[s][c] = v;
        }
        __syncthreads();
        for (int e = t; e < 1024; e += 256) {
            const long k = k0 + (e >> 4);
            if (k < N) x[k * 16 + (e & 15)] = (tile[e & 15][e >> 4]);
        }
    } else {
        for (int e = t; e < 1024; e += 256) {
            const long k = k0 + (e >> 4);
            if (k < N) tile[e & 15][e >> 4] = (x[k * 16 + (e & 15)]);
        }
        __syncthreads();
        for (int e = t; e < 1024; e += 256) {
            const int s = e >> 6, c = e & 63;
            const long k = k0 + c;
            if (s < na && k < N)
                z.out[(long)z.ridx[s] * z.rs + k] = cmul(tile[s][c], cmul(sx[k % Nx], sy[k / Nx]));
        }
    }
}

// separator values and the children's part of the boundary updates of a level
__global__ __launch_bounds__(256) void k_ndm_gather(NdLev lv, C* vp, C* up, const C* x) {
    const int f = lv.p + lv.b;
    const long e = blockIdx.x * 16L + (threadIdx.x >> 4);
    if (e >= (long)lv.cnt * f) return;
    const int s = threadIdx.x & 15, fr = (int)(e / f), i = (int)(e % f);
    const int k = lv.node[e];
    C v = mk<C>(R(0), R(0));
    if (k >= 0) {
        if (i < lv.p) v = gload(x + (long)k * 16 + s);
        const C* uc = up + (lv.offUc + (long)fr * lv.nch * lv.cb) * 16;
        const short* cm = lv.cm + (long)fr * 2 * f + i;
        if (lv.nch > 0 && cm[0] >= 0) v = cadd(v, gload(uc + (long)cm[0] * 16 + s));
        if (lv.nch > 1 && cm[f] >= 0) v = cadd(v, gload(uc + ((long)lv.cb + cm[f]) * 16 + s));
    }
    if (i < lv.p) gstore(vp + (lv.offV + (long)fr * lv.p + i) * 16 + s, v);
    else gstore(up + (lv.offU + (long)fr * lv.b + (i - lv.p)) * 16 + s, v);
}

// accumulators of a complex 16 x 16 tile: re = rr - ii, im = ri
struct ndm_acc {
    typename mfma_t<R>::acc rr = {0, 0, 0, 0}, ii = {0, 0, 0, 0}, ri = {0, 0, 0, 0};
    __device__ inline void step(C a, C b) {
        rr = mfma_t<R>::run(a.x, b.x, rr);
        ii = mfma_t<R>::run(a.y, b.y, ii);
        ri = mfma_t<R>::run(a.x, b.y, ri);
        ri = mfma_t<R>::run(a.y, b.x, ri);
    }
};

// sum of the KS waves' tiles through LDS (valid in wave 0)
template <int KS>
__device__ inline void ndm_reduce(C (&z)[4], C (*red)[4][64], int wv, int lane) {
    if constexpr (KS > 1) {
#pragma unroll
        for (int v = 0; v < 4; ++v) red[wv][v][lane] = z[v];
        __syncthreads();
        if (wv == 0)
            for (int w = 1; w < KS; ++w)
#pragma unroll
                for (int v = 0; v < 4; ++v) z[v] = cadd(z[v], red[w][v][lane]);
    }
}

constexpr int NDM_U = 4;  // K steps whose operands are loaded together

// u[j] -= sum_i Q[i][j] v[i], 16 boundary cells a tile
template <int KS>
__global__ __launch_bounds__(KS == 1 ? 256 : 64 * KS) void k_ndm_up(NdLev lv, const void* arena, const C* vp,
                                                               C* up, int nt) {
    using M = mfma_t<R>;
    __shared__ C red[KS > 1 ? KS : 1][4][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const long tile = KS == 1 ? blockIdx.x * 4L + wv : (long)blockIdx.x;
    if (KS == 1 && tile >= (long)lv.cnt * nt) return;
    const int fr = (int)(tile / nt), j0 = (int)(tile % nt) * 16;
    const int p = lv.p, b = lv.b, l16 = lane & 15, kg = lane >> 4;
    const C* Q = (const C*)arena + lv.offQ + (long)fr * p * b + min(j0 + l16, b - 1);
    const C* v = vp + (lv.offV + (long)fr * p) * 16 + l16;
    ndm_acc A;
    const int nst = p / 4;
    for (int s0 = KS == 1 ? 0 : wv * NDM_U; s0 < nst; s0 += KS * NDM_U) {
        C a[NDM_U], x[NDM_U];
#pragma unroll
        for (int q = 0; q < NDM_U; ++q) {
            const int i = 4 * min(s0 + q, nst - 1) + kg;
            a[q] = gload(Q + (long)i * b);
            x[q] = gload(v + (long)i * 16);
        }
#pragma unroll
        for (int q = 0; q < NDM_U; ++q)
            if (s0 + q < nst) A.step(a[q], x[q]);
    }
    C z[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) z[r] = mk<C>(A.rr[r] - A.ii[r], A.ri[r]);
    ndm_reduce<KS>(z, red, wv, lane);
    if (KS > 1 && wv != 0) return;
    C* u = up + (lv.offU + (long)fr * b) * 16 + l16;
    C old[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) old[r] = gload(u + (long)min(j0 + M::row(lane, r), b - 1) * 16);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int j = j0 + M::row(lane, r);
        if (j < b) gstore(u + (long)j * 16, csub(old[r], z[r]));
    }
}

// x = X v - Q x_boundary, 16 separator cells a tile.  X is symmetric, so its
// operand is read along rows (16 neighbouring columns); a lane reads four
// neighbouring entries of its row of Q and the K order is permuted to match.
template <int KS>
__global__ __launch_bounds__(KS == 1 ? 256 : 64 * KS) void k_ndm_down(NdLev lv, const void* arena, const C* vp,
                                                                 C* xp, int nt) {
    using M = mfma_t<R>;
    __shared__ C red[KS > 1 ? KS : 1][4][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const long tile = KS == 1 ? blockIdx.x * 4L + wv : (long)blockIdx.x;
    if (KS == 1 && tile >= (long)lv.cnt * nt) return;
    const int fr = (int)(tile / nt), i0 = (int)(tile % nt) * 16;
    const int p = lv.p, b = lv.b, l16 = lane & 15, kg = lane >> 4;
    const int* node = lv.node + (long)fr * (p + b);
    const int row = min(i0 + l16, p - 1);
    const C* X = (const C*)arena + lv.offX + (long)fr * p * p + row;
    const C* Q = (const C*)arena + lv.offQ + (long)fr * p * b + (long)row * b;
    const C* v = vp + (lv.offV + (long)fr * p) * 16 + l16;
    ndm_acc A, B;
    const int nst = p / 4;
    for (int s0 = KS == 1 ? 0 : wv * NDM_U; s0 < nst; s0 += KS * NDM_U) {
        C a[NDM_U], x[NDM_U];
#pragma unroll
        for (int q = 0; q < NDM_U; ++q) {
            const int k = 4 * min(s0 + q, nst - 1) + kg;
            a[q] = gload(X + (long)k * p);
            x[q] = gload(v + (long)k * 16);
        }
#pragma unroll
        for (int q = 0; q < NDM_U; ++q)
            if (s0 + q < nst) A.step(a[q], x[q]);
    }
    // four consecutive columns k0 + 4 kg .. + 3 per lane; b is a multiple of 4
    for (int k0 = KS == 1 ? 0 : 16 * wv; k0 < b; k0 += KS * 16) {
        const int k = k0 + 4 * kg;
        const bool ok = k < b;
        C a[4], x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int n = ok ? gload_s(node + p + k + q) : -1;
            a[q] = gload(Q + (ok ? k + q : 0));
            x[q] = gload(xp + (long)max(n, 0) * 16 + l16);
            if (n < 0) {
                a[q] = mk<C>(R(0), R(0));
                x[q] = a[q];
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) B.step(a[q], x[q]);
    }
    C z[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        z[r] = mk<C>((A.rr[r] - A.ii[r]) - (B.rr[r] - B.ii[r]), A.ri[r] - B.ri[r]);
    ndm_reduce<KS>(z, red, wv, lane);
    if (KS > 1 && wv != 0) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = i0 + M::row(lane, r);
        if (i < p) {
            const int k = node[i];
            if (k >= 0) gstore(xp + (long)k * 16 + l16, z[r]);
        }
    }
}

void launch_ndm_io(hipStream_t s, const NdVec& z, void* x, long N, int Nx, int na, bool pack) {
    const unsigned nb = (unsigned)((N + 63) / 64);
    if (pack) k_ndm_io<true><<<nb, 256, 0, s>>>(z, (C*)x, N, Nx, na);
    else k_ndm_io<false><<<nb, 256, 0, s>>>(z, (C*)x, N, Nx, na);
}
// waves that share a tile's K range: enough that a level of few tiles still
// covers the chip's 1024 SIMDs, at least 8 K steps a wave
static int ndm_split(long tiles, int k) {
    if (tiles >= 2048 || k < 128) return 1;
    return (tiles >= 512 || k < 512) ? 4 : 16;
}
void launch_ndm_up(hipStream_t s, const NdLev& lv, const void* arena, void* vp, void* up, const void* x) {
    const long n = (long)lv.cnt * (lv.p + lv.b);
    k_ndm_gather<<<(unsigned)((n + 15) / 16), 256, 0, s>>>(lv, (C*)vp, (C*)up, (const C*)x);
    if (lv.b == 0) return;
    const int nt = (lv.b + 15) / 16;
    const long tiles = (long)lv.cnt * nt;
    switch (ndm_split(tiles, lv.p)) {
        case 1: k_ndm_up<1><<<(unsigned)((tiles + 3) / 4), 256, 0, s>>>(lv, arena, (const C*)vp, (C*)up, nt); break;
        case 4: k_ndm_up<4><<<(unsigned)tiles, 256, 0, s>>>(lv, arena, (const C*)vp, (C*)up, nt); break;
        default: k_ndm_up<16><<<(unsigned)tiles, 1024, 0, s>>>(lv, arena, (const C*)vp, (C*)up, nt);
    }
}
void launch_ndm_down(hipStream_t s, const NdLev& lv, const void* arena, const void* vp, void* x) {
    const int nt = (lv.p + 15) / 16;
    const long tiles = (long)lv.cnt * nt;
    switch (ndm_split(tiles, lv.p + lv.b)) {
        case 1: k_ndm_down<1><<<(unsigned)((tiles + 3) / 4), 256, 0, s>>>(lv, arena, (const C*)vp, (C*)x, nt); break;
        case 4: k_ndm_down<4><<<(unsigned)tiles, 256, 0, s>>>(lv, arena, (const C*)vp, (C*)x, nt); break;
        default: k_ndm_down<16><<<(unsigned)tiles, 1024, 0, s>>>(lv, arena, (const C*)vp, (C*)x, nt);
    }
}

}  // namespace fdfd
