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
    // most pairs of a front are no neighbours on the torus
    const int dk = k > l ? k - l : l - k;
    if (dk > 1 && dk != Nx && dk != Nx - 1 && dk != (int)N - Nx) return v;
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
// In-place inversion by sweeps.  Sweeping cell k of a symmetric matrix M replaces
//   M_ij -= M_ik M_kj / d,  M_kj /= d,  M_ik /= -d,  M_kk = 1 / d,  d = M_kk,
// and sweeping the first np cells leaves M_ss^-1, Q = M_ss^-1 M_su above -Q^T,
// and the Schur complement.  Entries between swept and unswept cells are
// antisymmetric, all others symmetric, so only one triangle is kept; sweeps
// commute, so nothing is permuted.
//
// A matrix of 16 T cells is held in registers by the four waves of a
// workgroup, lower 16 x 16 tiles (I, J) in the MFMA accumulator layout, tile
// number I (I + 1) / 2 + J on wave (number % 4).  A block of 16 cells is swept at
// once:
//   a  the wave of tile (k, k) sweeps it on its own (nd_sweep16), the others put
//      the block row R_J = M_kJ into LDS;
//   b  Z_J = D^-1 R_J on MFMA, replacing tiles (k, J) by Z_J, (I, k) by -Z_I^T;
//   c  M_IJ -= sigma_I R_I^T Z_J on the other tiles, sigma = -1 for swept I;
//      the wave of the next diagonal tile goes on to its sweep meanwhile.
// The last block may end inside its tile: with its swept rows s and the others u,
// D holds D_ss^-1 and E = D_ss^-1 M_su, and b leaves R_uJ - E^T R_sJ in rows u.
// Cells are taken in order: with FP64 fronts and refinement the growth this
// allows (1e4 .. 1e5, like the near-resonances of the boxes) costs nothing that
// pivoting inside a separator would save.  What bounds a small inversion is the
// instruction count of its chain (a wave issues one in four cycles or more, an
// FP64 operation takes 16 from operand to result): sweeping 64 cells one by one
// with diagonal pivoting took 55 us on all four waves and 38 us in 16-cell
// tiles, four by four on all waves (817 instructions a step) 28 us.
// ---------------------------------------------------------------------------
__device__ inline C nd_rcp(C z) {
    // 1 / z from one hardware reciprocal of |z|^2 (about half the bits) and one
    // step r (1 + e + e^2), e = 1 - n r (the entries are scaled to O(1) and grow
    // by 1e6 or so: no range handling; NdPiv reports what is outside)
    const double n = fma(z.x, z.x, z.y * z.y), r0 = rcp_hw(n);
    const double e = fma(-n, r0, 1.0), r = fma(r0, fma(e, e, e), r0);
    return mk<C>(z.x * r, -z.y * r);
}
// a b + c in four fused steps
__device__ inline C cfma(C a, C b, C c) {
    return mk<C>(fma(a.x, b.x, fma(-a.y, b.y, c.x)), fma(a.x, b.y, fma(a.y, b.x, c.y)));
}

using F64 = mfma_t<double>;

// smallest and largest 2 x 2 pivot determinant (|re| + |im|), and whether one was
// out of the range that nd_rcp, which squares it, inverts
struct NdPiv {
    double mn = 1e300, mx = 0;
    bool bad = false;
    __device__ inline void add(C det) {
        const double m = cabs1(det);
        mn = fmin(mn, m);
        mx = fmax(mx, m);
        bad = bad || !(m > 1e-140 && m < 1e140);
    }
};

// inverse of a symmetric 2 x 2 block [a b; b c]
__device__ inline void nd_inv2(C a, C b, C c, C& x, C& y, C& z, NdPiv& pv) {
    const C det = cfma(a, c, cneg(cmul(b, b)));
    pv.add(det);
    const C r = nd_rcp(det);
    x = cmul(c, r);
    y = cneg(cmul(b, r));
    z = cmul(a, r);
}

// One wave sweeps the first kw cells (a multiple of 4) of its 16 x 16 tile, four
// at a time, the K of one 16 x 16 x 4 product: rows 4 v .. 4 v + 3 are entry v
// of the lanes, so the pivot rows are both operands as they stand,
//   M -= sigma R^T Z,  Z = D^-1 R,
// with the 4 x 4 pivot block D inverted by every lane (two 2 x 2 blocks, two
// reciprocals), pivot rows replaced by Z and pivot columns by -sigma R^T D^-1.
__device__ __attribute__((always_inline)) inline void nd_sweep16(d4v& mr, d4v& mi, int kw, C (*R)[17], NdPiv& pv) {
    const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    static_for<0, 4>([&](auto vc) {
        constexpr int v = decltype(vc)::value, k0 = 4 * v;
        if (k0 < kw) {  // uniform
            const bool quad = (l16 >> 2) == v;
            C a = mk<C>(mr[v], mi[v]);
            R[g][l16] = a;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            auto D = [&](int i, int j) { return R[i][k0 + j]; };
            const C d00 = D(0, 0), d01 = D(0, 1), d11 = D(1, 1), a0 = D(0, 2), a1 = D(0, 3), a2 = D(1, 2),
                    a3 = D(1, 3), d22 = D(2, 2), d23 = D(2, 3), d33 = D(3, 3);
            const C b0 = R[0][l16], b1 = R[1][l16], b2 = R[2][l16], b3 = R[3][l16];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            // D^-1 = [P + X S^-1 X^T, -X S^-1; ., S^-1], P = D11^-1, X = P D12,
            // S = D22 - D12^T X
            C p0, p1, p2, s0, s1, s2;
            nd_inv2(d00, d01, d11, p0, p1, p2, pv);
            const C x0 = cfma(p0, a0, cmul(p1, a2)), x1 = cfma(p0, a1, cmul(p1, a3));
            const C x2 = cfma(p1, a0, cmul(p2, a2)), x3 = cfma(p1, a1, cmul(p2, a3));
            const C na0 = cneg(a0), na1 = cneg(a1), na2 = cneg(a2), na3 = cneg(a3);
            nd_inv2(cfma(na0, x0, cfma(na2, x2, d22)), cfma(na0, x1, cfma(na2, x3, d23)),
                    cfma(na1, x1, cfma(na3, x3, d33)), s0, s1, s2, pv);
            const C y0 = cfma(x0, s0, cmul(x1, s1)), y1 = cfma(x0, s1, cmul(x1, s2));  // X S^-1
            const C y2 = cfma(x2, s0, cmul(x3, s1)), y3 = cfma(x2, s1, cmul(x3, s2));
            const C q0 = cfma(y0, x0, cfma(y1, x1, p0)), q1 = cfma(y0, x2, cfma(y1, x3, p1)),
                    q2 = cfma(y2, x2, cfma(y3, x3, p2));
            // this lane group's row of D^-1, and the entry for a pivot column
            auto pick = [&](int i, C a, C b, C c, C e) {
                const C lo = csel((i & 1) != 0, b, a), hi = csel((i & 1) != 0, e, c);
                return csel((i & 2) != 0, hi, lo);
            };
            const C n0 = cneg(y0), n1 = cneg(y1), n2 = cneg(y2), n3 = cneg(y3);
            const C r0 = pick(g, q0, q1, n0, n1), r1 = pick(g, q1, q2, n2, n3), r2 = pick(g, n0, n2, s0, s1),
                    r3 = pick(g, n1, n3, s1, s2);
            C z = cfma(r0, b0, cfma(r1, b1, cfma(r2, b2, cmul(r3, b3))));
            z = csel(quad, pick(l16, r0, r1, r2, r3), z);
            a = csel(l16 < k0, a, cneg(a));  // antisymmetric to swept cells
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                mr[w] = quad ? 0.0 : mr[w];
                mi[w] = quad ? 0.0 : mi[w];
            }
            mr = F64::run(a.x, z.x, mr);
            mi = F64::run(a.x, z.y, mi);
            mr = F64::run(-a.y, z.y, mr);
            mi = F64::run(a.y, z.x, mi);
            mr[v] = z.x;
            mi[v] = z.y;
        }
    });
}

// DB: the block row is double-buffered (one barrier less a block, more LDS).
// R and Z leave out the block being swept.
template <int T> struct NdSweep {
    static constexpr int NTL = T * (T + 1) / 2, NS = (NTL + 3) / 4;  // tiles, slots per wave
    static constexpr bool DB = T <= 4;
    C R[DB ? 2 : 1][T > 1 ? T - 1 : 1][16][17];
    C Z[T > 1 ? T - 1 : 1][16][17];
    C D[16][17];
    double pv[4][3];
};

// f(slot, I, J) for the tiles of this wave (I, J wave-uniform)
template <int T, typename F> __device__ __attribute__((always_inline)) inline void nd_each_tile(F&& f) {
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    static_for<0, NdSweep<T>::NS>([&](auto sc) {
        const int e = 4 * decltype(sc)::value + wv;
        if (e < NdSweep<T>::NTL) {
            int I = 0;
#pragma unroll
            for (int q = 1; q < T; ++q) I += e >= q * (q + 1) / 2;
            f(sc, I, e - I * (I + 1) / 2);
        }
    });
}
// f(slot, v, i, j, off) for the entries of this thread (off: an off-diagonal
// tile, whose mirror image is not stored)
template <int T, typename F> __device__ __attribute__((always_inline)) inline void nd_each_entry(F&& f) {
    const int lane = threadIdx.x & 63;
    nd_each_tile<T>([&](auto sc, int I, int J) {
#pragma unroll
        for (int v = 0; v < 4; ++v) f(sc, v, 16 * I + F64::row(lane, v), 16 * J + (lane & 15), I != J);
    });
}

// sweeps the first np cells (a multiple of 4); pst: pivot statistics, combined
// with what is there when `add`
template <int T>
__device__ __attribute__((always_inline)) inline void nd_sweep(d4v (&mr)[NdSweep<T>::NS], d4v (&mi)[NdSweep<T>::NS],
                                                               int np, NdSweep<T>& s, double* pst, bool add) {
    const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    NdPiv pv;
#pragma unroll 1
    for (int kb = 0; 16 * kb < np; ++kb) {
        const int kw = min(16, np - 16 * kb);
        C(*R)[16][17] = s.R[NdSweep<T>::DB ? kb & 1 : 0];
        auto at = [&](int I) { return I - (I > kb); };
        // the diagonal tile of block kb is in slot e / 4 of wave e % 4
        const int e = kb * (kb + 3) / 2;
        nd_each_tile<T>([&](auto sc, int I, int J) {
            if (I != J && I == kb) {
#pragma unroll
                for (int v = 0; v < 4; ++v) R[at(J)][F64::row(lane, v)][l16] = mk<C>(mr[sc][v], mi[sc][v]);
            } else if (I != J && J == kb) {
#pragma unroll
                for (int v = 0; v < 4; ++v) R[at(I)][l16][F64::row(lane, v)] = mk<C>(mr[sc][v], mi[sc][v]);
            }
        });
        if ((e & 3) == __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) {
            // one copy of the sweep's code for all slots
            d4v xr = mr[0], xi = mi[0];
#pragma unroll
            for (int q = 1; q < NdSweep<T>::NS; ++q)
                if ((e >> 2) == q) {
                    xr = mr[q];
                    xi = mi[q];
                }
            nd_sweep16(xr, xi, kw, s.D, pv);
#pragma unroll
            for (int q = 0; q < NdSweep<T>::NS; ++q)
                if ((e >> 2) == q) {
                    mr[q] = xr;
                    mi[q] = xi;
                }
#pragma unroll
            for (int v = 0; v < 4; ++v) s.D[F64::row(lane, v)][l16] = mk<C>(l16 < kw ? xr[v] : -xr[v], l16 < kw ? xi[v] : -xi[v]);
        }
        if (T == 1) break;
        __syncthreads();
        const int kq = kw >> 2;  // K steps
        nd_each_tile<T>([&](auto sc, int I, int J) {
            if ((I == kb) == (J == kb)) return;
            const bool rowt = I == kb;  // tile (k, J), else (I, k)
            // (k, J): D^-1 R_J; (I, k): R_I^T D^-1 (D^-1 is symmetric)
            const C(*Ap)[17] = rowt ? s.D : R[at(I)];
            const C(*Bp)[17] = rowt ? R[at(J)] : s.D;
            d4v xr = {0, 0, 0, 0}, xi = {0, 0, 0, 0}, yr = {0, 0, 0, 0}, yi = {0, 0, 0, 0};
            if (kw < 16) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const bool un = (rowt ? F64::row(lane, v) : l16) >= kw;
                    xr[v] = un ? mr[sc][v] : 0.0;
                    xi[v] = un ? mi[sc][v] : 0.0;
                }
            }
            const bool ng = !rowt && l16 < kw;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (q < kq) {
                    const C av = Ap[4 * q + g][l16], bv = Bp[4 * q + g][l16];
                    xr = F64::run(av.x, bv.x, xr);
                    xi = F64::run(av.x, bv.y, xi);
                    yr = F64::run(av.y, bv.y, yr);
                    yi = F64::run(av.y, bv.x, yi);
                }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const C z = mk<C>(xr[v] - yr[v], xi[v] + yi[v]);
                if (rowt) s.Z[at(J)][F64::row(lane, v)][l16] = z;
                else s.Z[at(I)][l16][F64::row(lane, v)] = z;
                mr[sc][v] = ng ? -z.x : z.x;
                mi[sc][v] = ng ? -z.y : z.y;
            }
        });
        __syncthreads();
        nd_each_tile<T>([&](auto sc, int I, int J) {
            if (I == kb || J == kb) return;
            const C(*Ap)[17] = R[at(I)];
            const C(*Bp)[17] = s.Z[at(J)];
            const unsigned long long sg = I > kb ? 0x8000000000000000ull : 0ull;  // subtract unless swept
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (q < kq) {
                    C av = Ap[4 * q + g][l16];
                    const C bv = Bp[4 * q + g][l16];
                    av.x = __longlong_as_double(__double_as_longlong(av.x) ^ (long long)sg);
                    av.y = __longlong_as_double(__double_as_longlong(av.y) ^ (long long)sg);
                    mr[sc] = F64::run(av.x, bv.x, mr[sc]);
                    mi[sc] = F64::run(av.x, bv.y, mi[sc]);
                    mr[sc] = F64::run(-av.y, bv.y, mr[sc]);
                    mi[sc] = F64::run(av.y, bv.x, mi[sc]);
                }
        });
        if (!NdSweep<T>::DB) __syncthreads();
    }
    // every lane of a wave has the same pivots
    if (lane == 0) {
        double* w = s.pv[threadIdx.x >> 6];
        w[0] = pv.mn;
        w[1] = pv.mx;
        w[2] = pv.bad ? 1.0 : 0.0;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double lo = add ? pst[0] : 1e300, hi = add ? pst[1] : 0.0, bad = add ? pst[2] : 0.0;
        for (int w = 0; w < 4; ++w) {
            lo = fmin(lo, s.pv[w][0]);
            hi = fmax(hi, s.pv[w][1]);
            bad = fmax(bad, s.pv[w][2]);
        }
        pst[0] = lo;
        pst[1] = hi;
        pst[2] = bad;
    }
}

// The operator at up to NF cells of a front, in LDS: one load a thread in place
// of a branch and a load for each entry that is not zero
template <int NF> struct NdCells {
    C cc[NF], ce[NF], cn[NF];
    int x[NF], y[NF];  // x < 0: no cell
    __device__ inline void load(const int* node, int n, const double2* coef, long N, int Nx) {
        for (int e = threadIdx.x; e < 3 * NF; e += 256) {
            const int i = e % NF;
            put(i, e / NF, i < n ? node[i] : -1, coef, N, Nx);
        }
    }
    // plane pl of row i, cell k
    __device__ inline void put(int i, int pl, int k, const double2* coef, long N, int Nx) {
        const int kk = max(k, 0);
        const C c = gload(coef + (long)(pl == 0 ? CC : pl == 1 ? CE : CN) * N + kk);
        (pl == 0 ? cc : pl == 1 ? ce : cn)[i] = c;
        if (pl == 0) {
            x[i] = k < 0 ? -1 : k % Nx;
            y[i] = kk / Nx;
        }
    }
    // entry (i, j) of the symmetrised operator, a unit row where there is no cell
    __device__ inline C entry(int i, int j, int Nx, int Ny) const {
        C z = mk<C>(0, 0);
        const int xi = x[i], xj = x[j], yi = y[i], yj = y[j];
        if (xi < 0 || xj < 0) {
            z = mk<C>(i == j ? 1 : 0, 0);
        } else if (yi == yj) {
            if (i == j) z = cc[i];
            if (xj == (xi + 1 == Nx ? 0 : xi + 1)) z = cadd(z, ce[i]);
            if (xi == (xj + 1 == Nx ? 0 : xj + 1)) z = cadd(z, ce[j]);
        } else if (xi == xj) {
            if (yj == (yi + 1 == Ny ? 0 : yi + 1)) z = cadd(z, cn[i]);
            if (yi == (yj + 1 == Ny ? 0 : yj + 1)) z = cadd(z, cn[j]);
        }
        return z;
    }
};

// Leaves: one workgroup per leaf, its whole front, the separator and then the
// boundary, swept in registers.  The chain of the sweep bounds a workgroup (some
// 50 us for 52 cells), so what counts is how many share a compute unit: a leaf
// of 7 x 7 cells is 80 rows, 15 tiles, 166 VGPRs and 39 kB of LDS, three
// workgroups.  The 16384 leaves of a 1024 x 1024 grid take 1.09 ms; 1.71 ms with
// the boundary behind whole tiles of separator (96 rows, 21 tiles, two
// workgroups), 1.19 ms with the entries gathered one by one from memory.
template <int T>
__global__ __launch_bounds__(256, 3) void k_nd_leaf(NdLev lv, const NdFac* fac, int Nx, int Ny, void* Sv) {
    const NdFac F = fac[blockIdx.y];
    const int p = lv.p, b = lv.b, fr = blockIdx.x;
    const long N = (long)Nx * Ny;
    constexpr int NF = 16 * T;
    __shared__ union {
        NdSweep<T> w;
        NdCells<NF> g;
    } s;
    s.g.load(lv.node + (long)fr * (p + b), p + b, F.coef, N, Nx);
    __syncthreads();
    constexpr int NS = NdSweep<T>::NS;
    d4v mr[NS], mi[NS];
    nd_each_entry<T>([&](auto sc, int v, int i, int j, bool) {
        C z = mk<C>(0, 0);
        if (i < p || j < p) z = s.g.entry(i, j, Nx, Ny);
        mr[sc][v] = z.x;
        mi[sc][v] = z.y;
    });
    __syncthreads();
    nd_sweep<T>(mr, mi, p, s.w, F.pivstat + 3 * (long)(lv.stat + fr), false);
    C* X = (C*)F.arena + lv.offX + (long)fr * p * p;
    C* Q = (C*)F.arena + lv.offQ + (long)fr * p * b;
    C* S = (C*)Sv + ((long)blockIdx.y * lv.cnt + fr) * b * b;
    nd_each_entry<T>([&](auto sc, int v, int i, int j, bool off) {
        const C z = mk<C>(mr[sc][v], mi[sc][v]);
        const int ib = i - p, jb = j - p;
        if (i < p && j < p) {
            gstore(X + i * p + j, z);
            if (off) gstore(X + j * p + i, z);
        } else if (ib >= 0 && ib < b && j < p) {
            gstore(Q + j * b + ib, cneg(z));
        } else if (ib >= 0 && ib < b && jb >= 0 && jb < b) {
            gstore(S + ib * b + jb, z);
            if (off) gstore(S + jb * b + ib, z);
        }
    });
}

static_assert(nd::LEAF_FRONT <= 80, "a leaf fits the largest kernel");
void launch_nd_leaf(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, int Nx, int Ny, void* S) {
    const int f = lv.p + lv.b;
    const dim3 g(lv.cnt, B);
    if (f <= 32) k_nd_leaf<2><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, S);
    else if (f <= 48) k_nd_leaf<3><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, S);
    else if (f <= 64) k_nd_leaf<4><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, S);
    else k_nd_leaf<5><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, S);
}

// ---------------------------------------------------------------------------
// Assembly of a level's fronts (operator entries plus the children's Schur
// complements, padded separator cells as unit rows) and the start of their
// inversion, in one launch:
//   blocks [0, cnt):  the leading 16 T <= 64 separator cells are gathered into
//                     registers and swept; the inverse goes to X when that is
//                     the whole separator, else to D (64 x 64, zero-padded);
//   blocks [cnt, ..): ASM_ROWS rows of F12, and of the lower triangle of F11
//                     when the separator is longer than 64 cells.
// ---------------------------------------------------------------------------
constexpr int ASM_ROWS = 8;
constexpr int NB = 64;  // block of the inversion

template <int T>
__global__ __launch_bounds__(256, 2) void k_nd_front(NdLev lv, const NdFac* fac, int Nx, int Ny, const void* Scv,
                                                  NdInv w, int nchunk) {
    const int q = blockIdx.y, p = lv.p, b = lv.b, f = p + b;
    const NdFac F = fac[q];
    const long N = (long)Nx * Ny;
    const bool inv = (int)blockIdx.x < lv.cnt;
    const int e = (int)blockIdx.x - lv.cnt;
    const int fr = inv ? (int)blockIdx.x : e / nchunk;
    const long job = (long)q * lv.cnt + fr;
    const int* node = lv.node + (long)fr * f;
    const short* cm = lv.cm + (long)fr * 2 * f;
    const C* Sc = (const C*)Scv + ((long)q * lv.cnt * lv.nch + (long)fr * lv.nch) * lv.cb * lv.cb;
    if (inv) {
        constexpr int NF = 16 * T;
        __shared__ union {
            NdSweep<T> w;
            struct {
                NdCells<NF> c;
                short m[2][NF];  // the cells' places in the children
            } g;
        } s;
        const int np = min(p, NB), two = lv.nch > 1 ? 1 : 0;
        s.g.c.load(node, np, F.coef, N, Nx);
        for (int i = threadIdx.x; i < 2 * NF; i += 256) {
            const int c = i / NF, k = i % NF;
            s.g.m[c][k] = k < np && c <= two ? cm[c * f + k] : -1;
        }
        __syncthreads();
        constexpr int NS = NdSweep<T>::NS;
        d4v mr[NS], mi[NS];
        // the children's entries are all loaded before the first is used (entry 0
        // where there is none)
        C o0[NS][4], o1[NS][4];
        nd_each_entry<T>([&](auto sc, int v, int i, int j, bool) {
            const int i0 = s.g.m[0][i], j0 = s.g.m[0][j], i1 = s.g.m[1][i], j1 = s.g.m[1][j];
            o0[sc][v] = gload(Sc + (i0 >= 0 && j0 >= 0 ? (long)i0 * lv.cb + j0 : 0));
            o1[sc][v] = gload(Sc + (i1 >= 0 && j1 >= 0 ? ((long)lv.cb + i1) * lv.cb + j1 : 0));
        });
        nd_each_entry<T>([&](auto sc, int v, int i, int j, bool) {
            const bool k0 = s.g.m[0][i] >= 0 && s.g.m[0][j] >= 0, k1 = s.g.m[1][i] >= 0 && s.g.m[1][j] >= 0;
            const C z = s.g.c.entry(i, j, Nx, Ny);
            mr[sc][v] = z.x + (k0 ? o0[sc][v].x : 0.0) + (k1 ? o1[sc][v].x : 0.0);
            mi[sc][v] = z.y + (k0 ? o0[sc][v].y : 0.0) + (k1 ? o1[sc][v].y : 0.0);
        });
        __syncthreads();
        nd_sweep<T>(mr, mi, np, s.w, F.pivstat + 3 * (long)(lv.stat + fr), false);
        const bool whole = p <= NB;
        C* out = whole ? (C*)F.arena + lv.offX + (long)fr * p * p : (C*)w.D + job * 2 * NB * NB;
        const int ld = whole ? p : NB;
        nd_each_entry<T>([&](auto sc, int v, int i, int j, bool off) {
            const C z = mk<C>(mr[sc][v], mi[sc][v]);
            if (i < np && j < np) {
                gstore(out + i * ld + j, z);
                if (off) gstore(out + j * ld + i, z);
            }
        });
        return;
    }
    const int r0 = (e % nchunk) * ASM_ROWS, j0 = p > NB ? 0 : p, nr = min(ASM_ROWS, p - r0);
    C* Y = (C*)w.Y + job * p * p;
    C* R = (C*)w.R + job * NB * p;
    C* G = (C*)w.F12 + job * p * b;
    for (int j = j0 + (int)threadIdx.x; j < f; j += 256) {
        const int kj = node[j], c0 = cm[j], c1 = lv.nch > 1 ? cm[f + j] : -1;
        // every row's contributions are loaded before the first is used
        C v0[ASM_ROWS], v1[ASM_ROWS];
#pragma unroll
        for (int r = 0; r < ASM_ROWS; ++r) {
            const int i = r0 + min(r, nr - 1), m0 = cm[i], m1 = lv.nch > 1 ? cm[f + i] : -1;
            const bool k0 = m0 >= 0 && c0 >= 0, k1 = m1 >= 0 && c1 >= 0;
            v0[r] = gload(Sc + (k0 ? (long)m0 * lv.cb + c0 : 0));
            v1[r] = gload(Sc + (k1 ? ((long)lv.cb + m1) * lv.cb + c1 : 0));
        }
#pragma unroll
        for (int r = 0; r < ASM_ROWS; ++r) {
            const int i = r0 + min(r, nr - 1), ki = node[i], m0 = cm[i], m1 = lv.nch > 1 ? cm[f + i] : -1;
            C v = mk<C>(0, 0);
            if (ki >= 0 && kj >= 0) v = nd_entry(F.coef, N, Nx, Ny, ki, kj);
            else if (i == j) v = mk<C>(1, 0);
            v = cadd(v, csel(m0 >= 0 && c0 >= 0, v0[r], mk<C>(0, 0)));
            v = cadd(v, csel(m1 >= 0 && c1 >= 0, v1[r], mk<C>(0, 0)));
            if (r < nr) {
                if (j >= p) gstore(G + (long)i * b + (j - p), v);
                else if (j <= (i | (NB - 1))) gstore(Y + (long)i * p + j, v);
                if (j < NB && i >= NB && p > NB) gstore(R + (long)j * p + i, v);  // the first block row
            }
        }
    }
}

void launch_nd_front(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, int Nx, int Ny, const void* Sc,
                     const NdInv& w) {
    const int nch = (lv.b == 0 && lv.p <= NB) ? 0 : (lv.p + ASM_ROWS - 1) / ASM_ROWS;
    const dim3 g(lv.cnt * (1 + nch), B);
    if (lv.p <= 16) k_nd_front<1><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, Sc, w, nch);
    else if (lv.p <= 32) k_nd_front<2><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, Sc, w, nch);
    else if (lv.p <= 48) k_nd_front<3><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, Sc, w, nch);
    else k_nd_front<4><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, Sc, w, nch);
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

// ---------------------------------------------------------------------------
// Small fronts whole, one workgroup each (p <= 16, b <= 16 BT): wave 0 gathers and
// sweeps F11 while the others gather F12, both stay in LDS, then
//   Q = X F12  and  S = F22 - F12^T Q
// by 16 x 16 tiles.  The lowest levels have thousands of such fronts and do little
// arithmetic: what counts is that S is written and the children's read once, and
// that F12 never leaves the chip.  8192 fronts of 8 cells and 44 boundary cells (1024 x
// 1024): 173 us, of which 110 at the copy rate; 332 us as assembly, Q and S in turn.
// 16 cells with 92: 142 us against 184.
// ---------------------------------------------------------------------------
template <int BT>
__global__ __launch_bounds__(256, 2) void k_nd_small(NdLev lv, const NdFac* fac, int Nx, int Ny, const void* Scv,
                                                     void* Sv) {
    constexpr int NF = 16 + 16 * BT, LC = 16 * BT + 1;
    __shared__ NdCells<NF> cl;
    __shared__ short cm[2][NF];  // places in the children; front rows: 16 for F11, then b
    __shared__ C F12[16][LC], Qs[16][LC], X[16][17];
    const int q = blockIdx.y, fr = blockIdx.x, p = lv.p, b = lv.b, f = p + b;
    const NdFac F = fac[q];
    const int t = threadIdx.x, lane = t & 63, l16 = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const long N = (long)Nx * Ny, job = (long)q * lv.cnt + fr;
    const C* Sc = (const C*)Scv + ((long)q * lv.cnt * lv.nch + (long)fr * lv.nch) * lv.cb * lv.cb;
    const int* node = lv.node + (long)fr * f;
    const short* cmg = lv.cm + (long)fr * 2 * f;
    // row r of the padded front -> index in the front, -1 outside
    auto at = [&](int r) { return r < 16 ? (r < p ? r : -1) : (r - 16 < b ? p + r - 16 : -1); };
    for (int e = t; e < 3 * NF; e += 256) {
        const int r = e % NF, pl = e / NF, i = at(r), k = i >= 0 ? node[i] : -1;
        cl.put(r, pl, k, F.coef, N, Nx);
        if (pl > 0) cm[pl - 1][r] = i >= 0 && pl <= lv.nch ? cmg[(pl - 1) * f + i] : -1;
    }
    __syncthreads();
    // the children's part of rows 4 v + g and column c: loaded (entry 0 where there is
    // none) before any is used
    auto kids = [&](int r0, int c, C (&o)[4]) {
        const int n0 = cm[0][c], n1 = cm[1][c];
        C a[4], d[4];
        int m0[4], m1[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            m0[v] = cm[0][r0 + F64::row(lane, v)];
            m1[v] = cm[1][r0 + F64::row(lane, v)];
            a[v] = gload(Sc + (m0[v] >= 0 && n0 >= 0 ? (long)m0[v] * lv.cb + n0 : 0));
            d[v] = gload(Sc + (m1[v] >= 0 && n1 >= 0 ? ((long)lv.cb + m1[v]) * lv.cb + n1 : 0));
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const bool k0 = m0[v] >= 0 && n0 >= 0, k1 = m1[v] >= 0 && n1 >= 0;
            o[v] = mk<C>((k0 ? a[v].x : 0.0) + (k1 ? d[v].x : 0.0), (k0 ? a[v].y : 0.0) + (k1 ? d[v].y : 0.0));
        }
    };
    if (wv == 0) {
        C o[4];
        kids(0, l16, o);
        d4v mr, mi;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const C z = cl.entry(F64::row(lane, v), l16, Nx, Ny);
            mr[v] = z.x + o[v].x;
            mi[v] = z.y + o[v].y;
        }
        NdPiv pv;
        nd_sweep16(mr, mi, p, X, pv);
        C* Xg = (C*)F.arena + lv.offX + (long)fr * p * p;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = F64::row(lane, v);
            const C z = mk<C>(mr[v], mi[v]);
            X[i][l16] = z;
            if (i < p && l16 < p) gstore(Xg + i * p + l16, z);
        }
        if (lane == 0) {
            double* pst = F.pivstat + 3 * (long)(lv.stat + fr);
            pst[0] = pv.mn;
            pst[1] = pv.mx;
            pst[2] = pv.bad ? 1.0 : 0.0;
        }
    } else {
        for (int c = wv - 1; 16 * c < b; c += 3) {
            C o[4];
            kids(0, 16 + 16 * c + l16, o);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = F64::row(lane, v), j = 16 * c + l16;
                const bool ok = i < p && j < b;
                F12[i][j] = csel(ok, cadd(cl.entry(i, 16 + j, Nx, Ny), o[v]), mk<C>(0, 0));
            }
        }
    }
    __syncthreads();
    const int nt = (b + 15) / 16;
    C* Qg = (C*)F.arena + lv.offQ + (long)fr * p * b;
    for (int c = wv; c < nt; c += 4) {
        ndm_acc A;
#pragma unroll
        for (int s = 0; s < 4; ++s) A.step(X[4 * s + g][l16], F12[4 * s + g][16 * c + l16]);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = F64::row(lane, v), j = 16 * c + l16;
            const C z = mk<C>(A.rr[v] - A.ii[v], A.ri[v]);
            Qs[i][j] = z;
            if (i < p && j < b) gstore(Qg + i * b + j, z);
        }
    }
    __syncthreads();
    C* S = (C*)Sv + job * b * b;
    for (int e = wv; e < nt * (nt + 1) / 2; e += 4) {
        int I = 0;
#pragma unroll
        for (int u = 1; u < BT; ++u) I += e >= u * (u + 1) / 2;
        const int J = e - I * (I + 1) / 2, j = 16 * J + l16;
        C o[4];
        kids(16 + 16 * I, 16 + j, o);
        ndm_acc A;
#pragma unroll
        for (int s = 0; s < 4; ++s) A.step(F12[4 * s + g][16 * I + l16], Qs[4 * s + g][j]);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 16 * I + F64::row(lane, v);
            const C z = csub(o[v], mk<C>(A.rr[v] - A.ii[v], A.ri[v]));
            if (i < b && j < b) {
                gstore(S + (long)i * b + j, z);
                if (I != J) gstore(S + (long)j * b + i, z);  // (four lanes write 64 bytes)
            }
        }
    }
}

bool launch_nd_small(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, int Nx, int Ny, const void* Sc,
                     void* S) {
    if (lv.p > 16 || lv.b == 0 || lv.b > 96) return false;
    const dim3 g(lv.cnt, B);
    if (lv.b <= 64) k_nd_small<4><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, Sc, S);
    else k_nd_small<6><<<g, 256, 0, s>>>(lv, fac, Nx, Ny, Sc, S);
    return true;
}

// ---------------------------------------------------------------------------
// Separators longer than 64 cells: block sweeps of 64 on the lower tiles of Y,
// one launch a block.  For block k with inverse D^-1 and block row R_J = M_kJ,
// the workgroup of a lower tile (I, J), I, J != k, forms
//   Z_J = D^-1 R_J  and  M_IJ -= sigma_I R_I^T Z_J, sigma = -1 for swept I < k,
// Z_J once more for every I: the chip is mostly idle here, and a launch of its
// own for Z was 12 us of the chain.  Tile (J, J)'s workgroup also writes Z_J to
// tile (k, J), or -Z_J^T to (J, k) for J > k.  The first workgroup takes tile
// (k + 1, k + 1) in the layout of the sweep and sweeps it: the next D^-1; the last
// one writes its Z for it.  Block rows and inverses are kept twice, the next ones
// written (by whoever updates a tile of block k + 1) while the present ones are
// read.
// The chain of a block is two products and the sweep (23 us).  It bounds a level
// of few fronts: 45 us a block on a 1024 x 1024 grid (separators of 1024 cells
// and less), 47 and a launch more with Z on its own, 76 with both products and the
// sweep in one workgroup before the update's launch.  200 x 120: 35 us, 37.
// ---------------------------------------------------------------------------
// The operands of a product over 64 K rows, 64 rows by TN columns, staged 16 K
// rows at a time through LDS; mm(kk) multiplies K rows kk .. kk + 3 of a stage.
// pa(k, i) and pb(k, j) give an entry's address, clamped where oka / okb, which
// zero it at the store to LDS, are false.
struct NdTile {
    double sAr[16][NB + 16], sAi[16][NB + 16], sBr[16][NB + 16], sBi[16][NB + 16];
};
template <int TN, typename PA, typename PB, typename OA, typename OB, typename MM>
__device__ __attribute__((always_inline)) inline void nd_staged(NdTile& s, PA&& pa, PB&& pb, OA&& oka, OB&& okb,
                                                                MM&& mm) {
    constexpr int NE = TN / 16;
    const int t = threadIdx.x;
    C ra[4], rb[NE];
    auto load = [&](int k0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) ra[e] = gload(pa(k0 + ((t + 256 * e) >> 6), t & 63));
#pragma unroll
        for (int e = 0; e < NE; ++e) rb[e] = gload(pb(k0 + (t + 256 * e) / TN, t % TN));
    };
    load(0);
    for (int k0 = 0; k0 < NB; k0 += 16) {
        __syncthreads();  // the previous stage (or the caller's use of s) is consumed
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k = (t + 256 * e) >> 6, i = t & 63;
            const bool oa = oka(k0 + k, i);
            s.sAr[k][i] = oa ? ra[e].x : 0.0;
            s.sAi[k][i] = oa ? ra[e].y : 0.0;
        }
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            const int k = (t + 256 * e) / TN, j = t % TN;
            const bool ob = okb(k0 + k, j);
            s.sBr[k][j] = ob ? rb[e].x : 0.0;
            s.sBi[k][j] = ob ? rb[e].y : 0.0;
        }
        __syncthreads();
        if (k0 + 16 < NB) load(k0 + 16);
#pragma unroll
        for (int kk = 0; kk < 16; kk += 4) mm(kk);
    }
}
// Accumulators of a 64 x TN tile on four waves of 32 x TN / 2, three real products
// per complex one
template <int TN> struct NdAcc {
    static constexpr int BN = TN / 32;
    d4v c1[2][BN] = {}, c2[2][BN] = {}, c3[2][BN] = {};
    __device__ __attribute__((always_inline)) inline void mul(const NdTile& s, int kk) {
        const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, wr = wv >> 1, wc = wv & 1;
        const int lr = lane & 15, lk = lane >> 4;
        double ar[2], ai[2], as[2], br[BN], bi[BN], bs[BN];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            ar[x] = s.sAr[kk + lk][wr * 32 + x * 16 + lr];
            ai[x] = s.sAi[kk + lk][wr * 32 + x * 16 + lr];
            as[x] = ar[x] + ai[x];
        }
#pragma unroll
        for (int y = 0; y < BN; ++y) {
            br[y] = s.sBr[kk + lk][wc * (TN / 2) + y * 16 + lr];
            bi[y] = s.sBi[kk + lk][wc * (TN / 2) + y * 16 + lr];
            bs[y] = br[y] + bi[y];
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < BN; ++y) c1[x][y] = F64::run(ar[x], br[y], c1[x][y]);
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < BN; ++y) c2[x][y] = F64::run(ai[x], bi[y], c2[x][y]);
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < BN; ++y) c3[x][y] = F64::run(as[x], bs[y], c3[x][y]);
    }
    // f(i, j, value) for this thread's entries of the product
    template <typename F> __device__ __attribute__((always_inline)) inline void each(F&& f) const {
        const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, wr = wv >> 1, wc = wv & 1;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < BN; ++y)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    f(wr * 32 + x * 16 + F64::row(lane, v), wc * (TN / 2) + y * 16 + (lane & 15),
                      mk<C>(c1[x][y][v] - c2[x][y][v], c3[x][y][v] - c1[x][y][v] - c2[x][y][v]));
    }
};

__global__ __launch_bounds__(256, 2) void k_nd_block(NdLev lv, const NdFac* fac, NdInv w, int k, int nb, int ntile) {
    __shared__ union {
        NdTile s;
        NdSweep<4> w;
    } u;
    NdTile& s = u.s;
    const int fr = blockIdx.x / (ntile + 1), q = blockIdx.y, p = lv.p;
    const long job = (long)q * lv.cnt + fr;
    // tile number -> (I, J), I >= J, over the blocks other than k; number 0 and
    // that of (k + 1, k + 1) change places, and the last workgroup does what that of
    // (k + 1, k + 1) has no time for
    const bool more = k + 1 < nb;
    const int en = more ? k * (k + 3) / 2 : 0, e0 = blockIdx.x % (ntile + 1);
    const bool extra = e0 == ntile;
    const int e = e0 == 0 || extra ? en : e0 == en ? 0 : e0;
    int I = (int)((sqrtf(8.0f * e + 1.0f) - 1.0f) * 0.5f);
    while ((I + 1) * (I + 2) / 2 <= e) ++I;
    while (I * (I + 1) / 2 > e) --I;
    int J = e - I * (I + 1) / 2;
    I += I >= k;
    J += J >= k;
    const int kw = min(NB, p - k * NB), iw = min(NB, p - I * NB), jw = min(NB, p - J * NB);
    C* Yf = (C*)w.Y + job * p * p;
    C* Y = Yf + (long)I * NB * p + J * NB;
    const C* R0 = (const C*)((k & 1) ? w.R1 : w.R) + job * NB * p;
    C* R1 = (C*)((k & 1) ? w.R : w.R1) + job * NB * p;
    const C* D = (const C*)w.D + (job * 2 + (k & 1)) * NB * NB;
    C* Dn = (C*)w.D + (job * 2 + (~k & 1)) * NB * NB;
    const int t = threadIdx.x, lane = t & 63, lr = lane & 15, lk = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6), wr = wv >> 1, wc = wv & 1;
    // Z_J, this thread's entries
    C z[2][2][4];
    {
        NdAcc<NB> A;
        nd_staged<NB>(
            s, [&](int kk, int i) { return D + kk * NB + i; },
            [&](int kk, int j) { return R0 + (long)min(kk, kw - 1) * p + J * NB + min(j, jw - 1); },
            [&](int kk, int i) { return kk < kw && i < kw; }, [&](int kk, int j) { return kk < kw && j < jw; },
            [&](int kk) { A.mul(s, kk); });
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    z[x][y][v] = mk<C>(A.c1[x][y][v] - A.c2[x][y][v],
                                       A.c3[x][y][v] - A.c1[x][y][v] - A.c2[x][y][v]);
    }
    // sum over the 64 rows of R_I^T Z_J: R_I staged from memory, Z_J from registers
    auto product = [&](auto&& mm) {
        C ra[4];
        auto load = [&](int k0) {
#pragma unroll
            for (int h = 0; h < 4; ++h)
                ra[h] = gload(R0 + (long)min(k0 + ((t + 256 * h) >> 6), kw - 1) * p + I * NB + min(t & 63, iw - 1));
        };
        load(0);
        static_for<0, 4>([&](auto sc) {
            constexpr int st = decltype(sc)::value, k0 = 16 * st;
            __syncthreads();  // the previous stage is consumed
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const int kr = (t + 256 * h) >> 6, i = t & 63;
                const bool ok = k0 + kr < kw && i < iw;
                s.sAr[kr][i] = ok ? ra[h].x : 0.0;
                s.sAi[kr][i] = ok ? ra[h].y : 0.0;
            }
            if (wr == (st >> 1)) {
#pragma unroll
                for (int y = 0; y < 2; ++y)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        s.sBr[F64::row(lane, v)][wc * 32 + y * 16 + lr] = z[st & 1][y][v].x;
                        s.sBi[F64::row(lane, v)][wc * 32 + y * 16 + lr] = z[st & 1][y][v].y;
                    }
            }
            __syncthreads();
            if (st < 3) load(k0 + 16);
#pragma unroll
            for (int kk = 0; kk < 16; kk += 4) mm(kk);
        });
    };
    // what else becomes of Z_J, by the workgroup of tile (J, J)
    auto spread = [&]() {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int i = wr * 32 + x * 16 + F64::row(lane, v), j = wc * 32 + y * 16 + lr;
                    if (i < kw && j < jw) {
                        if (J < k) gstore(Yf + (long)(k * NB + i) * p + J * NB + j, z[x][y][v]);
                        else gstore(Yf + (long)(J * NB + j) * p + k * NB + i, cneg(z[x][y][v]));
                        if (more && J == k + 1) gstore(R1 + (long)j * p + k * NB + i, cneg(z[x][y][v]));
                    }
                }
    };
    if (extra) {
        for (int i = t; i < NB * NB; i += 256) {  // tile (k, k) <- D^-1
            const int r = i >> 6, j = i & 63;
            if (r < kw && j < kw) gstore(Yf + (long)(k * NB + r) * p + k * NB + j, gload(D + i));
        }
        if (more) spread();
        return;
    }
    if (!more || I != k + 1 || J != k + 1) {
        NdAcc<NB> A;
        product([&](int kk) { A.mul(s, kk); });
        const double sg = I < k ? 1.0 : -1.0;
        A.each([&](int i, int j, C v) {
            if (i < iw && j < jw) {
                C* y = Y + (long)i * p + j;
                const C m = cadd(gload(y), cscale(v, sg));
                gstore(y, m);
                if (more && I == k + 1) gstore(R1 + (long)i * p + J * NB + j, m);
                else if (more && J == k + 1) gstore(R1 + (long)j * p + I * NB + i, m);
            }
        });
        if (I == J) spread();
        return;
    }
    // the lower 16 x 16 tiles in the layout of the sweep
    constexpr int NS = NdSweep<4>::NS;
    d4v mr[NS], mi[NS], c1[NS] = {}, c2[NS] = {}, c3[NS] = {};
    product([&](int kk) {
        nd_each_tile<4>([&](auto sc, int ti, int tj) {
            const double ar = s.sAr[kk + lk][16 * ti + lr], ai = s.sAi[kk + lk][16 * ti + lr];
            const double br = s.sBr[kk + lk][16 * tj + lr], bi = s.sBi[kk + lk][16 * tj + lr];
            c1[sc] = F64::run(ar, br, c1[sc]);
            c2[sc] = F64::run(ai, bi, c2[sc]);
            c3[sc] = F64::run(ar + ai, br + bi, c3[sc]);
        });
    });
    nd_each_entry<4>([&](auto sc, int v, int i, int j, bool) {
        const C y = gload(Y + (long)min(i, iw - 1) * p + min(j, iw - 1));
        mr[sc][v] = y.x;
        mi[sc][v] = y.y;
    });
    nd_each_entry<4>([&](auto sc, int v, int i, int j, bool) {
        const bool ok = i < iw && j < iw;
        const double re = c1[sc][v] - c2[sc][v], im = c3[sc][v] - c1[sc][v] - c2[sc][v];
        mr[sc][v] = ok ? mr[sc][v] - re : (i == j ? 1.0 : 0.0);
        mi[sc][v] = ok ? mi[sc][v] - im : 0.0;
    });
    __syncthreads();
    nd_sweep<4>(mr, mi, iw, u.w, fac[q].pivstat + 3 * (long)(lv.stat + fr), true);
    nd_each_entry<4>([&](auto sc, int v, int i, int j, bool off) {
        const C x = mk<C>(mr[sc][v], mi[sc][v]);
        gstore(Dn + i * NB + j, x);
        if (off) gstore(Dn + j * NB + i, x);
    });
}

// X (whole) from the lower tiles of Y
__global__ __launch_bounds__(256) void k_nd_mirror(NdLev lv, const NdFac* fac, NdInv w) {
    __shared__ C tile[32][33];
    const int q = blockIdx.y, p = lv.p, np = (p + 31) / 32;
    const int fr = blockIdx.x / (np * np), e = blockIdx.x % (np * np), I = e / np, J = e % np;
    if (J > I) return;
    const long job = (long)q * lv.cnt + fr;
    const C* Y = (const C*)w.Y + job * p * p;
    C* X = (C*)fac[q].arena + lv.offX + (long)fr * p * p;
    const int c = threadIdx.x & 31, r0 = threadIdx.x >> 5;
    for (int r = r0; r < 32; r += 8) {
        const int i = I * 32 + r, j = J * 32 + c;
        if (i < p && j < p) {
            const C v = gload(Y + (long)i * p + j);
            tile[r][c] = v;
            gstore(X + (long)i * p + j, v);
        }
    }
    if (I == J) return;
    __syncthreads();
    for (int r = r0; r < 32; r += 8) {
        const int i = J * 32 + r, j = I * 32 + c;
        if (i < p && j < p) gstore(X + (long)i * p + j, tile[c][r]);
    }
}

void launch_nd_invert(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, const NdInv& w) {
    if (lv.p <= NB) return;
    const int nb = (lv.p + NB - 1) / NB, nt = (nb - 1) * nb / 2, np = (lv.p + 31) / 32;
    for (int k = 0; k < nb; ++k) {
        k_nd_block<<<dim3(lv.cnt * (nt + 1), B), 256, 0, s>>>(lv, fac, w, k, nb, nt);
    }
    k_nd_mirror<<<dim3(lv.cnt * np * np, B), 256, 0, s>>>(lv, fac, w);
}

// ---------------------------------------------------------------------------
// Batched complex products of a level on MFMA, complex values as three real
// products (Gauss):
//   SCHUR = false:  Q = X F12                          (p x b, K = p)
//   SCHUR = true:   S = gather(children) - F12^T Q     (b x b, K = p),
// the latter only on tiles that meet the lower triangle; entries below the
// diagonal are written to both halves.  Operands are staged KT rows of K at a
// time through LDS, the next stage loading into registers meanwhile.
//
// Tiles of 32 x 32, one accumulator set per wave: with few fronts (512 x 2048
// at four of them) larger tiles leave CUs without work, and with many the
// epilogue of S (gathers from two children and two writes of each entry)
// dominates and wants workgroups to overlap with.  All levels of a 1024 x 1024
// grid, S and Q: 128 x 64 tiles 5.04 + 1.53 ms, 64 x 64 4.33 + 1.26, 64 x 32
// 4.05 + 1.32, 32 x 32 3.98 + 1.25; of a 200 x 120 grid 152 + 95 us against 89 + 53.
// ---------------------------------------------------------------------------
template <int TM, int TN, int KT, int WR, int WC, bool SCHUR>
__global__ __launch_bounds__(64 * WR * WC, 2) void k_nd_gemm(NdLev lv, const NdFac* fac, const void* F12v,
                                                        const void* Scv, void* Sv, int ntm, int ntn) {
    using M = mfma_t<R>;
    using acc_t = typename M::acc;
    constexpr int NT = 64 * WR * WC;
    constexpr int WM = TM / WR, WN = TN / WC, BM = WM / 16, BN = WN / 16;
    constexpr int PA = TM + 16, PB = TN + 16;
    constexpr int AE = TM * KT / NT, BE = TN * KT / NT;
    static_assert(AE >= 1 && BE >= 1 && BM >= 1 && BN >= 1, "tile shape");
    __shared__ struct {
        double ar[KT][PA], ai[KT][PA], br[KT][PB], bi[KT][PB];
    } sh;
    auto &sAr = sh.ar, &sAi = sh.ai;
    auto &sBr = sh.br, &sBi = sh.bi;
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
    // clamped addresses; entries outside are zeroed when they are stored to LDS
    // (a select here would wait for the load)
    const C* Ag = SCHUR ? F12 : X;
    const int lda = SCHUR ? b : p;  // X is symmetric: read along its rows
    auto load = [&](int kb) {
#pragma unroll
        for (int e = 0; e < AE; ++e) {
            const int id = t + NT * e, k = kb + id / TM, i = i0 + id % TM;
            ra[e] = gload(Ag + (long)min(k, p - 1) * lda + min(i, Mr - 1));
        }
#pragma unroll
        for (int e = 0; e < BE; ++e) {
            const int id = t + NT * e, k = kb + id / TN, j = j0 + id % TN;
            rb[e] = gload(Bg + (long)min(k, p - 1) * b + min(j, b - 1));
        }
    };
    auto store = [&](int kb) {
#pragma unroll
        for (int e = 0; e < AE; ++e) {
            const int id = t + NT * e, k = id / TM, i = id % TM;
            const bool ok = kb + k < p && i0 + i < Mr;
            sAr[k][i] = ok ? ra[e].x : 0.0;
            sAi[k][i] = ok ? ra[e].y : 0.0;
        }
#pragma unroll
        for (int e = 0; e < BE; ++e) {
            const int id = t + NT * e, k = id / TN, j = id % TN;
            const bool ok = kb + k < p && j0 + j < b;
            sBr[k][j] = ok ? rb[e].x : 0.0;
            sBi[k][j] = ok ? rb[e].y : 0.0;
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
        store(kb);
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
    if (!SCHUR) {
#pragma unroll
        for (int x = 0; x < BM; ++x)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = i0 + wr * WM + x * 16 + M::row(lane, v);
#pragma unroll
                for (int y = 0; y < BN; ++y) {
                    const int j = j0 + wc * WN + y * 16 + lr;
                    if (i < p && j < b)
                        gstore(Q + (long)i * b + j, mk<C>(c1[x][y][v] - c2[x][y][v], c3[x][y][v] - c1[x][y][v] - c2[x][y][v]));
                }
            }
        return;
    }
    // S: the children's entries of a 16 x 16 block are loaded before they are
    // used (entry 0 where there is none), the block is written row by row, and
    // its mirror image row by row after a transpose through the wave's LDS
    const short *cm = lv.cm + (long)fr * 2 * (p + b) + p, *cm1 = cm + (p + b);
    const C* Sc = (const C*)Scv + ((long)q * lv.cnt * lv.nch + (long)fr * lv.nch) * lv.cb * lv.cb;
    C* S = (C*)Sv + job * b * b;
    const bool two = lv.nch > 1;
    C(*tr)[17] = (C(*)[17])((C*)&sAr[0][0] + wv * 16 * 17);  // (the stages are consumed)
    static_assert(sizeof(C) * WR * WC * 16 * 17 <= sizeof(double) * 2 * KT * (PA + PB), "transpose tiles fit the stages");
#pragma unroll
    for (int x = 0; x < BM; ++x) {
        const int ib = i0 + wr * WM + x * 16;
        int m0[4], m1[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = min(ib + M::row(lane, v), b - 1);
            m0[v] = cm[i];
            m1[v] = two ? cm1[i] : -1;
        }
#pragma unroll
        for (int y = 0; y < BN; ++y) {
            const int jb = j0 + wc * WN + y * 16, j = jb + lr;
            if (jb > ib || jb >= b) continue;  // uniform: above the diagonal, or outside
            const int n0 = cm[min(j, b - 1)], n1 = two ? cm1[min(j, b - 1)] : -1;
            C o0[4], o1[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                o0[v] = gload(Sc + (m0[v] >= 0 && n0 >= 0 ? (long)m0[v] * lv.cb + n0 : 0));
                o1[v] = gload(Sc + (m1[v] >= 0 && n1 >= 0 ? ((long)lv.cb + m1[v]) * lv.cb + n1 : 0));
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const bool k0 = m0[v] >= 0 && n0 >= 0, k1 = m1[v] >= 0 && n1 >= 0;
                const double re = c1[x][y][v] - c2[x][y][v], im = c3[x][y][v] - c1[x][y][v] - c2[x][y][v];
                const C z = mk<C>((k0 ? o0[v].x : 0.0) + (k1 ? o1[v].x : 0.0) - re,
                                  (k0 ? o0[v].y : 0.0) + (k1 ? o1[v].y : 0.0) - im);
                const int i = ib + M::row(lane, v);
                if (i < b && j < b) gstore(S + (long)i * b + j, z);
                tr[M::row(lane, v)][lr] = z;
            }
            if (ib == jb) continue;  // a diagonal block is whole
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int jj = jb + M::row(lane, v), i = ib + lr;
                if (i < b && jj < b) gstore(S + (long)jj * b + i, tr[lr][M::row(lane, v)]);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
}

void launch_nd_gemm(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, const void* F12,
                    const void* Sc, void* S, bool schur) {
    auto go = [&](auto kern, int TM, int TN, int NT) {
        const int ntm = ((schur ? lv.b : lv.p) + TM - 1) / TM, ntn = (lv.b + TN - 1) / TN;
        kern<<<dim3(lv.cnt * ntm * ntn, B), NT, 0, s>>>(lv, fac, F12, Sc, S, ntm, ntn);
    };
    if (schur) go(k_nd_gemm<32, 32, 16, 2, 2, true>, 32, 32, 256);
    else go(k_nd_gemm<32, 32, 16, 2, 2, false>, 32, 32, 256);
}

// smallest and largest pivot and zero-pivot flag of each factor's fronts
constexpr int STAT_T = 1024;  // (256, one load after another: 60 us for the 32767 fronts of 1024 x 1024; 17 so)
__global__ __launch_bounds__(STAT_T) void k_nd_stat(const NdFac* fac, int nfronts, double* out) {
    const double* ps = fac[blockIdx.x].pivstat;
    double mn = __builtin_huge_val(), mx = 0, z = 0;
#pragma unroll 4
    for (int i = threadIdx.x; i < nfronts; i += STAT_T) {
        mn = fmin(mn, ps[3 * i]);
        mx = fmax(mx, ps[3 * i + 1]);
        z = fmax(z, ps[3 * i + 2]);
    }
    __shared__ double r[3][STAT_T];
    r[0][threadIdx.x] = mn;
    r[1][threadIdx.x] = mx;
    r[2][threadIdx.x] = z;
    __syncthreads();
    for (int o = STAT_T / 2; o > 0; o >>= 1) {
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
    k_nd_stat<<<B, STAT_T, 0, s>>>(fac, nfronts, out);
}

// ---------------------------------------------------------------------------
// Reduced solve for one right-hand side: a launch per level and direction,
// memory-bound on the leaves and bound by latency on all levels above, so a
// kernel keeps its chain short: what addresses the matrix does not depend on the
// vectors, and its loads are issued before the gathers (list, then value) that
// the vectors take; no workgroup barrier comes before the products; edges are
// clamped addresses against a zero operand, not branches.  A solve on a 512 x 512
// grid: 295 us in 30 launches (leaves 17 up and 58 down, 4.7 TB/s; the levels above
// 3 to 11 each), against 490 us with v staged by the workgroup before it loads Q
// and rows of X and Q in turn (leaves 26 and 111, levels 9 to 19).
//
// Grid row y is a solve of its own: the sideband factors of a modulated device are
// applied in one launch a level (three on 500 x 200: 8.2 ms a solve, 10.9 one by one).
// A lone solve passes its own arguments only.
//
// Upward step of a level: the separator values
//   v = scaled right-hand side + children's updates
// and the boundary update u = children's updates - Q^T v.  A task is CL boundary
// columns of one front: the lanes of a wave are CL columns by 64 / CL rows, and
// KW waves take a part of the separator each.
// ---------------------------------------------------------------------------
constexpr int UP_MU = 8;  // rows of Q a lane loads at a time

template <int CL, int KW, int NS>
__global__ __launch_bounds__(KW > 4 ? 64 * KW : 256) void k_nd_up(NdLev lv, NdBatch<NS> bt, int Nx, int nchunk) {
    const NdVec& z = bt.s[NS > 1 ? blockIdx.y : 0].z;
    const void* arena = bt.s[NS > 1 ? blockIdx.y : 0].arena;
    constexpr int RG = 64 / CL, NW = KW > 4 ? KW : 4;  // row groups of a wave, waves
    __shared__ C vs[NW][64];
    __shared__ C red[KW > 1 ? KW : 1][CL];
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wk = KW > 1 ? wv : 0;
    const int task = KW > 1 ? (int)blockIdx.x : (int)blockIdx.x * NW + wv;
    if (KW == 1 && task >= lv.cnt * nchunk) return;  // (no barrier follows)
    const int fr = task / nchunk, ch = task % nchunk;
    const int p = lv.p, b = lv.b, f = p + b, nch = lv.nch;
    const int src = z.ridx ? z.ridx[0] : 0;
    const double2* in = z.in + (long)src * z.rs;
    const double2* uc = z.u + lv.offUc + (long)fr * nch * lv.cb;
    const int* node = lv.node + (long)fr * f;
    const short* cm = lv.cm + (long)fr * 2 * f;
    const int col = lane % CL, rg = lane / CL, j = ch * CL + col;
    const C* Q = (const C*)arena + lv.offQ + (long)fr * p * b + min(j, b - 1);
    auto kids = [&](int m0, int m1) {
        C a = mk<C>(0, 0);
        if (nch > 0) {
            const C a0 = uc[max(m0, 0)];
            a = csel(m0 >= 0, a0, a);
            if (nch > 1) {
                const C a1 = uc[lv.cb + max(m1, 0)];
                a = cadd(a, csel(m1 >= 0, a1, mk<C>(0, 0)));
            }
        }
        return a;
    };
    // children's share of this task's columns, for the first lane group
    const bool fin = wk == 0 && rg == 0 && j < b;
    int n0 = -1, n1 = -1;
    if (nch > 0 && b > 0) n0 = cm[p + min(j, b - 1)];
    if (nch > 1 && b > 0) n1 = cm[f + p + min(j, b - 1)];
    const int PW = KW > 1 ? (p + KW - 1) / KW : p, ib = wk * PW, ie = min(p, ib + PW);
    C acc = mk<C>(0, 0);
    for (int i0 = ib; i0 < ie; i0 += 64) {
        const int n = min(64, ie - i0), i = i0 + min(lane, n - 1);
        const int k = node[i], m0 = nch > 0 ? cm[i] : -1, m1 = nch > 1 ? cm[f + i] : -1;
        C q[UP_MU];
        auto load = [&](int r0) {
#pragma unroll
            for (int m = 0; m < UP_MU; ++m) q[m] = gload(Q + (long)(i0 + min(r0 + rg + RG * m, n - 1)) * b);
        };
        if (b > 0) load(0);
        const int kk = max(k, 0);
        C v = cadd(cmul(in[kk], cmul(z.six[kk % Nx], z.siy[kk / Nx])), kids(m0, m1));
        v = csel(k >= 0 && lane < n, v, mk<C>(0, 0));
        if (ch == 0 && lane < n) z.v[lv.offV + (long)fr * p + i] = v;
        if (b == 0) continue;
        __builtin_amdgcn_wave_barrier();
        vs[wv][lane] = v;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int r0 = 0; r0 < n; r0 += UP_MU * RG) {
            if (r0 > 0) load(r0);
#pragma unroll
            for (int m = 0; m < UP_MU; ++m) {
                const int r = r0 + rg + RG * m;
                const C x = csel(r < n, vs[wv][min(r, 63)], mk<C>(0, 0));
                acc = cfma(q[m], x, acc);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (b == 0) return;
    const C own = kids(n0, n1);
#pragma unroll
    for (int o = CL; o < 64; o <<= 1) {
        acc.x += shfl_x(acc.x, o);
        acc.y += shfl_x(acc.y, o);
    }
    if (KW > 1) {
        if (rg == 0) red[wk][col] = acc;
        __syncthreads();
        if (!fin) return;
#pragma unroll
        for (int w = 1; w < KW; ++w) acc = cadd(acc, red[w][col]);
    }
    if (fin) z.u[lv.offU + (long)fr * b + j] = csub(own, acc);
}

// Downward step: x = X v - Q x_boundary.  A task is RW rows of one front, whose
// columns (of X, then of Q) are spread over the lanes of KW waves; the sums over
// the lanes are folded so that each exchange halves the rows a lane holds.
template <int RW, int KW, int NS>
__global__ __launch_bounds__(256) void k_nd_down(NdLev lv, NdBatch<NS> bt, int Nx, int nchunk) {
    const NdVec& z = bt.s[NS > 1 ? blockIdx.y : 0].z;
    const void* arena = bt.s[NS > 1 ? blockIdx.y : 0].arena;
    constexpr int MU = RW >= 8 ? 2 : 8 / RW;  // columns a lane takes at a time
    __shared__ C red[KW][RW];
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wk = KW > 1 ? wv : 0;
    const int task = KW > 1 ? (int)blockIdx.x : (int)blockIdx.x * 4 + wv;
    if (KW == 1 && task >= lv.cnt * nchunk) return;  // (no barrier follows)
    const int fr = task / nchunk, r0 = (task % nchunk) * RW;
    const int p = lv.p, b = lv.b, f = p + b;
    const int src = z.ridx ? z.ridx[0] : 0;
    double2* out = z.out + (long)src * z.rs;
    double2* xg = z.x;
    const double2* vb = z.v + lv.offV + (long)fr * p;
    const int* node = lv.node + (long)fr * f;
    const C* X = (const C*)arena + lv.offX + (long)fr * p * p;
    const C* Q = (const C*)arena + lv.offQ + (long)fr * p * b;
    // the row that the folds leave in this lane, its cell and scaling
    constexpr int FB = RW == 8 ? 3 : RW == 4 ? 2 : RW == 2 ? 1 : 0;  // folds
    const int row = lane >> (6 - FB), ni = node[min(r0 + row, p - 1)];
    C acc[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) acc[r] = mk<C>(0, 0);
    for (int k0 = wk * 64 + lane; __any(k0 < f); k0 += 64 * KW * MU) {
        C a[MU][RW], x[MU];
        int kn[MU];
#pragma unroll
        for (int m = 0; m < MU; ++m) {
            const int k = min(k0 + 64 * KW * m, f - 1);
            kn[m] = node[k];
            x[m] = vb[min(k, p - 1)];
        }
#pragma unroll
        for (int m = 0; m < MU; ++m) {
            const int k = min(k0 + 64 * KW * m, f - 1);
            const bool q = k >= p;
            const C* M = q ? Q + (k - p) : X + k;
            const int ld = q ? b : p;
#pragma unroll
            for (int r = 0; r < RW; ++r) a[m][r] = gload(M + (long)min(r0 + r, p - 1) * ld);
        }
#pragma unroll
        for (int m = 0; m < MU; ++m) {
            const int k = k0 + 64 * KW * m;
            const C xb = xg[max(kn[m], 0)];
            C y = csel(k < p, x[m], csel(kn[m] >= 0, cneg(xb), mk<C>(0, 0)));
            y = csel(k < f, y, mk<C>(0, 0));
#pragma unroll
            for (int r = 0; r < RW; ++r) acc[r] = cfma(a[m][r], y, acc[r]);
        }
    }
    const int nc = max(ni, 0);
    const C sc = cmul(z.sox[nc % Nx], z.soy[nc / Nx]);
    static_for<0, FB>([&](auto s) {
        constexpr int h = RW >> (decltype(s)::value + 1), o = 32 >> decltype(s)::value;
        const bool up = (lane & o) != 0;
#pragma unroll
        for (int r = 0; r < h; ++r) {
            const C keep = csel(up, acc[r + h], acc[r]), give = csel(up, acc[r], acc[r + h]);
            acc[r] = mk<C>(keep.x + shfl_x(give.x, o), keep.y + shfl_x(give.y, o));
        }
    });
#pragma unroll
    for (int o = 32 >> FB; o > 0; o >>= 1) {
        acc[0].x += shfl_x(acc[0].x, o);
        acc[0].y += shfl_x(acc[0].y, o);
    }
    const bool head = (lane & ((64 >> FB) - 1)) == 0;
    C y = acc[0];
    if (KW > 1) {
        if (head) red[wk][row] = y;
        __syncthreads();
        if (wk > 0 || !head) return;
#pragma unroll
        for (int w = 1; w < KW; ++w) y = cadd(y, red[w][row]);
    }
    if (head && r0 + row < p && ni >= 0) {
        xg[ni] = y;
        out[ni] = cmul(y, sc);
    }
}

// The widest task that still makes ND_WAVES waves (one for each SIMD); below,
// narrower ones with the sums split over the waves of a workgroup.  Some 390
// applications on a 512 x 512 grid with 512 / 1024 / 2048 / 4096 waves: 158 / 146 /
// 160 / 186 ms; a modulated device of 500 x 200: 10.6 / 10.5 / 11.4 / 11.8 ms.
constexpr long ND_WAVES = 1024;

template <int NS>
void launch_nd_up(hipStream_t s, const NdLev& lv, const NdBatch<NS>& bt, int nb, int Nx) {
    auto chunks = [&](int CL) { return std::max(1, (lv.b + CL - 1) / CL); };
    auto tasks = [&](int CL) { return (long)lv.cnt * chunks(CL) * nb; };
    auto go = [&](auto kern, int CL, int KW) {
        const int n = lv.cnt * chunks(CL), per = KW > 1 ? 1 : 4, NT = KW > 4 ? 64 * KW : 256;
        kern<<<dim3((n + per - 1) / per, nb), NT, 0, s>>>(lv, bt, Nx, chunks(CL));
    };
    if (lv.p <= 16 && tasks(64) >= ND_WAVES) go(k_nd_up<64, 1, NS>, 64, 1);
    else if (tasks(32) >= ND_WAVES) go(k_nd_up<32, 1, NS>, 32, 1);
    else if (tasks(16) >= ND_WAVES) go(k_nd_up<16, 1, NS>, 16, 1);
    else if (lv.p <= 64 || tasks(16) * 4 >= ND_WAVES) go(k_nd_up<16, 4, NS>, 16, 4);
    else go(k_nd_up<8, 16, NS>, 8, 16);
}
template <int NS>
void launch_nd_down(hipStream_t s, const NdLev& lv, const NdBatch<NS>& bt, int nb, int Nx) {
    auto chunks = [&](int RW) { return (lv.p + RW - 1) / RW; };
    auto tasks = [&](int RW) { return (long)lv.cnt * chunks(RW) * nb; };
    auto go = [&](auto kern, int RW, int KW) {
        const int n = lv.cnt * chunks(RW), per = KW > 1 ? 1 : 4;
        kern<<<dim3((n + per - 1) / per, nb), 256, 0, s>>>(lv, bt, Nx, chunks(RW));
    };
    if (tasks(8) >= ND_WAVES) go(k_nd_down<8, 1, NS>, 8, 1);
    else if (tasks(4) * 4 >= ND_WAVES) go(k_nd_down<4, 4, NS>, 4, 4);
    else if (tasks(2) * 4 >= ND_WAVES) go(k_nd_down<2, 4, NS>, 2, 4);
    else go(k_nd_down<1, 4, NS>, 1, 4);
}
template void launch_nd_up(hipStream_t, const NdLev&, const NdBatch<1>&, int, int);
template void launch_nd_up(hipStream_t, const NdLev&, const NdBatch<ND_SOLVES>&, int, int);
template void launch_nd_down(hipStream_t, const NdLev&, const NdBatch<1>&, int, int);
template void launch_nd_down(hipStream_t, const NdLev&, const NdBatch<ND_SOLVES>&, int, int);

// ---------------------------------------------------------------------------
// The reduced solve for 2 .. 16 sources on MFMA (16 x 16 x 4).  Work vectors
// keep the sources innermost (entry (i, s) at 16 i + s, zero past the active
// ones), so a row of 16 sources is one contiguous piece of every gather and
// the product's B operand; the factor streams straight into the A operand, so
// it is read once for all sources.  With one wave a tile of 16 outputs, a
// CU's four SIMDs consume about 16 B of factor a clock, above its share of the
// memory rate, so the products cost no more than the stream.  Levels with few tiles split K over KS waves of a workgroup.
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
    C v = mk<C>(0, 0);
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

// f(r, value) for the tile's entries v = r of this wave's lanes; with KS waves their
// tiles are added through LDS, entry r by wave r
template <int KS, typename F>
__device__ __attribute__((always_inline)) inline void ndm_finish(const C (&z)[4], C (*red)[4][64], int wv, int lane,
                                                                 F&& f) {
    if constexpr (KS == 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) f(r, z[r]);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wv][r][lane] = z[r];
        __syncthreads();
        if (wv >= 4) return;
        C s = red[0][wv][lane];
#pragma unroll
        for (int w = 1; w < KS; ++w) s = cadd(s, red[w][wv][lane]);
        f(0, s);
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
    // what this wave's entries are subtracted from
    C* u = up + (lv.offU + (long)fr * b) * 16 + l16;
    constexpr int NR = KS == 1 ? 4 : 1;
    int row[NR];
    C old[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        row[r] = j0 + M::row(lane, KS == 1 ? r : wv & 3);
        old[r] = gload(u + (long)min(row[r], b - 1) * 16);
    }
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
    ndm_finish<KS>(z, red, wv, lane, [&](int r, C s) {
        if (row[r] < b) gstore(u + (long)row[r] * 16, csub(old[r], s));
    });
}

// x = X v - Q x_boundary, 16 separator cells a tile.  X is symmetric, so its
// operand is read along rows (16 neighbouring columns); a lane reads four
// neighbouring entries of its row of Q and the K order is permuted to match.
// A level of few tiles is bound by the chain list, value, product: the list is read
// two groups ahead, and the waves' tiles are added by four of them (13 us for 256 x
// 1020 on two fronts, 23 us with the list read in turn and one wave adding; 16
// sources on 384 x 512 1.66 -> 1.49 ms).
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
    // the cells of this wave's entries (-1: none)
    constexpr int NR = KS == 1 ? 4 : 1;
    int cell[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int i = i0 + M::row(lane, KS == 1 ? r : wv & 3);
        cell[r] = i < p ? node[i] : -1;
    }
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
    // four consecutive columns k0 + 4 kg .. + 3 per lane (b is a multiple of 4), of
    // two groups of 16; the next two groups' cells are looked up meanwhile
    auto look = [&](int k0, int (&n)[2][4]) {
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int k = k0 + KS * 16 * g + 4 * kg + q;
                n[g][q] = node[p + min(k, b - 1)];
            }
    };
    int n[2][4];
    const int kb = KS == 1 ? 0 : 16 * wv;
    if (b > 0) look(kb, n);
    for (int k0 = kb; k0 < b; k0 += 2 * KS * 16) {
        C a[2][4], x[2][4];
        int nn[2][4];
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int k = k0 + KS * 16 * g + 4 * kg + q;
                a[g][q] = gload(Q + min(k, b - 1));
                x[g][q] = gload(xp + (long)max(n[g][q], 0) * 16 + l16);
            }
        look(k0 + 2 * KS * 16, nn);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            if (g == 1 && k0 + KS * 16 >= b) break;  // uniform
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const bool ok = n[g][q] >= 0 && k0 + KS * 16 * g + 4 * kg + q < b;
                B.step(csel(ok, a[g][q], mk<C>(0, 0)), csel(ok, x[g][q], mk<C>(0, 0)));
            }
        }
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int q = 0; q < 4; ++q) n[g][q] = nn[g][q];
    }
    C z[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        z[r] = mk<C>((A.rr[r] - A.ii[r]) - (B.rr[r] - B.ii[r]), A.ri[r] - B.ri[r]);
    ndm_finish<KS>(z, red, wv, lane, [&](int r, C s) {
        if (cell[r] >= 0) gstore(xp + (long)cell[r] * 16 + l16, s);
    });
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
