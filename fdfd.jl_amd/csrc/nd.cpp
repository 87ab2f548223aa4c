// Nested-dissection factorization and reduced solve (host side).
//
// The torus of cells is dissected by nd_plan.h; every tree level is one batch
// of equal-sized fronts (k_nd.hip).  Leaves are eliminated in registers; a
// level above assembles [F11 | F12] from the operator and its children's
// Schur complements, inverts F11 by symmetric block sweeps, and forms
// Q = X F12 and the Schur complement F22 - F12^T Q on MFMA.
//
// Against the block cyclic reduction of the lines (bcr.cpp) this takes of
// the order of N^1.5 operations and N log N storage instead of n^3 m and
// n^2 m, at the price of a fixed pivot order (4 x 4 blocks).  A factor with a
// pivot block that cannot be inverted is rebuilt by the line reduction, and so is
// one on which the refinement stalls above what rounding allows.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <memory>
#include <vector>

#include "../../include/fdfd.h"
#include "nd_dev.h"
#include "runtime.h"

namespace fdfd {

int rt_assemble(Handle* h, Factor* F);

// Tree and index maps of one grid shape on the device, shared by the factors
// built with it; lev[0] is the root.
struct NdPlan {
    int Nx = 0, Ny = 0, fronts = 0;
    std::vector<NdLev> lev;
    long arena = 0;            // complex entries of a factor
    long vlen = 0, ulen = 0;   // solve work: separator values, boundary updates
    long maxY = 0, maxF12 = 0, maxS[2] = {0, 0}, maxp = 0, maxcnt = 0;  // scratch, per factor
    void* base = nullptr;
    ~NdPlan() {
        if (base) (void)hipFree(base);
    }
};

namespace {

constexpr size_t ELEM = sizeof(double2);  // factor entries are complex128 (k_nd.hip)
constexpr int PLAN_CACHE = 4;  // grid shapes whose plans a handle keeps

void size_plan(NdPlan& P, const std::vector<nd::Level>& L) {
    long off = 0;
    P.fronts = 0;
    P.vlen = P.ulen = 0;
    for (size_t i = 0; i < L.size(); ++i) {
        const long cnt = (long)L[i].box.size(), p = L[i].p, b = L[i].b;
        NdLev v{};
        v.kind = L[i].kind;
        v.nch = L[i].nch;
        v.cnt = (int)cnt;
        v.p = (int)p;
        v.b = (int)b;
        v.stat = P.fronts;
        v.offX = off;
        off += cnt * p * p;
        v.offQ = off;
        off += cnt * p * b;
        v.offV = P.vlen;
        v.offU = P.ulen;
        P.vlen += cnt * p;
        P.ulen += cnt * b;
        P.fronts += (int)cnt;
        P.maxS[i & 1] = std::max(P.maxS[i & 1], cnt * b * b);
        if (L[i].nch > 0) P.maxF12 = std::max(P.maxF12, cnt * p * b);
        if (L[i].nch > 0 && p > 64) {  // separators inverted in blocks
            P.maxY = std::max(P.maxY, cnt * p * p);
            P.maxp = std::max(P.maxp, cnt * p);
            P.maxcnt = std::max(P.maxcnt, cnt);
        }
        P.lev.push_back(v);
    }
    for (size_t i = 0; i + 1 < P.lev.size(); ++i) {
        P.lev[i].cb = P.lev[i + 1].b;
        P.lev[i].offUc = P.lev[i + 1].offU;
    }
    P.arena = off;
}

// scratch of B factors built together: separators, F12, block rows and inverses
// (NdInv) of the largest level, and the Schur complements of two neighbouring
// levels
struct Scratch {
    size_t bytes = 0;
    size_t oY, oF12, oR, oR1, oD, oS[2], ofac, ostat;
    Scratch(const NdPlan& P, int B) {
        auto take = [&](size_t n) {
            const size_t o = bytes;
            bytes += (n + 255) & ~(size_t)255;
            return o;
        };
        oY = take(ELEM * P.maxY * B);
        oF12 = take(ELEM * P.maxF12 * B);
        oR = take(ELEM * P.maxp * 64 * B);
        oR1 = take(ELEM * P.maxp * 64 * B);
        oD = take(ELEM * P.maxcnt * 2 * 64 * 64 * B);
        for (int k = 0; k < 2; ++k) oS[k] = take(ELEM * P.maxS[k] * B);
        ofac = take(sizeof(NdFac) * B);
        ostat = take(sizeof(double) * 3 * B);
    }
};

}  // namespace

// the plan of the handle's grid, from the handle's cache or built
static int nd_plan(Handle* h, int Nx, int Ny, std::shared_ptr<NdPlan>& out) {
    for (size_t i = 0; i < h->nd_plans.size(); ++i)
        if (h->nd_plans[i]->Nx == Nx && h->nd_plans[i]->Ny == Ny) {
            out = h->nd_plans[i];
            h->nd_plans.erase(h->nd_plans.begin() + i);
            h->nd_plans.insert(h->nd_plans.begin(), out);
            return FDFD_OK;
        }
    const std::vector<nd::Level> L = nd::make_plan(Nx, Ny);
    auto P = std::make_shared<NdPlan>();
    P->Nx = Nx;
    P->Ny = Ny;
    size_plan(*P, L);
    // one buffer: node and child maps of every level, then the boxes
    size_t bytes = 0;
    auto take = [&](size_t n) {
        const size_t o = bytes;
        bytes += (n + 255) & ~(size_t)255;
        return o;
    };
    std::vector<size_t> on(L.size()), oc(L.size()), ob(L.size());
    for (size_t i = 0; i < L.size(); ++i) {
        const size_t f = (size_t)L[i].box.size() * (L[i].p + L[i].b);
        on[i] = take(sizeof(int) * f);
        oc[i] = take(sizeof(short) * 2 * f);
    }
    const size_t boxes0 = bytes;
    std::vector<nd::Box> all;
    for (size_t i = 0; i < L.size(); ++i) {
        ob[i] = boxes0 + sizeof(nd::Box) * all.size();
        all.insert(all.end(), L[i].box.begin(), L[i].box.end());
    }
    bytes += sizeof(nd::Box) * all.size();
    if (hipMalloc(&P->base, bytes) != hipSuccess) {
        (void)hipGetLastError();
        P->base = nullptr;
        return fail(h, FDFD_ERR_OOM, "dissection maps do not fit in device memory");
    }
    char* base = (char*)P->base;
    COPY(h, base + boxes0, all.data(), sizeof(nd::Box) * all.size(), hipMemcpyHostToDevice);
    for (size_t i = 0; i < L.size(); ++i) {
        NdLev& v = P->lev[i];
        v.node = (const int*)(base + on[i]);
        v.cm = (const short*)(base + oc[i]);
        NdMapArgs a{};
        a.kind = v.kind;
        a.nch = v.nch;
        a.cnt = v.cnt;
        a.p = v.p;
        a.b = v.b;
        a.wrapx = L[i].wrapx;
        a.wrapy = L[i].wrapy;
        a.Nx = Nx;
        a.Ny = Ny;
        a.box = (const nd::Box*)(base + ob[i]);
        if (i + 1 < L.size()) {
            a.cwrapx = L[i + 1].wrapx;
            a.cwrapy = L[i + 1].wrapy;
            a.cbox = (const nd::Box*)(base + ob[i + 1]);
        }
        launch_nd_maps(h->stream, a, (int*)v.node, (short*)v.cm);
    }
    HIPCHK(h, hipGetLastError());
    // a factor on another stream may use the plan next
    HIPCHK(h, hipStreamSynchronize(h->stream));
    h->nd_plans.insert(h->nd_plans.begin(), P);
    if (h->nd_plans.size() > PLAN_CACHE) h->nd_plans.pop_back();
    out = P;
    return FDFD_OK;
}

// Whether factors of this grid are built by nested dissection: not when a
// variant, panel width or full pivot search of the line reduction was asked
// for, and not on grids of few lines
bool rt_nd_applies(const Handle* h, int Nx, int Ny) {
    return !h->nd_off && !h->env_knobs && !h->full_pivot_search && h->panel_width == 0 &&
           std::min(Nx, Ny) >= ND_MIN_LINE;
}

// bytes of a factor (arena) and of the scratch one more factor adds to a build
// (a tree is built for them where the handle has none of this shape: about 1 ms at
// 1024 x 1024)
void rt_nd_bytes(const Handle* h, int Nx, int Ny, size_t* arena, size_t* scratch) {
    auto bytes = [&](const NdPlan& P) {
        *arena = (size_t)P.arena * ELEM;
        *scratch = Scratch(P, 1).bytes;
    };
    for (const auto& P : h->nd_plans)
        if (P->Nx == Nx && P->Ny == Ny) return bytes(*P);
    NdPlan P;
    size_plan(P, nd::make_plan(Nx, Ny));
    bytes(P);
}

int rt_nd_prepare(Handle* h, int Nx, int Ny) {
    std::shared_ptr<NdPlan> P;
    return nd_plan(h, Nx, Ny, P);
}

// Builds Fs by nested dissection; `bad` receives the factors whose pivots
// failed their check (their storage is kept, their result is not usable).
int rt_build_nd(Handle* h, const std::vector<Factor*>& Fs, std::vector<int>& bad, int poor) {
    const GridDesc& g = h->g;
    const int B = (int)Fs.size();
    const bool prof = h->prof.enabled;
    int rc;
    std::shared_ptr<NdPlan> P;
    if ((rc = nd_plan(h, g.Nx, g.Ny, P))) return rc;
    if ((rc = ensure_solve_work(h, (long)g.Nx * g.Ny))) return rc;
    const Scratch sc(*P, B);
    if (h->nd_scratch_bytes < sc.bytes) {
        if (h->nd_scratch) (void)hipFree(h->nd_scratch);
        h->nd_scratch = nullptr;
        h->nd_scratch_bytes = 0;
        HIPCHK(h, hipMalloc(&h->nd_scratch, sc.bytes));
        h->nd_scratch_bytes = sc.bytes;
    }
    char* w = (char*)h->nd_scratch;
    hipStream_t st = h->stream;
    std::vector<NdFac> fac(B);
    for (int f = 0; f < B; ++f) {
        Factor* F = Fs[f];
        if ((rc = rt_assemble(h, F))) return rc;
        F->blocks_bytes = (size_t)P->arena * ELEM;
        F->blocks = arena_take(h, F->blocks_bytes);
        F->ndu = (double2*)buf_alloc(h, sizeof(double2) * 2 * (g.Nx + g.Ny));
        F->pivstat = (double*)buf_alloc(h, sizeof(double) * 3 * P->fronts);
        if (!F->blocks || !F->ndu || !F->pivstat)
            return fail(h, FDFD_ERR_OOM, "factor storage (" + std::to_string(F->blocks_bytes >> 20) +
                                             " MiB) does not fit in device memory");
        F->nd = P;
        launch_nd_symmetrise(st, F->coef, F->ndu, F->form == 1 ? F->sxb : F->sxf,
                             F->form == 1 ? F->syb : F->syf, g.Nx, g.Ny);
        fac[f] = NdFac{F->coef, F->blocks, F->pivstat};
    }
    NdFac* dfac = (NdFac*)(w + sc.ofac);
    COPY(h, dfac, fac.data(), sizeof(NdFac) * B, hipMemcpyHostToDevice);
    const NdInv iw{w + sc.oY, w + sc.oF12, w + sc.oR, w + sc.oR1, w + sc.oD};
    hipEvent_t e0, e1;
    HIPCHK(h, hipEventCreate(&e0));
    HIPCHK(h, hipEventCreate(&e1));
    HIPCHK(h, hipEventRecord(e0, st));
    auto scope = [&](int id, double fl, double by) { return prof ? new ProfScope(h, id, fl, by, st) : nullptr; };
    for (int li = (int)P->lev.size() - 1; li >= 0; --li) {
        const NdLev& v = P->lev[li];
        const double p = v.p, b = v.b, nj = (double)v.cnt * B;
        void* S = w + sc.oS[li & 1];
        const void* Sc = w + sc.oS[(li + 1) & 1];
        ProfScope* ps = scope(P_SCHUR, 0, (p + b) * (p + b) * nj * ELEM);
        if (v.nch == 0) {
            launch_nd_leaf(st, v, dfac, B, g.Nx, g.Ny, S);
            delete ps;
            continue;
        }
        if (launch_nd_small(st, v, dfac, B, g.Nx, g.Ny, Sc, S)) {
            delete ps;
            continue;
        }
        launch_nd_front(st, v, dfac, B, g.Nx, g.Ny, Sc, iw);
        delete ps;
        ps = scope(P_PANEL, 4 * p * p * p * nj, 0);
        launch_nd_invert(st, v, dfac, B, iw);
        delete ps;
        if (v.b == 0) continue;
        ps = scope(P_GEMM, 8 * p * p * b * nj, 0);
        launch_nd_gemm(st, v, dfac, B, iw.F12, nullptr, nullptr, false);
        delete ps;
        ps = scope(P_GEMM, 4 * p * b * b * nj, 0);
        launch_nd_gemm(st, v, dfac, B, iw.F12, Sc, S, true);
        delete ps;
    }
    if (poor != 0 && std::abs(poor) <= B) {  // injected: the inverse of the last separator
        double2* X = (double2*)Fs[std::abs(poor) - 1]->blocks + P->lev[0].offX;
        const double a = poor > 0 ? 0.0 : std::numeric_limits<double>::quiet_NaN();
        launch_scale_copy(st, X, X, make_double2(a, 0), (long)P->lev[0].p * P->lev[0].p);
    }
    double* dstat = (double*)(w + sc.ostat);
    launch_nd_stat(st, dfac, B, P->fronts, dstat);
    hipError_t le = hipGetLastError();
    (void)hipEventRecord(e1, st);
    std::vector<double> stat(3 * (size_t)B);
    rc = le == hipSuccess ? FDFD_OK : fail(h, FDFD_ERR_HIP, std::string("dissection kernels: ") + hipGetErrorString(le));
    if (!rc) rc = stream_copy(h, stat.data(), dstat, sizeof(double) * stat.size(), hipMemcpyDeviceToHost);
    float ms = 0;
    if (!rc) (void)hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    for (int f = 0; f < B; ++f) {
        Factor* F = Fs[f];
        buf_free(h, F->coef);  // the solves apply the operator matrix-free
        F->coef = nullptr;
        const double mn = stat[3 * f], mx = stat[3 * f + 1];
        F->t_factor_ms = ms;
        F->singular_line = -1;
        F->pivot_fallback = 0;
        // (the statistics are of 2 x 2 determinants)
        F->pivot_growth = mn > 0 ? std::sqrt(mx / mn) : std::numeric_limits<double>::infinity();
        if (stat[3 * f + 2] != 0 || !(mn > 0) || !std::isfinite(mx)) bad.push_back(f);
    }
    return FDFD_OK;
}

// work vectors of `count` solves, in the handle's buffer
static int nd_vectors(Handle* h, long per, int count, double2** v) {
    const size_t need = sizeof(double2) * (size_t)per * count;
    if (h->nd_vec_bytes < need) {
        if (h->nd_vec) {
            HIPCHK(h, hipStreamSynchronize(h->stream));
            (void)hipFree(h->nd_vec);
        }
        h->nd_vec = nullptr;
        h->nd_vec_bytes = 0;
        HIPCHK(h, hipMalloc(&h->nd_vec, need));
        h->nd_vec_bytes = need;
    }
    *v = (double2*)h->nd_vec;
    return FDFD_OK;
}

// in -> out with the factor's scalings; v: its work vectors
static NdVec nd_vec(const Factor* F, int trans, const double2* in, double2* out, long rs, const int* ridx, double2* v) {
    const NdPlan& P = *F->nd;
    const double2 *ux = F->ndu, *uxi = ux + P.Nx, *uy = ux + 2 * P.Nx, *uyi = uy + P.Ny;
    return NdVec{in, out, rs, ridx, v, v + P.vlen, v + P.vlen + P.ulen,
                 trans ? ux : uxi, trans ? uy : uyi, trans ? uxi : ux, trans ? uyi : uy};
}

// out = A'^-1 in or A'^-T in for na sources (source ridx[i] at ridx[i] * rs;
// ridx null: one source).  S = U^-1 A' U gives A'^-1 = U S^-1 U^-1 and
// A'^-T = U^-1 S^-1 U.
int rt_nd_solve(Handle* h, Factor* F, int trans, const double2* in, double2* out, long rs,
                const int* ridx, int na, bool prof) {
    const NdPlan& P = *F->nd;
    const long N = (long)P.Nx * P.Ny, per = P.vlen + P.ulen + N;
    double2* v;
    int rc = nd_vectors(h, per, na == 1 ? 1 : KMULTI, &v);
    if (rc) return rc;
    static_assert(KMULTI == 16, "the multi-source kernels hold 16 sources");
    const NdVec z = nd_vec(F, trans, in, out, rs, ridx, v);
    const int nl = (int)P.lev.size();
    ProfScope* ps = prof ? new ProfScope(h, P_SWEEP, 0, 0) : nullptr;
    if (na > 1) {
        double2 *vp = v, *up = vp + P.vlen * KMULTI, *xp = up + P.ulen * KMULTI;
        launch_ndm_io(h->stream, z, xp, N, P.Nx, na, true);
        for (int li = nl - 1; li >= 0; --li) launch_ndm_up(h->stream, P.lev[li], F->blocks, vp, up, xp);
        for (int li = 0; li < nl; ++li) launch_ndm_down(h->stream, P.lev[li], F->blocks, vp, xp);
        launch_ndm_io(h->stream, z, xp, N, P.Nx, na, false);
    } else {
        NdBatch<1> bt{};
        bt.s[0].z = z;
        bt.s[0].arena = F->blocks;
        for (int li = nl - 1; li >= 0; --li) launch_nd_up(h->stream, P.lev[li], bt, 1, P.Nx);
        for (int li = 0; li < nl; ++li) launch_nd_down(h->stream, P.lev[li], bt, 1, P.Nx);
    }
    delete ps;
    return FDFD_OK;
}

// out_j = M_j^-1 in_j for the factors of one grid, N values apart
int rt_nd_solve_each(Handle* h, const std::vector<Factor*>& Fs, const double2* in, double2* out, bool prof) {
    const NdPlan& P = *Fs[0]->nd;
    const long N = (long)P.Nx * P.Ny, per = P.vlen + P.ulen + N;
    const int nf = (int)Fs.size(), nl = (int)P.lev.size();
    double2* v;
    int rc = nd_vectors(h, per, std::min(nf, ND_SOLVES), &v);
    if (rc) return rc;
    ProfScope* ps = prof ? new ProfScope(h, P_SWEEP, 0, 0) : nullptr;
    for (int f0 = 0; f0 < nf; f0 += ND_SOLVES) {
        const int nb = std::min(ND_SOLVES, nf - f0);
        NdBatch<ND_SOLVES> bt{};
        for (int q = 0; q < nb; ++q) {
            const long o = (long)(f0 + q) * N;
            bt.s[q].z = nd_vec(Fs[f0 + q], 0, in + o, out + o, 0, nullptr, v + q * per);
            bt.s[q].arena = Fs[f0 + q]->blocks;
        }
        for (int li = nl - 1; li >= 0; --li) launch_nd_up(h->stream, P.lev[li], bt, nb, P.Nx);
        for (int li = 0; li < nl; ++li) launch_nd_down(h->stream, P.lev[li], bt, nb, P.Nx);
    }
    delete ps;
    return FDFD_OK;
}

}  // namespace fdfd
