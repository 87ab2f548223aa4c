// Arguments of the nested-dissection kernels (k_nd.hip), filled by nd.cpp.
#pragma once

#include "fdfd_common.h"
#include "nd_plan.h"

namespace fdfd {

// one level of the tree on the device; offsets are in complex entries
struct NdLev {
    int kind, nch, cnt, p, b;
    int cb;           // boundary size of the child level
    int stat;         // first pivot-statistics slot of the level
    const int* node;  // cnt x (p + b) cells, -1 padding
    const short* cm;  // cnt x 2 x (p + b) positions in the children's boundaries
    long offX, offQ;        // X (cnt x p x p) and Q (cnt x p x b) in the arena
    long offV, offU, offUc; // solve vectors: separator values, boundary updates, children's updates
};

struct NdMapArgs {
    int kind, nch, cnt, p, b, wrapx, wrapy, cwrapx, cwrapy, Nx, Ny;
    const nd::Box *box, *cbox;
};

// per factor
struct NdFac {
    const double2* coef;  // symmetrised operator planes (CC, CE, CN)
    void* arena;
    double* pivstat;      // 3 per front
};

// inversion scratch of a level, one slot per (factor, front): the separator
// block, F12, the block row and its product of a block sweep (64 x p each) and
// two 64 x 64 block inverses
struct NdInv {
    void *Y, *F12, *R, *R1, *D;
};

// vectors of a reduced solve: source ridx[s] (0 without a list) at in / out
// + ridx * rs, one source's work vectors, and the scaling of the input
// (six (x) siy) and output (sox (x) soy)
struct NdVec {
    const double2* in;
    double2* out;
    long rs;
    const int* ridx;
    double2 *v, *u, *x;
    const double2 *six, *siy, *sox, *soy;
};

void launch_nd_maps(hipStream_t s, const NdMapArgs& a, int* node, short* cm);
void launch_nd_symmetrise(hipStream_t s, double2* coef, double2* us, const double2* wx,
                          const double2* wy, int Nx, int Ny);
void launch_nd_leaf(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, int Nx, int Ny, void* S);
// a level of small fronts in one launch; false if they are not
bool launch_nd_small(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, int Nx, int Ny, const void* Sc,
                     void* S);
void launch_nd_front(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, int Nx, int Ny, const void* Sc,
                     const NdInv& w);
void launch_nd_invert(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, const NdInv& w);
void launch_nd_gemm(hipStream_t s, const NdLev& lv, const NdFac* fac, int B, const void* F12,
                    const void* Sc, void* S, bool schur);
void launch_nd_stat(hipStream_t s, const NdFac* fac, int B, int nfronts, double* out);
// independent solves with factors of one tree, side by side
constexpr int ND_SOLVES = 8;
template <int N> struct NdBatch {
    struct {
        NdVec z;
        const void* arena;
    } s[N];
};
template <int N> void launch_nd_up(hipStream_t s, const NdLev& lv, const NdBatch<N>& bt, int nb, int Nx);
template <int N> void launch_nd_down(hipStream_t s, const NdLev& lv, const NdBatch<N>& bt, int nb, int Nx);
// several sources (at most 16): pack / unpack, one level up, one level down
void launch_ndm_io(hipStream_t s, const NdVec& z, void* x, long N, int Nx, int na, bool pack);
void launch_ndm_up(hipStream_t s, const NdLev& lv, const void* arena, void* vp, void* up, const void* x);
void launch_ndm_down(hipStream_t s, const NdLev& lv, const void* arena, const void* vp, void* x);

}  // namespace fdfd
