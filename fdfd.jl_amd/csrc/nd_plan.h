// Nested dissection of the periodic grid (host/device, integers only).
//
// The cells of an Nx x Ny torus are split level by level into a binary tree
// of boxes.  A box has one separator, the cells eliminated at its node of the
// tree, and a boundary, the cells adjacent to it outside (its up to four
// sides; the 5-point stencil couples no corners).  Every box of a level has
// the same kind of separator, so the fronts of a level (separator plus
// boundary) form one batch of equal padded sizes:
//   ND_CUTX    the box wraps around in x: its last column is eliminated and
//              one child remains that no longer wraps (ND_CUTY: last row);
//   ND_SPLITX  the middle column is eliminated, the two sides are the
//              children (ND_SPLITY: middle row);
//   ND_LEAF    all cells of the box.
// A wrapped dimension counts half its length when the longer side is chosen,
// since separating it takes two lines: a square torus is cut in x, split in
// x, then cut in y, which keeps every separator at most min(Nx, Ny) cells
// long (+- the first cut), also on elongated grids.
//
// Front indices: [0, p) separator cells, [p, p + b) boundary cells; a box's
// own counts are at most the level's padded p and b.  nd_node gives the cell
// of a front index (-1: padding) and nd_bpos the boundary position of a cell.
#pragma once

#include <vector>

#ifdef __HIPCC__
#define ND_HD __host__ __device__
#else
#define ND_HD
#endif

namespace fdfd {
namespace nd {

enum { ND_LEAF = 0, ND_CUTX = 1, ND_CUTY = 2, ND_SPLITX = 3, ND_SPLITY = 4 };

struct Box {
    int x0, w, y0, h;
};

// largest leaf: cells, and rows of the leaf kernel's front (cells and boundary,
// each padded to a multiple of 4)
constexpr int LEAF_CELLS = 49;
constexpr int LEAF_FRONT = 80;

// sides of a box: the columns left and right of it (nx of them: none when it
// wraps in x, one when both are the same column) and the rows below and above
struct Sides {
    int nx, xl, xr, ny, yl, yr;
};
ND_HD inline Sides sides(const Box& b, int wrapx, int wrapy, int Nx, int Ny) {
    Sides s;
    s.xl = b.x0 == 0 ? Nx - 1 : b.x0 - 1;
    s.xr = b.x0 + b.w >= Nx ? b.x0 + b.w - Nx : b.x0 + b.w;
    s.nx = wrapx ? 0 : (s.xl == s.xr ? 1 : 2);
    s.yl = b.y0 == 0 ? Ny - 1 : b.y0 - 1;
    s.yr = b.y0 + b.h >= Ny ? b.y0 + b.h - Ny : b.y0 + b.h;
    s.ny = wrapy ? 0 : (s.yl == s.yr ? 1 : 2);
    return s;
}

ND_HD inline int sep_count(int kind, const Box& b) {
    if (kind == ND_LEAF) return b.w * b.h;
    return (kind == ND_CUTX || kind == ND_SPLITX) ? b.h : b.w;
}
ND_HD inline int bnd_count(const Box& b, int wrapx, int wrapy, int Nx, int Ny) {
    const Sides s = sides(b, wrapx, wrapy, Nx, Ny);
    return s.nx * b.h + s.ny * b.w;
}

// cell (linear, x fastest) of separator index i, -1 past the separator
ND_HD inline int sep_node(int kind, const Box& b, int i, int Nx) {
    if (i >= sep_count(kind, b)) return -1;
    int x, y;
    switch (kind) {
        case ND_LEAF: x = b.x0 + i % b.w; y = b.y0 + i / b.w; break;
        case ND_CUTX: x = b.x0 + b.w - 1; y = b.y0 + i; break;
        case ND_CUTY: x = b.x0 + i; y = b.y0 + b.h - 1; break;
        case ND_SPLITX: x = b.x0 + (b.w - 1) / 2; y = b.y0 + i; break;
        default: x = b.x0 + i; y = b.y0 + (b.h - 1) / 2; break;
    }
    return x + Nx * y;
}
// cell of boundary index j (order: left, right, bottom, top), -1 past it
ND_HD inline int bnd_node(const Box& b, int wrapx, int wrapy, int j, int Nx, int Ny) {
    const Sides s = sides(b, wrapx, wrapy, Nx, Ny);
    if (j < s.nx * b.h) {
        const int x = j < b.h ? s.xl : s.xr;
        return x + Nx * (b.y0 + (j < b.h ? j : j - b.h));
    }
    j -= s.nx * b.h;
    if (j < s.ny * b.w) {
        const int y = j < b.w ? s.yl : s.yr;
        return b.x0 + (j < b.w ? j : j - b.w) + Nx * y;
    }
    return -1;
}
// boundary position of a cell, -1 if it is not on the boundary
ND_HD inline int bnd_pos(const Box& b, int wrapx, int wrapy, int node, int Nx, int Ny) {
    if (node < 0) return -1;
    const int x = node % Nx, y = node / Nx;
    const Sides s = sides(b, wrapx, wrapy, Nx, Ny);
    const bool iny = y >= b.y0 && y < b.y0 + b.h, inx = x >= b.x0 && x < b.x0 + b.w;
    if (s.nx > 0 && iny) {
        if (x == s.xl) return y - b.y0;
        if (s.nx > 1 && x == s.xr) return b.h + y - b.y0;
    }
    if (s.ny > 0 && inx) {
        if (y == s.yl) return s.nx * b.h + x - b.x0;
        if (s.ny > 1 && y == s.yr) return s.nx * b.h + b.w + x - b.x0;
    }
    return -1;
}

// child c of a box of a split or cut level
ND_HD inline Box child(int kind, const Box& b, int c) {
    Box r = b;
    switch (kind) {
        case ND_CUTX: r.w = b.w - 1; break;
        case ND_CUTY: r.h = b.h - 1; break;
        case ND_SPLITX: {
            const int m = (b.w - 1) / 2;
            if (c == 0) r.w = m;
            else { r.x0 = b.x0 + m + 1; r.w = b.w - 1 - m; }
            break;
        }
        default: {
            const int m = (b.h - 1) / 2;
            if (c == 0) r.h = m;
            else { r.y0 = b.y0 + m + 1; r.h = b.h - 1 - m; }
        }
    }
    return r;
}

struct Level {
    int kind = ND_LEAF, wrapx = 0, wrapy = 0;
    int nch = 0;        // children per box (0: leaf, 1: cut, 2: split)
    int p = 0, b = 0;   // padded separator and boundary sizes (multiples of 4)
    std::vector<Box> box;
};

// level 0 is the root (one box, the torus); child c of box i of level l is
// box nch * i + c of level l + 1; the last level holds the leaves
inline std::vector<Level> make_plan(int Nx, int Ny) {
    auto up4 = [](int v) { return (v + 3) & ~3; };
    std::vector<Level> L;
    Level cur;
    cur.wrapx = cur.wrapy = 1;
    cur.box.push_back(Box{0, Nx, 0, Ny});
    for (;;) {
        int W = 0, H = 0, wmin = Nx, hmin = Ny;
        for (const Box& b : cur.box) {
            W = b.w > W ? b.w : W;
            H = b.h > H ? b.h : H;
            wmin = b.w < wmin ? b.w : wmin;
            hmin = b.h < hmin ? b.h : hmin;
        }
        const bool open = !cur.wrapx && !cur.wrapy;
        const bool canx = cur.wrapx ? wmin >= 2 : wmin >= 3, cany = cur.wrapy ? hmin >= 2 : hmin >= 3;
        if ((open && W * H <= LEAF_CELLS && ((W * H + 3) & ~3) + ((2 * (W + H) + 3) & ~3) <= LEAF_FRONT) || (!canx && !cany)) {
            cur.kind = ND_LEAF;
        } else {
            const double ex = cur.wrapx ? 0.5 * W : W, ey = cur.wrapy ? 0.5 * H : H;
            // the longer side; a wrapped one first when they are equal
            bool dox = ex > ey || (ex == ey && (cur.wrapx || !cur.wrapy));
            if (dox && !canx) dox = false;
            else if (!dox && !cany) dox = true;
            cur.kind = dox ? (cur.wrapx ? ND_CUTX : ND_SPLITX) : (cur.wrapy ? ND_CUTY : ND_SPLITY);
        }
        cur.nch = cur.kind == ND_LEAF ? 0 : (cur.kind == ND_CUTX || cur.kind == ND_CUTY) ? 1 : 2;
        int p = 0, bb = 0;
        for (const Box& b : cur.box) {
            const int q = sep_count(cur.kind, b), r = bnd_count(b, cur.wrapx, cur.wrapy, Nx, Ny);
            p = q > p ? q : p;
            bb = r > bb ? r : bb;
        }
        cur.p = up4(p);
        cur.b = up4(bb);
        L.push_back(cur);
        if (cur.kind == ND_LEAF) break;
        Level nx;
        nx.wrapx = cur.kind == ND_CUTX ? 0 : cur.wrapx;
        nx.wrapy = cur.kind == ND_CUTY ? 0 : cur.wrapy;
        for (const Box& b : cur.box)
            for (int c = 0; c < cur.nch; ++c) nx.box.push_back(child(cur.kind, b, c));
        cur = nx;
    }
    return L;
}

}  // namespace nd
}  // namespace fdfd
