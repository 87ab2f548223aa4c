// Host arrays into the solver's layout (x fastest, one source after another).
//
// A row-major Nx x Ny array, or sources in the last axis of an Nx x Ny x n
// array, is a transposition.  An element at a time it touches a new cache line
// for each value: 3.1 ms for one of 16 sources of 256 x 256 (1 MB), 53 ms for
// all of them, twice the time of the batched solve behind it.  Here tiles are read
// along the source's runs into a buffer of 17 kB and written from it along x (rows
// a multiple of 4 kB apart share their cache sets: tiles without the buffer took
// 2.7 ms for 1024 x 768 values), by a few threads where the array is large.
#include <algorithm>
#include <cstdlib>
#include <thread>
#include <vector>

#include "../../include/fdfd.h"

namespace {

struct PackJob {
    const fdfd_complex* src;
    long long sx, sy, sr;
    int Nx, Ny, nr;
    fdfd_complex* dst;
};

// rows [y0, y1) of every source
void pack_rows(const PackJob& j, int y0, int y1) {
    const int T = j.nr > 1 ? 8 : 32, RB = 16;
    fdfd_complex buf[16 * 8 * 9];  // [r][y][x] of 16 x 8 x 8 or 1 x 32 x 32, x rows padded by one
    const int P = T + 1;
    for (int r0 = 0; r0 < j.nr; r0 += RB)
        for (int yt = y0; yt < y1; yt += T)
            for (int xt = 0; xt < j.Nx; xt += T) {
                const int nr = std::min(RB, j.nr - r0), ny = std::min(T, y1 - yt), nx = std::min(T, j.Nx - xt);
                const fdfd_complex* s = j.src + xt * j.sx + yt * j.sy + r0 * j.sr;
                if (std::llabs(j.sr) < std::llabs(j.sy)) {
                    for (int x = 0; x < nx; ++x)
                        for (int y = 0; y < ny; ++y)
                            for (int r = 0; r < nr; ++r)
                                buf[(r * T + y) * P + x] = s[x * j.sx + y * j.sy + r * j.sr];
                } else {
                    for (int r = 0; r < nr; ++r)
                        for (int x = 0; x < nx; ++x)
                            for (int y = 0; y < ny; ++y)
                                buf[(r * T + y) * P + x] = s[x * j.sx + y * j.sy + r * j.sr];
                }
                for (int r = 0; r < nr; ++r)
                    for (int y = 0; y < ny; ++y)
                        std::copy_n(buf + (r * T + y) * P, nx,
                                    j.dst + ((long long)(r0 + r) * j.Ny + yt + y) * j.Nx + xt);
            }
}

}  // namespace

extern "C" int fdfd_pack(const fdfd_complex* src, long long sx, long long sy, long long sr, int Nx, int Ny, int nr,
                         fdfd_complex* dst) {
    if (!src || !dst || Nx < 1 || Ny < 1 || nr < 1) return FDFD_ERR_INVALID;
    const PackJob job{src, sx, sy, sr, Nx, Ny, nr, dst};
    // a thread costs some 50 us, which it takes to move half a megabyte
    const double mb = 16e-6 * Nx * (double)Ny * nr;
    const int hw = (int)std::thread::hardware_concurrency();
    const int nt = std::max(1, std::min({8, hw, Ny, (int)std::min(mb, 64.0)}));
    std::vector<std::thread> th;
    int y0 = 0;
    try {
        th.reserve(nt);
        for (int t = 1; t < nt; ++t) {
            const int y1 = (int)((long long)Ny * t / nt);
            th.emplace_back(pack_rows, std::cref(job), y0, y1);
            y0 = y1;
        }
    } catch (...) {  // no thread to be had: the rest is done here
    }
    pack_rows(job, y0, Ny);
    for (auto& t : th) t.join();
    return FDFD_OK;
}
