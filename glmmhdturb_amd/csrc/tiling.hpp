// tiling.hpp -- z-chunk lengths of the march kernels (host).
//
// A march workgroup owns a column tile and `chunk` z planes; besides them it spends about `lead` planes
// on loading its window and on the faces it shares with its neighbours.  Short chunks give every CU
// work on small grids, long ones spend less on lead-in.  Every chunk length gives the same bits.
#pragma once
#include <cstddef>

namespace glm {

// Concurrent workgroups of a kernel: CUs and resident workgroups per CU (the occupancy API).
struct Resident {
    int cus = 256, occ = 1;
};

// Modelled time, in planes of a workgroup that has its CU for itself, of W workgroups of `len` planes:
// the CU with the most workgroups takes n = ceil(W / cus) of them, occ at a time, and m resident
// workgroups slow each other down by 1 + share (m - 1).  share 0 would be perfect overlap, 1 none; the
// measured GLM and CT marches lie at 0.5-0.7 in FP64 (two resident: 7.7 us a plane alone, 11.8 together)
// and 0.29-0.38 in FP32 (three or four resident), the hydro march, which keeps the VALU busier alone, at
// 0.9 and 0.6.  Against the sweep of all chunk lengths on grids from
// 32^3 to 256^3 the choice is within 5% of the best.  (Counting whole rounds over all slots as if
// resident workgroups did not slow each other, with chunks of at least 8 planes, took 72 us instead
// of 25 for 32^3 FP64 and 60 instead of 40 for 64^3 FP32.)
inline double chunk_cost(long W, double len, const Resident& r, double share)
{
    const long n = (W + r.cus - 1) / r.cus, full = n / r.occ, rest = n % r.occ;
    return len * ((double)full * (1.0 + share * (r.occ - 1)) + (rest ? 1.0 + share * (double)(rest - 1) : 0.0));
}

// Planes per chunk of one grid with `cols` column tiles.
inline int chunk_planes(long cols, int nz, const Resident& r, double lead, double share)
{
    int best = nz;
    double least = -1.0;
    for (int c = 1; c <= nz; ++c) {
        const int zc = (nz + c - 1) / c, n = (nz + zc - 1) / zc;   // chunks actually formed
        if (n != c) continue;
        const double t = chunk_cost(cols * n, zc + lead, r, share);
        if (least < 0.0 || t < least) { least = t; best = zc; }
    }
    return best;
}

// Tiles and z-chunks of an (nx, ny, nz) grid in ox x oy column tiles, with the requested chunk length
// or, for zreq <= 0, the modelled one.
inline void march_tiles(int nx, int ny, int nz, int ox, int oy, int zreq, const Resident& r, double lead, double share,
                        int& tiles_x, int& tiles_y, int& nzc, int& zchunk)
{
    tiles_x = (nx + ox - 1) / ox;
    tiles_y = (ny + oy - 1) / oy;
    zchunk = zreq > 0 ? (zreq < nz ? zreq : nz) : chunk_planes((long)tiles_x * tiles_y, nz, r, lead, share);
    nzc = (nz + zchunk - 1) / zchunk;
}

}  // namespace glm
