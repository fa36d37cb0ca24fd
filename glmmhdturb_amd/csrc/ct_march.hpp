// ct_march.hpp -- fused constrained-transport step as one z-march kernel (spike_ctm.cu:250-298
// ct_march; physics of ct_mhd.jl:20-184).
//
// What it computes is the multi-pass CT step of ct_impl.hpp in one pass over HBM: cell-centred B
// and primitives, the lower-face fluxes with the face-normal field (each face solved once), the
// Balsara-Spicer edge EMFs, the hydro update and the face-B curl update, with the optional floor
// and OU kick.  The point functions are the same ones (ct_cell_states, ct_riemann).
//
// Layout on the GPU (the GLM march's, adapted to CT):
//   * A workgroup of 256 lanes owns a 16 x 12 column tile and a z-chunk.  Lanes 0..191 own the
//     tile row by row; lanes 192..251 are the one-cell ring around it, corners included (the
//     EMF at an edge of the tile needs fluxes of the ring's corner cells).  Every lane builds the
//     x, y and z face states of its cell; the LDS plane holds the primitives of plane q over the
//     tile grown by two cells (the in-plane neighbours of the ring).
//   * Per plane q: (1) +x/+y face states through LDS, x and y faces solved once; (2) fluxes back
//     through LDS, then the z face q-1/2 from the +z state carried from plane q-1 (solved after
//     the x/y fluxes have left the registers); (3) the z flux's field part through LDS; (4) the edge
//     EMFs of plane q (ex, ey need the y/x fluxes of plane q-1, carried per column); (5) the
//     update of plane q-1, whose curl needs ex, ey of plane q and the EMFs of plane q-1 (kept in
//     a two-plane LDS ring); (6) the prefetch and publish of plane q+1.
//   * HBM traffic: one read and one write of the 8 planes per cell and step, plus the halo and
//     the update base read again from L2.  The CFL of the result is a separate reduction.
//   * The OU kick's interpolation is cached per column in LDS (force.hpp): its corner loads happen
//     only when the column crosses a forcing plane.
#pragma once
#include "ct_impl.hpp"
#include "ct_launch.hpp"
#include "force.hpp"
#include "gpu_util.hpp"
#include "tiling.hpp"

namespace glm {

constexpr int CM_OX = 16, CM_OY = 12;
constexpr int CM_NO = CM_OX * CM_OY;                           // owned lanes
constexpr int CM_NH = 2 * (CM_OX + 2) + 2 * CM_OY;             // one-cell ring with corners
constexpr int CM_NL = CM_NO + CM_NH;                           // 252 lanes with a cell of their own
constexpr int CM_NT = 256;                                     // and 4 that only help (they repeat the last lane)
constexpr int CM_PX = CM_OX + 4, CM_PY = CM_OY + 4;            // LDS plane (two-cell ring)
constexpr int CM_NPL = CM_PX * CM_PY;
constexpr int CM_LX = CM_OX + 2;                               // row of the lanes' grown tile
static_assert(CM_LX * (CM_OY + 2) == CM_OX * CM_OY + 2 * (CM_OX + 2) + 2 * CM_OY, "one lane per grown-tile cell");
constexpr int CM_NHELP = 2 * (CM_OX + 2) + 2 * (CM_OY + 2);    // two-cell ring without its corners
static_assert(CM_NL <= CM_NT && CM_NT - CM_NO >= CM_NHELP && CM_NO % 64 == 0, "CT tile shape");
static_assert(CM_NT == CT_MARCH_THREADS, "launch width of the CT march");

#ifndef GLM_CT_WAVES_F64
#define GLM_CT_WAVES_F64 2
#endif
#ifndef GLM_CT_WAVES_F32
#define GLM_CT_WAVES_F32 3
#endif
#define GLM_CT_WAVES_PER_EU(T) (sizeof(T) == 8 ? GLM_CT_WAVES_F64 : GLM_CT_WAVES_F32)
// With species the FP64 LDS (93.5 KB) admits one workgroup per CU, which may then use every register;
// in FP32 two workgroups with no spills run 1.2-1.4x faster than three held to 168 registers
// (480^3, measured).
#define GLM_CT_WAVES_PER_EU_NS(T, NS) ((NS) > 0 ? (sizeof(T) == 8 ? 1 : 2) : GLM_CT_WAVES_PER_EU(T))
// The parabolic-edge builds without species: FP64 at one wave per SIMD (all 512 registers; at two
// they spill ~300 bytes per lane and run 8-12% slower, 320^3), FP32 at three like PLM (two: no gain).
#ifndef GLM_CT_PPM_WAVES_F64
#define GLM_CT_PPM_WAVES_F64 1
#endif
#ifndef GLM_CT_PPM_WAVES_F32
#define GLM_CT_PPM_WAVES_F32 3
#endif
#define GLM_CT_WAVES_RC(T, NS, RC) \
    ((NS) == 0 && (RC) == RECON_PPM_SPIKE ? (sizeof(T) == 8 ? GLM_CT_PPM_WAVES_F64 : GLM_CT_PPM_WAVES_F32) \
                                          : GLM_CT_WAVES_PER_EU_NS(T, NS))

template <typename T>
struct CTMArgs {
    const T* q[10];        // the 8 CT planes, then up to 2 species rho X_s
    T* o[10];
    int nx, ny, nz;
    int tiles_x, tiles_y, nzc, zchunk;
    T gamma, igm1, smallr, smallp, dtdx, half_dtdx, dt, dx, lx, ly, lz, smallc, turb_min_rho, ramp;
    int face_slope, recon, update_floor, do_turb, tgs;
    const T* afield;
    unsigned long long* cmax;   // cleared here for the CFL reduction that follows, or null
};

// Lane t's cell (tx, ty) in the tile grown by one cell (tx in 0..OX+1, ty in 0..OY+1).
GLM_DEV void cm_lane_cell(int t, int& tx, int& ty)
{
    if (t < CM_NO) { tx = 1 + t % CM_OX; ty = 1 + t / CM_OX; return; }
    const int h = t - CM_NO;
    if (h < CM_OX + 2) { tx = h; ty = 0; }
    else if (h < 2 * (CM_OX + 2)) { tx = h - (CM_OX + 2); ty = CM_OY + 1; }
    else if (h < 2 * (CM_OX + 2) + CM_OY) { tx = 0; ty = 1 + h - 2 * (CM_OX + 2); }
    else { tx = CM_OX + 1; ty = 1 + h - 2 * (CM_OX + 2) - CM_OY; }
}

// LDS plane position (px, py) of helper cell h: the two-cell ring without its four corners.
GLM_DEV void cm_helper_cell(int h, int& px, int& py)
{
    if (h < CM_OX + 2) { px = 1 + h; py = 0; }
    else if (h < 2 * (CM_OX + 2)) { px = 1 + h - (CM_OX + 2); py = CM_PY - 1; }
    else if (h < 2 * (CM_OX + 2) + CM_OY + 2) { px = 0; py = 1 + h - 2 * (CM_OX + 2); }
    else { px = CM_PX - 1; py = 1 + h - 2 * (CM_OX + 2) - (CM_OY + 2); }
}

// The exchange buffers XB/YB hold one slot per lane (the tile grown by one cell, row CM_LX); the
// primitive plane and the EMF ring cover the tile grown by two cells (row CM_PX).
template <typename T, int NV = 8>
struct CTMarchLDS {
    T P[NV][CM_NPL];       // primitives (and species fractions) of plane q (two-cell ring)
    T XB[NV][CM_NL];       // +x face states, then x fluxes (0..4 and species 8.., By in 6) and the z flux's Bx (5), By (7)
    T YB[NV][CM_NL];       // +y face states, then y fluxes (0..4 and species 8.., Bx in 5)
    T E[2][3][CM_NPL];     // edge EMFs ex, ey, ez of the last two planes (plane k in slot k & 1)
    T FCB[6][CM_NO];       // forcing interpolation cache (ForceCache) of the owned columns
};

// A column (x, y) of the grid and the byte offsets, within a z plane, of its cells and of their upper x
// and y neighbours, for planes below 4 GiB: the plane's base is one for the wavefront and an access adds
// its offset itself, where 64-bit lane addresses take a multiplication or two and an addition each.  256^3 in
// us with 64-bit addresses and with offsets, for LLF, HLL and HLLD:
//   used:      FP64 PLM 1558, 1589, 2146 -> 1529, 1543, 1977
//              FP32 PPM 1094, 1102, 1242 -> 948, 958, 1091; FP32 PLM HLLD 1069 -> 1025
//   not used:  FP32 PLM LLF and HLL 870, 856 -> 907, 906; with species 1254, 1262, 1348 -> 1272, 1284, 1405
//              FP64 PPM 2362, 2410, 2718 -> 2509, 2577, 2907; PLM with species 2498, 2523, 2823 -> 2646, 2661, 3003
// (the FP64 builds not using them run one wavefront a SIMD, have the registers and wait longer for the
// pointers).  64^3 to 192^3 are on the same side, or within 1% of the line.
template <typename T, int RIEM, int NS, int RC>
constexpr bool CM_OFFSETS = NS == 0 && (sizeof(T) == 8 ? RC == RECON_PLM : RIEM == RIEM_HLLD || RC != RECON_PLM);
struct CmColumn {
    int x, y;
    unsigned c, x1, y1;
};
template <typename T>
GLM_DEV CmColumn cm_column(int x, int y, int nx, int ny)
{
    const unsigned row = (unsigned)nx * (unsigned)y;
    return {x, y, (unsigned)sizeof(T) * ((unsigned)x + row), (unsigned)sizeof(T) * ((unsigned)cwrap(x + 1, nx) + row),
            (unsigned)sizeof(T) * ((unsigned)x + (unsigned)nx * (unsigned)cwrap(y + 1, ny))};
}

// Primitives with cell-centred B of a cell (ct_mhd.jl:26-34, :85-96) from its values and the face
// fields of its upper neighbours, then the species fractions X_s = rho X_s / max(rho, smallr)
// (spike_ctm.cu:260-263).
template <typename T, int NV>
GLM_DEV void cm_prim_of(const CTMArgs<T>& a, const T u[NV], T bx1, T by1, T bz1, T p[NV])
{
    const T bx = T(0.5) * (u[5] + bx1), by = T(0.5) * (u[6] + by1), bz = T(0.5) * (u[7] + bz1);
    T rho = tmax(u[0], a.smallr), ir = trcp(rho);
    T vx = u[1] * ir, vy = u[2] * ir, vz = u[3] * ir;
    T pr = ct_pressure(u[4], rho, vx, vy, vz, bx, by, bz, a.gamma, a.smallp);
    p[0] = rho; p[1] = vx; p[2] = vy; p[3] = vz; p[4] = pr; p[5] = bx; p[6] = by; p[7] = bz;
#pragma unroll
    for (int v = 8; v < NV; ++v) p[v] = u[v] * ir;
}
// of cell (x, y, z)
template <typename T, int NV = 8>
GLM_DEV void cm_prim(const CTMArgs<T>& a, int x, int y, int z, T p[NV])
{
    const size_t pl = (size_t)a.nx * a.ny;
    const size_t c = (size_t)x + (size_t)a.nx * y + pl * z;
    T u[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) u[v] = gload(a.q[v] + c);
    const T bx1 = gload(a.q[5] + ((size_t)cwrap(x + 1, a.nx) + (size_t)a.nx * y + pl * z));
    const T by1 = gload(a.q[6] + ((size_t)x + (size_t)a.nx * cwrap(y + 1, a.ny) + pl * z));
    const T bz1 = gload(a.q[7] + ((size_t)x + (size_t)a.nx * y + pl * cwrap(z + 1, a.nz)));
    cm_prim_of<T, NV>(a, u, bx1, by1, bz1, p);
}
// of a column's cell in plane z, by offsets where `narrow`
template <typename T, int NV, bool OFF, typename A>
GLM_DEV void cm_prim_at(const A& a, CmColumn k, int z, bool narrow, T p[NV])
{
    if constexpr (OFF) {
        if (__builtin_expect(narrow, 1)) {
            const auto* ap = &a;
            renew_s(ap);
            const size_t pl = (size_t)a.nx * a.ny, z0 = pl * z, z1 = pl * cwrap(z + 1, a.nz);
            renew_v(k.c); renew_v(k.x1); renew_v(k.y1);
            T u[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) u[v] = gload_at((const T*)ap->q[v] + z0, k.c);
            const T bx1 = gload_at((const T*)ap->q[5] + z0, k.x1);
            const T by1 = gload_at((const T*)ap->q[6] + z0, k.y1);
            const T bz1 = gload_at((const T*)ap->q[7] + z1, k.c);
            cm_prim_of<T, NV>(a, u, bx1, by1, bz1, p);
            return;
        }
        renew_v(k.x);   // nothing of the wide addresses is kept across the march
        renew_v(k.y);
    }
    cm_prim<T, NV>(a, k.x, k.y, z, p);
}

// Tiles and z-chunks of the CT march (lead-in: two whole planes of face states and fluxes).
template <typename T>
inline void ct_march_tiling(int nx, int ny, int nz, int zchunk_req, const Resident& r, int& tiles_x, int& tiles_y,
                            int& nzc, int& zchunk)
{
    march_tiles(nx, ny, nz, CM_OX, CM_OY, zchunk_req, r, 2.0, sizeof(T) == 8 ? 0.7 : 0.38, tiles_x, tiles_y, nzc, zchunk);
}

// One step of the CT state with NS passive species (spike_ctm.cu -DNSP: their fluxes ride the
// mass flux and are updated with the hydro planes): workgroup w marches tile xcd_block(w).  RC: the
// reconstruction (RECON_PLM or RECON_PPM_SPIKE), a template argument so that each build holds the
// registers of its own path only.
template <typename T, int RIEM, int NS = 0, int RC = RECON_PLM>
__global__ void __launch_bounds__(CM_NT) __attribute__((amdgpu_waves_per_eu(GLM_CT_WAVES_RC(T, NS, RC))))
ct_march_kernel(CTMArgs<T> a_)
{
    // the argument block read in place (kernarg_ref): HLLD + PLM at 320^3 FP64 5.75 -> 6.08 Gcell/s,
    // at 480^3 FP32 16.05 -> 16.58 (HLL PLM 0.5-1.4% slower, PPM within 1%)
    const auto& a = kernarg_ref<CTMArgs<T>>();
    constexpr int NV = 8 + NS, NH = 5 + NS;   // values per cell; hydro-updated values (species at 5..)
    __shared__ CTMarchLDS<T, NV> L;
    T (&P)[NV][CM_NPL] = L.P;
    T (&XB)[NV][CM_NL] = L.XB;
    T (&YB)[NV][CM_NL] = L.YB;
    const int tid = threadIdx.x;
    if (a.cmax && blockIdx.x == 0 && tid == 0) *a.cmax = 0ull;
    int tile = xcd_block((int)blockIdx.x, (int)gridDim.x);
    int tx, ty;
    cm_lane_cell(tid < CM_NL ? tid : CM_NL - 1, tx, ty);
    const int tile_x = tile % a.tiles_x; tile /= a.tiles_x;
    const int tile_y = tile % a.tiles_y; tile /= a.tiles_y;
    const int zs = tile * a.zchunk;
    const int ze = min(zs + a.zchunk, a.nz);
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const size_t plane = (size_t)nx * ny;
    const int gxu = tile_x * CM_OX - 1 + tx, gyu = tile_y * CM_OY - 1 + ty;
    const int gx = cwrap(gxu, nx), gy = cwrap(gyu, ny);
    const bool owned = tid < CM_NO && gxu < nx && gyu < ny;
    const bool corner = (tx == 0 || tx == CM_OX + 1) && (ty == 0 || ty == CM_OY + 1);
    const bool need_x = tx >= 1;                      // this lane solves the x face at tx - 1/2
    const bool need_y = ty >= 1;                      // and the y face at ty - 1/2
    const bool need_z = !corner;                      // and the z face below its cell
    const bool emf_z = tx >= 1 && ty >= 1;            // ez at the lane's lower x-y edge
    const bool emf_x = tx >= 1 && tx <= CM_OX && ty >= 1;
    const bool emf_y = tx >= 1 && ty >= 1 && ty <= CM_OY;
    constexpr bool OFF = CM_OFFSETS<T, RIEM, NS, RC>;
    const bool narrow = OFF && plane * sizeof(T) <= 0xffffffffu;
    auto wide = [&] {   // the column's index within a z plane
        int x = gx, y = gy;
        if (OFF) { renew_v(x); renew_v(y); }
        return (size_t)x + (size_t)nx * y;
    };
    const CmColumn col = cm_column<T>(gx, gy, nx, ny);
    const int lo = (ty + 1) * CM_PX + (tx + 1);
    const int li = ty * CM_LX + tx;
    const bool helper = tid >= CM_NO;   // the halo wavefront, which has no update, brings in the two-cell ring (by
                                        // the first owned one the HLLD + PLM step at 256^3 FP64 took 10% longer)
    int hx = 0, hy = 0;
    cm_helper_cell(helper ? tid - CM_NO : 0, hx, hy);
    const CmColumn hcol =
        cm_column<T>(cwrap(tile_x * CM_OX - 2 + hx, nx), cwrap(tile_y * CM_OY - 2 + hy, ny), nx, ny);
    const int lo_ring = hy * CM_PX + hx;

    // column window: primitives of planes q-1 and q+1 (plane q is read back from LDS)
    T pm[NV], pp[NV];
    {
        T p0[NV];
        cm_prim_at<T, NV, OFF>(a, col, cwrap(zs - 2, nz), narrow, pm);
        cm_prim_at<T, NV, OFF>(a, col, cwrap(zs - 1, nz), narrow, p0);
        cm_prim_at<T, NV, OFF>(a, col, cwrap(zs, nz), narrow, pp);
#pragma unroll
        for (int v = 0; v < NV; ++v) P[v][lo] = p0[v];
        if (helper) {
            T h[NV];
            cm_prim_at<T, NV, OFF>(a, hcol, cwrap(zs - 1, nz), narrow, h);
#pragma unroll
            for (int v = 0; v < NV; ++v) P[v][lo_ring] = h[v];
        }
    }
    __syncthreads();

    T zprev[NV];                // +z face state of plane q-1
    T fzp[NH];                  // hydro (and species) part of the z flux below plane q-1
    T pend[NH];                 // (Fx_lo - Fx_hi) + (Fy_lo - Fy_hi) of plane q-1
    T fxbz = T(0), fybz = T(0); // Fx[Bz], Fy[Bz] of this cell in plane q-1
#pragma unroll
    for (int v = 0; v < NV; ++v) zprev[v] = T(0);
#pragma unroll
    for (int v = 0; v < NH; ++v) { fzp[v] = T(0); pend[v] = T(0); }
    ForceCache<T, CM_NO> fc;
    fc.k0 = -0x7fffffff;
    fc.b = &L.FCB[0][tid < CM_NO ? tid : 0];

    for (int q = zs - 1; q <= ze; ++q) {
        const int zq = cwrap(q, nz);
        const bool lead = q == zs - 1;

        // face-normal fields of this cell's lower faces, loaded ahead of their Riemann solves
        T bnx, bny, bnz;
        if (__builtin_expect(narrow, 1)) {
            const auto* ap = &a;
            unsigned off = col.c;
            renew_s(ap);
            renew_v(off);
            bnx = gload_at((const T*)ap->q[5] + plane * zq, off);
            bny = gload_at((const T*)ap->q[6] + plane * zq, off);
            bnz = gload_at((const T*)ap->q[7] + plane * zq, off);
        } else {
            const size_t off = wide() + plane * zq;
            bnx = gload(a.q[5] + off); bny = gload(a.q[6] + off); bnz = gload(a.q[7] + off);
        }

        // ---- x and y face states of this lane's cell in plane q -----------------------------------
        T xlo[NV], ylo[NV];
        {
            T l[NV], c0[NV], r[NV], hi[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) { l[v] = P[v][lo - 1]; c0[v] = P[v][lo]; r[v] = P[v][lo + 1]; }
            ct_cell_states<T, 0, NV, RC>(l, c0, r, a, xlo, hi);
#pragma unroll
            for (int v = 0; v < NV; ++v) XB[v][li] = hi[v];
#pragma unroll
            for (int v = 0; v < NV; ++v) { l[v] = P[v][lo - CM_PX]; r[v] = P[v][lo + CM_PX]; }
            ct_cell_states<T, 1, NV, RC>(l, c0, r, a, ylo, hi);
#pragma unroll
            for (int v = 0; v < NV; ++v) YB[v][li] = hi[v];
        }
        __syncthreads();

        // ---- x and y faces ------------------------------------------------------------------------
        T fx[NV], fy[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) { fx[v] = T(0); fy[v] = T(0); }
        if (need_x) {
            T Lx[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) Lx[v] = XB[v][li - 1];
            ct_riemann<T, RIEM, 0, NV>(Lx, xlo, bnx, a, fx);
        }
        if (need_y) {
            // FP64 HLLD + PLM without species: the -y state again from the plane rather than held
            // across the x solve (200 -> 136 B of spills per lane, 6.08 -> 6.25 Gcell/s at 320^3; the
            // other builds run 5-10% slower with the extra cell state, so they keep it in registers)
            if constexpr (sizeof(T) == 8 && RIEM == RIEM_HLLD && RC == RECON_PLM && NS == 0) {
                T l[NV], c0[NV], r[NV], hi[NV];
#pragma unroll
                for (int v = 0; v < NV; ++v) { l[v] = P[v][lo - CM_PX]; c0[v] = P[v][lo]; r[v] = P[v][lo + CM_PX]; }
                ct_cell_states<T, 1, NV, RC>(l, c0, r, a, ylo, hi);
            }
            T Ly[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) Ly[v] = YB[v][li - CM_LX];
            ct_riemann<T, RIEM, 1, NV>(Ly, ylo, bny, a, fy);
        }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 5; ++v) { XB[v][li] = fx[v]; YB[v][li] = fy[v]; }
#pragma unroll
        for (int v = 8; v < NV; ++v) { XB[v][li] = fx[v]; YB[v][li] = fy[v]; }
        XB[6][li] = fx[6];
        YB[5][li] = fy[5];
        const T fx7 = fx[7], fy7 = fy[7];
        __asm__ volatile("" ::: "memory");   // the other flux components are read back from LDS below

        // ---- z face q-1/2 (the plane's LDS cells are untouched until the publish) -----------------
        T fz[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) fz[v] = T(0);
        {
            T c0[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) c0[v] = P[v][lo];
            T zlo[NV], zhi[NV];
            ct_cell_states<T, 2, NV, RC>(pm, c0, pp, a, zlo, zhi);
            if (need_z && !lead) ct_riemann<T, RIEM, 2, NV>(zprev, zlo, bnz, a, fz);
#pragma unroll
            for (int v = 0; v < NV; ++v) zprev[v] = zhi[v];
        }
        if (!lead) { XB[5][li] = fz[5]; XB[7][li] = fz[6]; }
        __syncthreads();

        if (!lead) {
            // ---- edge EMFs of plane q (ct_mhd.jl:139-154) ----------------------------------------
            // ez at (i-1/2, j-1/2), ex at (j-1/2, k-1/2), ey at (i-1/2, k-1/2) of this lane's cell
            T ex = T(0), ey = T(0), ez = T(0);
            if (emf_z) ez = T(0.25) * (YB[5][li] + YB[5][li - 1] - XB[6][li] - XB[6][li - CM_LX]);
            if (emf_x) ex = T(0.25) * (fz[6] + XB[7][li - CM_LX] - fy7 - fybz);
            if (emf_y) ey = T(0.25) * (fx7 + fxbz - fz[5] - XB[5][li - 1]);
            T (&Ec)[3][CM_NPL] = L.E[q & 1];
            T (&Ep)[3][CM_NPL] = L.E[(q - 1) & 1];
            Ec[0][lo] = ex; Ec[1][lo] = ey; Ec[2][lo] = ez;

            // ---- update of plane q-1 (ct_mhd.jl:124-136, :156-171) --------------------------------
            if (owned && q >= zs + 1) {
                const int zu = cwrap(q - 1, nz);
                const size_t zo = plane * zu;
                size_t ow = OFF ? 0 : wide() + zo;
                T r[NH], b0[NH], bo[3];   // hydro values, then species (plane 8 + s at index 5 + s); face fields
                const auto* ap = &a;
                renew_s(ap);
                if (__builtin_expect(narrow, 1)) {
                    unsigned off = col.c;
                    renew_v(off);
#pragma unroll
                    for (int t = 0; t < NH; ++t) b0[t] = gload_at((const T*)ap->q[t < 5 ? t : t + 3] + zo, off);
#pragma unroll
                    for (int t = 0; t < 3; ++t) bo[t] = gload_at((const T*)ap->q[5 + t] + zo, off);
                } else {
                    if (OFF) ow = wide() + zo;
#pragma unroll
                    for (int t = 0; t < NH; ++t) b0[t] = gload(a.q[t < 5 ? t : t + 3] + ow);
#pragma unroll
                    for (int t = 0; t < 3 && OFF; ++t) bo[t] = gload(a.q[5 + t] + ow);
                }
#pragma unroll
                for (int t = 0; t < NH; ++t) r[t] = b0[t] + a.dtdx * (pend[t] + (fzp[t] - fz[t < 5 ? t : t + 3]));
                const T ex0 = Ep[0][lo], ey0 = Ep[1][lo], ez0 = Ep[2][lo];
                auto face_b = [&](int t) { return OFF ? bo[t] : gload(a.q[5 + t] + ow); };
                const T bxn = face_b(0) - a.dtdx * ((Ep[2][lo + CM_PX] - ez0) - (ey - ey0));
                const T byn = face_b(1) - a.dtdx * ((ex - ex0) - (Ep[2][lo + 1] - ez0));
                const T bzn = face_b(2) - a.dtdx * ((Ep[1][lo + 1] - ey0) - (Ep[0][lo + CM_PX] - ex0));
                if (a.update_floor && r[0] < a.smallr) {
                    T emag = T(0.5) * (pm[5] * pm[5] + pm[6] * pm[6] + pm[7] * pm[7]);
                    r[0] = a.smallr; r[1] = T(0); r[2] = T(0); r[3] = T(0); r[4] = a.smallp * a.igm1 + emag;
                    // the species keep their fraction: rho X = smallr X_old
#pragma unroll
                    for (int t = 5; t < NH; ++t) r[t] = a.smallr * (b0[t] * trcp(tmax(b0[0], a.smallr)));
                }
                if (a.do_turb && r[0] >= a.turb_min_rho) {
                    T acc[3];
                    force_accel(fc, a, gx, gy, zu, acc);
                    T rho = r[0], rhom = tmax(rho, a.smallr), irm = trcp(rhom), fl = rho * a.smallc * a.smallc, e = r[4];
                    e = tmax(e - T(0.5) * r[1] * r[1] * irm, fl);
                    e = tmax(e - T(0.5) * r[2] * r[2] * irm, fl);
                    e = tmax(e - T(0.5) * r[3] * r[3] * irm, fl);
                    T m2 = r[1] + rhom * acc[0] * a.dt, m3 = r[2] + rhom * acc[1] * a.dt, m4 = r[3] + rhom * acc[2] * a.dt;
                    e = tmax(e + T(0.5) * m2 * m2 * irm, fl);
                    e = tmax(e + T(0.5) * m3 * m3 * irm, fl);
                    e = tmax(e + T(0.5) * m4 * m4 * irm, fl);
                    r[1] = m2; r[2] = m3; r[3] = m4; r[4] = e;
                }
                const T bn[3] = {bxn, byn, bzn};
                renew_s(ap);
                if (__builtin_expect(narrow, 1)) {
                    unsigned off = col.c;
                    renew_v(off);
#pragma unroll
                    for (int t = 0; t < NH; ++t) gstore_nt_at(r[t], (T*)ap->o[t < 5 ? t : t + 3] + zo, off);
#pragma unroll
                    for (int t = 0; t < 3; ++t) gstore_nt_at(bn[t], (T*)ap->o[5 + t] + zo, off);
                } else {
                    if (OFF) ow = wide() + zo;
#pragma unroll
                    for (int t = 0; t < NH; ++t) gstore_nt(r[t], (T*)a.o[t < 5 ? t : t + 3] + ow);
#pragma unroll
                    for (int t = 0; t < 3; ++t) gstore_nt(bn[t], (T*)a.o[5 + t] + ow);
                }
            }
            // in-plane flux differences of plane q for its update in the next pass
            if (owned) {
#pragma unroll
                for (int t = 0; t < NH; ++t) {
                    const int v = t < 5 ? t : t + 3;
                    pend[t] = (XB[v][li] - XB[v][li + 1]) + (YB[v][li] - YB[v][li + CM_LX]);
                }
            }
#pragma unroll
            for (int t = 0; t < NH; ++t) fzp[t] = fz[t < 5 ? t : t + 3];
        }
        fxbz = fx7;
        fybz = fy7;
        if (q == ze) break;

        // ---- prefetch and publish plane q+1 -------------------------------------------------------
        // The prefetch and publish run ahead of the other workgroup's wavefront on this SIMD, so the
        // workgroups reach the plane's last barrier sooner (FP32 PPM +2%, FP64 HLLD + PLM +1.7%).
        __builtin_amdgcn_s_setprio(1);
        T pn[NV], hn[NV];
        cm_prim_at<T, NV, OFF>(a, col, cwrap(q + 2, nz), narrow, pn);
        if (helper) cm_prim_at<T, NV, OFF>(a, hcol, cwrap(q + 1, nz), narrow, hn);
        __syncthreads();   // every read of plane q's LDS cells and of the flux exchange is done
#pragma unroll
        for (int v = 0; v < NV; ++v) { pm[v] = P[v][lo]; P[v][lo] = pp[v]; pp[v] = pn[v]; }
        if (helper) {
#pragma unroll
            for (int v = 0; v < NV; ++v) P[v][lo_ring] = hn[v];
        }
        __syncthreads();
        __builtin_amdgcn_s_setprio(0);
    }
}

}  // namespace glm
