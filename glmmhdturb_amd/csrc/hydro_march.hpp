// hydro_march.hpp -- the 5-variable hydro line march (spike_25d.cu:383-516 as build_march.sh
// builds it: -DHANCOCK1D, optional -DLLF_FALLBACK) as one z-march kernel for gfx950.
//
// Scheme per cell and direction d: primitive state (:196-202), MonCen slopes of the cells at
// -1, 0, +1 (:207-221), the normal-only Hancock half step (:287-301), face states at mh -/+ s/2
// clamped at SMALLR/SMALLP (:222-230), HLL (:302-330) or HLL with the LLF fallback (:335-376),
// div += F(+1/2) - F(-1/2) in the order x, y, z (:486-487), U1 = toCons(prim(U0)) - dtdx*div
// (:432, :492).  Periodic in all three axes.
//
// Layout: 5 SoA planes [rho, mx, my, mz, E], cell (i,j,k) at i + nx*(j + ny*k); with NSP = 2
// passive scalars (-DSCALARS, :115-119) two more planes of rho*s, advected as s (:191, :241,
// :251, :298), their flux the HLL/LLF flux of rho*s or, with CMA (-DCMA), the HLL mass flux times
// the upwind face value of s (:321, :367).
//
// Kernel shape.  A workgroup of 256 lanes owns a 30 x 16 column tile and a chunk of z planes.  Half a
// wavefront is one row of 32 cells (the 30 owned and one more on each side), and each lane carries the
// columns of two neighbouring rows.  What bounds it is the issue of VALU instructions, so each face
// state and face is computed as few times as its direction allows without a workgroup barrier:
//   x: every lane builds the states of its own cell once and solves its lower face; the upper face of the
//      lower neighbour and the flux of the upper one come from the next lane (DPP wave shift, no LDS
//      round trip);
//   y: four cells' states and three faces for a lane's two rows, from the LDS plane;
//   z: one cell's states and one face per plane and row; the upper state is carried to the next plane.
// Per owned cell that is 4 slopes and half steps and 3.5 solves (times 32/30), where a lane per column
// with both its faces in each direction took 8 and 5: 480^3 FP32 2.52 -> 1.90 ms (1.99 with the flux sums below).
//   LDS holds the primitives of planes k and k+1 over the tile grown by two cells (34 x 20): a lane's own
// cells reach plane k+2 in registers, the halo's plane k+1 is fetched during plane k, so one barrier
// per plane suffices.  The loop starts two planes early so that the chunk's first z states and face
// come from the loop's own code, and the flux functions are not contracted by the compiler (their
// fused operations are written out): a face has the same bits in every row, lane and chunking.
#pragma once
#include "gpu_util.hpp"
#include "tiling.hpp"

namespace glm {

constexpr int HM_OX = 30, HM_OY = 16;
constexpr int HM_W = HM_OX + 2;                      // lanes of a row
constexpr int HM_LX = HM_OX + 4, HM_LY = HM_OY + 4;  // LDS plane: the tile grown by two cells
constexpr int HM_NPL = HM_LX * HM_LY;
constexpr int HM_NT = HM_W * HM_OY / 2;              // 256 lanes, two rows each
constexpr int HM_NHALO = 4 * HM_W + 2 * HM_OY;       // plane cells no lane owns: two rows below and above, the outer columns
constexpr int HM_SEAM_X = 32, HM_SEAM_Y = 8;         // the reference's 32 x 8 tiles, whose seams HY_DONOR treats
static_assert(HM_W == 32 && HM_NT == 256 && HM_NHALO <= HM_NT, "two rows of 32 lanes per wavefront");

constexpr int HM_NVMAX = 7;   // 5 hydro variables + 2 passive scalars (-DSCALARS)

// Storage formats of the state in HBM (spike_25d.cu:64-95, the compact-storage builds):
//   HY_CONS   conserved planes of T (the build_march.sh library);
//   HY_F16P   -DF16STATE: primitive rho, vx, vy, vz, p as f16;
//   HY_U16P   -DU16STATE: primitive, rho and p as uint16 log2 over [-32, 32], velocities uint16
//             linear over [-8, 8];
//   HY_U16SP  -DU16SP: conserved hydro planes of T, the two species fractions as uint16 log2 over
//             [-110, 0], reconstructed in log2 (the CMA flux and the conserved rho X decode X).
// The compact formats compute in FP32.
enum { HY_CONS = 0, HY_F16P = 1, HY_U16P = 2, HY_U16SP = 3 };

template <typename T>
struct HydroArgs {
    const T* q[HM_NVMAX];
    T* o[HM_NVMAX];
    const unsigned short* qh[HM_NVMAX];   // 16-bit planes of the compact formats
    unsigned short* oh[HM_NVMAX];
    int nx, ny, nz;
    int tiles_x, tiles_y, nzc, zchunk;
    T gm1, igm1, gamma, dtdx, smallr, smallp, fb_dmin, fb_pmin;
};

// uint16 codecs (spike_25d.cu:157-168): log2 over [-110, 0] (species), velocity linear over
// [-8, 8], log2 over [-32, 32] (rho, p); encode rounds to nearest and clamps.  Not contracted:
// each is a float multiply and a float add, so a codec is a fixed function of its input.
GLM_DEV float hy_dec_log2(unsigned short u)
{
#pragma clang fp contract(off)
    return -110.f + (float)u * (110.f / 65535.f);
}
GLM_DEV unsigned short hy_enc_log2(float l2)
{
#pragma clang fp contract(off)
    float t = (l2 + 110.f) * (65535.f / 110.f);
    t = fminf(fmaxf(t, 0.f), 65535.f);
    return (unsigned short)(t + 0.5f);
}
GLM_DEV float hy_dec_vel(unsigned short u)
{
#pragma clang fp contract(off)
    return -8.f + (float)u * (16.f / 65535.f);
}
GLM_DEV unsigned short hy_enc_vel(float x)
{
#pragma clang fp contract(off)
    const float t = (fminf(fmaxf(x, -8.f), 8.f) + 8.f) * (65535.f / 16.f);
    return (unsigned short)(t + 0.5f);
}
GLM_DEV float hy_dec_log2s(unsigned short u)
{
#pragma clang fp contract(off)
    return -32.f + (float)u * (64.f / 65535.f);
}
GLM_DEV unsigned short hy_enc_log2s(float l2)
{
#pragma clang fp contract(off)
    float t = (l2 + 32.f) * (65535.f / 64.f);
    t = fminf(fmaxf(t, 0.f), 65535.f);
    return (unsigned short)(t + 0.5f);
}
GLM_DEV float hy_f16_to_f32(unsigned short h) { return (float)__builtin_bit_cast(_Float16, h); }
GLM_DEV unsigned short hy_f32_to_f16(float x) { return __builtin_bit_cast(unsigned short, (_Float16)x); }
template <typename T>
GLM_HD T hy_exp2(T x) { return (T)exp2f((float)x); }

// spike_25d.cu:196-202 prim_from_cons (:183-194 with scalars: s = (rho s) / rho; with LG the scalar
// planes already hold log2 X, :188-190)
template <typename T, int NV, bool LG = false>
GLM_DEV void hy_c2p(const T c[NV], T q[NV], const HydroArgs<T>& a)
{
#pragma clang fp contract(off)   // the same bits at every call site of the kernel
    const T r = tmax(c[0], a.smallr);
    const T ir = trcp(r);
    q[0] = r;
    q[1] = c[1] * ir;
    q[2] = c[2] * ir;
    q[3] = c[3] * ir;
    const T ke = T(0.5) * r * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]);
    q[4] = tmax(a.gm1 * (c[4] - ke), a.smallp);
#pragma unroll
    for (int v = 5; v < NV; ++v) q[v] = LG ? c[v] : c[v] * ir;
}

// a*b + c as one operation.  The flux functions below are compiled without contraction and write their
// fused operations out, so that every copy of them (two rows, three faces, three directions) rounds alike.
GLM_HD double tfma(double a, double b, double c) { return __builtin_fma(a, b, c); }
GLM_HD float tfma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// spike_25d.cu:245-255 toCons of the old primitives less dt/dx of the flux differences (with LG the scalars are
// log2 X, decoded for the conserved rho X, :248-250).  The products of toCons are fused into the sum, so
// that a value is rounded once at its own size (128^3 FP32, error of the momenta after a step 3.85e-8 -> 3.57e-8).
template <typename T, int NV, bool LG = false>
GLM_HD void hy_update(const T q[NV], const T div[NV], T u[NV], const HydroArgs<T>& a)
{
#pragma clang fp contract(off)
    u[0] = tfma(-a.dtdx, div[0], q[0]);
#pragma unroll
    for (int c = 1; c < 4; ++c) u[c] = tfma(q[0], q[c], -a.dtdx * div[c]);
    const T v2 = tfma(q[1], q[1], tfma(q[2], q[2], q[3] * q[3]));
    u[4] = tfma(q[4], a.igm1, tfma(T(0.5) * q[0], v2, -a.dtdx * div[4]));
#pragma unroll
    for (int v = 5; v < NV; ++v) u[v] = tfma(q[0], LG ? hy_exp2(q[v]) : q[v], -a.dtdx * div[v]);
}

// Scheme variants of the march (spike_25d.cu build flags): HY_PLM the light march (-DHANCOCK1D:
// MonCen slopes, normal-only Hancock half step, edges clamped at SMALLR/SMALLP, :462-466); HY_PPM1D
// the parabolic-edge variant (-DPPM1D, :467-483: the monotonized 3-point parabola's edge plus the
// half step's change mh - c, no clamp, HLL without the fallback); HY_DONOR (-DDONOR, :438-454): the
// light march with donor-cell HLL of the two cell states at the x and y faces of the 32 x 8 tiles
// (a face at x = i - 1/2 with i mod 32 = 0, at y = j - 1/2 with j mod 8 = 0; z has none), HLL
// without the fallback.
enum { HY_PLM = 0, HY_PPM1D = 1, HY_DONOR = 2 };

// The two face states of cell c along D from its neighbours l and r: half the MonCen slope (:207-221), the
// normal-only Hancock half step mh (:287-301), then mh -+ half slope clamped at SMALLR/SMALLP (:222-230)
// or the PPM1D parabola's edges plus mh - c, unclamped (:476-479).
template <typename T, int D, int NV, int SV>
GLM_DEV void hy_states(const T l[NV], const T c[NV], const T r[NV], T lo[NV], T hi[NV], const HydroArgs<T>& a)
{
#pragma clang fp contract(off)
    T hs[NV], mh[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) hs[v] = moncen_half(c[v] - l[v], r[v] - c[v]);
    // the half step is dt/dx times the half slope
    const T un = c[1 + D], sn = hs[1 + D], k = -a.dtdx;
    const T kn = k * un;
#pragma unroll
    for (int v = 0; v < NV; ++v) mh[v] = tfma(kn, hs[v], c[v]);   // advection, the whole of a scalar's half step (:298)
    mh[0] = tfma(k * c[0], sn, mh[0]);
    mh[1 + D] = tfma(k * trcp(c[0]), hs[4], mh[1 + D]);
    mh[4] = tfma(k * a.gamma * c[4], sn, mh[4]);
    if (SV == HY_PPM1D) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            T dl, dr;   // the edge is c - dl or c + dr; plus mh - c
            ppm_offsets_spike(l[v], c[v], r[v], dl, dr);
            lo[v] = mh[v] - dl;
            hi[v] = mh[v] + dr;
        }
    } else {
#pragma unroll
        for (int v = 0; v < NV; ++v) { lo[v] = mh[v] - hs[v]; hi[v] = mh[v] + hs[v]; }
        lo[0] = tmax(lo[0], a.smallr); hi[0] = tmax(hi[0], a.smallr);
        lo[4] = tmax(lo[4], a.smallp); hi[4] = tmax(hi[4], a.smallp);
    }
}

// HLL (spike_25d.cu:302-330); with FB, LLF where a face state is below the fallback floors
// (riemann_fb, :335-376).  With CMA the scalar fluxes of the HLL fan are the mass flux times the upwind
// face value (:321, :367).
//
// F = wL FL + wR FR + k (UL - UR) with wL = sR / (sR - sL), wR = -sL / (sR - sL) and k = -sL wL; weights
// of 1/2 and k = max(|u| + a)/2 make it LLF: three selects instead of one per component.  The jumps are formed
// before they are multiplied: as wL (FL - sL UL) + wR (FR - sR UR), 12 operations less, the terms -+k U are
// rounded before they cancel, and at Mach 0.01 with 2% jumps the mass flux loses a factor of 70 of its accuracy.
//
// Where both waves go one way the flux is that side's, and nothing of the other side enters it, be it infinite or
// NaN.  By a branch, or with SEL by selects: the branch is the faster one (480^3 FP32 1.99 ms, with
// selects 2.05) except in the FP64 builds whose registers it makes spill (256^3 705 us with 36 B spilled,
// with selects 670; PPM1D at 192^3 488 and 376).
template <typename T, int D, bool FB, int NV, bool CMA, bool LG = false, bool SEL = false>
GLM_HD void hy_riemann(const T L_[NV], const T R_[NV], T F[NV], const HydroArgs<T>& a)
{
#pragma clang fp contract(off)
    T L[NV], R[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) { L[v] = L_[v]; R[v] = R_[v]; }
    const T aL = tsqrt_pos(a.gamma * L[4] * trcp(L[0])), aR = tsqrt_pos(a.gamma * R[4] * trcp(R[0]));
    const T sL = tmin(L[1 + D] - aL, R[1 + D] - aR), sR = tmax(L[1 + D] + aL, R[1 + D] + aR);
    const bool llf = FB && (L[0] < a.fb_dmin || L[4] < a.fb_pmin || R[0] < a.fb_dmin || R[4] < a.fb_pmin);
    const bool up = sL >= T(0) && !llf, down = sR <= T(0) && !llf;
    if (!SEL && (up || down)) {
        T X[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) X[v] = up ? L[v] : R[v];
        const T m = X[0] * X[1 + D];
        const T E = tfma(X[4], a.igm1, T(0.5) * X[0] * tfma(X[1], X[1], tfma(X[2], X[2], X[3] * X[3])));
        F[0] = m;
#pragma unroll
        for (int c = 1; c < 4; ++c) F[c] = m * X[c];
        F[1 + D] = F[1 + D] + X[4];
        F[4] = (E + X[4]) * X[1 + D];
#pragma unroll
        for (int v = 5; v < NV; ++v) F[v] = m * (LG ? hy_exp2(X[v]) : X[v]);
        return;
    }
    const T inv = trcp(sR - sL);
    T wL = sR * inv, wR = -sL * inv, k = -sL * wL;
    if (FB) {
        const T sm = tmax(tabs(L[1 + D]) + aL, tabs(R[1 + D]) + aR);
        wL = llf ? T(0.5) : wL;
        wR = llf ? T(0.5) : wR;
        k = llf ? T(0.5) * sm : k;
    }
    if (SEL) {   // both sides the one
#pragma unroll
        for (int v = 0; v < NV; ++v) { L[v] = down ? R_[v] : L_[v]; R[v] = up ? L_[v] : R_[v]; }
        wL = up || down ? T(1) : wL;
        wR = up || down ? T(0) : wR;
        k = up || down ? T(0) : k;
    }
    const T bL = wL * L[1 + D], bR = wR * R[1 + D];
    const T mL = L[0] * bL, mR = R[0] * bR;
    F[0] = tfma(k, L[0] - R[0], tfma(L[0], bL, mR));
#pragma unroll
    for (int c = 1; c < 4; ++c) {
        const T uy = R[0] * R[c];
        F[c] = tfma(k, tfma(L[0], L[c], -uy), tfma(mL, L[c], bR * uy));
    }
    F[1 + D] = F[1 + D] + tfma(wL, L[4], wR * R[4]);
    const T EL = tfma(L[4], a.igm1, T(0.5) * L[0] * tfma(L[1], L[1], tfma(L[2], L[2], L[3] * L[3])));
    const T ER = tfma(R[4], a.igm1, T(0.5) * R[0] * tfma(R[1], R[1], tfma(R[2], R[2], R[3] * R[3])));
    F[4] = tfma(k, EL - ER, tfma(bL, EL + L[4], bR * (ER + R[4])));
#pragma unroll
    for (int v = 5; v < NV; ++v) {
        if (CMA && !llf) {
            const T x = F[0] >= T(0) ? L[v] : R[v];
            F[v] = F[0] * (LG ? hy_exp2(x) : x);
        } else {
            const T xL = LG ? hy_exp2(L[v]) : L[v], ux = R[0] * (LG ? hy_exp2(R[v]) : R[v]);
            F[v] = tfma(k, tfma(L[0], xL, -ux), tfma(mL, xL, bR * ux));
        }
    }
}

// The value of the previous / next lane of the wavefront.
GLM_DEV float lane_prev(float x)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x138, 0xf, 0xf, false));
}
GLM_DEV float lane_next(float x)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x130, 0xf, 0xf, false));
}
GLM_DEV double lane_prev(double x)
{
    int2 w = __builtin_bit_cast(int2, x);
    w.x = __builtin_amdgcn_update_dpp(0, w.x, 0x138, 0xf, 0xf, false);
    w.y = __builtin_amdgcn_update_dpp(0, w.y, 0x138, 0xf, 0xf, false);
    return __builtin_bit_cast(double, w);
}
GLM_DEV double lane_next(double x)
{
    int2 w = __builtin_bit_cast(int2, x);
    w.x = __builtin_amdgcn_update_dpp(0, w.x, 0x130, 0xf, 0xf, false);
    w.y = __builtin_amdgcn_update_dpp(0, w.y, 0x130, 0xf, 0xf, false);
    return __builtin_bit_cast(double, w);
}

// Tiles and z-chunks of the hydro march (lead-in: the two priming iterations and the window's load; a
// plane takes 2.65 us alone and 6.0 with three resident in FP32, 3.9 and 8 with two in FP64).
template <typename T>
inline void hydro_tiling(int nx, int ny, int nz, int zchunk_req, const Resident& r, int& tiles_x, int& tiles_y, int& nzc,
                         int& zchunk)
{
    march_tiles(nx, ny, nz, HM_OX, HM_OY, zchunk_req, r, 0.7, sizeof(T) == 8 ? 0.9 : 0.6, tiles_x, tiles_y, nzc, zchunk);
}

// Resident wavefronts per SIMD that the register allocation is held to (480^3).  FP32: 3 (144 to 168 registers,
// no spills, 2.09 ms; at 4, 128 registers with 76 B of spills, 2.55), with scalars 2 (2.83 ms; 3 with 108 B of
// spills 3.60).  FP64: 2 (4.23 ms, at one 4.57; with the fallback 4.38 and 4.74, PPM1D 5.57 and 5.79), with
// scalars or donor seams, which would spill 140-552 B at 256 registers, 1 (scalars 5.9 ms, at two 9.7; donor
// 4.8, at two 6.5).
#ifndef GLM_HY_WAVES
#define GLM_HY_WAVES(T, NSP, SV) (sizeof(T) == 8 ? ((NSP) || (SV) == HY_DONOR ? 1 : 2) : ((NSP) ? 2 : 3))
#endif

template <typename T, bool FB, int NSP, bool CMA, int FMT = HY_CONS, int SV = HY_PLM>
__global__ void __launch_bounds__(HM_NT) __attribute__((amdgpu_waves_per_eu(GLM_HY_WAVES(T, NSP, SV))))
hydro_march_kernel(HydroArgs<T> a)
{
    constexpr int NV = 5 + NSP;
    constexpr bool LG = FMT == HY_U16SP;      // species held as log2 X
    constexpr bool PRIM = FMT == HY_F16P || FMT == HY_U16P;   // primitive storage: no conversion on load
    constexpr bool fb = FB && SV == HY_PLM;
    constexpr bool sel = sizeof(T) == 8 && GLM_HY_WAVES(T, NSP, SV) > 1 && !fb;   // hy_riemann
    static_assert(FMT == HY_CONS || (sizeof(T) == 4 && (FMT != HY_U16SP || (NSP == 2 && CMA)) &&
                                     (FMT == HY_U16SP || NSP == 0)), "compact formats: FP32; U16SP with 2 CMA species");
    __shared__ T P[2][NV][HM_NPL];   // primitives of plane j in P[j & 1]
    const int tid = threadIdx.x;
    const int lx = tid % HM_W, ly = tid / HM_W * 2;   // the lane's column in the row of 32, its lower row
    const int ntile = a.tiles_x * a.tiles_y;
    const int w = xcd_block((int)blockIdx.x, (int)gridDim.x);   // neighbouring tiles share an XCD's L2
    const int tile = w % ntile, zc = w / ntile;
    const int x0 = (tile % a.tiles_x) * HM_OX, y0 = (tile / a.tiles_x) * HM_OY;
    const int k0 = zc * a.zchunk;
    const int k1 = k0 + a.zchunk < a.nz ? k0 + a.zchunk : a.nz;
    const size_t plane = (size_t)a.nx * a.ny;
    // the lane's columns; those outside the tile or the grid are wrapped and store nothing
    const int gx = wrapi(x0 - 1 + lx, a.nx), gy0 = wrapi(y0 + ly, a.ny), gy1 = wrapi(y0 + ly + 1, a.ny);
    const size_t col[2] = {(size_t)gx + (size_t)a.nx * gy0, (size_t)gx + (size_t)a.nx * gy1};
    const bool ownx = lx >= 1 && lx <= HM_OX && x0 - 1 + lx < a.nx;
    const bool own[2] = {ownx && y0 + ly < a.ny, ownx && y0 + ly + 1 < a.ny};
    const int li = (ly + 2) * HM_LX + lx + 1;   // the lower row's cell of the LDS plane
    // the halo cell this lane brings in: rows -2, -1, 16, 17 of the lanes' columns, then columns -2 and 31
    const bool halo = tid < HM_NHALO;
    int hpx = 1 + lx, hpy = ly / 2 < 2 ? ly / 2 : HM_OY + ly / 2;
    if (tid >= 4 * HM_W) {
        hpx = (tid & 1) ? HM_LX - 1 : 0;
        hpy = 2 + (tid - 4 * HM_W) / 2;
    }
    const int hi_ = halo ? hpy * HM_LX + hpx : 0;
    const size_t hcol = halo ? (size_t)wrapi(x0 - 2 + hpx, a.nx) + (size_t)a.nx * wrapi(y0 - 2 + hpy, a.ny) : 0;

    // a cell as it lies in HBM, decoded (cell g of the state)
    auto fetch = [&](size_t g, T c[NV]) {
        if (FMT == HY_CONS) {
#pragma unroll
            for (int v = 0; v < NV; ++v) c[v] = gload(a.q[v] + g);
        } else if (FMT == HY_F16P) {
#pragma unroll
            for (int v = 0; v < 5; ++v) c[v] = (T)hy_f16_to_f32(gload(a.qh[v] + g));
        } else if (FMT == HY_U16P) {   // spike_25d.cu:397-402
            c[0] = (T)exp2f(hy_dec_log2s(gload(a.qh[0] + g)));
#pragma unroll
            for (int v = 1; v < 4; ++v) c[v] = (T)hy_dec_vel(gload(a.qh[v] + g));
            c[4] = (T)exp2f(hy_dec_log2s(gload(a.qh[4] + g)));
        } else {                       // HY_U16SP, :409-411
#pragma unroll
            for (int v = 0; v < 5; ++v) c[v] = gload(a.q[v] + g);
#pragma unroll
            for (int v = 5; v < NV; ++v) c[v] = (T)hy_dec_log2(gload(a.qh[v] + g));
        }
    };
    // its primitives: every primitive value of the kernel comes from here
    auto prim = [&](const T c[NV], T q[NV]) {
        if (PRIM) {   // make_prim (spike_25d.cu:204-206)
#pragma unroll
            for (int v = 0; v < NV; ++v) q[v] = c[v];
            q[0] = tmax(q[0], a.smallr);
            q[4] = tmax(q[4], a.smallp);
        } else {
            hy_c2p<T, NV, LG>(c, q, a);
        }
    };
    auto zoff = [&](int k) { return (size_t)wrapi(k, a.nz) * plane; };
    auto lds = [&](int k, int at, T q[NV]) {
#pragma unroll
        for (int v = 0; v < NV; ++v) q[v] = P[k & 1][v][at];
    };
    // U1 = toCons(prim(U0)) - dtdx div of cell g
    auto store = [&](size_t g, const T p0[NV], const T div[NV]) {
        T U[NV];
        hy_update<T, NV, LG>(p0, div, U, a);
        if (FMT == HY_CONS) {
#pragma unroll
            for (int v = 0; v < NV; ++v) a.o[v][g] = U[v];
        } else if (PRIM) {   // c2p -> store primitive (spike_25d.cu:499-511)
            const T ir = T(1) / tmax(U[0], a.smallr);
            const T vx = U[1] * ir, vy = U[2] * ir, vz = U[3] * ir;
            const T ke = T(0.5) * U[0] * (vx * vx + vy * vy + vz * vz);
            const T pp = tmax(a.gm1 * (U[4] - ke), a.smallp);
            if (FMT == HY_F16P) {
                a.oh[0][g] = hy_f32_to_f16((float)U[0]);
                a.oh[1][g] = hy_f32_to_f16((float)vx);
                a.oh[2][g] = hy_f32_to_f16((float)vy);
                a.oh[3][g] = hy_f32_to_f16((float)vz);
                a.oh[4][g] = hy_f32_to_f16((float)pp);
            } else {
                a.oh[0][g] = hy_enc_log2s(log2f((float)tmax(U[0], a.smallr)));
                a.oh[1][g] = hy_enc_vel((float)vx);
                a.oh[2][g] = hy_enc_vel((float)vy);
                a.oh[3][g] = hy_enc_vel((float)vz);
                a.oh[4][g] = hy_enc_log2s(log2f((float)pp));
            }
        } else {             // HY_U16SP: X_new = (rho X)_new / rho_new -> log2 -> uint16 (:514-517)
#pragma unroll
            for (int v = 0; v < 5; ++v) a.o[v][g] = U[v];
            const T rinv = T(1) / tmax(U[0], a.smallr);
#pragma unroll
            for (int v = 5; v < NV; ++v) a.oh[v][g] = hy_enc_log2(log2f(fmaxf((float)(U[v] * rinv), 7.7e-34f)));
        }
    };

    T pp[2][NV];      // the lane's cells of plane k+1
    T zprev[2][NV];   // upper z states of its cells of plane k
    T Fz[2][NV];      // z fluxes through face k-1/2
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        T c[NV], q[NV];
        fetch(zoff(k0 - 2) + col[r], c);
        prim(c, q);
#pragma unroll
        for (int v = 0; v < NV; ++v) { P[k0 & 1][v][li + r * HM_LX] = q[v]; zprev[r][v] = T(1); Fz[r][v] = T(0); }
        fetch(zoff(k0 - 1) + col[r], c);
        prim(c, pp[r]);
    }

    // iterations k0-2 and k0-1 only form the z states and the face below plane k0
#pragma clang loop unroll(disable)
    for (int k = k0 - 2; k < k1; ++k) {
        T pre[2][NV], hpre[NV];   // plane k+2 of the lane's cells, plane k+1 of its halo cell
        const bool more = k + 1 >= k0 && k + 1 < k1;
#pragma unroll
        for (int r = 0; r < 2; ++r) fetch(zoff(k + 2) + col[r], pre[r]);
        if (more && halo) fetch(zoff(k + 1) + hcol, hpre);
        // plane k+1 into the buffer of plane k-1, last read before the previous barrier
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int v = 0; v < NV; ++v) P[(k + 1) & 1][v][li + r * HM_LX] = pp[r][v];

        T div[2][NV];
        if (k >= k0) {
            // ---- x: the lane's own states, its lower face; the neighbours by wave shift ----------------
            const bool seam = SV == HY_DONOR && gx % HM_SEAM_X == 0;
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                T l[NV], c[NV], n[NV], lo[NV], hi[NV], F[NV];
                lds(k, li + r * HM_LX - 1, l);
                lds(k, li + r * HM_LX, c);
                lds(k, li + r * HM_LX + 1, n);
                hy_states<T, 0, NV, SV>(l, c, n, lo, hi, a);
#pragma unroll
                for (int v = 0; v < NV; ++v) hi[v] = lane_prev(hi[v]);
                if (seam) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) { hi[v] = l[v]; lo[v] = c[v]; }
                }
                hy_riemann<T, 0, fb, NV, CMA, LG, sel>(hi, lo, F, a);
#pragma unroll
                for (int v = 0; v < NV; ++v) div[r][v] = lane_next(F[v]) - F[v];
            }
            // ---- y: rows -1 .. 2 around the lane's rows 0 and 1, three faces -----------------------------
            const bool seam0 = SV == HY_DONOR && gy0 % HM_SEAM_Y == 0, seam1 = SV == HY_DONOR && gy1 % HM_SEAM_Y == 0;
            const bool seam2 = SV == HY_DONOR && ((gy1 + 1) % a.ny) % HM_SEAM_Y == 0;
            T l[NV], c[NV], n[NV], up[NV], lo[NV], hi[NV], F0[NV], F1[NV];
            lds(k, li - 2 * HM_LX, l);
            lds(k, li - HM_LX, c);
            lds(k, li, n);
            hy_states<T, 1, NV, SV>(l, c, n, lo, up, a);
#pragma unroll
            for (int f = 0; f < 3; ++f) {   // face below row f: (c | n) with c's upper state in `up`
                T nn[NV];
                lds(k, li + (f + 1) * HM_LX, nn);
                hy_states<T, 1, NV, SV>(c, n, nn, lo, hi, a);
                if (f == 0 ? seam0 : f == 1 ? seam1 : seam2) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) { up[v] = c[v]; lo[v] = n[v]; }
                }
                hy_riemann<T, 1, fb, NV, CMA, LG, sel>(up, lo, F1, a);
                if (f > 0) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) div[f - 1][v] += F1[v] - F0[v];
                }
#pragma unroll
                for (int v = 0; v < NV; ++v) { F0[v] = F1[v]; c[v] = n[v]; n[v] = nn[v]; up[v] = hi[v]; }
            }
        }
        // ---- z: states of plane k+1, the face k+1/2, the update of plane k ---------------------------------
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            T p0[NV], pn[NV], lo[NV], hi[NV], F[NV];
            lds(k, li + r * HM_LX, p0);
            prim(pre[r], pn);
            hy_states<T, 2, NV, SV>(p0, pp[r], pn, lo, hi, a);
            hy_riemann<T, 2, fb, NV, CMA, LG, sel>(zprev[r], lo, F, a);
            if (k >= k0 && own[r]) {
#pragma unroll
                for (int v = 0; v < NV; ++v) div[r][v] += F[v] - Fz[r][v];
                store((size_t)k * plane + col[r], p0, div[r]);
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) { zprev[r][v] = hi[v]; Fz[r][v] = F[v]; pp[r][v] = pn[v]; }
        }
        if (more && halo) {
            T q[NV];
            prim(hpre, q);
#pragma unroll
            for (int v = 0; v < NV; ++v) P[(k + 1) & 1][v][hi_] = q[v];
        }
        __syncthreads();
    }
}

}  // namespace glm
