// launch.hpp -- host-side launchers of the gfx950 kernels (defined in march_f64.hip,
// march_f32.hip, aux.hip, ct.hip) used by the C-ABI in capi.hip.
#pragma once
#include <hip/hip_runtime.h>
#include "march_impl.hpp"
#include "tiling.hpp"

namespace glm {

// One (precision, predictor, Riemann) family of march kernels; the 3 reconstructions x 2 limiters
// of a family are instantiated in one object built from march_inst.hip.
template <typename T, int PRED, int RIEM>
hipError_t launch_march_pr(const MarchArgs<T>& a, int recon, int slope, hipStream_t st);
template <typename T, int PRED, int RIEM>
const void* march_kernel_ptr_pr(int recon, int slope);
template <typename T, int PRED, int RIEM>
hipError_t launch_march_pr_sp(const MarchArgs<T>& a, int recon, int slope, hipStream_t st);
template <typename T, int PRED, int RIEM>
const void* march_kernel_ptr_pr_sp(int recon, int slope);
template <typename T, int PRED, int RIEM>
hipError_t launch_ens_pr(const EnsLaunch<T>& e, int recon, int slope, int grid, hipStream_t st);
template <typename T, int PRED, int RIEM>
const void* ens_kernel_ptr_pr(int recon, int slope);
// The march's memory floor (march_floor_kernel; built in the full-predictor HLLD object).
template <typename T>
hipError_t launch_march_floor(const MarchArgs<T>& a, hipStream_t st);
template <typename T>
const void* march_floor_ptr();

// nsp = 0: the 9-plane march; nsp = 2: with two passive species (11 planes).
template <typename T>
inline hipError_t launch_march(const MarchArgs<T>& a, int pred, int riem, int recon, int slope, hipStream_t st,
                               int nsp = 0)
{
#define GLM_CASE(P, R) \
    if (pred == P && riem == R) \
        return nsp ? launch_march_pr_sp<T, P, R>(a, recon, slope, st) : launch_march_pr<T, P, R>(a, recon, slope, st);
    GLM_CASE(PRED_FULL, RIEM_LLF) GLM_CASE(PRED_FULL, RIEM_LLFB) GLM_CASE(PRED_FULL, RIEM_HLL) GLM_CASE(PRED_FULL, RIEM_HLLD)
    GLM_CASE(PRED_ONED, RIEM_LLF) GLM_CASE(PRED_ONED, RIEM_LLFB) GLM_CASE(PRED_ONED, RIEM_HLL) GLM_CASE(PRED_ONED, RIEM_HLLD)
#undef GLM_CASE
    return hipErrorInvalidValue;
}

// Kernel symbol of one march variant (for resource queries); nullptr if unknown.
template <typename T>
inline const void* march_kernel_ptr(int pred, int riem, int recon, int slope, int nsp = 0)
{
#define GLM_CASE(P, R) \
    if (pred == P && riem == R) \
        return nsp ? march_kernel_ptr_pr_sp<T, P, R>(recon, slope) : march_kernel_ptr_pr<T, P, R>(recon, slope);
    GLM_CASE(PRED_FULL, RIEM_LLF) GLM_CASE(PRED_FULL, RIEM_LLFB) GLM_CASE(PRED_FULL, RIEM_HLL) GLM_CASE(PRED_FULL, RIEM_HLLD)
    GLM_CASE(PRED_ONED, RIEM_LLF) GLM_CASE(PRED_ONED, RIEM_LLFB) GLM_CASE(PRED_ONED, RIEM_HLL) GLM_CASE(PRED_ONED, RIEM_HLLD)
#undef GLM_CASE
    return nullptr;
}

template <typename T>
inline hipError_t launch_ens(const EnsLaunch<T>& e, int pred, int riem, int recon, int slope, int grid, hipStream_t st)
{
#define GLM_CASE(P, R) \
    if (pred == P && riem == R) return launch_ens_pr<T, P, R>(e, recon, slope, grid, st);
    GLM_CASE(PRED_FULL, RIEM_LLF) GLM_CASE(PRED_FULL, RIEM_LLFB) GLM_CASE(PRED_FULL, RIEM_HLL) GLM_CASE(PRED_FULL, RIEM_HLLD)
    GLM_CASE(PRED_ONED, RIEM_LLF) GLM_CASE(PRED_ONED, RIEM_LLFB) GLM_CASE(PRED_ONED, RIEM_HLL) GLM_CASE(PRED_ONED, RIEM_HLLD)
#undef GLM_CASE
    return hipErrorInvalidValue;
}

template <typename T>
inline const void* ens_kernel_ptr(int pred, int riem, int recon, int slope)
{
#define GLM_CASE(P, R) \
    if (pred == P && riem == R) return ens_kernel_ptr_pr<T, P, R>(recon, slope);
    GLM_CASE(PRED_FULL, RIEM_LLF) GLM_CASE(PRED_FULL, RIEM_LLFB) GLM_CASE(PRED_FULL, RIEM_HLL) GLM_CASE(PRED_FULL, RIEM_HLLD)
    GLM_CASE(PRED_ONED, RIEM_LLF) GLM_CASE(PRED_ONED, RIEM_LLFB) GLM_CASE(PRED_ONED, RIEM_HLL) GLM_CASE(PRED_ONED, RIEM_HLLD)
#undef GLM_CASE
    return nullptr;
}

// Workgroup tiling of the march for an (nx, ny, nz) grid.  A chunk costs about 1.3 planes besides its
// own: the window's first planes, the lead-in plane's predictor and the face above the last plane.
// share: the FP64 PPM + HLLD march 0.55, FP32 marches (four resident) 0.29-0.34.
constexpr double MARCH_LEAD = 1.3;
inline double march_share(int prec) { return prec == 8 ? 0.55 : 0.32; }
template <typename T>
inline void march_tiling(int nx, int ny, int nz, int zchunk_req, const Resident& r, int& tiles_x, int& tiles_y, int& nzc,
                         int& zchunk)
{
    march_tiles(nx, ny, nz, OX, OY, zchunk_req, r, MARCH_LEAD, march_share((int)sizeof(T)), tiles_x, tiles_y, nzc, zchunk);
}

}  // namespace glm
