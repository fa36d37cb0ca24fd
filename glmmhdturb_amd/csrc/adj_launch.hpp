// adj_launch.hpp -- host side of the reverse step (adj.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "physics.hpp"
#include "tiling.hpp"

namespace glm {

constexpr int ADJ_NT = 256;

// Scratch planes of the reverse step (n doubles each, interleaved row by row: adj_impl.hpp adj_index).
constexpr int ADJ_W = 0, ADJ_MH = 9, ADJ_FS = 18, ADJ_LPRE = 72, ADJ_LFS = 81, ADJ_CON = 135, ADJ_MHB = 198,
              ADJ_NPLANES = 207;

// face-state slot: direction d, side 0 (low face) or 1 (high face)
__host__ __device__ constexpr int fs_slot(int d, int side) { return (d * 2 + side) * 9; }

struct AdjArgs {
    const double* u0[9];
    const double* lam1[9];
    double* lam0[9];
    int nx, ny, nz, tgs;
    Phys<double> ph;
    double dtdx, half_dtdx, glm_fac, smallc, turb_min_rho, ramp, dt, dx, lx, ly, lz;
    int mh_revert, face_guard, update_floor, do_turb;
    const double* afield;   // 3 planes of tgs^3 (the step's forcing field), or null
    double* scr;            // ADJ_NPLANES planes of n
    double* part;           // per-workgroup partial sums of a_bar . a (front half)
};


// Device scratch of one reverse step over n cells, in bytes (ADJ_NPLANES planes plus the
// front half's partial sums: its workgroups are at most as many as the cells).
size_t adj_scratch_bytes(size_t n);
template <typename T>
struct MarchArgs;
// One (predictor, Riemann) family of front kernels (adj_front.hpp), built from adj_front_inst.hip.
template <int PRED, int RIEM>
hipError_t launch_adj_front_pr(const MarchArgs<double>& m, const AdjArgs& a, int recon, int slope, hipStream_t st);
template <int PRED, int RIEM>
const void* adj_front_ptr_pr(int recon, int slope);   // the kernel (occupancy queries)

// Concurrent workgroups of a scheme's reverse kernels on the present device (the front half, the back half,
// the HLLD adjoint) and the modelled chunk lengths of the two marches on a grid.
struct AdjResident {
    Resident front, back, hlld;
    int zfront, zback;
};
hipError_t adj_resident(int nx, int ny, int nz, int pred, int riem, int recon, int slope, AdjResident& out);

// Launch the reverse step and add the step's sum of (kick acceleration adjoint . acceleration)
// to *fdot (device).  With fused, the face-state and predictor adjoints and the gather run as one
// z-march kernel (adj_march.hpp, z planes per tile: zchunk, 0 = the occupancy model) where a z plane
// of the scratch is below 4 GiB; otherwise as the separate passes 5 and 6.  a.scr and a.part must come
// from a scratch of adj_scratch_bytes(n).  Returns hipErrorInvalidValue for an unsupported scheme.
hipError_t launch_step_adjoint(AdjArgs a, const AdjResident& r, void* scratch, int pred, int riem, int recon,
                               int slope, double* fdot, bool fused, int zchunk, hipStream_t st);

}  // namespace glm
