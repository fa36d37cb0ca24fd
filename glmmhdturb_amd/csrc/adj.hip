// adj.hip -- launches of the reverse step (adj_impl.hpp).
#include "adj_impl.hpp"
#include "adj_march.hpp"
#include "launch.hpp"

#include <cstring>

namespace glm {

constexpr unsigned ADJ_GRID_MAX = 2048;

static unsigned adj_grid(size_t n)
{
    size_t g = (n + ADJ_NT - 1) / ADJ_NT;
    return (unsigned)(g < ADJ_GRID_MAX ? (g > 0 ? g : 1) : ADJ_GRID_MAX);
}

size_t adj_scratch_bytes(size_t n) { return (size_t)(ADJ_NPLANES + 1) * n * sizeof(double); }

static const void* front_ptr(int pred, int riem, int recon, int slope)
{
#define GLM_CASE(P, R) if (pred == P && riem == R) return adj_front_ptr_pr<P, R>(recon, slope);
    GLM_CASE(PRED_FULL, RIEM_LLF) GLM_CASE(PRED_FULL, RIEM_LLFB) GLM_CASE(PRED_FULL, RIEM_HLL) GLM_CASE(PRED_FULL, RIEM_HLLD)
    GLM_CASE(PRED_ONED, RIEM_LLF) GLM_CASE(PRED_ONED, RIEM_LLFB) GLM_CASE(PRED_ONED, RIEM_HLL) GLM_CASE(PRED_ONED, RIEM_HLLD)
#undef GLM_CASE
    return nullptr;
}

// Passes 1-3 as one march; nparts: the workgroups, each with a partial sum in a.part.
static hipError_t dispatch_front(const AdjArgs& a, const AdjResident& r, int zchunk, hipStream_t st, int pred, int riem,
                                 int recon, int slope, int& nparts)
{
    MarchArgs<double> m;
    memset(&m, 0, sizeof m);
    for (int v = 0; v < 9; ++v) m.q[v] = a.u0[v];
    m.nx = a.nx; m.ny = a.ny; m.nz = a.nz;
    march_tiling<double>(a.nx, a.ny, a.nz, zchunk > 0 ? zchunk : r.zfront, r.front, m.tiles_x, m.tiles_y, m.nzc, m.zchunk);
    m.ph = a.ph;
    m.dtdx = a.dtdx; m.half_dtdx = a.half_dtdx; m.glm_fac = a.glm_fac;
    m.smallc = a.smallc; m.turb_min_rho = a.turb_min_rho; m.ramp = a.ramp; m.dt = a.dt;
    m.dx = a.dx; m.lx = a.lx; m.ly = a.ly; m.lz = a.lz;
    m.recon = recon; m.slope = slope;
    m.mh_revert = a.mh_revert; m.face_guard = a.face_guard; m.update_floor = a.update_floor;
    m.do_turb = a.do_turb; m.tgs = a.tgs; m.afield = a.afield;
    nparts = m.tiles_x * m.tiles_y * m.nzc;
#define GLM_CASE(P, R) if (pred == P && riem == R) return launch_adj_front_pr<P, R>(m, a, recon, slope, st);
    GLM_CASE(PRED_FULL, RIEM_LLF) GLM_CASE(PRED_FULL, RIEM_LLFB) GLM_CASE(PRED_FULL, RIEM_HLL) GLM_CASE(PRED_FULL, RIEM_HLLD)
    GLM_CASE(PRED_ONED, RIEM_LLF) GLM_CASE(PRED_ONED, RIEM_LLFB) GLM_CASE(PRED_ONED, RIEM_HLL) GLM_CASE(PRED_ONED, RIEM_HLLD)
#undef GLM_CASE
    return hipErrorInvalidValue;
}

template <int PRED, int RECON, int SLOPE>
static void launch_cellwise(const AdjArgs& a, dim3 g, hipStream_t st)
{
    hipLaunchKernelGGL((adj_cell_dir_kernel<PRED, RECON, SLOPE, 0>), g, dim3(ADJ_NT), 0, st, a);
    hipLaunchKernelGGL((adj_cell_dir_kernel<PRED, RECON, SLOPE, 1>), g, dim3(ADJ_NT), 0, st, a);
    hipLaunchKernelGGL((adj_cell_dir_kernel<PRED, RECON, SLOPE, 2>), g, dim3(ADJ_NT), 0, st, a);
    if (PRED == PRED_FULL) hipLaunchKernelGGL((adj_hancock_kernel<SLOPE>), g, dim3(ADJ_NT), 0, st, a);
}

static void dispatch_cellwise(const AdjArgs& a, dim3 g, hipStream_t st, int pred, int recon, int slope)
{
#define GLM_CASE(P, RC, SL)                                          \
    if (pred == P && recon == RC && slope == SL) launch_cellwise<P, RC, SL>(a, g, st);
    GLM_CASE(PRED_FULL, RECON_PLM, SLOPE_MONCEN) GLM_CASE(PRED_FULL, RECON_PLM, SLOPE_MINMOD)
    GLM_CASE(PRED_FULL, RECON_PPM, SLOPE_MONCEN) GLM_CASE(PRED_FULL, RECON_PPM, SLOPE_MINMOD)
    GLM_CASE(PRED_ONED, RECON_PLM, SLOPE_MONCEN) GLM_CASE(PRED_ONED, RECON_PLM, SLOPE_MINMOD)
    GLM_CASE(PRED_ONED, RECON_PPM, SLOPE_MONCEN) GLM_CASE(PRED_ONED, RECON_PPM, SLOPE_MINMOD)
#undef GLM_CASE
}

// HLLD: the grid is what is resident (one workgroup a CU) and each walks its share of the cells (adj_riemann_kernel).
static void dispatch_riemann(const AdjArgs& a, const AdjResident& r, dim3 g, hipStream_t st, int riem)
{
    const unsigned most = (unsigned)(r.hlld.cus * r.hlld.occ);
    if (riem == RIEM_HLLD && g.x > most) g.x = most;
#define GLM_CASE(R) \
    if (riem == R) hipLaunchKernelGGL((adj_riemann_kernel<R>), g, dim3(ADJ_NT), 0, st, a);
    GLM_CASE(RIEM_LLF) GLM_CASE(RIEM_LLFB) GLM_CASE(RIEM_HLL) GLM_CASE(RIEM_HLLD)
#undef GLM_CASE
}

static const void* back_ptr(int pred, int recon, int slope)
{
#define GLM_CASE(P, RC, SL) if (pred == P && recon == RC && slope == SL) return (const void*)&adj_back_kernel<P, RC, SL>;
    GLM_CASE(PRED_FULL, RECON_PLM, SLOPE_MONCEN) GLM_CASE(PRED_FULL, RECON_PLM, SLOPE_MINMOD)
    GLM_CASE(PRED_FULL, RECON_PPM, SLOPE_MONCEN) GLM_CASE(PRED_FULL, RECON_PPM, SLOPE_MINMOD)
    GLM_CASE(PRED_ONED, RECON_PLM, SLOPE_MONCEN) GLM_CASE(PRED_ONED, RECON_PLM, SLOPE_MINMOD)
    GLM_CASE(PRED_ONED, RECON_PPM, SLOPE_MONCEN) GLM_CASE(PRED_ONED, RECON_PPM, SLOPE_MINMOD)
#undef GLM_CASE
    return nullptr;
}

static void dispatch_back(const AdjArgs& a, const AdjResident& r, int zchunk, hipStream_t st, int pred, int recon, int slope)
{
    int tx, ty, nzc, zc;
    march_tiling<double>(a.nx, a.ny, a.nz, zchunk > 0 ? zchunk : r.zback, r.back, tx, ty, nzc, zc);
    const dim3 g((unsigned)(tx * ty * nzc));
#define GLM_CASE(P, RC, SL)                                                                          \
    if (pred == P && recon == RC && slope == SL)                                                     \
        hipLaunchKernelGGL((adj_back_kernel<P, RC, SL>), g, dim3(NT), 0, st, a, tx, ty, zc);
    GLM_CASE(PRED_FULL, RECON_PLM, SLOPE_MONCEN) GLM_CASE(PRED_FULL, RECON_PLM, SLOPE_MINMOD)
    GLM_CASE(PRED_FULL, RECON_PPM, SLOPE_MONCEN) GLM_CASE(PRED_FULL, RECON_PPM, SLOPE_MINMOD)
    GLM_CASE(PRED_ONED, RECON_PLM, SLOPE_MONCEN) GLM_CASE(PRED_ONED, RECON_PLM, SLOPE_MINMOD)
    GLM_CASE(PRED_ONED, RECON_PPM, SLOPE_MONCEN) GLM_CASE(PRED_ONED, RECON_PPM, SLOPE_MINMOD)
#undef GLM_CASE
}

static hipError_t resident(const void* fn, int threads, Resident& r)
{
    int dev = 0;
    r.occ = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&r.cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&r.occ, fn, threads, 0);
    if (r.occ < 1) r.occ = 1;
    return e;
}

hipError_t adj_resident(int nx, int ny, int nz, int pred, int riem, int recon, int slope, AdjResident& out)
{
    const void *front = front_ptr(pred, riem, recon, slope), *back = back_ptr(pred, recon, slope);
    if (!front || !back) return hipErrorInvalidValue;
    hipError_t e = resident(front, NT, out.front);
    if (e == hipSuccess) e = resident(back, NT, out.back);
    if (e == hipSuccess) e = resident((const void*)&adj_riemann_kernel<RIEM_HLLD>, ADJ_NT, out.hlld);
    int tx, ty, nzc;
    march_tiling<double>(nx, ny, nz, 0, out.front, tx, ty, nzc, out.zfront);
    march_tiling<double>(nx, ny, nz, 0, out.back, tx, ty, nzc, out.zback);
    return e;
}

hipError_t launch_step_adjoint(AdjArgs a, const AdjResident& r, void* scratch, int pred, int riem, int recon,
                               int slope, double* fdot, bool fused, int zchunk, hipStream_t st)
{
    if (recon == RECON_PPM_SPIKE) return hipErrorInvalidValue;
    const size_t n = (size_t)a.nx * a.ny * a.nz;
    a.scr = (double*)scratch;
    a.part = a.scr + (size_t)ADJ_NPLANES * n;
    const dim3 g(adj_grid(n));
    int nparts = 0;
    const hipError_t e = dispatch_front(a, r, zchunk, st, pred, riem, recon, slope, nparts);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(adj_fdot_kernel, dim3(1), dim3(ADJ_NT), 0, st, (const double*)a.part, nparts, fdot);
    dispatch_riemann(a, r, g, st, riem);
    // the march's 32-bit offsets reach over one z plane of the scratch (2.59 million cells)
    if (fused && (size_t)ADJ_NPLANES * sizeof(double) * a.nx * a.ny <= UINT32_MAX) {
        dispatch_back(a, r, zchunk, st, pred, recon, slope);
    } else {
        dispatch_cellwise(a, g, st, pred, recon, slope);
        hipLaunchKernelGGL(adj_gather_kernel, g, dim3(ADJ_NT), 0, st, a);
    }
    return hipGetLastError();
}

}  // namespace glm
