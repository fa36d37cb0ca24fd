// adj_front_inst.hip -- one family of the reverse step's front kernels: predictor GLM_PRED, Riemann
// solver GLM_RIEM (set by the build), the reconstructions and limiters that have an adjoint.
#include "adj_front.hpp"

#ifndef GLM_PRED
#error "build with -DGLM_PRED=0|1 -DGLM_RIEM=0..3"
#endif

namespace glm {

template <>
hipError_t launch_adj_front_pr<GLM_PRED, GLM_RIEM>(const MarchArgs<double>& m, const AdjArgs& a, int recon, int slope,
                                                   hipStream_t st)
{
    const FrontArgs f{m, a};
    const dim3 grid((unsigned)(m.tiles_x * m.tiles_y * m.nzc));
#define GLM_CASE(RC, SL)                                                                               \
    if (recon == RC && slope == SL) {                                                                  \
        hipLaunchKernelGGL((adj_front_kernel<GLM_PRED, GLM_RIEM, RC, SL>), grid, dim3(NT), 0, st, f); \
        return hipGetLastError();                                                                      \
    }
    GLM_CASE(RECON_PLM, SLOPE_MONCEN) GLM_CASE(RECON_PPM, SLOPE_MONCEN)
    GLM_CASE(RECON_PLM, SLOPE_MINMOD) GLM_CASE(RECON_PPM, SLOPE_MINMOD)
#undef GLM_CASE
    return hipErrorInvalidValue;
}

template <>
const void* adj_front_ptr_pr<GLM_PRED, GLM_RIEM>(int recon, int slope)
{
#define GLM_CASE(RC, SL) \
    if (recon == RC && slope == SL) return (const void*)&adj_front_kernel<GLM_PRED, GLM_RIEM, RC, SL>;
    GLM_CASE(RECON_PLM, SLOPE_MONCEN) GLM_CASE(RECON_PPM, SLOPE_MONCEN)
    GLM_CASE(RECON_PLM, SLOPE_MINMOD) GLM_CASE(RECON_PPM, SLOPE_MINMOD)
#undef GLM_CASE
    return nullptr;
}

}  // namespace glm
