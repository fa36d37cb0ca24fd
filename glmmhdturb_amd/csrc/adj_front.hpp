// adj_front.hpp -- the front half of the reverse step: the forward march (march_impl.hpp) with its
// stages' values kept (FP64).
//
// One launch re-derives the step and leaves in the scratch what the reverse needs of it: W = c2p(u0),
// the predicted state before the revert (full predictor), the six guarded face states of every cell,
// and, where the march would update the cell, the adjoint of the state before the epilogue (LPRE).
// As four passes (c2p; predictor and face states; fluxes; divergence and epilogue adjoint) each at the
// rate of its reads and writes, the same values moved 270 planes, 99 now: 0.90 -> 0.57 ms at 128^3 (streaming stores; with
// cached ones 0.59, with one workgroup a CU 0.69).
#pragma once
#include "adjoint.hpp"
#include "adj_launch.hpp"
#include "march_impl.hpp"

namespace glm {

struct FrontArgs {
    MarchArgs<double> m;
    AdjArgs a;
};

// march_tile's stages for the reverse step; every value is stored by the lane that owns the cell.
// A: the kernel's AdjArgs.
template <typename A>
struct ReverseStages {
    static constexpr bool REVERSE = true;
    const A& a;
    double fdot;

    GLM_DEV void put(int p, int i, int j, int k, const double* x) const
    {
        size_t o = (size_t)i + (size_t)a.nx * ADJ_NPLANES * ((size_t)j + (size_t)a.ny * k);
        // opaque (c below too), or the 81 addresses are computed before the march and spilled
        asm volatile("" : "+v"(o));
        double* b = a.scr + (size_t)p * a.nx + o;
#pragma unroll
        for (int v = 0; v < 9; ++v) gstore_nt(x[v], b + (size_t)v * a.nx);   // read once, by the next kernel
    }
    GLM_DEV void prim(int i, int j, int k, const double q[9]) const { put(ADJ_W, i, j, k, q); }
    GLM_DEV void predicted(int i, int j, int k, const double mh[9]) const { put(ADJ_MH, i, j, k, mh); }
    GLM_DEV void faces(int d, int i, int j, int k, const double lo[9], const double hi[9]) const
    {
        put(ADJ_FS + fs_slot(d, 0), i, j, k, lo);
        put(ADJ_FS + fs_slot(d, 1), i, j, k, hi);
    }
    // u: the cell's state at the start of the step; acc: its flux sum
    GLM_DEV void update(const double u[9], const double acc[9], const ColdArgs<double>& ca, ForceCache<double, NO>& fc,
                        const Phys<double>& s, int i, int j, int k)
    {
        double r[9], lam[9], rb[9], a3[3] = {0.0, 0.0, 0.0}, a3b[3] = {0.0, 0.0, 0.0};
        size_t c = (size_t)i + (size_t)a.nx * ((size_t)j + (size_t)a.ny * k);
        asm volatile("" : "+v"(c));
#pragma unroll
        for (int v = 0; v < 9; ++v) {
            lam[v] = gload(a.lam1[v] + c);
            r[v] = u[v] + ca.dtdx * acc[v];
            rb[v] = 0.0;
        }
        if (ca.do_turb) force_accel(fc, ca, i, j, k, a3);
        epilogue_adj<double>(r, a3, ca.glm_fac, ca.smallc, ca.turb_min_rho, ca.dt, UpdOpts{ca.update_floor, ca.do_turb},
                             s, lam, rb, a3b);
        put(ADJ_LPRE, i, j, k, rb);
        fdot += a3b[0] * a3[0] + a3b[1] * a3[1] + a3b[2] * a3[2];
    }
};

template <int PRED, int RIEM, int RECON, int SLOPE>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2))) adj_front_kernel(FrontArgs f)
{
    __shared__ MarchLDS<double> L;
    const auto& k = kernarg_ref<FrontArgs>();
    if (threadIdx.x == 0) stage_cold(f.m, L.ca);
    __syncthreads();
    ReverseStages<decltype(k.a)> h{k.a, 0.0};
    march_tile<double, PRED, RIEM, RECON, SLOPE>(k.m, L, xcd_block((int)blockIdx.x, (int)gridDim.x), h);
    // the workgroup's sum of (kick adjoint . acceleration), in lane order
    __syncthreads();
    double* red = &L.XB[0][0];
    red[threadIdx.x] = h.fdot;
    __syncthreads();
    if (threadIdx.x < 64) {
        double s = 0.0;
        for (int t = threadIdx.x; t < NT; t += 64) s += red[t];
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
        if (threadIdx.x == 0) k.a.part[blockIdx.x] = s;
    }
}

}  // namespace glm
