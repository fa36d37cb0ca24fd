// adj_impl.hpp -- reverse (adjoint) step of the GLM-MHD march for gfx950, FP64.
//
// Given the state u0 a step started from and the adjoint lam1 of the state it produced, the
// kernels below compute lam0 = (dU1/dU0)^T lam1 for that step with its scalars (dt, ch, psi
// decay, ramp, forcing field) held fixed.  The step is re-derived in passes, one thread per cell
// (every pass is a stencil over the periodic grid):
//   1 prim    W = c2p(u0)
//   2 faces   predictor (full Hancock) and the six face states of every cell
//   3 upre    the flux through every face, each solved once (FLX), then the step's flux
//             divergence -> the pre-epilogue state and the epilogue adjoint (kick, psi decay,
//             floor): LPRE = adjoint of the pre-epilogue state
//   4 riemann per lower face: lambda_F = dtdx (LPRE(c) - LPRE(c - e_d)), Riemann adjoint ->
//             adjoints of the two face states meeting there (each slot has one writer)
//   5 cell    face-state adjoints (one launch per direction) and the predictor adjoint of every
//             cell -> contributions to the primitive adjoints of the cell and its six
//             neighbours (7 x 9 values per cell)
//   6 gather  each cell sums the contributions aimed at it, then c2p adjoint: lam0
// Every pass writes only its own cell's slots (pass 4 writes the slots of the two face states of
// one face), so there are no atomics and the result is deterministic.
#pragma once
#include "adjoint.hpp"
#include "adj_launch.hpp"

namespace glm {

GLM_DEV int adj_wrap(int i, int n)
{
    int m = i % n;
    return m < 0 ? m + n : m;
}

struct Cell {
    size_t c, o;   // index in the caller's planes and in the scratch
    int i, j, k;
};
// Scratch index: the ADJ_NPLANES values of a cell row lie together, row by row.  As planes of n cells the
// 60 to 120 streams of a pass were as many pages, and every access of a wavefront a translation of its
// own: the Riemann adjoint took 618 us at 128^3 (505 now), the reverse step as a whole 6% more.
GLM_DEV size_t adj_index(const AdjArgs& a, int i, int j, int k)
{
    return (size_t)i + (size_t)a.nx * ADJ_NPLANES * ((size_t)j + (size_t)a.ny * k);
}
GLM_DEV Cell cell_of(const AdjArgs& a, size_t c)
{
    Cell r;
    r.c = c;
    r.i = (int)(c % a.nx);
    r.j = (int)((c / a.nx) % a.ny);
    r.k = (int)(c / ((size_t)a.nx * a.ny));
    r.o = adj_index(a, r.i, r.j, r.k);
    return r;
}
// scratch index of the neighbour in direction d (0..2), offset o (-1 or +1)
GLM_DEV size_t nbr(const AdjArgs& a, const Cell& x, int d, int o)
{
    int i = x.i, j = x.j, k = x.k;
    if (d == 0) i = adj_wrap(i + o, a.nx);
    else if (d == 1) j = adj_wrap(j + o, a.ny);
    else k = adj_wrap(k + o, a.nz);
    return adj_index(a, i, j, k);
}

// plane p of the scratch; the nine planes of a group are a.nx apart
GLM_DEV double* plane(const AdjArgs& a, int p) { return a.scr + (size_t)p * a.nx; }
GLM_DEV void ld9(const AdjArgs& a, int p, size_t o, double x[9])
{
    const double* b = plane(a, p) + o;
#pragma unroll
    for (int v = 0; v < 9; ++v) x[v] = b[(size_t)v * a.nx];
}
GLM_DEV void st9(const AdjArgs& a, int p, size_t o, const double x[9])
{
    double* b = plane(a, p) + o;
#pragma unroll
    for (int v = 0; v < 9; ++v) b[(size_t)v * a.nx] = x[v];
}

// The predicted state as the face states use it: MH holds the predictor's result before the revert,
// which is what its adjoint needs.
GLM_DEV void mh_revert(const AdjArgs& a, const double p0[9], double mh[9])
{
    const bool rev = hancock_reverts(mh, a.mh_revert, a.ph);
#pragma unroll
    for (int v = 0; v < 9; ++v) mh[v] = rev ? p0[v] : mh[v];
}
// face-state slot: direction d, side 0 (low face) or 1 (high face)
GLM_DEV int fs_slot(int d, int side) { return (d * 2 + side) * 9; }

// ---- pass 1 ----------------------------------------------------------------------------------
__global__ void __launch_bounds__(ADJ_NT) adj_prim_kernel(AdjArgs a)
{
    const size_t n = (size_t)a.nx * a.ny * a.nz;
    for (size_t c = (size_t)blockIdx.x * ADJ_NT + threadIdx.x; c < n; c += (size_t)gridDim.x * ADJ_NT) {
        double u[9], w[9];
#pragma unroll
        for (int v = 0; v < 9; ++v) u[v] = a.u0[v][c];
        cons2prim(u, w, a.ph);
        st9(a, ADJ_W, cell_of(a, c).o, w);
    }
}

// PPM strong-pressure-jump flag of a cell from its pressure stencil (glmmhd_turb.jl:959)
GLM_DEV bool ppm_up(const double p0[9], const double (*nb)[9])
{
    return !(spj(nb[0][4], p0[4], nb[1][4]) || spj(nb[2][4], p0[4], nb[3][4]) || spj(nb[4][4], p0[4], nb[5][4]));
}

GLM_DEV void load_p(const AdjArgs& a, size_t o, double* out9) { ld9(a, ADJ_W, o, out9); }
GLM_DEV void load_stencil(const AdjArgs& a, const Cell& x, double p0[9], double nb[6][9])
{
    load_p(a, x.o, p0);
    for (int d = 0; d < 3; ++d) {
        load_p(a, nbr(a, x, d, -1), nb[2 * d]);
        load_p(a, nbr(a, x, d, +1), nb[2 * d + 1]);
    }
}

// ---- pass 2 ----------------------------------------------------------------------------------
template <int PRED, int RECON, int SLOPE>
__global__ void __launch_bounds__(ADJ_NT) adj_faces_kernel(AdjArgs a)
{
    const size_t n = (size_t)a.nx * a.ny * a.nz;
    const FaceOpts o{a.mh_revert, a.face_guard};
    for (size_t c = (size_t)blockIdx.x * ADJ_NT + threadIdx.x; c < n; c += (size_t)gridDim.x * ADJ_NT) {
        const Cell x = cell_of(a, c);
        double p0[9], nb[6][9], mh[9], lo[9], hi[9];
        load_stencil(a, x, p0, nb);
        const bool up = RECON == RECON_PPM ? ppm_up(p0, nb) : true;
        if (PRED == PRED_FULL) {
            hancock_fwd<double, SLOPE>(p0, nb, mh, a.half_dtdx, 0, a.ph);
            st9(a, ADJ_MH, x.o, mh);
            mh_revert(a, p0, mh);
        }
        faces_fwd<double, PRED, RECON, SLOPE, 0>(nb[0], p0, nb[1], mh, up, a.half_dtdx, o, a.ph, lo, hi);
        st9(a, ADJ_FS + fs_slot(0, 0), x.o, lo);
        st9(a, ADJ_FS + fs_slot(0, 1), x.o, hi);
        faces_fwd<double, PRED, RECON, SLOPE, 1>(nb[2], p0, nb[3], mh, up, a.half_dtdx, o, a.ph, lo, hi);
        st9(a, ADJ_FS + fs_slot(1, 0), x.o, lo);
        st9(a, ADJ_FS + fs_slot(1, 1), x.o, hi);
        faces_fwd<double, PRED, RECON, SLOPE, 2>(nb[4], p0, nb[5], mh, up, a.half_dtdx, o, a.ph, lo, hi);
        st9(a, ADJ_FS + fs_slot(2, 0), x.o, lo);
        st9(a, ADJ_FS + fs_slot(2, 1), x.o, hi);
    }
}

// Forcing acceleration at the centre of cell (i,j,k) (glmmhd_turb.jl:483-505), ramp applied.
GLM_DEV void adj_force(const AdjArgs& a, int i, int j, int k, double a3[3])
{
    const int g = a.tgs;
    const double gg = (double)g;
    const double cx = (((double)i + 0.5) * a.dx) / a.lx * gg;
    const double cy = (((double)j + 0.5) * a.dx) / a.ly * gg;
    const double cz = (((double)k + 0.5) * a.dx) / a.lz * gg;
    const double fx = floor(cx), fy = floor(cy), fz = floor(cz);
    const int i0 = (int)fx, j0 = (int)fy, k0 = (int)fz;
    const double wx = cx - fx, wy = cy - fy, wz = cz - fz;
    const int i0w = adj_wrap(i0, g), i1w = adj_wrap(i0 + 1, g), j0w = adj_wrap(j0, g), j1w = adj_wrap(j0 + 1, g);
    const int k0w = adj_wrap(k0, g), k1w = adj_wrap(k0 + 1, g);
    const size_t g3 = (size_t)g * g * g;
    for (int cc = 0; cc < 3; ++cc) {
        const double* af = a.afield + cc * g3;
        auto at = [&](int ii, int jj, int kk) { return af[(size_t)ii + (size_t)g * ((size_t)jj + (size_t)g * kk)]; };
        const double b0 = (at(i0w, j0w, k0w) * (1.0 - wx) + at(i1w, j0w, k0w) * wx) * (1.0 - wy) +
                          (at(i0w, j1w, k0w) * (1.0 - wx) + at(i1w, j1w, k0w) * wx) * wy;
        const double b1 = (at(i0w, j0w, k1w) * (1.0 - wx) + at(i1w, j0w, k1w) * wx) * (1.0 - wy) +
                          (at(i0w, j1w, k1w) * (1.0 - wx) + at(i1w, j1w, k1w) * wx) * wy;
        a3[cc] = a.ramp * (b0 * (1.0 - wz) + b1 * wz);
    }
}

template <int RIEM, int D>
GLM_DEV void face_flux(const AdjArgs& a, size_t cl, size_t cr, double f[9])
{
    double L[9], R[9];
    ld9(a, ADJ_FS + fs_slot(D, 1), cl, L);
    ld9(a, ADJ_FS + fs_slot(D, 0), cr, R);
    riemann<double, RIEM, D>(L, R, f, a.ph);
}

// ---- pass 3 ----------------------------------------------------------------------------------
// 3a: the flux through each cell's three lower faces, each face solved once -> FLX (27 planes)
template <int RIEM>
__global__ void __launch_bounds__(ADJ_NT) adj_flux_kernel(AdjArgs a)
{
    const size_t n = (size_t)a.nx * a.ny * a.nz;
    for (size_t c = (size_t)blockIdx.x * ADJ_NT + threadIdx.x; c < n; c += (size_t)gridDim.x * ADJ_NT) {
        const Cell x = cell_of(a, c);
        double f[9];
        face_flux<RIEM, 0>(a, nbr(a, x, 0, -1), x.o, f);
        st9(a, ADJ_FLX, x.o, f);
        face_flux<RIEM, 1>(a, nbr(a, x, 1, -1), x.o, f);
        st9(a, ADJ_FLX + 9, x.o, f);
        face_flux<RIEM, 2>(a, nbr(a, x, 2, -1), x.o, f);
        st9(a, ADJ_FLX + 18, x.o, f);
    }
}

// 3b: flux divergence from FLX, then the epilogue adjoint
__global__ void __launch_bounds__(ADJ_NT) adj_upre_kernel(AdjArgs a)
{
    __shared__ double red[ADJ_NT];
    const size_t n = (size_t)a.nx * a.ny * a.nz;
    const UpdOpts o{a.update_floor, a.do_turb};
    double fdot = 0.0;
    for (size_t c = (size_t)blockIdx.x * ADJ_NT + threadIdx.x; c < n; c += (size_t)gridDim.x * ADJ_NT) {
        const Cell x = cell_of(a, c);
        double acc[9], fl[9], fh[9];
        ld9(a, ADJ_FLX, x.o, fl);
        ld9(a, ADJ_FLX, nbr(a, x, 0, +1), fh);
#pragma unroll
        for (int v = 0; v < 9; ++v) acc[v] = fl[v] - fh[v];
        ld9(a, ADJ_FLX + 9, x.o, fl);
        ld9(a, ADJ_FLX + 9, nbr(a, x, 1, +1), fh);
#pragma unroll
        for (int v = 0; v < 9; ++v) acc[v] += fl[v] - fh[v];
        ld9(a, ADJ_FLX + 18, x.o, fl);
        ld9(a, ADJ_FLX + 18, nbr(a, x, 2, +1), fh);
        double r[9], lam[9], rb[9];
#pragma unroll
        for (int v = 0; v < 9; ++v) {
            acc[v] += fl[v] - fh[v];
            r[v] = a.u0[v][c] + a.dtdx * acc[v];
            lam[v] = a.lam1[v][c];
            rb[v] = 0.0;
        }
        double a3[3] = {0.0, 0.0, 0.0}, a3b[3] = {0.0, 0.0, 0.0};
        if (a.do_turb) adj_force(a, x.i, x.j, x.k, a3);
        epilogue_adj<double>(r, a3, a.glm_fac, a.smallc, a.turb_min_rho, a.dt, o, a.ph, lam, rb, a3b);
        st9(a, ADJ_LPRE, x.o, rb);
        fdot += a3b[0] * a3[0] + a3b[1] * a3[1] + a3b[2] * a3[2];
    }
    red[threadIdx.x] = fdot;
    __syncthreads();
    for (int s = ADJ_NT / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) a.part[blockIdx.x] = red[0];
}

// ---- pass 4 ----------------------------------------------------------------------------------
template <int RIEM, int D>
GLM_DEV void face_adj(const AdjArgs& a, const Cell& x)
{
    const size_t cl = nbr(a, x, D, -1), cr = x.o;
    double L[9], R[9], lr[9], ll[9], ob[9];
    ld9(a, ADJ_FS + fs_slot(D, 1), cl, L);
    ld9(a, ADJ_FS + fs_slot(D, 0), cr, R);
    ld9(a, ADJ_LPRE, cr, lr);
    ld9(a, ADJ_LPRE, cl, ll);
    double Lb[9], Rb[9];
#pragma unroll
    for (int v = 0; v < 9; ++v) {
        ob[v] = a.dtdx * (lr[v] - ll[v]);
        Lb[v] = 0.0;
        Rb[v] = 0.0;
    }
    riemann_adj<double, RIEM, D>(L, R, ob, Lb, Rb, a.ph);
    st9(a, ADJ_LFS + fs_slot(D, 1), cl, Lb);
    st9(a, ADJ_LFS + fs_slot(D, 0), cr, Rb);
}
template <int RIEM>
__global__ void __launch_bounds__(ADJ_NT) adj_riemann_kernel(AdjArgs a)
{
    const size_t n = (size_t)a.nx * a.ny * a.nz;
    for (size_t c = (size_t)blockIdx.x * ADJ_NT + threadIdx.x; c < n; c += (size_t)gridDim.x * ADJ_NT) {
        const Cell x = cell_of(a, c);
        face_adj<RIEM, 0>(a, x);
        face_adj<RIEM, 1>(a, x);
        face_adj<RIEM, 2>(a, x);
    }
}

// ---- pass 5 ----------------------------------------------------------------------------------
// CON slot k of a cell: 0 the cell itself, 1 + 2d its -d neighbour, 2 + 2d its +d neighbour.
// 5d (one launch per direction D): face-state adjoints of the cell's two faces in D -> slots
// 1 + 2D and 2 + 2D, plus the cell's own slot 0 and the predictor adjoint MHB (the D = 0 launch
// stores, the others add).  5h (full predictor): the predictor adjoint -> slots 0..6 (added).
// One direction per launch keeps each thread's live set small.
template <int PRED, int RECON, int SLOPE, int D>
__global__ void __launch_bounds__(ADJ_NT) adj_cell_dir_kernel(AdjArgs a)
{
    const size_t n = (size_t)a.nx * a.ny * a.nz;
    const FaceOpts o{a.mh_revert, a.face_guard};
    for (size_t c = (size_t)blockIdx.x * ADJ_NT + threadIdx.x; c < n; c += (size_t)gridDim.x * ADJ_NT) {
        const Cell x = cell_of(a, c);
        double p0[9], l[9], r[9], mh[9], lob[9], hib[9], lb[9], m0b[9], rb[9], mhb[9];
        load_p(a, x.o, p0);
        load_p(a, nbr(a, x, D, -1), l);
        load_p(a, nbr(a, x, D, +1), r);
        bool up = true;
        if (RECON == RECON_PPM) {
            const double* P = plane(a, ADJ_W + 4);
            double pr[6];
            for (int d = 0; d < 3; ++d) {
                pr[2 * d] = P[nbr(a, x, d, -1)];
                pr[2 * d + 1] = P[nbr(a, x, d, +1)];
            }
            up = !(spj(pr[0], p0[4], pr[1]) || spj(pr[2], p0[4], pr[3]) || spj(pr[4], p0[4], pr[5]));
        }
        if (PRED == PRED_FULL) {
            ld9(a, ADJ_MH, x.o, mh);
            mh_revert(a, p0, mh);
        } else for (int v = 0; v < 9; ++v) mh[v] = 0.0;
        ld9(a, ADJ_LFS + fs_slot(D, 0), x.o, lob);
        ld9(a, ADJ_LFS + fs_slot(D, 1), x.o, hib);
        for (int v = 0; v < 9; ++v) { lb[v] = 0.0; m0b[v] = 0.0; rb[v] = 0.0; mhb[v] = 0.0; }
        faces_adj<double, PRED, RECON, SLOPE, D>(l, p0, r, mh, up, a.half_dtdx, o, a.ph, lob, hib, lb, m0b, rb, mhb);
        st9(a, ADJ_CON + (1 + 2 * D) * 9, x.o, lb);
        st9(a, ADJ_CON + (2 + 2 * D) * 9, x.o, rb);
        if (D > 0) {
            double t[9];
            ld9(a, ADJ_CON, x.o, t);
            for (int v = 0; v < 9; ++v) m0b[v] += t[v];
            if (PRED == PRED_FULL) {
                ld9(a, ADJ_MHB, x.o, t);
                for (int v = 0; v < 9; ++v) mhb[v] += t[v];
            }
        }
        st9(a, ADJ_CON, x.o, m0b);
        if (PRED == PRED_FULL) st9(a, ADJ_MHB, x.o, mhb);
    }
}

template <int SLOPE, int D>
GLM_DEV void hancock_dir_add(const AdjArgs& a, const Cell& x, const double p0[9], const double accb[9],
                             double p0b[9])
{
    double l[9], r[9], lb[9], rb[9], t[9];
    const size_t cl = nbr(a, x, D, -1), cr = nbr(a, x, D, +1);
    load_p(a, cl, l);
    load_p(a, cr, r);
    for (int v = 0; v < 9; ++v) { lb[v] = 0.0; rb[v] = 0.0; }
    hancock_adj_dir<double, SLOPE, D>(p0, l, r, accb, p0b, lb, rb, a.ph);
    ld9(a, ADJ_CON + (1 + 2 * D) * 9, x.o, t);
    for (int v = 0; v < 9; ++v) t[v] += lb[v];
    st9(a, ADJ_CON + (1 + 2 * D) * 9, x.o, t);
    ld9(a, ADJ_CON + (2 + 2 * D) * 9, x.o, t);
    for (int v = 0; v < 9; ++v) t[v] += rb[v];
    st9(a, ADJ_CON + (2 + 2 * D) * 9, x.o, t);
}
template <int SLOPE>
__global__ void __launch_bounds__(ADJ_NT) adj_hancock_kernel(AdjArgs a)
{
    const size_t n = (size_t)a.nx * a.ny * a.nz;
    for (size_t c = (size_t)blockIdx.x * ADJ_NT + threadIdx.x; c < n; c += (size_t)gridDim.x * ADJ_NT) {
        const Cell x = cell_of(a, c);
        double p0[9], mh[9], mhb[9], p0b[9], accb[9];
        load_p(a, x.o, p0);
        ld9(a, ADJ_MHB, x.o, mhb);
        ld9(a, ADJ_MH, x.o, mh);
        for (int v = 0; v < 9; ++v) p0b[v] = 0.0;
        if (hancock_adj_core(p0, mh, mhb, p0b, accb, a.half_dtdx, a.mh_revert, a.ph)) {
            hancock_dir_add<SLOPE, 0>(a, x, p0, accb, p0b);
            hancock_dir_add<SLOPE, 1>(a, x, p0, accb, p0b);
            hancock_dir_add<SLOPE, 2>(a, x, p0, accb, p0b);
        }
        double t[9];
        ld9(a, ADJ_CON, x.o, t);
        for (int v = 0; v < 9; ++v) t[v] += p0b[v];
        st9(a, ADJ_CON, x.o, t);
    }
}

// ---- pass 6 ----------------------------------------------------------------------------------
__global__ void __launch_bounds__(ADJ_NT) adj_gather_kernel(AdjArgs a)
{
    const size_t n = (size_t)a.nx * a.ny * a.nz;
    for (size_t c = (size_t)blockIdx.x * ADJ_NT + threadIdx.x; c < n; c += (size_t)gridDim.x * ADJ_NT) {
        const Cell x = cell_of(a, c);
        double wb[9], t[9], w[9], lb[9];
        ld9(a, ADJ_CON, x.o, wb);
        for (int d = 0; d < 3; ++d) {
            // the -d neighbour's +d contribution and the +d neighbour's -d contribution aim at c
            ld9(a, ADJ_CON + (2 + 2 * d) * 9, nbr(a, x, d, -1), t);
            for (int v = 0; v < 9; ++v) wb[v] += t[v];
            ld9(a, ADJ_CON + (1 + 2 * d) * 9, nbr(a, x, d, +1), t);
            for (int v = 0; v < 9; ++v) wb[v] += t[v];
        }
        load_p(a, x.o, w);
        ld9(a, ADJ_LPRE, x.o, lb);
        cons2prim_adj_q(w, wb, lb, a.ph);
#pragma unroll
        for (int v = 0; v < 9; ++v) a.lam0[v][c] = lb[v];
    }
}

// Sum of the per-block partials of pass 3, added to *acc.  One block: thread t sums partials
// t, t + 256, ... in order, then a fixed tree; deterministic for a given grid.
__global__ void __launch_bounds__(ADJ_NT) adj_fdot_kernel(const double* part, int nparts, double* acc)
{
    __shared__ double red[ADJ_NT];
    double s = 0.0;
    for (int b = threadIdx.x; b < nparts; b += ADJ_NT) s += part[b];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = ADJ_NT / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *acc += red[0];
}

}  // namespace glm
