// adj_impl.hpp -- reverse (adjoint) step of the GLM-MHD march for gfx950, FP64.
//
// Given the state u0 a step started from and the adjoint lam1 of the state it produced, the
// kernels below compute lam0 = (dU1/dU0)^T lam1 for that step with its scalars (dt, ch, psi
// decay, ramp, forcing field) held fixed.  The step is re-derived in passes over the periodic grid:
//   1-3 front (adj_front.hpp, a z-march): W = c2p(u0), the predicted state, the six face states of
//             every cell; the step's flux divergence -> the pre-epilogue state and the epilogue
//             adjoint (kick, psi decay, floor): LPRE = adjoint of the pre-epilogue state
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
// own: at 128^3 the Riemann adjoint took 618 us instead of 505 (before its loads were requested ahead), the reverse step
// as a whole 6% more.
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
GLM_DEV void load_p(const AdjArgs& a, size_t o, double* out9) { ld9(a, ADJ_W, o, out9); }

// ---- pass 4 ----------------------------------------------------------------------------------
// One thread a cell and its three lower faces.  The HLLD adjoint takes some 390 registers, so a SIMD
// has one wavefront and nothing hides its loads: there a face's values are requested while the
// face before is solved, the next cell's first face with the last, and the grid is what is resident, so
// that nearly every cell has a cell before it (dispatch_riemann).  At 128^3 0.48 -> 0.40 ms, the rate of its
// reads and writes (with 2048 workgroups 0.44).  The other solvers run two wavefronts a SIMD and lose the
// second to the registers this takes (same time at 128^3, 4% of the reverse step at 64^3).
struct FaceIn {
    double L[9], R[9], ll[9];   // the states meeting at the face; LPRE of the cell below it
};
template <int D>
GLM_DEV void face_load(const AdjArgs& a, const Cell& x, FaceIn& f)
{
    const size_t cl = nbr(a, x, D, -1);
    ld9(a, ADJ_FS + fs_slot(D, 1), cl, f.L);
    ld9(a, ADJ_FS + fs_slot(D, 0), x.o, f.R);
    ld9(a, ADJ_LPRE, cl, f.ll);
    __builtin_amdgcn_sched_barrier(0);
}
template <int RIEM, int D>
GLM_DEV void face_adj(const AdjArgs& a, const Cell& x, const FaceIn& f, const double lr[9])
{
    double ob[9], Lb[9], Rb[9];
#pragma unroll
    for (int v = 0; v < 9; ++v) {
        ob[v] = a.dtdx * (lr[v] - f.ll[v]);
        Lb[v] = 0.0;
        Rb[v] = 0.0;
    }
    riemann_adj<double, RIEM, D>(f.L, f.R, ob, Lb, Rb, a.ph);
    st9(a, ADJ_LFS + fs_slot(D, 1), nbr(a, x, D, -1), Lb);
    st9(a, ADJ_LFS + fs_slot(D, 0), x.o, Rb);
}
template <int RIEM, int D>
GLM_DEV void face_here(const AdjArgs& a, const Cell& x)
{
    FaceIn f;
    double lr[9];
    face_load<D>(a, x, f);
    ld9(a, ADJ_LPRE, x.o, lr);
    face_adj<RIEM, D>(a, x, f, lr);
}
template <int RIEM>
__global__ void __launch_bounds__(ADJ_NT) adj_riemann_kernel(AdjArgs a)
{
    const size_t n = (size_t)a.nx * a.ny * a.nz, step = (size_t)gridDim.x * ADJ_NT;
    size_t c = (size_t)blockIdx.x * ADJ_NT + threadIdx.x;
    if (RIEM != RIEM_HLLD) {
        for (; c < n; c += step) {
            const Cell x = cell_of(a, c);
            face_here<RIEM, 0>(a, x);
            face_here<RIEM, 1>(a, x);
            face_here<RIEM, 2>(a, x);
        }
        return;
    }
    if (c >= n) return;
    Cell x = cell_of(a, c);
    FaceIn f, g;
    double lr[9], ln[9];
    face_load<0>(a, x, f);
    ld9(a, ADJ_LPRE, x.o, lr);
    for (;;) {
        c += step;
        const bool more = c < n;
        const Cell y = cell_of(a, more ? c : 0);
        face_load<1>(a, x, g);
        face_adj<RIEM, 0>(a, x, f, lr);
        face_load<2>(a, x, f);
        face_adj<RIEM, 1>(a, x, g, lr);
        if (more) {
            face_load<0>(a, y, g);
            ld9(a, ADJ_LPRE, y.o, ln);
        }
        face_adj<RIEM, 2>(a, x, f, lr);
        if (!more) break;
        x = y;
        f = g;
        for (int v = 0; v < 9; ++v) lr[v] = ln[v];
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

// Sum of the front half's per-workgroup partials, added to *acc.  One block: thread t sums partials
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
