// adj_march.hpp -- the back half of the reverse step as one z-march kernel (FP64).
//
// It replaces passes 5 and 6 of adj_impl.hpp (the face-state and predictor adjoints of every cell,
// their contributions to the primitive adjoints of the cell and its six neighbours, the gather and
// the c2p adjoint) with one pass that keeps those contributions on chip instead of writing and
// re-reading 63 + 9 contribution planes.  Inputs are the planes the front passes wrote: W = c2p(u0),
// the predicted states MH, the face-state adjoints LFS and LPRE; the output is lam0.
//
// Layout: the forward march's tile (march_impl.hpp): 252 lanes, a 16 x 12 owned tile and its
// one-cell ring, each lane one column, marching z; W of plane q over the tile grown by two cells in
// LDS.  Per plane q every lane takes the face-state adjoints of its cell in x, y, z and then the
// predictor adjoint in x, y, z.  The contributions to in-plane neighbours change hands through LDS
// after each direction, the one to the cell below finishes plane q-1, the one to the cell above
// starts plane q+1.
//
// What bounds it: 3300 FP64 instructions and 300 LDS accesses a lane and plane in a chain of eight
// exchanges.  One workgroup a CU with everything in 512 registers left the chain's latencies bare
// (VALU busy 24%, 224 B spilled, 1.64 ms at 128^3).  Two workgroups need 256 registers and 80 KiB of
// LDS each: so the variables of a stage are finished one by one, what a later stage can read again
// from LDS is not kept, Wb of the plane below rests in LDS, and a stage's planes are requested where
// the stage before has let go of its registers: 0.78 ms.  The last wavefront holds the ring, whose
// loads take a line per lane: it skips the z contributions, which nobody reads (0.73), and LDS rows have
// odd pitches for its columns (0.70, VALU busy 43%).  Requests two stages ahead or spread over a stage,
// the c2p adjoint behind the next plane's barrier, and 3 or 9 variables at a time measured 2 to 4% slower.
#pragma once
#include "adj_impl.hpp"
#include "gpu_util.hpp"
#include "march_impl.hpp"

namespace glm {

// Workgroups a CU (wavefronts a SIMD).  The normal-only predictor couples the variables of each
// direction's face states, does not fit 256 registers and is faster with 512 (its reverse step with PPM
// and HLLD at 128^3: 1.62 against 2.64 ms).  The full predictor's fits and needs no second half (1.59).
constexpr int adj_waves(int pred) { return pred == PRED_FULL ? 2 : 1; }
constexpr int ADJ_GRP = 2;     // variables in work at a time
// LDS rows: odd pitches, so that the ring's columns (one lane a row) fall on different banks.
constexpr int APX = OX + 5, ANPL = APX * PY;            // W: the tile with its two-cell ring
constexpr int ADJ_EX = OX + 3, ADJ_EXN = ADJ_EX * (OY + 2);   // exchange: the tile with its one-cell ring

struct AdjBackLDS {
    double P[9][ANPL];                     // W of plane q (two-cell ring)
    double LO[9][ADJ_EXN], HI[9][ADJ_EXN];   // a lane's contributions to its lower and its upper neighbour
    double PT[9][ADJ_EXN];                // Wb of plane q-1 without plane q's share (each lane its own slot)
};

// After every lane has left its contributions to its two neighbours STEP slots away: take the two that
// are aimed at it.
template <int STEP, int NV>
GLM_DEV void adj_collect(const AdjBackLDS& L, int e, bool owned, double s0[9])
{
    __syncthreads();
    if (owned) {
#pragma unroll
        for (int v = 0; v < NV; ++v) s0[v] += L.HI[v][e - STEP] + L.LO[v][e + STEP];
    }
    __syncthreads();
}

// LDS reads behind this point are made again: the values read before it would cost two registers each
// across a stage that has none to spare.
GLM_DEV void reread()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// One direction's face-state adjoints of the lane's cell.  lr(v, l, p0, r) reads a variable and its two
// neighbours, out(v, lb, rb) takes the contributions to them; the cell's own go to s0 and mhb.
// With the full predictor the variables are independent once the guards are known, so each one is read,
// finished and handed out by itself: nine of anything would not fit the registers next to the march's
// state.  give: the lane's contributions are wanted (the halo's in z are not).  m0, m4: the predicted density and pressure (the guards look at those two only).
template <int PRED, int RECON, int SLOPE, int D, class LR, class OUT>
GLM_DEV void back_faces(const AdjArgs& a, bool up, double m0, double m4, double lob[9], double hib[9], LR lr, OUT out,
                        bool give, double s0[9], double mhb[9])
{
    const FaceOpts o{a.mh_revert, a.face_guard};
    if (PRED == PRED_ONED) {
        double l[9], p0[9], r[9], lb[9], rb[9];
#pragma unroll
        for (int v = 0; v < 9; ++v) { lr(v, l[v], p0[v], r[v]); lb[v] = 0.0; rb[v] = 0.0; }
        faces_adj<double, PRED, RECON, SLOPE, D>(l, p0, r, p0, up, a.half_dtdx, o, a.ph, lob, hib, lb, s0, rb, mhb);
#pragma unroll
        for (int v = 0; v < 9; ++v) out(v, lb[v], rb[v]);
        return;
    }
    // guards (faces_adj): iflo hands the whole face's adjoint to the cell, clamp drops the clamped entry
    if (a.face_guard != GUARD_NONE) {
        double fl[2], fh[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            double l, p0, r, el, eh;
            lr(4 * k, l, p0, r);
            const double m = k == 0 ? m0 : m4;
            const double h = half_slope<double, SLOPE>(l, p0, r);
            if (RECON == RECON_PPM) {
                ppm_edges(l, p0, r, el, eh);
                fl[k] = up ? m + el - p0 : m - h;
                fh[k] = up ? m + eh - p0 : m + h;
            } else {
                fl[k] = m - h;
                fh[k] = m + h;
            }
        }
        if (a.face_guard == GUARD_IFLO) {
            if (fl[0] < a.ph.smallr || fl[1] < a.ph.pfl)
                for (int v = 0; v < 9; ++v) { s0[v] += lob[v]; lob[v] = 0.0; }
            if (fh[0] < a.ph.smallr || fh[1] < a.ph.pfl)
                for (int v = 0; v < 9; ++v) { s0[v] += hib[v]; hib[v] = 0.0; }
        } else {
            lob[0] = fl[0] > a.ph.smallr ? lob[0] : 0.0;
            lob[4] = fl[1] > a.ph.pfl ? lob[4] : 0.0;
            hib[0] = fh[0] > a.ph.smallr ? hib[0] : 0.0;
            hib[4] = fh[1] > a.ph.pfl ? hib[4] : 0.0;
        }
    }
    if (!give) {
#pragma unroll
        for (int v = 0; v < 9; ++v) mhb[v] += lob[v] + hib[v];
    } else if (RECON == RECON_PPM && up) {
#pragma unroll
        for (int v = 0; v < 9; ++v) {
            double l, p0, r, lb, rb;
            lr(v, l, p0, r);
            mhb[v] += lob[v] + hib[v];
            ppm_offsets_adj(l, p0, r, lob[v], hib[v], lb, s0[v], rb);
            out(v, lb, rb);
            if (v % ADJ_GRP == ADJ_GRP - 1) __builtin_amdgcn_sched_barrier(0);
        }
    } else {
#pragma unroll
        for (int v = 0; v < 9; ++v) {
            double l, p0, r, lb, rb;
            lr(v, l, p0, r);
            mhb[v] += lob[v] + hib[v];
            half_slope_adj_set<double, SLOPE>(l, p0, r, hib[v] - lob[v], lb, s0[v], rb);
            out(v, lb, rb);
            if (v % ADJ_GRP == ADJ_GRP - 1) __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// One direction's share of the predictor adjoint, in the same manner (ok: the predictor did not revert;
// psi has no share).  mid runs between the flux part, where the registers are full, and the slopes'.
template <int SLOPE, int D, class LR, class OUT, class MID>
GLM_DEV void back_hancock(const AdjArgs& a, bool ok, const double accb[9], LR lr, OUT out, MID mid, double s0[9])
{
    double hsb[8];
    if (ok) {
        double p0[9], hs[9];
        p0[8] = hs[8] = 0.0;
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            double l, r;
            lr(v, l, p0[v], r);
            hs[v] = half_slope<double, SLOPE>(l, p0[v], r);
            if (v % ADJ_GRP == ADJ_GRP - 1) __builtin_amdgcn_sched_barrier(0);
        }
        hancock_adj_flux<double, D>(p0, hs, accb, s0, hsb, a.ph);
    } else {
#pragma unroll
        for (int v = 0; v < 8; ++v) hsb[v] = 0.0;
    }
    reread();
    mid();
#pragma unroll
    for (int v = 0; v < 8; ++v) {
        double l, p0, r, lb, rb;
        lr(v, l, p0, r);
        half_slope_adj_set<double, SLOPE>(l, p0, r, hsb[v], lb, s0[v], rb);
        out(v, lb, rb);
        if (v % ADJ_GRP == ADJ_GRP - 1) __builtin_amdgcn_sched_barrier(0);
    }
}

template <int PRED, int RECON, int SLOPE>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(adj_waves(PRED))))
adj_back_kernel(AdjArgs a, int tiles_x, int tiles_y, int zchunk)
{
    __shared__ AdjBackLDS L;
    double (&P)[9][ANPL] = L.P;
    const int tid = threadIdx.x;
    int tile = xcd_block((int)blockIdx.x, (int)gridDim.x);
    int tx, ty;
    lane_cell(tid, tx, ty);
    const int tile_x = tile % tiles_x; tile /= tiles_x;
    const int tile_y = tile % tiles_y; tile /= tiles_y;
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int zs = tile * zchunk;
    const int ze = min(zs + zchunk, nz);
    const size_t pl = (size_t)nx * ny;
    const int gxu = tile_x * OX - 1 + tx, gyu = tile_y * OY - 1 + ty;
    const int gx = wrapi(gxu, nx), gy = wrapi(gyu, ny);
    const bool owned = tid < NO, inside = owned && gxu < nx && gyu < ny;
    // byte offsets within a z plane of the scratch and of the caller's planes (launch_step_adjoint takes
    // this kernel only where the former stay below 4 GiB)
    const unsigned row = 8u * ADJ_NPLANES * (unsigned)nx;
    const unsigned col = 8u * (unsigned)gx + row * (unsigned)gy, ccol = 8u * (unsigned)(gx + nx * gy);
    const int lo = (ty + 1) * APX + (tx + 1), e = ty * ADJ_EX + tx;
    const bool helper = tid >= NO && tid - NO < NHELP;
    int hx = 0, hy = 0;
    helper_cell(helper ? tid - NO : 0, hx, hy);
    const unsigned hcol =
        8u * (unsigned)wrapi(tile_x * OX - 2 + hx, nx) + row * (unsigned)wrapi(tile_y * OY - 2 + hy, ny);
    const int lo_ring = hy * APX + hx;
    // nine planes of the scratch from plane p on, of z plane q at the lane's offset.  The offset is made
    // opaque per use: hoisted out of the loop as 64 bits it costs an addition and two registers a load,
    // next to the load it is the load's own offset operand.
    auto at = [&](int p, int q, unsigned off) {
        return gload_at(a.scr + ((size_t)wrapi(q, nz) * ADJ_NPLANES * ny + p) * nx, off);
    };
    auto ldp = [&](int p, int q, unsigned off, double x[9]) {
        asm volatile("" : "+v"(off));
#pragma unroll
        for (int v = 0; v < 9; ++v) x[v] = at(p + v, q, off);
    };

    // W window: planes q-1 and q+1 in registers, plane q in LDS
    double pm[9], pp[9];
    {
        double p0[9];
        ldp(ADJ_W, zs - 2, col, pm);
        ldp(ADJ_W, zs - 1, col, p0);
        ldp(ADJ_W, zs, col, pp);
#pragma unroll
        for (int v = 0; v < 9; ++v) P[v][lo] = p0[v];
        if (helper) {
            double h[9];
            ldp(ADJ_W, zs - 1, hcol, h);
#pragma unroll
            for (int v = 0; v < 9; ++v) P[v][lo_ring] = h[v];
        }
    }
    __syncthreads();

    double up1[9];   // plane q's share for plane q+1
#pragma unroll
    for (int v = 0; v < 9; ++v) { L.PT[v][e] = 0.0; up1[v] = 0.0; }

    // The planes of a direction, of the predictor and of the last stage are requested one stage ahead,
    // where the registers of the stage before are free.
    double lob[9], hib[9], m0 = 0.0, m4 = 0.0, pr = pp[4];
    auto ldL = [&](int d, int q) {
        ldp(ADJ_LFS + fs_slot(d, 0), q, col, lob);
        ldp(ADJ_LFS + fs_slot(d, 1), q, col, hib);
    };
    auto ldM = [&](int q) {
        if (PRED == PRED_FULL) {
            m0 = at(ADJ_MH, q, col);
            m4 = at(ADJ_MH + 4, q, col);
        }
    };
    ldM(zs - 1);
    ldL(0, zs - 1);

    for (int q = zs - 1;; ++q) {
        double s0[9], mhb[9];
#pragma unroll
        for (int v = 0; v < 9; ++v) { s0[v] = up1[v]; up1[v] = 0.0; mhb[v] = 0.0; }
        auto lrx = [&](int v, double& l, double& m, double& r) { l = P[v][lo - 1]; m = P[v][lo]; r = P[v][lo + 1]; };
        auto lry = [&](int v, double& l, double& m, double& r) { l = P[v][lo - APX]; m = P[v][lo]; r = P[v][lo + APX]; };
        auto lrz = [&](int v, double& l, double& m, double& r) { l = pm[v]; m = P[v][lo]; r = pp[v]; };
        auto side = [&](int v, double lb, double rb) { L.LO[v][e] = lb; L.HI[v][e] = rb; };
        auto column = [&](int v, double lb, double rb) { L.PT[v][e] += lb; up1[v] += rb; };
        // the last stage's planes: LPRE of the cell below, or W of the ring's next plane
        auto ldX = [&](double x[9]) {
            if (helper) ldp(ADJ_W, q + 1, hcol, x);
            else ldp(ADJ_LPRE, q - 1, col, x);
        };
        double xp[9];

        // face-state adjoints, one direction at a time
        {
            const double p0 = P[4][lo];
            if (PRED == PRED_FULL && a.mh_revert && (m0 <= a.ph.smallr || m4 <= a.ph.pfl)) { m0 = P[0][lo]; m4 = p0; }
            bool up = true;   // PPM strong-pressure-jump flag (glmmhd_turb.jl:959), stencil order of ppm_up
            if (RECON == RECON_PPM)
                up = !(spj(P[4][lo - 1], p0, P[4][lo + 1]) || spj(P[4][lo - APX], p0, P[4][lo + APX]) || spj(pm[4], p0, pr));
            back_faces<PRED, RECON, SLOPE, 0>(a, up, m0, m4, lob, hib, lrx, side, true, s0, mhb);
            ldL(1, q);
            adj_collect<1, 9>(L, e, owned, s0);
            back_faces<PRED, RECON, SLOPE, 1>(a, up, m0, m4, lob, hib, lry, side, true, s0, mhb);
            ldL(2, q);
            adj_collect<ADJ_EX, 9>(L, e, owned, s0);
            if (PRED != PRED_FULL) ldX(xp);
            back_faces<PRED, RECON, SLOPE, 2>(a, up, m0, m4, lob, hib, lrz, column, owned, s0, mhb);
        }

        // predictor adjoint
        if (PRED == PRED_FULL) {
            reread();
            double accb[9];
            bool ok;
            {
                double p0[9], mh[9];
                ldp(ADJ_MH, q, col, mh);
#pragma unroll
                for (int v = 0; v < 9; ++v) p0[v] = P[v][lo];
                ok = hancock_adj_core(p0, mh, mhb, s0, accb, a.half_dtdx, a.mh_revert, a.ph);
            }
            reread();
            auto none = [] {};
            back_hancock<SLOPE, 0>(a, ok, accb, lrx, side, none, s0);
            adj_collect<1, 8>(L, e, owned, s0);
            back_hancock<SLOPE, 1>(a, ok, accb, lry, side, none, s0);
            adj_collect<ADJ_EX, 8>(L, e, owned, s0);
            if (owned) back_hancock<SLOPE, 2>(a, ok, accb, lrz, column, [&] { ldX(xp); }, s0);
            else ldX(xp);
        }
        const bool last = q == ze;
        if (!last) {
            ldM(q + 1);
            ldL(0, q + 1);
            pr = at(ADJ_W + 4, q + 2, col);
        }

        // plane q-1 is complete with this plane's share: the c2p adjoint
        if (inside && q >= zs + 1) {
            double wb[9];
#pragma unroll
            for (int v = 0; v < 9; ++v) wb[v] = L.PT[v][e];
            cons2prim_adj_q(pm, wb, xp, a.ph);
            unsigned off = ccol;
            asm volatile("" : "+v"(off));
#pragma unroll
            for (int v = 0; v < 9; ++v) gstore_at(a.lam0[v] + pl * (q - 1), off, xp[v]);
        }
        if (last) break;

        // publish plane q+1 (the exchanges' barriers are behind every read of plane q's neighbours)
#pragma unroll
        for (int v = 0; v < 9; ++v) { L.PT[v][e] = s0[v]; pm[v] = P[v][lo]; P[v][lo] = pp[v]; }
        if (helper) {
#pragma unroll
            for (int v = 0; v < 9; ++v) P[v][lo_ring] = xp[v];
        }
        ldp(ADJ_W, q + 2, col, pp);
        __syncthreads();
    }
}

}  // namespace glm
