// flux_check.cpp -- the kernels' two-wave fluxes (HLL, LLF) as host functions, for their rounding error and their
// one-sided limits.  Built by tests/native/Makefile (a host-only pass of hipcc); used by the CPU tests.
#include "../../glmmhdturb_amd/csrc/hydro_march.hpp"

using namespace glm;

namespace {

// n faces: x-frame states of nine values each (rho, vx, vy, vz, p, Bx, By, Bz, psi), no floors, no cleaning
template <typename T>
void mhd(int llf, const T* L, const T* R, T* f, long n, double gamma)
{
    Phys<T> s;
    s.gamma = (T)gamma; s.igm1 = (T)(1.0 / (gamma - 1.0)); s.smallr = T(0); s.pfl = T(0);
    s.ch = T(0); s.ch2 = T(0); s.half_ich = T(0); s.llf_dmin = T(0); s.llf_pmin = T(0);
    for (long i = 0; i < n; ++i) {
        if (llf) llf_x<T, false>(L + 9 * i, R + 9 * i, f + 9 * i, s);
        else hll_x(L + 9 * i, R + 9 * i, f + 9 * i, s);
    }
}

// n faces normal to x: states of seven values each (rho, vx, vy, vz, p and two scalars), solved by HLL or LLF;
// SEL: the one-sided fluxes by selects
template <typename T, bool SEL = false>
void hydro(int llf, const T* L, const T* R, T* f, long n, double gamma)
{
    HydroArgs<T> a;
    a.gamma = (T)gamma; a.igm1 = (T)(1.0 / (gamma - 1.0));
    a.fb_dmin = llf ? T(1e30) : T(0); a.fb_pmin = T(0);
    for (long i = 0; i < n; ++i) hy_riemann<T, 0, true, 7, false, false, SEL>(L + 7 * i, R + 7 * i, f + 7 * i, a);
}

template <typename T>
void update(const T* q, const T* div, T* u, long n, double dtdx)
{
    HydroArgs<T> a;
    a.igm1 = T(2.5); a.dtdx = (T)dtdx;
    for (long i = 0; i < n; ++i) hy_update<T, 7>(q + 7 * i, div + 7 * i, u + 7 * i, a);
}

}  // namespace

extern "C" {
void fc_mhd_f32(int llf, const float* L, const float* R, float* f, long n, double g) { mhd(llf, L, R, f, n, g); }
void fc_mhd_f64(int llf, const double* L, const double* R, double* f, long n, double g) { mhd(llf, L, R, f, n, g); }
void fc_hydro_f32(int llf, const float* L, const float* R, float* f, long n, double g) { hydro(llf, L, R, f, n, g); }
void fc_hydro_f64(int llf, const double* L, const double* R, double* f, long n, double g) { hydro(llf, L, R, f, n, g); }
void fc_hydro_sel_f32(int llf, const float* L, const float* R, float* f, long n, double g) { hydro<float, true>(llf, L, R, f, n, g); }
void fc_hydro_sel_f64(int llf, const double* L, const double* R, double* f, long n, double g) { hydro<double, true>(llf, L, R, f, n, g); }
void fc_update_f32(const float* q, const float* div, float* u, long n, double dtdx) { update(q, div, u, n, dtdx); }
void fc_update_f64(const double* q, const double* div, double* u, long n, double dtdx) { update(q, div, u, n, dtdx); }
}
