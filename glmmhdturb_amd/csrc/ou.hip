// ou.hip -- host side of the band-limited OU forcing (ou_impl.hpp): per-box buffers and the
// batched advance.
#include <cmath>
#include <cstring>
#include <vector>

#include "ou_impl.hpp"

namespace glm {

static size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

int ou_band_width(int g, double kmax)
{
    int K = kmax >= 0.0 ? (int)std::floor(kmax) : 0;
    int nb = 2 * K + 1;
    return nb < g ? nb : g;
}

hipError_t ou_box_alloc(OUBox& b, int g, double kmin, double kmax, double T, int ndt, double comp, double amp,
                        unsigned long long seed, int prec, hipStream_t st)
{
    memset(&b, 0, sizeof b);
    b.g = g;
    b.nb = ou_band_width(g, kmax);
    b.K = kmax >= 0.0 ? (int)std::floor(kmax) : 0;
    b.kmin = kmin; b.kmax = kmax;
    const double dt = T / ndt;                 // glmmhd_turb.jl:2148-2150
    b.alpha = 1.0 - dt / T;
    b.beta = std::sqrt(2.0 * dt / T);
    b.comp = comp; b.sol = 1.0 - comp;
    b.scale = amp / ((double)g * (double)g * (double)g);
    b.seed = seed;
    const size_t nb = b.nb, gg = (size_t)g * g;
    const size_t n_f = 3 * nb * nb * nb, n_w1 = 3 * nb * nb * g, n_w2 = 3 * nb * gg, n_a = 3 * gg * g;
    const size_t sz_f = al256(n_f * 8), sz_w1 = al256(n_w1 * 8), sz_w2 = al256(n_w2 * 8), sz_t = al256((size_t)g * 8);
    const size_t total = 2 * sz_f + 2 * sz_w1 + 2 * sz_w2 + 2 * sz_t + al256(n_a * prec);
    char* base = nullptr;
    hipError_t e = hipMalloc(&base, total);
    if (e != hipSuccess) return e;
    char* p = base;
    b.fre = (double*)p; p += sz_f;
    b.fim = (double*)p; p += sz_f;
    b.w1r = (double*)p; p += sz_w1;
    b.w1i = (double*)p; p += sz_w1;
    b.w2r = (double*)p; p += sz_w2;
    b.w2i = (double*)p; p += sz_w2;
    double* cs = (double*)p; p += sz_t;
    double* sn = (double*)p; p += sz_t;
    b.cs = cs; b.sn = sn;
    b.afield = p;
    std::vector<double> hc(g), hs(g);
    for (int m = 0; m < g; ++m) {
        hc[m] = std::cos(2.0 * M_PI * m / g);
        hs[m] = std::sin(2.0 * M_PI * m / g);
    }
    if ((e = hipMemcpy(cs, hc.data(), g * 8, hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = hipMemcpy(sn, hs.data(), g * 8, hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = hipMemsetAsync(base, 0, 2 * sz_f, st)) != hipSuccess) return e;
    return hipMemsetAsync(b.afield, 0, n_a * prec, st);
}

void ou_box_free(OUBox& b)
{
    if (b.fre) (void)hipFree(b.fre);
    memset(&b, 0, sizeof b);
}

static unsigned blocks_for(size_t work, int nbox)
{
    size_t cap = (size_t)(2048 / (nbox > 0 ? nbox : 1));
    if (cap < 16) cap = 16;
    size_t bl = (work + 255) / 256;
    if (bl > cap) bl = cap;
    return (unsigned)(bl > 0 ? bl : 1);
}

hipError_t launch_ou_advance(int prec, const OUBox* d_boxes, int nbox, int gmax, int nbmax, long long step_all,
                             hipStream_t st)
{
    const size_t g = gmax, nb = nbmax;
    dim3 bl(256);
    hipLaunchKernelGGL(ou_band_step_kernel, dim3(blocks_for(nb * nb * nb, nbox), nbox), bl, 0, st, d_boxes, step_all);
    hipLaunchKernelGGL(ou_pass_x_kernel, dim3(blocks_for(3 * nb * nb * g, nbox), nbox), bl, 0, st, d_boxes, step_all);
    // The y and z passes as one kernel, a workgroup a plane, where a plane's nb x g complex values fit LDS and either
    // the planes fill the device or a plane has so few terms that the launch saved is the larger part.  One kernel
    // against two, whole advances in us: 8 boxes on 64^3 with kmax 3: 70 against 117; two of them (384 planes, where
    // the lines cross): 38 against 41, with kmax 16 218 against 197; one: 33.6 against 28.5, with kmax 16 186
    // against 111.  One on 32^3 with kmax 3: 17.7 against 19.0, kmax 5 (15136 terms a plane): 26.5 against 24.1.
    // An ensemble (step_all < 0) launches the passes in each sweep, due or not, so there the launch counts for more:
    // one box of 32^3 with kmax 3 on 64^3 takes 33 us a sweep with one kernel and 35.6 with two, with kmax 16
    // on a box of 64^3 117 and 104.
    const size_t lds = 2 * nb * g * sizeof(double);
    const bool filled = 3 * g * nbox >= 384, few_terms = nb * g * (nb + g) <= (step_all < 0 ? 40000u : 10000u);
    if (lds <= 64 * 1024 && (filled || few_terms)) {
        dim3 gp((unsigned)(3 * g), nbox);
        if (prec == 8) hipLaunchKernelGGL((ou_pass_yz_kernel<double>), gp, bl, lds, st, d_boxes, step_all);
        else hipLaunchKernelGGL((ou_pass_yz_kernel<float>), gp, bl, lds, st, d_boxes, step_all);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(ou_pass_y_kernel, dim3(blocks_for(3 * nb * g * g, nbox), nbox), bl, 0, st, d_boxes, step_all);
    dim3 gz(blocks_for(3 * g * g * g, nbox), nbox);
    if (prec == 8) hipLaunchKernelGGL((ou_pass_z_kernel<double>), gz, bl, 0, st, d_boxes, step_all);
    else hipLaunchKernelGGL((ou_pass_z_kernel<float>), gz, bl, 0, st, d_boxes, step_all);
    return hipGetLastError();
}

hipError_t launch_ou_reset(int prec, const OUBox* d_boxes, int nbox, int gmax, hipStream_t st)
{
    hipLaunchKernelGGL(ou_reset_kernel, dim3(blocks_for(3 * (size_t)gmax * gmax * gmax, nbox), nbox), dim3(256), 0, st, d_boxes, prec);
    return hipGetLastError();
}

}  // namespace glm
