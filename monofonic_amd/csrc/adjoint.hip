// Differentiable 2LPT: the forward map from real-space white noise to the
// 2LPT displacement fields and its hand-written adjoint (reverse mode).
//
// Forward (ic_generator.cc:378-383, 509-555, 916-970 with the NGenIC
// convention of empty Nyquist planes, random_ngenic.cc:117):
//   w = P_N r2c(delta)                 P_N: zero the i, j or k = N/2 planes
//   phi1 = S w,  S(k) = -A(k) / (k^2 volfac), DC := 0
//   phi2 = lap^-1 mu2(phi1),  mu2 = T[xx yy + xx zz + yy zz - xy^2 - xz^2 - yz^2]
//   Psi_d = c2r( i g_d (g1 phi1 + g2 phi2) ) * unit, DC := 0
// with T the Orszag truncation (convolution.hh:495-651).  Adjoint, for
// cotangents G_d of Psi_d and the full-spectrum inner product:
//   lam = unit * sum_d (-i g_d) r2c(G_d), DC := 0
//   lam1 = g1 lam;  lam_mu = P_N lap^-1 (g2 lam)
//   lam1 += D_xx T(lam_mu (H_yy + H_zz)) + D_yy T(lam_mu (H_xx + H_zz))
//         + D_zz T(lam_mu (H_xx + H_yy)) - 2 D_xy T(lam_mu H_xy)
//         - 2 D_xz T(lam_mu H_xz) - 2 D_yz T(lam_mu H_yz)
//   grad = c2r( P_N S lam1 )
// (the adjoint of a -> T(a b) is l -> T(l b) for real band-limited b, and
// D_ab = -g_a g_b, S and lap^-1 are real diagonal multipliers).  phi1 is
// recomputed from delta in the adjoint instead of being stored.
//
// The six products share their transforms: lam_mu and the six Hessians of
// phi1 go through the padded passes once, one row pass forms all products,
// and the D_ab act per axis on the way back (padded_hessian_adjoint).
// Bound by those passes; forward and adjoint of a 256^3 FP32 box through
// autograd 3.57 ms, 7.24 ms as six two-operand convolutions.
#include <cmath>
#include <string>

#include "cosmology.hpp"
#include "fft_core.hpp"
#include "kspace.hpp"
#include "mfic_internal.hpp"

namespace mfic {

namespace {

struct Geo {
    int n0, n1, n2, nc;
    double kf0, kf1, kf2;
    __device__ __forceinline__ void ijk(size_t idx, int& i, int& j, int& k) const {
        k = (int)(idx % nc);
        const size_t r = idx / nc;
        j = (int)(r % n1);
        i = (int)(r / n1);
    }
    // Grid_FFT::gradient component (grid_fft.hh:376-385): 0 at index n/2
    __device__ __forceinline__ double g(int d, int i, int j, int k) const {
        const int idx = d == 0 ? i : (d == 1 ? j : k);
        const int n = d == 0 ? n0 : (d == 1 ? n1 : n2);
        const double kf = d == 0 ? kf0 : (d == 1 ? kf1 : kf2);
        return idx == n / 2 ? 0.0 : ((double)idx - (double)(idx > n / 2) * n) * kf;
    }
};

Geo geo_of(mfic_grid g) {
    Geo G;
    G.n0 = (int)g->n[0];
    G.n1 = (int)g->n[1];
    G.n2 = (int)g->n[2];
    G.nc = (int)g->nc();
    const double pi2 = 2.0 * 3.14159265358979323846;
    G.kf0 = pi2 / g->L[0];
    G.kf1 = pi2 / g->L[1];
    G.kf2 = pi2 / g->L[2];
    return G;
}

// lam = unit * sum_d (-i g_d) G_d, DC := 0, and lam_mu = lap^-1 (g2 lam) with
// empty Nyquist planes
template <typename T>
__global__ void k_grad_adjoint(cx<T>* __restrict__ lam, cx<T>* __restrict__ lmu, const cx<T>* __restrict__ gx,
                               const cx<T>* __restrict__ gy, const cx<T>* __restrict__ gz, Geo G, size_t nk,
                               double unit, double g2) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nk) return;
    int i, j, k;
    G.ijk(idx, i, j, k);
    const cx<T> in[3] = {gx[idx], gy[idx], gz[idx]};
    const double g[3] = {G.g(0, i, j, k), G.g(1, i, j, k), G.g(2, i, j, k)};
    double re = 0.0, im = 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {  // (-i g)(x + i y) = g y - i g x
        re += g[d] * (double)in[d].y;
        im -= g[d] * (double)in[d].x;
    }
    re *= unit;
    im *= unit;
    const bool nyq = i == G.n0 / 2 || j == G.n1 / 2 || k == G.n2 / 2;
    lam[idx] = idx == 0 ? cx<T>{0, 0} : cx<T>{(T)re, (T)im};
    // off the Nyquist planes g is the wave vector
    const double f = idx == 0 || nyq ? 0.0 : -g2 / (g[0] * g[0] + g[1] * g[1] + g[2] * g[2]);
    lmu[idx] = cx<T>{(T)(re * f), (T)(im * f)};
}

unsigned nblk(size_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

void kspace_grad_adjoint(mfic_grid lam, mfic_grid lmu, mfic_grid gx, mfic_grid gy, mfic_grid gz, double unit,
                         double g2) {
    const Geo G = geo_of(lam);
    const size_t nk = (size_t)G.n0 * G.n1 * G.nc;
    ProfScope prof(lam->ctx, "adjoint_gradient", 5.0 * lam->bytes());
    if (lam->prec == MFIC_F64)
        hipLaunchKernelGGL(k_grad_adjoint<double>, dim3(nblk(nk)), dim3(256), 0, lam->ctx->stream, (cx<double>*)lam->d,
                           (cx<double>*)lmu->d, (const cx<double>*)gx->d, (const cx<double>*)gy->d,
                           (const cx<double>*)gz->d, G, nk, unit, g2);
    else
        hipLaunchKernelGGL(k_grad_adjoint<float>, dim3(nblk(nk)), dim3(256), 0, lam->ctx->stream, (cx<float>*)lam->d,
                           (cx<float>*)lmu->d, (const cx<float>*)gx->d, (const cx<float>*)gy->d,
                           (const cx<float>*)gz->d, G, nk, unit, g2);
    MFIC_LAUNCH_CHECK();
}

}  // namespace mfic
