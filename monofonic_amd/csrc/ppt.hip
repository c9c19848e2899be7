// Complex-to-complex 3D FFT (Grid_FFT<ccomplex_t>, grid_fft.cc:56-63,
// 207-270) and the semiclassical perturbation theory (PPT) fields of the
// field_eulerian output (ic_generator.cc:786-897): psi = sqrt(rho)
// exp(i (phi + phi2) / (hbar D+)), one kinetic drift exp(-i hbar k^2 D+ / 2)
// in k-space, the second-order kick exp(i phi2 / (hbar D+)), then the density
// |psi|^2 - 1 and the velocity hbar Im(psi* grad psi) / (1 + delta).
//
// A complex grid is [n0][n1][n2] complex.  The c2c transform runs the
// contiguous axis as row transforms in LDS and the two strided axes as the
// pencil passes of the r2c/c2r transforms; both directions are unitary.
//
// This file is compiled once per precision (MFIC_UNIT 32 or 64).
#include <cmath>
#include <vector>

#include "fft_core.hpp"
#include "mfic_internal.hpp"
#include "ppt.hpp"

namespace mfic {

static inline unsigned nblk(size_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// complex rows of length L along the contiguous axis, RW rows per block
template <typename T, int L, int RW, bool FWD>
__global__ void __launch_bounds__(Plan<L>::P * RW)
k_rows_c2c(cx<T>* __restrict__ data, long nrows, T scale, const cx<T>* __restrict__ tw) {
    constexpr int E = Plan<L>::E, P = Plan<L>::P, RP = row_lds_pitch<L>();
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int q = threadIdx.x % P, rw = threadIdx.x / P;
    const long row = (long)blockIdx.x * RW + rw;
    const bool active = row < nrows;
    cx<T>* r = data + (active ? row : 0) * (long)L;
    cx<T> v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = active ? r[q + P * e] : cx<T>{0, 0};
    fft_regs_row<T, L, FWD>(v, q, lds, rw * RP, tw);
    if (active) {
#pragma unroll
        for (int e = 0; e < E; ++e) r[q + P * e] = cscale(v[e], scale);
    }
}

template <typename T, int L, bool FWD>
static void launch_rows_c2c(mfic_ctx ctx, cx<T>* data, long nrows, T scale) {
    constexpr int P = Plan<L>::P;
    int rw = 1;
    while (rw < 64 && P * rw * 2 <= 256) rw *= 2;
    while (rw > 1 && (size_t)row_lds_pitch<L>() * rw * sizeof(cx<T>) > (size_t)ctx->max_lds) rw /= 2;
    const cx<T>* tw = static_cast<const cx<T>*>(twiddles(ctx, L, 0, sizeof(T) == 8 ? MFIC_F64 : MFIC_F32));
    const size_t lds = (size_t)row_lds_pitch<L>() * rw * sizeof(cx<T>);
    const dim3 grid((unsigned)((nrows + rw - 1) / rw));
    ProfScope prof(ctx, std::string("fft_rows_c2c_n") + std::to_string(L) + (sizeof(T) == 8 ? "_f64" : "_f32"),
                   2.0 * (double)nrows * L * sizeof(cx<T>));
    switch (rw) {
#define RWCASE(K)                                                                                                   \
    case K:                                                                                                         \
        if constexpr (P * K <= 1024)                                                                                \
            hipLaunchKernelGGL((k_rows_c2c<T, L, K, FWD>), grid, dim3(P * K), lds, ctx->stream, data, nrows, scale, tw); \
        break;
        RWCASE(1) RWCASE(2) RWCASE(4) RWCASE(8) RWCASE(16) RWCASE(32) RWCASE(64)
#undef RWCASE
    default:
        throw Error(MFIC_ERR_SIZE, "bad row tile");
    }
    MFIC_LAUNCH_CHECK();
}

#define MFIC_C2C_SIZES(X) \
    X(4) X(6) X(8) X(9) X(12) X(16) X(18) X(24) X(32) X(36) X(48) X(64) X(72) X(96) X(128) X(144) X(192) X(256) X(288) X(384) X(512) X(576) X(768)

template <typename T> void fft_c2c(mfic_ctx ctx, void* data, const size_t n[3], bool forward, double scale) {
    for (int a = 0; a < 3; ++a)
        MFIC_CHECK(fft_length_supported(n[a]), MFIC_ERR_SIZE,
                   "unsupported complex FFT length " + std::to_string(n[a]) + " (n = 2^a 3^b, 4 <= n <= 768)");
    cx<T>* d = static_cast<cx<T>*>(data);
    const long rows = (long)(n[0] * n[1]);
    switch ((int)n[2]) {
#define X(S)                                                                               \
    case S:                                                                                \
        if (forward) launch_rows_c2c<T, S, true>(ctx, d, rows, (T)1);                     \
        else launch_rows_c2c<T, S, false>(ctx, d, rows, (T)1);                            \
        break;
        MFIC_C2C_SIZES(X)
#undef X
    }
    fft_pencils<T>(ctx, data, (int)n[1], (long)n[2], (long)(n[1] * n[2]), (int)n[2], (long)n[0], forward, 1.0,
                   "_c2c_ax1");
    fft_pencils<T>(ctx, data, (int)n[0], (long)(n[1] * n[2]), 0, (int)(n[1] * n[2]), 1, forward, scale, "_c2c_ax0");
}
#if MFIC_UNIT == 64
template void fft_c2c<double>(mfic_ctx, void*, const size_t*, bool, double);
#else
template void fft_c2c<float>(mfic_ctx, void*, const size_t*, bool, double);
#endif

// ----------------------------------------------------------- PPT kernels --
// Grid_FFT::get_k component of index i, in units of 2 pi / L (n/2 maps to
// +n/2)
__device__ __forceinline__ double ppt_k(int i, int n) { return (double)(i > n / 2 ? i - n : i); }

// per-block maxima of |phi(i+1,j,k) - phi|, |phi(i,j+1,k) - phi|,
// |phi(i,j,k+1) - phi| over i < n-1 (periodic in j, k): the loop of
// ic_generator.cc:819-836, which leaves out the last x-plane
template <typename T>
__global__ void k_ppt_maxdphi(const T* __restrict__ phi, int n, double* __restrict__ part) {
    __shared__ double red[256];
    const long pitch = n + 2;
    double m = 0.0;
    for (int row = blockIdx.x; row < (n - 1) * n; row += gridDim.x) {
        const int i = row / n, j = row - i * n;
        const T* p0 = phi + (long)row * pitch;
        const T* px = p0 + n * pitch;
        const T* py = j == n - 1 ? phi + (long)i * n * pitch : p0 + pitch;
        for (int k = threadIdx.x; k < n; k += 256) {
            const double p = p0[k];
            m = fmax(m, fmax(fabs((double)px[k] - p),
                             fmax(fabs((double)py[k] - p), fabs((double)p0[k == n - 1 ? 0 : k + 1] - p))));
        }
    }
    red[threadIdx.x] = m;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// The fields take seven passes over psi where three gradients by 3D
// transforms took 24 (plus one pass per pointwise step): the pointwise steps
// run on the elements of the transform passes beside them, and since i k_d
// depends on one index only, the transforms of the other two axes cancel and
// a gradient component is a forward and an inverse transform along its own
// axis.  HBM bound: 11 elements of psi read or written a cell (and 7 real
// values) where it took about 70.  The whole call at 192^3 FP64, order 2: 2.74
// -> 0.69 ms, a third of it the two potentials' transforms; the passes run at
// 3.2-4.5 TB/s, the ones with two transforms on a load the slowest.

// 1. psi = exp(i (phi + phi2) / (hbar D+)) with sqrt(rho) = 1 (no baryon-CDM
// offset: C_species = 0, or delta_bc = 0 for Eisenstein & Hu), transformed
// forward along its rows.  The phases go through LDS (own slots, no
// exchange) so that sincos is expanded once and not per element.
template <typename T, int L, int RW>
__global__ void __launch_bounds__(Plan<L>::P * RW)
k_ppt_rows_init(cx<T>* __restrict__ psi, const T* __restrict__ phi, const T* __restrict__ phi2, long nrows,
                double inv, const cx<T>* __restrict__ tw) {
    constexpr int E = Plan<L>::E, P = Plan<L>::P, RP = row_lds_pitch<L>();
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int q = threadIdx.x % P, rw = threadIdx.x / P;
    const long row = (long)blockIdx.x * RW + rw;
    const bool active = row < nrows;
    const long o = (active ? row : 0) * (long)(L + 2);
    cx<T>* slot = lds + rw * RP + q;
#pragma unroll 1
    for (int e = 0; e < E; ++e) {
        const long c = o + q + P * e;
        double a = (double)phi[c];
        if (phi2) a += (double)phi2[c];
        double s, co;
        sincos(a * inv, &s, &co);
        slot[P * e] = cx<T>{(T)co, (T)s};
    }
    cx<T> v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = slot[P * e];
    __syncthreads();
    fft_regs_row<T, L, true>(v, q, lds, rw * RP, tw);
    if (active) {
        cx<T>* r = psi + row * (long)L;
#pragma unroll
        for (int e = 0; e < E; ++e) r[q + P * e] = v[e];
    }
}

// exp(-i (hbar D+ / 2) k^2) for every index of one axis; the drift factor of
// a mode is the product of its three
static __global__ void k_ppt_drift_table(cx<double>* __restrict__ tab, int n, double half_hbar_d, double kf) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double k = ppt_k(i, n) * kf;
    double s, co;
    sincos(-half_hbar_d * (k * k), &s, &co);
    tab[i] = cx<double>{co, s};
}

// pencils per workgroup of the axis passes: LDS of at most 48 KB (three
// workgroups a CU), at most 512 threads, at least 8 neighbouring pencils
template <typename T, int L> constexpr int ppt_tile() {
    int tk = 64;
    while (tk > 8 && (L * tk * (int)sizeof(T) > 49152 || Plan<L>::P * tk > 512)) tk /= 2;
    return tk;
}

// 2. (between the axis-1 passes) axis 0 forward, the drift
// exp(-i hbar |k|^2 D+ / 2) and both unitary scales, axis 0 backward
template <typename T, int L, int TK>
__global__ void __launch_bounds__(Plan<L>::P * TK)
k_ppt_drift(cx<T>* __restrict__ psi, const cx<double>* __restrict__ tab, double scale,
            const cx<T>* __restrict__ tw) {
    constexpr int E = Plan<L>::E, P = Plan<L>::P;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int t = threadIdx.x % TK, q = threadIdx.x / TK;
    const int col = blockIdx.x * TK + t;
    const bool active = col < L * L;
    const int j = (active ? col : 0) / L, k = (active ? col : 0) % L;
    cx<T>* base = psi + (active ? col : 0);
    cx<T> v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = base[(long)(q + P * e) * (L * L)];
    const cx<double> c = cscale(cmul(tab[j], tab[k]), scale);
    fft_pencil<T, L, true>(v, q, lds, LdsMap{t, TK}, tw);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const cx<double> w = cmul(cmul(tab[q + P * e], c), cx<double>{(double)v[e].x, (double)v[e].y});
        v[e] = cx<T>{(T)w.x, (T)w.y};
    }
    fft_pencil<T, L, false>(v, q, lds, LdsMap{t, TK}, tw);
    if (active) {
#pragma unroll
        for (int e = 0; e < E; ++e) base[(long)(q + P * e) * (L * L)] = v[e];
    }
}

// v_d = vunit Re[(psi* g - psi g*) / (2 i / hbar)] / (1 + delta)
//     = vunit hbar Im(psi* g) / (1 + delta)     (ic_generator.cc:889-896),
// delta = |psi|^2 - 1 rounded to T
template <typename T> __device__ __forceinline__ T ppt_delta(cx<T> p) {
    return (T)((double)p.x * p.x + (double)p.y * p.y - 1.0);
}
template <typename T> __device__ __forceinline__ T ppt_velocity(cx<T> p, cx<T> g, double vh) {
    const double im = (double)p.x * g.y - (double)p.y * g.x;
    return (T)(vh * im / (1.0 + (double)ppt_delta(p)));
}
// i k_d times a transformed element at index pos; kf carries 2 pi / L and
// the 1 / n of the transform pair
template <typename T> __device__ __forceinline__ cx<T> ppt_ik(cx<T> v, int pos, int n, double kf) {
    const double kd = ppt_k(pos, n) * kf;
    return cx<T>{(T)(-kd * v.y), (T)(kd * v.x)};
}

// 3. rows backward, the kick exp(i phi2 / (hbar D+)), psi and delta =
// |psi|^2 - 1 stored, and the z velocity from the same rows
template <typename T, int L, int RW>
__global__ void __launch_bounds__(Plan<L>::P * RW)
k_ppt_rows_final(cx<T>* __restrict__ psi, const T* __restrict__ phi2, T* __restrict__ delta, T* __restrict__ vz,
                 long nrows, double inv, double kf, double vh, const cx<T>* __restrict__ tw) {
    constexpr int E = Plan<L>::E, P = Plan<L>::P, RP = row_lds_pitch<L>();
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int q = threadIdx.x % P, rw = threadIdx.x / P;
    const long row = (long)blockIdx.x * RW + rw;
    const bool active = row < nrows;
    cx<T>* r = psi + (active ? row : 0) * (long)L;
    const long o = (active ? row : 0) * (long)(L + 2);
    cx<T> v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = r[q + P * e];
    fft_regs_row<T, L, false>(v, q, lds, rw * RP, tw);
    cx<T>* slot = lds + rw * RP + q;
#pragma unroll
    for (int e = 0; e < E; ++e) slot[P * e] = v[e];
#pragma unroll 1
    for (int e = 0; e < E; ++e) {
        cx<T> p = slot[P * e];
        const int k = q + P * e;
        if (phi2) {
            double s, co;
            sincos((double)phi2[o + k] * inv, &s, &co);
            p = cx<T>{(T)((double)p.x * co - (double)p.y * s), (T)((double)p.x * s + (double)p.y * co)};
            slot[P * e] = p;
        }
        if (active) {
            r[k] = p;
            delta[o + k] = ppt_delta(p);
        }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = slot[P * e];
    __syncthreads();
    fft_regs_row<T, L, true>(v, q, lds, rw * RP, tw);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = ppt_ik(v[e], q + P * e, L, kf);
    fft_regs_row<T, L, false>(v, q, lds, rw * RP, tw);
    if (active) {
#pragma unroll
        for (int e = 0; e < E; ++e) vz[o + q + P * e] = ppt_velocity(r[q + P * e], v[e], vh);
    }
}

// 4. velocity along axis AX (0 or 1) from pencils of psi
template <typename T, int L, int TK, int AX>
__global__ void __launch_bounds__(Plan<L>::P * TK)
k_ppt_pencil_velocity(const cx<T>* __restrict__ psi, T* __restrict__ vel, double kf, double vh,
                      const cx<T>* __restrict__ tw) {
    constexpr int E = Plan<L>::E, P = Plan<L>::P;
    constexpr long PS = AX == 0 ? (long)L * L : L, PV = AX == 0 ? (long)L * (L + 2) : L + 2;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int t = threadIdx.x % TK, q = threadIdx.x / TK;
    // neighbouring tiles of axis-1 pencils share cache lines of the velocity rows
    const int col = (int)(AX == 0 ? (long)blockIdx.x : xcd_tile(blockIdx.x, gridDim.x)) * TK + t;
    const bool active = col < L * L;
    const int hi = (active ? col : 0) / L, k = (active ? col : 0) % L;
    const cx<T>* p = psi + (AX == 0 ? (long)hi * L : (long)hi * L * L) + k;
    cx<T> v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = p[(q + P * e) * PS];
    fft_pencil<T, L, true>(v, q, lds, LdsMap{t, TK}, tw);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = ppt_ik(v[e], q + P * e, L, kf);
    fft_pencil<T, L, false>(v, q, lds, LdsMap{t, TK}, tw);
    if (active) {
        T* o = vel + (AX == 0 ? (long)hi * (L + 2) : (long)hi * L * (L + 2)) + k;
#pragma unroll
        for (int e = 0; e < E; ++e) o[(q + P * e) * PV] = ppt_velocity(p[(q + P * e) * PS], v[e], vh);
    }
}

template <typename T, int L>
static void ppt_passes(mfic_ctx ctx, const PptInput& in, double hbar, T* delta, T* vel[3]) {
    constexpr int P = Plan<L>::P, TK = ppt_tile<T, L>();
    constexpr int RW = P >= 256 ? 1 : (256 / P > 64 ? 64 : 256 / P);
    const int prec = sizeof(T) == 8 ? MFIC_F64 : MFIC_F32;
    const std::string tag = "_n" + std::to_string(L) + (sizeof(T) == 8 ? "_f64" : "_f32");
    const double inv = 1.0 / (hbar * in.Dplus0), kf = 2.0 * 3.14159265358979323846 / in.L, n3 = (double)L * L * L;
    const long rows = (long)L * L;
    const cx<T>* tw = static_cast<const cx<T>*>(twiddles(ctx, L, 0, prec));
    const T* phi = static_cast<const T*>(in.phi_r);
    const T* phi2 = in.order >= 2 ? static_cast<const T*>(in.phi2_r) : nullptr;
    cx<T>* psi = static_cast<cx<T>*>(in.psi);
    cx<double>* tab = static_cast<cx<double>*>(ctx_scratch(ctx, "ppt_drift", L * sizeof(cx<double>)));
    const dim3 rgrid((unsigned)((rows + RW - 1) / RW)), pgrid((unsigned)((rows + TK - 1) / TK));
    const size_t rlds = (size_t)row_lds_pitch<L>() * RW * sizeof(cx<T>), plds = (size_t)L * TK * sizeof(T);
    MFIC_CHECK(rlds <= ctx->max_lds && plds <= ctx->max_lds, MFIC_ERR_SIZE, "PPT pass exceeds the LDS of a workgroup");
    hipLaunchKernelGGL(k_ppt_drift_table, dim3((L + 63) / 64), dim3(64), 0, ctx->stream, tab, L,
                       0.5 * hbar * in.Dplus0, kf);
    MFIC_LAUNCH_CHECK();
    {
        ProfScope prof(ctx, "ppt_rows_init" + tag, n3 * (sizeof(cx<T>) + (phi2 ? 2 : 1) * sizeof(T)));
        hipLaunchKernelGGL((k_ppt_rows_init<T, L, RW>), rgrid, dim3(P * RW), rlds, ctx->stream, psi, phi, phi2, rows,
                           inv, tw);
        MFIC_LAUNCH_CHECK();
    }
    fft_pencils<T>(ctx, psi, L, (long)L, rows, L, (long)L, true, 1.0, "_c2c_ax1");
    {
        ProfScope prof(ctx, "ppt_drift" + tag, 2.0 * n3 * sizeof(cx<T>));
        hipLaunchKernelGGL((k_ppt_drift<T, L, TK>), pgrid, dim3(P * TK), plds, ctx->stream, psi, tab, 1.0 / n3, tw);
        MFIC_LAUNCH_CHECK();
    }
    fft_pencils<T>(ctx, psi, L, (long)L, rows, L, (long)L, false, 1.0, "_c2c_ax1");
    const double vh = in.vunit * hbar, kn = kf / L;
    {
        ProfScope prof(ctx, "ppt_rows_final" + tag, n3 * (2 * sizeof(cx<T>) + (phi2 ? 3 : 2) * sizeof(T)));
        hipLaunchKernelGGL((k_ppt_rows_final<T, L, RW>), rgrid, dim3(P * RW), rlds, ctx->stream, psi, phi2, delta,
                           vel[2], rows, inv, kn, vh, tw);
        MFIC_LAUNCH_CHECK();
    }
    // a buffer given for several components ends up with the last of them, z
    // (written above) before y before x
    ProfScope prof(ctx, "ppt_pencil_velocity" + tag, 2.0 * n3 * (sizeof(cx<T>) + sizeof(T)));
    if (vel[0] != vel[2]) {
        hipLaunchKernelGGL((k_ppt_pencil_velocity<T, L, TK, 0>), pgrid, dim3(P * TK), plds, ctx->stream, psi, vel[0],
                           kn, vh, tw);
        MFIC_LAUNCH_CHECK();
    }
    if (vel[1] != vel[2]) {
        hipLaunchKernelGGL((k_ppt_pencil_velocity<T, L, TK, 1>), dim3((unsigned)xcd_grid(pgrid.x)), dim3(P * TK), plds,
                           ctx->stream, psi, vel[1], kn, vh, tw);
        MFIC_LAUNCH_CHECK();
    }
}

template <typename T>
void ppt_fields_t(mfic_ctx ctx, const PptInput& in, T* delta, T* vel[3], double* hbar_out) {
    const int n = in.n;
    // hbar from the largest neighbour jump of the growth-scaled phi
    // (ic_generator.cc:815-841)
    const unsigned nb = 1024;
    double* part = static_cast<double*>(ctx_scratch(ctx, "ppt_maxdphi", nb * sizeof(double)));
    hipLaunchKernelGGL(k_ppt_maxdphi<T>, dim3(nb), dim3(256), 0, ctx->stream, static_cast<const T*>(in.phi_r), n, part);
    MFIC_LAUNCH_CHECK();
    std::vector<double> hp(nb);
    MFIC_HIP(hipMemcpyAsync(hp.data(), part, nb * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    MFIC_HIP(hipStreamSynchronize(ctx->stream));
    double maxdphi = 0.0;
    for (double x : hp) maxdphi = std::fmax(maxdphi, x);
    const double hbar = maxdphi / 3.14159265358979323846 / in.Dplus0 * 1.01;
    MFIC_CHECK(hbar > 0.0, MFIC_ERR_STATE, "PPT: the potential is constant (hbar = 0)");
    if (hbar_out) *hbar_out = hbar;
    switch (n) {
#define X(S)                                          \
    case S:                                           \
        ppt_passes<T, S>(ctx, in, hbar, delta, vel);  \
        break;
        MFIC_C2C_SIZES(X)
#undef X
    default:
        throw Error(MFIC_ERR_SIZE, "unsupported complex FFT length " + std::to_string(n) +
                                       " (n = 2^a 3^b, 4 <= n <= 768)");
    }
}

#if MFIC_UNIT == 64
template void ppt_fields_t<double>(mfic_ctx, const PptInput&, double*, double*[3], double*);
#else
extern template void ppt_fields_t<double>(mfic_ctx, const PptInput&, double*, double*[3], double*);
void ppt_fields(mfic_ctx ctx, int prec, const PptInput& in, void* delta, void* vel[3], double* hbar) {
    if (prec == MFIC_F64) {
        double* v[3] = {static_cast<double*>(vel[0]), static_cast<double*>(vel[1]), static_cast<double*>(vel[2])};
        ppt_fields_t<double>(ctx, in, static_cast<double*>(delta), v, hbar);
    } else {
        float* v[3] = {static_cast<float*>(vel[0]), static_cast<float*>(vel[1]), static_cast<float*>(vel[2])};
        ppt_fields_t<float>(ctx, in, static_cast<float*>(delta), v, hbar);
    }
}
#endif

}  // namespace mfic
