// Fused padded row pass for the LPT sources (ic_generator.cc:523-629 with
// the Orszag 3/2 rule of convolution.hh:495-532).
//
// One workgroup takes one or a few padded rows (i', j').  Each input field's
// compact half-spectrum row (kz <= N/2, after the axis-0 and axis-1 c2r
// passes) is brought to real space in LDS by its own thread group, the
// source products are formed pointwise from LDS with FP64 sums, and every
// output row is transformed back (r2c) and written as a compact
// half-spectrum row for the axis-1 / axis-0 r2c passes.  The padded real
// fields therefore never reach HBM: per row the pass reads NI and writes NO
// compact rows.
//
// Each transform's threads lie inside one wavefront (groups start on
// power-of-two lane boundaries), so Stockham stages synchronise per
// wavefront and idle output groups simply skip the r2c; workgroup barriers
// separate the three phases.  Two forms: one half-length transform per row
// (k_rows_fused) or two rows per full-length complex transform
// (k_rows_fused_pair, the default), chosen per length and precision at run
// time.  The products of the convolver and of the 2LPT adjoint use the second.
//
// This file is compiled once per precision (MFIC_UNIT 32 or 64).
#include <cmath>

#include "fft_core.hpp"
#include "fused.hpp"
#include "mfic_internal.hpp"

namespace mfic {

// Products at one real point: NF fields in, NOF products out.  The paired form
// takes ROWS padded rows together.  With two, a pair is two neighbouring rows
// of one field: an odd number of inputs or outputs pairs up, and fields of
// different size (the operands of a convolver call, the adjoint's lambda)
// keep their own rounding, where a shared transform would give the smaller
// one the larger one's.
// Hessian component order in every source: xx yy zz xy xz yz
// 2LPT source (ic_generator.cc:536-541)
struct ProdSrc2 {
    static constexpr int NF = 6, NOF = 1, ROWS = 2, WAVES = 3;
    static constexpr bool OUT32 = false;
    __device__ static __forceinline__ void eval(const double* h, double* o) {
        o[0] = h[0] * (h[1] + h[2]) + h[1] * h[2] - h[3] * h[3] - h[4] * h[4] - h[5] * h[5];
    }
};
// 2LPT source plus the inner products of the 3a terms grouped by their outer
// factor: Qzz = xx yy - xy^2, Qyz = xy xz, Qxx = yz^2, Qyy = xz^2
// (ic_generator.cc:581-585)
struct ProdSrc2Q {
    static constexpr int NF = 6, NOF = 5, ROWS = 2, WAVES = 3;
    static constexpr bool OUT32 = false;
    __device__ static __forceinline__ void eval(const double* h, double* o) {
        ProdSrc2::eval(h, o);
        o[1] = h[0] * h[1] - h[3] * h[3];
        o[2] = h[3] * h[4];
        o[3] = h[5] * h[5];
        o[4] = h[4] * h[4];
    }
};
// phi3 source (3a outer products with the truncated Q fields + 3b,
// ic_generator.cc:581-609) and A3 (ic_generator.cc:614-627).  Inputs: phi1
// Hessians a[0..5], phi2 Hessians b[6..11], Qzz Qyz Qxx Qyy [12..15]
struct ProdSrc3 {
    // registers for two waves per SIMD (no spills), i.e. two workgroups per CU
    static constexpr int NF = 16, NOF = 4, ROWS = 1, WAVES = 2;
    // half-length form: the four output transforms on 32 threads each (two
    // waves) instead of 16 (one wave): the output phase was a third of the pass
    static constexpr bool OUT32 = true;
    __device__ static __forceinline__ void eval(const double* h, double* o) {
        const double* a = h;
        const double* b = h + 6;
        const double* Q = h + 12;
        const double c5 = -5.0 / 7.0, c10 = 10.0 / 7.0;
        o[0] = Q[0] * a[2] + 2.0 * (Q[1] * a[5]) - Q[2] * a[0] - Q[3] * a[1] +
               c5 * (a[0] * (b[1] + b[2]) + a[1] * (b[2] + b[0]) + a[2] * (b[0] + b[1])) +
               c10 * (a[3] * b[3] + a[4] * b[4] + a[5] * b[5]);
        // A3[d] = b_{dd'} a_{dd''} - b_{dd''} a_{dd'} + a_{d'd''} (b_{d'd'} - b_{d''d''})
        //         - b_{d'd''} (a_{d'd'} - a_{d''d''}),  d' = d+1, d'' = d+2 (mod 3)
        o[1] = b[3] * a[4] - b[4] * a[3] + a[5] * (b[1] - b[2]) - b[5] * (a[1] - a[2]);
        o[2] = b[5] * a[3] - b[3] * a[5] + a[4] * (b[2] - b[0]) - b[4] * (a[2] - a[0]);
        o[3] = b[4] * a[5] - b[5] * a[4] + a[3] * (b[0] - b[1]) - b[3] * (a[0] - a[1]);
    }
};
// convolver products: two operands, or one with itself
struct ProdMul {
    static constexpr int NF = 2, NOF = 1, ROWS = 2;
    __device__ static __forceinline__ void eval(const double* h, double* o) { o[0] = h[0] * h[1]; }
};
struct ProdSquare {
    static constexpr int NF = 1, NOF = 1, ROWS = 2;
    __device__ static __forceinline__ void eval(const double* h, double* o) { o[0] = h[0] * h[0]; }
};
// adjoint of the 2LPT source: phi1 Hessians a[0..5] and lambda [6] -> lambda
// times the derivative of the source with respect to each Hessian
struct ProdAdjoint2 {
    static constexpr int NF = 7, NOF = 6, ROWS = 2;
    __device__ static __forceinline__ void eval(const double* a, double* o) {
        const double l = a[6];
        o[0] = l * (a[1] + a[2]);
        o[1] = l * (a[0] + a[2]);
        o[2] = l * (a[0] + a[1]);
        o[3] = -2.0 * (l * a[3]);
        o[4] = -2.0 * (l * a[4]);
        o[5] = -2.0 * (l * a[5]);
    }
};

template <int M, int NI> constexpr int fused_rows_per_block() {
    constexpr int tpr = NI * lane_slot<Plan<M>::P>();
    return tpr >= 256 ? 1 : (256 / tpr > 8 ? 8 : 256 / tpr);
}

// FP32: at least PR::WAVES waves per SIMD (register budget 512 / WAVES)
template <typename T, int M, class PR>
__global__ void __launch_bounds__((fused_rows_per_block<M, PR::NF>() * PR::NF * lane_slot<Plan<M>::P>()))
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? PR::WAVES : 1, 8)))
k_rows_fused(const cx<T>* __restrict__ in, long istride, cx<T>* __restrict__ out, long ostride, int kc, long nrows,
             T scale, const cx<T>* __restrict__ tw, const cx<T>* __restrict__ tw2) {
    constexpr int NI = PR::NF, NO = PR::NOF, NG = NI;
    constexpr int E = Plan<M>::E, P = Plan<M>::P, SL = lane_slot<P>();
    constexpr int RP = row_lds_pitch<M>(), RB = fused_rows_per_block<M, NG>(), TPR = NG * SL;
    constexpr int NPOS = (M + TPR - 1) / TPR;
    static_assert(P <= 64 && 64 % SL == 0, "a transform must fit in one wavefront");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int tr = threadIdx.x % TPR, rb = threadIdx.x / TPR;
    const int g = tr / SL, q = tr % SL;
    const bool lane = q < P;
    const long row = xcd_tile(blockIdx.x, gridDim.x) * RB + rb;
    const bool active = row < nrows;
    const cx<T>* uw = tw + plan_tw_size<M>();

    // 1. c2r of input g: half-spectrum row (kz < kc, kz = 0 and the padded
    // Nyquist real) -> M complex = 2M real values, kept in its input's region
    if (lane) {
        // kc = N/2 + 1 with N = 4M/3: positions below KC carry data, the rest
        // of the padded row is the zero band
        constexpr int KC = 2 * M / 3 + 1;
        const cx<T>* src = in + g * istride + (active ? row : 0) * (long)KC;
        const LdsRowMap lm{(rb * NI + g) * RP};
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = q + P * e;
            cx<T> x = cx<T>{0, 0};
            if (P * e + P <= KC) x = src[k];
            else if (P * e < KC) x = k < KC ? src[k] : cx<T>{0, 0};
            if (k == 0) x.y = 0;
            lds[lm.at(k)] = x;
        }
        if (q == 0) lds[lm.at(M)] = cx<T>{0, 0};
        WaveSync::sync();
        cx<T> v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = q + P * e;
            const cx<T> xk = lds[lm.at(k)], xm = lds[lm.at(M - k)];
            const cx<T> A = {xk.x + xm.x, xk.y - xm.y};
            const cx<T> D = {xk.x - xm.x, xk.y + xm.y};
            const cx<T> B = cmulc(D, uw[k]);
            v[e] = cx<T>{A.x - B.y, A.y + B.x};
        }
        WaveSync::sync();
        fft_regs_row<T, M, false, WaveSync>(v, q, lds, lm.base, tw);
#pragma unroll
        for (int e = 0; e < E; ++e) lds[lm.at(q + P * e)] = cscale(v[e], scale);
    }
    __syncthreads();

    // 2. source products at each complex slot (two real points), FP64 sums
    // rounded once to T.  Slot p of every row is read and written by one
    // thread only, so outputs overwrite the first NO input rows in place.
#pragma unroll
    for (int u = 0; u < NPOS; ++u) {
        const int p = tr + u * TPR;
        if (p < M) {
            cx<T> x[NI];
#pragma unroll
            for (int f = 0; f < NI; ++f) x[f] = lds[(rb * NI + f) * RP + p];
            T res[NO][2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                double h[NI], o[NO];
#pragma unroll
                for (int f = 0; f < NI; ++f) h[f] = (double)(c ? x[f].y : x[f].x);
                PR::eval(h, o);
#pragma unroll
                for (int r = 0; r < NO; ++r) res[r][c] = (T)o[r];
            }
#pragma unroll
            for (int o = 0; o < NO; ++o) lds[(rb * NI + o) * RP + p] = cx<T>{res[o][0], res[o][1]};
        }
    }
    __syncthreads();

    // 3. r2c of outputs g, g + NG, ... < NO, first kc half-spectrum values written
    constexpr int RV = row_alt_plan<M>();
    constexpr bool O32 = PR::OUT32 && RV == 2 && RB == 1 && NO * Plan<M, RV>::P <= NG * SL;
    if constexpr (O32) {
        constexpr int E2 = Plan<M, RV>::E, P2 = Plan<M, RV>::P;
        const int o = tr / P2, q2 = tr % P2;
        const cx<T>* uw2 = tw2 + plan_tw_size<M, RV>();
        if (o < NO) {
            const int base = (rb * NI + o) * RP;
            cx<T> v[E2];
#pragma unroll
            for (int e = 0; e < E2; ++e) v[e] = lds[base + q2 + P2 * e];
            WaveSync::sync();
            fft_regs_row<T, M, true, WaveSync, RV>(v, q2, lds, base, tw2);
#pragma unroll
            for (int e = 0; e < E2; ++e) lds[base + q2 + P2 * e] = v[e];
            WaveSync::sync();
            if (active) {
                cx<T>* dst = out + o * ostride + row * (long)kc;
#pragma unroll
                for (int e = 0; e < E2; ++e) {
                    const int k = q2 + P2 * e;
                    if (k >= kc) continue;
                    const cx<T> zk = v[e], zm = lds[base + (k == 0 ? 0 : M - k)];
                    const cx<T> Ek = {(zk.x + zm.x) * (T)0.5, (zk.y - zm.y) * (T)0.5};
                    const cx<T> Ok = {(zk.y + zm.y) * (T)0.5, (zm.x - zk.x) * (T)0.5};
                    dst[k] = cadd(Ek, cmul(uw2[k], Ok));
                }
            }
        }
    } else if (lane) {
        for (int o = g; o < NO; o += NG) {
            const LdsRowMap lm{(rb * NI + o) * RP};
            cx<T> v[E];
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = lds[lm.at(q + P * e)];
            WaveSync::sync();
            fft_regs_row<T, M, true, WaveSync>(v, q, lds, lm.base, tw);
#pragma unroll
            for (int e = 0; e < E; ++e) lds[lm.at(q + P * e)] = v[e];
            WaveSync::sync();
            if (active) {
                cx<T>* dst = out + o * ostride + row * (long)kc;
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const int k = q + P * e;
                    if (k >= kc) continue;
                    const cx<T> zk = v[e], zm = lds[lm.at(k == 0 ? 0 : M - k)];
                    const cx<T> Ek = {(zk.x + zm.x) * (T)0.5, (zk.y - zm.y) * (T)0.5};
                    const cx<T> Ok = {(zk.y + zm.y) * (T)0.5, (zm.x - zk.x) * (T)0.5};
                    dst[k] = cadd(Ek, cmul(uw[k], Ok));
                }
            }
        }
    }
}

// Paired form of the fused row pass: two real rows per complex transform of
// the full padded length L2 = 2M.  Inputs 2g and 2g+1 of a row are brought
// to real space together, z = x_2g + i x_2g+1, from the Hermitian spectrum
// Z[k] = X_2g[k] + i X_2g+1[k] (k <= N/2) and conj(X_2g[L2-k]) +
// i conj(X_2g+1[L2-k]) (k >= L2 - N/2), read straight from the compact rows:
// no half-length untangle, no LDS round trip before the transform.  Outputs
// are paired the same way, w = o_2p + i o_2p+1, and separated after the
// forward transform as O_2p[k] = W[k] + conj(W[L2-k]),
// O_2p+1[k] = -i (W[k] - conj(W[L2-k])) (the 1/2 and both normalisations
// are one FP64 factor on the products).
//
// Bound by vector issue and by latency: 65% of the issue slots at 3 waves a
// SIMD, which is what whole complex rows in LDS left room for.  So an exchange
// takes real and imaginary parts in turn and the product stage half the
// points at a time, which halves the LDS (4 waves and more), the factors
// between stages are read from LDS (from memory, the lanes' spread-out reads
// of them kept the vector cache busier than the data), and the plans avoid
// the 24-point butterfly.  6-, 16- and 7-input passes:
//   768 FP32 4.37 -> 3.97 ms, 8.79 -> 7.2 ms; 384 FP32 0.62 -> 0.46, 1.11 ->
//   0.82, 0.73 -> 0.53 ms; 288 FP64 0.48 -> 0.45, 0.85 -> 0.76 ms; 384 FP64
//   1.45 -> 0.95, 2.79 -> 1.63 ms; 576 FP64 5.36 -> 4.07, 9.30 -> 6.73 ms
// without the transforms the same loads and stores take 5.1 ms (768, 16
// inputs), 0.76 (384) and 0.56 (288 FP64).
template <typename T, int L2> constexpr int pair_variant() {
    // 24 values to a thread in FP32 (576 points, which have no plan of that
    // kind with power-of-two spans: 12), 12 in FP64
    return sizeof(T) == 8 || L2 == 576 ? pair_wide_plan<L2>() : pair_narrow_plan<L2>();
}
// waves per SIMD to fit the registers to: 4 hold 12 FP64 or 24 FP32 values
// without spilling (288 points FP64, 16 inputs: 0.76 ms, 0.88 with the
// compiler's own choice of 3), except for four-stage FP64 plans with their
// precomputed exchange addresses (384 points, 2 inputs: 0.27 ms with 3, 0.31
// with 4)
template <typename T, int L2> constexpr int pair_waves() {
    return sizeof(T) == 8 && Plan<L2, pair_variant<T, L2>()>::S > 3 ? 3 : 4;
}
template <typename T, int L2, int GI> constexpr int pair_rows_per_block() {
    constexpr int tpr = GI * lane_slot<Plan<L2, pair_variant<T, L2>()>::P>();
    return tpr >= 256 ? 1 : (256 / tpr > 8 ? 8 : 256 / tpr);
}
template <class PR> constexpr int pair_inputs() { return PR::NF * PR::ROWS / 2; }
template <class PR> constexpr int pair_outputs() { return (PR::NOF * PR::ROWS + 1) / 2; }
template <typename T, int L2, class PR> constexpr int pair_block_threads() {
    constexpr int GI = pair_inputs<PR>();
    return pair_rows_per_block<T, L2, GI>() * GI * lane_slot<Plan<L2, pair_variant<T, L2>()>::P>();
}
// LDS of a pair row, in T: an exchange takes real and imaginary parts in turn
// and the product stage half the points at a time, so a row needs L2 values
// of T, not L2 complex ones.  The pitch puts the transforms that share a
// 32-lane group a lane slot apart modulo the 32 banks.
template <int L2, int SL> constexpr int pair_row_pitch() { return L2 + (((SL < 2 ? 2 : SL) - L2) % 32 + 32) % 32; }

template <typename T, int L2, class PR>
__global__ void __launch_bounds__((pair_block_threads<T, L2, PR>()))
__attribute__((amdgpu_waves_per_eu(pair_waves<T, L2>(), 8)))
k_rows_fused_pair(const cx<T>* __restrict__ in, long istride, cx<T>* __restrict__ out, long ostride, long nrows,
                  double scale2, const cx<T>* __restrict__ tw) {
    constexpr int NF = PR::NF, NOF = PR::NOF, ROWS = PR::ROWS, NI = NF * ROWS, NO = NOF * ROWS;
    constexpr int GI = pair_inputs<PR>(), GO = pair_outputs<PR>();
    constexpr int V = pair_variant<T, L2>(), E = Plan<L2, V>::E, P = Plan<L2, V>::P, SL = lane_slot<P>();
    constexpr int RB = pair_rows_per_block<T, L2, GI>(), TPR = GI * SL, RP = pair_row_pitch<L2, SL>();
    constexpr int KC = L2 / 3 + 1;  // N/2 + 1 values per compact row, N = 2 L2 / 3
    constexpr int H = L2 / 2, HP = RP / 2, NPOS = (H + TPR - 1) / TPR;
    static_assert(E % 2 == 0 && L2 % 2 == 0 && RP % 2 == 0, "rows are handled in halves");
    static_assert(NI % 2 == 0, "inputs come in pairs");
    static_assert(P <= 64 && 64 % SL == 0, "a transform must fit in one wavefront");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int tr = threadIdx.x % TPR, rb = threadIdx.x / TPR;
    const int g = tr / SL, q = tr % SL;
    // groups of ROWS consecutive rows; input i of a group is field i / ROWS
    // of its row i % ROWS, output o product o / ROWS of its row o % ROWS
    const long tile = xcd_tile(blockIdx.x, gridDim.x);
    const long group = tile * RB + rb, ngroups = nrows / ROWS;

    // the inter-stage factors go to LDS once for the block: read from memory
    // by every lane they cost more cycles in the vector cache than the data
    // (FP32: stored once the data loads are under way, 768 points 4.09 -> 3.94
    // ms; FP64, where they would take registers from the data, at once)
    constexpr int NTW = plan_tw_size<L2, V>(), NT = pair_block_threads<T, L2, PR>();
    cx<T>* ltw = lds + RB * GI * HP;
    TwStage<T, L2, V, NT> tws;
    if constexpr (sizeof(T) == 4) {
        tws.load(tw);
    } else {
#pragma unroll
        for (int i = 0; i < NTW; i += NT)
            if (i + (int)threadIdx.x < NTW) ltw[i + threadIdx.x] = tw[i + threadIdx.x];
    }

    // 1. inverse transform of input pair g: all compact-row loads first, the
    // zero band (N/2 < k < L2 - N/2) never loaded
    cx<T> v[E], a[E], b[E];
    if (q < P) {
        const long r0 = (group < ngroups ? group : 0) * (long)(ROWS * KC);
        const int i0 = 2 * g, i1 = 2 * g + 1;
        const cx<T>* s0 = in + (i0 / ROWS) * istride + r0 + (i0 % ROWS) * KC;
        const cx<T>* s1 = in + (i1 / ROWS) * istride + r0 + (i1 % ROWS) * KC;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = q + P * e;
            a[e] = b[e] = cx<T>{0, 0};
            if (P * e + P <= KC) {
                a[e] = s0[k];
                b[e] = s1[k];
            } else if (P * e > L2 - KC) {
                a[e] = s0[L2 - k];
                b[e] = s1[L2 - k];
            } else if (P * e < KC || P * e + P > L2 - KC + 1) {
                if (k < KC) {
                    a[e] = s0[k];
                    b[e] = s1[k];
                } else if (k > L2 - KC) {
                    a[e] = s0[L2 - k];
                    b[e] = s1[L2 - k];
                }
            }
        }
    }
    if constexpr (sizeof(T) == 4) tws.store(ltw);
    __syncthreads();
    if (q < P) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = q + P * e;
            if (P * e > L2 - KC || (P * e + P > L2 - KC + 1 && k > L2 - KC)) {
                v[e] = cx<T>{a[e].x + b[e].y, b[e].x - a[e].y};  // conj(A) + i conj(B)
            } else {
                if (e == 0 && k == 0) a[e].y = b[e].y = 0;  // the DC imaginary parts are not data
                v[e] = cx<T>{a[e].x - b[e].y, a[e].y + b[e].x};  // A + i B
            }
        }
        fft_regs_row<T, L2, false, WaveSync, V, true, true>(v, q, lds, (rb * GI + g) * RP, ltw);
    }

    // 2. products at every real point n from the NI/2 pair rows, in FP64,
    // times the normalisation, half the points at a time; outputs paired over
    // the first pair rows (a point is read and written by one thread only)
    // and taken by their transforms' threads
    const int rbo = (threadIdx.x / SL) / GO, po = (threadIdx.x / SL) % GO;
    // the position again, as a value of its own: or the compiler holds the
    // inverse transforms' factors and addresses in registers for the forward
    // ones and spills (768 points, 6 inputs: 5.0 against 4.0 ms)
    int qo = q;
    asm("" : "+v"(qo));
    const bool olane = rbo < RB && qo < P;
    const int obase = (rbo * GI + po) * HP;
    cx<T> w[E];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        if (q < P) {
            const int base = (rb * GI + g) * HP;
#pragma unroll
            for (int e = 0; e < E / 2; ++e) lds[base + q + P * e] = v[e + half * (E / 2)];
        }
        __syncthreads();
        // the second half starts half a row of threads on, where the first
        // half's last round may have left threads without a point
        const int t0 = half ? (tr + TPR / 2) % TPR : tr;
#pragma unroll
        for (int u = 0; u < NPOS; ++u) {
            const int n = t0 + u * TPR;
            if (n < H) {
                double h[NI], o[NO];
#pragma unroll
                for (int p = 0; p < GI; ++p) {
                    const cx<T> z = lds[(rb * GI + p) * HP + n];
                    h[2 * p] = (double)z.x;
                    h[2 * p + 1] = (double)z.y;
                }
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                    double hr[NF], orow[NOF];
#pragma unroll
                    for (int f = 0; f < NF; ++f) hr[f] = h[f * ROWS + r];
                    PR::eval(hr, orow);
#pragma unroll
                    for (int f = 0; f < NOF; ++f) o[f * ROWS + r] = orow[f];
                }
#pragma unroll
                for (int p = 0; p < GO; ++p) {
                    const T lo = (T)(o[2 * p] * scale2);
                    const T hi = 2 * p + 1 < NO ? (T)(o[2 * p + 1] * scale2) : (T)0;
                    lds[(rb * GI + p) * HP + n] = cx<T>{lo, hi};
                }
            }
        }
        __syncthreads();
        if (olane) {
#pragma unroll
            for (int e = 0; e < E / 2; ++e) w[e + half * (E / 2)] = lds[obase + qo + P * e];
        }
        if (half == 0) __syncthreads();
    }

    // 3. forward transform of output pair po, separated into the two outputs'
    // first KC modes
    if (olane) {
        WaveSync::sync();
        fft_regs_row<T, L2, true, WaveSync, V, true, true>(w, qo, lds, 2 * obase, ltw);
        // partners W[L2 - k] of the kept modes sit at L2 - KC + 1 .. L2 - 1,
        // in the upper half of the row
#pragma unroll
        for (int e = E / 2; e < E; ++e)
            if (P * e + P > L2 - KC + 1) lds[obase + qo + P * e - H] = w[e];
        WaveSync::sync();
        const long groupo = tile * RB + rbo;
        if (groupo < ngroups) {
            const int o0 = 2 * po, o1 = 2 * po + 1 < NO ? 2 * po + 1 : 2 * po;
            cx<T>* d0 = out + (o0 / ROWS) * ostride + (groupo * ROWS + o0 % ROWS) * (long)KC;
            cx<T>* d1 = out + (o1 / ROWS) * ostride + (groupo * ROWS + o1 % ROWS) * (long)KC;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int k = qo + P * e;
                if (P * e >= KC || k >= KC) continue;
                const cx<T> x = w[e], xm = k == 0 ? w[e] : lds[obase + H - k];
                d0[k] = cx<T>{x.x + xm.x, x.y - xm.y};
                if (2 * po + 1 < NO) d1[k] = cx<T>{x.y + xm.y, xm.x - x.x};
            }
        }
    }
}

template <typename T, int L2, class PR>
static void launch_fused_pair(mfic_ctx ctx, const void* in, void* out, long stride, int kc, long nrows, double scale,
                              const char* name) {
    constexpr int GI = pair_inputs<PR>();
    constexpr int RB = pair_rows_per_block<T, L2, GI>(), V = pair_variant<T, L2>();
    MFIC_CHECK(3 * (kc - 1) == L2 && nrows % PR::ROWS == 0, MFIC_ERR_SIZE,
               "half-spectrum rows must hold N/2 + 1 values of a 3N/2 padded row");
    constexpr int RP = pair_row_pitch<L2, lane_slot<Plan<L2, V>::P>()>();
    const size_t lds = (size_t)RB * GI * RP * sizeof(T) + plan_tw_size<L2, V>() * sizeof(cx<T>);
    MFIC_CHECK(lds <= (size_t)ctx->max_lds, MFIC_ERR_SIZE, "fused row pass exceeds the LDS of a workgroup");
    const int prec = sizeof(T) == 8 ? MFIC_F64 : MFIC_F32;
    const cx<T>* tw = static_cast<const cx<T>*>(twiddles(ctx, L2, 3, prec, V));
    dim3 grid((unsigned)xcd_grid((nrows / PR::ROWS + RB - 1) / RB));
    ProfScope prof(ctx, std::string(name) + "_n" + std::to_string(L2) + (sizeof(T) == 8 ? "_f64" : "_f32"),
                   (double)nrows * (PR::NF + PR::NOF) * kc * sizeof(cx<T>));
    hipLaunchKernelGGL((k_rows_fused_pair<T, L2, PR>), grid, dim3(pair_block_threads<T, L2, PR>()), lds, ctx->stream,
                       static_cast<const cx<T>*>(in), stride, static_cast<cx<T>*>(out), stride, nrows,
                       0.5 * scale * scale, tw);
    MFIC_LAUNCH_CHECK();
}

template <typename T, int M, class PR>
static void launch_fused(mfic_ctx ctx, const void* in, void* out, long stride, int kc, long nrows, double scale,
                         const char* name) {
    constexpr int NI = PR::NF, NO = PR::NOF, NG = NI, SL = lane_slot<Plan<M>::P>();
    constexpr int RB = fused_rows_per_block<M, NG>(), RP = row_lds_pitch<M>();
    MFIC_CHECK(3 * (kc - 1) == 2 * M, MFIC_ERR_SIZE, "half-spectrum rows must hold N/2 + 1 values of a 3N/2 padded row");
    const size_t lds = (size_t)RB * NI * RP * sizeof(cx<T>);
    MFIC_CHECK(lds <= (size_t)ctx->max_lds, MFIC_ERR_SIZE, "fused row pass exceeds the LDS of a workgroup");
    const cx<T>* tw = static_cast<const cx<T>*>(twiddles(ctx, M, 1, sizeof(T) == 8 ? MFIC_F64 : MFIC_F32));
    // the output transforms' own plan (row plan 2) where the pass uses one
    const cx<T>* tw2 = (PR::OUT32 && row_alt_plan<M>() == 2 && RB == 1)
                           ? static_cast<const cx<T>*>(twiddles(ctx, M, 1, sizeof(T) == 8 ? MFIC_F64 : MFIC_F32, 2))
                           : tw;
    dim3 grid((unsigned)xcd_grid((nrows + RB - 1) / RB));
    ProfScope prof(ctx, std::string(name) + "_n" + std::to_string(2 * M) + (sizeof(T) == 8 ? "_f64" : "_f32"),
                   (double)nrows * (NI + NO) * kc * sizeof(cx<T>));
    hipLaunchKernelGGL((k_rows_fused<T, M, PR>), grid, dim3(RB * NG * SL), lds, ctx->stream,
                       static_cast<const cx<T>*>(in), stride, static_cast<cx<T>*>(out), stride, kc, nrows, (T)scale,
                       tw, tw2);
    MFIC_LAUNCH_CHECK();
}

// Last c2r pass of the three displacement (or velocity) components fused
// with the lattice readout (particle_generator.hh:499-544, 597-639): each
// group transforms one component row in LDS, then the row's particles are
// written as interleaved FP64 [p][3], q + Psi for positions
// ((ijk + shift)/N * lunit per axis, grid_fft.hh:242-252, not wrapped) or Psi
// for velocities.  blockIdx.y takes the sets one after another.
struct ParticleSets { ParticleRows s[8]; };
template <typename T, int M>
__global__ void __launch_bounds__((fused_rows_per_block<M, 3>() * 3 * lane_slot<Plan<M>::P>()))
k_rows_c2r_particles(ParticleSets sets, long nrows, T scale, const cx<T>* __restrict__ tw, double lunit) {
    constexpr int E = Plan<M>::E, P = Plan<M>::P, SL = lane_slot<P>(), N = 2 * M;
    constexpr int RP = row_lds_pitch<M>(), RB = fused_rows_per_block<M, 3>(), TPR = 3 * SL;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int tr = threadIdx.x % TPR, rb = threadIdx.x / TPR;
    const int g = tr / SL, q = tr % SL;
    const long row = (long)blockIdx.x * RB + rb;
    const bool active = row < nrows;
    const LdsRowMap lm{(rb * 3 + g) * RP};
    const cx<T>* uw = tw + plan_tw_size<M>();
    if (q < P) {
        // the untangle's partner M - k is loaded from global memory beside k
        // (same cache lines), so it runs in registers without an LDS round
        // trip (4.96 -> 4.13 ms for the four 512^3 launches)
        const ParticleRows& ps = sets.s[blockIdx.y];
        const cx<T>* __restrict__ src = static_cast<const cx<T>*>(g == 0 ? ps.f[0] : (g == 1 ? ps.f[1] : ps.f[2])) +
                                        (active ? row : 0) * (long)(M + 1);
        cx<T> raw[E], rev[E], v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = q + P * e;
            raw[e] = active ? src[k] : cx<T>{0, 0};
            rev[e] = active ? src[M - k] : cx<T>{0, 0};
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = q + P * e;
            cx<T> xk = raw[e], xm = rev[e];
            if (k == 0) { xk.y = 0; xm.y = 0; }  // kz = 0 and the Nyquist M are real
            const cx<T> A = {xk.x + xm.x, xk.y - xm.y};
            const cx<T> D = {xk.x - xm.x, xk.y + xm.y};
            const cx<T> B = cmulc(D, uw[k]);
            v[e] = cx<T>{A.x - B.y, A.y + B.x};
        }
        fft_regs_row<T, M, false, WaveSync>(v, q, lds, lm.base, tw);
#pragma unroll
        for (int e = 0; e < E; ++e) lds[lm.at(q + P * e)] = cscale(v[e], scale);
    }
    __syncthreads();
    if (!active) return;
    const int i = (int)(row / N), j = (int)(row % N);
    const bool is_pos = sets.s[blockIdx.y].is_pos != 0;
    const double sh0 = sets.s[blockIdx.y].shift[0], sh1 = sets.s[blockIdx.y].shift[1], sh2 = sets.s[blockIdx.y].shift[2];
    double* __restrict__ out = sets.s[blockIdx.y].dst + 3 * (size_t)row * N;
    for (int idx = tr; idx < 3 * N; idx += TPR) {
        const int p = idx / 3, c = idx - 3 * p;
        const cx<T> w = lds[(rb * 3 + c) * RP + (p >> 1)];
        double val = (double)((p & 1) ? w.y : w.x);
        if (is_pos) {
            const int ijk = c == 0 ? i : (c == 1 ? j : p);
            const double sh = c == 0 ? sh0 : (c == 1 ? sh1 : sh2);
            val = (((double)ijk + sh) / (double)N) * lunit + val;
        }
        out[idx] = val;
    }
}

template <typename T, int M>
static void launch_particles(mfic_ctx ctx, const ParticleSets& sets, int count, double lunit) {
    constexpr int SL = lane_slot<Plan<M>::P>(), RB = fused_rows_per_block<M, 3>(), RP = row_lds_pitch<M>();
    const long nrows = (long)(2 * M) * (2 * M);
    const size_t lds = (size_t)RB * 3 * RP * sizeof(cx<T>);
    MFIC_CHECK(lds <= (size_t)ctx->max_lds, MFIC_ERR_SIZE, "particle row pass exceeds the LDS of a workgroup");
    const cx<T>* tw = static_cast<const cx<T>*>(twiddles(ctx, M, 1, sizeof(T) == 8 ? MFIC_F64 : MFIC_F32));
    const double N = 2.0 * M;
    ProfScope prof(ctx, std::string("rows_c2r_particles_n") + std::to_string(2 * M) + (sizeof(T) == 8 ? "_f64" : "_f32"),
                   (double)nrows * (3.0 * (M + 1) * sizeof(cx<T>) + 3.0 * 2 * M * 8.0) * count);
    const dim3 grid((unsigned)((nrows + RB - 1) / RB), count);
    hipLaunchKernelGGL((k_rows_c2r_particles<T, M>), grid, dim3(RB * 3 * SL), lds, ctx->stream, sets, nrows,
                       (T)(1.0 / std::sqrt(N * N * N)), tw, lunit);
    MFIC_LAUNCH_CHECK();
}

#define MFIC_PARTICLE_ROWS(X) X(8) X(12) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384)

template <typename T>
void particle_rows(mfic_ctx ctx, const ParticleRows* sets, int count, int n, double lunit) {
    MFIC_CHECK(count >= 1 && count <= 8, MFIC_ERR_ARG, "one to eight particle sets");
    ParticleSets ps{};
    for (int m = 0; m < count; ++m) ps.s[m] = sets[m];
    switch (n / 2) {
#define X(M) case M: launch_particles<T, M>(ctx, ps, count, lunit); break;
        MFIC_PARTICLE_ROWS(X)
#undef X
    default:
        throw Error(MFIC_ERR_SIZE, "unsupported particle grid size " + std::to_string(n));
    }
}

#ifndef MFIC_FUSED_SIZES
#define MFIC_FUSED_SIZES(X) X(12) X(18) X(24) X(36) X(48) X(72) X(96) X(144) X(192) X(288) X(384) X(576) X(768)
#endif

template <typename T, class PR, bool HALF>
static void fused_t(mfic_ctx ctx, size_t n, const void* in, void* out, const char* name) {
    const int N = (int)n, np = 3 * N / 2, kc = N / 2 + 1;
    const long stride = (long)np * np * kc, rows = (long)np * np;
    const double norm = 1.0 / std::sqrt((double)np * (double)np * (double)np);
    // form 0 (default): two rows per full-length transform; form 1 (LPT
    // sources only): one half-length transform per row
    const bool paired = !HALF || plan_variant(ctx, np, MFIC_PASS_FUSED_ROWS, sizeof(T) == 8 ? MFIC_F64 : MFIC_F32) == 0;
    switch (np) {
#define X(S)                                                                                    \
    case S:                                                                                     \
        if (paired) launch_fused_pair<T, S, PR>(ctx, in, out, stride, kc, rows, norm, name);    \
        else if constexpr (HALF) launch_fused<T, S / 2, PR>(ctx, in, out, stride, kc, rows, norm, name); \
        break;
        MFIC_FUSED_SIZES(X)
#undef X
    default:
        throw Error(MFIC_ERR_SIZE, "unsupported padded size " + std::to_string(np));
    }
}

template <typename T> void fused_rows(mfic_ctx ctx, FusedKind kind, size_t n, const void* in, void* out) {
    switch (kind) {
    case FusedKind::Src2: fused_t<T, ProdSrc2, true>(ctx, n, in, out, "fused_src2"); break;
    case FusedKind::Src2Q: fused_t<T, ProdSrc2Q, true>(ctx, n, in, out, "fused_src2q"); break;
    case FusedKind::Src3: fused_t<T, ProdSrc3, true>(ctx, n, in, out, "fused_src3"); break;
    case FusedKind::Mul: fused_t<T, ProdMul, false>(ctx, n, in, out, "fused_mul"); break;
    case FusedKind::Square: fused_t<T, ProdSquare, false>(ctx, n, in, out, "fused_square"); break;
    case FusedKind::Adjoint2: fused_t<T, ProdAdjoint2, false>(ctx, n, in, out, "fused_adjoint2"); break;
    }
}

#define MFIC_FUSED_T(MODE, T)                                                                                        \
    MODE template void particle_rows<T>(mfic_ctx, const ParticleRows*, int, int, double);                            \
    MODE template void fused_rows<T>(mfic_ctx, FusedKind, size_t, const void*, void*);

#if MFIC_UNIT == 64
MFIC_FUSED_T(, double)
#else
MFIC_FUSED_T(extern, double)

void rows_c2r_particles(mfic_ctx ctx, int prec, const ParticleRows* sets, int count, int n, double lunit) {
    if (prec == MFIC_F64) particle_rows<double>(ctx, sets, count, n, lunit);
    else particle_rows<float>(ctx, sets, count, n, lunit);
}

void fused_source_rows(mfic_ctx ctx, int prec, FusedKind kind, size_t n, const void* in, void* out) {
    if (prec == MFIC_F64) fused_rows<double>(ctx, kind, n, in, out);
    else fused_rows<float>(ctx, kind, n, in, out);
}
#endif

}  // namespace mfic
