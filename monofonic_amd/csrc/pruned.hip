// Pruned and fused 3/2-padded transforms for the Orszag products
// (convolution.hh:495-651) on gfx950.
//
// The padded spectrum of an N-grid operand is nonzero only for source rows
// (i, j in [0, N/2] U (N, 3N/2)) and kz <= N/2, and the truncation keeps
// exactly those modes again.  So:
//   c2r  A: axis-0 pass over the (j, kz <= N/2) source columns, reading the
//           N-grid operand (Hessian / gradient / identity evaluated on the fly,
//           x (3/2)^{3/2}) and writing the full padded axis;
//        B: axis-1 pass over (i', kz <= N/2), the zero band of j' is not read;
//   the contiguous axis, the products and the transform back along it are one
//   fused row pass (fused.hip), which reads and writes kz <= N/2 only;
//   r2c  B': axis-1 pass, only the kept j' written;
//        A': axis-0 pass, only the kept i' written straight into the N-grid
//           with the unpad rules (Nyquist planes zeroed, / (3/2)^{3/2}), the
//           output operator and optionally -1/k^2.
// Padded k-space intermediates use a compact [Np][Np][N/2+1] layout.  Every
// skipped element is an exact zero of the unpruned algorithm, and every
// dropped output is one the unpad discards, so results equal the full
// transforms up to rounding order.
//
// One launch takes all the fields a pass runs over (members: blockIdx.y,
// consecutive compact buffers), so that small grids fill the chip and large
// ones pay one tail; the members of a launch run one after another, in the
// order of separate launches.
//
// This file is compiled once per precision (MFIC_UNIT 32 or 64).
#include <algorithm>
#include <cmath>

#include "fft_core.hpp"
#include "mfic_internal.hpp"
#include "pruned.hpp"

namespace mfic {

// ---------------------------------------------------------- loaders / stores
//
// Every padded pass runs pencils of length L = 3N/2 and every loader and
// store below is instantiated with that L, so N, N/2 + 1 and the strides are
// compile-time constants.  Element e of a pencil sits on lane q at position
// pos = q + P e; once the element loop is unrolled, which side of the zero
// band it lies on is a constant for all lanes except the two elements that
// straddle N/2 and N, so band tests and gradient factors cost nothing for the
// others.

template <int L, int V = 0> struct PadGeo {
    static constexpr int P = Plan<L, V>::P, N = 2 * L / 3, NH = N / 2, KC = NH + 1;
    static_assert(3 * N == 2 * L, "padded length must be 3N/2");
    // 0: every lane below N/2, 1: every lane above N, 2: every lane in the
    // zero band N/2 < pos <= N, 3: mixed
    static __device__ __forceinline__ constexpr int side(int e) {
        return P * e + P - 1 < NH ? 0 : (P * e > N ? 1 : (P * e > NH && P * e + P - 1 <= N ? 2 : 3));
    }
    static __device__ __forceinline__ bool band(int q, int e) {
        const int pos = q + P * e;
        const int sd = side(e);
        return sd == 2 || (sd == 3 && pos > NH && pos <= N);
    }
    // source index behind pos (convolution.hh:562-571), -1 in the band
    static __device__ __forceinline__ int src(int q, int e) {
        const int pos = q + P * e;
        switch (side(e)) {
        case 0: return pos;
        case 1: return pos - NH;
        case 2: return -1;
        default: return pos <= NH ? pos : (pos > N ? pos - NH : -1);
        }
    }
    // gradient factor of the source mode behind pos: signed index times kf,
    // 0 at the source Nyquist N/2 (never used in the band)
    template <typename T> static __device__ __forceinline__ T grad(int q, int e, T kf) {
        const int pos = q + P * e;
        switch (side(e)) {
        case 0: return (T)q * kf + (T)(P * e) * kf;
        case 1: return (T)q * kf + (T)(P * e - L) * kf;
        default: return pos == NH ? T(0) : (T)(pos - (pos > NH ? L : 0)) * kf;
        }
    }
};

// gradient factor of an unpadded index
template <typename T> __device__ __forceinline__ T grad_t(int idx, int n, T kf) {
    return idx == n / 2 ? T(0) : (T)(idx - (idx > n / 2) * n) * kf;
}

// pass A: operand of an N-grid k-space field.  Along a pencil only the
// axis-0 gradient g_i varies, so every operand multiplier is a polynomial
// s(g_i) = (alpha g_i + beta) g_i + gamma fixed per column (imaginary for a
// single gradient); the (3/2)^{3/2} pad factor is folded in.
template <typename T> struct LdOperand {
    struct Op { const cx<T>* f; int kind, d0, d1, d2, d3; };
    Op op[2];
    double kf[3], scale;  // 2 pi / L of each axis
    struct Col { const cx<T>* p; double al, be, ga; bool imag; };
    // product -(g_a g_b) as polynomial coefficients in g_i
    __device__ __forceinline__ static void prod2(int a, int b, double gj, double gk, double sg, double& al, double& be,
                                                 double& ga) {
        const double ga_ = a == 1 ? gj : gk, gb_ = b == 1 ? gj : gk;
        if (a == 0 && b == 0) al += -sg;
        else if (a == 0) be += -sg * gb_;
        else if (b == 0) be += -sg * ga_;
        else ga += -sg * (ga_ * gb_);
    }
    template <int L> __device__ __forceinline__ Col column(long col, int m) const {
        using G = PadGeo<L>;
        Col c;
        const int j = (int)(col / G::KC), k = (int)(col % G::KC);
        const Op o = op[m];
        const int d0 = o.d0, d1 = o.d1, d2 = o.d2, d3 = o.d3;
        c.p = o.f + col;
        const double gj = grad_t<double>(j, G::N, kf[1]), gk = grad_t<double>(k, G::N, kf[2]);
        c.al = c.be = c.ga = 0.0;
        c.imag = false;
        switch (o.kind) {
        case MFIC_OPND_HESS: prod2(d0, d1, gj, gk, 1.0, c.al, c.be, c.ga); break;
        case MFIC_OPND_SUM_HESS:
            prod2(d0, d1, gj, gk, 1.0, c.al, c.be, c.ga);
            prod2(d2, d3, gj, gk, 1.0, c.al, c.be, c.ga);
            break;
        case MFIC_OPND_DIFF_HESS:
            prod2(d0, d1, gj, gk, 1.0, c.al, c.be, c.ga);
            prod2(d2, d3, gj, gk, -1.0, c.al, c.be, c.ga);
            break;
        case MFIC_OPND_GRAD:
            c.imag = true;
            if (d0 == 0) c.be = 1.0; else c.ga = d0 == 1 ? gj : gk;
            break;
        default: c.ga = 1.0; break;
        }
        c.al *= scale;
        c.be *= scale;
        c.ga *= scale;
        return c;
    }
    template <int L, int V = 0> __device__ __forceinline__ cx<T> load(const Col& c, int q, int e) const {
        using G = PadGeo<L, V>;
        const int i = G::src(q, e);
        return i < 0 ? cx<T>{0, 0} : c.p[(long)i * (G::N * G::KC)];
    }
    template <int L, int V = 0> __device__ __forceinline__ cx<T> fix(const Col& c, int q, int e, cx<T> v) const {
        using G = PadGeo<L, V>;
        if (G::band(q, e)) return v;
        const double g = G::template grad<double>(q, e, kf[0]);
        const double s = (c.al * g + c.be) * g + c.ga;
        return c.imag ? cx<T>{(T)(-s * (double)v.y), (T)(s * (double)v.x)}
                      : cx<T>{(T)(s * (double)v.x), (T)(s * (double)v.y)};
    }
};
// pass A store: padded column (j' = pad(j)) of the compact k buffer
template <typename T> struct StPadCol {
    cx<T>* kb;
    struct Col { cx<T>* p; };
    template <int L> __device__ __forceinline__ Col column(long col, int m) const {
        using G = PadGeo<L>;
        const int j = (int)(col / G::KC), k = (int)(col % G::KC);
        return Col{kb + m * (long)(L * G::KC) * L + (long)(j > G::NH ? j + G::NH : j) * G::KC + k};
    }
    template <int L, int V = 0> __device__ __forceinline__ void store(const Col& c, int q, int e, cx<T> v) const {
        using G = PadGeo<L, V>;
        c.p[(long)(q + G::P * e) * (L * G::KC)] = v;
    }
};
// passes B / B': axis-1 pencils of the compact buffer, column = (i', kz)
template <typename T, bool SKIP_BAND> struct LdAx1 {
    const cx<T>* kb;
    struct Col { const cx<T>* p; };
    template <int L> __device__ __forceinline__ Col column(long col, int m) const {
        using G = PadGeo<L>;
        const long ip = col / G::KC, k = col % G::KC;
        return Col{kb + m * (long)(L * G::KC) * L + ip * (L * G::KC) + k};
    }
    template <int L, int V = 0> __device__ __forceinline__ cx<T> load(const Col& c, int q, int e) const {
        using G = PadGeo<L, V>;
        if (SKIP_BAND && G::band(q, e)) return cx<T>{0, 0};
        return c.p[(long)(q + G::P * e) * G::KC];
    }
    template <int L, int V = 0> __device__ __forceinline__ cx<T> fix(const Col&, int, int, cx<T> v) const { return v; }
};
template <typename T, bool DROP_BAND> struct StAx1 {
    cx<T>* kb;
    struct Col { cx<T>* p; };
    template <int L> __device__ __forceinline__ Col column(long col, int m) const {
        using G = PadGeo<L>;
        const long ip = col / G::KC, k = col % G::KC;
        return Col{kb + m * (long)(L * G::KC) * L + ip * (L * G::KC) + k};
    }
    template <int L, int V = 0> __device__ __forceinline__ void store(const Col& c, int q, int e, cx<T> v) const {
        using G = PadGeo<L, V>;
        if (DROP_BAND && G::band(q, e)) return;
        c.p[(long)(q + G::P * e) * G::KC] = v;
    }
};
// pass A' load: padded column of the compact buffer for kept j
template <typename T> struct LdPadCol {
    const cx<T>* kb;
    struct Col { const cx<T>* p; };
    template <int L> __device__ __forceinline__ Col column(long col, int m) const {
        using G = PadGeo<L>;
        const int j = (int)(col / G::KC), k = (int)(col % G::KC);
        return Col{kb + m * (long)(L * G::KC) * L + (long)(j > G::NH ? j + G::NH : j) * G::KC + k};
    }
    template <int L, int V = 0> __device__ __forceinline__ cx<T> load(const Col& c, int q, int e) const {
        using G = PadGeo<L, V>;
        return c.p[(long)(q + G::P * e) * (L * G::KC)];
    }
    template <int L, int V = 0> __device__ __forceinline__ cx<T> fix(const Col&, int, int, cx<T> v) const { return v; }
};
// pass A' store: unpad rules + output operator (+ optional -1/k^2) into the N-grid
template <typename T> struct StUnpad {
    cx<T>* out[4];
    int op, invlap;
    double scale, coef, kf;
    struct Col { cx<T>* p; double kj, kk; bool nyq; };
    template <int L> __device__ __forceinline__ Col column(long col, int m) const {
        using G = PadGeo<L>;
        Col c;
        const int j = (int)(col / G::KC), k = (int)(col % G::KC);
        c.p = out[m] + col;
        c.kj = ((double)j - (double)(j > G::NH) * G::N) * kf;
        c.kk = ((double)k - (double)(k > G::NH) * G::N) * kf;
        c.nyq = (j == G::NH) || (k == G::NH);
        return c;
    }
    template <int L, int V = 0> __device__ __forceinline__ void store(const Col& c, int q, int e, cx<T> v) const {
        using G = PadGeo<L, V>;
        const int i = G::src(q, e);
        if (i < 0) return;
        double re = 0.0, im = 0.0;
        if (!(c.nyq || i == G::NH)) {
            double f = scale;
            if (invlap) {  // one FP64 division per element, shared by both parts
                const double ki = G::template grad<double>(q, e, kf);
                const double k2 = ki * ki + c.kj * c.kj + c.kk * c.kk;
                f = k2 > 0.0 ? -scale / k2 : 0.0;
            }
            re = (double)v.x * f;
            im = (double)v.y * f;
        }
        cx<T>* dst = c.p + (long)i * (G::N * G::KC);
        if (op == MFIC_OP_ASSIGN) { *dst = cx<T>{(T)re, (T)im}; return; }
        const cx<T> o = *dst;
        if (op == MFIC_OP_ADD) *dst = cx<T>{(T)((double)o.x + re), (T)((double)o.y + im)};
        else if (op == MFIC_OP_SUB) *dst = cx<T>{(T)((double)o.x - re), (T)((double)o.y - im)};
        else *dst = cx<T>{(T)((double)o.x + re * coef), (T)((double)o.y + im * coef)};
    }
};
// axis-0 pencils of the compact buffer over every row j', column = (j', kz)
template <typename T> struct LdAx0 {
    const cx<T>* kb;
    struct Col { const cx<T>* p; };
    template <int L> __device__ __forceinline__ Col column(long col, int m) const {
        return Col{kb + m * (long)(L * PadGeo<L>::KC) * L + col};
    }
    template <int L, int V = 0> __device__ __forceinline__ cx<T> load(const Col& c, int q, int e) const {
        using G = PadGeo<L, V>;
        return c.p[(long)(q + G::P * e) * (L * G::KC)];
    }
};
template <typename T> struct StAx0 {
    cx<T>* kb;
    struct Col { cx<T>* p; };
    template <int L> __device__ __forceinline__ Col column(long col, int m) const {
        return Col{kb + m * (long)(L * PadGeo<L>::KC) * L + col};
    }
    template <int L, int V = 0> __device__ __forceinline__ void store(const Col& c, int q, int e, cx<T> v) const {
        using G = PadGeo<L, V>;
        c.p[(long)(q + G::P * e) * (L * G::KC)] = v;
    }
};

// ------------------------------------------------------------- kernels ----

template <typename T, int L, int TK, bool FWD, class LD, class ST, int V = 0>
__global__ void __launch_bounds__((Plan<L, V>::P * TK))
k_pencils_f(LD ld, ST st, long ncols, const cx<T>* __restrict__ tw, int xcd) {
    constexpr int E = Plan<L, V>::E;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int t = threadIdx.x % TK, q = threadIdx.x / TK, m = blockIdx.y;
    using Tw = PencilTw<T, L, V, Plan<L, V>::P * TK>;
    Tw tws;
    tws.load(tw);
    const long col = (xcd ? xcd_tile(blockIdx.x, gridDim.x) : (long)blockIdx.x) * TK + t;
    const bool active = col < ncols;
    const long c = active ? col : 0;
    const auto lc = ld.template column<L>(c, m);
    cx<T> v[E];
    // every load of the pencil is issued before any multiplier is applied;
    // lanes past the last column read column 0 and store nothing, so no load
    // carries a branch
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = ld.template load<L, V>(lc, q, e);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = ld.template fix<L, V>(lc, q, e, v[e]);
    const cx<T>* ltw = tws.store(lds, L * TK, tw);
    fft_pencil<T, L, FWD, V, Tw::LDS>(v, q, lds, LdsMap{t, TK}, ltw);
    if (active) {
        const auto sc = st.template column<L>(c, m);
#pragma unroll
        for (int e = 0; e < E; ++e) st.template store<L, V>(sc, q, e, v[e]);
    }
}

// The six Hessians (xx yy zz xy xz yz) of an N-grid field factorise per axis:
// -g_a g_b = -(g_i^p)(g_j^q)(g_k^r).  Pass A makes one buffer per x power p,
// pass B one buffer per Hessian from the buffer of its p.  In pass order the
// Hessians are yy zz yz (p = 0), xy xz (1), xx (2).
struct HessOrder {
    // slot, p, q, r of entry i, two bits (slot: four) each
    static __device__ __forceinline__ int slot(int i) { return (0x043521 >> (4 * i)) & 15; }
    static __device__ __forceinline__ int p(int i) { return i < 3 ? 0 : (i < 5 ? 1 : 2); }
    static __device__ __forceinline__ int q(int i) { return i == 0 ? 2 : (i == 2 || i == 3 ? 1 : 0); }
    static __device__ __forceinline__ int r(int i) { return i == 1 ? 2 : (i == 2 || i == 4 ? 1 : 0); }
    // entries of member y: every x power by itself (3 members) or every
    // Hessian by itself (6)
    static __device__ __forceinline__ int first(int y, int ny) { return ny == 6 ? y : (y == 0 ? 0 : (y == 1 ? 3 : 5)); }
    static __device__ __forceinline__ int last(int y, int ny) { return ny == 6 ? y + 1 : (y == 0 ? 3 : (y == 1 ? 5 : 6)); }
};

// A workgroup reads a tile of source pencils once and makes the outputs of
// all x powers (gridDim.y = 1) or one (3).  KEEP holds the pencil in
// registers for the next power; else it is read again, from cache.  The weights
// are formed and applied in W: T for the LPT sources, FP64 for the 2LPT adjoint
// (256^3 FP32: pass A 110 us against 98, pass B 314 against 313).
template <typename T, typename W, int L, int TK, int V, bool KEEP>
__global__ void __launch_bounds__((Plan<L, V>::P * TK))
k_hess_a(const cx<T>* __restrict__ f, StPadCol<T> st, long ncols, W kf, W scale, const cx<T>* __restrict__ tw) {
    using G = PadGeo<L, V>;
    constexpr int E = Plan<L, V>::E;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int t = threadIdx.x % TK, q = threadIdx.x / TK;
    using Tw = PencilTw<T, L, V, Plan<L, V>::P * TK>;
    Tw tws;
    tws.load(tw);
    const long col = (long)blockIdx.x * TK + t;
    const bool active = col < ncols;
    const cx<T>* src = f + (active ? col : 0);
    cx<T> raw[KEEP ? E : 1];
    auto load = [&](int e) {
        const int i = G::src(q, e);
        return i < 0 ? cx<T>{0, 0} : src[(long)i * (G::N * G::KC)];
    };
    if constexpr (KEEP) {
#pragma unroll
        for (int e = 0; e < E; ++e) raw[e] = load(e);
    }
    const int top = gridDim.y == 1 ? 2 : 2 - (int)blockIdx.y, end = gridDim.y == 1 ? 0 : top;
    const cx<T>* ltw = tws.store(lds, L * TK, tw);
#pragma unroll 1
    for (int p = top; p >= end; --p) {
        cx<T> v[E];
        if constexpr (!KEEP) {
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = load(e);
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const W g = G::template grad<W>(q, e, kf);
            const W m = scale * (p > 0 ? g : W(1)) * (p > 1 ? g : W(1));
            const cx<T> x = KEEP ? raw[KEEP ? e : 0] : v[e];
            v[e] = cx<T>{(T)(m * x.x), (T)(m * x.y)};
        }
        fft_pencil<T, L, false, V, Tw::LDS>(v, q, lds, LdsMap{t, TK}, ltw);
        if (active) {
            const auto sc = st.template column<L>(col, p);
#pragma unroll
            for (int e = 0; e < E; ++e) st.template store<L, V>(sc, q, e, v[e]);
        }
    }
}

// Pass B: g_j^q along the pencil (zero band skipped) times the per-column
// factor -g_k^r; gridDim.y = 3 reads the pencils of an x power once for all
// its Hessians, 6 takes each Hessian by itself.
template <typename T, typename W, int L, int TK, int V, bool KEEP>
__global__ void __launch_bounds__((Plan<L, V>::P * TK))
k_hess_b(LdAx1<T, true> ld, StAx1<T, false> st, long ncols, W kf, const cx<T>* __restrict__ tw) {
    using G = PadGeo<L, V>;
    constexpr int E = Plan<L, V>::E;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int t = threadIdx.x % TK, q = threadIdx.x / TK;
    using Tw = PencilTw<T, L, V, Plan<L, V>::P * TK>;
    Tw tws;
    tws.load(tw);
    const long col = xcd_tile(blockIdx.x, gridDim.x) * TK + t;
    const bool active = col < ncols;
    const long c = active ? col : 0;
    const int first = HessOrder::first(blockIdx.y, gridDim.y), last = HessOrder::last(blockIdx.y, gridDim.y);
    const auto lc = ld.template column<L>(c, HessOrder::p(first));
    const W gk = grad_t<W>((int)(c % G::KC), G::N, kf);
    cx<T> raw[KEEP ? E : 1];
    if constexpr (KEEP) {
#pragma unroll
        for (int e = 0; e < E; ++e) raw[e] = ld.template load<L, V>(lc, q, e);
    }
    const cx<T>* ltw = tws.store(lds, L * TK, tw);
#pragma unroll 1
    for (int i = first; i < last; ++i) {
        const int pq = HessOrder::q(i), pr = HessOrder::r(i);
        const W cm = pr == 0 ? W(-1) : (pr == 1 ? W(-1) * gk : W(-1) * (gk * gk));
        cx<T> v[E];
        if constexpr (!KEEP) {
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = ld.template load<L, V>(lc, q, e);
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const W g = G::template grad<W>(q, e, kf);
            const W m = cm * (pq > 0 ? g : W(1)) * (pq > 1 ? g : W(1));
            const cx<T> x = KEEP ? raw[KEEP ? e : 0] : v[e];
            v[e] = cx<T>{(T)(m * x.x), (T)(m * x.y)};
        }
        fft_pencil<T, L, false, V, Tw::LDS>(v, q, lds, LdsMap{t, TK}, ltw);
        if (active) {
            const auto sc = st.template column<L>(c, HessOrder::slot(i));
#pragma unroll
            for (int e = 0; e < E; ++e) st.template store<L, V>(sc, q, e, v[e]);
        }
    }
}

// Adjoint of the Hessian passes, for sum_h D_h T(r_h) with D_h = -g_a g_b and
// six real fields r_h given as r2c'd rows (slot order as the Hessians).  The
// factors separate per axis, so pass B' sums the fields of an x power after
// their axis-1 transforms, weighted by -g_j^q g_k^r, and pass A' the three
// sums after theirs, weighted by g_i^p: three axis-0 transforms and one write
// of the result for six of each.  Weights and multiply-adds are FP64, the sums
// are rounded to T at each addition, as sums kept in memory field by field
// would be (FP64 sums put pass B' on one wave a SIMD: forward and adjoint 3.74
// ms against 3.57).  Bound by memory: at 256^3 FP32 pass B' 270 us (4.5 TB/s)
// for six fields, pass A' 159 us (2.8 TB/s; 16 columns to a tile), where one
// field took 63 + 45 us and 58 us for its weighted sum.
template <typename T, int L, int TK, int V>
__global__ void __launch_bounds__((Plan<L, V>::P * TK))
k_hess_bt(LdAx1<T, false> ld, StAx1<T, true> st, long ncols, double kf, const cx<T>* __restrict__ tw) {
    using G = PadGeo<L, V>;
    constexpr int E = Plan<L, V>::E;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int t = threadIdx.x % TK, q = threadIdx.x / TK;
    using Tw = PencilTw<T, L, V, Plan<L, V>::P * TK>;
    Tw tws;
    tws.load(tw);
    const long col = xcd_tile(blockIdx.x, gridDim.x) * TK + t;
    const bool active = col < ncols;
    const long c = active ? col : 0;
    const int first = HessOrder::first(blockIdx.y, 3), last = HessOrder::last(blockIdx.y, 3);
    const double gk = grad_t<double>((int)(c % G::KC), G::N, kf);
    cx<T> acc[E];
#pragma unroll
    for (int e = 0; e < E; ++e) acc[e] = cx<T>{0, 0};
    const cx<T>* ltw = tws.store(lds, L * TK, tw);
#pragma unroll 1
    for (int i = first; i < last; ++i) {
        const int pq = HessOrder::q(i), pr = HessOrder::r(i);
        const double cm = pr == 0 ? -1.0 : (pr == 1 ? -gk : -(gk * gk));
        const auto lc = ld.template column<L>(c, HessOrder::slot(i));
        cx<T> v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = ld.template load<L, V>(lc, q, e);
        fft_pencil<T, L, true, V, Tw::LDS>(v, q, lds, LdsMap{t, TK}, ltw);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const double g = G::template grad<double>(q, e, kf);  // band elements are not stored
            const double m = cm * (pq > 0 ? g : 1.0) * (pq > 1 ? g : 1.0);
            acc[e] = cx<T>{(T)(acc[e].x + m * v[e].x), (T)(acc[e].y + m * v[e].y)};
        }
    }
    if (active) {
        const auto sc = st.template column<L>(c, HessOrder::p(first));
#pragma unroll
        for (int e = 0; e < E; ++e) st.template store<L, V>(sc, q, e, acc[e]);
    }
}
// out = F(|n|^2) / volfac * (g1 lam + scale * sum_p g_i^p (pass A' of slot p)),
// Nyquist planes zeroed: F is the -A(k)/k^2 table of phi1
template <typename T> struct AdjointOut {
    cx<T>* out;
    const cx<T>* lam;
    const double* tab;
    double g1, scale, volfac;
};
template <typename T, int L, int TK, int V>
__global__ void __launch_bounds__((Plan<L, V>::P * TK))
k_hess_at(LdPadCol<T> ld, AdjointOut<T> o, long ncols, double kf, const cx<T>* __restrict__ tw) {
    using G = PadGeo<L, V>;
    constexpr int E = Plan<L, V>::E;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int t = threadIdx.x % TK, q = threadIdx.x / TK;
    using Tw = PencilTw<T, L, V, Plan<L, V>::P * TK>;
    Tw tws;
    tws.load(tw);
    const long col = (long)blockIdx.x * TK + t;
    const bool active = col < ncols;
    const long c = active ? col : 0;
    cx<T> acc[E];
#pragma unroll
    for (int e = 0; e < E; ++e) acc[e] = cx<T>{0, 0};
    const cx<T>* ltw = tws.store(lds, L * TK, tw);
#pragma unroll 1
    for (int p = 0; p < 3; ++p) {
        const auto lc = ld.template column<L>(c, p);
        cx<T> v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = ld.template load<L, V>(lc, q, e);
        fft_pencil<T, L, true, V, Tw::LDS>(v, q, lds, LdsMap{t, TK}, ltw);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const double g = G::template grad<double>(q, e, kf);
            const double m = (p > 0 ? g : 1.0) * (p > 1 ? g : 1.0);
            acc[e] = cx<T>{(T)(acc[e].x + m * v[e].x), (T)(acc[e].y + m * v[e].y)};
        }
    }
    if (!active) return;
    const int j = (int)(c / G::KC), k = (int)(c % G::KC), sj = j - (j > G::NH) * G::N;
    const bool nyq = j == G::NH || k == G::NH;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = G::src(q, e);
        if (i < 0) continue;
        const long at = (long)i * (G::N * G::KC) + c;
        cx<T> r = {0, 0};
        if (!nyq && i != G::NH) {
            const int si = i - (i > G::NH) * G::N;
            const double F = o.tab[si * si + sj * sj + k * k];
            const cx<T> l = o.lam[at];
            r = cx<T>{(T)((o.g1 * (double)l.x + o.scale * (double)acc[e].x) / o.volfac * F),
                      (T)((o.g1 * (double)l.y + o.scale * (double)acc[e].y) / o.volfac * F)};
        }
        o.out[at] = r;
    }
}

// Orszag truncation followed by re-padding along one axis of a compact
// padded buffer that is real-space along that axis: forward transform, keep
// the source modes (not the zero band, not the source Nyquist N/2), inverse
// transform.  Equal to the unpad (convolution.hh:600-651) then pad_insert
// (convolution.hh:552-594) pair of a two-stage product restricted to that
// axis; the column mask zeroes kz = N/2 and `scale` carries the pad factors.
template <typename T, int L, int TK, class LD, class ST, int V = 0>
__global__ void __launch_bounds__((Plan<L, V>::P * TK))
k_pencils_filter(LD ld, ST st, long ncols, const cx<T>* __restrict__ tw, int xcd, int zero_kz_nyquist, T scale) {
    using G = PadGeo<L, V>;
    constexpr int E = Plan<L, V>::E;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
    const int t = threadIdx.x % TK, q = threadIdx.x / TK, m = blockIdx.y;
    using Tw = PencilTw<T, L, V, Plan<L, V>::P * TK>;
    Tw tws;
    tws.load(tw);
    const long col = (xcd ? xcd_tile(blockIdx.x, gridDim.x) : (long)blockIdx.x) * TK + t;
    const bool active = col < ncols;
    const long c = active ? col : 0;
    const auto lc = ld.template column<L>(c, m);
    cx<T> v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = ld.template load<L, V>(lc, q, e);
    const cx<T>* ltw = tws.store(lds, L * TK, tw);
    fft_pencil<T, L, true, V, Tw::LDS>(v, q, lds, LdsMap{t, TK}, ltw);
    const bool colzero = zero_kz_nyquist && (int)(c % G::KC) == G::NH;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        // keep the source modes: not the zero band, not the source Nyquist
        const bool keep = !colzero && !G::band(q, e) && q + G::P * e != G::NH;
        v[e] = keep ? cscale(v[e], scale) : cx<T>{0, 0};
    }
    // a position of its own, so that the factors of the first transform do not
    // stay in registers for the second
    int q2 = q;
    if constexpr (Tw::LDS) asm("" : "+v"(q2));
    fft_pencil<T, L, false, V, Tw::LDS>(v, q2, lds, LdsMap{t, TK}, ltw);
    if (active) {
        const auto sc = st.template column<L>(c, m);
#pragma unroll
        for (int e = 0; e < E; ++e) st.template store<L, V>(sc, q, e, v[e]);
    }
}

// ------------------------------------------------------------- launchers --

// tile of a padded pass: the override of its own kind, else the override of
// every strided pass of the length (kind 0), else 128-byte row segments (16
// pencils in FP32, 8 in FP64).  Twice that at two lengths: 384 points in the
// passes with one output (`wide`), whose workgroups are small (16 threads to a
// transform, where the neighbouring lengths have 24 and 32), and 288 points in
// FP32, where the Hessian passes take 106 + 277 us per 192^3 3LPT box against
// 121 + 327.
// Against the widest tile of 68 KB, which this is at 768 points: the two r2c
// passes of four fields 84 -> 66 us at 192 points FP64, 42 -> 39 at 192 FP32.
// Tiles below 4 run as 4.
template <typename T, int L, int V>
static int pick_tile(mfic_ctx ctx, int pass, bool wide) {
    constexpr int P = Plan<L, V>::P;
    int tk = sizeof(T) == 8 ? 8 : 16;
    if ((wide && L == 384) || (sizeof(T) == 4 && L == 288)) tk *= 2;
    const int prec = sizeof(T) == 8 ? MFIC_F64 : MFIC_F32;
    auto ov = ctx->tiles.find(std::make_tuple(L, pass, prec));
    if (ov == ctx->tiles.end()) ov = ctx->tiles.find(std::make_tuple(L, 0, prec));
    if (ov != ctx->tiles.end()) tk = ov->second.first;
    while (tk > 4 && ((size_t)L * tk * sizeof(T) > 139264 || P * tk > 1024)) tk /= 2;
    return tk < 4 ? 4 : tk;
}

template <typename T, int L, int V> constexpr size_t pencil_lds(int tk) {
    return PencilTw<T, L, V, 64>::bytes((size_t)L * tk);
}

template <typename T> constexpr int prec_of() { return sizeof(T) == 8 ? MFIC_F64 : MFIC_F32; }
template <typename T, int L> static std::string pass_name(const char* name) {
    return std::string(name) + "_L" + std::to_string(L) + (sizeof(T) == 8 ? "_f64" : "_f32");
}

#define MFIC_TILE_SWITCH(P_, CALL)                 \
    switch (tk) {                                  \
    case 4: CALL(4) break;                         \
    case 8: CALL(8) break;                         \
    case 16: if constexpr (P_ * 16 <= 1024) { CALL(16) } break; \
    case 32: if constexpr (P_ * 32 <= 1024) { CALL(32) } break; \
    case 64: if constexpr (P_ * 64 <= 1024) { CALL(64) } break; \
    default: throw Error(MFIC_ERR_SIZE, "bad tile"); \
    }

template <typename T, int L, bool FWD, class LD, class ST, int V>
static void launch_fv(mfic_ctx ctx, int pass, const LD& ld, const ST& st, long ncols, int members, const char* name,
                      double bytes, bool xcd) {
    constexpr int P = Plan<L, V>::P;
    const int tk = pick_tile<T, L, V>(ctx, pass, true);
    const cx<T>* tw = static_cast<const cx<T>*>(twiddles(ctx, L, PencilTw<T, L, V, 64>::KIND, prec_of<T>(), V));
    const size_t lds = pencil_lds<T, L, V>(tk);
    // axis-1 passes: 16-column tiles of rows with an odd pitch share cache
    // lines with their neighbours, which the XCD-aware order keeps in one L2
    const long ntiles = (ncols + tk - 1) / tk;
    const dim3 grid((unsigned)(xcd ? xcd_grid(ntiles) : ntiles), members);
    ProfScope prof(ctx, pass_name<T, L>(name), bytes * members);
#define CALL(K)                                                                                                  \
    hipLaunchKernelGGL((k_pencils_f<T, L, K, FWD, LD, ST, V>), grid, dim3(P * K), lds, ctx->stream, ld, st, ncols, \
                       tw, xcd ? 1 : 0);
    MFIC_TILE_SWITCH(P, CALL)
#undef CALL
    MFIC_LAUNCH_CHECK();
}

// a strided padded pass with the radix plan selected for its kind (pass)
template <typename T, int L, bool FWD, class LD, class ST>
static void launch_f(mfic_ctx ctx, int pass, const LD& ld, const ST& st, long ncols, int members, const char* name,
                     double bytes, bool xcd = false) {
    if (plan_variant(ctx, L, pass, prec_of<T>()) == 1)
        launch_fv<T, L, FWD, LD, ST, alt_plan<L>()>(ctx, pass, ld, st, ncols, members, name, bytes, xcd);
    else
        launch_fv<T, L, FWD, LD, ST, 0>(ctx, pass, ld, st, ncols, members, name, bytes, xcd);
}

#ifndef MFIC_PADDED_SIZES
#define MFIC_PADDED_SIZES(X) X(12) X(18) X(24) X(36) X(48) X(72) X(96) X(144) X(192) X(288) X(384) X(576) X(768)
#endif
#define MFIC_PADDED_SWITCH(NP)                                                          \
    switch (NP) {                                                                       \
        MFIC_PADDED_SIZES(X)                                                            \
    default:                                                                            \
        throw Error(MFIC_ERR_SIZE, "unsupported padded size " + std::to_string(NP));    \
    }

template <typename T>
void operands_to_kbuf(mfic_ctx ctx, const OperandDesc* o, int count, size_t n, const double L[3], void* kbuf) {
    const int N = (int)n, np = 3 * N / 2, kc = N / 2 + 1;
    LdOperand<T> la{};
    for (int m = 0; m < count; ++m)
        la.op[m] = {static_cast<const cx<T>*>(o[m].f), o[m].kind, o[m].d[0], o[m].d[1], o[m].d[2], o[m].d[3]};
    for (int a = 0; a < 3; ++a) la.kf[a] = 2.0 * 3.14159265358979323846 / L[a];
    la.scale = std::pow(1.5, 1.5);
    StPadCol<T> sa{static_cast<cx<T>*>(kbuf)};
    LdAx1<T, true> lb{static_cast<const cx<T>*>(kbuf)};
    StAx1<T, false> sb{static_cast<cx<T>*>(kbuf)};
    const double cs = sizeof(cx<T>);
    const long colsA = (long)N * kc, colsB = (long)np * kc;
#define X(S)                                                                                                         \
    case S:                                                                                                          \
        launch_f<T, S, false>(ctx, MFIC_PASS_PAD_C2R_A, la, sa, colsA, count, "fft_c2rA", (double)colsA * (N + np) * cs); \
        launch_f<T, S, false>(ctx, MFIC_PASS_PAD_C2R_B, lb, sb, colsB, count, "fft_c2rB",                            \
                              (double)colsB * (N + np) * cs, true);                                                  \
        break;
    MFIC_PADDED_SWITCH(np)
#undef X
}

template <typename T>
void r2c_from_kbuf(mfic_ctx ctx, size_t n, double L, void* kbuf, int count, void* const* out, int op, double coef,
                   bool invlap) {
    const int N = (int)n, np = 3 * N / 2, kc = N / 2 + 1;
    const double rfac = std::sqrt((double)np * np * np) / std::sqrt((double)N * N * N);
    const double norm = 1.0 / std::sqrt((double)np * (double)np * (double)np);
    LdAx1<T, false> lb{static_cast<const cx<T>*>(kbuf)};
    StAx1<T, true> sb{static_cast<cx<T>*>(kbuf)};
    LdPadCol<T> la{static_cast<const cx<T>*>(kbuf)};
    StUnpad<T> sa{};
    for (int m = 0; m < count; ++m) sa.out[m] = static_cast<cx<T>*>(out[m]);
    sa.op = op;
    sa.invlap = invlap ? 1 : 0;
    sa.scale = norm / rfac;
    sa.coef = coef;
    sa.kf = 2.0 * 3.14159265358979323846 / L;
    const double cs = sizeof(cx<T>);
    const long colsA = (long)N * kc, colsB = (long)np * kc;
#define X(S)                                                                                                         \
    case S:                                                                                                          \
        launch_f<T, S, true>(ctx, MFIC_PASS_PAD_R2C_B, lb, sb, colsB, count, "fft_r2cB",                             \
                             (double)colsB * (np + N) * cs, true);                                                   \
        launch_f<T, S, true>(ctx, MFIC_PASS_PAD_R2C_A, la, sa, colsA, count, "fft_r2cA",                             \
                             (double)colsA * (np + N * (op == MFIC_OP_ASSIGN ? 1 : 2)) * cs);                        \
        break;
    MFIC_PADDED_SWITCH(np)
#undef X
}

// Hessian passes keep the source pencil in registers where it and the one
// being transformed take at most 192 of them: against reading it again for
// each output, pass B of 512^3 FP32 2.92 -> 2.68 ms, 256^3 FP64 712 -> 636 us
template <typename T, int L, int V> constexpr bool hess_keep() { return Plan<L, V>::E * sizeof(cx<T>) <= 384; }

// One workgroup makes every x power of its pencils once there are enough
// tiles to fill the chip several times over, else a power each (pass A of
// 512^3 FP32: 0.77 ms as one member, 1.01 as three, 1.84 as three launches
// that read the field each time; 64^3 FP64 8.3, 5.8 and 24 us).
template <typename T, typename W, int L, int V>
static void launch_hess(mfic_ctx ctx, const cx<T>* f, cx<T>* xb, W kf, W scale) {
    constexpr int P = Plan<L, V>::P, N = 2 * L / 3, kc = N / 2 + 1;
    constexpr bool KEEP = hess_keep<T, L, V>();
    const int tk = pick_tile<T, L, V>(ctx, MFIC_PASS_PAD_C2R_A, false);
    const cx<T>* tw = static_cast<const cx<T>*>(twiddles(ctx, L, PencilTw<T, L, V, 64>::KIND, prec_of<T>(), V));
    const long cols = (long)N * kc;
    const long ntiles = (cols + tk - 1) / tk;
    const int members = ntiles >= 4096 ? 1 : 3;
    const dim3 grid((unsigned)ntiles, members);
    ProfScope prof(ctx, pass_name<T, L>("fft_c2rAh"), (double)cols * (members * N + 3 * L) * sizeof(cx<T>));
#define CALL(K)                                                                                                \
    hipLaunchKernelGGL((k_hess_a<T, W, L, K, V, KEEP>), grid, dim3(P * K), (pencil_lds<T, L, V>(K)), ctx->stream, \
                       f, StPadCol<T>{xb}, cols, kf, scale, tw);
    MFIC_TILE_SWITCH(P, CALL)
#undef CALL
    MFIC_LAUNCH_CHECK();
}
// Pass B: a member per x power (its Hessians from one read) from about four
// workgroups a CU on, below that a member per Hessian (512^3 FP32: 2.68 ms
// against 3.06 as six members and 3.5 as six launches on the same plan;
// 256^3 FP32 317, 394 and 380 us; 64^3 FP32 9.4, 7.8 and 26 us).
template <typename T, typename W, int L, int V>
static void launch_hess_b(mfic_ctx ctx, const cx<T>* xb, cx<T>* out, W kf) {
    constexpr int P = Plan<L, V>::P, N = 2 * L / 3, kc = N / 2 + 1;
    constexpr bool KEEP = hess_keep<T, L, V>();
    const int tk = pick_tile<T, L, V>(ctx, MFIC_PASS_PAD_C2R_B, false);
    const cx<T>* tw = static_cast<const cx<T>*>(twiddles(ctx, L, PencilTw<T, L, V, 64>::KIND, prec_of<T>(), V));
    const long cols = (long)L * kc;
    const long ntiles = (cols + tk - 1) / tk;
    const int members = ntiles * 3 >= 1024 ? 3 : 6;
    const dim3 grid((unsigned)xcd_grid(ntiles), members);
    ProfScope prof(ctx, pass_name<T, L>("fft_c2rBh"), (double)cols * (members * N + 6 * L) * sizeof(cx<T>));
#define CALL(K)                                                                                                \
    hipLaunchKernelGGL((k_hess_b<T, W, L, K, V, KEEP>), grid, dim3(P * K), (pencil_lds<T, L, V>(K)), ctx->stream, \
                       LdAx1<T, true>{xb}, StAx1<T, false>{out}, cols, kf, tw);
    MFIC_TILE_SWITCH(P, CALL)
#undef CALL
    MFIC_LAUNCH_CHECK();
}

template <typename T, typename W>
void hessians_to_kbuf(mfic_ctx ctx, const void* f, size_t n, double L, void* xbuf, void* out) {
    const int np = 3 * (int)n / 2;
    const W kf = (W)(2.0 * 3.14159265358979323846 / L), rfac = (W)std::pow(1.5, 1.5);
    const cx<T>* src = static_cast<const cx<T>*>(f);
    cx<T>*xb = static_cast<cx<T>*>(xbuf), *ob = static_cast<cx<T>*>(out);
#define X(S)                                                                                   \
    case S:                                                                                    \
        if (plan_variant(ctx, S, MFIC_PASS_PAD_C2R_A, prec_of<T>()) == 1)                      \
            launch_hess<T, W, S, alt_plan<S>()>(ctx, src, xb, kf, rfac);                       \
        else launch_hess<T, W, S, 0>(ctx, src, xb, kf, rfac);                                  \
        if (plan_variant(ctx, S, MFIC_PASS_PAD_C2R_B, prec_of<T>()) == 1)                      \
            launch_hess_b<T, W, S, alt_plan<S>()>(ctx, xb, ob, kf);                            \
        else launch_hess_b<T, W, S, 0>(ctx, xb, ob, kf);                                       \
        break;
    MFIC_PADDED_SWITCH(np)
#undef X
}

template <typename T, int L, int V> static void launch_hess_bt(mfic_ctx ctx, const cx<T>* in, cx<T>* zb, double kf) {
    constexpr int P = Plan<L, V>::P, N = 2 * L / 3, kc = N / 2 + 1;
    const int tk = pick_tile<T, L, V>(ctx, MFIC_PASS_PAD_R2C_B, false);
    const cx<T>* tw = static_cast<const cx<T>*>(twiddles(ctx, L, PencilTw<T, L, V, 64>::KIND, prec_of<T>(), V));
    const long cols = (long)L * kc;
    const dim3 grid((unsigned)xcd_grid((cols + tk - 1) / tk), 3);
    ProfScope prof(ctx, pass_name<T, L>("fft_r2cBt"), (double)cols * (6 * L + 3 * N) * sizeof(cx<T>));
#define CALL(K)                                                                                                \
    hipLaunchKernelGGL((k_hess_bt<T, L, K, V>), grid, dim3(P * K), (pencil_lds<T, L, V>(K)), ctx->stream,     \
                       LdAx1<T, false>{in}, StAx1<T, true>{zb}, cols, kf, tw);
    MFIC_TILE_SWITCH(P, CALL)
#undef CALL
    MFIC_LAUNCH_CHECK();
}
template <typename T, int L, int V>
static void launch_hess_at(mfic_ctx ctx, const cx<T>* zb, const AdjointOut<T>& o, double kf) {
    constexpr int P = Plan<L, V>::P, N = 2 * L / 3, kc = N / 2 + 1;
    const int tk = pick_tile<T, L, V>(ctx, MFIC_PASS_PAD_R2C_A, false);
    const cx<T>* tw = static_cast<const cx<T>*>(twiddles(ctx, L, PencilTw<T, L, V, 64>::KIND, prec_of<T>(), V));
    const long cols = (long)N * kc;
    const dim3 grid((unsigned)((cols + tk - 1) / tk));
    ProfScope prof(ctx, pass_name<T, L>("fft_r2cAt"), (double)cols * (3 * L + 2 * N) * sizeof(cx<T>));
#define CALL(K)                                                                                                \
    hipLaunchKernelGGL((k_hess_at<T, L, K, V>), grid, dim3(P * K), (pencil_lds<T, L, V>(K)), ctx->stream,     \
                       LdPadCol<T>{zb}, o, cols, kf, tw);
    MFIC_TILE_SWITCH(P, CALL)
#undef CALL
    MFIC_LAUNCH_CHECK();
}

template <typename T>
void hessian_adjoint(mfic_ctx ctx, size_t n, double L, const void* prod, void* zbuf, const void* lam,
                     const double* tab, double g1, double volfac, void* out) {
    const int np = 3 * (int)n / 2;
    const double kf = 2.0 * 3.14159265358979323846 / L;
    const double rfac = std::sqrt((double)np * np * np) / std::sqrt((double)n * n * n);
    const double norm = 1.0 / std::sqrt((double)np * (double)np * (double)np);
    const AdjointOut<T> o{static_cast<cx<T>*>(out), static_cast<const cx<T>*>(lam), tab, g1, norm / rfac, volfac};
    cx<T>* zb = static_cast<cx<T>*>(zbuf);
#define X(S)                                                                                                        \
    case S:                                                                                                         \
        if (plan_variant(ctx, S, MFIC_PASS_PAD_R2C_B, prec_of<T>()) == 1)                                           \
            launch_hess_bt<T, S, alt_plan<S>()>(ctx, static_cast<const cx<T>*>(prod), zb, kf);                      \
        else launch_hess_bt<T, S, 0>(ctx, static_cast<const cx<T>*>(prod), zb, kf);                                 \
        if (plan_variant(ctx, S, MFIC_PASS_PAD_R2C_A, prec_of<T>()) == 1) launch_hess_at<T, S, alt_plan<S>()>(ctx, zb, o, kf); \
        else launch_hess_at<T, S, 0>(ctx, zb, o, kf);                                                               \
        break;
    MFIC_PADDED_SWITCH(np)
#undef X
}

template <typename T, int L, class LD, class ST, int V>
static void launch_filter_v(mfic_ctx ctx, int pass, const LD& ld, const ST& st, long ncols, int members, bool xcd,
                            int zk, double scale, const char* name) {
    constexpr int P = Plan<L, V>::P;
    const int tk = pick_tile<T, L, V>(ctx, pass, true);
    const cx<T>* tw = static_cast<const cx<T>*>(twiddles(ctx, L, PencilTw<T, L, V, 64>::KIND, prec_of<T>(), V));
    const size_t lds = pencil_lds<T, L, V>(tk);
    const long ntiles = (ncols + tk - 1) / tk;
    const dim3 grid((unsigned)(xcd ? xcd_grid(ntiles) : ntiles), members);
    ProfScope prof(ctx, pass_name<T, L>(name), 2.0 * (double)ncols * L * sizeof(cx<T>) * members);
#define CALL(K)                                                                                                    \
    hipLaunchKernelGGL((k_pencils_filter<T, L, K, LD, ST, V>), grid, dim3(P * K), lds, ctx->stream, ld, st, ncols, \
                       tw, xcd ? 1 : 0, zk, (T)scale);
    MFIC_TILE_SWITCH(P, CALL)
#undef CALL
    MFIC_LAUNCH_CHECK();
}

template <typename T, int L, class LD, class ST>
static void launch_filter(mfic_ctx ctx, int pass, const LD& ld, const ST& st, long ncols, int members, bool xcd, int zk,
                          double scale, const char* name) {
    if (plan_variant(ctx, L, pass, prec_of<T>()) == 1)
        launch_filter_v<T, L, LD, ST, alt_plan<L>()>(ctx, pass, ld, st, ncols, members, xcd, zk, scale, name);
    else
        launch_filter_v<T, L, LD, ST, 0>(ctx, pass, ld, st, ncols, members, xcd, zk, scale, name);
}

template <typename T> void truncate_repad(mfic_ctx ctx, size_t n, void* kbuf, int count) {
    const int N = (int)n, np = 3 * N / 2, kc = N / 2 + 1;
    const double norm = 1.0 / std::sqrt((double)np * (double)np * (double)np);
    cx<T>* kb = static_cast<cx<T>*>(kbuf);
    LdAx1<T, false> l1{kb};
    StAx1<T, false> s1{kb};
    LdAx0<T> l0{kb};
    StAx0<T> s0{kb};
    const long cols = (long)np * kc;
#define X(S)                                                                                                     \
    case S:                                                                                                      \
        launch_filter<T, S>(ctx, MFIC_PASS_TRUNC_AX1, l1, s1, cols, count, true, 1, norm, "fft_truncate_ax1");   \
        launch_filter<T, S>(ctx, MFIC_PASS_TRUNC_AX0, l0, s0, cols, count, false, 0, 1.0, "fft_truncate_ax0");   \
        break;
    MFIC_PADDED_SWITCH(np)
#undef X
}

#define MFIC_PRUNED_T(MODE, T)                                                                                        \
    MODE template void operands_to_kbuf<T>(mfic_ctx, const OperandDesc*, int, size_t, const double*, void*);                \
    MODE template void r2c_from_kbuf<T>(mfic_ctx, size_t, double, void*, int, void* const*, int, double, bool);       \
    MODE template void hessians_to_kbuf<T, T>(mfic_ctx, const void*, size_t, double, void*, void*);                   \
    MODE template void hessian_adjoint<T>(mfic_ctx, size_t, double, const void*, void*, const void*, const double*,   \
                                          double, double, void*);                                                     \
    MODE template void truncate_repad<T>(mfic_ctx, size_t, void*, int);

#if MFIC_UNIT == 64
MFIC_PRUNED_T(, double)
#else
MFIC_PRUNED_T(extern, double)

void padded_hessians_to_kbuf(mfic_ctx ctx, int prec, const void* f, size_t n, double L, void* xbuf, void* out,
                             bool weights64) {
    if (prec == MFIC_F64) hessians_to_kbuf<double, double>(ctx, f, n, L, xbuf, out);
    else if (weights64) hessians_to_kbuf<float, double>(ctx, f, n, L, xbuf, out);
    else hessians_to_kbuf<float, float>(ctx, f, n, L, xbuf, out);
}

void padded_hessian_adjoint(mfic_ctx ctx, int prec, size_t n, double L, const void* prod, void* zbuf, const void* lam,
                            const double* tab, double g1, double volfac, void* out) {
    if (prec == MFIC_F64) hessian_adjoint<double>(ctx, n, L, prod, zbuf, lam, tab, g1, volfac, out);
    else hessian_adjoint<float>(ctx, n, L, prod, zbuf, lam, tab, g1, volfac, out);
}

void padded_truncate_repad(mfic_ctx ctx, int prec, size_t n, void* kbuf, int count) {
    if (prec == MFIC_F64) truncate_repad<double>(ctx, n, kbuf, count);
    else truncate_repad<float>(ctx, n, kbuf, count);
}

void padded_operands_to_kbuf(mfic_ctx ctx, int prec, const OperandDesc* o, int count, size_t n, const double L[3],
                             void* kbuf) {
    MFIC_CHECK(count == 1 || count == 2, MFIC_ERR_ARG, "one or two operands");
    if (prec == MFIC_F64) operands_to_kbuf<double>(ctx, o, count, n, L, kbuf);
    else operands_to_kbuf<float>(ctx, o, count, n, L, kbuf);
}

void padded_r2c_from_kbuf(mfic_ctx ctx, int prec, size_t n, double L, void* kbuf, int count, void* const* out, int op,
                          double coef, bool invlap) {
    MFIC_CHECK(count >= 1 && count <= 4, MFIC_ERR_ARG, "one to four fields");
    if (prec == MFIC_F64) r2c_from_kbuf<double>(ctx, n, L, kbuf, count, out, op, coef, invlap);
    else r2c_from_kbuf<float>(ctx, n, L, kbuf, count, out, op, coef, invlap);
}
#endif

}  // namespace mfic
