// NGenIC white noise on the device (random_ngenic.cc:39-154).
//
// Each (i, j) column of the k-space grid is an independent RANLUX stream
// reseeded from the seed table, so one lane generates one column.  The
// RANLUX state (12 words of 48 bits) lives in registers; every 202-step cycle
// is unrolled with static indices and the register names are rotated by 10
// afterwards, so a cycle always starts at word 0 and the 12 outputs of the
// cycle are words 0..11 in order.  The numbers go through LDS to the lanes
// that turn them into Gaussian draws, one mode a lane: correctly rounded log,
// sin and cos from a short double-double evaluation with a rounding test, or,
// where the test leaves the rounding open, from the long one (the operation
// sequence of the CPU oracle), giving bit-identical draws.
//
// This file is compiled with -ffp-contract=off: every fma is explicit.
#include <cmath>
#include <cstdint>
#include <vector>

#include "fft_core.hpp"
#include "mfic_internal.hpp"
#include "ngenic.hpp"

namespace mfic {

// ----------------------------------------------------- double-double ----
struct dd { double hi, lo; };

__host__ __device__ inline dd two_sum(double a, double b) {
    double s = a + b, bb = s - a;
    return {s, (a - (s - bb)) + (b - bb)};
}
__host__ __device__ inline dd fast_two_sum(double a, double b) {
    double s = a + b;
    return {s, b - (s - a)};
}
__host__ __device__ inline dd two_prod(double a, double b) {
    double p = a * b;
    return {p, fma(a, b, -p)};
}
__host__ __device__ inline dd dd_add(dd x, dd y) {
    dd s = two_sum(x.hi, y.hi), t = two_sum(x.lo, y.lo);
    double c = s.lo + t.hi;
    dd v = fast_two_sum(s.hi, c);
    c = t.lo + v.lo;
    return fast_two_sum(v.hi, c);
}
__host__ __device__ inline dd dd_mul(dd x, dd y) {
    dd p = two_prod(x.hi, y.hi);
    double e = fma(x.hi, y.lo, x.lo * y.hi) + p.lo;
    return fast_two_sum(p.hi, e);
}
__host__ __device__ inline dd dd_mul_d(dd x, double d) {
    dd p = two_prod(x.hi, d);
    double e = fma(x.lo, d, p.lo);
    return fast_two_sum(p.hi, e);
}
__host__ __device__ inline dd dd_div(dd x, dd y) {
    double q1 = x.hi / y.hi;
    dd p = dd_mul_d(y, q1);
    dd r = dd_add(x, dd{-p.hi, -p.lo});
    double q2 = r.hi / y.hi;
    p = dd_mul_d(y, q2);
    r = dd_add(r, dd{-p.hi, -p.lo});
    double q3 = r.hi / y.hi;
    dd q = fast_two_sum(q1, q2);
    return dd_add(q, dd{q3, 0.0});
}
__host__ __device__ inline dd dd_recip_d(double d) {
    double hi = 1.0 / d;
    double r = fma(-hi, d, 1.0);
    return {hi, r / d};
}

// series coefficients, computed once on the host with the same operations as
// the CPU oracle: log: 1/(2k+1), k = 0..26;  sin / cos Taylor terms
struct CrTables {
    double logc[27][2];
    double sinc[16][2];
    double cosc[16][2];
};

static CrTables make_tables() {
    CrTables t;
    for (int k = 0; k <= 26; ++k) {
        dd r = dd_recip_d((double)(2 * k + 1));
        t.logc[k][0] = r.hi; t.logc[k][1] = r.lo;
    }
    dd cs = {1.0, 0.0}, cc = {1.0, 0.0};
    t.sinc[0][0] = 1.0; t.sinc[0][1] = 0.0; t.cosc[0][0] = 1.0; t.cosc[0][1] = 0.0;
    for (int k = 1; k <= 15; ++k) {
        cs = dd_div(cs, dd{(double)((2 * k) * (2 * k + 1)), 0.0});
        cc = dd_div(cc, dd{(double)((2 * k - 1) * (2 * k)), 0.0});
        t.sinc[k][0] = cs.hi; t.sinc[k][1] = cs.lo;
        t.cosc[k][0] = cc.hi; t.cosc[k][1] = cc.lo;
    }
    return t;
}

__device__ inline double cr_log(double x, const CrTables& T) {
    // x in (0, 1) here: positive, finite, normal
    int e;
    double m = frexp(x, &e);
    if (m < 0.70710678118654752440) { m *= 2.0; e -= 1; }
    dd num = {m - 1.0, 0.0};
    dd den = two_sum(m, 1.0);
    dd s = dd_div(num, den);
    dd t = dd_mul(s, s);
    dd p = {T.logc[26][0], T.logc[26][1]};
    for (int k = 25; k >= 0; --k) {
        p = dd_mul(p, t);
        p = dd_add(p, dd{T.logc[k][0], T.logc[k][1]});
    }
    dd lm = dd_mul(s, p);
    lm.hi *= 2.0; lm.lo *= 2.0;
    dd el = dd_mul_d(dd{6.93147180559945286227e-01, 2.31904681384629955842e-17}, (double)e);
    dd r = dd_add(el, lm);
    return r.hi + r.lo;
}

__device__ inline void cr_sincos(double x, double* sn, double* cs, const CrTables& T) {
    const double PIO2_1 = 1.57079632679489655800e+00, PIO2_2 = 6.12323399573676603587e-17,
                 PIO2_3 = -1.49738490485916983634e-33;
    double qd = rint(x * 0.63661977236758134308);
    dd r;
    if (qd == 0.0) {
        r = dd{x, 0.0};
    } else {
        dd p1 = two_prod(qd, PIO2_1), p2 = two_prod(qd, PIO2_2);
        double p3 = qd * PIO2_3;
        r = two_sum(x, -p1.hi);
        r = dd_add(r, dd{-p1.lo, 0.0});
        r = dd_add(r, dd{-p2.hi, -p2.lo});
        r = dd_add(r, dd{-p3, 0.0});
    }
    dd t = dd_mul(r, r);
    const int K = 15;
    dd ps = {-T.sinc[K][0], -T.sinc[K][1]}, pc = {-T.cosc[K][0], -T.cosc[K][1]};  // K odd
    for (int k = K - 1; k >= 0; --k) {
        dd a = {T.sinc[k][0], T.sinc[k][1]}, b = {T.cosc[k][0], T.cosc[k][1]};
        if (k & 1) { a.hi = -a.hi; a.lo = -a.lo; b.hi = -b.hi; b.lo = -b.lo; }
        ps = dd_add(dd_mul(ps, t), a);
        pc = dd_add(dd_mul(pc, t), b);
    }
    dd ss = dd_mul(ps, r);
    double sv = ss.hi + ss.lo, cv = pc.hi + pc.lo;
    long q = (long)qd;
    switch (((q % 4) + 4) % 4) {
    case 0: *sn = sv; *cs = cv; break;
    case 1: *sn = cv; *cs = -sv; break;
    case 2: *sn = -sv; *cs = -cv; break;
    default: *sn = -cv; *cs = sv; break;
    }
}

// ------------------------------------------------------------- RANLUX ----
constexpr uint64_t kMask48 = (uint64_t(1) << 48) - 1;

// gsl_rng_set seeding of ranlxd: 31-bit shift register (taps 0 and 18),
// 48 complemented register bits per word.  Host form: the seed is held in a
// C int exactly as there.
inline void ranlux_seed_host(uint64_t x[12], unsigned long seed) {
    if (seed == 0) seed = 1;
    int i = (int)(uint32_t)(seed & 0xFFFFFFFFUL);
    int xbit[31];
    for (int k = 0; k < 31; ++k) { xbit[k] = i % 2; i /= 2; }
    int ibit = 0, jbit = 18;
    for (int k = 0; k < 12; ++k) {
        uint64_t w = 0;
        for (int l = 1; l <= 48; ++l) {
            const int y = (xbit[ibit] + 1) % 2;
            w = 2 * w + (uint64_t)(int64_t)y;
            xbit[ibit] = (xbit[ibit] + xbit[jbit]) % 2;
            ibit = (ibit + 1) % 31;
            jbit = (jbit + 1) % 31;
        }
        x[k] = w & kMask48;
    }
}

// x_ir <- x_jr - x_ir - c  (mod 2^48), jr = ir + 7 (mod 12)
#define MFIC_SWB(IR)                                                          \
    {                                                                         \
        uint64_t d_ = x[((IR) + 7) % 12] + (uint64_t(1) << 48) - x[(IR)] - c; \
        c = 1 - (int)(d_ >> 48);                                              \
        x[(IR)] = d_ & kMask48;                                               \
    }

// one luxury-202 cycle starting at word 0; afterwards the words are renamed
// so that the 12 outputs (the last 12 produced, oldest first) are x[0..11]
// and the next cycle again starts at word 0
inline void ranlux_cycle202(uint64_t x[12], int& c) {
    for (int blk = 0; blk < 16; ++blk) {
#pragma unroll
        for (int r = 0; r < 12; ++r) MFIC_SWB(r)
    }
#pragma unroll
    for (int r = 0; r < 10; ++r) MFIC_SWB(r)
    const uint64_t a = x[10], b = x[11];
#pragma unroll
    for (int r = 11; r >= 2; --r) x[r] = x[r - 2];
    x[0] = a;
    x[1] = b;
}
#undef MFIC_SWB

// ------------------------------------------------- device: the stream ----
// Words as a 32-bit low part and a 16-bit high part, so that a step is two
// subtractions on the carry flag and one mask (3 instructions, against 8 for
// the 64-bit form above).
struct DevRanlux {
    uint32_t l[12], h[12];
    unsigned c;

    // Seeds in [0, 2^31): the shift register's bits follow s[t + 31] = s[t] ^
    // s[t + 18] and a word is 48 complemented bits, first bit highest.  `win`
    // holds the next bits of the sequence, first bit lowest; 31 known bits
    // give 26 more in two steps, 24 of which are taken at a time.
    __device__ __forceinline__ void seed(uint32_t s) {
        uint64_t win = (s == 0 ? 1u : s) & 0x7fffffffu;
        auto take24 = [&win]() {
            win |= ((win ^ (win >> 18)) & 0x1fffu) << 31;
            win |= (((win >> 13) ^ (win >> 31)) & 0x1fffu) << 44;
            const uint32_t v = __brev(~(uint32_t)win) >> 8;
            win >>= 24;
            return v;
        };
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            const uint32_t hi = take24(), lo = take24();
            h[k] = hi >> 8;
            l[k] = (hi << 24) | lo;
        }
        c = 0;
    }
    // x_ir <- x_jr - x_ir - c  (mod 2^48), jr = ir + 7 (mod 12)
    template <int IR> __device__ __forceinline__ void step() {
        unsigned b, d;
        l[IR] = __builtin_subc(l[(IR + 7) % 12], l[IR], c, &b);
        h[IR] = __builtin_subc(h[(IR + 7) % 12], h[IR], b, &d) & 0xffffu;
        c = d;
    }
    // ranlux_cycle202 on the device
    __device__ __forceinline__ void cycle() {
#pragma unroll 2
        for (int blk = 0; blk < 16; ++blk) {
            step<0>(); step<1>(); step<2>(); step<3>(); step<4>(); step<5>();
            step<6>(); step<7>(); step<8>(); step<9>(); step<10>(); step<11>();
        }
        step<0>(); step<1>(); step<2>(); step<3>(); step<4>();
        step<5>(); step<6>(); step<7>(); step<8>(); step<9>();
        const uint32_t l0 = l[10], l1 = l[11], h0 = h[10], h1 = h[11];
#pragma unroll
        for (int r = 11; r >= 2; --r) { l[r] = l[r - 2]; h[r] = h[r - 2]; }
        l[0] = l0; l[1] = l1; h[0] = h0; h[1] = h1;
    }
    __device__ __forceinline__ uint64_t word(int r) const { return (uint64_t)h[r] << 32 | l[r]; }
};

// ------------------------------------- device: correctly rounded draws ----
constexpr double kPio2a = 1.57079632679489655800e+00, kPio2b = 6.12323399573676603587e-17,
                 kPio2c = -1.49738490485916983634e-33;  // pi/2 in three parts
constexpr double kLn2a = 6.93147180559945286227e-01, kLn2b = 2.31904681384629955842e-17;

// x * t + (ch + cl) on double-doubles with |c| >= |x t|
__device__ __forceinline__ dd dd_horner(dd x, dd t, double ch, double cl) {
    const dd p = two_prod(x.hi, t.hi);
    const double e = fma(x.hi, t.lo, fma(x.lo, t.hi, p.lo));
    const dd s = fast_two_sum(ch, p.hi);
    return {s.hi, s.lo + (e + cl)};
}
// x * y, low part not renormalised
__device__ __forceinline__ dd dd_mul_fast(dd x, dd y) {
    const dd p = two_prod(x.hi, y.hi);
    return {p.hi, fma(x.hi, y.lo, fma(x.lo, y.hi, p.lo))};
}
// rounds hi + lo, an approximation within 2^-68 |hi|, to *y; false when the
// rounding of the exact value stays open
__device__ __forceinline__ bool round_settled(dd x, double* y) {
    const double d = fabs(x.hi) * 0x1p-68;
    const double a = x.hi + (x.lo - d), b = x.hi + (x.lo + d);
    *y = a;
    return a == b;
}
// The short evaluations behind the rounding test (relative error below
// 2^-70, tested at 2^-68): every series runs in double from the term whose
// share of the sum is below 2^-21, so that its rounding is below 2^-72, and
// in double-double below that: 4 or 5 steps where the full evaluation takes
// 26 and 15.  log: 2 s sum t^k / (2k + 1), s = (m - 1) / (m + 1), t = s^2 <=
// 0.0295, terms to k = 13 (the next is 2^-76).  sin, cos on |r| <= pi/4:
// terms to k = 10 (the next are 2^-82 and 2^-77).
__device__ __forceinline__ bool log_short(double x, const CrTables& T, double* y) {
    double m = __builtin_amdgcn_frexp_mant(x);
    int e = __builtin_amdgcn_frexp_exp(x);
    if (m < 0.70710678118654752440) { m *= 2.0; e -= 1; }
    const double num = m - 1.0;
    const dd den = two_sum(m, 1.0);
    const double inv = 1.0 / den.hi;
    dd s;
    s.hi = num * inv;
    s.lo = fma(-s.hi, den.lo, fma(-s.hi, den.hi, num)) * inv;
    const dd t = dd_mul_fast(s, s);
    double q = T.logc[13][0];
#pragma unroll
    for (int k = 12; k >= 4; --k) q = fma(q, t.hi, T.logc[k][0]);
    dd p = {q, 0.0};
#pragma unroll
    for (int k = 3; k >= 0; --k) p = dd_horner(p, t, T.logc[k][0], T.logc[k][1]);
    dd lm = dd_mul_fast(s, p);
    lm.hi *= 2.0; lm.lo *= 2.0;
    const double ed = (double)e;
    dd el = two_prod(ed, kLn2a);
    el.lo = fma(ed, kLn2b, el.lo);
    const dd r = two_sum(el.hi, lm.hi);
    return round_settled(fast_two_sum(r.hi, r.lo + (el.lo + lm.lo)), y);
}
__device__ __forceinline__ bool sincos_short(double x, const CrTables& T, double* sn, double* cs) {
    const double q = rint(x * 0.63661977236758134308);  // x in [0, 2 pi): q = 0 .. 4
    const dd p1 = two_prod(q, kPio2a), p2 = two_prod(q, kPio2b);
    dd r = two_sum(x - p1.hi, -p1.lo);  // x - p1.hi is exact
    const double l1 = r.lo;
    r = two_sum(r.hi, -p2.hi);
    r = fast_two_sum(r.hi, r.lo + (l1 - fma(q, kPio2c, p2.lo)));
    const dd t = dd_mul_fast(r, r);
    double us = T.sinc[10][0], uc = T.cosc[10][0];
#pragma unroll
    for (int k = 9; k >= 4; --k) us = fma(us, t.hi, k & 1 ? -T.sinc[k][0] : T.sinc[k][0]);
#pragma unroll
    for (int k = 9; k >= 5; --k) uc = fma(uc, t.hi, k & 1 ? -T.cosc[k][0] : T.cosc[k][0]);
    dd ps = {us, 0.0}, pc = {uc, 0.0};
    pc = dd_horner(pc, t, T.cosc[4][0], T.cosc[4][1]);
#pragma unroll
    for (int k = 3; k >= 0; --k) {
        const double sg = k & 1 ? -1.0 : 1.0;
        ps = dd_horner(ps, t, sg * T.sinc[k][0], sg * T.sinc[k][1]);
        pc = dd_horner(pc, t, sg * T.cosc[k][0], sg * T.cosc[k][1]);
    }
    double sv, cv;
    const dd ss = dd_mul_fast(ps, r);
    const bool oks = round_settled(fast_two_sum(ss.hi, ss.lo), &sv);
    const bool okc = round_settled(fast_two_sum(pc.hi, pc.lo), &cv);
    const int qi = (int)q;
    const double a = qi & 1 ? cv : sv, b = qi & 1 ? sv : cv;
    *sn = qi & 2 ? -a : a;
    *cs = (qi + 1) & 2 ? -b : b;
    return oks && okc;
}
// FP32 draws: z = sqrt(-log u) exp(i phase) in plain double, relative error
// below 2^-46 (series as above, to 2^-49; reciprocal and square root by two
// and one Newton steps).  When every double within 2^-42 of a part rounds to
// the same float, that float is also the rounding of the correctly rounded
// double, so the FP32 noise stays bit-identical.
__device__ __forceinline__ bool float_rounding_settled(double y) {
    const double d = fabs(y) * 0x1p-42;
    return (float)(y - d) == (float)(y + d);
}
__device__ __forceinline__ bool gauss_float(double phase, double ampl, const CrTables& T, double* zr, double* zi) {
    double m = __builtin_amdgcn_frexp_mant(ampl);
    int e = __builtin_amdgcn_frexp_exp(ampl);
    if (m < 0.70710678118654752440) { m *= 2.0; e -= 1; }
    const double den = m + 1.0;
    double inv = __builtin_amdgcn_rcp(den);
    inv = fma(fma(-den, inv, 1.0), inv, inv);
    inv = fma(fma(-den, inv, 1.0), inv, inv);
    const double s = (m - 1.0) * inv, t = s * s;
    double p = T.logc[8][0];
#pragma unroll
    for (int k = 7; k >= 0; --k) p = fma(p, t, T.logc[k][0]);
    const double w = -fma((double)e, kLn2a, 2.0 * s * p);  // -log u > 0
    double y = __builtin_amdgcn_rsq(w);
    y = fma(y * fma(-w * y, y, 1.0), 0.5, y);
    const double g = w * y, a = fma(fma(-g, g, w), 0.5 * y, g);
    const double q = rint(phase * 0.63661977236758134308);
    const double r = fma(-q, kPio2b, fma(-q, kPio2a, phase)), r2 = r * r;
    double ps = -T.sinc[7][0], pc = T.cosc[8][0];
#pragma unroll
    for (int k = 6; k >= 0; --k) ps = fma(ps, r2, k & 1 ? -T.sinc[k][0] : T.sinc[k][0]);
#pragma unroll
    for (int k = 7; k >= 0; --k) pc = fma(pc, r2, k & 1 ? -T.cosc[k][0] : T.cosc[k][0]);
    const double sv = ps * r;
    const int qi = (int)q;
    const double sn = qi & 1 ? pc : sv, cs = qi & 1 ? sv : pc;
    *zi = a * (qi & 2 ? -sn : sn);
    *zr = a * ((qi + 1) & 2 ? -cs : cs);
    return float_rounding_settled(*zr) && float_rounding_settled(*zi);
}

// one value of the white-noise field from a (phase, amplitude) draw pair
template <typename T>
__device__ __forceinline__ cx<T> ngenic_value(double phase, double ampl, const CrTables& tabs) {
    double zr, zi;
    if constexpr (sizeof(T) == 4) {
        if (gauss_float(phase, ampl, tabs, &zr, &zi)) return cx<T>{(T)zr, (T)zi};
    }
    double lg, sn, cs;
    bool ok = log_short(ampl, tabs, &lg);
    ok = sincos_short(phase, tabs, &sn, &cs) && ok;
    if (!ok) {
        lg = cr_log(ampl, tabs);
        cr_sincos(phase, &sn, &cs, tabs);
    }
    const double a = sqrt(-lg);
    return cx<T>{(T)(a * cs), (T)(a * sn)};
}

// ------------------------------------------------- device: the kernel ----
// PHI: store phi1 = sg * w / volfac * F(|n|^2) instead of the noise w (the
// values k_phi1_tab forms from the stored noise, from the same T-rounded w),
// with F the FP64 -A(k)/k^2 table per integer |n|^2 of a cubic box and w
// normalised to |w| = 1 when fixing
struct Phi1Fold {
    const double* tab = nullptr;
    double sg = 1.0, volfac = 1.0;
    int fixing = 0;
};
template <typename T>
__device__ __forceinline__ cx<T> phi1_fold(cx<T> w, int si, int sj, int k, const Phi1Fold& f) {
    double wr = w.x, wi = w.y;
    if (f.fixing) {
        const double a = hypot(wr, wi);
        if (a != 0.0) { wr /= a; wi /= a; }
    }
    const double F = f.tab[si * si + sj * sj + k * k];
    return cx<T>{(T)(f.sg * wr / f.volfac * F), (T)(f.sg * wi / f.volfac * F)};
}

// A workgroup takes NGENIC_COLS columns: wave 0 runs their RANLUX streams, a
// column a lane, into a ring of raw numbers in LDS, one tile of KT modes per
// column ahead of the other waves, which turn the previous tile into draws,
// lanes along kz, and store it.
// A column uses a number for the phase of a mode and the next nonzero one for
// its amplitude, so the pairs of mode k sit at ring positions 2k, 2k + 1.
// Every mode of the grid is written.
//
// Bound by instruction issue and, with few columns, by the length of one
// stream: 606 dependent carry instructions per 12 numbers.  The split lets
// the streams of a small grid (one wave per 64 columns, 64 waves at 64^3)
// run while other waves do the far longer transform, and the short
// evaluations cut the FP64 draw from about 2000 instructions to 300.  Noise
// with phi1 folded in, against one thread a column with the long
// evaluations: FP64 64^3 194 -> 33 us, 256^3 786 -> 214 us, 512^3 5.65 ->
// 1.31 ms; FP32 64^3 72 -> 27 us, 256^3 262 -> 135 us, 512^3 1.22 -> 0.85
// ms.  Four waves and 6 modes a tile (19 KB of LDS, eight workgroups a CU)
// measured best or within 2%; three waves lose 5-15%, tiles of 24 modes half
// the speed at 512^3, one wave doing both parts 30-100% up to 256^3.
constexpr int NGENIC_COLS = 64, NGENIC_NW = 4, NGENIC_KT = 6;
// ring slots of a column: the tile being read, the one being written and the
// rest of a cycle; two more keep pairs 16-byte aligned and columns on
// different banks
constexpr int NGENIC_RING = 4 * NGENIC_KT + 12, NGENIC_PITCH = NGENIC_RING + 2;
template <typename T, bool PHI>
__global__ void __launch_bounds__(64 * NGENIC_NW)
k_ngenic_fill(cx<T>* __restrict__ g, const uint32_t* __restrict__ table, int n, CrTables tabs, Phi1Fold pf) {
    constexpr int NW = NGENIC_NW, KT = NGENIC_KT;
    __shared__ __align__(16) uint64_t raw[NGENIC_COLS * NGENIC_PITCH];
    const int cols = n * n, nc = n / 2 + 1, nh = n / 2;
    const int col0 = (int)blockIdx.x * NGENIC_COLS;
    const bool producer = threadIdx.x < 64;
    const int ntile = (nc + KT - 1) / KT, total = 2 * nh;  // kz = n/2 is zero: no numbers
    const int i0 = col0 / n, j0 = col0 - i0 * n;  // the same for the whole workgroup

    DevRanlux rl;
    int pos = 0, slot = 0;
    uint64_t* ring = raw + (threadIdx.x % 64) * NGENIC_PITCH;
    bool draws = false;
    if (producer) {
        const int col = col0 + (int)threadIdx.x, i = col / n, j = col % n;
        draws = col < cols && i != nh && j != nh;
        rl.seed(draws ? table[col] : 1u);
    }
    auto produce = [&](int upto) {
        upto = upto < total ? upto : total;
        while (draws && pos < upto) {
            rl.cycle();
#pragma unroll
            for (int r = 0; r < 12; ++r) {
                const uint64_t w = rl.word(r);
                ring[slot] = w;
                if (!((pos & 1) && w == 0)) {  // an amplitude of 0 is drawn again
                    ++pos;
                    slot = slot == NGENIC_RING - 1 ? 0 : slot + 1;
                }
            }
        }
    };
    auto consume = [&](int t, int at) {
        const int base = (2 * KT * t) % NGENIC_RING;
        for (int idx = at; idx < NGENIC_COLS * KT; idx += 64 * (NW - 1)) {
            const int c = idx / KT, kk = idx % KT, k = t * KT + kk, col = col0 + c;
            if (k >= nc || col >= cols) continue;
            int i = i0, j = j0 + c;
            for (; j >= n; j -= n) ++i;
            cx<T>* dst = g + (long)col * nc + k;
            if (i == nh || j == nh || k == nh || (col == 0 && k == 0)) {
                *dst = cx<T>{0, 0};
                continue;
            }
            // kz = 0: half of the plane is drawn, and gives its mirror (-i, -j) too
            if (k == 0 && !(i == 0 ? j < nh : i < nh)) continue;
            int p = base + 2 * kk;
            p -= p >= NGENIC_RING ? NGENIC_RING : 0;
            const ulonglong2 u = *reinterpret_cast<const ulonglong2*>(raw + c * NGENIC_PITCH + p);
            const double phase = (double)u.x * (1.0 / 281474976710656.0) * 2 * 3.14159265358979323846;
            const double ampl = (double)u.y * (1.0 / 281474976710656.0);
            cx<T> z = ngenic_value<T>(phase, ampl, tabs);
            // the mirror has the same |n|^2: its value is conj(z) either way
            if constexpr (PHI) z = phi1_fold(z, i - (i > nh) * n, j - (j > nh) * n, k, pf);
            *dst = z;
            if (k == 0) {
                const int ii = i > 0 ? n - i : 0, jj = j > 0 ? n - j : 0;
                g[((long)ii * n + jj) * nc] = cx<T>{z.x, -z.y};
            }
        }
    };
    if (producer) produce(2 * KT);
    __syncthreads();
    for (int t = 0; t < ntile; ++t) {
        if (producer) produce(2 * KT * (t + 2));
        else consume(t, (int)threadIdx.x - 64);
        __syncthreads();
    }
}

// ------------------------------------------------------------- host -----

namespace {
struct HostRanlux {
    uint64_t x[12];
    int carry = 0, pos = 12;
    explicit HostRanlux(unsigned long seed) { ranlux_seed_host(x, seed); }
    double uniform() {
        if (pos == 12) { ranlux_cycle202(x, carry); pos = 0; }
        return (double)x[pos++] * (1.0 / 281474976710656.0);
    }
};
}  // namespace

void ngenic_seedtable(long seed, size_t n, uint32_t* T) {
    HostRanlux r((unsigned long)seed);
    auto draw = [&r]() { return (uint32_t)(2147483647.0 * r.uniform()); };
    for (size_t q = 0; q < n * n; ++q) T[q] = 0;
    for (size_t i = 0; i < n / 2; ++i) {
        for (size_t j = 0; j < i; j++) T[i * n + j] = draw();
        for (size_t j = 0; j < i + 1; j++) T[j * n + i] = draw();
        for (size_t j = 0; j < i; j++) T[(n - 1 - i) * n + j] = draw();
        for (size_t j = 0; j < i + 1; j++) T[(n - 1 - j) * n + i] = draw();
        for (size_t j = 0; j < i; j++) T[i * n + (n - 1 - j)] = draw();
        for (size_t j = 0; j < i + 1; j++) T[j * n + (n - 1 - i)] = draw();
        for (size_t j = 0; j < i; j++) T[(n - 1 - i) * n + (n - 1 - j)] = draw();
        for (size_t j = 0; j < i + 1; j++) T[(n - 1 - j) * n + (n - 1 - i)] = draw();
    }
}

template <typename T, bool PHI>
static void launch_ngenic(mfic_grid g, const uint32_t* dev_table, const Phi1Fold& pf) {
    MFIC_CHECK(g->n[0] == g->n[1] && g->n[1] == g->n[2], MFIC_ERR_SIZE, "NGenIC needs a cubic grid");
    MFIC_CHECK(g->n[0] % 2 == 0, MFIC_ERR_SIZE, "NGenIC needs an even grid size");
    MFIC_CHECK(g->n[0] <= 32768, MFIC_ERR_SIZE, "NGenIC column index exceeds 32 bits");
    static const CrTables tabs = make_tables();
    const int n = (int)g->n[0];
    const long cols = (long)n * n;
    ProfScope prof(g->ctx, PHI ? "ngenic_phi1" : "ngenic_fill", (double)cols * (n / 2 + 1) * sizeof(cx<T>));
    hipLaunchKernelGGL((k_ngenic_fill<T, PHI>), dim3((unsigned)((cols + NGENIC_COLS - 1) / NGENIC_COLS)),
                       dim3(64 * NGENIC_NW), 0, g->ctx->stream, (cx<T>*)g->d, dev_table, n, tabs, pf);
    MFIC_LAUNCH_CHECK();
}

void ngenic_fill(mfic_grid g, const uint32_t* dev_table) {
    if (g->prec == MFIC_F64) launch_ngenic<double, false>(g, dev_table, Phi1Fold{});
    else launch_ngenic<float, false>(g, dev_table, Phi1Fold{});
}

void ngenic_phi1_fill(mfic_grid phi, const uint32_t* dev_table, const double* phitab, double volfac, int fixing,
                      int inversion) {
    Phi1Fold pf;
    pf.tab = phitab;
    pf.sg = inversion ? -1.0 : 1.0;
    pf.volfac = volfac;
    pf.fixing = fixing;
    if (phi->prec == MFIC_F64) launch_ngenic<double, true>(phi, dev_table, pf);
    else launch_ngenic<float, true>(phi, dev_table, pf);
}

}  // namespace mfic
