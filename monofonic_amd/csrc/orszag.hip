// Orszag 3/2-rule dealiased products (convolution.hh:412-651) and the LPT
// source block of ic_generator::run (ic_generator.cc:523-629).
//
// Two entry levels:
//  * convolve2 / convolve3: the reference's per-product schedule for the
//    drop-in OrszagConvolver interface: both operands through the axis-0 and
//    axis-1 padded c2r passes, one fused row pass for the product, and the
//    r2c passes with the unpad rules and the output operator;
//  * lpt_sources: the reorganised schedule used by the pipeline.  Each
//    Hessian of phi1 and phi2 goes through the axis-0 / axis-1 padded c2r
//    passes once; one fused row pass per LPT order brings all of them to
//    real space in LDS, sums every product sharing one truncation (in FP64)
//    and returns the r2c'd rows, so padded real fields never reach HBM.  The
//    cubic 3a terms keep their two-stage truncation trunc(trunc(a b) c)
//    (convolution.hh:525-532) with the inner products grouped by their outer
//    factor.  Equal to the reference schedule in exact arithmetic (every step
//    is linear in the grouped quantity).
#include "fused.hpp"
#include "mfic_internal.hpp"
#include "orszag.hpp"
#include "pruned.hpp"

namespace mfic {

ConvCore::ConvCore(mfic_ctx c, const size_t n[3], const double L[3], int p) : ctx(c), prec(p) {
    // the passes take every stride and column count from one size
    MFIC_CHECK(n[0] == n[1] && n[1] == n[2], MFIC_ERR_SIZE, "the Orszag convolver needs the same grid size on every axis");
    for (int i = 0; i < 3; ++i) {
        MFIC_CHECK(n[i] % 2 == 0, MFIC_ERR_SIZE, "Orszag convolver for LPTorder>1 requires even grid size!");
        N[i] = n[i];
        Np[i] = 3 * n[i] / 2;
        len[i] = L[i];
    }
    MFIC_CHECK(Np[2] % 2 == 0, MFIC_ERR_SIZE, "padded contiguous axis 3N/2 must be even (N multiple of 4)");
    for (int i = 0; i < 3; ++i)
        MFIC_CHECK(fft_length_supported(N[i]) && fft_length_supported(Np[i]), MFIC_ERR_SIZE,
                   "unsupported grid size for the Orszag convolver");
}

size_t ConvCore::grid_reals() const { return N[0] * N[1] * (N[2] + 2); }
size_t ConvCore::esize() const { return prec == MFIC_F64 ? 8 : 4; }
size_t ConvCore::kbuf_reals() const { return 2 * Np[0] * Np[1] * (N[2] / 2 + 1); }

// convolution.hh:495-518.  The padded real fields stay in the row pass's LDS
// where they went through HBM, and a product of an operand with itself pads
// and transforms it once: the seven products of the 2LPT source and one
// convolve3 at 192^3 FP32 1.72 -> 1.03 ms.  Bound by the four strided passes
// (4.3-5.1 TB/s).
void ConvCore::convolve2(const OperandDesc& a, const OperandDesc& b, void* out, int op, double coef, void* kbuf) const {
    const bool square = a.same(b);
    const OperandDesc o[2] = {a, b};
    void* prod = static_cast<char*>(kbuf) + 2 * kbuf_reals() * esize();
    padded_operands_to_kbuf(ctx, prec, o, square ? 1 : 2, N[0], len, kbuf);
    fused_source_rows(ctx, prec, square ? FusedKind::Square : FusedKind::Mul, N[0], kbuf, prod);
    padded_r2c_from_kbuf(ctx, prec, N[0], len[0], prod, 1, &out, op, coef, false);
}

void ConvCore::convolve3(const OperandDesc& a, const OperandDesc& b, const OperandDesc& c, void* out, int op,
                         double coef, void* kbuf, void* fbuf) const {
    convolve2(a, b, fbuf, MFIC_OP_ASSIGN, 0.0, kbuf);
    OperandDesc id{fbuf, MFIC_OPND_IDENT, {0, 0, 0, 0}};
    convolve2(id, c, out, op, coef, kbuf);
}

// ------------------------------------------------- reorganised sources ----

void lpt_sources(mfic_ctx ctx, int order, mfic_grid phi1, mfic_grid phi2, mfic_grid phi3, mfic_grid A3x,
                 mfic_grid A3y, mfic_grid A3z) {
    if (order < 2) return;
    ConvCore C(ctx, phi1->n, phi1->L, phi1->prec);
    MFIC_CHECK(phi1->L[0] == phi1->L[1] && phi1->L[1] == phi1->L[2], MFIC_ERR_SIZE, "LPT sources need equal box sides");
    const size_t n = phi1->n[0];
    const double L = phi1->L[0];
    const int prec = phi1->prec;
    // compact padded half-spectrum buffers, consecutive: inputs of the fused
    // row pass (phi1 Hessians, phi2 Hessians, Q) and its outputs
    const size_t kb = C.kbuf_reals() * C.esize();
    const FusedKind k1 = order >= 3 ? FusedKind::Src2Q : FusedKind::Src2;
    // inputs of the row passes, consecutive: phi1 Hessians [0, 6), phi2
    // Hessians [6, 12), Q [12, 16).  The 2LPT pass writes its outputs (phi2
    // source, Q) to [11, 16): slot 11 is consumed before the phi2 Hessians
    // fill it.
    char* kin = static_cast<char*>(ctx_scratch(ctx, "fused_in", (size_t)(order >= 3 ? 16 : 7) * kb));
    void* xbuf = ctx_scratch(ctx, "hess_x", 3 * kb);
    padded_hessians_to_kbuf(ctx, prec, phi1->d, n, L, xbuf, kin);
    char* src2 = kin + (order >= 3 ? 11 : 6) * kb;
    // phi2 source (ic_generator.cc:536-541) and, for 3LPT, the inner 3a
    // products Qzz Qyz Qxx Qyy (ic_generator.cc:581-585) from one row pass
    fused_source_rows(ctx, prec, k1, n, kin, src2);
    padded_r2c_from_kbuf(ctx, prec, n, L, src2, 1, &phi2->d, MFIC_OP_ASSIGN, 0.0, true);  // -1/k^2: ic_generator.cc:554
    phi2->space = MFIC_KSPACE;
    if (order < 3) return;
    // Q: truncated once (first stage of trunc(trunc(a b) c), convolution.hh:
    // 525-532) and padded again for the outer products, in place
    padded_truncate_repad(ctx, prec, n, kin + 12 * kb, 4);
    padded_hessians_to_kbuf(ctx, prec, phi2->d, n, L, xbuf, kin + 6 * kb);
    // phi3 source (3a outer + 3b, ic_generator.cc:581-609) and A3
    // (ic_generator.cc:614-627), then -1/k^2 each
    char* kout = static_cast<char*>(ctx_scratch(ctx, "fused_out", 4 * kb));
    fused_source_rows(ctx, prec, FusedKind::Src3, n, kin, kout);
    void* outs[4] = {phi3->d, A3x->d, A3y->d, A3z->d};
    // one launch writes them all: a grid given several times takes the last,
    // the others go to the x powers' buffers, whose work is done
    for (int o = 0; o < 3; ++o)
        for (int e = o + 1; e < 4; ++e)
            if (outs[o] == outs[e]) {
                outs[o] = static_cast<char*>(xbuf) + o * kb;
                break;
            }
    padded_r2c_from_kbuf(ctx, prec, n, L, kout, 4, outs, MFIC_OP_ASSIGN, 0.0, true);
    for (mfic_grid g : {phi3, A3x, A3y, A3z}) g->space = MFIC_KSPACE;
}

}  // namespace mfic
