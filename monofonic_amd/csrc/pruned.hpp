// Pruned / fused 3/2-padded transforms (pruned.hip).
#pragma once
#include "mfic_internal.hpp"
#include "orszag.hpp"

namespace mfic {

// operands of N-grid k-space fields -> consecutive compact padded buffers
// ([Np][Np][N/2+1] complex each) after the axis-0 and axis-1 c2r passes
// (half-spectrum rows ready for a row pass) in a box of sides L; one or two
// operands
void padded_operands_to_kbuf(mfic_ctx ctx, int prec, const OperandDesc* o, int count, size_t n, const double L[3],
                             void* kbuf);
// the six Hessians xx yy zz xy xz yz of an N-grid k-space field -> six
// consecutive compact padded buffers (out) after the axis-0 and axis-1 c2r
// passes; xbuf is scratch for three compact buffers; weights64: gradient
// factors in FP64 whatever the precision
void padded_hessians_to_kbuf(mfic_ctx ctx, int prec, const void* f, size_t n, double L, void* xbuf, void* out,
                             bool weights64 = false);
// consecutive compact padded buffers of r2c'd rows of products (real space
// along axes 0 and 1) -> the same buffers truncated to the source modes with
// Nyquist planes zeroed and padded again, ready as inputs of a row pass: the
// unpad / pad_insert pair of a two-stage product, as two in-place filter passes
void padded_truncate_repad(mfic_ctx ctx, int prec, size_t n, void* kbuf, int count);
// consecutive compact padded buffers of r2c'd rows (one to four) -> axis-1
// and axis-0 r2c passes with the unpad rules, output operator and optional
// -1/k^2 into the N-grids out[]; kbuf is overwritten
void padded_r2c_from_kbuf(mfic_ctx ctx, int prec, size_t n, double L, void* kbuf, int count, void* const* out, int op,
                          double coef, bool invlap);

// the adjoint of the Hessian passes with the last stage of the 2LPT adjoint:
// six consecutive compact buffers of r2c'd rows (slot order as the Hessians)
// -> out = F(|n|^2) / volfac (g1 lam + sum_h -g_a g_b T(r_h)) in k-space with
// empty Nyquist planes, F the -A(k)/k^2 table of phi1_table; zbuf is scratch
// for three compact buffers
void padded_hessian_adjoint(mfic_ctx ctx, int prec, size_t n, double L, const void* prod, void* zbuf, const void* lam,
                            const double* tab, double g1, double volfac, void* out);

}  // namespace mfic
