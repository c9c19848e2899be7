// Fused padded row pass of the LPT sources (fused.hip).
#pragma once
#include <cstddef>

#include "mfic_internal.hpp"

namespace mfic {

enum class FusedKind {
    Src2,   // in: 6 phi1 Hessians; out: 2LPT source
    Src2Q,  // in: 6 phi1 Hessians; out: 2LPT source, Qzz, Qyz, Qxx, Qyy
    Src3,   // in: 6 phi1 + 6 phi2 Hessians + 4 Q; out: phi3 source, A3x, A3y, A3z
    Mul,       // in: two operands; out: their product
    Square,    // in: one operand; out: its square
    Adjoint2,  // in: 6 phi1 Hessians, lambda; out: lambda d(2LPT source)/d(Hessian), 6 products
};

// in / out: consecutive compact padded half-spectrum buffers ([Np][Np][N/2+1]
// complex each) after the axis-0 and axis-1 c2r passes / before the axis-1
// and axis-0 r2c passes
void fused_source_rows(mfic_ctx ctx, int prec, FusedKind kind, size_t n, const void* in, void* out);
// last (contiguous-axis) c2r pass of three component grids (k-space after the
// axis-0 and axis-1 passes, [n][n][n/2+1] complex) fused with the lattice
// readout into FP64 [p][3]; positions sit at (ijk + shift) cells per axis.
// Up to eight such sets (sub-lattices, positions and velocities) per call.
struct ParticleRows {
    const void* f[3];
    double* dst;
    int is_pos;
    double shift[3];
};
void rows_c2r_particles(mfic_ctx ctx, int prec, const ParticleRows* sets, int count, int n, double lunit);

}  // namespace mfic
