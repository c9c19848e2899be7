// Orszag 3/2 convolver core and the reorganised LPT source schedule.
#pragma once
#include "mfic_internal.hpp"

namespace mfic {

struct OperandDesc {
    const void* f;  // k-space N-grid field (device)
    int kind;       // mfic_opkind
    int d[4];
    bool same(const OperandDesc& o) const {
        if (f != o.f || kind != o.kind) return false;
        const int used = kind == MFIC_OPND_IDENT ? 0 : kind == MFIC_OPND_GRAD ? 1 : kind == MFIC_OPND_HESS ? 2 : 4;
        for (int i = 0; i < used; ++i)
            if (d[i] != o.d[i]) return false;
        return true;
    }
};

// Padded-grid operations for one N-grid size (OrszagConvolver, convolution.hh:412-651)
struct ConvCore {
    mfic_ctx ctx;
    int prec;
    size_t N[3], Np[3];
    double len[3];
    ConvCore(mfic_ctx c, const size_t n[3], const double L[3], int prec);
    size_t grid_reals() const;
    size_t esize() const;
    // reals of a compact padded buffer ([Np][Np][N/2+1] complex)
    size_t kbuf_reals() const;
    // kbuf: three compact buffers; fbuf: an N-grid
    void convolve2(const OperandDesc& a, const OperandDesc& b, void* out, int op, double coef, void* kbuf) const;
    void convolve3(const OperandDesc& a, const OperandDesc& b, const OperandDesc& c, void* out, int op, double coef,
                   void* kbuf, void* fbuf) const;
};

// phi2 (order >= 2), phi3 / A3 (order 3) from phi1, inverse Laplacian applied,
// growth factors not applied
void lpt_sources(mfic_ctx ctx, int order, mfic_grid phi1, mfic_grid phi2, mfic_grid phi3, mfic_grid A3x,
                 mfic_grid A3y, mfic_grid A3z);

}  // namespace mfic
