// C ABI, differentiable 2LPT: forward map white noise -> 2LPT displacement
// and its adjoint (the maths is in adjoint.hip); plus wrapping of external
// device buffers as grids for framework bindings.  No reference
// counterpart: monofonIC has no derivative of its initial-condition map.
#include <cmath>
#include <memory>
#include <string>

#include "cosmology.hpp"
#include "fused.hpp"
#include "kspace.hpp"
#include "lpt.hpp"
#include "mfic_internal.hpp"
#include "orszag.hpp"
#include "pruned.hpp"

namespace mfic {
void kspace_grad_adjoint(mfic_grid lam, mfic_grid lmu, mfic_grid gx, mfic_grid gy, mfic_grid gz, double unit,
                         double g2);
}  // namespace mfic

using mfic::Error;

namespace {
void ck(int rc) {
    if (rc != MFIC_OK) throw Error(rc, mfic_last_error());
}
struct GridPtr {
    mfic_grid g = nullptr;
    GridPtr() = default;
    GridPtr(const GridPtr&) = delete;
    ~GridPtr() {
        if (g) (void)mfic_grid_destroy(g);
    }
};
}  // namespace

struct mfic_lpt2_s {
    mfic_ctx ctx = nullptr;
    size_t n = 0;
    double L = 0.0, unit = 1.0;
    int prec = MFIC_F32;
    mfic::EhParams eh{};
    mfic_lpt_coef coef{};
    GridPtr phi1, phi2, lam, lmu, t[3];
    std::unique_ptr<mfic::ConvCore> core;  // sizes of the padded passes
    void* ws = nullptr;    // compact padded buffers of the adjoint
    void* d_tk = nullptr;  // spline nodes of a tabulated transfer function
    ~mfic_lpt2_s() {
        if (ws) (void)hipFree(ws);
        if (d_tk) (void)hipFree(d_tk);
    }
};

namespace {
// compact padded buffers: Hessians of phi1 [0, 6), lam_mu [6], the six products
// [7, 13); the x powers pass through [7, 10) on the way in and [0, 3) on the
// way out
constexpr size_t WS_BUFFERS = 13;
void make(mfic_lpt2_s* p, GridPtr& g, int space) {
    const size_t n3[3] = {p->n, p->n, p->n};
    const double L3[3] = {p->L, p->L, p->L};
    ck(mfic_grid_create(p->ctx, n3, L3, p->prec, space, &g.g));
}
void check_io(const mfic_lpt2_s* p, mfic_grid g, const char* what) {
    MFIC_CHECK(g && g->d, MFIC_ERR_ARG, std::string("null grid: ") + what);
    MFIC_CHECK(g->n[0] == p->n && g->n[1] == p->n && g->n[2] == p->n && g->prec == p->prec, MFIC_ERR_ARG,
               std::string("grid size / precision differs from the plan: ") + what);
}
// r2c of real grids into k-space grids of the plan
template <typename T> void to_kspace(mfic_lpt2_s* p, mfic_grid* src, mfic_grid* dst, int count) {
    const T* s[3];
    T* d[3];
    for (int m = 0; m < count; ++m) {
        s[m] = static_cast<const T*>(src[m]->d);
        d[m] = static_cast<T*>(dst[m]->d);
        dst[m]->space = MFIC_KSPACE;
    }
    const size_t n3[3] = {p->n, p->n, p->n};
    mfic::fft_r2c<T>(p->ctx, s, d, count, n3, 1.0 / std::sqrt((double)p->n * p->n * p->n));
}
// c2r in place
template <typename T> void to_real(mfic_lpt2_s* p, mfic_grid* g, int count) {
    T* d[3];
    for (int m = 0; m < count; ++m) {
        d[m] = static_cast<T*>(g[m]->d);
        g[m]->space = MFIC_RSPACE;
    }
    const size_t n3[3] = {p->n, p->n, p->n};
    mfic::fft_c2r<T>(p->ctx, d, d, count, n3, 1.0 / std::sqrt((double)p->n * p->n * p->n));
}
// phi1 = S P_N r2c(noise) (the forward map's first linear stage)
void phi1_of(mfic_lpt2_s* p, mfic_grid noise) {
    if (p->prec == MFIC_F64) to_kspace<double>(p, &noise, &p->phi1.g, 1);
    else to_kspace<float>(p, &noise, &p->phi1.g, 1);
    mfic::phi1_from_noise(p->phi1.g, p->phi1.g, p->eh, p->coef.volfac, 0, 0, nullptr, true);
}
}  // namespace

extern "C" {

int mfic_grid_wrap(mfic_ctx ctx, const size_t n[3], const double L[3], int prec, int space, void* device_ptr,
                   mfic_grid* out) {
    return mfic::guard_call([&] {
        MFIC_CHECK(ctx && n && L && device_ptr && out, MFIC_ERR_ARG, "null argument");
        MFIC_CHECK(prec == MFIC_F32 || prec == MFIC_F64, MFIC_ERR_ARG, "precision must be MFIC_F32 or MFIC_F64");
        MFIC_CHECK(space == MFIC_KSPACE || space == MFIC_RSPACE, MFIC_ERR_ARG, "bad space");
        MFIC_CHECK(n[0] > 0 && n[1] > 0 && n[2] > 0 && n[2] % 2 == 0, MFIC_ERR_SIZE, "bad grid size");
        MFIC_CHECK(((uintptr_t)device_ptr % (prec == MFIC_F64 ? 16 : 8)) == 0, MFIC_ERR_ARG,
                   "device buffer must be aligned to one complex element");
        MFIC_HIP(hipSetDevice(ctx->device));
        mfic::require_device_memory(device_ptr, "the wrapped buffer");
        auto* g = new mfic_grid_s();
        g->ctx = ctx;
        for (int i = 0; i < 3; ++i) { g->n[i] = n[i]; g->L[i] = L[i]; }
        g->prec = prec;
        g->space = space;
        g->nreal = n[0] * n[1] * (n[2] + 2);
        g->d = device_ptr;
        g->owns = false;
        ++ctx->children;
        *out = g;
    });
}

int mfic_lpt2_create(mfic_ctx ctx, size_t n, double L, int prec, const mfic_cosmo_params* cosmo, double unit,
                     mfic_lpt2* out) {
    return mfic::guard_call([&] {
        MFIC_CHECK(ctx && cosmo && out, MFIC_ERR_ARG, "null argument");
        MFIC_CHECK(prec == MFIC_F32 || prec == MFIC_F64, MFIC_ERR_ARG, "bad precision");
        MFIC_CHECK(L > 0.0, MFIC_ERR_CONFIG, "BoxLength must be positive");
        auto p = std::make_unique<mfic_lpt2_s>();
        p->ctx = ctx;
        p->n = n;
        p->L = L;
        p->prec = prec;
        p->unit = unit;
        mfic_cosmo_scalars sc;
        mfic::cosmo_compute(*cosmo, &sc, &p->eh);
        {
            const size_t n3[3] = {n, n, n};
            const double L3[3] = {L, L, L};
            mfic::check_tk_range(*cosmo, n3, L3);
        }
        p->d_tk = mfic::tk_upload(*cosmo, &p->eh);
        ck(mfic_lpt_coefficients(cosmo, n, L, 2, &p->coef));
        make(p.get(), p->phi1, MFIC_KSPACE);
        make(p.get(), p->phi2, MFIC_KSPACE);
        make(p.get(), p->lam, MFIC_KSPACE);
        make(p.get(), p->lmu, MFIC_KSPACE);
        for (auto& t : p->t) make(p.get(), t, MFIC_KSPACE);
        const size_t n3[3] = {n, n, n};
        const double L3[3] = {L, L, L};
        p->core = std::make_unique<mfic::ConvCore>(ctx, n3, L3, prec);
        const size_t wsb = WS_BUFFERS * p->core->kbuf_reals() * p->core->esize();
        p->ws = mfic::device_alloc(wsb);
        MFIC_CHECK(p->ws, MFIC_ERR_ALLOC, "2LPT plan: workspace allocation of " + std::to_string(wsb) + " bytes failed");
        ++ctx->children;
        *out = p.release();
    });
}

int mfic_lpt2_destroy(mfic_lpt2 p) {
    return mfic::guard_call([&] {
        if (!p) return;
        (void)hipStreamSynchronize(p->ctx->stream);
        mfic_ctx ctx = p->ctx;
        delete p;
        --ctx->children;
    });
}

int mfic_lpt2_forward(mfic_lpt2 p, mfic_grid noise, mfic_grid psi_x, mfic_grid psi_y, mfic_grid psi_z) {
    return mfic::guard_call([&] {
        MFIC_CHECK(p, MFIC_ERR_ARG, "null plan");
        check_io(p, noise, "noise");
        mfic_grid psi[3] = {psi_x, psi_y, psi_z};
        for (auto g : psi) check_io(p, g, "displacement");
        phi1_of(p, noise);
        mfic::lpt_sources(p->ctx, 2, p->phi1.g, p->phi2.g, nullptr, nullptr, nullptr, nullptr);
        // the three components in one pass over phi1 and phi2
        const double cf[4] = {p->coef.g1, p->coef.g2, 0.0, 0.0};
        const void* phi[3] = {p->phi1.g->d, p->phi2.g->d, nullptr};
        const void* A3[3] = {nullptr, nullptr, nullptr};
        // a buffer given for two components ends up with the later one
        for (int d = 0; d < 2; ++d)
            for (int e = d + 1; e < 3; ++e)
                if (psi[d]->d == psi[e]->d) {
                    psi[d]->space = MFIC_RSPACE;
                    psi[d] = p->t[d].g;
                    break;
                }
        void* outs[12] = {psi[0]->d, psi[1]->d, psi[2]->d};
        mfic::assemble_all(p->ctx, p->prec, p->n, p->L, 2, cf, cf, p->unit, p->unit, mfic::PltDev{}, phi, A3, outs, 1);
        if (p->prec == MFIC_F64) to_real<double>(p, psi, 3);
        else to_real<float>(p, psi, 3);
    });
}

int mfic_lpt2_adjoint(mfic_lpt2 p, mfic_grid noise, mfic_grid cot_x, mfic_grid cot_y, mfic_grid cot_z,
                      mfic_grid grad) {
    return mfic::guard_call([&] {
        MFIC_CHECK(p, MFIC_ERR_ARG, "null plan");
        check_io(p, noise, "noise");
        check_io(p, grad, "gradient");
        mfic_grid cot[3] = {cot_x, cot_y, cot_z};
        for (auto g : cot) check_io(p, g, "cotangent");
        phi1_of(p, noise);  // recomputed, not stored by the forward call
        mfic_grid t[3] = {p->t[0].g, p->t[1].g, p->t[2].g};
        if (p->prec == MFIC_F64) to_kspace<double>(p, cot, t, 3);
        else to_kspace<float>(p, cot, t, 3);
        // lam = unit sum_d (-i g_d) G_d (adjoint of the gradient, unit and
        // DC := 0) and lam_mu = P_N lap^-1 (g2 lam) of the phi2 branch
        mfic::kspace_grad_adjoint(p->lam.g, p->lmu.g, t[0], t[1], t[2], p->unit, p->coef.g2);
        const size_t kb = p->core->kbuf_reals() * p->core->esize();
        char* ws = static_cast<char*>(p->ws);
        mfic::padded_hessians_to_kbuf(p->ctx, p->prec, p->phi1.g->d, p->n, p->L, ws + 7 * kb, ws, true);
        const mfic::OperandDesc lmu{p->lmu.g->d, MFIC_OPND_IDENT, {0, 0, 0, 0}};
        mfic::padded_operands_to_kbuf(p->ctx, p->prec, &lmu, 1, p->n, p->core->len, ws + 6 * kb);
        mfic::fused_source_rows(p->ctx, p->prec, mfic::FusedKind::Adjoint2, p->n, ws, ws + 7 * kb);
        // phi1 branch and the adjoint of phi1 = S P_N r2c(noise)
        mfic::padded_hessian_adjoint(p->ctx, p->prec, p->n, p->L, ws + 7 * kb, ws, p->lam.g->d,
                                     mfic::phi1_table(p->phi1.g, p->eh), p->coef.g1, p->coef.volfac, grad->d);
        if (p->prec == MFIC_F64) to_real<double>(p, &grad, 1);
        else to_real<float>(p, &grad, 1);
    });
}

}  // extern "C"
