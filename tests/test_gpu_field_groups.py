"""Passes over several fields per launch: the sub-lattice passes of grouped
components, and convolver products through the fused row pass: operands of
very different size (a product must keep the precision of the smaller one),
squares, and a square against the general product.  Tolerances are those of
the convolver tests (FP64 1e-10, FP32 1e-5 rel-L2)."""
import numpy as np
import pytest

from monofonic_amd import F32, F64, Grid, _lib as L, lpt
from oracle import oracle as O

from _gpu_helpers import rel_l2

TOL = {F64: 1e-10, F32: 1e-5}


def k_grid(ctx, field, prec, box):
    n = field.shape[0]
    g = Grid(ctx, (n,) * 3, (box,) * 3, prec=prec)
    g.upload(field)
    g.set_space(L.KSPACE)
    return g


@pytest.mark.gpu
@pytest.mark.parametrize("n,prec", [(8, F32), (24, F64), (32, F32), (48, F32), (64, F64)])
def test_products_of_unequal_operands(ctx, n, prec):
    box = 40.0
    a, b = O.ngenic_fill(5, n), O.ngenic_fill(6, n) * 1e6
    ga, gb = k_grid(ctx, a, prec, box), k_grid(ctx, b, prec, box)
    go = Grid(ctx, (n,) * 3, (box,) * 3, prec=prec, space=L.KSPACE)
    conv = lpt.OrszagConvolver(ctx, (n,) * 3, (box,) * 3, prec)
    kinds = {"hess": (L.HESS, O.HESS, (0, 1)), "ident": (L.IDENT, O.IDENT, (0, 0)), "grad": (L.GRAD, O.GRAD, (2, 0)),
             "sum": (L.SUM_HESS, O.SUM_HESS, (0, 0, 1, 2))}
    for ka, kb in (("hess", "ident"), ("grad", "sum"), ("ident", "hess")):
        ref = O.empty_field(n)
        da, db = kinds[ka][2], kinds[kb][2]
        pad = lambda d: tuple(d) + (0,) * (4 - len(d))  # noqa: E731
        O.convolve2(n, box, O.operand(a, kinds[ka][1], pad(da)), O.operand(b, kinds[kb][1], pad(db)), ref, O.ASSIGN)
        conv.convolve2(lpt._operand(ga, kinds[ka][0], da), lpt._operand(gb, kinds[kb][0], db), go)
        err = rel_l2(go.download_k(), O.kview(ref))
        assert err < TOL[prec], (ka, kb, err)
    # cubic product whose first stage is far smaller than the third operand
    ref = O.empty_field(n)
    h = (0, 0, 0, 0)
    O.convolve3(n, box, O.operand(a, O.HESS, h), O.operand(a, O.HESS, (1, 1, 0, 0)), O.operand(b, O.HESS, (2, 2, 0, 0)),
                ref, O.ASSIGN)
    conv.convolve3(lpt._operand(ga, L.HESS, (0, 0)), lpt._operand(ga, L.HESS, (1, 1)), lpt._operand(gb, L.HESS, (2, 2)),
                   go)
    assert rel_l2(go.download_k(), O.kview(ref)) < TOL[prec]
    for x in (conv, ga, gb, go):
        x.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,prec", [(8, F64), (24, F32), (32, F64), (96, F32)])
def test_square_is_the_general_product(ctx, n, prec):
    """one operand given twice takes the path that transforms it once; the
    same values in another grid take the general one; unused direction slots
    do not matter"""
    box = 30.0
    f = O.ngenic_fill(9, n)
    g1, g2 = k_grid(ctx, f, prec, box), k_grid(ctx, f, prec, box)
    outs = [Grid(ctx, (n,) * 3, (box,) * 3, prec=prec, space=L.KSPACE) for _ in range(3)]
    conv = lpt.OrszagConvolver(ctx, (n,) * 3, (box,) * 3, prec)
    a = lpt._operand(g1, L.HESS, (0, 2))
    conv.convolve2(a, lpt._operand(g1, L.HESS, (0, 2, 1, 1)), outs[0])
    conv.convolve2(a, lpt._operand(g2, L.HESS, (0, 2)), outs[1])
    conv.convolve2(a, lpt._operand(g1, L.HESS, (2, 0)), outs[2])  # the same Hessian, other order
    ref = O.empty_field(n)
    o = O.operand(f, O.HESS, (0, 2, 0, 0))
    O.convolve2(n, box, o, o, ref, O.ASSIGN)
    for g in outs:
        assert rel_l2(g.download_k(), O.kview(ref)) < TOL[prec]
    for x in (conv, g1, g2, *outs):
        x.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,lattice,baryons,prec", [(16, L.FCC, True, F64), (24, L.BCC, False, F32),
                                                    (48, L.FCC, False, F64), (96, L.SC, False, F64)])
def test_grouped_components(ctx, n, lattice, baryons, prec):
    """particles of a run (components and sub-lattices grouped into launches)
    against the per-component entry points"""
    box, order = 100.0, 1
    cfg = lpt.ICConfig(n=n, box=box, zstart=24.0, lpt_order=order, lattice=lattice, prec=prec, seed=3, particles=True,
                       baryons=baryons)
    run = lpt.ICRun(ctx, cfg)
    run.execute()
    first = [run.particles(b) for b in ((False, True) if baryons else (False,))]
    run.execute()  # the components are rebuilt from the potentials
    coef = lpt.lpt_coefficients(lpt.baseline_cosmology(24.0), n, box, order)
    import torch
    for idx, (pos, vel) in enumerate(first):
        again = run.particles(bool(idx))
        assert np.array_equal(again[0], pos) and np.array_equal(again[1], vel)
        for d in range(3):
            for comp, want, is_pos in ((d, pos, 1), (d + 3, vel, 0)):
                f = Grid(ctx, (n,) * 3, (box,) * 3, prec=prec, space=L.KSPACE)
                lpt.lpt_component(ctx, order, comp, coef, (run.potential(0), None, None, (None,) * 3), f, 1.0 / box * box / box)
                f.FourierTransformBackward()
                dst = torch.zeros(3 * len(pos), dtype=torch.float64, device="cuda")
                torch.cuda.synchronize()
                L.call("mfic_lattice_readout_index", f.h, lattice, idx, d, is_pos, 1.0, dst.data_ptr())
                ctx.sync()
                got = dst.cpu().numpy().reshape(-1, 3)[:, d]
                scale = np.abs(want[:, d] - (np.round(want[:, d] * 2 * n) / (2 * n) if is_pos else 0.0)).max()
                assert np.abs(got - want[:, d]).max() < (1e-10 if prec == F64 else 2e-5) * max(scale, 1e-3), (idx, comp)
                f.close()
    run.close()
