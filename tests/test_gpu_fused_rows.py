"""The two forms of the fused row pass of the LPT sources against each other:
two rows per full-length complex transform (in halves, with the factors in
LDS) and one row per half-length transform, which share no transform code
beyond the butterflies.  Every padded length they are built for: one and
several transforms to a wavefront, blocks of several rows, 12 and 24 values to
a thread.  FP64: the forms against each other to 1e-13 rel-L2 (rounding of two
transforms of ~10 stages; the cubic terms pass through two products, twice
that).  FP32: the error of the paired form against FP64 is
at most twice that of the half-length form.  (No absolute bound there: the
inverse Laplacian weighs the white rounding noise of the sources towards the
low modes, where the sources themselves vanish, so the error of either form
grows with n.)"""
import numpy as np
import pytest

from monofonic_amd import F32, F64, Grid, _lib as L, batch, lpt

from _gpu_helpers import rel_l2


def potentials(ctx, n, prec, form):
    grids = [Grid(ctx, (n,) * 3, (50.0,) * 3, prec=prec, space=L.KSPACE) for _ in range(6)]
    lpt.ngenic_fill(grids[0], 7)
    batch.set_plan(ctx, 3 * n // 2, L.PASS_FUSED_ROWS, prec, form)
    try:
        lpt.lpt_sources(ctx, 3, grids[0], grids[1], grids[2], grids[3:])
    finally:
        batch.set_plan(ctx, 3 * n // 2, L.PASS_FUSED_ROWS, prec, -1)
    out = [g.download_k().copy() for g in grids[1:]]
    for g in grids:
        g.close()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("n", [8, 16, 24, 32, 48, 64, 96, 128, 192, 256, 384])
def test_forms_agree(ctx, n):
    ref = potentials(ctx, n, F64, 1)
    for i, (a, b) in enumerate(zip(potentials(ctx, n, F64, 0), ref)):
        err = rel_l2(a, b)
        assert err < 1e-13 * (1 if i == 0 else 2), (i, err)
    errs = [[rel_l2(np.asarray(a, dtype=np.complex128), b) for a, b in zip(potentials(ctx, n, F32, form), ref)]
            for form in (0, 1)]
    assert all(e0 <= 2 * e1 for e0, e1 in zip(*errs)), errs
