"""Grids that the convolver's and the LPT sources' passes would address with
another grid's strides are refused on the host, before anything is launched:
unequal sizes per axis, operands and outputs of another size or precision."""
import ctypes as C
import itertools

import numpy as np
import pytest

from monofonic_amd import F32, F64, Grid, _lib as L, lpt

ERR_ARG, ERR_SIZE = -1, -2


def status(name, *args):
    return getattr(L.load(), name)(*args)


@pytest.mark.parametrize("n", [(32, 16, 16), (16, 32, 16), (16, 16, 32), (12, 16, 24), (48, 16, 16)])
def test_unequal_sizes_are_refused_before_any_device_call(n):
    """the size check precedes the first use of the context, so a zeroed block
    stands for one and no device is needed"""
    block = C.create_string_buffer(1 << 14)
    h = C.c_void_p()
    rc = status("mfic_conv_create", C.cast(block, C.c_void_p), (C.c_size_t * 3)(*n), (C.c_double * 3)(1, 1, 1), F64,
                C.byref(h))
    assert rc == ERR_SIZE and not h
    assert b"same grid size" in L.load().mfic_last_error()


def k_grid(ctx, n, prec):
    return Grid(ctx, (n,) * 3, (20.0,) * 3, prec=prec, space=L.KSPACE)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [F32, F64])
def test_operands_match_the_convolver(ctx, prec):
    n, other = 16, F32 if prec == F64 else F64
    conv = lpt.OrszagConvolver(ctx, (n,) * 3, (20.0,) * 3, prec)
    good, out = k_grid(ctx, n, prec), k_grid(ctx, n, prec)
    bad = [k_grid(ctx, n, other), k_grid(ctx, 8, prec), k_grid(ctx, 32, prec)]
    op = lambda g: lpt._operand(g, L.IDENT, ())  # noqa: E731
    before = out.download_k().copy()
    for g in bad:
        for a, b in ((g, good), (good, g)):
            assert status("mfic_conv_convolve2", conv.h, C.byref(op(a)), C.byref(op(b)), out.h, L.OP_ASSIGN, 0.0) == ERR_ARG
        for at in range(3):
            o = [op(g if i == at else good) for i in range(3)]
            assert status("mfic_conv_convolve3", conv.h, *[C.byref(x) for x in o], out.h, L.OP_ASSIGN, 0.0) == ERR_ARG
        assert status("mfic_conv_convolve2", conv.h, C.byref(op(good)), C.byref(op(good)), g.h, L.OP_ASSIGN, 0.0) == ERR_ARG
    assert np.array_equal(out.download_k(), before)
    for x in (conv, good, out, *bad):
        x.close()


@pytest.mark.gpu
def test_potentials_match_phi1(ctx):
    n = 16
    g = [k_grid(ctx, n, F64) for _ in range(6)]
    bad = [k_grid(ctx, n, F32), k_grid(ctx, 8, F64), k_grid(ctx, 32, F64)]
    coef = lpt.lpt_coefficients(lpt.baseline_cosmology(24.0), n, 20.0, 3)
    out = k_grid(ctx, n, F64)
    for b, at in itertools.product(bad, range(1, 6)):
        h = [(b if i == at else x).h for i, x in enumerate(g)]
        assert status("mfic_lpt_sources", ctx.h, 3, *h) == ERR_ARG
        assert status("mfic_lpt_component", ctx.h, 3, 0, C.byref(coef), None, 1.0, *h, out.h) == ERR_ARG
    for b in bad:
        assert status("mfic_lpt_component", ctx.h, 3, 0, C.byref(coef), None, 1.0, *[x.h for x in g], b.h) == ERR_ARG
    for x in (*g, *bad, out):
        x.close()
