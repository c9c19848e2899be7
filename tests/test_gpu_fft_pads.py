"""Tiles and LDS pads of the N-grid strided passes: the pitch moves the
exchange and the twiddles behind it, not the arithmetic, so every override
gives the bits of the built-in choice.  9 is the one odd length: with an odd
pad its exchange has an odd number of reals."""
import ctypes as C

import numpy as np
import pytest
import torch  # noqa: F401  before the library, whose HIP runtime is then torch's

from monofonic_amd import F32, F64, Grid, _lib as L


def transform(ctx, x, prec):
    g = Grid(ctx, x.shape, (10.0,) * 3, prec=prec)
    a = np.zeros(g.shape_real)
    a[:, :, : x.shape[2]] = x
    g.upload(a)
    g.FourierTransformForward()
    k = g.download_k().copy()
    g.FourierTransformBackward()
    r = g.download_r().copy()
    g.close()
    return k, r


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [F32, F64])
@pytest.mark.parametrize("shape", [(9, 9, 12), (9, 18, 16), (48, 9, 24), (36, 64, 18)])
def test_pads_change_nothing(ctx, shape, prec):
    x = np.random.default_rng(sum(shape)).standard_normal(shape)
    want = transform(ctx, x, prec)
    assert np.linalg.norm(want[0] - np.fft.rfftn(x, norm="ortho")) < (1e-12 if prec == F64 else 2e-6) * np.linalg.norm(x)
    lengths = set(shape[:2])
    try:
        for tile in (1, 4, 16, 64):
            for pad in (0, 1, 3, 8):
                for n in lengths:
                    L.call("mfic_fft_set_tile", ctx.h, n, 0, prec, tile, pad)
                for a, b in zip(transform(ctx, x, prec), want):
                    assert np.array_equal(a, b), (tile, pad)
    finally:
        for n in lengths:
            L.call("mfic_fft_set_tile", ctx.h, n, 0, prec, 0, 0)


@pytest.mark.gpu
def test_reported_tiles_are_those_that_run(ctx):
    t, pad = C.c_int(), C.c_int()
    for length, kind in ((64, 0), (64, 1), (64, 2), (96, L.PASS_PAD_C2R_A), (96, L.PASS_TRUNC_AX1)):
        try:
            for tile in (1, 2, 4, 16):
                L.call("mfic_fft_set_tile", ctx.h, length, kind, F32, tile, 0)
                L.call("mfic_fft_get_tile", ctx.h, length, kind, F32, C.byref(t), C.byref(pad))
                assert t.value == (tile if kind == 1 else max(tile, 4)), (length, kind, tile)
        finally:
            L.call("mfic_fft_set_tile", ctx.h, length, kind, F32, 0, 0)
