"""Shapes of boxes in the convolver and the LPT sources.  Grids that their
passes would address with another grid's strides are refused on the host,
before anything is launched: unequal sizes per axis, operands and outputs of
another size or precision.  A convolver's gradients follow the box side of
their own axis; the sources and the assembly, which have one side, refuse
unequal ones."""
import ctypes as C
import itertools

import numpy as np
import pytest
import torch  # noqa: F401  before the library, whose HIP runtime is then torch's

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


def padded_real(f, n, m):
    """values on the m^3 grid of the modes f of an n^3 field (complex128,
    [n][n][n/2+1], empty Nyquist planes), unnormalised"""
    p = np.zeros((m, m, m // 2 + 1), dtype=np.complex128)
    h = n // 2
    at = [(slice(0, h), slice(0, h)), (slice(-h + 1, None), slice(-h + 1, None))]
    for si, di in at:
        for sj, dj in at:
            p[di, dj, :h] = f[si, sj, :h]
    return np.fft.irfftn(p, s=(m, m, m), axes=(0, 1, 2)) * m ** 3


def truncated(r, n, m):
    p = np.fft.rfftn(r) / m ** 3
    h = n // 2
    f = np.zeros((n, n, h + 1), dtype=np.complex128)
    at = [slice(0, h), slice(-h + 1, None)]
    for si in at:
        for sj in at:
            f[si, sj, :h] = p[si, sj, :h]
    return f


@pytest.mark.gpu
@pytest.mark.parametrize("n,prec,sides", [(16, F64, (20.0, 35.0, 50.0)), (24, F64, (50.0, 20.0, 20.0)),
                                          (32, F32, (20.0, 20.0, 31.0))])
def test_gradients_follow_their_axis(ctx, n, prec, sides):
    """every operand kind in a box of unequal sides against numpy in 64 bits
    (the tolerances of the convolver tests: FP64 1e-10, FP32 1e-5 rel-L2)"""
    rng = np.random.default_rng(n)
    h, m = n // 2, 3 * n // 2
    f = []
    for _ in range(2):  # real fields without Nyquist planes
        k = np.fft.rfftn(rng.standard_normal((n, n, n))) / n ** 1.5
        k[h], k[:, h], k[:, :, h] = 0, 0, 0
        f.append(k.astype(np.complex64).astype(np.complex128) if prec == F32 else k)
    idx = np.fft.fftfreq(n, 1.0 / n)
    g = [2 * np.pi / s * x for s, x in zip(sides, np.meshgrid(idx, idx, np.arange(h + 1.0), indexing="ij"))]
    kinds = {"hess": (L.HESS, (0, 1), -g[0] * g[1]), "hess2": (L.HESS, (2, 2), -g[2] * g[2]),
             "sum": (L.SUM_HESS, (0, 0, 1, 2), -g[0] * g[0] - g[1] * g[2]),
             "diff": (L.DIFF_HESS, (1, 1, 0, 2), -g[1] * g[1] + g[0] * g[2]),
             "grad": (L.GRAD, (1,), 1j * g[1]), "ident": (L.IDENT, (), 1.0)}
    grids = [Grid(ctx, (n,) * 3, sides, prec=prec, space=L.KSPACE) for _ in range(3)]
    for gr, k in zip(grids, f):
        gr.upload_k(k)
    conv = lpt.OrszagConvolver(ctx, (n,) * 3, sides, prec)
    for a, b in (("hess", "hess2"), ("sum", "grad"), ("diff", "ident"), ("grad", "hess"), ("hess2", "sum")):
        conv.convolve2(lpt._operand(grids[0], *kinds[a][:2]), lpt._operand(grids[1], *kinds[b][:2]), grids[2])
        # unitary transforms of an n^3 grid: a product of fields carries n^{-3/2}
        want = truncated(padded_real(f[0] * kinds[a][2], n, m) * padded_real(f[1] * kinds[b][2], n, m), n, m) / n ** 1.5
        got = grids[2].download_k()
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        print(f"n {n} sides {sides} {a} x {b}: {err:.1e}")
        assert err < (1e-10 if prec == F64 else 1e-5), (a, b, err)
    for x in (conv, *grids):
        x.close()


@pytest.mark.gpu
@pytest.mark.parametrize("sides", [(20.0, 20.0, 21.0), (20.0, 19.0, 20.0), (21.0, 20.0, 20.0)])
def test_unequal_sides_of_a_potential_are_refused(ctx, sides):
    g = [Grid(ctx, (16,) * 3, sides, prec=F64, space=L.KSPACE) for _ in range(2)]
    out = Grid(ctx, (16,) * 3, sides, prec=F64, space=L.KSPACE)
    coef = lpt.lpt_coefficients(lpt.baseline_cosmology(24.0), 16, 20.0, 2)
    assert status("mfic_lpt_sources", ctx.h, 2, g[0].h, g[1].h, None, None, None, None) == ERR_SIZE
    assert status("mfic_lpt_component", ctx.h, 2, 0, C.byref(coef), None, 1.0, g[0].h, g[1].h, None, None, None, None,
                  out.h) == ERR_SIZE
    for x in (*g, out):
        x.close()


@pytest.mark.gpu
@pytest.mark.parametrize("prec,n", [(F64, 32), (F32, 96)])
@pytest.mark.parametrize("same", [(0, 1), (1, 2, 3), (0, 3), (0, 1, 2, 3)])
def test_one_grid_for_several_potentials(ctx, same, prec, n):
    """of phi3, A3x, A3y, A3z given the same grid, it holds the last"""
    g = [k_grid(ctx, n, prec) for _ in range(6)]
    lpt.ngenic_fill(g[0], 4)
    lpt.lpt_sources(ctx, 3, g[0], g[1], g[2], g[3:])
    want = [x.download_k().copy() for x in g[2:]]
    out = [g[2 + (same[0] if i in same else i)] for i in range(4)]
    for rep in range(3):
        for x in g[1:]:
            x.zero()
        lpt.lpt_sources(ctx, 3, g[0], g[1], out[0], out[1:])
        for i in range(4):
            assert np.array_equal(out[i].download_k(), want[same[-1] if i in same else i]), (rep, i)
    for x in g:
        x.close()
