"""Padded passes and row products at the lengths above 384 points, where other
plans and tiles take over, with bounds from rounding theory: with unit roundoff
eps a transform has a relative error of about eps sqrt(log2 of its points) in
the norm (rounding at random, half an ulp a stage), and a path through several
adds their squares.  References in 64 bits: torch transforms for products, the
transpose identity (exact for a quadratic map) for the adjoint, and the FP64
sources for the FP32 ones, compared before the inverse Laplacian, which would
weigh the rounding noise of the sources towards the modes where they vanish."""
import math

import pytest
import torch

from monofonic_amd import F32, F64, Grid, _lib as L, batch, lpt
from monofonic_amd.adjoint import LPT2
from monofonic_amd.lpt import _operand

EPS = 2.0 ** -24
# the terms of the 2LPT source cancel: root sum of their squared norms over the
# norm of their sum, for white noise in 64 bits
CANCEL = 2.1


def k_grid(ctx, n, prec, box=50.0):
    return Grid(ctx, (n,) * 3, (box,) * 3, prec=prec, space=L.KSPACE)


def on_gpu(grid):
    return torch.tensor(grid.download_k(), device="cuda")


def band(n):
    """the modes of an n^3 spectrum that are no Nyquist mode, and their place in
    the spectrum of a 3n/2 grid"""
    i = torch.cat([torch.arange(0, n // 2), torch.arange(n // 2 + 1, n)])
    return i.cuda(), torch.where(i > n // 2, i + n // 2, i).cuda()


def padded(k, n):
    m = 3 * n // 2
    src, dst = band(n)
    p = torch.zeros(m, m, m // 2 + 1, dtype=torch.complex128, device="cuda")
    p[dst[:, None], dst[None, :], : n // 2] = k[src][:, src, : n // 2]
    return torch.fft.irfftn(p, s=(m, m, m), norm="ortho") * 1.5 ** 1.5


def truncated(r, n):
    src, dst = band(n)
    p = torch.fft.rfftn(r, norm="ortho") / 1.5 ** 1.5
    k = torch.zeros(n, n, n // 2 + 1, dtype=torch.complex128, device="cuda")
    k[src[:, None], src[None, :], : n // 2] = p[dst][:, dst, : n // 2]
    return k


def rel(a, b):
    return ((a - b).norm() / b.norm()).item()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [96, 128, 192, 256, 384, 512])
def test_products(ctx, n):
    """general product and square: three transforms of 3 log2(3n/2) stages, the
    operands' errors and the result's; a margin of two"""
    print(f"products n={n}", flush=True)
    for prec in (F32, F64):
        g = [k_grid(ctx, n, prec) for _ in range(3)]
        lpt.ngenic_fill(g[0], 5)
        lpt.ngenic_fill(g[1], 6)
        conv = lpt.OrszagConvolver(ctx, (n,) * 3, (50.0,) * 3, prec)
        a, b = [padded(on_gpu(x), n) for x in g[:2]]
        bound = 2 * (EPS if prec == F32 else 2.0 ** -53) * math.sqrt(3 * 3 * math.log2(1.5 * n))
        for name, rb, other in (("general", b, g[1]), ("square", a, g[0])):
            conv.convolve2(_operand(g[0], L.IDENT, ()), _operand(other, L.IDENT, ()), g[2])
            want = truncated(a * rb, n)
            err = rel(on_gpu(g[2]), want)
            print(f"  {name} prec {prec}: {err:.2e} (bound {bound:.2e})", flush=True)
            assert err < bound
            del want
        del a, b
        for x in (conv, *g):
            x.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [32, 96, 192, 256, 384, 512])
@pytest.mark.parametrize("form", [0, 1])
def test_fp32_sources(ctx, n, form):
    """both forms of the row passes: errors of k^2 phi2 (products of two fields,
    whose cancellation weighs the errors of the terms) and of k^2 phi3, k^2 A3
    (the inner product's error, three more transforms and the terms of the outer
    product) against the FP64 sources of the same noise; a margin of two"""
    print(f"sources n={n} form={form}", flush=True)
    k = torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64, device="cuda")
    k2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + torch.arange(n // 2 + 1, device="cuda")[None, None, :] ** 2
    out = {}
    for prec in (F64, F32):
        g = [k_grid(ctx, n, prec) for _ in range(6)]
        lpt.ngenic_fill(g[0], 7)
        batch.set_plan(ctx, 3 * n // 2, L.PASS_FUSED_ROWS, prec, form)
        try:
            lpt.lpt_sources(ctx, 3, g[0], g[1], g[2], g[3:])
        finally:
            batch.set_plan(ctx, 3 * n // 2, L.PASS_FUSED_ROWS, prec, -1)
        if prec == F64:
            out = [(on_gpu(x) * k2).cpu() for x in g[1:]]
        else:
            stages = 3 * math.log2(1.5 * n)
            for i, x in enumerate(g[1:]):
                err = rel(on_gpu(x) * k2, out[i].cuda())
                bound = 2 * EPS * (CANCEL * math.sqrt(3 * stages) if i == 0 else CANCEL ** 2 * math.sqrt(6 * stages))
                print(f"  field {i}: {err:.2e} (bound {bound:.2e})", flush=True)
                assert err < bound, i
        for x in g:
            x.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [32, 128, 256, 384, 512])
def test_adjoint(ctx, n):
    """FP64 (to 384): the transpose identity.  FP32: two transforms of 3 log2 n
    stages (cotangents in, gradient out) dominate, the second-order branch is
    smaller; a margin of two"""
    print(f"adjoint n={n}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    draw = lambda *s: torch.randn(*s, generator=gen, device="cuda").double()  # noqa: E731
    x, C = draw(n, n, n), draw(3, n, n, n)
    p64 = LPT2(ctx, n, 100.0, prec=F64)
    grad = p64.adjoint(x, C).contiguous()
    if n <= 384:
        v = draw(n, n, n)
        jv = (p64.forward(x + 0.5 * v) - p64.forward(x - 0.5 * v)).contiguous()
        lhs, rhs = (jv * C).sum().item(), (grad * v).sum().item()
        assert abs(lhs - rhs) <= 1e-11 * jv.norm().item() * C.norm().item()
        del jv, v
    p64.close()
    p32 = LPT2(ctx, n, 100.0, prec=F32)
    err = rel(p32.adjoint(x.float(), C.float()).double(), grad)
    p32.close()
    bound = 2 * EPS * math.sqrt(2 * 3 * math.log2(n))
    print(f"  FP32: {err:.2e} (bound {bound:.2e})", flush=True)
    assert err < bound
