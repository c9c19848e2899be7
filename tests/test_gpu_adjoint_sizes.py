"""The padded passes of the 2LPT adjoint at the sizes where their tiles and
plans change: against the forward map by the dot-product identity, which is
exact for a quadratic map (central difference), and FP32 against FP64."""
import pytest

from monofonic_amd import F32, F64

torch = pytest.importorskip("torch")
from monofonic_amd.adjoint import LPT2  # noqa: E402

# smallest, a column count that is no multiple of a tile, several tiles,
# three-times-a-power sizes and the long plans
SIZES = [16, 32, 48, 64, 96, 128, 192, 256]


@pytest.mark.gpu
@pytest.mark.parametrize("n", SIZES)
def test_adjoint_is_the_transpose(ctx, n):
    box = 100.0
    rng = torch.Generator().manual_seed(n)
    draw = lambda *s: torch.randn(*s, generator=rng, dtype=torch.float64).cuda()  # noqa: E731
    x, v, C = draw(n, n, n), draw(n, n, n), draw(3, n, n, n)
    plan = LPT2(ctx, n, box, prec=F64)
    grad = plan.adjoint(x, C)
    eps = 0.5
    jv = (plan.forward(x + eps * v) - plan.forward(x - eps * v)) / (2 * eps)
    lhs, rhs = (jv * C).sum().item(), (grad * v).sum().item()
    plan.close()
    # rounding of sums of random terms, relative to their norms
    scale = jv.norm().item() * C.norm().item()
    print(f"n {n}: {lhs:.12e} {rhs:.12e} diff/scale {abs(lhs - rhs) / scale:.1e}")
    assert abs(lhs - rhs) <= 1e-11 * scale
    p32 = LPT2(ctx, n, box, prec=F32)
    g32 = p32.adjoint(x.float(), C.float()).double()
    p32.close()
    assert ((g32 - grad).norm() / grad.norm()).item() < 5e-6


@pytest.mark.gpu
def test_one_buffer_for_two_components(ctx):
    """a displacement grid given twice holds the later component; the gradient
    may replace an input"""
    n = 32
    plan = LPT2(ctx, n, 50.0, prec=F64)
    rng = torch.Generator().manual_seed(1)
    pad = lambda t: torch.nn.functional.pad(t, (0, 2)).contiguous().cuda()  # noqa: E731
    x, C = torch.randn(n, n, n, generator=rng, dtype=torch.float64), torch.randn(3, n, n, n, generator=rng, dtype=torch.float64)
    want = plan.forward(x.cuda())
    noise, a, b = pad(x), torch.zeros(n, n, n + 2, dtype=torch.float64, device="cuda"), None
    b = torch.zeros_like(a)
    plan._call(lambda g: plan.forward_grids(g[0], [g[1], g[1], g[2]]), [noise, a, b])
    assert torch.equal(a[:, :, :n], want[1]) and torch.equal(b[:, :, :n], want[2])
    grad = plan.adjoint(x.cuda(), C.cuda())
    cots = [pad(C[d]) for d in range(3)]
    plan._call(lambda g: plan.adjoint_grids(g[0], g[1:4], g[2]), [noise] + cots)
    assert torch.equal(cots[1][:, :, :n], grad)
    plan.close()
