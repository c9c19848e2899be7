"""A device allocation that fails is reported by the call that made it, and by
no later one: the next launch on the thread does not find its error."""
import pytest
import torch  # noqa: F401  before the library, whose HIP runtime is then torch's

from monofonic_amd import F64, Grid, _lib as L, lpt

ERR_ALLOC = -4
HUGE = 8192  # 4.4 TB as an FP64 grid


@pytest.mark.gpu
def test_a_failed_allocation_is_reported_once(ctx):
    g = Grid(ctx, (32,) * 3, (10.0,) * 3, prec=F64)
    lpt.ngenic_fill(g, 1)
    want = g.download_k().copy()
    with pytest.raises(L.MficError) as e:
        Grid(ctx, (HUGE,) * 3, (10.0,) * 3, prec=F64)
    print(e.value)
    assert L.load().mfic_last_error() and "alloc" in str(e.value).lower()
    lpt.ngenic_fill(g, 1)
    assert (g.download_k() == want).all()
    g.close()
