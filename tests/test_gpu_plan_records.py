"""A record of chosen plans names every plan that is not the built-in one, so
that setting them on another context repeats the choice."""
import pytest
import torch  # noqa: F401  before the library, whose HIP runtime is then torch's

from monofonic_amd import F32, F64, Context, _lib as L, batch


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [F32, F64])
@pytest.mark.parametrize("variant", [0, 1])
def test_a_record_repeats_the_choice(prec, variant):
    n = 512
    a, b = Context(0), Context(0)
    try:
        assert batch.chosen_plans(a, n, prec) == {}
        keys = [(length, p) for length in (n, 3 * n // 2) for p in L.PASSES if p != L.PASS_FUSED_ROWS] \
            + [(3 * n // 2, L.PASS_FUSED_ROWS)]
        for length, p in keys:
            batch.set_plan(a, length, p, prec, variant)
        for (length, p), v in batch.chosen_plans(a, n, prec).items():
            batch.set_plan(b, length, p, prec, v)
        for length, p in keys:
            assert batch.get_plan(b, length, p, prec) == variant, (length, p)
    finally:
        a.close()
        b.close()
