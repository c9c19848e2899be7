"""A record of chosen plans names every plan that is not the built-in one, so
that setting them on another context repeats the choice (also where plan 0 was
chosen for a pass with another default)."""
import ctypes as C

import pytest
import torch  # noqa: F401  before the library, whose HIP runtime is then torch's

from monofonic_amd import F32, F64, Context, _lib as L, batch


def test_default_plans():
    for length in (48, 512, 576, 768):
        for p in L.PASSES:
            for prec in (F32, F64):
                want = int(length == 768 and prec == F32 and p in (L.PASS_TRUNC_AX0, L.PASS_TRUNC_AX1))
                assert batch.default_plan(length, p, prec) == want
    v = C.c_int()
    lib = L.load()
    assert lib.mfic_fft_default_plan(7, L.PASS_PAD_C2R_A, F32, C.byref(v)) == -2
    assert lib.mfic_fft_default_plan(768, 1, F32, C.byref(v)) == -1
    assert lib.mfic_fft_default_plan(768, L.PASS_TRUNC_AX0, 7, C.byref(v)) == -1
    assert lib.mfic_fft_default_plan(768, L.PASS_TRUNC_AX0, F32, None) == -1


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
