"""Work spaces that a captured graph uses stay where they are while a later,
larger box outgrows them: replays give the bits of the eager run, and the
outgrown buffers are given back with the last graph.  The 2LPT adjoint works in
a space of its plan."""
import ctypes as C

import numpy as np
import pytest

from monofonic_amd import F32, F64, Context, Grid, lpt
from monofonic_amd.batch import capture
from monofonic_amd.lpt import ICConfig, ICRun

torch = pytest.importorskip("torch")
from monofonic_amd.adjoint import LPT2  # noqa: E402


def free_bytes():
    hip = lpt._hip()
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
    f, t = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


def fields(run):
    return [run.field(c).download_r().copy() for c in range(6)]


@pytest.mark.gpu
@pytest.mark.parametrize("prec,order,n,large", [(F32, 3, 64, (96, 128)), (F64, 2, 64, (128,)), (F64, 3, 32, (48, 64, 96))])
def test_replay_after_a_larger_box(prec, order, n, large):
    ctx = Context(0)  # of its own: nothing has grown yet
    try:
        small = ICRun(ctx, ICConfig(n=n, box=80.0, zstart=24.0, lpt_order=order, prec=prec, seed=11))
        small.execute()
        want = fields(small)
        graphs = [capture(ctx, lambda: small.execute(blocking=False)) for _ in range(2)]
        for m in large:
            r = ICRun(ctx, ICConfig(n=m, box=80.0, zstart=24.0, lpt_order=order, prec=prec, seed=12))
            r.execute()
            # whatever was given back holds other values now
            junk = [torch.full((1 << 20,), float("nan"), device="cuda") for _ in range(64)]
            torch.cuda.synchronize()
            for g in graphs:
                for c in range(6):
                    small.field(c).zero()
                g.launch()
                for c, (a, b) in enumerate(zip(fields(small), want)):
                    assert np.array_equal(a, b), (m, c)
            del junk
            r.close()
        graphs[0].close()
        graphs[1].launch()
        assert all(np.array_equal(a, b) for a, b in zip(fields(small), want))
        ctx.sync()
        before = free_bytes()
        graphs[1].close()
        # at least the inputs of the row passes: 7 (16) compact padded buffers
        np_, kc, es = 3 * n // 2, n // 2 + 1, 8 if prec == F64 else 4
        held = (16 if order == 3 else 7) * np_ * np_ * kc * 2 * es
        print(f"given back with the last graph: {free_bytes() - before} bytes (row pass inputs {held})")
        assert free_bytes() - before >= held
        small.execute()
        assert all(np.array_equal(a, b) for a, b in zip(fields(small), want))
        small.close()
    finally:
        ctx.close()


@pytest.mark.gpu
def test_growth_without_a_graph_keeps_nothing():
    """outgrown buffers are freed at once where no graph is alive, also after
    one was"""
    ctx = Context(0)
    try:
        def run(n):
            r = ICRun(ctx, ICConfig(n=n, box=80.0, zstart=24.0, lpt_order=3, prec=F64, seed=5))
            r.execute()
            r.close()
            return free_bytes()

        run(48)
        r = ICRun(ctx, ICConfig(n=48, box=80.0, zstart=24.0, lpt_order=3, prec=F64, seed=5))
        r.execute()
        capture(ctx, lambda: r.execute(blocking=False)).close()
        r.close()
        at96 = run(96)
        for _ in range(2):
            assert abs(run(96) - at96) <= 2 << 20
        at128 = run(128)
        # 128^3 takes (16 + 3 + 4) buffers of its own and none of 96^3's beside them
        kb = lambda n: (3 * n // 2) ** 2 * (n // 2 + 1) * 16  # noqa: E731
        grown = 23 * (kb(128) - kb(96))
        print(f"96^3 -> 128^3: {at96 - at128} bytes more, {grown} expected")
        assert at96 - at128 <= grown + (16 << 20)  # tables and allocation granules
    finally:
        ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("prec,n,larger", [(F32, 32, 96), (F64, 48, 64)])
def test_adjoint_replay_after_a_larger_plan(prec, n, larger):
    ctx = Context(0)
    try:
        rng = np.random.default_rng(n)
        dtype = np.float64 if prec == F64 else np.float32
        plan = LPT2(ctx, n, 100.0, prec=prec)
        grids = [Grid(ctx, (n,) * 3, (100.0,) * 3, prec=prec) for _ in range(5)]
        for g in grids[:4]:
            g.upload(rng.standard_normal(g.shape_real).astype(dtype))
        adjoint = lambda: plan.adjoint_grids(grids[0], grids[1:4], grids[4])  # noqa: E731
        adjoint()
        want = grids[4].download_r().copy()
        graph = capture(ctx, adjoint)
        big = LPT2(ctx, larger, 100.0, prec=prec)
        x = torch.randn(larger, larger, larger, dtype=torch.float64, device="cuda")
        big.adjoint(x, torch.stack([x, -x, 2 * x]))
        for rep in range(3):
            grids[4].zero()
            graph.launch()
            assert np.array_equal(grids[4].download_r(), want), rep
            if rep == 0:
                big.close()
        graph.close()
        for o in (plan, *grids):
            o.close()
    finally:
        ctx.close()


@pytest.mark.gpu
def test_a_plan_owns_its_workspace():
    """taken when the plan is made, not at the first adjoint, and given back
    with the plan"""
    ctx = Context(0)
    try:
        n, prec = 128, F32
        x = torch.randn(n, n, n, device="cuda")
        cot = torch.stack([x, x, x])
        first = LPT2(ctx, n, 100.0, prec=prec)  # allocates what the context keeps
        first.forward(x), first.adjoint(x, cot)
        first.close()
        before = free_bytes()
        plan = LPT2(ctx, n, 100.0, prec=prec)
        made = free_bytes()
        workspace = 13 * (3 * n // 2) ** 2 * (n // 2 + 1) * 8
        assert before - made >= workspace
        plan.adjoint(x, cot)
        assert made - free_bytes() <= 2 << 20
        plan.close()
        assert before - free_bytes() <= 2 << 20
    finally:
        ctx.close()
