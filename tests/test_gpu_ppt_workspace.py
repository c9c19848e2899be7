"""The work arrays of the semiclassical PT fields belong to their run."""
import ctypes as C

import numpy as np
import pytest
import torch  # noqa: F401  before the library, whose HIP runtime is then torch's

from monofonic_amd import F64, Context, Grid, _lib as L, batch, lpt


@pytest.mark.gpu
def test_work_arrays_go_with_the_run():
    """a run's work arrays are made once and given back when it is closed; the
    context keeps nothing of their size"""
    hip = lpt._hip()
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    n, box = 96, 100.0
    ctx = Context(0)
    try:
        outs = [Grid(ctx, (n,) * 3, (box,) * 3, prec=F64) for _ in range(4)]

        def cycle():
            run = lpt.ICRun(ctx, lpt.ICConfig(n=n, box=box, zstart=24.0, lpt_order=2, prec=F64, seed=3))
            run.execute()
            marks = [free()]
            for _ in range(2):
                L.call("mfic_ppt_fields", run.h, 1.0, *[g.h for g in outs], None)
                marks.append(free())
            run.close()
            return marks + [free()]

        cycle()  # tables
        start = free()
        made, first, second, closed = cycle()
        assert made - first >= 4 * n ** 3 * 8 and first == second
        assert start - closed <= 2 << 20
        for g in outs:
            g.close()
    finally:
        ctx.close()


@pytest.mark.gpu
def test_fields_are_refused_under_capture(ctx):
    n = 16
    run = lpt.ICRun(ctx, lpt.ICConfig(n=n, box=50.0, zstart=24.0, lpt_order=2, prec=F64, seed=3))
    run.execute()
    outs, _ = lpt.ppt_fields(run)
    want = [g.download_r().copy() for g in outs]

    def both():
        assert L.load().mfic_ppt_fields(run.h, 1.0, *[g.h for g in outs], None) == -5
        run.execute(blocking=False)

    graph = batch.capture(ctx, both)  # the refusal leaves the capture whole
    graph.launch()
    again, _ = lpt.ppt_fields(run)
    for a, b in zip(again, want):
        assert np.array_equal(a.download_r(), b)
    for o in (graph, *outs, *again, run):
        o.close()


@pytest.mark.gpu
@pytest.mark.parametrize("same", [(0, 1), (0, 2), (1, 2), (0, 1, 2)])
def test_one_grid_for_several_velocities(ctx, same):
    """holds the last of its components, as passes in the order x, y, z leave it"""
    n = 24
    run = lpt.ICRun(ctx, lpt.ICConfig(n=n, box=50.0, zstart=24.0, lpt_order=2, prec=F64, seed=3))
    run.execute()
    want, _ = lpt.ppt_fields(run)
    ref = [g.download_r().copy() for g in want]
    outs = [Grid(ctx, (n,) * 3, (50.0,) * 3, prec=F64) for _ in range(4)]
    vel = [outs[1 + (same[0] if d in same else d)] for d in range(3)]
    L.call("mfic_ppt_fields", run.h, 1.0, outs[0].h, *[g.h for g in vel], None)
    assert np.array_equal(outs[0].download_r(), ref[0])
    for d in range(3):
        last = same[-1] if d in same else d
        assert np.array_equal(vel[d].download_r(), ref[1 + last]), d
    for o in (*want, *outs, run):
        o.close()
