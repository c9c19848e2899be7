"""Semiclassical PT fields at the edges of their passes' tiles: lengths whose
transform fits one thread (8, 12), ragged radices (18, 36, 72, whose rows and
pencils leave partial workgroups) and a three-stage plan (96), against the
oracle.  FP64 rel-L2 1e-9 (phases of 10^2 radians and FFT rounding stay below
1e-12); FP32 1e-4 (phases of tens of radians in 24 bits)."""
import ctypes as C

import pytest

from monofonic_amd import F32, F64, Grid, _lib as L, lpt
from oracle import oracle as O

from _gpu_helpers import rel_l2


@pytest.mark.gpu
@pytest.mark.parametrize("n,order,prec", [(8, 2, F64), (12, 2, F32), (18, 1, F64), (36, 1, F32), (72, 1, F64),
                                          (96, 2, F64)])
def test_ppt_sizes(ctx, n, order, prec):
    box, z, seed, vu = 3.0 * n, 30.0, 777 + n, 1.5
    print(f"PPT n={n} order={order} prec={prec}", flush=True)
    cfg = O.ic_cfg(n, box, order, seed)
    oc = O.baseline_cosmology(z)
    phi, phi2, _, _ = O.potentials(cfg, oc, O.ngenic_fill(seed, n))
    want, hb_want = O.ppt_fields(cfg, O.lpt_coefs(cfg, oc), phi, phi2, vu)
    run = lpt.ICRun(ctx, lpt.ICConfig(n=n, box=box, zstart=z, lpt_order=order, prec=prec, seed=seed))
    run.execute()
    outs = [Grid(ctx, (n,) * 3, (box,) * 3, prec=prec) for _ in range(4)]
    hb = C.c_double()
    for _ in range(2):  # the second call finds its workspace used
        L.call("mfic_ppt_fields", run.h, vu, *[g.h for g in outs], C.byref(hb))
        assert abs(hb.value / hb_want - 1) < (1e-9 if prec == F64 else 1e-5)
        for name, g, w in zip(("delta", "vx", "vy", "vz"), outs, want):
            err = rel_l2(g.download_r(), O.rview(w))
            assert err < (1e-9 if prec == F64 else 1e-4), (name, err)
    for g in outs:
        g.close()
    run.close()
