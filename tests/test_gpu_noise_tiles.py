"""White noise at the edges of the noise kernel's tiles (64 columns a
workgroup, 6 modes a tile): partial column groups, rows of modes shorter than,
equal to and one longer than a tile, several rows of columns in one group, and
a size with enough draws that some need the long evaluation behind the
rounding test.  FP64 is bit-exact with the oracle, FP32 its rounding, and
every mode is written whatever the grid held."""
import numpy as np
import pytest

from monofonic_amd import F32, F64, Grid, lpt
from oracle import oracle as O


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 4, 6, 10, 12, 22, 24, 26, 96])
def test_noise_tile_edges(ctx, n):
    print(f"noise n={n}", flush=True)
    ref = O.ngenic_fill(2024 + n, n)
    for prec, dtype in ((F64, np.float64), (F32, np.float32)):
        g = Grid(ctx, (n,) * 3, (50.0,) * 3, prec=prec)
        g.upload(np.full(g.shape_real, 7.5, dtype=dtype))
        lpt.ngenic_fill(g, 2024 + n)
        # bits up to the sign of zero
        assert np.array_equal(g.download(dtype), ref.astype(dtype))
        g.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,prec", [(8, F64), (8, F32), (12, F64), (18, F32), (36, F64)])
def test_folded_phi1_equals_two_steps(ctx, n, prec):
    """a run's phi1 (formed in the noise stores) is phi1_from_noise of the noise"""
    cfg = lpt.ICConfig(n=n, box=80.0, zstart=30.0, lpt_order=1, prec=prec, seed=99)
    run = lpt.ICRun(ctx, cfg)
    run.execute()
    got = run.potential(0).download(np.float64)
    wn, phi = (Grid(ctx, (n,) * 3, (80.0,) * 3, prec=prec) for _ in range(2))
    lpt.ngenic_fill(wn, 99)
    lpt.phi1_from_noise(phi, wn, lpt.baseline_cosmology(30.0))
    assert np.array_equal(got, phi.download(np.float64))
    for o in (wn, phi, run):
        o.close()
