"""3D grids on both sides of the tile rule of the dataflow schedule (tiles of
2 x 2 x 8 points on small grids, pencils of 4 x 4 x 8 on large ones), at the
edges of the tiles: against the CPU oracle (condition-scaled error <= 1e-4
fp32), and bit for bit against the band schedule (4 x 4 x 8 tiles)."""
import numpy as np
import pytest

import oracle as O
from kmtest import TOL_F32, assert_close
from test_scannd_gpu import _stable_nd_inputs, kappa, run_device

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

SMALL = [((2, 2, 8), 4, 16), ((3, 5, 9), 8, 8), ((1, 4, 17), 16, 4), ((5, 1, 8), 4, 16), ((4, 7, 1), 32, 2),
         ((9, 3, 25), 20, 16), ((7, 8, 16), 2, 32), ((7, 5, 10), 1024, 16)]
# Fronts of more than 768 waves: pencils (one channel group per 4 channels).
LARGE = [((9, 6, 11), 832, 16), ((7, 6, 10), 1024, 16), ((5, 12, 9), 448, 32)]
# 2050 bands of 4 x 4 x 8 tiles (pencils: 1), whose 4101 of 2 x 2 x 8 would not
# fit the host's tables; 801 and 778 bands of 2 x 2 x 8 tiles, more than the
# dataflow schedule's table holds.
LONG = [((8200, 4, 8), 4, 16), ((1600, 4, 8), 4, 16), ((6, 1550, 9), 4, 16)]


@pytest.mark.parametrize("dims,D,M", SMALL + LARGE + LONG)
def test_tile_rule_edges(dims, D, M, monkeypatch):
    x, A, B, Cm, dt = _stable_nd_inputs(dims, D, M, "tiles3")
    y, h = run_device(dims, x, A, B, Cm, dt)
    yr, hr = O.scannd_ref(dims, x, A, B, Cm, dt, nthreads=8, fast=True)
    ya, ha = kappa(dims, x, A, B, Cm, dt)
    assert_close(y, yr, TOL_F32, "y", ya)
    assert_close(h, hr, TOL_F32, "h", ha)
    for name, value in (("KM_SCANND_PENCIL", "0"), ("KM_SCANND_SCHED", "band")):
        monkeypatch.setenv(name, value)
        y2, h2 = run_device(dims, x, A, B, Cm, dt)
        assert np.array_equal(h.view(np.uint32), h2.view(np.uint32)), name
        assert np.array_equal(y.view(np.uint32), y2.view(np.uint32)), name
