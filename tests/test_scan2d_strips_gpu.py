"""2D grids at the edges of the row strips (7 rows, blocks of 4 columns, 4
blocks of operands in flight, rings of 8 blocks): against the CPU oracle
(condition-scaled error <= 1e-4 fp32), and the states bit for bit against the
band schedule, which adds the same terms in the same order."""
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

import oracle as O
from kmtest import TOL_F32, assert_close
from test_scannd_gpu import FUSED_CASES, _BUDGET0, _stable_nd_inputs, bwd_inputs, kappa, run_bwd, run_device

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# Rows: one short strip, a full one, one more row, two strips, many; columns:
# less than a block, ragged blocks, fewer and more blocks than in flight and
# than a ring holds. M covers every lane sum; one channel group leaves seven
# XCDs without work.
STRIPS = [((2, 2), 4, 16), ((7, 3), 64, 1), ((8, 4), 96, 2), ((14, 5), 48, 4), ((15, 16), 8, 8),
          ((22, 33), 20, 16), ((3, 37), 10, 32), ((40, 2), 3, 64), ((29, 70), 36, 16), ((1, 41), 8, 8),
          ((30, 1), 8, 8)]


@pytest.mark.parametrize("dims,D,M", STRIPS)
def test_strip_edges(dims, D, M, monkeypatch):
    x, A, B, Cm, dt = _stable_nd_inputs(dims, D, M, "strips")
    y, h = run_device(dims, x, A, B, Cm, dt)
    yr, hr = O.scannd_ref(dims, x, A, B, Cm, dt, nthreads=8, fast=True)
    ya, ha = kappa(dims, x, A, B, Cm, dt)
    assert_close(y, yr, TOL_F32, "y", ya)
    assert_close(h, hr, TOL_F32, "h", ha)
    monkeypatch.setenv("KM_SCANND_SCHED", "band")
    _, hb = run_device(dims, x, A, B, Cm, dt)
    assert np.array_equal(h.view(np.uint32), hb.view(np.uint32))


# (24 states: the adjoint sums no lanes and takes any M.)
@pytest.mark.parametrize("dims,D,M", STRIPS + [((16, 19), 8, 24)])
def test_strip_edges_backward(dims, D, M, monkeypatch):
    ins = bwd_inputs(dims, D, M, 8)
    a = run_bwd(dims, *ins)
    want = O.scannd_backward(dims, *ins, fast=True)
    for k in want:
        assert np.isfinite(a[k]).all(), k
        err = np.abs(a[k] - want[k]).max() / max(np.abs(want[k]).max(), 1e-30)
        assert err <= 1e-4, f"{k}: normwise error {err:.2e}"
    monkeypatch.setenv("KM_SCANND_SCHED", "band")
    b = run_bwd(dims, *ins)
    for k in a:
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), k


# Small 2D grids run the two passes by default; forced, the fused backward
# gives the same values (dA sums its terms in another order). The last grid
# is over the line, so its default is the fused one.
@pytest.mark.parametrize("dims,D,M", [c for c in FUSED_CASES if len(c[0]) == 2] + [((9, 10), 4096, 16)])
def test_fused_forced_matches_default(dims, D, M, monkeypatch):
    ins = bwd_inputs(dims, D, M, 9)
    a = run_bwd(dims, *ins)
    for forced in ("1", "0"):
        monkeypatch.setenv("KM_SCANND_BWD_FUSED", forced)
        b = run_bwd(dims, *ins)
        for k in ("dx", "ddelta", "dB", "dC"):
            assert np.isfinite(a[k]).all() and np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), k
        np.testing.assert_allclose(a["dA"], b["dA"], rtol=1e-5, atol=1e-6 * float(np.abs(b["dA"]).max()))


def test_wait_budget_exhausted_fails_loudly_and_sync_api_recovers(tmp_path):
    # No polls at all (the budget is read once per process): the couriers hand
    # NaN to every strip but the first, the status says so, and the
    # synchronous entry point runs the call again by bands.
    root = Path(__file__).resolve().parent.parent
    dims, D, M = (20, 9), 4, 16
    x, A, B, Cm, dt = _stable_nd_inputs(dims, D, M, "strips-budget0")
    src, dst = tmp_path / "in.npz", tmp_path / "out.npz"
    np.savez(src, dims=np.array(dims), x=x, A=A, B=B, C=Cm, dt=dt)
    r = subprocess.run([sys.executable, "-c", _BUDGET0, str(src), str(root / "k-mamba_amd"),
                        str(root / "oracle"), str(dst)], env=dict(os.environ, KM_SCANND_FLOW_SPIN="0"),
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    out = np.load(dst)
    yr, hr = O.scannd_ref(dims, x, A, B, Cm, dt, nthreads=8, fast=True)
    ya, ha = kappa(dims, x, A, B, Cm, dt)
    assert int(out["status_async"]) == 1 and int(out["status_noalloc"]) == 1
    assert int(out["rc"]) == 0 and int(out["status_sync"]) == 0
    assert_close(out["y_sync"], yr, TOL_F32, "y after re-run", ya)
    assert_close(out["h_sync"], hr, TOL_F32, "h after re-run", ha)
    yg = out["y_async"].reshape(dims + (D,))
    assert np.isnan(yg[7:]).all()
    assert_close(yg[:7].reshape(-1, D), yr[:63], TOL_F32, "first strip", ya[:63])
