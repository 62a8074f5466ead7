"""GPU parity of the segmented Scan1D forward on sequences that are not whole
64-step blocks, with checkpoints, with the state updated in place, and under
stream capture, against the CPU oracle (condition-scaled error <= 1e-4 fp32)."""
import ctypes as C

import numpy as np
import pytest

import kmamba as K
import oracle as O
from kmtest import (TOL_F32, assert_close, rel_err_cond, rng_for, scan1d_bwd_kappa, scan1d_inputs,
                    scan1d_kappa)

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"
N = 16


def T(a, dtype=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV, dtype)


# Few channel groups and a last segment of 1, 41, 63, 9 and 64 steps; D not a
# multiple of 32 leaves lanes without a channel.
RAGGED = [(1, 1025, 64), (2, 1001, 40), (3, 1023, 100), (1, 777, 32), (1, 4160, 96)]


@pytest.mark.parametrize("Bsz,L,D", RAGGED)
@pytest.mark.parametrize("layout", ["shared", "per_channel"])
def test_ragged_segments_with_checkpoints(Bsz, L, D, layout):
    x, dt, A, _, _ = scan1d_inputs(Bsz, L, D, N, seed=31)
    g = rng_for("segments", Bsz, L, D)
    h0 = g.standard_normal((Bsz, D, N)).astype(np.float32)
    shape = (Bsz, L, N) if layout == "shared" else (Bsz, L, D, N)
    strides = (L * N, N, 0) if layout == "shared" else (L * D * N, D * N, N)
    Bm, Cm = ((g.standard_normal(shape) * 0.25).astype(np.float32) for _ in range(2))
    yr, hr, hhr = O.scan1d_batched(x, dt, A, Bm, Cm, h0=h0, bc_strides=strides, hist=True)
    ky, kh, khh = scan1d_kappa(x, dt, A, Bm, Cm, h0=h0, bc_strides=strides)
    # The checkpoint after every 32 steps and after the last one.
    at = np.minimum(np.arange(31, L + 31, 32), L - 1)
    ck = torch.full((Bsz, len(at), D, N), float("nan"), device=DEV)
    y = torch.full((Bsz, L, D), float("nan"), device=DEV)
    hf = torch.empty((Bsz, D, N), device=DEV)
    hh = torch.full((Bsz, L, D, N), float("nan"), device=DEV)
    ins = [T(a) for a in (x, dt, A, Bm, Cm)]
    for hist in (None, hh):
        K.scan1d_fwd(*ins, y, h0=T(h0), h_final=hf, h_hist=hist, h_ckpt=ck, bc_strides=strides)
        assert_close(y.cpu().numpy(), yr, TOL_F32, "y", ky)
        assert_close(hf.cpu().numpy(), hr, TOL_F32, "h_final", kh)
        assert_close(ck.cpu().numpy(), hhr[:, at], TOL_F32, "checkpoints", khh[:, at])
    assert_close(hh.cpu().numpy(), hhr, TOL_F32, "history", khh)


@pytest.mark.parametrize("L", [1024, 1001])
@pytest.mark.parametrize("peak", [1.0, 4000.0])
def test_state_updated_in_place(L, peak):
    # h_final is h0's own memory; with peak = 4000 the states of a few steps
    # leave [-1000, 1000], so the whole sequence is re-run from h0.
    Bsz, D = 2, 40
    x, dt, A, Bm, Cm = scan1d_inputs(Bsz, L, D, N, seed=32)
    Bm = Bm.copy()
    Bm[:, 500:505] *= peak
    h0 = rng_for("in-place", L).standard_normal((Bsz, D, N)).astype(np.float32) * 50
    yr, hr, _ = O.scan1d_batched(x, dt, A, Bm, Cm, h0=h0)
    ky, kh, _ = scan1d_kappa(x, dt, A, Bm, Cm, h0=h0)
    h = T(h0)
    y = torch.empty((Bsz, L, D), device=DEV)
    K.scan1d_fwd(*(T(a) for a in (x, dt, A, Bm, Cm)), y, h0=h, h_final=h)
    assert_close(y.cpu().numpy(), yr, TOL_F32, "y", ky)
    assert_close(h.cpu().numpy(), hr, TOL_F32, "h", kh)


def test_captured_call_takes_no_scratch():
    # A capture of a shape that would be split needs no allocation, and its
    # replays follow changed inputs.
    Bsz, L, D = 1, 1001, 64
    x, dt, A, Bm, Cm = (T(a) for a in scan1d_inputs(Bsz, L, D, N, seed=33))
    y, hf = torch.empty_like(x), torch.empty((Bsz, D, N), device=DEV)
    s = torch.cuda.Stream()
    args = K.scan1d_fwd_args(x, dt, A, Bm, Cm, y, h_final=hf)
    held = K.km_device_bytes_held()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        assert K.km_scan1d_fwd_c(C.byref(args), C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    assert K.km_device_bytes_held() == held
    for i in range(3):
        xi = rng_for("graph", i).standard_normal((Bsz, L, D)).astype(np.float32)
        x.copy_(T(xi))
        g.replay()
        torch.cuda.synchronize()
        yr, hr, _ = O.scan1d_batched(xi, *(a.cpu().numpy() for a in (dt, A, Bm, Cm)))
        ky, kh, _ = scan1d_kappa(xi, *(a.cpu().numpy() for a in (dt, A, Bm, Cm)))
        assert rel_err_cond(y.cpu().numpy(), yr, ky) <= TOL_F32
        assert rel_err_cond(hf.cpu().numpy(), hr, kh) <= TOL_F32


# --- the backward split over workgroups ------------------------------------------

def _bwd(x, dt, A, Bm, Cm, dy, *, mode, strides, h0=None, hist=None, workspace=None):
    ins = [T(a) for a in (x, dt, A, Bm, Cm)]
    Bsz, L, D = x.shape
    out = [torch.full_like(ins[0], float("nan")), torch.full_like(ins[0], float("nan")),
           torch.full((D, N), float("nan"), device=DEV), torch.full_like(ins[3], float("nan")),
           torch.full_like(ins[4], float("nan"))]
    th0 = None if h0 is None else T(h0)
    kw = dict(h0=th0, bc_strides=strides)
    if mode == "hist":
        kw["h_hist"] = T(hist)
    elif mode == "ckpt":
        kw["h_ckpt"] = torch.empty((Bsz, -(-L // 32), D, N), device=DEV)
        K.scan1d_fwd(*ins, None, h0=th0, h_ckpt=kw["h_ckpt"], bc_strides=strides)
    args = K.scan1d_bwd_args(*ins, T(dy), *out, **kw)
    need = K.km_scan1d_bwd_workspace_bytes(C.byref(args))
    if workspace == "queried":
        kw["workspace"] = torch.empty(need, dtype=torch.uint8, device=DEV)
    K.scan1d_bwd(*ins, T(dy), *out, **kw)
    torch.cuda.synchronize()
    return [t.cpu().numpy() for t in out], need


def _unsplit_bytes(Bsz, L, D, *, shared, wide, mode):
    """The workspace without a split: dB/dC slots, dA partials, checkpoints."""
    up = lambda v: -(-v // 256) * 256   # noqa: E731
    groups = -(-D // (32 if wide else 16))
    return (up(8 * Bsz * groups * L * N) * shared + up(4 * Bsz * D * N) +
            up(4 * Bsz * -(-L // 32) * D * N) * (mode == "recompute"))


def _check_backward(Bsz, L, D, *, mode, per_channel, wide):
    x, dt, A, Bm, Cm = scan1d_inputs(Bsz, L, D, N, seed=41)
    g = rng_for("segments-bwd", Bsz, L, D)
    if D == 40:
        A = (A * g.uniform(0.02, 1.0, size=A.shape)).astype(np.float32)   # generic, slow decays
    h0 = g.standard_normal((Bsz, D, N)).astype(np.float32)
    dy = g.standard_normal((Bsz, L, D)).astype(np.float32)
    strides = (L * N, N, 0)
    if per_channel:
        strides = (L * D * N, D * N, N)
        Bm, Cm = ((g.standard_normal((Bsz, L, D, N)) * 0.25).astype(np.float32) for _ in range(2))
    kw = dict(h0=h0, bc_strides=strides, nthreads=8, fast=True)
    hh = O.scan1d_batched(x, dt, A, Bm, Cm, hist=True, **kw)[2]
    ref = O.scan1d_batched_backward(x, dt, A, Bm, Cm, dy, hh, **kw)
    kap = scan1d_bwd_kappa(x, dt, A, Bm, Cm, dy, h0=h0, bc_strides=strides)
    got, need = _bwd(x, dt, A, Bm, Cm, dy, mode=mode, strides=strides, h0=h0, hist=hh)
    assert need > _unsplit_bytes(Bsz, L, D, shared=not per_channel, wide=wide, mode=mode)
    for n, a, r, k in zip(("dx", "ddelta", "dA", "dB", "dC"), got, ref, kap):
        assert_close(a, r, TOL_F32, n, k)
    # The caller's own workspace of the queried size: the same bits.
    again, _ = _bwd(x, dt, A, Bm, Cm, dy, mode=mode, strides=strides, h0=h0, hist=hh, workspace="queried")
    for a, b in zip(got, again):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


# Last segments of 1, 41, 31 and 64 steps, two of them with per-channel B/C.
@pytest.mark.parametrize("Bsz,L,D", [(1, 1025, 64), (2, 1001, 40), (1, 799, 200), (1, 1024, 33)])
@pytest.mark.parametrize("mode", ["hist", "ckpt", "recompute"])
def test_backward_segments_vs_oracle(Bsz, L, D, mode):
    _check_backward(Bsz, L, D, mode=mode, per_channel=D in (40, 33), wide=False)


# The same on 16-wave workgroups of 32 channels: forced on small shapes, and
# where the rule takes them (260 groups, 3 segments of 384 steps).
@pytest.mark.parametrize("Bsz,L,D", [(1, 1025, 64), (2, 1001, 40), (1, 799, 200)])
@pytest.mark.parametrize("mode", ["hist", "ckpt"])
def test_backward_segments_of_32_channels(Bsz, L, D, mode, monkeypatch):
    monkeypatch.setenv("KM_SCAN1D_BWD_WIDE", "1")
    _check_backward(Bsz, L, D, mode=mode, per_channel=False, wide=True)


def test_backward_segments_where_32_channels_fill_the_chip():
    _check_backward(5, 1123, 1664, mode="ckpt", per_channel=False, wide=True)


def test_backward_segments_clamped_states():
    # States leave [-1000, 1000] around steps 500-505 of 1001: the segments
    # they pass through recompute them with the per-step clamp.
    Bsz, L, D = 2, 1001, 40
    x, dt, A, Bm, Cm = scan1d_inputs(Bsz, L, D, N, seed=42)
    g = rng_for("segments-clamp")
    A = (A * g.uniform(0.001, 0.01, size=A.shape)).astype(np.float32)
    Bm = Bm.copy()
    Bm[:, 500:506] *= 4000.0
    dy = g.standard_normal((Bsz, L, D)).astype(np.float32)
    strides = (L * N, N, 0)
    kw = dict(bc_strides=strides, nthreads=8, fast=True)
    hh = O.scan1d_batched(x, dt, A, Bm, Cm, hist=True, **kw)[2]
    assert np.abs(hh).max() == 1000.0
    ref = O.scan1d_batched_backward(x, dt, A, Bm, Cm, dy, hh, **kw)
    kap = scan1d_bwd_kappa(x, dt, A, Bm, Cm, dy, bc_strides=strides)
    got, _ = _bwd(x, dt, A, Bm, Cm, dy, mode="ckpt", strides=strides)
    for n, a, r, k in zip(("dx", "ddelta", "dA", "dB", "dC"), got, ref, kap):
        assert_close(a, r, TOL_F32, n, k)


# --- per-channel B / C read in 16-byte loads --------------------------------------

@pytest.mark.parametrize("io,tol", [(torch.float32, TOL_F32), (torch.bfloat16, 2e-2)])
def test_per_channel_rows_of_any_alignment(io, tol):
    # Whole rows; from an odd element on; channels 17 elements apart: the same
    # values, so the same bits, and the oracle's to rounding.
    Bsz, L, D = 2, 1001, 40
    x, dt, A, _, _ = scan1d_inputs(Bsz, L, D, N, seed=34)
    g = rng_for("alignment", L)
    Bm, Cm = ((g.standard_normal((Bsz, L, D, N)) * 0.25).astype(np.float32) for _ in range(2))
    dy = g.standard_normal((Bsz, L, D)).astype(np.float32)
    st = (L * D * N, D * N, N)
    xd, dtd, dyd = (T(a, io) for a in (x, dt, dy))
    runs = []
    for first, gap in ((0, N), (1, N), (0, N + 1)):
        flat = [torch.zeros(first + Bsz * L * D * gap, dtype=io, device=DEV) for _ in range(4)]
        M = [f[first:] for f in flat]
        for m, a in zip(M, (Bm, Cm)):
            m.view(Bsz, L, D, gap)[..., :N] = T(a, io)
        stg = (L * D * gap, D * gap, gap)
        y, hf = torch.empty_like(xd), torch.empty((Bsz, D, N), device=DEV)
        K.scan1d_fwd(xd, dtd, T(A), M[0], M[1], y, h_final=hf, bc_strides=stg)
        dx, ddt, dA = torch.empty_like(xd), torch.empty_like(xd), torch.empty((D, N), device=DEV)
        K.scan1d_bwd(xd, dtd, T(A), M[0], M[1], dyd, dx, ddt, dA, M[2], M[3], bc_strides=stg)
        runs.append([y, hf, dx, ddt, dA] + [m.view(Bsz, L, D, gap)[..., :N].clone() for m in M[2:]])
    for other in runs[1:]:
        for a, b in zip(runs[0], other):
            assert torch.equal(a, b)
    yr, hr, _ = O.scan1d_batched(x, dt, A, Bm, Cm, bc_strides=st)
    ky, kh, _ = scan1d_kappa(x, dt, A, Bm, Cm, bc_strides=st)
    assert_close(runs[0][0].float().cpu().numpy(), yr, tol, "y", ky)
    assert_close(runs[0][1].cpu().numpy(), hr, tol, "h_final", kh)


# --- decays over a whole segment that are out of range -----------------------------

def _growing(Bsz, L, D, kind):
    """Decays of up to e^2 a step: over the parts of a split (64 steps or more)
    they overflow, while the 20 steps that carry data keep every value finite."""
    x, dt, _, Bm, Cm = scan1d_inputs(Bsz, L, D, N, seed=51)
    dt = np.full_like(dt, 0.5)
    if kind == "structured":
        A = np.tile(np.arange(1, N + 1, dtype=np.float32) / 4, (D, 1))
    elif kind == "generic":
        A = np.tile(np.where(np.arange(N) % 2, -3.0, 4.0).astype(np.float32), (D, 1))
    else:                                       # negative steps
        A = -np.tile(np.arange(1, N + 1, dtype=np.float32) / 4, (D, 1))
        dt = -dt
    return x, dt, A, Bm, Cm


@pytest.mark.parametrize("L", [1024, 1001])
@pytest.mark.parametrize("kind", ["structured", "generic", "negative delta"])
def test_growing_decays_keep_padding_zero(L, kind):
    Bsz, D = 2, 40
    x, dt, A, Bm, Cm = _growing(Bsz, L, D, kind)
    x[:, :L - 20] = 0.0                         # padded at the front
    yr, hr, _ = O.scan1d_batched(x, dt, A, Bm, Cm, clamp=False)
    assert np.isfinite(yr).all() and np.isfinite(hr).all()
    ky, kh, _ = (np.abs(a) for a in scan1d_kappa(x, np.abs(dt), A * np.sign(dt[0, 0, 0]), Bm, Cm))
    y = torch.full((Bsz, L, D), float("nan"), device=DEV)
    hf = torch.full((Bsz, D, N), float("nan"), device=DEV)
    K.scan1d_fwd(*(T(a) for a in (x, dt, A, Bm, Cm)), y, h_final=hf, clamp=False)
    assert_close(y.cpu().numpy(), yr, TOL_F32, "y", ky)
    assert_close(hf.cpu().numpy(), hr, TOL_F32, "h_final", kh)


def test_overflowed_state_stays_infinite():
    # Without the clamp an infinite state decays to itself, however far the
    # decay over the following segments underflows.
    Bsz, L, D = 1, 1001, 64
    x, dt, A, Bm, Cm = scan1d_inputs(Bsz, L, D, N, seed=52)
    x[:, 100] = 3e38
    Bm[:, 100] = 40.0
    hr = O.scan1d_batched(x, dt, A, Bm, Cm, clamp=False)[1]
    assert np.isposinf(hr).all()
    hf = torch.zeros((Bsz, D, N), device=DEV)
    K.scan1d_fwd(*(T(a) for a in (x, dt, A, Bm, Cm)), torch.empty((Bsz, L, D), device=DEV), h_final=hf, clamp=False)
    assert np.isposinf(hf.cpu().numpy()).all()


@pytest.mark.parametrize("L", [1024, 1001])
@pytest.mark.parametrize("kind", ["structured", "generic"])
@pytest.mark.parametrize("mode", ["hist", "ckpt"])
def test_growing_decays_backward_of_masked_loss(L, kind, mode):
    # dy reaches only the first 20 steps: the adjoint is exactly zero after.
    Bsz, D = 2, 40
    x, dt, A, Bm, Cm = _growing(Bsz, L, D, kind)
    dy = rng_for("masked", L).standard_normal((Bsz, L, D)).astype(np.float32)
    dy[:, 20:] = 0.0
    if mode == "ckpt":
        x[:, 30:] = 0.0                         # the clamp keeps the states finite
    strides = (L * N, N, 0)
    hh = O.scan1d_batched(x, dt, A, Bm, Cm, hist=True)[2]
    ref = O.scan1d_batched_backward(x, dt, A, Bm, Cm, dy, hh)
    assert all(np.isfinite(r).all() for r in ref)
    ax, aB, aC, ady = (np.abs(a) for a in (x, Bm, Cm, dy))
    kap = O.scan1d_batched_backward(ax, dt, np.abs(A) if kind == "structured" else A, aB, aC, ady, np.abs(hh))
    got, _ = _bwd(x, dt, A, Bm, Cm, dy, mode=mode, strides=strides, hist=hh)
    for n, a, r, k in zip(("dx", "ddelta", "dA", "dB", "dC"), got, ref, kap):
        assert np.isfinite(a).all(), n
        if kind == "structured":
            assert_close(a, r, TOL_F32, n, np.abs(k))
        else:                                   # mixed signs of A: per tensor
            assert np.abs(a - r).max() <= TOL_F32 * np.abs(r).max(), n


# --- scratch in the caller's workspace ------------------------------------------------

def test_backward_with_workspace_takes_no_scratch():
    # Without checkpoints the backward runs the forward first: split or not, a
    # call that was given its workspace allocates nothing.
    Bsz, L, D = 1, 1001, 64
    x, dt, A, Bm, Cm = (T(a) for a in scan1d_inputs(Bsz, L, D, N, seed=61))
    dy = T(rng_for("ws", L).standard_normal((Bsz, L, D)).astype(np.float32))
    outs = [[torch.full_like(t, float("nan")) for t in (x, dt, A, Bm, Cm)] for _ in range(2)]
    args = K.scan1d_bwd_args(x, dt, A, Bm, Cm, dy, *outs[0])
    ws = torch.empty(K.km_scan1d_bwd_workspace_bytes(C.byref(args)), dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    held = K.km_device_bytes_held()
    K.scan1d_bwd(x, dt, A, Bm, Cm, dy, *outs[0], workspace=ws, stream=s)
    s.synchronize()
    assert K.km_device_bytes_held() == held
    K.scan1d_bwd(x, dt, A, Bm, Cm, dy, *outs[1])          # the library's scratch: the same bits
    torch.cuda.synchronize()
    for a, b in zip(*outs):
        assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("whole", [True, False])
def test_mamba1_block_with_workspace_takes_no_scratch(whole):
    # A workspace of the queried size, and one that holds the activations only.
    Bsz, L, dim, R = 1, 1001, 64, 8
    di = 2 * dim
    g = torch.Generator().manual_seed(62)
    rn = lambda *s, std=0.1: (torch.randn(s, generator=g) * std).to(DEV)   # noqa: E731
    bf = torch.bfloat16
    w = {"W_in": rn(2 * di, dim).to(bf), "conv_w": rn(4, di, std=0.5), "conv_b": rn(di),
         "W_x": rn(R + 2 * N, di).to(bf), "W_dt": rn(di, R).to(bf), "dt_bias": rn(di) - 1,
         "A": -torch.arange(1, N + 1, device=DEV, dtype=torch.float32).repeat(di, 1).contiguous(),
         "Dskip": rn(di), "W_out": rn(dim, di).to(bf)}
    x = rn(Bsz, L, dim, std=1.0).to(bf)
    up = lambda v: (v + 255) // 256 * 256   # noqa: E731
    nb = 5 * up(Bsz * L * di * 2) + up(Bsz * L * (R + 2 * N) * 2)
    st = K.mamba1_weights(w)
    if whole:
        nb = K.km_mamba1_block_workspace_bytes(C.byref(st), Bsz, L)
    ws = torch.empty(nb, dtype=torch.uint8, device=DEV)
    out, want = torch.empty_like(x), torch.empty_like(x)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    held = K.km_device_bytes_held()
    K.mamba1_block_fwd(w, x, out, workspace=ws, stream=s)
    s.synchronize()
    assert K.km_device_bytes_held() == held
    K.mamba1_block_fwd(w, x, want)
    torch.cuda.synchronize()
    # Split or not: the scan's fp32 sums in another order, rounded to bf16 once.
    assert (out.float() - want.float()).norm() <= (1e-6 if whole else 4e-3) * want.float().norm()


def test_captured_backward_with_workspace():
    # The split's scratch is the caller's: forward (states again) and backward are
    # split inside a capture too, and each replay equals an eager call.
    Bsz, L, D = 1, 1001, 64
    x, dt, A, Bm, Cm = (T(a) for a in scan1d_inputs(Bsz, L, D, N, seed=63))
    dy = T(rng_for("graph-ws", L).standard_normal((Bsz, L, D)).astype(np.float32))
    outs, want = ([torch.zeros_like(t) for t in (x, x, A, Bm, Cm)] for _ in range(2))
    args = K.scan1d_bwd_args(x, dt, A, Bm, Cm, dy, *outs)
    ws = torch.empty(K.km_scan1d_bwd_workspace_bytes(C.byref(args)), dtype=torch.uint8, device=DEV)
    args = K.scan1d_bwd_args(x, dt, A, Bm, Cm, dy, *outs, workspace=ws)
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    held = K.km_device_bytes_held()
    with torch.cuda.graph(g, stream=s):
        assert K.km_scan1d_bwd_c(C.byref(args), C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    assert K.km_device_bytes_held() == held
    for i in range(3):
        x.copy_(T(rng_for("graph-ws-x", i).standard_normal((Bsz, L, D)).astype(np.float32)))
        g.replay()
        torch.cuda.synchronize()
        K.scan1d_bwd(x, dt, A, Bm, Cm, dy, *want)
        torch.cuda.synchronize()
        for a, b in zip(outs, want):
            assert torch.isfinite(a).all() and torch.equal(a, b)
