"""The work that users of libkmamba have it do, as measurable cases.

Each case runs one pass through the library's public entry points on inputs
that live where a user's program would have them. The argument structures are
filled in once, as a C caller keeps them; every output is returned whole.

    listed()            the named cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program has in hand before the call
    run(state)          one pass, and its outputs
    work(case)          bytes and operations a pass cannot do without
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   the same outputs in 64 bits, in plain torch

State size N (M for the grids) is 16 throughout, as in every configuration of
the benchmark.
"""
from __future__ import annotations

import ctypes as C
import math
import os
import sys

import numpy as np
import torch

# The working folder is the repository's root; the package is not installed.
_PKG = os.path.join(os.getcwd(), "k-mamba_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import kmamba as K  # noqa: E402

N = 16
DEV = "cuda"
BF = torch.bfloat16
F64 = torch.float64


def listed():
    return [
        # One short sequence at a small model's width: the time is launch and latency.
        {"name": "scan1d_fwd_short", "kind": "scan1d", "B": 1, "L": 128, "D": 384, "dtype": "f32",
         "gated": False},
        # A training batch's forward in fp32, without gradients (evaluation).
        {"name": "scan1d_fwd_batch", "kind": "scan1d", "B": 8, "L": 4096, "D": 1024, "dtype": "f32",
         "gated": False},
        # Prefill of one long prompt of any length: bf16 activations, SiLU(z) gate and skip.
        {"name": "scan1d_prompt_bf16", "kind": "scan1d", "B": 1, "L": 5003, "D": 1536, "dtype": "bf16",
         "gated": True},
        # A training step of the scan layer: forward with checkpoints, then every gradient.
        {"name": "scan1d_step_f32", "kind": "scan1d_step", "B": 8, "L": 4096, "D": 1024, "dtype": "f32"},
        # The same in bf16 on a small batch of sequences of an odd length.
        {"name": "scan1d_step_bf16_odd", "kind": "scan1d_step", "B": 2, "L": 1999, "D": 768,
         "dtype": "bf16"},
        # An image's wavefront scan, inference.
        {"name": "scan2d_fwd", "kind": "grid", "dims": "256x256", "D": 256},
        # A training step on a small image of odd sizes.
        {"name": "scan2d_step_odd", "kind": "grid_step", "dims": "45x61", "D": 96},
        # A training step on a volume.
        {"name": "scan3d_step", "kind": "grid_step", "dims": "64x64x64", "D": 128},
        # A training step of the per-channel causal convolution on an image.
        {"name": "conv2d_step", "kind": "conv_step", "dims": "512x512", "D": 64, "K": 3},
        # The Mamba-1 block forward at a small language model's width.
        {"name": "mamba1_block", "kind": "mamba1", "B": 8, "L": 2048, "dim": 1024},
        # The Mamba-3 block forward, activations on the GPU.
        {"name": "mamba3_block", "kind": "mamba3", "B": 8, "L": 2048, "dim": 1024, "R": 1},
        # A whole call: host tokens in, host logits out.
        {"name": "model_forward", "kind": "model", "V": 32768, "dim": 1024, "L": 2048, "layers": 4},
    ]


def _log_int(rng, lo, hi, step=1):
    """An integer of [lo, hi], uniform in its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, step * round(v / step))))


def draw(rng):
    kind = rng.choice(["scan1d", "scan1d", "scan1d_step", "scan1d_step", "grid", "grid_step", "grid_step",
                       "conv_step", "mamba1", "mamba1", "mamba3", "model"])
    if kind in ("scan1d", "scan1d_step"):
        L = _log_int(rng, 64, 8192)
        D = _log_int(rng, 64, 2048, rng.choice([64, 32, 8, 1]))
        B = _log_int(rng, 1, max(1, min(16, 8 * 4096 * 1024 // (L * D))))
        c = {"kind": kind, "B": B, "L": L, "D": D, "dtype": rng.choice(["f32", "bf16"])}
        if kind == "scan1d":
            c["gated"] = rng.random() < 0.5
        return c
    if kind in ("grid", "grid_step"):
        if rng.random() < 0.6:
            dims, D = [_log_int(rng, 12, 256) for _ in range(2)], _log_int(rng, 16, 256, 16)
        else:
            dims, D = [_log_int(rng, 6, 64) for _ in range(3)], _log_int(rng, 16, 128, 16)
        return {"kind": kind, "dims": "x".join(map(str, dims)), "D": D}
    if kind == "conv_step":
        if rng.random() < 0.5:
            dims, k = [_log_int(rng, 24, 512) for _ in range(2)], rng.choice([2, 3, 4])
        else:
            dims, k = [_log_int(rng, 10, 64) for _ in range(3)], rng.choice([2, 3])
        return {"kind": kind, "dims": "x".join(map(str, dims)), "D": _log_int(rng, 16, 128, 8), "K": k}
    if kind == "mamba1":
        return {"kind": kind, "B": _log_int(rng, 1, 8), "L": _log_int(rng, 64, 2048),
                "dim": _log_int(rng, 256, 1024, 128)}
    if kind == "mamba3":
        return {"kind": kind, "B": _log_int(rng, 1, 8), "L": _log_int(rng, 64, 2048),
                "dim": _log_int(rng, 128, 1024, 4), "R": rng.choice([1, 1, 2, 4])}
    return {"kind": kind, "V": _log_int(rng, 1000, 32768), "dim": _log_int(rng, 128, 1024, 4),
            "L": _log_int(rng, 64, 2048), "layers": rng.randint(1, 4)}


def _dims(case):
    return tuple(int(v) for v in case["dims"].split("x"))


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _check(rc):
    if rc != 0:
        raise RuntimeError(K.km_last_error())


# --- inputs, from the seed alone ------------------------------------------------

def _scan1d_inputs(case, seed):
    """x ~ N(0,1); delta = softplus(0.5 N(0,1) - 1); A = -(1..N); B, C ~ N(0, 1/N)
    shared over channels; gate z and incoming gradient ~ N(0,1)."""
    B, L, D = case["B"], case["L"], case["D"]
    io = BF if case["dtype"] == "bf16" else torch.float32
    g = _gen(seed)
    rn = lambda *s: torch.randn(s, device=DEV, generator=g)  # noqa: E731
    x = rn(B, L, D).to(io)
    dt = torch.nn.functional.softplus(0.5 * rn(B, L, D) - 1.0).to(io)
    A = -torch.arange(1, N + 1, device=DEV, dtype=torch.float32).repeat(D, 1).contiguous()
    Bm, Cm = (rn(B, L, N) / N ** 0.5).to(io), (rn(B, L, N) / N ** 0.5).to(io)
    extra = rn(B, L, D).to(io)                       # z, or dy of a training step
    skip = 1.0 + 0.1 * rn(D)
    return x, dt, A, Bm, Cm, extra, skip


def _grid_inputs(case, seed):
    """x, dy ~ N(0,1); delta in [0.8, 1.2]; A = log U(0.05, 0.9/nd), so the decays of a
    point sum to less than one; B, C ~ N(0, 1/N) per point."""
    dims, D = _dims(case), case["D"]
    nd, P = len(dims), int(np.prod(dims))
    g = _gen(seed)
    x = torch.randn((P, D), device=DEV, generator=g)
    A = torch.log(0.05 + (0.9 / nd - 0.05) * torch.rand((nd, D, N), device=DEV, generator=g))
    B = torch.randn((P, D, N), device=DEV, generator=g).mul_(0.25)
    Cm = torch.randn((P, D, N), device=DEV, generator=g).mul_(0.25)
    dt = torch.rand((nd, P, D), device=DEV, generator=g).mul_(0.4).add_(0.8)
    dy = torch.randn((P, D), device=DEV, generator=g)
    return x, A, B, Cm, dt, dy


def _conv_inputs(case, seed):
    dims, D, k = _dims(case), case["D"], case["K"]
    P, KV = int(np.prod(dims)), k ** len(dims)
    g = _gen(seed)
    inp = torch.randn((P, D), device=DEV, generator=g)
    ker = torch.randn((KV, D), device=DEV, generator=g) / KV ** 0.5
    bias = torch.randn((D,), device=DEV, generator=g) * 0.1
    dy = torch.randn((P, D), device=DEV, generator=g)
    return inp, ker, bias, dy


def _mamba1_inputs(case, seed):
    """Weights ~ N(0, 0.02), A = -(1..N), x ~ N(0,1); d_inner = 2 dim, dt_rank = dim / 16
    rounded up to 8, convolution over 4 steps."""
    dim = case["dim"]
    di, R = 2 * dim, (dim // 16 + 7) // 8 * 8
    g = _gen(seed)
    rn = lambda *s, std=0.02: torch.randn(s, device=DEV, generator=g) * std  # noqa: E731
    w = {"W_in": rn(2 * di, dim).to(BF), "conv_w": rn(4, di, std=0.5), "conv_b": rn(di, std=0.1),
         "W_x": rn(R + 2 * N, di).to(BF), "W_dt": rn(di, R).to(BF), "dt_bias": rn(di, std=0.5) - 2.0,
         "A": -torch.arange(1, N + 1, device=DEV, dtype=torch.float32).repeat(di, 1).contiguous(),
         "Dskip": 1.0 + rn(di, std=0.1), "W_out": rn(dim, di).to(BF)}
    x = torch.randn((case["B"], case["L"], dim), device=DEV, generator=g).to(BF)
    return w, x


def _block_params(rng, dim, R):
    """A Mamba-3 block's host parameters, distributed as mamba_block_init draws them,
    with delta_proj and lambda_proj wide enough that the step sizes vary."""
    f = np.float32
    uni = lambda r, c: ((rng.random((r, c), dtype=f) * 2 - 1) * f(math.sqrt(6.0 / (r + c))))  # noqa: E731
    return {"W_in": uni(R, dim), "W_out": uni(dim, R), "A_log": -(0.5 + rng.random((N, 1), dtype=f)),
            "W_B": uni(N * R, dim), "W_C": uni(N * R, dim),
            "delta_proj": (rng.standard_normal((1, dim), dtype=f) * f(2.0 / math.sqrt(dim))),
            "lambda_proj": (rng.random((1, dim), dtype=f) - f(0.5)) * f(0.1),
            "b_B": rng.standard_normal(N * R, dtype=f) * f(0.02),
            "b_C": rng.standard_normal(N * R, dtype=f) * f(0.02),
            "theta": rng.random(N // 2, dtype=f) * f(2 * math.pi / N)}


def _fill_block(blk, params):
    b = blk.contents
    for name, v in params.items():
        dst = getattr(b, name)
        ptr = dst.data if isinstance(dst, K.MBMatrix) else dst
        np.ctypeslib.as_array(ptr, shape=(v.size,))[:] = v.ravel()


_DT = {"dt_scale": 0.1, "dt_min": 1e-3, "dt_max": 1.0}


class _Block:
    """A block that a program keeps, freed with its last reference."""

    def __init__(self, dim, L, R, params):
        cfg = K.MBConfig()
        cfg.dim, cfg.state_size, cfg.seq_len, cfg.mimo_rank = dim, N, L, R
        cfg.dt_scale, cfg.dt_min, cfg.dt_max = _DT["dt_scale"], _DT["dt_min"], _DT["dt_max"]
        self.p = K.mamba_block_create(C.byref(cfg))
        if not self.p:
            raise RuntimeError(K.km_last_error())
        _fill_block(self.p, params)

    def __del__(self):
        K.mamba_block_free(self.p)


class _Model:
    def __init__(self, case, emb, head, layers):
        cfg = K.KMambaConfig()
        cfg.vocab_size, cfg.dim, cfg.state_size = case["V"], case["dim"], N
        cfg.seq_len, cfg.n_layers, cfg.mimo_rank = case["L"], case["layers"], 1
        cfg.dt_scale, cfg.dt_min, cfg.dt_max = _DT["dt_scale"], _DT["dt_min"], _DT["dt_max"]
        self.p = K.kmamba_create(C.byref(cfg))
        if not self.p:
            raise RuntimeError(K.km_last_error())
        m = self.p.contents
        np.ctypeslib.as_array(m.embedding, shape=(emb.size,))[:] = emb.ravel()
        np.ctypeslib.as_array(m.head, shape=(head.size,))[:] = head.ravel()
        for i, params in enumerate(layers):
            _fill_block(m.layers[i], params)

    def __del__(self):
        K.kmamba_free(self.p)


def _model_inputs(case, seed):
    V, D = case["V"], case["dim"]
    rng = np.random.default_rng(int(seed))
    s = np.float32(math.sqrt(6.0 / (V + D)))
    # Made on the GPU for speed, kept on the host as the model keeps them.
    g = _gen(seed)
    host = lambda *sh: ((torch.rand(sh, device=DEV, generator=g) * 2 - 1) * float(s)).cpu().numpy()  # noqa: E731
    emb, head = host(V, D), host(D, V)
    layers = [_block_params(rng, D, 1) for _ in range(case["layers"])]
    toks = rng.integers(0, V, case["L"]).astype(np.uint32)
    return emb, head, layers, toks


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("scan1d", "scan1d_step"):
        x, dt, A, Bm, Cm, extra, skip = _scan1d_inputs(case, seed)
        B, L, D = x.shape
        y = torch.empty_like(x)
        if kind == "scan1d":
            hf = torch.empty((B, D, N), device=DEV)
            kw = {"z": extra, "Dskip": skip} if case["gated"] else {}
            args = K.scan1d_fwd_args(x, dt, A, Bm, Cm, y, h_final=hf, **kw)
            return {"kind": kind, "fwd": args, "out": (y, hf), "keep": (x, dt, A, Bm, Cm, extra, skip)}
        ck = torch.empty((B, -(-L // K.KM_SCAN1D_CKPT_STEPS), D, N), device=DEV)
        dx, ddt, dA = torch.empty_like(x), torch.empty_like(x), torch.empty_like(A)
        dB, dC = torch.empty_like(Bm), torch.empty_like(Cm)
        fwd = K.scan1d_fwd_args(x, dt, A, Bm, Cm, y, h_ckpt=ck)
        bwd = K.scan1d_bwd_args(x, dt, A, Bm, Cm, extra, dx, ddt, dA, dB, dC, h_ckpt=ck)
        return {"kind": kind, "fwd": fwd, "bwd": bwd, "out": (y, dx, ddt, dA, dB, dC),
                "keep": (x, dt, A, Bm, Cm, extra, ck)}
    if kind in ("grid", "grid_step"):
        dims = _dims(case)
        x, A, B, Cm, dt, dy = _grid_inputs(case, seed)
        h, y = torch.empty_like(B), torch.empty_like(x)
        fwd, keep = K.scannd_params(dims, x, A, B, Cm, dt, h, y)
        s = {"kind": kind, "fwd": fwd, "out": (h, y), "keep": (keep, x, A, B, Cm, dt, dy)}
        if kind == "grid_step":
            dx, ddt, dA = torch.empty_like(x), torch.empty_like(dt), torch.empty_like(A)
            dB, dC = torch.empty_like(B), torch.empty_like(Cm)
            p = K.ptr
            s["bwd"] = K.KMScanNDBwd(keep, len(dims), case["D"], N, p(x), p(A), p(B), p(Cm), p(dt), p(h),
                                     p(dy), p(dx), p(ddt), p(dA), p(dB), p(dC), None, 0)
            s["out"] += (dx, ddt, dA, dB, dC)
        return s
    if kind == "conv_step":
        inp, ker, bias, dy = _conv_inputs(case, seed)
        out, din = torch.empty_like(inp), torch.empty_like(inp)
        dker, db = torch.empty_like(ker), torch.empty_like(bias)
        args, keep = K.convnd_params(_dims(case), inp, ker, bias, out, dy, din, dker, db, D=case["D"],
                                     K=case["K"])
        return {"kind": kind, "args": args, "out": (out, din, dker, db), "keep": (keep, inp, ker, bias, dy)}
    if kind == "mamba1":
        w, x = _mamba1_inputs(case, seed)
        out = torch.empty_like(x)
        st = K.mamba1_weights(w)
        nb = K.km_mamba1_block_workspace_bytes(C.byref(st), case["B"], case["L"])
        ws = torch.empty(nb, dtype=torch.uint8, device=DEV)
        return {"kind": kind, "w": st, "x": x, "out": (out,), "ws": ws, "nb": nb, "B": case["B"],
                "L": case["L"], "keep": w}
    if kind == "mamba3":
        params = _block_params(np.random.default_rng(int(seed)), case["dim"], case["R"])
        x = torch.randn((case["B"], case["L"], case["dim"]), device=DEV, generator=_gen(seed))
        return {"kind": kind, "blk": _Block(case["dim"], case["L"], case["R"], params), "x": x,
                "out": (torch.empty_like(x),), "B": case["B"]}
    emb, head, layers, toks = _model_inputs(case, seed)
    return {"kind": kind, "model": _Model(case, emb, head, layers), "toks": toks,
            "out": (np.empty((case["L"], case["V"]), np.float32),)}


def run(s):
    kind = s["kind"]
    if kind == "scan1d":
        _check(K.km_scan1d_fwd_c(C.byref(s["fwd"]), _stream()))
    elif kind == "scan1d_step":
        _check(K.km_scan1d_fwd_c(C.byref(s["fwd"]), _stream()))
        _check(K.km_scan1d_bwd_c(C.byref(s["bwd"]), _stream()))
    elif kind == "grid":
        _check(K.km_scannd_fwd_c(C.byref(s["fwd"]), _stream()))
    elif kind == "grid_step":
        _check(K.km_scannd_fwd_c(C.byref(s["fwd"]), _stream()))
        _check(K.km_scannd_bwd_c(C.byref(s["bwd"]), _stream()))
    elif kind == "conv_step":
        _check(K.km_convnd_fwd_c(C.byref(s["args"]), 1, _stream()))
        _check(K.km_convnd_bwd_c(C.byref(s["args"]), 1, _stream()))
    elif kind == "mamba1":
        _check(K.km_mamba1_block_fwd_c(C.byref(s["w"]), s["x"].data_ptr(), s["out"][0].data_ptr(), s["B"],
                                       s["L"], s["ws"].data_ptr(), s["nb"], _stream()))
    elif kind == "mamba3":
        K.mamba_block_forward(s["blk"].p, s["out"][0].data_ptr(), s["x"].data_ptr(), s["B"])
        if K.km_last_error_c():
            raise RuntimeError(K.km_last_error())
    else:
        _check(K.kmamba_forward(s["model"].p, s["toks"].ctypes.data, s["out"][0].ctypes.data))
    return s["out"]


def work(case):
    kind = case["kind"]
    if kind in ("scan1d", "scan1d_step"):
        B, L, D = case["B"], case["L"], case["D"]
        e = 2 if case["dtype"] == "bf16" else 4
        ld, bc = B * L * D * e, B * L * N * e
        upd = B * L * D * N
        if kind == "scan1d":
            return {"bytes": (3 + case["gated"]) * ld + 2 * bc + 4 * D * N + 4 * B * D * N,
                    "flops": 6 * upd}
        # Forward: x, delta, B, C, A in, y out. Backward: x, delta, dy, B, C, A in, five gradients out.
        return {"bytes": 8 * ld + 6 * bc + 3 * 4 * D * N, "flops": 6 * upd + 16 * upd}
    if kind in ("grid", "grid_step"):
        dims, D = _dims(case), case["D"]
        nd, P = len(dims), int(np.prod(dims))
        pd, pdm, a = 4 * P * D, 4 * P * D * N, 4 * nd * D * N
        fwd = (2 + nd) * pd + 3 * pdm + a
        flops = (2 * nd + 5) * P * D * N
        if kind == "grid":
            return {"bytes": fwd, "flops": flops}
        return {"bytes": fwd + (3 + 2 * nd) * pd + 5 * pdm + 2 * a, "flops": flops + (7 * nd + 10) * P * D * N}
    if kind == "conv_step":
        dims, D, KV = _dims(case), case["D"], case["K"] ** len(_dims(case))
        pd = 4 * int(np.prod(dims)) * D
        return {"bytes": 5 * pd + 3 * 4 * KV * D + 2 * 4 * D, "flops": 6 * KV * pd // 4}
    if kind == "mamba1":
        dim, T = case["dim"], case["B"] * case["L"]
        di, R = 2 * dim, (dim // 16 + 7) // 8 * 8
        wts = 2 * (2 * di * dim + (R + 2 * N) * di + di * R + dim * di) + 4 * (4 * di + 3 * di + di * N)
        return {"bytes": 4 * T * dim + wts,
                "flops": 2 * T * (2 * di * dim + (R + 2 * N) * di + R * di + dim * di)
                + T * di * (6 * N + 8 + 8)}
    if kind == "mamba3":
        dim, T, R = case["dim"], case["B"] * case["L"], case["R"]
        J = R + 2 + 2 * N * R
        return {"bytes": 8 * T * dim + 4 * (J + R) * dim, "flops": 2 * T * dim * (J + R) + 20 * T * N * R}
    D, V, L, n = case["dim"], case["V"], case["L"], case["layers"]
    J = 3 + 2 * N
    return {"bytes": 4 * (L * D + D * V + L * V + n * (J + 1) * D),
            "flops": 2 * L * D * V + n * (2 * L * D * (J + 1) + 20 * L * N)}


def tolerance(case):
    # About four times the errors measured against exact(): up to 5.7e-7 where sums run in
    # 32 bits, 1.7e-3 for bf16 results, 3.9e-3 for the Mamba-1 block, whose activations are
    # rounded to bf16 between its layers. Single elements sit on cancelling sums (32 bits)
    # or differ by a bf16 step.
    kind = case["kind"]
    if kind == "mamba1":
        return {"rel": 1.6e-2, "max": 0.1}
    if kind in ("scan1d", "scan1d_step") and case["dtype"] == "bf16":
        return {"rel": 7e-3, "max": 0.05}
    return {"rel": 4e-6, "max": 4e-4}


# --- the same in 64 bits -----------------------------------------------------------

def _scan1d_fwd64(x, dt, A, Bm, Cm, keep_h):
    """y [B, L, D], the final state and (keep_h) every state [L, B, D, N]."""
    B, L, D = x.shape
    h = torch.zeros((B, D, N), device=DEV, dtype=F64)
    y = torch.empty((B, L, D), device=DEV, dtype=F64)
    hist = torch.empty((L, B, D, N), device=DEV, dtype=F64) if keep_h else None
    for t in range(L):
        u = (dt[:, t] * x[:, t])[..., None]
        h = torch.exp(dt[:, t, :, None] * A) * h + u * Bm[:, t, None, :]
        y[:, t] = (h * Cm[:, t, None, :]).sum(-1)
        if keep_h:
            hist[t] = h
    return y, h, hist


def _scan1d_exact(case, seed):
    x, dt, A, Bm, Cm, extra, skip = (t.double() for t in _scan1d_inputs(case, seed))
    step = case["kind"] == "scan1d_step"
    y, h, hist = _scan1d_fwd64(x, dt, A, Bm, Cm, step)
    if not step:
        if case["gated"]:
            y = (y + skip * x) * torch.nn.functional.silu(extra)
        return y, h
    B, L, D = x.shape
    dy, adj = extra, torch.zeros_like(h)
    dx, ddt, dA = torch.empty_like(x), torch.empty_like(x), torch.zeros_like(A)
    dB, dC = torch.empty_like(Bm), torch.empty_like(Cm)
    for t in range(L - 1, -1, -1):
        d, xt, g = dt[:, t, :, None], x[:, t, :, None], dy[:, t, :, None]
        ah = adj + g * Cm[:, t, None, :]
        adj = ah * torch.exp(d * A)
        q = adj * hist[t - 1] if t > 0 else torch.zeros_like(adj)      # ah e h_{t-1}
        sb = (ah * Bm[:, t, None, :]).sum(-1)
        dx[:, t] = d[..., 0] * sb
        ddt[:, t] = (A * q).sum(-1) + xt[..., 0] * sb
        dA += (d * q).sum(0)
        dB[:, t] = (ah * (d * xt)).sum(1)
        dC[:, t] = (g * hist[t]).sum(1)
    return y, dx, ddt, dA, dB, dC


def _levels(dims):
    """Point indices by wavefront level (sum of the coordinates), ascending."""
    grid = torch.meshgrid(*[torch.arange(n, device=DEV) for n in dims], indexing="ij")
    lev = sum(grid).reshape(-1)
    order = torch.argsort(lev, stable=True)
    sizes = torch.bincount(lev).tolist()
    return torch.split(order, sizes), [g.reshape(-1) for g in grid]


def _grid_exact(case, seed):
    dims, D = _dims(case), case["D"]
    nd, P = len(dims), int(np.prod(dims))
    x, A, B, Cm, dt, dy = _grid_inputs(case, seed)
    st = [int(np.prod(dims[a + 1:])) for a in range(nd)]
    levels, co = _levels(dims)
    A = A.double()
    dtb = dt.double().mean(0)
    h = torch.empty((P, D, N), device=DEV, dtype=F64)
    for idx in levels:
        v = (dtb[idx] * x[idx].double())[..., None] * B[idx].double()
        for a in range(nd):
            ok = co[a][idx] > 0
            q = idx[ok]
            v[ok] += torch.exp(dt[a, q].double()[..., None] * A[a]) * h[q - st[a]]
        h[idx] = v
    y = torch.empty((P, D), device=DEV, dtype=F64)
    for c in torch.arange(P, device=DEV).split(4096):
        y[c] = (h[c] * Cm[c].double()).sum(-1)
    if case["kind"] == "grid":
        return h, y
    g = torch.empty_like(h)
    for idx in reversed(levels):
        v = dy[idx].double()[..., None] * Cm[idx].double()
        for a in range(nd):
            ok = co[a][idx] + 1 < dims[a]
            nx = idx[ok] + st[a]
            v[ok] += torch.exp(dt[a, nx].double()[..., None] * A[a]) * g[nx]
        g[idx] = v
    dx, ddt = torch.empty_like(y), torch.empty((nd, P, D), device=DEV, dtype=F64)
    dA, dC = torch.zeros_like(A), torch.empty_like(h)
    for c in torch.arange(P, device=DEV).split(4096):
        gv, bv, xv, db = g[c], B[c].double(), x[c].double(), dtb[c]
        dC[c] = dy[c].double()[..., None] * h[c]
        s = (gv * bv).sum(-1)
        dx[c] = s * db
        for a in range(nd):
            ok = (co[a][c] > 0).double()[:, None, None]
            prev = h[(c - st[a]).clamp(min=0)] * ok
            gh = gv * torch.exp(dt[a, c].double()[..., None] * A[a]) * prev
            ddt[a, c] = s * xv / nd + (gh * A[a]).sum(-1)
            dA[a] += (gh * dt[a, c].double()[..., None]).sum(0)
        g[c] = gv * (db * xv)[..., None]                              # dB, in g's memory
    return h, y, dx, ddt, dA, g, dC


def _conv_exact(case, seed):
    dims, D, k = _dims(case), case["D"], case["K"]
    nd = len(dims)
    inp, ker, bias, dy = (t.double() for t in _conv_inputs(case, seed))
    inp, dy = inp.view(*dims, D), dy.view(*dims, D)
    out, din, dker = bias.expand(*dims, D).clone(), torch.zeros_like(inp), torch.empty_like(ker)
    for kl in range(k ** nd):
        rem, off = kl, []
        for _ in range(nd):
            off.insert(0, k - 1 - rem % k)
            rem //= k
        to = tuple(slice(min(o, n), n) for o, n in zip(off, dims))     # out[c] reads in[c - off]
        fr = tuple(slice(0, max(n - o, 0)) for o, n in zip(off, dims))
        out[to] += inp[fr] * ker[kl]
        din[fr] += dy[to] * ker[kl]
        dker[kl] = (dy[to] * inp[fr]).reshape(-1, D).sum(0)
    return (out.view(-1, D), din.view(-1, D), dker, dy.reshape(-1, D).sum(0))


def _mamba1_exact(case, seed):
    w, x = _mamba1_inputs(case, seed)
    w = {n: v.double() for n, v in w.items()}
    x = x.double()
    di, R = w["W_in"].shape[0] // 2, w["W_dt"].shape[1]
    L = x.shape[1]
    xz = x @ w["W_in"].t()
    xi, z = xz[..., :di], xz[..., di:]
    pad = torch.nn.functional.pad(xi, (0, 0, 3, 0))
    u = torch.nn.functional.silu(sum(pad[:, j:j + L] * w["conv_w"][j] for j in range(4)) + w["conv_b"])
    dbl = u @ w["W_x"].t()
    dt = torch.nn.functional.softplus(dbl[..., :R] @ w["W_dt"].t() + w["dt_bias"])
    y = _scan1d_fwd64(u, dt, w["A"], dbl[..., R:R + N], dbl[..., R + N:], False)[0]
    return (((y + w["Dskip"] * u) * torch.nn.functional.silu(z)) @ w["W_out"].t(),)


def _mamba3_fwd64(params, x):
    p = {n: torch.from_numpy(v).to(DEV).double() for n, v in params.items()}
    B, L, _ = x.shape
    R = p["W_in"].shape[0]
    u = torch.nn.functional.silu(x @ p["W_in"].t())                                     # [B, L, R]
    dt = torch.nn.functional.softplus(x @ p["delta_proj"][0]).clamp(float(np.float32(_DT["dt_min"])),
                                                                    float(np.float32(_DT["dt_max"])))
    lam = torch.sigmoid(x @ p["lambda_proj"][0])
    Bt = (x @ p["W_B"].t() + p["b_B"]).view(B, L, R, N)
    Ct = (x @ p["W_C"].t() + p["b_C"]).view(B, L, R, N)
    bu = (Bt * u[..., None]).sum(2)                                                     # [B, L, N]
    alpha = torch.exp(dt[..., None] * p["A_log"][:, 0])
    prev = torch.nn.functional.pad(bu, (0, 0, 1, 0))[:, :L]
    drive = ((1 - lam) * dt)[..., None] * alpha * prev + (lam * dt)[..., None] * bu
    cs, sn = torch.cos(p["theta"]), torch.sin(p["theta"])
    h, H = torch.zeros((B, N), device=DEV, dtype=F64), torch.empty((B, L, N), device=DEV, dtype=F64)
    for t in range(L):
        h0, h1 = h[:, 0::2], h[:, 1::2]
        r = torch.stack((cs * h0 - sn * h1, sn * h0 + cs * h1), -1).reshape(B, N)
        h = alpha[:, t] * r + drive[:, t]
        H[:, t] = h
    y = (Ct * H[:, :, None]).sum(-1)                                                    # [B, L, R]
    return x + y @ p["W_out"].t()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("scan1d", "scan1d_step"):
        return _scan1d_exact(case, seed)
    if kind in ("grid", "grid_step"):
        return _grid_exact(case, seed)
    if kind == "conv_step":
        return _conv_exact(case, seed)
    if kind == "mamba1":
        return _mamba1_exact(case, seed)
    if kind == "mamba3":
        params = _block_params(np.random.default_rng(int(seed)), case["dim"], case["R"])
        x = torch.randn((case["B"], case["L"], case["dim"]), device=DEV, generator=_gen(seed))
        return (_mamba3_fwd64(params, x.double()),)
    emb, head, layers, toks = _model_inputs(case, seed)
    x = torch.from_numpy(emb[toks.astype(np.int64)]).to(DEV).double()[None]
    for params in layers:
        x = _mamba3_fwd64(params, x)
    return ((x[0] @ torch.from_numpy(head).to(DEV).double()),)
