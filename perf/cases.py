"""Timed work of the token sampler and its logits projection.

Each case is one pass through a public entry point of gs_sampler.py, as a
decoding program makes it:

  row     Sampler.sample: one row, one token (the chat loop's call)
  batch   Sampler.sample_batch: B device rows, one token each
  gemv    QMatrix.gemv: B logit vectors from a quantized output matrix
  decode  Decoder.step: the projection, the sampling and the commit of B rows

listed() holds the sizes of the configurations, tests and benchmark; draw()
spreads over the same ranges.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gguf-rs-cli_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import gs_sampler as gs  # noqa: E402

# GGUF block types: id, weights per block, bytes per block.
QTYPES = {
    "q4_0": (2, 32, 18), "q4_1": (3, 32, 20), "q8_0": (8, 32, 34), "q3_k": (11, 256, 110),
    "q4_k": (12, 256, 144), "q5_k": (13, 256, 176), "q6_k": (14, 256, 210),
}
MAX_NEW = 16384  # generated ids kept per decoding row


def listed():
    return [
        # One chat row with the command line's default settings: the latency of a token.
        dict(name="row_32000", kind="row", V=32000, T=0.7, k=40, p=0.9, rep=1.1, W=64, sigma=3.0, spikes=5, host=False),
        # The same call as a host program makes it: the logits are in host memory.
        dict(name="row_host_152064", kind="row", V=152064, T=0.7, k=40, p=0.9, rep=1.1, W=64, sigma=3.0, spikes=5,
             host=True),
        # A small serving batch with top-k, one setting for all rows.
        dict(name="topk_64x128256", kind="batch", B=64, V=128256, T=0.8, k=40, p=0.9, rep=1.1, W=128, sigma=2.5,
             spikes=10, mixed=False),
        # A few rows that sample from the whole vocabulary (no top-k), odd row length, windows.
        dict(name="nucleus_8x50257", kind="batch", B=8, V=50257, T=0.8, k=0, p=0.9, rep=1.1, W=64, sigma=2.5,
             spikes=3, mixed=False),
        # A full batch of flat rows with a wide nucleus: the whole vocabulary counts in every row.
        dict(name="nucleus_256x152064", kind="batch", B=256, V=152064, T=1.0, k=0, p=0.95, rep=1.0, W=0, sigma=2.0,
             spikes=0, mixed=False),
        # Rows of many users: temperature, top-k, top-p and penalty of their own.
        dict(name="mixed_512x256000", kind="batch", B=512, V=256000, T=0.0, k=0, p=0.0, rep=0.0, W=256, sigma=3.0,
             spikes=3, mixed=True),
        # A large batch with top-k and long windows (one step of a device-resident loop).
        dict(name="topk_1024x152064", kind="batch", B=1024, V=152064, T=0.7, k=50, p=0.9, rep=1.3, W=1024, sigma=3.0,
             spikes=0, mixed=False),
        # The projection alone, a few vectors (parallel conversations on one card).
        dict(name="gemv_q8_0_32000x4096_b4", kind="gemv", q="q8_0", rows=32000, cols=4096, B=4),
        # The projection of a serving batch.
        dict(name="gemv_q4_k_128256x4096_b16", kind="gemv", q="q4_k", rows=128256, cols=4096, B=16),
        # One vector of a wider model.
        dict(name="gemv_q5_k_32000x8192_b1", kind="gemv", q="q5_k", rows=32000, cols=8192, B=1),
        # The whole step of one conversation with the default settings.
        dict(name="decode_q6_k_152064x3584_b1", kind="decode", q="q6_k", rows=152064, cols=3584, B=1, T=0.7, k=40,
             p=0.9, rep=1.1, W=64),
        # The whole step of a serving batch.
        dict(name="decode_q4_k_152064x3584_b32", kind="decode", q="q4_k", rows=152064, cols=3584, B=32, T=0.7, k=40,
             p=0.9, rep=1.1, W=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("row", "batch", "batch", "batch", "gemv", "gemv", "gemv", "decode"))
    T = round(rng.uniform(0.5, 1.3), 3)
    k = rng.choice((0, 20, 40, 50, 100))
    p = round(rng.uniform(0.8, 1.0), 3)
    rep = rng.choice((1.0, 1.1, 1.3))
    W = rng.choice((0, 64, 128, 1024))
    sigma = round(rng.uniform(1.5, 3.5), 3)
    spikes = rng.choice((0, 3, 10))
    if kind == "row":
        return dict(kind=kind, V=_log(rng, 4000, 256000), T=T, k=k, p=p, rep=rep, W=W, sigma=sigma, spikes=spikes,
                    host=rng.random() < 0.5)
    if kind == "batch":
        V = _log(rng, 4000, 256000)
        V -= V % 4 if rng.random() < 0.5 else 0
        B = min(_log(rng, 1, 1024), 131072000 // V)
        return dict(kind=kind, B=B, V=V, T=T, k=k, p=p, rep=rep, W=W, sigma=sigma, spikes=spikes,
                    mixed=rng.random() < 0.25)
    q = rng.choice(sorted(QTYPES))
    cols = _log(rng, 1024, 8192)
    cols -= cols % QTYPES[q][1]
    rows = min(_log(rng, 4000, 152064), 545000000 // cols)
    B = _log(rng, 1, 32)
    if kind == "gemv":
        return dict(kind=kind, q=q, rows=rows, cols=cols, B=B)
    return dict(kind=kind, q=q, rows=rows, cols=cols, B=B, T=T, k=k, p=p, rep=rep, W=W)


def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 16 + what)
    return g


def _logits(case, B, seed):
    """B rows N(0, sigma^2), a few entries raised (what a model is sure of)."""
    g = _gen(seed, 1)
    V = case["V"]
    x = torch.randn((B, V), generator=g, device="cuda")
    x *= case["sigma"]
    if case["spikes"]:
        at = torch.randint(0, V, (B, case["spikes"]), generator=g, device="cuda")
        up = 5.0 + 7.0 * torch.rand((B, case["spikes"]), generator=g, device="cuda")
        x.scatter_(1, at, x.gather(1, at) + up)
    return x


def _window(case, B, V, seed):
    """B windows of recent ids (int32 holds their bits)."""
    if not case["W"]:
        return None
    return torch.randint(0, V, (B, case["W"]), generator=_gen(seed, 2), device="cuda", dtype=torch.int32)


def _blocks(q, rows, cols, seed):
    """Raw GGUF blocks of a rows x cols matrix: any quant bits and sub-block
    scales, small positive block scales (weights of about 1e-3 to 1e-1)."""
    _, w, nb = QTYPES[q]
    g = _gen(seed, 3)
    n = rows * (cols // w)
    b = torch.randint(0, 256, (n, nb), generator=g, device="cuda", dtype=torch.uint8)

    def f16(scale):
        v = (torch.rand(n, generator=g, device="cuda") + 0.25) * scale
        return v.to(torch.float16).view(torch.uint8).reshape(n, 2)

    if q in ("q4_0", "q8_0"):
        b[:, 0:2] = f16(0.002)
    elif q == "q4_1":
        b[:, 0:2] = f16(0.002)
        b[:, 2:4] = f16(-0.02)
    elif q == "q3_k":
        b[:, 108:110] = f16(0.0005)
    elif q in ("q4_k", "q5_k"):
        b[:, 0:2] = f16(0.0002)
        b[:, 2:4] = f16(0.0005)
    else:
        b[:, 208:210] = f16(0.00005)
    return b


def _x(cols, B, seed):
    """B normalized hidden states: channels of unequal size."""
    g = _gen(seed, 4)
    gain = torch.exp(0.5 * torch.randn(cols, generator=g, device="cuda"))
    return torch.randn((B, cols), generator=g, device="cuda") * gain


def prepare(case, seed):
    kind = case["kind"]
    if kind == "row":
        s = gs.Sampler(case["T"], case["k"], case["p"], case["rep"], seed=seed)
        s.reserve(1, case["V"])
        x = _logits(case, 1, seed)[0]
        win = _window(case, 1, case["V"], seed)
        win = np.zeros(0, np.uint32) if win is None else win[0].cpu().numpy().view(np.uint32)
        return dict(case=case, s=s, x=x.cpu().numpy() if case["host"] else x, win=win)
    if kind == "batch":
        B, V = case["B"], case["V"]
        g = _gen(seed, 5)
        s = gs.Sampler(case["T"], case["k"], case["p"], case["rep"], seed=seed)
        s.reserve(B, V)
        params = None
        if case["mixed"]:
            r = np.random.default_rng(seed)
            params = gs.params_array(zip(r.uniform(0.3, 1.5, B), r.choice([0, 1, 20, 100], B), r.uniform(0.5, 1.0, B),
                                         r.uniform(1.0, 1.3, B)))
            params = torch.from_numpy(params.view(np.uint8)).cuda()
        return dict(case=case, s=s, x=_logits(case, B, seed), params=params, win=_window(case, B, V, seed),
                    u=torch.rand(B, generator=g, device="cuda"),
                    tokens=torch.zeros(B, dtype=torch.int32, device="cuda"),
                    status=torch.zeros(B, dtype=torch.int32, device="cuda"))
    q, rows, cols, B = case["q"], case["rows"], case["cols"], case["B"]
    m = gs.QMatrix(QTYPES[q][0], _blocks(q, rows, cols, seed).cpu().numpy().reshape(-1), rows, cols)
    st = dict(case=case, m=m, x=_x(cols, B, seed), out=torch.zeros((B, rows), device="cuda"))
    if kind == "decode":
        st["s"] = gs.Sampler(case["T"], case["k"], case["p"], case["rep"], seed=seed)
        st["s"].reserve(B, rows)
        st["d"] = gs.Decoder(B, W=case["W"], max_new=MAX_NEW)
        win = _window(case, B, rows, seed)
        st["d"].init(st["s"], [seed + b for b in range(B)],
                     init_recent=None if win is None else win.cpu().numpy().view(np.uint32))
    return st


def run(state):
    kind = state["case"]["kind"]
    if kind == "row":
        return state["s"].sample(state["x"], state["win"])
    if kind == "batch":
        state["s"].sample_batch(state["x"], state["tokens"], params=state["params"], recent=state["win"],
                                u=state["u"], status=state["status"])
        return dict(tokens=state["tokens"], status=state["status"])
    if kind == "gemv":
        state["m"].gemv(state["x"], state["out"], B=state["case"]["B"])
        return state["out"]
    d = state["d"]
    d.step(state["s"], logits=state["out"], lm_head=state["m"], x=state["x"])
    return dict(logits=state["out"], tokens=d.tokens, status=d.status, next=d.next, window=d.window, u=d.u)


def work(case):
    kind = case["kind"]
    if kind == "row":
        return dict(bytes=4 * case["V"] + 4 * case["W"] + 4, flops=0)
    if kind == "batch":
        return dict(bytes=case["B"] * (4 * case["V"] + 4 * case["W"] + 12 + (16 if case["mixed"] else 0)), flops=0)
    _, w, nb = QTYPES[case["q"]]
    rows, cols, B = case["rows"], case["cols"], case["B"]
    nbytes = rows * (cols // w) * nb + 4 * B * cols + 4 * B * rows
    if kind == "decode":
        nbytes += B * (4 * case["W"] + 12)
    return dict(bytes=nbytes, flops=2 * rows * cols * B)


def tolerance(case):
    # Tokens are exact.  The projection sums in 32 bits, in an order of its own.
    return "exact" if case["kind"] in ("row", "batch") else dict(rel=1e-5, differ=0.001)


def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _weights(q, b):
    """[n blocks, weights] in 64 bits from raw blocks [n, bytes]."""
    n = b.shape[0]
    u = b.to(torch.int16)
    if q == "q8_0":
        return _f16(b[:, 0:2]) * b[:, 2:34].contiguous().view(torch.int8).double()
    if q in ("q4_0", "q4_1"):
        o = 4 if q == "q4_1" else 2
        v = torch.cat([u[:, o:o + 16] & 15, u[:, o:o + 16] >> 4], 1).double()
        return (v - 8) * _f16(b[:, 0:2]) if q == "q4_0" else v * _f16(b[:, 0:2]) + _f16(b[:, 2:4])
    if q == "q6_k":
        out = torch.empty((n, 8, 32), dtype=torch.float64, device=b.device)
        for h in range(2):
            qh = u[:, 128 + 32 * h:160 + 32 * h]
            for j in range(4):
                ql = u[:, 64 * h + 32 * (j & 1):64 * h + 32 * (j & 1) + 32]
                out[:, 4 * h + j] = (((ql >> (4 * (j >> 1))) & 15) | (((qh >> (2 * j)) & 3) << 4)) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        return out.reshape(n, 256) * (sc * _f16(b[:, 208:210])).repeat_interleave(16, 1)
    if q == "q3_k":
        out = torch.empty((n, 8, 32), dtype=torch.float64, device=b.device)
        for h in range(2):
            for j in range(4):
                lo = (u[:, 32 + 32 * h:64 + 32 * h] >> (2 * j)) & 3
                out[:, 4 * h + j] = lo + 4 * ((u[:, 0:32] >> (4 * h + j)) & 1) - 4
        s = u[:, 96:108]
        low = torch.cat([s[:, 0:8] & 15, s[:, 0:8] >> 4], 1)
        top = torch.cat([(s[:, 8:12] >> (2 * k)) & 3 for k in range(4)], 1)
        sc = (low + 16 * top - 32).double()
        return out.reshape(n, 256) * (sc * _f16(b[:, 108:110])).repeat_interleave(16, 1)
    s = u[:, 4:16]
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double() * _f16(b[:, 0:2])
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double() * _f16(b[:, 2:4])
    out = torch.empty((n, 8, 32), dtype=torch.float64, device=b.device)
    qs = u[:, 48:176] if q == "q5_k" else u[:, 16:144]
    for j in range(8):
        v = (qs[:, 32 * (j >> 1):32 * (j >> 1) + 32] >> (4 * (j & 1))) & 15
        if q == "q5_k":
            v = v + 16 * ((u[:, 16:48] >> j) & 1)
        out[:, j] = v
    return (out * sc[:, :, None] - mn[:, :, None]).reshape(n, 256)


def exact(case, seed):
    """The logits in 64 bits.  Tokens are defined by 32-bit sums in a fixed
    order: 64 bits give no other value to compare them with."""
    if case["kind"] in ("row", "batch"):
        return None
    q, rows, cols, B = case["q"], case["rows"], case["cols"], case["B"]
    b = _blocks(q, rows, cols, seed).reshape(rows, -1)
    x = _x(cols, B, seed).double()
    out = torch.empty((B, rows), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 25) // cols)
    for r in range(0, rows, step):
        w = _weights(q, b[r:r + step].reshape(-1, QTYPES[q][2])).reshape(-1, cols)
        out[:, r:r + step] = (w @ x.t().contiguous()).t()
    if case["kind"] == "gemv":
        return out
    return dict(logits=out, tokens=None, status=None, next=None, window=None, u=None)
