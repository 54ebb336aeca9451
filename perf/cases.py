"""The attention work that a program serving a model over quantized caches does.

Each case is one call sequence of the package's public entry points at one
size.  Kinds:

  decode   `quantized_sdpa` of one query position over quantized keys that
           the program holds (a shared prefix, another engine's cache)
  step     one decode step: the new token's K / V appended with
           `update_and_fetch`, then `cache_sdpa`
  verify   speculative decoding: a few draft tokens appended and attended to
  prompt   the first pass over a prompt: an empty cache filled, causal
           attention over what it returned
  chunk    a further prompt chunk: into a full rotating window (which is
           quantized again) with causal attention over it, or onto a
           left-padded batch under the mask that the batch cache makes
  layer    a whole attention layer's decode step (`Attention.forward`:
           projections, rotary positions, cache, attention)

Steps that grow a cache take the tokens back with `trim`, as a rejected
draft is, so that every pass is the same step.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "mlx-qsdpa_amd"))

import mlx_qsdpa_amd as mq  # noqa: E402

DEVICE = "cuda"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}


def _case(name, kind, cache, dtype, bits, gs, B, Hq, Hkv, D, N, L=1, pad=0, mask="none"):
    """N: keys attended to.  L: query positions.  pad: the batch's left
    padding is spread over [0, pad].  cache: plain, batch (left-padded),
    window (one ring buffer of N tokens), batch_window."""
    c = dict(kind=kind, cache=cache, dtype=dtype, bits=bits, gs=gs, B=B, Hq=Hq, Hkv=Hkv, D=D, N=N, L=L, pad=pad,
             mask=mask)
    return dict(c, name=name) if name else c


def listed():
    return [
        # A chat's decode step on a small model: the shortest calls, where launches and host time count.
        _case("step_short", "step", "plain", "f16", 4, 64, 1, 8, 2, 128, 4096),
        # Decode over a long context with wide head groups: the benchmark's headline workload.
        _case("decode_long", "decode", "none", "f16", 4, 32, 1, 32, 2, 256, 131072),
        # Continuous batching over long, uneven contexts.
        _case("step_batch", "step", "batch", "f16", 4, 64, 16, 32, 8, 128, 32768, pad=31744),
        # A serving batch with more sequences and shorter contexts, an odd number of them.
        _case("step_serve", "step", "batch", "bf16", 8, 64, 43, 32, 8, 128, 6000, pad=5200),
        # Sliding-window decode of four sequences.
        _case("step_window", "step", "batch_window", "bf16", 8, 128, 4, 16, 4, 128, 4096),
        # A 512-token chunk into a full sliding window.
        _case("chunk_window", "chunk", "batch_window", "bf16", 8, 128, 4, 16, 4, 128, 4096, L=512),
        # A fresh prompt of odd length.
        _case("prompt", "prompt", "plain", "f16", 4, 64, 1, 32, 8, 128, 3000, L=3000),
        # The next chunk of a batch of left-padded prompts, under the mask that the batch cache makes.
        _case("chunk_batch", "chunk", "batch", "bf16", 8, 64, 8, 32, 8, 128, 1500, L=500, pad=700, mask="cache"),
        # Four drafts and the last token verified over a long context.
        _case("verify", "verify", "plain", "f16", 4, 32, 1, 32, 2, 256, 65536, L=5),
        # Decode of a batch on a model with 64-wide heads.
        _case("step_d64", "step", "plain", "f16", 4, 64, 8, 32, 8, 64, 8192),
        # A prompt on such a model.
        _case("prompt_d64", "prompt", "plain", "bf16", 8, 64, 1, 32, 8, 64, 1500, L=1500),
        # One attention layer's decode step, projections and rotary positions included.
        _case("layer_step", "layer", "plain", "f16", 4, 64, 2, 16, 4, 128, 4096),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "step", "step", "step", "verify", "prompt", "prompt", "chunk", "layer"])
    dtype, bits = rng.choice(["f16", "bf16"]), rng.choice([4, 8])
    D = rng.choice([64, 128, 128, 256])
    gs = rng.choice([g for g in (32, 64, 128) if g <= D])
    Hkv = rng.choice([1, 2, 4, 8])
    G = rng.choice([1, 4, 4, 7, 8, 16])
    G = min(G, 8) if Hkv == 8 else G
    row = Hkv * (D * bits // 8 + 4 * D // gs) * 2  # K and V bytes of a token
    budget = 240e6                                  # below the largest listed case's
    mask = "none"
    if kind == "decode":
        B = _log(rng, 1, 16)
        N = min(_log(rng, 200, 131072), max(200, int(budget / (B * row))))
        mask = rng.choice(["none", "none", "bool"])
        return _case(None, kind, "none", dtype, bits, gs, B, G * Hkv, Hkv, D, N, mask=mask)
    if kind == "step":
        cache = rng.choice(["plain", "batch", "batch", "window", "batch_window"])
        B = 1 if cache in ("window",) else _log(rng, 1, 64)
        N = min(_log(rng, 200, 32768), max(200, int(budget / (B * row))))
        pad = int(N * rng.uniform(0.2, 0.95)) if cache == "batch" else 0
        return _case(None, kind, cache, dtype, bits, gs, B, G * Hkv, Hkv, D, N, pad=pad)
    if kind == "verify":
        L = rng.randint(2, 12)
        N = min(_log(rng, 1000, 65536), max(1000, int(budget / row / 4)))
        return _case(None, kind, "plain", dtype, bits, gs, 1, G * Hkv, Hkv, D, N, L=L)
    if kind == "chunk":
        cache, B = rng.choice([("batch_window", 1), ("batch_window", 4), ("batch", 2), ("batch", 7)])
        N = _log(rng, 1024, 4096)
        # The pairs of heads of 64 are fewer: those calls cost more of them.
        L = min(_log(rng, 33, 512), max(17, int((4.5e9 if D == 64 else 16e9) / (B * G * Hkv * N * D))))
        batch = cache == "batch"
        return _case(None, kind, cache, dtype, bits, gs, B, G * Hkv, Hkv, D, N, L=L, pad=N // 3 if batch else 0,
                     mask="cache" if batch else "none")
    if kind == "prompt":
        B = rng.choice([1, 1, 2, 5])
        heads = G * Hkv
        N = min(_log(rng, 100, 3000), int(math.sqrt((4.5e9 if D == 64 else 12e9) / (B * heads * D))))
        return _case(None, kind, "batch" if B > 1 else "plain", dtype, bits, gs, B, heads, Hkv, D, N, L=N,
                     pad=int(N * 0.6) if B > 1 else 0)
    heads = min(G * Hkv, 4096 // D // Hkv * Hkv)
    return _case(None, "layer", "plain", dtype, bits, gs, rng.choice([1, 2, 4]), heads, Hkv, D, _log(rng, 512, 8192))


# ---- inputs ----------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _rows(case, g, n):
    """Keys or values [B, Hkv, n, D]: normal, with a few louder channels as
    real keys have."""
    x = torch.randn(case["B"], case["Hkv"], n, case["D"], generator=g, device=DEVICE, dtype=DTYPES[case["dtype"]])
    x[..., :: max(1, case["D"] // 4)] *= 3
    return x


def _queries(case, g):
    q = torch.randn(case["B"], case["Hq"], case["L"], case["D"], generator=g, device=DEVICE) * 1.5
    return q.to(DTYPES[case["dtype"]])


def _padding(case):
    B = case["B"]
    return [0] * B if not case["pad"] else [(i * 7919 % B) * case["pad"] // max(1, B - 1) for i in range(B)]


def _held(case):
    """Tokens that the cache holds before the pass (a window is full)."""
    if case["kind"] == "decode" or case["cache"] in ("window", "batch_window"):
        return case["N"]
    return case["N"] - case["L"]


def _inputs(case, seed):
    """(keys, values held; new keys, new values; queries or layer input) from the seed alone."""
    g = _gen(seed)
    held = _held(case)
    k, v = (_rows(case, g, held), _rows(case, g, held)) if held else (None, None)
    kn = vn = None
    if case["kind"] in ("step", "verify", "prompt", "chunk"):
        kn, vn = _rows(case, g, case["L"]), _rows(case, g, case["L"])
    if case["kind"] == "layer":
        dim = case["Hq"] * case["D"]
        x = torch.randn(case["B"], 1, dim, generator=g, device=DEVICE).to(DTYPES[case["dtype"]])
    else:
        x = _queries(case, g)
    if case["mask"] == "bool":
        keep = torch.rand(case["B"], 1, 1, case["N"], generator=g, device=DEVICE) < 0.8
        keep[..., -1] = True
    else:
        keep = None
    return k, v, kn, vn, x, keep


def _layer(case, seed):
    """The layer, its weights drawn from the seed."""
    g = torch.Generator().manual_seed(int(seed) + 1)
    dim = case["Hq"] * case["D"]
    layer = mq.Attention(dim, case["Hq"], case["Hkv"], head_dim=case["D"], dtype=DTYPES[case["dtype"]])
    layer.reset_parameters(g)
    return layer


def _new_cache(case):
    kw = dict(bits=case["bits"], group_size=case["gs"])
    if case["cache"] == "batch":
        return mq.BatchQuantizedSDPACache(_padding(case), **kw)
    if case["cache"] == "window":
        return mq.QuantizedRotatingSDPACache(case["N"], **kw)
    if case["cache"] == "batch_window":
        return mq.BatchQuantizedRotatingSDPACache(_padding(case), case["N"], **kw)
    return mq.QuantizedSDPACache(**kw)


def prepare(case, seed):
    k, v, kn, vn, x, keep = _inputs(case, seed)
    s = {"case": case, "kn": kn, "vn": vn, "x": x, "mask": keep}
    if case["kind"] == "decode":
        s["k"] = mq.quantize(k, case["gs"], case["bits"])
        s["v"] = mq.quantize(v, case["gs"], case["bits"])
        return s
    cache = _new_cache(case)
    if k is not None:
        cache.update_and_fetch(k, v)
    if case["cache"] in ("window", "batch_window"):
        # The window as a saved prompt cache: every pass restores it.
        s["window"] = (type(cache), cache.state, cache.meta_state)
    elif case["kind"] != "prompt":
        s["cache"] = cache
    if case["kind"] == "layer":
        s["layer"] = _layer(case, seed).to(DEVICE)
    return s


def _whole(kv):
    """A cache's (packed, scales, biases), the codes as int32 words."""
    return kv[0].view(torch.int32), kv[1], kv[2]


# ---- the passes ------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        k, v = s["k"], s["v"]
        return mq.quantized_sdpa(s["x"], k[0], v[0], k[1], v[1], k[2], v[2], mask=s["mask"], bits=case["bits"],
                                 group_size=case["gs"])
    if kind == "layer":
        with torch.no_grad():
            out = s["layer"](s["x"], cache=s["cache"])
        state = tuple(_whole(t) for t in s["cache"].state)
        s["cache"].trim(1)
        return out, state
    if "window" in s:
        cls, state, meta = s["window"]
        cache = cls.from_state(state, meta)
    else:
        cache = s["cache"] if "cache" in s else _new_cache(case)
    mask = "causal" if case["L"] > 1 else None
    start = None
    if case["mask"] == "cache":
        mask = cache.make_mask(case["L"])
    k, v = cache.update_and_fetch(s["kn"], s["vn"])
    if case["cache"] == "batch" and case["mask"] != "cache":
        start = cache.kv_start(DEVICE)
    out = mq.cache_sdpa(s["x"], k, v, cache, mask=mask, kv_start=start)
    if "cache" in s:
        cache.trim(case["L"])
    return out, _whole(k), _whole(v)


# ---- what a pass cannot do without -----------------------------------------
def _pairs(case):
    """(query position, key) pairs that are attended to, over the batch."""
    N, L = case["N"], case["L"]
    total = 0
    for p in _padding(case):
        if case["mask"] == "cache":  # keys [p, N - L + i - p] for query i
            total += sum(max(0, N - L + i - 2 * p + 1) for i in range(L))
        elif L == 1:
            total += N - p
        else:  # query i sees keys [p, N - L + i]
            total += sum(max(0, N - L + i - p + 1) for i in range(L))
    return total


def work(case):
    B, Hq, Hkv, D, L, N = (case[x] for x in ("B", "Hq", "Hkv", "D", "L", "N"))
    row = 2 * Hkv * (D * case["bits"] // 8 + 4 * (D // case["gs"]))  # K and V bytes of a token
    tokens = sum(N - p for p in _padding(case))
    qo = 2 * B * Hq * L * D * 2
    new = B * L * Hkv * D * 2 * 2  # new keys and values in 16 bits
    kind = case["kind"]
    flops = 4.0 * _pairs(case) * Hq * D
    if kind == "decode":
        return {"bytes": tokens * row + qo + (B * N if case["mask"] == "bool" else 0), "flops": flops}
    if kind == "layer":
        dim = Hq * D
        weights = 2 * dim * (2 * dim + 2 * Hkv * D)
        return {"bytes": tokens * row + weights + 2 * B * dim * 2, "flops": flops + B * weights}
    if kind == "prompt":  # written once; what is attended to comes from the caches on the way
        return {"bytes": B * N * row + qo + new, "flops": flops}
    if case["mask"] == "cache":  # and the mask, once
        return {"bytes": tokens * row + qo + new + B * L * N, "flops": flops}
    if kind == "chunk":  # the window read and written again, then attended to
        return {"bytes": 2 * B * N * row + qo + new, "flops": flops}
    return {"bytes": tokens * row + qo + new, "flops": flops}


def tolerance(case):
    # About four times the error against 64 bits that was seen: 16-bit
    # outputs and softmax weights.  Codes, scales and biases stay as they are,
    # but for the layer's own new row, which the projections' rounding reaches.
    rel = {"f16": 2e-3, "bf16": 1e-2}[case["dtype"]]
    if case["kind"] == "layer":
        return {"rel": 2 * rel, "max": 0.2, "differ": 2e-4}
    return {"rel": rel, "max": 0.1}


# ---- the same in 64 bits ---------------------------------------------------
def _quantized(x, bits, gs):
    """The affine format's values of x: each group's codes under its 16-bit
    scale and bias, the value rounded to x's type as a stored one is."""
    def over(a, b):  # the correctly rounded 32-bit quotient, on any device
        return (a.double() / b.double()).float()

    bins = torch.tensor(float((1 << bits) - 1), device=x.device)
    w = x.float().unflatten(-1, (-1, gs))
    lo, hi = w.amin(-1, keepdim=True), w.amax(-1, keepdim=True)
    scale = over(hi - lo, bins).clamp_min(1e-7)
    low = lo.abs() > hi.abs()
    scale = torch.where(low, scale, -scale)
    edge = torch.where(low, lo, hi)
    q0 = torch.round(over(edge, scale))
    scale = torch.where(q0 != 0, over(edge, q0), scale)
    bias = torch.where(q0 != 0, edge, torch.zeros_like(edge))
    codes = torch.round(over(w - bias, scale)).clamp(0, float(bins))
    s, b = scale.to(x.dtype).double(), bias.to(x.dtype).double()
    return (s * codes.double() + b).float().to(x.dtype).flatten(-2)


def _attention(q, k, v, keep):
    """[Hq, L, D] over [Hkv, N, D] in 64 bits; keep: bool, broadcastable to [L, N]."""
    Hq, L, D = q.shape
    Hkv, N = k.shape[:2]
    out = torch.empty(Hq, L, D, dtype=torch.float64, device=q.device)
    G = Hq // Hkv
    for h in range(Hkv):
        s = torch.matmul(q[h * G:(h + 1) * G].double(), k[h].double().t().contiguous()) * D ** -0.5
        if keep is not None:
            s = s.masked_fill(~keep, float("-inf"))
        s = s - s.amax(-1, keepdim=True).clamp_min(-1e300)
        e = torch.exp(s)
        out[h * G:(h + 1) * G] = torch.matmul(e, v[h].double()) / e.sum(-1, keepdim=True).clamp_min(1e-300)
    return out


def _rotated(x, pos, theta=10000.0):
    """Rotary positions, half-split layout: x [B, H, D] in 64 bits, all at position pos."""
    D = x.shape[-1]
    ang = pos * theta ** (-torch.arange(0, D, 2, device=x.device, dtype=torch.float64) / D)
    x1, x2 = x[..., : D // 2], x[..., D // 2:]
    return torch.cat([x1 * ang.cos() - x2 * ang.sin(), x2 * ang.cos() + x1 * ang.sin()], -1)


def exact(case, seed):
    k, v, kn, vn, x, keep = _inputs(case, seed)
    T, bits, gs = DTYPES[case["dtype"]], case["bits"], case["gs"]
    B, Hq, Hkv, D, N, L = (case[n] for n in ("B", "Hq", "Hkv", "D", "N", "L"))
    weights = None
    if case["kind"] == "layer":
        layer = _layer(case, seed)
        w = [p.weight.detach().to(DEVICE).double() for p in (layer.q_proj, layer.k_proj, layer.v_proj, layer.o_proj)]
        x64 = x[:, 0].double()
        q, kn, vn = ((x64 @ m.t()).reshape(B, -1, D) for m in w[:3])
        x = _rotated(q, N - 1)[:, :, None]
        kn, vn = _rotated(kn, N - 1).to(T)[:, :, None], vn.to(T)[:, :, None]
        weights = w[3]
    pads = _padding(case)
    outs = []
    for b in range(B):
        if case["kind"] == "chunk" and case["cache"] == "batch_window":
            # The window's stored values, then the chunk, the newest N quantized again.
            kb, vb = ((torch.cat([_quantized(o[b], bits, gs), n[b]], 1))[:, -N:] for o, n in ((k, kn), (v, vn)))
        elif case["cache"] in ("window", "batch_window"):
            # One token in the place of the oldest (a full window; order does not matter to one query).
            kb, vb = torch.cat([k[b][:, 1:], kn[b]], 1), torch.cat([v[b][:, 1:], vn[b]], 1)
        elif kn is None:
            kb, vb = k[b], v[b]
        elif k is None:
            kb, vb = kn[b], vn[b]
        else:
            kb, vb = torch.cat([k[b], kn[b]], 1), torch.cat([v[b], vn[b]], 1)
        kb, vb = _quantized(kb, bits, gs), _quantized(vb, bits, gs)
        rows = torch.arange(L, device=DEVICE)[:, None] + (N - L)
        cols = torch.arange(N, device=DEVICE)[None, :]
        if keep is not None:
            m = keep[b, 0]
        elif case["mask"] == "cache":
            m = (rows - pads[b] >= cols) & (cols >= pads[b])
        else:
            m = (rows >= cols) & (cols >= pads[b])
        outs.append(_attention(x[b], kb, vb, m))
    out = torch.stack(outs)
    if case["kind"] == "layer":
        out = out.reshape(B, 1, Hq * D) @ weights.t()
        return out, (None, None)
    if case["kind"] == "decode":
        return out
    return out, None, None
