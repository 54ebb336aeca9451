"""64-wide heads on the matrix-core kernels, against the float64 oracle
(tests/torch_oracle.py).

Bars: a 16-bit output is off by half an ulp (2^-11 of a float16 value, 2^-9
of a bfloat16 one); P enters P.V with 22 (float16) or 16 (bfloat16)
significant bits and the sums are float32, which moves an output by less
than 2^-16 max|V|; both are allowed twice.
"""

import pytest
import torch

import torch_oracle as to

import mlx_qsdpa_amd as mq
from mlx_qsdpa_amd import dispatch, kernels

pytestmark = pytest.mark.gpu

D = 64
F16, BF16 = torch.float16, torch.bfloat16


def _inputs(B, Hq, Hkv, N, L, bits, gs, dtype, symmetric=False, seed=0):
    g = torch.Generator().manual_seed(1000 * N + L + seed)
    q = (torch.randn(B, Hq, L, D, generator=g) * 2).to(dtype).cuda()
    kv = [kernels.quantize(torch.randn(B, Hkv, N, D, generator=g).to(dtype).cuda(), gs, bits) for _ in range(2)]
    return (q, *((p, s, None if symmetric else b) for p, s, b in kv))


def _keep(q, N, mask, kv_start):
    L, dev = q.shape[2], q.device
    cols = torch.arange(N, device=dev)
    keep = torch.ones(1, 1, L, N, dtype=torch.bool, device=dev)
    if isinstance(mask, torch.Tensor):
        keep = keep & mask
    elif mask == "causal":
        keep = keep & (cols[None] <= (N - L) + torch.arange(L, device=dev)[:, None])
    if kv_start is not None:
        keep = keep & (cols >= kv_start.to(dev)[:, None, None, None])
    return keep


def _check(q, k, v, bits, gs, mask=None, kv_start=None, additive=None, **kw):
    print(f"q {tuple(q.shape)} keys {k[0].shape[2]} bits {bits} gs {gs} {q.dtype} {kw}", flush=True)
    N = k[0].shape[2]
    keep = _keep(q, N, mask, kv_start)
    ref_mask = keep if additive is None else additive.float().masked_fill(~keep, float("-inf"))
    want = to.quantized_sdpa(q, k, v, bits=bits, group_size=gs, mask=ref_mask)
    out = mq.quantized_sdpa(q, k[0], v[0], k[1], v[1], k[2], v[2], bits=bits, group_size=gs,
                            mask=mask if additive is None else additive, kv_start=kv_start, **kw)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(out).all())
    ulp = 2.0 ** -11 if q.dtype == F16 else 2.0 ** -9
    vmax = float(to.dequantize(*v, gs, bits, q.dtype).abs().max())
    err = (out.double() - want).abs()
    bad = err > 2 * ulp * want.abs() + 2 * 2.0 ** -16 * vmax
    assert not bool(bad.any()), f"{int(bad.sum())} outside, max err {float(err.max()):.3e}"
    return out


@pytest.mark.parametrize("dtype", [F16, BF16], ids=["f16", "bf16"])
@pytest.mark.parametrize("bits,gs", [(4, 32), (4, 64), (8, 32), (8, 64)])
def test_decode(device, bits, gs, dtype):
    """One position: part-filled tiles, single pass, in-launch merge, merge
    kernel; head groups of 1, 7 and 20 (two row blocks)."""
    for B, Hq, Hkv, N, splits in ((1, 2, 2, 1, None), (2, 14, 2, 33, 1), (1, 7, 1, 1000, 7), (1, 20, 1, 4100, None),
                                  (3, 8, 2, 515, None)):
        q, k, v = _inputs(B, Hq, Hkv, N, 1, bits, gs, dtype)
        _check(q, k, v, bits, gs, num_splits=splits)
    q, k, v = _inputs(2, 8, 2, 300, 1, bits, gs, dtype, symmetric=True)
    _check(q, k, v, bits, gs)


@pytest.mark.parametrize("dtype,bits", [(F16, 4), (BF16, 8)], ids=["f16", "bf16"])
def test_decode_masks_and_starts(device, dtype, bits):
    """Left padding (stream-K, an empty sequence among them), bool and
    additive masks, rows without keys."""
    B, N = 4, 3001
    q, k, v = _inputs(B, 8, 2, N, 1, bits, 32, dtype)
    ks = torch.tensor([0, 2990, N, 1234], dtype=torch.int32, device=device)
    out = _check(q, k, v, bits, 32, kv_start=ks)
    assert bool((out[2] == 0).all())
    keep = torch.rand(B, 1, 1, N, device=device) < 0.5
    keep[1] = False
    out = _check(q, k, v, bits, 32, mask=keep)
    assert bool((out[1] == 0).all())
    _check(q, k, v, bits, 32, mask=keep, kv_start=ks)
    _check(q, k, v, bits, 32, additive=torch.randn(1, 8, 1, N, device=device))


@pytest.mark.parametrize("dtype,bits,gs", [(F16, 4, 32), (F16, 8, 64), (BF16, 4, 64), (BF16, 8, 32)])
def test_several_positions(device, monkeypatch, dtype, bits, gs):
    """Several positions run fused (the fallback is made to fail): causal,
    left padding, a bool mask, a partial last row block."""
    monkeypatch.setattr(dispatch, "fallback_sdpa", None)
    for B, Hq, Hkv, N, L in ((1, 4, 1, 256, 5), (2, 8, 2, 700, 9), (2, 21, 3, 1500, 3), (1, 8, 2, 333, 333)):
        q, k, v = _inputs(B, Hq, Hkv, N, L, bits, gs, dtype)
        _check(q, k, v, bits, gs, mask="causal")
        ks = torch.tensor([40, N - 1][:B], device=device)
        _check(q, k, v, bits, gs, mask="causal", kv_start=ks)
        keep = torch.rand(B, 1, L, N, device=device) < 0.5
        _check(q, k, v, bits, gs, mask=keep)


@pytest.mark.parametrize("dtype,bits,gs", [(F16, 4, 32), (F16, 8, 64), (BF16, 4, 64), (BF16, 8, 32)])
def test_prefill(device, dtype, bits, gs):
    """The prefill kernel (at least 5 * 2^20 query-key pairs): one pass of
    several rounds, key splits, 128-key tiles cut by the end, a start inside a
    tile, the causal limit and masks, and a partial row group."""
    for B, Hq, Hkv, N, L in ((1, 8, 2, 830, 830), (2, 16, 4, 1100, 161), (1, 4, 1, 21000, 66), (1, 24, 8, 767, 300)):
        assert B * Hq * L * N >= 5 << 20 and Hq // Hkv * L >= 128
        q, k, v = _inputs(B, Hq, Hkv, N, L, bits, gs, dtype)
        _check(q, k, v, bits, gs, mask="causal")
        _check(q, k, v, bits, gs)
        _check(q, k, v, bits, gs, mask="causal", kv_start=torch.tensor([130, N - L // 2][:B], device=device))
        if N < 2000:
            keep = torch.rand(B, Hq if L < 200 else 1, L, N, device=device) < 0.5
            keep[0, 0, 3] = False
            _check(q, k, v, bits, gs, mask=keep)
    q, k, v = _inputs(1, 8, 2, 830, 830, bits, gs, dtype, symmetric=True)
    _check(q, k, v, bits, gs, mask="causal")


@pytest.mark.parametrize("size", [1e-9, 1e-3, 3e6])
def test_prefill_value_magnitudes(device, size):
    """bfloat16 V of any magnitude is scaled to the top of float16's range, so
    small values keep their 8 bits as large ones do."""
    q, k, v = _inputs(1, 8, 2, 830, 830, 8, 64, BF16)
    v = (v[0], (v[1].float() * size).to(BF16), (v[2].float() * size).to(BF16))
    _check(q, k, v, 8, 64, mask="causal")


def test_several_positions_on_the_fallback(device, monkeypatch):
    """What the kernel would mask otherwise stays on dequantize + attention."""
    q, k, v = _inputs(2, 4, 2, 300, 3, 4, 32, F16)
    low = torch.full((1, 1, 3, 300), torch.finfo(torch.float32).min, device=device)
    mean = to.dequantize(*v, 32, 4, F16).float().mean(2)  # every score the same
    out = mq.quantized_sdpa(q, k[0], v[0], k[1], v[1], k[2], v[2], mask=low)
    assert float((out.float() - mean.repeat_interleave(2, 1)[:, :, None]).abs().max()) < 2e-3
    column = torch.ones(1, 1, 3, 1, dtype=torch.bool, device=device)  # broadcasts over the keys
    whole = mq.quantized_sdpa(q, k[0], v[0], k[1], v[1], k[2], v[2])
    out = mq.quantized_sdpa(q, k[0], v[0], k[1], v[1], k[2], v[2], mask=column)
    assert float((out.float() - whole.float()).abs().max()) < 2e-3


def test_not_a_number_rows(device):
    """A query row of NaN or infinities gives zeros, as the float32 path's
    softmax gives, and leaves the other rows alone."""
    _nan_rows(3, 600)


def test_not_a_number_rows_prefill(device):
    _nan_rows(700, 2000)   # one pass
    _nan_rows(66, 21000)   # key splits


def _nan_rows(L, N):
    q, k, v = _inputs(1, 4, 1, N, L, 4, 32, F16)
    want = mq.fallback_sdpa(q, k, v, bits=4, group_size=32, scale=D ** -0.5)
    q[0, 1, 2, 5] = float("nan")
    q[0, 3, 0, :] = float("inf")
    out = mq.quantized_sdpa(q, k[0], v[0], k[1], v[1], k[2], v[2])
    ref = mq.fallback_sdpa(q, k, v, bits=4, group_size=32, scale=D ** -0.5)
    assert bool((ref[0, 1, 2] == 0).all()) and bool((out[0, 1, 2] == 0).all()) and bool((out[0, 3, 0] == 0).all())
    rest = torch.ones(4, L, dtype=torch.bool)
    rest[1, 2] = rest[3, 0] = False
    assert float((out[0][rest].float() - want[0][rest].float()).abs().max()) < 2e-3


@pytest.mark.parametrize("dtype,bits", [(F16, 4), (F16, 8), (BF16, 4), (BF16, 8)])
@pytest.mark.parametrize("L", [1, 5, 300])
def test_small_weights_beside_a_large_one(device, L, dtype, bits):
    """One key (an attention sink) holds nearly all of the softmax and its
    value is zero, so the output is the sum over keys of weight 2^-21: they
    keep float32's precision (16-bit terms of a fixed scale would be off by
    percents).  An output is off by its rounding (allowed twice), and by
    scores rounded in float32: 2^-14 of the sum of the weighted |V|."""
    Hq, Hkv, N, gs = 8, 2, 4096, 32
    g = torch.Generator(device="cuda").manual_seed(bits + L)
    u = torch.where(torch.rand(D, generator=g, device=device) < 0.5, 3.0, -3.0)
    kw = torch.randn(1, Hkv, N, D, generator=g, device=device) * 0.5
    vw = torch.randn(1, Hkv, N, D, generator=g, device=device) * 512
    kw[:, :, 7], vw[:, :, 7] = u, 0.0
    k, v = (kernels.quantize(x.to(dtype), gs, bits) for x in (kw, vw))
    q = (u * 0.2 + torch.randn(1, Hq, L, D, generator=g, device=device) * 0.3).to(dtype)
    print(f"sink L={L} {dtype} bits={bits}", flush=True)
    out = mq.quantized_sdpa(q, k[0], v[0], k[1], v[1], k[2], v[2], bits=bits, group_size=gs)
    kd, vd = (to.dequantize(*x, gs, bits, dtype).double().repeat_interleave(Hq // Hkv, 1) for x in (k, v))
    assert bool((vd[:, :, 7] == 0).all())
    p = torch.softmax(torch.matmul(q.double(), kd.transpose(2, 3).contiguous()) * D ** -0.5, -1)
    assert 2.0 ** -24 < float(p[..., :7].median()) < 2.0 ** -18
    want, size = torch.matmul(p, vd), torch.matmul(p, vd.abs())
    ulp = 2.0 ** -11 if dtype == F16 else 2.0 ** -8
    err = (out.double() - want).abs()
    assert bool((err <= 2 * ulp * want.abs() + 2.0 ** -14 * size + 2.0 ** -24).all()), \
        f"{float((err / size).max()):.2e} of the weighted values"


def test_an_infinite_value_stays_infinite(device):
    """A value past float16's range (codes of a group near it round up to
    infinity) makes the dims that read it infinite, as float32 weights do."""
    for L in (1, 5, 300):
        q, k, v = _inputs(1, 4, 1, 6000, L, 8, 32, F16)
        v[2][0, 0, 50, 1] = float("inf")  # the bias of dims 32..63
        out = mq.quantized_sdpa(q, k[0], v[0], k[1], v[1], k[2], v[2], bits=8, group_size=32)
        assert bool(torch.isposinf(out[..., 32:]).all()) and bool(torch.isfinite(out[..., :32]).all())


@pytest.mark.parametrize("alone", ["keys", "values"])
def test_biases_of_one_alone(device, alone):
    """Several positions with the biases of the keys or of the values alone:
    dequantize + attention's results, where they count."""
    q, k, v = _inputs(2, 4, 2, 300, 3, 4, 32, F16)
    k, v = (k, (v[0], v[1], None)) if alone == "keys" else ((k[0], k[1], None), v)
    for mask in (None, "causal"):
        out = mq.quantized_sdpa(q, k[0], v[0], k[1], v[1], k[2], v[2], mask=mask)
        want = mq.fallback_sdpa(q, k, v, bits=4, group_size=32, scale=D ** -0.5, mask=mask)
        assert torch.equal(out, want)


@pytest.mark.parametrize("dtype,bits", [(F16, 4), (BF16, 8)])
def test_several_positions_over_few_keys(device, monkeypatch, dtype, bits):
    """The shortest calls run fused too: key ranges within one tile and just
    past it, and positions that outnumber the keys (causal: zero rows)."""
    monkeypatch.setattr(dispatch, "fallback_sdpa", None)
    for B, Hq, Hkv, N, L in ((1, 4, 1, 1, 2), (2, 8, 2, 31, 31), (1, 14, 2, 33, 2), (2, 16, 1, 100, 100), (1, 8, 8, 20, 37),
                             (3, 32, 8, 255, 255)):
        q, k, v = _inputs(B, Hq, Hkv, N, L, bits, 32, dtype)
        out = _check(q, k, v, bits, 32, mask="causal")
        assert not bool(out[:, :, :max(0, L - N)].any())
        _check(q, k, v, bits, 32, kv_start=torch.tensor([0, N // 2, N - 1][:B], device=device))
        _check(q, k, v, bits, 32, mask=torch.rand(B, 1, L, N, device=device) < 0.5)


def test_queries_with_a_gradient(device):
    """Several positions with a gradient of either mode through the queries:
    dequantize + attention's torch operations."""
    q, k, v = _inputs(2, 4, 2, 300, 3, 4, 32, F16)
    call = lambda x: mq.quantized_sdpa(x, k[0], v[0], k[1], v[1], k[2], v[2], mask="causal")  # noqa: E731
    path = lambda x: mq.fallback_sdpa(x, k, v, bits=4, group_size=32, scale=D ** -0.5, mask="causal")  # noqa: E731
    plain, tangent = call(q), torch.randn_like(q)
    grads = []
    for f in (call, path):
        x = q.clone().requires_grad_()
        out = f(x)
        out.backward(tangent)
        grads.append(x.grad)
        with torch.no_grad():
            assert f(x).grad_fn is None
    assert torch.equal(*grads) and float(grads[0].abs().max()) > 0
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(q, tangent)
        got, want = (torch.autograd.forward_ad.unpack_dual(f(dual)) for f in (call, path))
        assert torch.equal(got.tangent, want.tangent)
    assert float((plain.float() - path(q).float()).abs().max()) < 2e-3
