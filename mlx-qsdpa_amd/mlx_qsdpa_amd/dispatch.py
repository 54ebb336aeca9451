"""quantized_sdpa: validation and routing onto the HIP decode kernels.

Mirrors mlx_qsdpa/dispatch.py:8-111 (same signature, same ValueError set,
same defaults for ``scale`` and for missing biases), with four MI355X
choices:

* Masked decode runs in-kernel (bool keep-mask or additive mask), where the
  reference falls back to dequantize + SDPA (dispatch.py:68-83).
* ``threshold`` keeps its meaning when given (N <= threshold: single pass,
  else split-K); the default ``None`` lets the library pick the split count
  for 256 CUs.
* ``kv_start`` (extension) skips keys before a per-sequence start index, the
  left padding of a batched cache, without reading them.

* Several query positions (qL > 1: speculative or chunked decoding,
  prefill) run on the fused matrix-core kernel, including mask="causal"
  (aligned to the last key), where the reference dequantizes and runs SDPA.
  Shapes that kernel does not take (unaligned views; at D = 64 additive
  masks and gradients) keep the reference's path: HIP dequantize, then
  float32 attention with torch on the GPU (dispatch.py:68-83).

Head dims the library does not compile (any other multiple of 32, e.g. 32
or 512, which the reference's validation accepts: dispatch.py:48-49) take
that same dequantize + attention path at every qL.
"""

from __future__ import annotations

import torch
from torch.autograd import forward_ad

from . import _lib, kernels


def _validate(q, packed_k, packed_v, bits, group_size):
    """dispatch.py:42-65."""
    if q.dim() != 4:
        raise ValueError(f"q must be 4D (B, H_q, qL, D), got ndim={q.dim()}")
    B, H_q, qL, D = q.shape
    if bits not in (4, 8):
        raise ValueError(f"bits must be 4 or 8, got {bits}")
    if D % 32 != 0:
        raise ValueError(f"D must be multiple of 32, got {D}")
    elems_per_int = 32 // bits
    pack_D = D // elems_per_int
    if packed_k.dim() != 4 or packed_v.dim() != 4:
        raise ValueError("packed_k and packed_v must be 4D (B, H_kv, N, pack_D)")
    _, H_kv, N, actual_pack_D = packed_k.shape
    if actual_pack_D != pack_D:
        raise ValueError(
            f"packed_k last dim {actual_pack_D} != expected pack_D={pack_D} "
            f"for bits={bits}, D={D}")
    if H_q % H_kv != 0:
        raise ValueError(f"H_q ({H_q}) must be divisible by H_kv ({H_kv})")
    return B, H_q, qL, D, H_kv, N


def attention_fp32(q, k, v, scale, mask=None, kv_start=None):
    """float32 SDPA on the GPU with MLX mask conventions.

    q [B,Hq,L,D], k/v [B,Hkv,N,D] (dequantized T), grouped-query heads.
    Bool masks keep True, float masks are added, "causal" is lower-right
    aligned; keys before kv_start[b] are skipped; rows with every key masked
    return 0.  Output has q's dtype.
    """
    B, Hq, L, D = q.shape
    Hkv, N = k.shape[1], k.shape[2]
    G = Hq // Hkv
    qf = q.float().reshape(B, Hkv, G * L, D)
    kt = k.float().transpose(-1, -2).contiguous()
    s = torch.matmul(qf, kt).reshape(B, Hq, L, N) * float(scale)
    cols = torch.arange(N, device=q.device)
    if isinstance(mask, str):
        if mask != "causal":
            raise ValueError(f"unknown mask {mask!r}")
        rows = torch.arange(L, device=q.device)[:, None] + (N - L)
        s = s.masked_fill(cols[None, :] > rows, float("-inf"))
    elif mask is not None:
        m = mask.to(q.device)
        s = s.masked_fill(~m, float("-inf")) if m.dtype == torch.bool else s + m.float()
    if kv_start is not None:
        ks = kv_start.to(q.device, torch.int64)
        s = s.masked_fill(cols[None, None, None, :] < ks[:, None, None, None], float("-inf"))
    p = torch.nan_to_num(torch.softmax(s, dim=-1), nan=0.0)
    o = torch.matmul(p.reshape(B, Hkv, G * L, N), v.float().contiguous())
    return o.reshape(B, Hq, L, D).to(q.dtype)


def dequantize_attention(q, k_quant, v_quant, *, bits, group_size, scale, mask, kv_start=None):
    """The reference's dequantize + SDPA path (dispatch.py:68-83)."""
    k = kernels.dequantize(*k_quant, group_size=group_size, bits=bits)
    v = kernels.dequantize(*v_quant, group_size=group_size, bits=bits)
    return attention_fp32(q, k, v, scale, mask, kv_start)


def fallback_sdpa(q, k_quant, v_quant, *, bits, group_size, scale, mask=None, kv_start=None):
    """Dequantize (HIP) + float32 attention: the path of dispatch.py:68-83.

    Missing biases are zeros (dispatch.py:71, 76); keys before kv_start[b]
    are masked.
    """
    kb = k_quant[2] if k_quant[2] is not None else torch.zeros_like(k_quant[1])
    vb = v_quant[2] if v_quant[2] is not None else torch.zeros_like(v_quant[1])
    return dequantize_attention(q, (k_quant[0], k_quant[1], kb), (v_quant[0], v_quant[1], vb),
                                bits=bits, group_size=group_size, scale=scale, mask=mask,
                                kv_start=kv_start)


def quantized_sdpa(
    q,
    packed_k,
    packed_v,
    k_scales,
    v_scales,
    k_biases=None,
    v_biases=None,
    scale=None,
    mask=None,
    bits=4,
    group_size=32,
    threshold=None,
    *,
    kv_start=None,
    num_splits=None,
):
    """Quantized scaled dot-product attention for decode (qL = 1).

    Args (as mlx_qsdpa.quantized_sdpa, dispatch.py:22-40):
        q:          (B, H_q, qL, D) float16/bfloat16
        packed_k/v: (B, H_kv, N, D*bits/32) uint32
        k/v_scales: (B, H_kv, N, D/group_size) q.dtype
        k/v_biases: same shape, or None for the symmetric format
        scale:      softmax scale (default D**-0.5)
        mask:       None, bool keep-mask or additive mask broadcastable to
                    (B, H_q, 1, N); "causal" (no-op for qL = 1)
        bits:       4 or 8;  group_size: 32, 64 or 128
        threshold:  N <= threshold -> single pass, else split-K;
                    None -> choose for the GPU
        kv_start:   optional (B,) int tensor: keys before it are ignored
        num_splits: optional explicit split count (overrides threshold)
    Returns (B, H_q, qL, D) in q's dtype.
    """
    # Calls whose tensors need no conversion go straight to the native host
    # path, which checks them itself; what it does not take comes back here.
    masked = isinstance(mask, torch.Tensor)
    if (mask is None or (masked and mask.is_cuda) or (isinstance(mask, str) and mask == "causal")) \
            and threshold is None and num_splits is None and q.dim() == 4 and q.shape[3] in kernels.HEAD_DIMS:
        several = q.shape[2] > 1
        both = k_biases is not None and v_biases is not None
        if not several or q.shape[3] != 64 or (packed_k.dim() == 4 and _d64_in_kernel(
                q, packed_k.shape[2], mask, kv_start, k_biases, v_biases)):
            out = kernels.decode_native(q, packed_k, packed_v, k_scales, v_scales, k_biases if both else None,
                                        v_biases if both else None,
                                        scale=q.shape[3] ** -0.5 if scale is None else scale, bits=bits,
                                        group_size=group_size, kv_start=kv_start,
                                        causal=several and mask is not None and not masked,
                                        mask=mask if masked else None)
            if out is not None:
                return out
    B, H_q, qL, D, H_kv, N = _validate(q, packed_k, packed_v, bits, group_size)
    if scale is None:
        scale = D ** -0.5                                          # dispatch.py:86-87
    # The kernels read packed rows in 16-byte pieces; a view whose rows are
    # not 16-byte aligned is copied first, as the reference's kernel builder
    # copies every input (ensure_row_contiguous, kernels.py:190).
    packed_k, packed_v = _row_aligned(packed_k), _row_aligned(packed_v)
    # A mask made on the host (as a cache's make_mask may make it) goes to
    # the device in stream order, without waiting.
    if isinstance(mask, torch.Tensor) and q.device.type == "cuda":
        mask = kernels.to_device(mask, q.device)
    if isinstance(kv_start, torch.Tensor) and q.device.type == "cuda":
        kv_start = kernels.to_device(kv_start, q.device)

    if D not in kernels.HEAD_DIMS or (qL > 1 and not (
            (D != 64 or _d64_in_kernel(q, N, mask, kv_start, k_biases, v_biases))
            and _fused_takes(q, packed_k, packed_v, k_scales, v_scales, k_biases, v_biases, scale, bits,
                             group_size))):
        return fallback_sdpa(q, (packed_k, k_scales, k_biases),    # dispatch.py:68-83
                             (packed_v, v_scales, v_biases), bits=bits, group_size=group_size,
                             scale=scale, mask=mask, kv_start=kv_start)

    has_biases = k_biases is not None and v_biases is not None     # dispatch.py:89-94
    if not has_biases:
        k_biases = v_biases = None
    causal = False
    if isinstance(mask, str):
        if mask != "causal":
            raise ValueError(f"unknown mask {mask!r}")
        causal = qL > 1                                            # qL == 1: sees every key
        mask = None

    if num_splits is None:
        if threshold is None:
            num_splits = 0
        elif N <= threshold:                                       # dispatch.py:98
            num_splits = 1
        else:
            auto, _ = kernels.decode_plan(q, packed_k, packed_v, k_scales, v_scales, k_biases,
                                          v_biases, scale=scale, bits=bits,
                                          group_size=group_size)
            num_splits = max(2, auto)
    return kernels.decode(q, packed_k, packed_v, k_scales, v_scales, k_biases, v_biases,
                          scale=scale, bits=bits, group_size=group_size, mask=mask,
                          kv_start=kv_start, num_splits=num_splits, causal=causal)


def _row_aligned(t):
    """`t` itself if its rows start on 16-byte boundaries, else a contiguous copy."""
    if t.data_ptr() % 16 == 0 and all(st % 4 == 0 for st in t.stride()[:3]) and t.stride(-1) == 1:
        return t
    return t.contiguous()


def _d64_in_kernel(q, N, mask, kv_start, k_biases, v_biases):
    """Whether several positions at D = 64 run fused: biases of both or of
    neither (one alone counts there, and not in the kernel), and masked as the
    dequantize + attention path masks them ("causal" or a bool mask over all
    keys, one start per sequence).  Fused they are the faster ones at every
    size: 8 to 26 us a call against 172 to 242 on that path for 2 to 255
    positions over 2 to 255 keys (1 to 8 sequences, 8 / 2 to 32 / 8 heads), 44
    against 878 at 1500 of each.  The path's other masks stay on it: additive ones (a row whose every score is the type's lowest value
    averages V there and is empty in the kernel, which scales the mask to
    base 2), masks that broadcast over the keys.  So do calls whose queries
    carry a gradient, which goes through its torch operations."""
    B, H_q, qL, _ = q.shape
    if N < 1 or (k_biases is None) != (v_biases is None) or _differentiated(q):
        return False
    if kv_start is not None and tuple(kv_start.shape) != (B,):
        return False
    if not isinstance(mask, torch.Tensor):
        return True
    if mask.dtype != torch.bool or not 1 <= mask.dim() <= 4:
        return False
    shape = (1,) * (4 - mask.dim()) + tuple(mask.shape)
    return shape[3] == N and shape[2] in (1, qL) and shape[1] in (1, H_q) and shape[0] in (1, B)


def _differentiated(q):
    """Whether a gradient, of either mode, is taken through q."""
    return (q.requires_grad and torch.is_grad_enabled()) \
        or (forward_ad._current_level >= 0 and forward_ad.unpack_dual(q).tangent is not None)


def _fused_takes(q, packed_k, packed_v, k_scales, v_scales, k_biases, v_biases, scale, bits,
                 group_size):
    """Whether the fused kernel takes several query positions for these
    inputs (the matrix-core path: D 64, 128 or 256, aligned views).  Extension:
    the reference sends every qL > 1 call to dequantize + attention."""
    if k_biases is None or v_biases is None:
        k_biases = v_biases = None
    try:
        kernels.decode_plan(q, packed_k, packed_v, k_scales, v_scales, k_biases, v_biases,
                            scale=scale, bits=bits, group_size=group_size)
    except _lib.QsdpaError as e:
        if e.code == _lib.QSDPA_ERR_UNSUPPORTED:
            return False
        raise
    return True
