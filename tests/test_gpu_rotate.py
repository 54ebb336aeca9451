"""Rotary positions in one launch (csrc/rotate.hip) against the same in 64 bits."""

import math

import pytest
import torch

from mlx_qsdpa_amd import attention, kernels

pytestmark = pytest.mark.gpu


def _exact(x, start, theta):
    """(value, bound): the float32 angle pos * theta^(-2i/D) is off by at most
    two units of its last place in powf and half a one in its own product
    (|angle| 2^-21 covers them), and by what a unit of the exponent 2i/D <= 1
    makes of theta to it (|angle| ln(theta) 2^-23); sin and cos by another
    2^-21; and the result is rounded to x's type (half a unit, 2^-25 in
    float16's subnormals)."""
    B, H, L, D = x.shape
    pos = start.double()[:, None] + torch.arange(L, dtype=torch.float64)
    ang = (pos[..., None] * theta ** (-torch.arange(0, D, 2, dtype=torch.float64) / D))[:, None].to(x.device)
    x1, x2 = x.double()[..., : D // 2], x.double()[..., D // 2:]
    y = torch.cat([x1 * ang.cos() - x2 * ang.sin(), x2 * ang.cos() + x1 * ang.sin()], -1)
    turn = (x1.abs() + x2.abs()) * (ang.abs() * (2.0 ** -21 + math.log(theta) * 2.0 ** -23) + 2.0 ** -21)
    return y, torch.cat([turn, turn], -1) + y.abs() * (2.0 ** -11 if x.dtype == torch.float16 else 2.0 ** -8) + 2.0 ** -25


# (B, Hq, Hkv, L, D, projected: a transposed view of a linear layer's output)
SHAPES = [(1, 1, 1, 1, 2, True), (2, 16, 4, 1, 128, True), (3, 7, 1, 5, 64, False), (65, 4, 2, 2, 96, True),
          (1, 3, 3, 300, 80, True), (2, 5, 1, 3, 30, False), (1, 2, 1, 2, 1024, True), (130, 2, 2, 1, 256, True)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,Hq,Hkv,L,D,projected", SHAPES)
def test_rotate(device, B, Hq, Hkv, L, D, projected, dtype):
    g = torch.Generator(device="cuda").manual_seed(B + D)
    q, k = ((torch.randn(B, L, h, D, generator=g, device="cuda").to(dtype).transpose(1, 2)) for h in (Hq, Hkv))
    if not projected:
        q, k = q.contiguous(), k.contiguous()
    starts = torch.arange(B) * 97 - 40
    for start in (starts, 4095, torch.tensor([131000])):
        got = kernels.rotate(q, k, start, 10000.0)
        assert got is not None
        s = torch.as_tensor(start).reshape(-1).expand(B)
        for y, x in zip(got, (q, k)):
            assert y.is_contiguous() and y.dtype == dtype
            want, bound = _exact(x, s, 10000.0)
            assert ((y.double() - want).abs() <= bound).all()
    # Rows off the 16-byte grid.
    wide = torch.randn(B, Hq, L, D + 3, generator=g, device="cuda").to(dtype)[..., 1:D + 1]
    got = kernels.rotate(wide, k, starts, 500.0)
    want, bound = _exact(wide, starts, 500.0)
    assert ((got[0].double() - want).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("theta", [10000.0, 500000.0])
@pytest.mark.parametrize("B,Hq,Hkv,L,D", [(2, 16, 4, 1, 128), (1, 3, 1, 700, 64), (3, 8, 2, 5, 256), (2, 4, 4, 9, 96),
                                          (1, 2, 2, 3, 80)])
def test_rotate_gives_the_bits_of_the_expression(device, B, Hq, Hkv, L, D, theta, dtype):
    """Operation for operation the layer's torch expression on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(B + D)
    q, k = ((torch.randn(B, L, h, D, generator=g, device="cuda") * 3).to(dtype).transpose(1, 2) for h in (Hq, Hkv))
    for start in (torch.arange(B) * 1777 + 3, torch.full((B,), 65000)):
        got = kernels.rotate(q, k, start, theta)
        pos = start[:, None] + torch.arange(L)[None, :]
        for y, x in zip(got, (q, k)):
            assert torch.equal(y, attention._rope(x, pos, theta))


def test_other_calls_keep_the_expression(device):
    q, k = torch.randn(2, 4, 3, 64, device="cuda").half(), torch.randn(2, 2, 3, 64, device="cuda").half()
    assert kernels.rotate(q.float(), k.float(), 0, 1e4) is None
    assert kernels.rotate(q, k[:1], 0, 1e4) is None
    assert kernels.rotate(q, k, torch.zeros(3, dtype=torch.int64), 1e4) is None
    assert kernels.rotate(q[..., :63], k[..., :63], 0, 1e4) is None
    g = q.clone().requires_grad_()
    assert kernels.rotate(g, k, 0, 1e4) is None
    a, _ = attention._rotated(g, k, 5, 1e4)
    a.float().sum().backward()
    assert g.grad is not None
    with torch.no_grad():
        b, _ = attention._rotated(g, k, 5, 1e4)
    assert b.grad_fn is None and (a - b).abs().max() <= 2.0 ** -9 * a.abs().max()
