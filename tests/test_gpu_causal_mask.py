"""The causal mask in one launch (csrc/causal_mask.hip) against the torch
expression on the CPU: whole values, so equal."""

import pytest
import torch

from mlx_qsdpa_amd import cache, kernels

pytestmark = pytest.mark.gpu


def _vectors(B, g):
    off = torch.randint(-20, 90, (B,), generator=g)
    off[0] = 90
    return off, torch.randint(0, 40, (B,), generator=g)


# Rows shorter than a 16-byte piece, rows off its grid, a mask that ends
# inside one, more sequences than one launch takes.
@pytest.mark.parametrize("B,N", [(1, 1), (2, 3), (3, 33), (65, 7), (129, 2), (4, 512)])
@pytest.mark.parametrize("window", [None, 1, 17, 5000])
@pytest.mark.parametrize("padded", [False, True])
def test_batched(device, B, N, window, padded):
    off, pad = _vectors(B, torch.Generator().manual_seed(B * N))
    pad = pad if padded else None
    got = kernels.causal_mask(N, off, pad, window, device)
    want = cache._create_causal_mask(N, off, window_size=window, left_padding=pad)
    assert got.dtype == torch.bool and got.shape == want.shape and got.is_contiguous()
    assert torch.equal(got.cpu(), want)
    assert torch.equal(cache._create_causal_mask(N, off, window, pad, device).cpu(), want)


@pytest.mark.parametrize("offset,N", [(0, 1), (0, 5), (3, 2), (100, 33), (1000, 500)])
@pytest.mark.parametrize("window", [None, 0, 9, 10**12])
def test_one_offset(device, offset, N, window):
    got = cache._create_causal_mask(N, offset, window_size=window, device=device)
    assert torch.equal(got.cpu(), cache._create_causal_mask(N, offset, window_size=window))


def test_what_it_does_not_take(device):
    off = torch.tensor([5, 3])
    assert kernels.causal_mask(0, off, None, None, device) is None
    assert kernels.causal_mask(2, off - 50, None, None, device) is None
    assert kernels.causal_mask(2, off, torch.tensor([1]), None, device) is None
    assert kernels.causal_mask(2, off + 2**33, None, None, device) is None
    assert kernels.causal_mask(2, off, None, 1.5, device) is None
