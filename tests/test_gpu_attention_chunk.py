"""The chunk attention kernel (16-bit types, head dims 32, 64 and 128, rows
16-byte aligned) against the general kernel, which the same values take when
their rows lie 8 bytes off, at the edges of its chunks (64 keys, 64 or 128
queries a workgroup) in every mask mode and bias type, and against the formula
in 64 bits.  At head dim 32, windows of 129 to 352 tokens run the tuned kernel
and those of few keys the general one, whatever their alignment: there the
first comparison is of that kernel with itself, and only the formula says more.

Tolerance: the two differ in the maxima that P is taken and rounded against;
each is held to the type's bound against the formula (2e-3 / 1e-2), so to
twice that of each other."""

from __future__ import annotations

import math

import pytest
import torch

import crumpet_amd
from crumpet_amd.fused_attention import fused_swin_attention, fused_swin_attention_shifted
from helpers import TOL

pytestmark = pytest.mark.gpu


def _off(t):
    """The same values with rows 8 bytes past 16-byte alignment."""
    flat = torch.empty(t.numel() + 4, dtype=t.dtype, device=t.device)[4:]
    return flat.view(t.shape).copy_(t)


def _both(call, q, k, v, dtype):
    a = call(q, k, v)
    b = call(_off(q), _off(k), _off(v))
    assert torch.isfinite(a).all()
    assert (a.float() - b.float()).abs().max().item() <= 2 * TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Dh", [32, 64, 128])
@pytest.mark.parametrize("N", [1, 15, 63, 64, 65, 127, 128, 129, 192, 353, 385, 512])
@pytest.mark.parametrize("mask_dtype,bias_dtype", [(None, torch.float32), (torch.float16, torch.bfloat16),
                                                   (torch.float32, torch.float16), (torch.bfloat16, torch.float32)])
def test_edges(dev, dtype, Dh, N, mask_dtype, bias_dtype):
    g = torch.Generator(device="cuda").manual_seed(N + Dh)
    q, k, v = (torch.randn((3, 2, N, Dh), generator=g, device="cuda").to(dtype) for _ in range(3))
    bias = torch.randn((2, N, N), generator=g, device="cuda").to(bias_dtype)
    mask = flags = None
    if mask_dtype is not None:
        mask = torch.where(torch.rand((3, N, N), generator=g, device="cuda") < 0.3, -100.0, 0.0).to(mask_dtype)
        mask[:, :, N // 2] = 0
        flags = torch.tensor([1, 0, 1], dtype=torch.uint8, device="cuda")
    _both(lambda q, k, v: fused_swin_attention(q, k, v, bias, mask, flags), q, k, v, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Dh", [32, 64, 128])
@pytest.mark.parametrize("ws,grid,shift", [((4, 4, 4), (2, 3, 1), (2, 2, 2)), ((3, 5, 4), (2, 2, 2), (1, 0, 2)),
                                           ((8, 8, 8), (1, 2, 2), (4, 4, 4)), ((7, 7, 7), (2, 1, 2), (3, 3, 3))])
def test_regions(dev, dtype, Dh, ws, grid, shift):
    g = torch.Generator(device="cuda").manual_seed(Dh)
    N, nw = ws[0] * ws[1] * ws[2], grid[0] * grid[1] * grid[2]
    dims = tuple(n * w for n, w in zip(grid, ws))
    q, k, v = (torch.randn((2 * nw, 3, N, Dh), generator=g, device="cuda").to(dtype) for _ in range(3))
    bias = torch.randn((3, N, N), generator=g, device="cuda")
    mask = crumpet_amd.compute_attn_mask_3d(*dims, ws, shift, torch.float32, "cuda").repeat(2, 1, 1)
    got = fused_swin_attention_shifted(q, k, v, bias, dims, ws, shift)
    want = fused_swin_attention(_off(q), _off(k), _off(v), bias, mask)
    assert (got.float() - want.float()).abs().max().item() <= 2 * TOL[dtype]


@pytest.mark.parametrize("mask_dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_lowest_and_infinite_masks(dev, mask_dtype):
    """Keys masked by the type's lowest value or -inf, whole chunks of them
    first: they have no part in the result."""
    g = torch.Generator(device="cuda").manual_seed(1)
    N = 200
    q, k, v = (torch.randn((2, 2, N, 64), generator=g, device="cuda").half() for _ in range(3))
    bias = torch.randn((2, N, N), generator=g, device="cuda")
    keep = torch.arange(N, device="cuda") >= 130
    want = torch.softmax((q.double() / 8) @ k.double()[:, :, keep].transpose(-2, -1).contiguous()
                         + bias.double()[:, :, keep], -1) @ v.double()[:, :, keep].contiguous()
    for low in (torch.finfo(mask_dtype).min, float("-inf")):
        mask = torch.zeros((2, N, N), dtype=mask_dtype, device="cuda")
        mask[:, :, ~keep] = low
        got = fused_swin_attention(q, k, v, bias, mask)
        assert (got.double() - want).abs().max().item() <= TOL[torch.float16]


@pytest.mark.parametrize("dtype,u", [(torch.float16, 2.0 ** -11), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("Dh,N", [(32, 400), (32, 512), (64, 343), (128, 343)])
def test_row_sums_of_unrounded_probabilities(dev, dtype, u, Dh, N):
    """One dominant key and equal small ones of a probability that 16 bits
    round by almost u, with values of no weight: the row sum alone decides
    the result, which is then off by its own rounding (u) and a few fp32
    roundings.  A sum of the rounded probabilities would add almost another u."""
    g = torch.Generator(device="cuda").manual_seed(Dh)
    q = torch.zeros((2, 2, N, Dh), device="cuda", dtype=dtype)
    v = torch.zeros_like(q)
    v[:, :, 7] = (1 + torch.rand((2, 2, Dh), generator=g, device="cuda")).to(dtype)
    bias = torch.full((2, N, N), math.log((1 + 0.98 * u) / 8), device="cuda")
    bias[:, :, 7] = 0
    got = fused_swin_attention(q, q, v, bias, None).double()
    want = v[:, :, 7:8].double() / (1 + (N - 1) * bias[0, 0, 0].double().exp())
    assert ((got - want).abs() / want).max().item() <= 1.05 * u


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Dh,N", [(32, 400), (32, 512), (64, 200), (128, 200)])
@pytest.mark.parametrize("mask_dtype,low", [(torch.float32, torch.finfo(torch.float32).min),
                                            (torch.bfloat16, torch.finfo(torch.bfloat16).min),
                                            (torch.float32, -1.5e38)])
def test_rows_masked_wholly_by_a_low_value(dev, dtype, Dh, N, mask_dtype, low):
    """Every key of a row at the lowest value: the scores vanish in it (they do
    not in fp16's, which leaves them 2^-8 steps of fp32) and the result is the mean of v, as of torch.softmax; with keys at -inf beside
    them, the mean of the others; a row all at -inf is NaN."""
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k, v = (torch.randn((1, 2, N, Dh), generator=g, device="cuda").to(dtype) for _ in range(3))
    bias = torch.randn((2, N, N), generator=g, device="cuda")
    mask = torch.zeros((1, N, N), dtype=mask_dtype, device="cuda")
    mask[:, 3] = low
    mask[:, 5] = low
    mask[:, 5, ::3] = float("-inf")
    mask[:, 6, :130] = low
    mask[:, 7, 130:] = low
    mask[:, 8] = float("-inf")
    got = fused_swin_attention(q, k, v, bias, mask).double()
    # the scores in fp32, where they vanish in the mask
    s = ((q.double() * Dh ** -0.5) @ k.double().transpose(-2, -1).contiguous() + bias.double()).float()
    want = torch.softmax((s + mask.float()[:, None]).double(), -1) @ v.double()
    assert torch.isnan(got[:, :, 8]).all()
    rows = torch.arange(N, device="cuda") != 8
    assert (got - want)[:, :, rows].abs().max().item() <= TOL[dtype]


def _formula(q, k, v, bias, mask):
    s = (q.double() * q.shape[-1] ** -0.5) @ k.double().transpose(-2, -1).contiguous() + bias.double()
    return torch.softmax(s if mask is None else s + mask.double()[:, None], -1) @ v.double()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Dh,N", [(32, n) for n in (1, 15, 16, 31, 32, 33, 64, 65, 127, 128, 353, 385, 450, 511, 512,
                                                    576, 640, 700, 729)]
                         + [(d, n) for d in (64, 128) for n in (1, 16, 63, 64, 65, 129, 192, 353)])
def test_few_and_many_keys_against_64_bits(dev, dtype, Dh, N):
    """Both sides of the line below which head dim 32 stays with the general
    kernel (16 keys with a mask tensor, 33 without), and of every chunk."""
    g = torch.Generator(device="cuda").manual_seed(N)
    q, k, v = (torch.randn((4, 2, N, Dh), generator=g, device="cuda").to(dtype) for _ in range(3))
    bias = torch.randn((2, N, N), generator=g, device="cuda")
    mask = torch.where(torch.rand((4, N, N), generator=g, device="cuda") < 0.3, -100.0, 0.0)
    mask[:, :, N // 2] = 0
    assert (fused_swin_attention(q, k, v, bias, None).double() - _formula(q, k, v, bias, None)).abs().max() <= TOL[dtype]
    assert (fused_swin_attention(q, k, v, bias, mask).double() - _formula(q, k, v, bias, mask)).abs().max() <= TOL[dtype]
    dims, ws, shift = (2, 2, N), (1, 1, N), (0, 0, N // 2)
    region = crumpet_amd.compute_attn_mask_3d(*dims, ws, shift, torch.float32, "cuda")
    got = fused_swin_attention_shifted(q, k, v, bias, dims, ws, shift)
    assert (got.double() - _formula(q, k, v, bias, region)).abs().max() <= TOL[dtype]
