"""window_qkv_3d / window_proj_3d where window_rows_kernel runs them (16-bit
types, C a multiple of 32 from 96 to 384): half steps of 64 channels, feature
counts off the 64-feature tile, last tiles of fewer than 32 tokens, padding,
shifts, no LayerNorm, no bias; against the oracle, to 4 units in the last
place (the rounding of the normalised row and of the result, and fp32 sums in
another order)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from crumpet_amd import fused_block

pytestmark = pytest.mark.gpu

ULP = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}
NAME = {torch.float16: "float16", torch.bfloat16: "bfloat16"}


def _check(got, want, dtype):
    got = got.double().cpu().numpy()
    assert got.shape == want.shape
    assert (np.abs(got - want) / np.maximum(np.abs(want), 1.0)).max() <= 4 * ULP[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("C,n_out", [(96, 288), (96, 48), (128, 384), (160, 80), (192, 576), (224, 16), (256, 64),
                                     (288, 864), (320, 112), (384, 1152)])
@pytest.mark.parametrize("dims,ws,ss", [((6, 6, 6), (6, 6, 6), (0, 0, 0)), ((5, 8, 3), (2, 7, 3), (1, 3, 0)),
                                        ((1, 1, 1), (1, 1, 1), (0, 0, 0))])
@pytest.mark.parametrize("x_fp32,bias,normalize", [(True, True, True), (False, False, True), (False, True, False)])
def test_rows(oracle, dev, dtype, C, n_out, dims, ws, ss, x_fp32, bias, normalize):
    g = torch.Generator().manual_seed(C + n_out)
    x = torch.randn((2, *dims, C), generator=g).to(torch.float32 if x_fp32 else dtype)
    w = (torch.randn((n_out, C), generator=g) / C ** 0.5).to(dtype)
    b = torch.randn((n_out,), generator=g).to(dtype) if bias else None
    up = lambda t: None if t is None else t.double().numpy()  # noqa: E731
    on = lambda t: None if t is None else t.to(dev)  # noqa: E731
    if normalize:
        got = fused_block.window_qkv_3d(on(x), on(w), on(b), ws, ss, dtype=dtype)
        want = oracle.window_qkv(up(x), ws, ss, up(w), up(b), dtype=NAME[dtype])
        _check(got, want, dtype)
    else:
        got = fused_block.window_qkv_3d(on(x), on(w), on(b), ws, ss, normalize=False, dtype=dtype)
        pad = [(-d) % s for d, s in zip(dims, ws)]
        xp = torch.nn.functional.pad(x, (0, 0, 0, pad[2], 0, pad[1], 0, pad[0]))
        rows = oracle.shift_partition(xp.double().numpy(), ws, ss)
        _check(got, rows @ up(w).T + (0 if b is None else up(b)), dtype)
    nwin = got.shape[0]
    win = torch.randn((nwin, got.shape[1], C), generator=g).to(dtype)
    y = fused_block.window_proj_3d(on(win), on(w), on(b), 2, *dims, ws, ss)
    _check(y, oracle.window_proj(up(win), 2, *dims, ws, ss, up(w), up(b)), dtype)
