"""What the patched attention half keeps of its parameters, used from another
stream than the one that made it: the values are waited for, and their memory
is not handed out again while that stream may still read it."""

from __future__ import annotations

import pytest
import torch

from crumpet_amd import monai_patch
from crumpet_amd import swin_unetr_compat as sw

pytestmark = pytest.mark.gpu


def _params(attn):
    bias, (wq, bq), (wp, bp) = monai_patch._block_params(attn, 343, torch.float16)
    return [t.clone() for t in (bias, wq, bq, wp, bp)]


def test_another_stream_waits_for_kept_parameters(dev):
    torch.manual_seed(0)
    attn = sw.WindowAttention(384, 24, (7, 7, 7), qkv_bias=True).to(dev).requires_grad_(False)
    want = _params(attn)
    monai_patch.forget_cached_params(attn)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        torch.cuda._sleep(20_000_000)  # some ms of work before the values are made
        _params(attn)
    with torch.cuda.stream(second):
        got = _params(attn)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_replaced_parameters_outlive_the_streams_that_read_them(dev):
    torch.manual_seed(0)
    attn = sw.WindowAttention(384, 24, (7, 7, 7), qkv_bias=True).to(dev).requires_grad_(False)
    want = _params(attn)
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(other):
        kept = monai_patch._block_params(attn, 343, torch.float16)
        torch.cuda._sleep(20_000_000)
        got = [t.clone() for t in monai_patch._tensors(kept)]
    del kept
    monai_patch.forget_cached_params(attn)
    # the freed blocks, were they free, would be the next ones of these sizes
    fill = [torch.full_like(t, 7.0) for t in want for _ in range(2)]
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want)) and len(fill) == 10
