"""The second half of a Swin block (fused_swin_mlp), patch merging and the
feature norm against plain torch in 64 bits, at the edges of their tiles (16
tokens and 16 or 32 features a tile, 32-deep steps shared by four waves), and
the patched encoder against its eager forward.

Tolerances: the results are rounded to the 16-bit type once, and so are the
normalised rows and the hidden layer; with unit-variance rows and weights
scaled by K^-1/2 each adds at most about one rounding (u = 2^-11 or 2^-8) of
the largest value, so 6 u of it bounds their sum."""

from __future__ import annotations

import copy

import pytest
import torch
import torch.nn.functional as F

import crumpet_amd
from crumpet_amd import fused_block, monai_patch
from crumpet_amd import swin_unetr_compat as sw

pytestmark = pytest.mark.gpu

U = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _close(got, want, dtype):
    want = want.double()
    err = (got.double() - want).abs().max().item()
    assert err <= 6 * U[dtype] * want.abs().max().item(), err


def _randn(g, *shape, dtype=torch.float32, std=1.0):
    return (torch.randn(shape, generator=g) * std).to("cuda", dtype)


def _norm(g, c, dtype):
    norm = torch.nn.LayerNorm(c, device="cuda", dtype=dtype).requires_grad_(False)
    norm.weight.copy_(1 + 0.1 * _randn(g, c))
    norm.bias.copy_(0.1 * _randn(g, c))
    return norm


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("c,hidden,rows", [(16, 32, 1), (32, 128, 17), (48, 192, 1000), (64, 256, 15), (80, 320, 33),
                                           (96, 384, 5000), (96, 512, 40), (128, 512, 31), (192, 768, 129),
                                           (384, 1536, 27), (768, 3072, 64), (192, 768, 13824)])
@pytest.mark.parametrize("x_fp32,with_add,bias", [(True, True, True), (False, True, True), (False, False, False)])
def test_swin_mlp(dev, dtype, c, hidden, rows, x_fp32, with_add, bias):
    g = torch.Generator().manual_seed(c + rows)
    xdt = torch.float32 if x_fp32 else dtype
    x = _randn(g, rows, c, dtype=xdt)
    add = _randn(g, rows, c, dtype=dtype) if with_add else None
    norm = _norm(g, c, xdt)
    l1 = (_randn(g, hidden, c, dtype=dtype, std=c ** -0.5), _randn(g, hidden, dtype=dtype, std=0.1) if bias else None)
    l2 = (_randn(g, c, hidden, dtype=dtype, std=hidden ** -0.5), _randn(g, c, dtype=dtype, std=0.1) if bias else None)
    got = fused_block.fused_swin_mlp(x, add, norm, l1, l2, dtype)
    assert got.dtype == xdt and got.shape == x.shape
    x1 = x if add is None else x + add
    a = F.layer_norm(x1.double(), (c,), norm.weight.double(), norm.bias.double(), norm.eps)
    up = lambda t: None if t is None else t.double()  # noqa: E731
    want = x1.double() + F.linear(F.gelu(F.linear(a, up(l1[0]), up(l1[1]))), up(l2[0]), up(l2[1]))
    _close(got, want, dtype)


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_swin_mlp_spreads_what_is_not_finite(dev, value):
    """A row with a value that is not finite is NaN, as in eager; the others stay."""
    g = torch.Generator().manual_seed(0)
    x = _randn(g, 40, 48, dtype=torch.float16)
    x[7, 3] = value
    norm = _norm(g, 48, torch.float16)
    l1 = (_randn(g, 192, 48, dtype=torch.float16, std=0.1), None)
    l2 = (_randn(g, 48, 192, dtype=torch.float16, std=0.1), None)
    got = fused_block.fused_swin_mlp(x, None, norm, l1, l2)
    assert torch.isnan(got[7]).all()
    assert torch.isfinite(got[torch.arange(40, device="cuda") != 7]).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dims,c", [((2, 2, 2), 8), ((5, 3, 4), 24), ((1, 1, 1), 48), ((7, 8, 9), 96), ((6, 6, 6), 384),
                                    ((3, 4, 2), 768)])
@pytest.mark.parametrize("kind", [sw.PatchMerging, sw.PatchMergingV2])
def test_patch_merging(dev, monkeypatch, dtype, dims, c, kind):
    torch.manual_seed(c)
    m = kind(c).to(dev).eval().requires_grad_(False)
    m.norm.weight.uniform_(0.9, 1.1)
    x = torch.randn((2, *dims, c), device=dev).to(dtype)
    want = m.to(torch.float64)(x.double())
    m = m.to(torch.float32)
    calls = []
    monkeypatch.setattr(monai_patch, "patch_merge_3d",
                        lambda *a: calls.append(1) or fused_block.patch_merge_3d(*a))
    with torch.no_grad(), torch.autocast("cuda", dtype=dtype):
        got = monai_patch._downsample(m, x, sw)
    assert calls and got.dtype == dtype and got.shape == want.shape
    _close(got, want, dtype)


@pytest.mark.parametrize("c,rows", [(8, 3), (48, 1000), (96, 65), (192, 17), (768, 100), (1536, 33), (6144, 5)])
@pytest.mark.parametrize("xdt,odt", [(torch.float32, torch.float32), (torch.float16, torch.float32),
                                     (torch.bfloat16, torch.bfloat16)])
def test_channel_norm(dev, c, rows, xdt, odt):
    x = (3 + 2 * torch.randn((rows, c), generator=torch.Generator().manual_seed(c))).to(dev, xdt)
    got = fused_block.channel_norm(x, dtype=odt)
    want = F.layer_norm(x.double(), (c,))
    # fp32: sums of c terms and a division, a few ulps of the largest value
    bound = (1e-6 if odt == torch.float32 else U[odt]) * 2 * want.abs().max().item()
    assert got.dtype == odt and (got.double() - want).abs().max().item() <= bound


def _encoder(dev, **kw):
    torch.manual_seed(0)
    return sw.SwinTransformer(in_chans=1, embed_dim=48, window_size=(7, 7, 7), patch_size=(2, 2, 2),
                              depths=(2, 2, 2, 2), num_heads=(3, 6, 12, 24), **kw).to(dev).eval()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, None])
@pytest.mark.parametrize("downsample", ["merging", "mergingv2"])
def test_patched_encoder(dev, monkeypatch, dtype, downsample):
    """Same shapes, strides and types as the eager encoder, and values no
    further from those of 64 bits than its own (2-norm over a feature, whose
    thousands of roundings differ by a few per cent between two orders of the
    sums; fp32 sums as short as here by more)."""
    m = _encoder(dev, downsample=downsample)
    x = torch.rand((2, 1, 32, 48, 40), device=dev)
    with torch.no_grad():
        exact = copy.deepcopy(m).cpu().double()(x.cpu().double())

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=dtype or torch.float16, enabled=dtype is not None):
            return m(x)

    fused = []
    for name in ("fused_swin_mlp", "patch_merge_3d"):
        monkeypatch.setattr(monai_patch, name, lambda *a, f=getattr(fused_block, name): fused.append(1) or f(*a))
    want = run()
    crumpet_amd.patch_monai_swin_unetr()
    try:
        got = run()
        assert len(fused) == (0 if dtype is None else 12)  # eight blocks, four mergings
    finally:
        crumpet_amd.unpatch_monai_swin_unetr()
    bound = 1e-4 if dtype is None else 64 * U[dtype]
    for a, b, e in zip(got, want, exact):
        assert a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype
        assert (a - b).abs().max().item() <= bound * b.abs().max().item()
        off = [((t.double().cpu() - e).norm() / e.norm()).item() for t in (a, b)]
        print(dtype, downsample, off)
        assert off[0] <= (1.5 if dtype is None else 1.1) * off[1], off


def test_patched_block_keeps_gradients_hooks_and_training(dev, monkeypatch):
    """Where more than the values is wanted the eager second half runs."""
    def fail(*a, **k):
        raise AssertionError("fused second half")

    monkeypatch.setattr(monai_patch, "fused_swin_mlp", fail)
    block = sw.SwinTransformerBlock(48, 3, (4, 4, 4), (0, 0, 0)).to(dev).eval()
    x = torch.randn((1, 8, 8, 8, 48), device=dev)
    crumpet_amd.patch_monai_swin_unetr()
    try:
        with torch.autocast("cuda", dtype=torch.float16):
            block(x, None).float().sum().backward()
            assert block.mlp.linear1.weight.grad is not None
            with torch.no_grad():
                seen = []
                handle = block.mlp.register_forward_hook(lambda *a: seen.append(1))
                block(x, None)
                handle.remove()
                assert seen
                block.mlp.drop1.train()
                block(x, None)
                block.mlp.drop1.eval()
                monkeypatch.setenv("CRUMPET_DISABLE_FUSED_BLOCK", "1")
                block(x, None)
    finally:
        crumpet_amd.unpatch_monai_swin_unetr()


def _patched(run):
    crumpet_amd.patch_monai_swin_unetr()
    try:
        return run()
    finally:
        crumpet_amd.unpatch_monai_swin_unetr()


def test_second_half_and_merging_follow_their_weights(dev):
    """Every pass uses the Linears' weights as they are then: after a write
    through .data (which moves no version counter), and with parameters that
    a call swaps in (whose storage may be one that an earlier call freed)."""
    torch.manual_seed(0)
    layer = sw.BasicLayer(48, 1, 3, (4, 4, 4), 0.0, downsample=sw.PatchMerging).to(dev).eval().requires_grad_(False)
    mlp, red = layer.blocks[0].mlp, layer.downsample.reduction
    x = torch.randn((1, 48, 8, 8, 8), device=dev)

    def both(swap=None):
        def run():
            with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16, cache_enabled=False):
                return layer(x) if swap is None else torch.func.functional_call(layer, swap(), (x,))
        return _patched(run), run()

    def agree(got, want):
        # four roundings to 16 bits on the way to the merged values, at most
        # doubled by the norm between them
        assert (got - want).abs().max().item() <= 8 * U[torch.float16] * want.abs().max().item()

    agree(*both())
    mlp.linear2.weight.data.mul_(3)
    mlp.linear1.bias.data.add_(0.5)
    agree(*both())
    red.weight.data.copy_(red.weight.flip(0))
    agree(*both())
    names = [n for n, _ in layer.named_parameters() if "mlp" in n or "reduction" in n]
    for i in range(6):
        start = {n: p.clone() for n, p in layer.named_parameters() if n in names}
        agree(*both(lambda: {n: p * (1 + 0.2 * i) for n, p in start.items()}))


@pytest.mark.parametrize("c", [48, 96, 192])  # one kernel, one with more than 64 KB of LDS, three kernels
def test_captured_second_half_reads_the_weights_at_replay(dev, c):
    torch.manual_seed(0)
    block = sw.SwinTransformerBlock(c, c // 16, (4, 4, 4), (0, 0, 0)).to(dev).eval().requires_grad_(False)
    x = torch.randn((1, 8, 8, 8, c), device=dev)

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16, cache_enabled=False):
            return block(x, None)

    def check():
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            run()
        torch.cuda.current_stream().wait_stream(s)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = run()
        for scale in (1.0, 2.0, 0.5, 1.0):
            block.mlp.linear2.weight.data.mul_(scale)
            torch.randn(1 << 20, device=dev).sum().item()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, run())

    _patched(check)


def test_jit_trace_keeps_the_modules_parameters(dev):
    """A trace of a patched block records the second half with the module's
    parameters, not with 16-bit copies of their values at that time."""
    torch.manual_seed(0)
    block = sw.SwinTransformerBlock(48, 3, (4, 4, 4), (0, 0, 0)).to(dev).eval().requires_grad_(False)
    x = torch.randn((1, 8, 8, 8, 48), device=dev)

    class Alone(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.block = block

        def forward(self, x):
            return self.block(x, None)

    def check():
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16, cache_enabled=False):
            block(x, None)  # a pass before the trace may have kept such copies
            traced = torch.jit.trace(Alone(), (x,), check_trace=False)
            block.mlp.linear2.weight.mul_(3)
            got, want = traced(x), block(x, None)
        assert (got - want).abs().max().item() <= 6 * U[torch.float16] * want.abs().max().item()

    _patched(check)


def test_channel_norm_over_more_rows_than_one_row_of_workgroups(dev):
    """64 rows a workgroup and 2^20 workgroups along x: rows past 2^26."""
    rows, c = (1 << 26) + 100, 8
    x = torch.zeros((rows, c), device=dev, dtype=torch.float16)
    parts = [slice(0, 1000), slice((1 << 26) - 1000, rows)]
    for part in parts:
        x[part] = torch.randn(x[part].shape, device=dev, dtype=torch.float16)
    got = fused_block.channel_norm(x)
    for part in parts:
        want = F.layer_norm(x[part].double(), (c,))
        assert (got[part].double() - want).abs().max().item() <= 2 * U[torch.float16] * want.abs().max().item()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("c,hidden", [(16, 32), (48, 192), (96, 384), (384, 1536)])
@pytest.mark.parametrize("form", ["contiguous", "transposed", "4 bytes off", "one converted already"])
def test_weights_converted_by_the_op(dev, dtype, c, hidden, form):
    """The op's conversion of fp32 parameters against torch's, bit for bit,
    through the results of the same kernels."""
    g = torch.Generator().manual_seed(c)
    x = _randn(g, 50, c)
    norm = _norm(g, c, torch.float32)
    w1, b1 = _randn(g, hidden, c, std=c ** -0.5), _randn(g, hidden, std=0.1)
    w2, b2 = _randn(g, c, hidden, std=hidden ** -0.5), _randn(g, c, std=0.1)
    u = U[dtype]
    w1[0, :4] = torch.tensor([1 + u, 1 + 3 * u, -1e-7, 6.1e-5], device=dev)  # ties, fp16's smallest
    if form == "transposed":
        w1 = w1.t().contiguous().t()
    elif form == "4 bytes off":
        w2, b1 = (torch.empty(t.numel() + 1, device=dev)[1:].view(t.shape).copy_(t) for t in (w2, b1))
    elif form == "one converted already":
        w2 = w2.to(dtype)
    got = fused_block.fused_swin_mlp(x, None, norm, (w1, b1), (w2, b2), dtype)
    cast = [t.to(dtype).contiguous() for t in (w1, b1, w2, b2)]
    want = fused_block.fused_swin_mlp(x, None, norm, cast[:2], cast[2:], dtype)
    assert torch.isfinite(want).all() and torch.equal(got, want)
