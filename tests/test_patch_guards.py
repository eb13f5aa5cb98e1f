"""When the patched encoder leaves its fused second half, patch merging and
channels-last chain for the eager modules (no GPU needed to decide that)."""

from __future__ import annotations

import copy
import pickle

import pytest
import torch
import torch.utils.flop_counter

import crumpet_amd
from crumpet_amd import monai_patch
from crumpet_amd import swin_unetr_compat as sw


def test_a_forward_set_on_the_module_is_called():
    linear = torch.nn.Linear(4, 4)
    assert monai_patch._unhooked(linear)
    linear.forward = lambda x: x
    assert not monai_patch._unhooked(linear)


@pytest.mark.parametrize("offset,takes", [(0, True), (8, True), (1, False), (4, False)])
@pytest.mark.parametrize("which", ["input", "parameter"])
def test_storage_off_the_16_byte_grid_stays_eager(offset, takes, which):
    flat = torch.zeros(128, dtype=torch.float16)
    part, whole = flat[offset:offset + 48], torch.zeros(48, dtype=torch.float16)
    x, p = (part, whole) if which == "input" else (whole, part)
    assert (monai_patch._half_compute(x, [p]) is torch.float16) == takes


@pytest.mark.parametrize("device", ["cpu", "meta"])
def test_other_devices_are_turned_away_before_the_block_is_looked_at(device):
    x = torch.empty((1, 2, 2, 2, 48), dtype=torch.float16, device=device)
    assert monai_patch._tail_dtype(object(), x) is None


def _fused(monkeypatch, block, c=32):
    """Whether the block's second half would run fused on a 16-bit volume;
    the checks that need a HIP device are answered in its place."""
    monkeypatch.setattr(monai_patch, "_computes_half", lambda x: True)
    monkeypatch.setattr(monai_patch, "_values_only", lambda x, params: True)
    return monai_patch._tail_dtype(block, torch.zeros((1, 4, 4, 4, c), dtype=torch.float16)) is torch.float16


def _block(cls=sw.SwinTransformerBlock, c=32):
    return cls(c, c // 16, (4, 4, 4), (0, 0, 0)).half().eval().requires_grad_(False)


class _OwnSecondHalf(sw.SwinTransformerBlock):
    def forward_part2(self, x):
        return x * 0


class _OwnFirstHalf(sw.SwinTransformerBlock):
    def forward_part1(self, x, mask_matrix):
        return x * 0


def test_a_second_half_of_the_programs_own_is_called(monkeypatch):
    assert _fused(monkeypatch, _block())
    assert _fused(monkeypatch, _block(_OwnFirstHalf))  # called either way
    assert not _fused(monkeypatch, _block(_OwnSecondHalf))
    block = _block()
    block.forward_part2 = lambda x: x * 0
    assert not _fused(monkeypatch, block)
    stock = sw.SwinTransformerBlock.forward_part2
    monkeypatch.setattr(sw.SwinTransformerBlock, "forward_part2", lambda self, x: stock(self, x) * 0)
    assert not _fused(monkeypatch, _block())


def test_a_block_forward_put_in_place_before_the_patch_stays(monkeypatch):
    calls = []
    monkeypatch.setattr(sw.SwinTransformerBlock, "forward", lambda self, x, mask: calls.append(1) or x)
    monkeypatch.setattr(monai_patch, "_tail_dtype", lambda *a: pytest.fail("fused second half"))
    crumpet_amd.patch_monai_swin_unetr()
    try:
        _block()(torch.zeros((1, 4, 4, 4, 32), dtype=torch.float16), None)
    finally:
        crumpet_amd.unpatch_monai_swin_unetr()
    assert calls


class _Scale(torch.nn.Identity):
    def forward(self, x):
        return 2 * x


def _like_named(cls):
    """Another class of the same name and attributes that computes something else."""
    return type(cls.__name__, (cls,), {"forward": lambda self, x: x * 0})


def test_modules_are_known_by_their_class_not_its_name(monkeypatch):
    block = _block()
    block.mlp.__class__ = _like_named(sw.MLPBlock)
    assert type(block.mlp).__name__ == "MLPBlock" and not _fused(monkeypatch, block)
    block = _block()
    monkeypatch.setattr(sw.MLPBlock, "forward", lambda self, x: x * 0)
    assert not _fused(monkeypatch, block)
    monkeypatch.undo()
    block.drop_path = _Scale()
    assert not _fused(monkeypatch, block)
    block.drop_path = type("DropPath", (torch.nn.Module,), {"forward": lambda self, x: x * 0})().eval()
    assert not _fused(monkeypatch, block)
    monkeypatch.setattr(sw, "DropPath", _OwnDropPath, raising=False)
    block.drop_path = _OwnDropPath().eval()
    assert _fused(monkeypatch, block)
    assert not _fused(monkeypatch, block.train())


class _OwnDropPath(torch.nn.Module):
    def forward(self, x):
        return x


def _encoder():
    return sw.SwinTransformer(in_chans=1, embed_dim=32, window_size=(4, 4, 4), patch_size=(2, 2, 2), depths=(1, 1),
                              num_heads=(2, 4)).eval().requires_grad_(False)


def _chained(monkeypatch, model):
    monkeypatch.setattr(monai_patch, "_values_only", lambda x, params: True)
    return monai_patch._channels_last_chain(model, torch.zeros((1, 1, 16, 16, 16)), True, sw)


class _Embed(torch.nn.Module):
    """A patch embedding of a program's own: any width, no attributes."""

    def __init__(self, width):
        super().__init__()
        self.width = width

    def forward(self, x):
        return torch.nn.functional.avg_pool3d(x, 2).expand(-1, self.width, -1, -1, -1)


def test_a_patch_embedding_of_the_programs_own(monkeypatch):
    crumpet_amd.patch_monai_swin_unetr()
    try:
        model = _encoder()
        model.patch_embed = _Embed(32)
        assert _chained(monkeypatch, model)
        # widths that the norm kernel does not take go through F.layer_norm
        x = torch.randn((1, 2, 3, 4, 30))
        want = torch.nn.functional.layer_norm(x, (30,)).permute(0, 4, 1, 2, 3)
        got = monai_patch._feature(x)
        assert torch.equal(got, want) and got.stride() == want.stride()
    finally:
        crumpet_amd.unpatch_monai_swin_unetr()


def test_encoder_steps_of_the_programs_own_are_called(monkeypatch):
    crumpet_amd.patch_monai_swin_unetr()
    try:
        assert _chained(monkeypatch, _encoder())
        with monkeypatch.context() as m:
            m.setattr(sw.SwinTransformer, "proj_out", staticmethod(lambda x, normalize=False: x))
            assert not _chained(m, _encoder())
        with monkeypatch.context() as m:
            m.setattr(sw.BasicLayer, "forward", lambda self, x: x)
            assert not _chained(m, _encoder())
        with monkeypatch.context() as m:
            m.setattr(sw.PatchMerging, "forward", lambda self, x: "called")
            m.setattr(monai_patch, "_computes_half", lambda x: True)
            x = torch.zeros((1, 4, 4, 4, 32), dtype=torch.float16)
            assert monai_patch._downsample(sw.PatchMerging(32).half().eval(), x, sw) == "called"
    finally:
        crumpet_amd.unpatch_monai_swin_unetr()


def test_an_encoder_forward_put_in_place_before_the_patch_stays(monkeypatch):
    calls = []
    monkeypatch.setattr(sw.SwinTransformer, "forward", lambda self, x, normalize=True: calls.append(1))
    monkeypatch.setattr(monai_patch, "_channels_last_chain", lambda *a: True)
    crumpet_amd.patch_monai_swin_unetr()
    try:
        _encoder()(torch.zeros((1, 1, 16, 16, 16)))
    finally:
        crumpet_amd.unpatch_monai_swin_unetr()
    assert calls


def test_what_follows_the_ops_sees_the_modules():
    seen = []

    def look(x):
        seen.append(monai_patch._watched())
        return x * 2

    x = torch.ones(3)
    look(x)
    torch.jit.trace(look, (x,), check_trace=False)
    torch.func.vmap(look)(x)
    with torch.autograd.forward_ad.dual_level():
        look(x)
    with torch.utils.flop_counter.FlopCounterMode(display=False):
        look(x)
    assert seen == [False, True, True, True, True]


@pytest.mark.parametrize("change", ["bias type", "weight strides"])
def test_norm_parameters_that_the_kernels_do_not_take(monkeypatch, change):
    """Eager LayerNorm under autocast takes both."""
    monkeypatch.setattr(torch, "is_autocast_enabled", lambda *a: True)
    monkeypatch.setattr(torch, "get_autocast_dtype", lambda *a: torch.float16)

    def spoil(norm):
        if change == "bias type":
            norm.bias = torch.nn.Parameter(norm.bias.float(), requires_grad=False)
        else:
            norm.weight = torch.nn.Parameter(norm.weight.repeat_interleave(2)[::2], requires_grad=False)

    block = _block()
    assert _fused(monkeypatch, block)
    spoil(block.norm2)
    assert not _fused(monkeypatch, block)

    def called(self, x):
        return "called"

    merge = sw.PatchMerging(32).half().eval().requires_grad_(False)
    monkeypatch.setattr(monai_patch, "patch_merge_3d", lambda *a: "fused")
    x = torch.zeros((1, 4, 4, 4, 32), dtype=torch.float16)
    assert monai_patch._downsample(merge, x, sw) == "fused"
    spoil(merge.norm)
    monkeypatch.setattr(sw.PatchMerging, "__call__", called)
    assert monai_patch._downsample(merge, x, sw) == "called"


class _Weight(torch.Tensor):
    pass


def test_weights_of_a_tensor_subclass_keep_their_ops():
    x = torch.zeros(8, dtype=torch.float16)
    assert monai_patch._half_compute(x, [x.clone(), torch.nn.Parameter(x.clone())]) is torch.float16
    assert monai_patch._half_compute(x, [torch.nn.Parameter(x.clone().as_subclass(_Weight))]) is None


@pytest.mark.parametrize("form", ["gradient", "broadcast", "unaligned"])
def test_the_first_half_may_need_the_eager_second(monkeypatch, form):
    """Parameters of the attention half that train in eval mode beside a
    frozen MLP keep their gradients; other forms of its result are added as
    eager adds them."""
    def first_half(self, x, mask_matrix):
        if form == "gradient":
            return x * torch.ones(32, dtype=torch.float16, requires_grad=True)
        if form == "broadcast":
            return x[..., :1]
        flat = torch.empty(x.numel() + 1, dtype=x.dtype)
        return flat[1:].view(x.shape).copy_(x)

    monkeypatch.setattr(monai_patch, "_tail_dtype", lambda *a: torch.float16)
    monkeypatch.setattr(monai_patch, "fused_swin_mlp", lambda *a: pytest.fail("fused second half"))
    crumpet_amd.patch_monai_swin_unetr()
    try:
        block = _block(type("Block", (sw.SwinTransformerBlock,), {"forward_part1": first_half}))
        y = block(torch.randn((1, 2, 2, 2, 32)).half(), None)
        assert y.shape == (1, 2, 2, 2, 32) and y.requires_grad == (form == "gradient")
    finally:
        crumpet_amd.unpatch_monai_swin_unetr()


def test_kept_parameters_are_not_known_by_a_reused_address():
    """Parameters that every call swaps in start at version 0, and without
    a hold on the last ones' storage land on the address that they left."""
    attn = _Bias(sw.WindowAttention(48, 3, (4, 4, 4)))
    shape = attn.attn.relative_position_bias_table.shape
    for i in range(20):
        table = torch.full(shape, float(i))
        assert (torch.func.functional_call(attn, {"attn.relative_position_bias_table": table}, ()) == i).all()
        del table


class _Bias(torch.nn.Module):
    def __init__(self, attn):
        super().__init__()
        self.attn = attn

    def forward(self):
        return monai_patch._window_bias(self.attn, 64)


def test_writes_into_data_are_seen_after_forgetting():
    block = _block(c=48)
    first = monai_patch._window_bias(block.attn, 64).clone()
    block.attn.relative_position_bias_table.data.add_(1)
    monai_patch.forget_cached_params(block)
    assert torch.equal(monai_patch._window_bias(block.attn, 64), first + 1)


def test_copies_of_a_module_start_without_kept_parameters():
    attn = sw.WindowAttention(48, 3, (4, 4, 4))
    first = monai_patch._window_bias(attn, 64)
    for other in (copy.deepcopy(attn), pickle.loads(pickle.dumps(attn))):
        assert not any(other.__dict__["_crumpet_cache"].values())
        other.relative_position_bias_table.data.add_(1)
        assert torch.equal(monai_patch._window_bias(other, 64), first + 1)


class _Plain(torch.nn.Module):
    """A block of a program's own, without attention."""

    def forward(self, x, mask_matrix):
        return x + 1


def test_stages_of_other_blocks_run(monkeypatch):
    monkeypatch.setattr(monai_patch, "compute_attn_mask_3d", lambda **k: torch.zeros(1))
    crumpet_amd.patch_monai_swin_unetr()
    try:
        model = _encoder()
        assert _chained(monkeypatch, model)
        model.layers1[0].blocks[0] = _Plain()
        assert not _chained(monkeypatch, model)
        assert model.layers1[0](torch.zeros((1, 32, 8, 8, 8))).shape == (1, 64, 4, 4, 4)
    finally:
        crumpet_amd.unpatch_monai_swin_unetr()
