"""Reversible patch of MONAI-style Swin UNETR models onto the gfx950 kernels.

Same entry points and patched methods as torch-ext/crumpet/monai_patch.py:
``patch_monai_swin_unetr()`` (idempotent; True when it installs the patch,
False when already active) and ``unpatch_monai_swin_unetr()`` (restores
the originals; True / False likewise) replace

* ``SwinTransformerBlock.forward_part1``: norm1, pad to the window grid,
  ``fused_shift_partition_3d``, window attention,
  ``fused_unshift_unpartition_3d``, crop (reference :72-114).  In inference
  mode, with a LayerNorm norm1 and Linear qkv / proj, the whole method runs
  as three kernels instead (``crumpet_amd.fused_block``): norm1 + pad +
  shift + partition + qkv in one, the fused attention, and proj + reverse +
  unshift + crop in one (opt out with ``CRUMPET_DISABLE_FUSED_BLOCK=1``);
* ``BasicLayer.forward``: channels-last stage loop with the cached
  ``compute_attn_mask_3d`` mask (reference :201-232);
* ``SwinTransformerBlock.forward``: in inference with a 16-bit compute type
  the residual sums, norm2 and the MLP run as ``fused_swin_mlp``;
* the patch merging at the end of a patched ``BasicLayer``: gather, norm and
  reduction as ``patch_merge_3d`` (same conditions);
* ``SwinTransformer.forward``: the stages hand each other channels-last
  volumes and the feature norm reads them in place, where the original
  transposes to channels-first and back around every stage (the results have
  the original's shapes and strides);
* ``WindowAttention.forward``: the eager ``q k^T + bias + mask -> softmax
  -> @ v`` chain becomes one gfx950 kernel call (reference :117-198).  It
  falls back to the original in training mode, with attention dropout,
  when ``CRUMPET_DISABLE_FUSED_ATTN=1``, or for a head dimension other
  than 16, 32, 64, 128 or 256 (the kernels' head dimensions; every stage of
  the feature-size-48 Swin UNETR has 16, feature size 96 gives 32).  The
  reference takes the fused path for any head dimension from 16 up
  (reference :144-149), which its Triton kernel compiles for powers of two.

Differences from the reference's patched attention, none of which changes
the math:

* q, k and v are passed to the kernel as strided views of the qkv linear's
  output (no ``.contiguous()`` copies), and the kernel writes straight into
  a ``[b, n, H, hd]`` buffer, so the ``transpose(1, 2).reshape`` copy
  disappears;
* in a shifted block whose mask came from the patched ``BasicLayer`` the
  kernel derives the shifted-window mask from the window geometry
  (``fused_swin_attention_shifted``): nothing is tiled with
  ``mask.repeat`` and no mask or boundary flags are read.  Any other mask is
  read as ``mask[b mod nW]`` with boundary flags computed on the ``nW``
  distinct windows only;
* the relative-position bias stays in the table's dtype (fp32), as in the
  eager MONAI chain, instead of being rounded to the activation dtype.

MONAI is optional: the patch applies to ``monai.networks.nets.swin_unetr``
when it is importable, and always to ``crumpet_amd.swin_unetr_compat`` (the
in-repo MONAI-compatible model used when MONAI is absent).
"""

from __future__ import annotations

import ctypes
import functools
import itertools
import os
import sys
from typing import Any

import torch
import torch.nn.functional as F
from torch.nn.modules import module as _module

from . import _native, compute_attn_mask_3d, fused_shift_partition_3d, fused_unshift_unpartition_3d
from .fused_attention import fused_swin_attention_shifted, fused_swin_attention_windows
from .fused_block import channel_norm, fused_swin_mlp, fused_window_msa_3d, patch_merge_3d

_STATE: dict[str, Any] = {}
_REQUIRED = ("SwinTransformerBlock", "BasicLayer", "WindowAttention", "get_window_size")
# Attribute names: the mask geometry tag set by the patched BasicLayer, and the
# per-call region handed from forward_part1 to the attention module.
_GEOMETRY_ATTR = "_crumpet_geometry"
_REGION_ATTR = "_crumpet_region"


def _fused_attn_enabled() -> bool:
    """Opt-out via ``CRUMPET_DISABLE_FUSED_ATTN=1`` (reference monai_patch.py:47-51)."""
    return os.environ.get("CRUMPET_DISABLE_FUSED_ATTN", "0") != "1"


def _swin_modules() -> list:
    """Modules to patch: MONAI's swin_unetr if importable, plus the in-repo one."""
    mods = []
    try:
        import monai.networks.nets.swin_unetr as monai_swin  # noqa: F401

        if all(hasattr(monai_swin, n) for n in _REQUIRED):
            mods.append(monai_swin)
    except Exception:
        pass
    from . import swin_unetr_compat

    mods.append(swin_unetr_compat)
    return mods


def _as_triple(value) -> tuple[int, int, int]:
    if len(value) != 3:
        raise RuntimeError("CRUMPET MONAI patch only supports 3D Swin blocks")
    return tuple(int(v) for v in value)


def _fused_block_enabled() -> bool:
    """Opt-out of the fused block projections via ``CRUMPET_DISABLE_FUSED_BLOCK=1``."""
    return os.environ.get("CRUMPET_DISABLE_FUSED_BLOCK", "0") != "1"


def _compute_dtype(x: torch.Tensor) -> torch.dtype:
    """The dtype the block's Linear layers run in: autocast's, else x's."""
    if torch.is_autocast_enabled(x.device.type):
        return torch.get_autocast_dtype(x.device.type)
    return x.dtype


_ESIZE = {torch.float32: 4, torch.float16: 2, torch.bfloat16: 2}
# head dimensions of the fused attention kernels
_HEAD_DIMS = (16, 32, 64, 128, 256)


def _fits_staging_tile(c: int, esize: int) -> bool:
    """The projections' LDS tile (window_linear.hip plan_tile): 64 staged rows
    of C channels, an output chunk of at least 16 features (rows padded by
    16 bytes each) and 64 row indices within 64 KiB."""
    pad = 16 // esize
    return 64 * (c + pad) * esize + 64 * (16 + pad) * esize + 64 * 4 <= 64 * 1024


def _fused_block_supported(block, x: torch.Tensor) -> bool:
    """Inference-mode blocks whose attention half the fused block kernels
    cover: LayerNorm norm1 over C, Linear qkv / proj, a head dimension the
    attention kernels take, no attention dropout, C a multiple of 16 that
    fits the staging tile."""
    attn = block.attn
    c = x.shape[-1]
    if block.training or not (_fused_attn_enabled() and _fused_block_enabled()):
        return False
    if x.device.type != "cuda" or x.dtype not in (torch.float32, torch.float16, torch.bfloat16):
        return False
    norm = block.norm1
    if not isinstance(norm, torch.nn.LayerNorm) or tuple(norm.normalized_shape) != (c,):
        return False
    if not isinstance(attn.qkv, torch.nn.Linear) or not isinstance(attn.proj, torch.nn.Linear):
        return False
    if attn.qkv.out_features != 3 * c or attn.proj.in_features != c or attn.proj.out_features != c:
        return False
    if attn.attn_drop.p != 0.0 or c % attn.num_heads != 0 or c // attn.num_heads not in _HEAD_DIMS:
        return False
    return c % 16 == 0 and c <= 384 and _fits_staging_tile(c, _ESIZE[_compute_dtype(x)])


def _tensors(value):
    """The tensors of a value that ``_cached`` keeps."""
    if isinstance(value, torch.Tensor):
        return [value]
    return [] if value is None else [t for v in value for t in _tensors(v)]


class _Entry:
    """A value that ``_cached`` keeps.  ``held`` are the source tensors'
    storages: while they live no other tensor can be found at their
    addresses.  Another stream than the one that made the value waits for it,
    and is noted with its memory.  Copies and pickles of a module start
    without the entry."""

    __slots__ = ("stamp", "held", "value", "device", "stream", "made")

    def __init__(self, stamp, sources, value):
        self.stamp, self.value = stamp, value
        self.held = tuple(t.detach() for t in sources)
        self.device, self.stream, self.made = sources[0].device, None, None
        if self.device.type == "cuda":
            current = torch.cuda.current_stream(self.device)
            self.stream, self.made = current.cuda_stream, current.record_event()

    def use(self):
        if self.made is not None and torch._C._cuda_getCurrentRawStream(self.device.index) != self.stream:
            current = torch.cuda.current_stream(self.device)
            current.wait_event(self.made)
            for t in _tensors(self.value):
                t.record_stream(current)
        return self.value

    def __deepcopy__(self, memo):
        return None

    def __reduce__(self):
        return type(None), ()


def _cached(module, key, sources, make):
    """``make()`` for ``key``, kept on ``module`` until a tensor in ``sources``
    changes: an in-place update bumps its version counter, reassigning it
    (also through ``.data``, or by a call that swaps parameters in) changes
    its storage.  A write *into* ``.data`` does neither and is not seen;
    ``forget_cached_params`` is for programs that write so.  Under graph
    capture nothing is cached or reused: the value is recomputed by kernels
    the graph records, so every replay reads the parameters as they are then
    (the reference recomputes the bias on every call for that reason,
    torch-ext/crumpet/monai_patch.py:157-162)."""
    if torch.cuda.is_available() and torch.cuda.is_current_stream_capturing():
        return make()
    stamp = tuple((t._version, t.data_ptr()) for t in sources)
    cache = module.__dict__.setdefault("_crumpet_cache", {})
    hit = cache.get(key)
    if hit is not None and hit.stamp == stamp:
        return hit.use()
    with torch.no_grad():
        value = make()
    cache[key] = _Entry(stamp, sources, value)
    return value


def forget_cached_params(model: torch.nn.Module) -> None:
    """Drop what the patched attention half keeps of its parameters (the
    gathered relative-position bias, the projections in the compute type), to
    be made anew by the next pass: for programs that write into a
    parameter's ``.data`` between passes, which nothing else shows."""
    for module in model.modules():
        module.__dict__.pop("_crumpet_cache", None)


def _window_bias(attn, n):
    """``[heads, n, n]`` relative-position bias of the first ``n`` window
    tokens, gathered from the transposed table (unit stride along keys) and
    kept in the table's dtype; cached on the module (``_cached``)."""
    def make():
        idx = attn.relative_position_index[:n, :n].reshape(-1)
        return attn.relative_position_bias_table.t()[:, idx].view(attn.num_heads, n, n)

    return _cached(attn, ("bias", n), (attn.relative_position_bias_table, attn.relative_position_index), make)


def _block_params(attn, n, dtype):
    """``(bias, (w_qkv, b_qkv), (w_proj, b_proj))`` of a window-attention
    module for the fused block: the gathered ``[heads, n, n]`` bias and both
    projections cast to ``dtype``, kept as one entry on the module
    (``_cached``), so a call checks the sources' versions once."""
    def make():
        idx = attn.relative_position_index[:n, :n].reshape(-1)
        bias = attn.relative_position_bias_table.t()[:, idx].view(attn.num_heads, n, n)
        cast = lambda t: None if t is None else t.to(dtype).contiguous()  # noqa: E731
        return bias, (cast(attn.qkv.weight), cast(attn.qkv.bias)), (cast(attn.proj.weight), cast(attn.proj.bias))

    sources = tuple(t for t in (attn.relative_position_bias_table, attn.relative_position_index,
                                attn.qkv.weight, attn.qkv.bias, attn.proj.weight, attn.proj.bias)
                    if t is not None)
    return _cached(attn, ("block", n, dtype), sources, make)


def _fused_block_forward(block, x, mask_matrix, swin):
    """forward_part1 as three kernels: window_qkv_3d (norm1, pad, shift,
    partition, qkv), the fused attention, window_proj_3d (proj, reverse,
    unshift, crop), launched by one dispatcher call unless a mask tensor
    without the geometry tag is passed.  The gathered bias and the cast
    projection weights are cached per module."""
    b, d, h, w, c = x.shape
    window_size, shift_size = swin.get_window_size((d, h, w), block.window_size, block.shift_size)
    ws = _as_triple(window_size)
    ss = _as_triple(shift_size)
    padded = tuple(-(-n // k) * k for n, k in zip((d, h, w), ws))
    attn = block.attn
    n = ws[0] * ws[1] * ws[2]
    dtype = _compute_dtype(x)
    bias, qkv, proj = _block_params(attn, n, dtype)
    shifted = any(s > 0 for s in ss)
    region = shifted and getattr(mask_matrix, _GEOMETRY_ATTR, None) == (*padded, ws, ss)
    return fused_window_msa_3d(x, block.norm1, qkv, proj, bias, attn.num_heads, attn.scale, ws, ss,
                               mask=mask_matrix if shifted else None, region=region, dtype=dtype)


def _patched_forward_part1(original, swin):
    @functools.wraps(original)
    def forward_part1(self, x, mask_matrix):
        if x.dim() != 5:
            return original(self, x, mask_matrix)
        if _fused_block_supported(self, x):
            return _fused_block_forward(self, x, mask_matrix, swin)
        x = self.norm1(x)
        b, d, h, w, c = x.shape
        window_size, shift_size = swin.get_window_size((d, h, w), self.window_size, self.shift_size)
        window_size = _as_triple(window_size)
        shift_size = _as_triple(shift_size)
        pad_d1 = (window_size[0] - d % window_size[0]) % window_size[0]
        pad_b = (window_size[1] - h % window_size[1]) % window_size[1]
        pad_r = (window_size[2] - w % window_size[2]) % window_size[2]
        if pad_d1 > 0 or pad_b > 0 or pad_r > 0:
            x = F.pad(x, (0, 0, 0, pad_r, 0, pad_b, 0, pad_d1))
        _, dp, hp, wp, _ = x.shape

        shifted = any(s > 0 for s in shift_size)
        attn_mask = mask_matrix if shifted else None
        region = None
        if shifted and getattr(mask_matrix, _GEOMETRY_ATTR, None) == (dp, hp, wp, window_size, shift_size):
            region = ((dp, hp, wp), window_size, shift_size)

        x_windows = fused_shift_partition_3d(x, window_size, shift_size)
        setattr(self.attn, _REGION_ATTR, region)
        try:
            attn_windows = self.attn(x_windows, mask=attn_mask)
        finally:
            setattr(self.attn, _REGION_ATTR, None)
        x = fused_unshift_unpartition_3d(attn_windows, B=b, D=dp, H=hp, W=wp, C=c,
                                         window_size=window_size, shift_size=shift_size)
        if pad_d1 > 0 or pad_r > 0 or pad_b > 0:
            x = x[:, :d, :h, :w, :].contiguous()
        return x

    return forward_part1


def _patched_window_attention_forward(original):
    @functools.wraps(original)
    def forward(self, x, mask):
        if self.training or self.attn_drop.p != 0.0 or not _fused_attn_enabled():
            return original(self, x, mask)
        b, n, c = x.shape
        heads = self.num_heads
        hd = c // heads
        if hd not in _HEAD_DIMS or hd * heads != c:
            return original(self, x, mask)

        qkv = self.qkv(x)  # [b, n, 3c]; channel = s*c + h*hd + d
        t = qkv.view(b, n, 3, heads, hd).permute(2, 0, 3, 1, 4)  # views [b, H, n, hd]
        bias = _window_bias(self, n)
        out = torch.empty((b, n, heads, hd), dtype=qkv.dtype, device=qkv.device)
        ov = out.permute(0, 2, 1, 3)
        region = getattr(self, _REGION_ATTR, None)
        if mask is not None and region is not None:
            volume, ws, ss = region
            fused_swin_attention_shifted(t[0], t[1], t[2], bias, volume, ws, ss, self.scale, ov)
        elif mask is not None:
            nw = mask.shape[0]
            flags = (mask.reshape(nw, -1).abs().amax(dim=1) > 0).to(torch.uint8)
            boundary = flags.repeat(b // nw).contiguous()
            fused_swin_attention_windows(t[0], t[1], t[2], bias, mask, boundary, self.scale, ov)
        else:
            fused_swin_attention_windows(t[0], t[1], t[2], bias, None, None, self.scale, ov)
        x = self.proj(out.view(b, n, c))
        return self.proj_drop(x)

    return forward


# ---- what the eager modules would do beyond the values ---------------------------

_HALF = (torch.float16, torch.bfloat16)
_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _computes_half(x: torch.Tensor) -> bool:
    """Whether the fused second half and patch merging may apply at all; asked
    first, so that an fp32 model, whose host is the slower side, pays for no
    other check."""
    return x.device.type == "cuda" and _compute_dtype(x) in _HALF


def _unhooked(*modules) -> bool:
    """Whether running the modules' math without calling them goes unnoticed:
    no hooks, and no forward that a program put on the object itself."""
    return not any(m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__ for m in modules) and not (
        _module._global_forward_hooks or _module._global_forward_pre_hooks)


_OWN: dict[tuple, Any] = {}


def _own(cls, name):
    """``cls.name`` as the module that defines ``cls`` wrote it; None while a
    program has another function there (unless the first was seen before)."""
    method = _OWN.get((cls, name))
    if method is None:
        here = getattr(cls, name)
        code = getattr(here, "__code__", None)
        if code is not None and code.co_filename == getattr(sys.modules.get(cls.__module__), "__file__", None):
            method = _OWN[cls, name] = here
    return method


def _stock(obj, cls, name) -> bool:
    """Whether ``obj.name`` is the method that ``cls``'s module wrote: not that
    of a subclass, nor one that a program put on the class or the object."""
    return getattr(type(obj), name, None) is _own(cls, name) and name not in obj.__dict__


def _watched() -> bool:
    """Whether something follows the ops that run, and would miss those that
    a fused kernel stands for: a function transform, forward-mode gradients,
    a dispatch mode, torch.jit.trace."""
    return (torch._C._functorch.peek_interpreter_stack() is not None or torch.autograd.forward_ad._current_level >= 0
            or torch._C._len_torch_dispatch_stack() > 0 or torch.jit.is_tracing())


def _values_only(x: torch.Tensor, params) -> bool:
    """Whether a pass over ``x`` needs nothing but its values: a plain HIP
    tensor, no gradient of any kind, nothing that follows the ops."""
    if type(x) is not torch.Tensor or x.device.type != "cuda" or _watched():
        return False
    return not (torch.is_grad_enabled() and (x.requires_grad or any(p.requires_grad for p in params)))


def _half_compute(x: torch.Tensor, params) -> torch.dtype | None:
    """The 16-bit type the Linears of ``params`` run in on ``x``, or None
    where they run in fp32, or where the eager ops mix types in another way
    (without autocast everything must share x's type).  Tensor subclasses
    (quantised or distributed weights) bring ops of their own; the kernels'
    16-byte accesses need what eager does not, aligned storage (parameters
    that are views of one flat vector often are not)."""
    if any(type(p) not in _PLAIN for p in params) or any(t.data_ptr() % 16 for t in (x, *params)):
        return None
    if torch.is_autocast_enabled("cuda"):
        dtype = torch.get_autocast_dtype("cuda")
        plain = x.dtype in (torch.float32, dtype) and all(
            p.dtype in (torch.float32, x.dtype) for p in params)
    else:
        dtype = x.dtype
        plain = all(p.dtype == dtype for p in params)
    return dtype if plain and dtype in _HALF else None


def _stock_module(module, swin, *names) -> bool:
    """Whether ``module`` is of a class that ``swin`` knows by one of
    ``names``, with that class's own forward (a class of the same name from
    elsewhere may compute anything)."""
    cls = type(module)
    return any(cls is getattr(swin, name, None) for name in names) and _stock(module, cls, "forward")


def _idle(drop, swin) -> bool:
    """A dropout or drop-path module that passes its input through."""
    if type(drop) is torch.nn.Identity:
        return True
    return not drop.training and (type(drop) is torch.nn.Dropout or _stock_module(drop, swin, "DropPath"))


def _linear_params(*linears):
    return [p for m in linears for p in (m.weight, m.bias) if p is not None]


def _affine_norm(norm, c) -> bool:
    """A LayerNorm over ``c`` whose parameters the kernels take: contiguous,
    and of one type (autocast brings both to fp32, whatever they are)."""
    if type(norm) is not torch.nn.LayerNorm or tuple(norm.normalized_shape) != (c,):
        return False
    params = _norm_params(norm)
    return all(p.is_contiguous() and p.dtype == params[0].dtype for p in params)


def _norm_params(norm):
    return [p for p in (norm.weight, norm.bias) if p is not None]


def _fusable_heads(block) -> bool:
    """Whether the block's attention runs fused.  Models whose head dimension
    is not covered keep every other eager op too, and with them eager's exact
    bits, and so do those whose blocks are something else."""
    try:
        attn = block.attn
        return _fused_attn_enabled() and attn.dim // attn.num_heads in _HEAD_DIMS and attn.attn_drop.p == 0.0
    except AttributeError:
        return False


@functools.lru_cache(maxsize=64)
def _one_kernel_mlp(c: int, hidden: int) -> bool:
    f = _native.hip_library().crumpet_swin_mlp_fits
    f.argtypes = [ctypes.c_int64, ctypes.c_int64]
    return bool(f(c, hidden))


def _tail_dtype(block, x, swin=None) -> torch.dtype | None:
    """The compute type of a block's fused second half, or None: inference,
    the module's own ``forward_part2`` (LayerNorm -> Linear -> exact GELU ->
    Linear) with idle dropouts, sizes that the kernels take (channels and
    hidden features multiples of 32, or of 16 where one kernel covers the
    block).  ``swin`` is the patched module, by default the in-repo one."""
    if torch.compiler.is_compiling() or not _computes_half(x):
        return None
    if block.training or x.dim() != 5 or not _fused_block_enabled():
        return None
    if swin is None:
        from . import swin_unetr_compat as swin
    if not _stock(block, swin.SwinTransformerBlock, "forward_part2"):
        return None
    if getattr(block, "use_checkpoint", False) or not _fusable_heads(block):
        return None
    norm, mlp, c = block.norm2, block.mlp, x.shape[-1]
    # MONAI's swin_unetr imports its MLPBlock as Mlp
    if not _stock_module(mlp, swin, "MLPBlock", "Mlp") or not _affine_norm(norm, c):
        return None
    l1, l2, fn = mlp.linear1, mlp.linear2, mlp.fn
    if type(l1) is not torch.nn.Linear or type(l2) is not torch.nn.Linear or type(fn) is not torch.nn.GELU:
        return None
    if fn.approximate != "none" or not all(
            _idle(m, swin) for m in (block.drop_path, mlp.drop1, mlp.drop2)):
        return None
    hidden = l1.out_features
    if l1.in_features != c or l2.in_features != hidden or l2.out_features != c or hidden % 32 or c > 6144:
        return None
    if c % 32 and not _one_kernel_mlp(c, hidden):
        return None
    if not _unhooked(norm, mlp, l1, l2, fn, block.drop_path, mlp.drop1, mlp.drop2):
        return None
    params = _linear_params(l1, l2) + _norm_params(norm)
    return _half_compute(x, params) if _values_only(x, params) else None


def _patched_block_forward(original, swin):
    own = _own(swin.SwinTransformerBlock, "forward") is original

    @functools.wraps(original)
    def forward(self, x, mask_matrix):
        dtype = _tail_dtype(self, x, swin) if own else None
        if dtype is None:
            return original(self, x, mask_matrix)
        half = self.forward_part1(x, mask_matrix)
        # a gradient through the attention half (its parameters may train while
        # the MLP's do not), or a half that a subclass gave another form
        if (half.dtype != dtype or half.requires_grad or half.shape != x.shape or type(half) is not torch.Tensor
                or half.data_ptr() % 16):
            x = x + half
            return x + self.forward_part2(x)
        return fused_swin_mlp(x, half, self.norm2, self.mlp.linear1, self.mlp.linear2, dtype)

    return forward


# sub-grid offsets (d, h, w) in concatenation order
_MERGE_V2 = tuple(itertools.product(range(2), repeat=3))
_MERGE_V1 = ((0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (0, 1, 0), (0, 0, 1), (1, 1, 1))


def _downsample(m, x, swin):
    """A stage's patch merging: one gather + norm pass and the reduction, or
    the module itself."""
    offsets = _MERGE_V1 if type(m) is getattr(swin, "PatchMerging", None) else _MERGE_V2
    if (torch.compiler.is_compiling() or not _computes_half(x) or m.training or x.dim() != 5
            or not _fused_block_enabled() or not _stock_module(m, swin, "PatchMerging", "PatchMergingV2")):
        return m(x)
    norm, red, c = m.norm, m.reduction, x.shape[-1]
    if (type(red) is not torch.nn.Linear or red.bias is not None or red.in_features != 8 * c
            or red.out_features % 16 or c % 4 or c > 768 or not _affine_norm(norm, 8 * c)
            or not _unhooked(m, norm, red)):
        return m(x)
    params = [red.weight] + _norm_params(norm)
    dtype = _half_compute(x, params) if _values_only(x, params) else None
    if dtype is None:
        return m(x)
    return patch_merge_3d(x, norm, red.weight, offsets, dtype)


def _layer_channels_last(layer, x, swin):
    """A stage on a contiguous ``[b, d, h, w, c]`` volume, channels-last out."""
    b, d, h, w, _ = x.shape
    window_size, shift_size = swin.get_window_size((d, h, w), layer.window_size, layer.shift_size)
    window_size = _as_triple(window_size)
    shift_size = _as_triple(shift_size)
    dp = -(-d // window_size[0]) * window_size[0]
    hp = -(-h // window_size[1]) * window_size[1]
    wp = -(-w // window_size[2]) * window_size[2]
    attn_mask = compute_attn_mask_3d(D=dp, H=hp, W=wp, window_size=window_size,
                                     shift_size=shift_size, dtype=x.dtype, device=x.device)
    setattr(attn_mask, _GEOMETRY_ATTR, (dp, hp, wp, window_size, shift_size))
    for blk in layer.blocks:
        x = blk(x, attn_mask)
    x = x.view(b, d, h, w, -1)
    if layer.downsample is not None:
        fused = _computes_half(x) and len(layer.blocks) > 0 and _fusable_heads(layer.blocks[-1])
        x = _downsample(layer.downsample, x, swin) if fused else layer.downsample(x)
    return x


def _patched_basic_layer_forward(original, swin):
    @functools.wraps(original)
    def forward(self, x):
        if x.dim() != 5:
            return original(self, x)
        x = _layer_channels_last(self, x.permute(0, 2, 3, 4, 1).contiguous(), swin)
        return x.permute(0, 4, 1, 2, 3).contiguous()

    return forward


def _channels_last_chain(model, x, normalize, swin) -> bool:
    """Whether the encoder's stages may hand each other channels-last
    volumes: inference on plain tensors, the module's own ``proj_out``, every
    stage the patched ``BasicLayer`` without hooks, normalised features."""
    if (torch.compiler.is_compiling() or model.training or not normalize or x.dim() != 5
            or type(model) is not swin.SwinTransformer or getattr(model, "use_v2", False)
            or not _stock(model, swin.SwinTransformer, "proj_out") or not _fused_block_enabled()):
        return False
    layers = [getattr(model, f"layers{i + 1}", ()) for i in range(model.num_layers)]
    if swin.BasicLayer.forward is not _STATE.get("basic_layer", {}).get(swin.BasicLayer):
        return False
    if not all(len(m) >= 1 and type(m[0]) is swin.BasicLayer and _unhooked(m[0]) and len(m[0].blocks)
               and _fusable_heads(m[0].blocks[0]) for m in layers):
        return False
    return _values_only(x, model.parameters())


def _feature(x):
    """The normalised feature, channels-first, of a channels-last volume."""
    # F.layer_norm runs and returns in fp32 under autocast
    dtype = torch.float32 if torch.is_autocast_enabled("cuda") else None
    c = x.shape[-1]
    fits = c % 8 == 0 and c <= 6144 and x.data_ptr() % 16 == 0  # the kernel's rows
    x = channel_norm(x, dtype=dtype) if fits else F.layer_norm(x, (c,))
    return x.permute(0, 4, 1, 2, 3)


def _patched_transformer_forward(original, swin):
    own = _own(swin.SwinTransformer, "forward") is original

    @functools.wraps(original)
    def forward(self, x, normalize=True):
        if not (own and _channels_last_chain(self, x, normalize, swin)):
            return original(self, x, normalize)
        x = self.pos_drop(self.patch_embed(x)).permute(0, 2, 3, 4, 1).contiguous()
        outs = [_feature(x)]
        for i in range(self.num_layers):
            x = _layer_channels_last(getattr(self, f"layers{i + 1}")[0], x, swin)
            outs.append(_feature(x))
        return outs

    return forward


def patch_monai_swin_unetr() -> bool:
    """Install the patch.  Returns True on the call that installs it and False
    if it is already active (reference monai_patch.py:235-261)."""
    if _STATE.get("patched"):
        return False
    saved = []
    basic_layer = {}

    def install(cls, name, make, *args):
        original = cls.__dict__[name]
        saved.append((cls, name, original))
        setattr(cls, name, make(original, *args))

    for swin in _swin_modules():
        install(swin.SwinTransformerBlock, "forward_part1", _patched_forward_part1, swin)
        install(swin.SwinTransformerBlock, "forward", _patched_block_forward, swin)
        install(swin.BasicLayer, "forward", _patched_basic_layer_forward, swin)
        basic_layer[swin.BasicLayer] = swin.BasicLayer.forward
        if hasattr(swin, "SwinTransformer"):
            install(swin.SwinTransformer, "forward", _patched_transformer_forward, swin)
        if _fused_attn_enabled():
            install(swin.WindowAttention, "forward", _patched_window_attention_forward)
    _STATE.update({"patched": True, "saved": saved, "basic_layer": basic_layer})
    return True


def unpatch_monai_swin_unetr() -> bool:
    """Restore the original methods.  Returns True if a patch was removed
    (reference monai_patch.py:264-275)."""
    if not _STATE.get("patched"):
        return False
    for cls, name, original in _STATE["saved"]:
        setattr(cls, name, original)
    _STATE.clear()
    return True


def is_patched() -> bool:
    return bool(_STATE.get("patched"))
