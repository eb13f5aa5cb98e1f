"""The work that crumpet_amd does for its users, as cases that can be timed.

Each case is one pass through the public entry points: the window gathers and
their gradients, the shifted-window mask, the window attention in its mask
modes, data types and head dimensions, the fused attention half of a Swin
block, and the patched Swin encoder as a whole.  Sizes are the Swin UNETR
stages at feature sizes 48 and 96 (windows of 7 and 6, heads of 16 and 32)
and the window sizes and head dimensions that the tests cover.  ``draw``
gives more cases of the same ranges.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import crumpet_amd
from crumpet_amd import fused_block
from crumpet_amd import swin_unetr_compat as swin
from crumpet_amd.fused_attention import fused_swin_attention, fused_swin_attention_shifted

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def _gather(name, B, grid, ws, shift, C, dtype, grad):
    """``grid`` windows of ``ws`` tokens per axis, cyclic shift ``shift``."""
    case = {"kind": "gather", "B": B, "C": C, "dtype": dtype, "grad": grad}
    for a, n, w, s in zip("dhw", grid, ws, shift):
        case.update({f"n{a}": n, f"ws_{a}": w, f"ss_{a}": s})
    return {"name": name, **case} if name else case


def _attention(name, B, grid, ws, heads, hd, dtype, mode, layout):
    """B volumes of ``grid`` windows.  mode: "none", "shifted" (the mask comes
    from the geometry), "kept" (a mask tensor that the program keeps) or
    "new" (the mask of a geometry not seen before).  layout: "qkv" (views of
    a qkv projection's output) or "split" (contiguous q, k and v)."""
    case = {"kind": "attention", "B": B, "heads": heads, "hd": hd, "dtype": dtype, "mode": mode, "layout": layout}
    for a, n, w in zip("dhw", grid, ws):
        case.update({f"n{a}": n, f"ws_{a}": w})
    return {"name": name, **case} if name else case


def _block(name, B, dims, ws, C, hd, shifted, x_dtype, dtype):
    case = {"kind": "block", "B": B, "C": C, "hd": hd, "shifted": shifted, "x_dtype": x_dtype, "dtype": dtype}
    for a, n, w in zip("dhw", dims, ws):
        case.update({a: n, f"ws_{a}": w})
    return {"name": name, **case} if name else case


def _encoder(name, B, dims, feature, dtype):
    case = {"kind": "encoder", "B": B, "feature": feature, "dtype": dtype}
    case.update(zip("dhw", dims))
    return {"name": name, **case} if name else case


def listed():
    return [
        # one small crop's tokens into shifted windows and back: the launches count
        _gather("gather_crop_bf16", 1, (2, 2, 2), (7, 7, 7), (3, 3, 3), 48, "bf16", False),
        # a 196^3 scan at patch size 2, stage 0, the whole volume at once
        _gather("gather_volume_fp16", 1, (14, 14, 14), (7, 7, 7), (3, 3, 3), 48, "fp16", False),
        # training at feature size 12 (24-byte tokens), ragged grid, both directions and their gradients
        _gather("gather_train_narrow", 2, (5, 7, 6), (7, 7, 7), (3, 3, 3), 12, "fp16", True),
        # stage 0 of four 96^3 crops under fp16 autocast, shifted block
        _attention("attn_shifted_fp16", 4, (7, 7, 7), (7, 7, 7), 3, 16, "fp16", "shifted", "qkv"),
        # a new volume size: its mask is made, then read by the first attention of the stage
        _attention("attn_new_mask_fp16", 1, (14, 14, 14), (7, 7, 7), 3, 16, "fp16", "new", "split"),
        # one 96^3 crop, bf16, the mask tensor kept by the program
        _attention("attn_kept_mask_bf16", 1, (7, 7, 7), (7, 7, 7), 3, 16, "bf16", "kept", "split"),
        # one 96^3 crop without autocast: everything in fp32
        _attention("attn_shifted_fp32", 1, (7, 7, 7), (7, 7, 7), 3, 16, "fp32", "shifted", "qkv"),
        # wide heads, shifted 7^3 windows
        _attention("attn_hd64_bf16", 1, (5, 5, 5), (7, 7, 7), 6, 64, "bf16", "shifted", "qkv"),
        # 8^3 windows, heads of 32
        _attention("attn_long_fp16", 2, (4, 4, 4), (8, 8, 8), 6, 32, "fp16", "none", "qkv"),
        # the attention half of a shifted stage-0 block of four 96^3 crops (padded to 49^3)
        _block("block_stage0_fp16", 4, (48, 48, 48), (7, 7, 7), 48, 16, True, "fp32", "fp16"),
        # the deepest stage of the same crops: 6^3 windows, no shift
        _block("block_stage3_bf16", 4, (6, 6, 6), (6, 6, 6), 384, 16, False, "fp32", "bf16"),
        # the whole patched encoder on one 96^3 crop
        _encoder("encoder_fp16", 1, (96, 96, 96), 48, "fp16"),
    ]


_WINDOWS = ((7, 7, 7), (7, 7, 7), (7, 7, 7), (6, 6, 6), (4, 4, 4), (8, 8, 8), (2, 7, 7), (5, 6, 7), (3, 5, 4))


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["bytes"] <= 6.0e8 and w["flops"] <= 5.0e10:
            return case


def _draw(rng):
    kind = rng.choice(("gather", "attention", "attention", "attention", "block", "block", "encoder"))
    ws = rng.choice(_WINDOWS)
    dtype = rng.choice(("fp16", "bf16", "fp32"))
    if kind == "gather":
        grid = tuple(_log_int(rng, 1, 14) for _ in range(3))
        shift = tuple(w // 2 for w in ws) if rng.random() < 0.7 else (0, 0, 0)
        C = rng.choice((12, 24, 33, 36, 48, 60, 96, 192, 384))
        return _gather(None, rng.randint(1, 4), grid, ws, shift, C, dtype, rng.random() < 0.5)
    if kind == "attention":
        grid = tuple(_log_int(rng, 1, 12) for _ in range(3))
        hd = rng.choice((16, 16, 16, 32, 32, 64, 128))
        mode = rng.choice(("none", "shifted", "shifted", "kept", "new"))
        layout = rng.choice(("qkv", "split"))
        return _attention(None, rng.randint(1, 4), grid, ws, rng.choice((3, 4, 6, 12, 24)), hd, dtype, mode, layout)
    if kind == "block":
        dims = tuple(_log_int(rng, 6, 48) for _ in range(3))
        ws = tuple(min(w, d) for w, d in zip(rng.choice(((7, 7, 7), (7, 7, 7), (6, 6, 6), (4, 4, 4))), dims))
        C, hd = rng.choice(((48, 16), (96, 16), (192, 16), (384, 16), (96, 32), (192, 32), (384, 32)))
        if C == 384 and dtype == "fp32":
            C = 192  # the widest block that the fp32 projections take
        x_dtype = rng.choice(("fp32", dtype))
        return _block(None, rng.randint(1, 4), dims, ws, C, hd, rng.random() < 0.5, x_dtype, dtype)
    dims = tuple(16 * rng.randint(2, 6) for _ in range(3))
    return _encoder(None, rng.randint(1, 2), dims, rng.choice((48, 48, 96)), dtype)


# ---- inputs ----------------------------------------------------------------


def _randn(gen, shape, dtype, std=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * std).to(dtype)


def _triple(case, prefix):
    return tuple(case[prefix + a] for a in "dhw")


def _attention_geometry(case):
    ws = _triple(case, "ws_")
    grid = _triple(case, "n")
    dims = tuple(n * w for n, w in zip(grid, ws))
    shift = tuple(w // 2 for w in ws)
    return dims, ws, shift, grid[0] * grid[1] * grid[2], ws[0] * ws[1] * ws[2]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    dtype = DTYPES[case["dtype"]]
    s = {"case": case}
    if case["kind"] == "gather":
        s["ws"], s["shift"] = _triple(case, "ws_"), _triple(case, "ss_")
        s["dims"] = tuple(n * w for n, w in zip(_triple(case, "n"), s["ws"]))
        shape = (case["B"], *s["dims"], case["C"])
        s["x"] = _randn(gen, shape, dtype).requires_grad_(case["grad"])
        if case["grad"]:
            s["g"] = _randn(gen, shape, dtype)
    elif case["kind"] == "attention":
        dims, ws, shift, nw, n = _attention_geometry(case)
        B, H, hd = case["B"] * nw, case["heads"], case["hd"]
        if case["layout"] == "qkv":
            t = _randn(gen, (B, n, 3, H, hd), dtype).permute(2, 0, 3, 1, 4)
            # the result goes where the output projection reads it
            s["out"] = torch.empty((B, n, H, hd), dtype=dtype, device="cuda").permute(0, 2, 1, 3)
        else:
            t = _randn(gen, (3, B, H, n, hd), dtype)
            s["out"] = None
        s["q"], s["k"], s["v"] = t[0], t[1], t[2]
        s["bias"] = _randn(gen, (H, n, n), torch.float32, 0.2)
        s["geometry"] = (dims, ws, shift)
        if case["mode"] in ("kept", "new"):
            mask = crumpet_amd.compute_attn_mask_3d(*dims, ws, shift, dtype, "cuda")
            flags = (mask.abs().amax(dim=(1, 2)) > 0).to(torch.uint8)
            s["flags"] = flags.repeat(case["B"])
            if case["mode"] == "kept":
                # the entry point takes one mask per window of the batch
                s["mask"] = mask if case["B"] == 1 else mask.repeat(case["B"], 1, 1)
    elif case["kind"] == "block":
        C = case["C"]
        dims = tuple(case[a] for a in "dhw")
        s["ws"] = _triple(case, "ws_")
        s["shift"] = tuple(w // 2 if case["shifted"] and d > w else 0 for d, w in zip(dims, s["ws"]))
        n = s["ws"][0] * s["ws"][1] * s["ws"][2]
        s["x"] = _randn(gen, (case["B"], *dims, C), DTYPES[case["x_dtype"]])
        s["norm"] = torch.nn.LayerNorm(C, device="cuda", dtype=DTYPES[case["x_dtype"]]).requires_grad_(False)
        s["norm"].weight.copy_(1.0 + _randn(gen, (C,), torch.float32, 0.1))
        s["norm"].bias.copy_(_randn(gen, (C,), torch.float32, 0.1))
        # weights cast to the compute type once, as the patched model keeps them
        s["qkv"] = (_randn(gen, (3 * C, C), dtype, C ** -0.5), _randn(gen, (3 * C,), dtype, 0.1))
        s["proj"] = (_randn(gen, (C, C), dtype, C ** -0.5), _randn(gen, (C,), dtype, 0.1))
        s["bias"] = _randn(gen, (C // case["hd"], n, n), torch.float32, 0.2)
    else:
        torch.manual_seed(int(seed))
        with torch.device("cuda"):
            model = swin.SwinTransformer(in_chans=1, embed_dim=case["feature"], window_size=(7, 7, 7),
                                         patch_size=(2, 2, 2), depths=(2, 2, 2, 2), num_heads=(3, 6, 12, 24))
        s["model"] = model.eval().requires_grad_(False)
        s["x"] = torch.rand((case["B"], 1, *(case[a] for a in "dhw")), generator=gen, device="cuda")
        crumpet_amd.patch_monai_swin_unetr()
    return s


# ---- one pass --------------------------------------------------------------


def run(s):
    case = s["case"]
    if case["kind"] == "gather":
        windows = crumpet_amd.fused_shift_partition_3d(s["x"], s["ws"], s["shift"])
        y = crumpet_amd.fused_unshift_unpartition_3d(windows, case["B"], *s["dims"], case["C"], s["ws"], s["shift"])
        if not case["grad"]:
            return [windows, y]
        (gx,) = torch.autograd.grad(y, s["x"], s["g"])
        return [windows.detach(), y.detach(), gx]
    if case["kind"] == "attention":
        dims, ws, shift = s["geometry"]
        q, k, v, bias = s["q"], s["k"], s["v"], s["bias"]
        if case["mode"] == "shifted":
            return [fused_swin_attention_shifted(q, k, v, bias, dims, ws, shift, out=s["out"])]
        if case["mode"] == "none":
            return [fused_swin_attention(q, k, v, bias, None, out=s["out"])]
        if case["mode"] == "kept":
            return [fused_swin_attention(q, k, v, bias, s["mask"], s["flags"], out=s["out"])]
        crumpet_amd.clear_mask_cache()  # a geometry that was not seen before
        mask = crumpet_amd.compute_attn_mask_3d(*dims, ws, shift, q.dtype, q.device)
        tiled = mask if case["B"] == 1 else mask.repeat(case["B"], 1, 1)
        return [mask, fused_swin_attention(q, k, v, bias, tiled, s["flags"], out=s["out"])]
    if case["kind"] == "block":
        hd = case["hd"]
        return [fused_block.fused_window_msa_3d(s["x"], s["norm"], s["qkv"], s["proj"], s["bias"], case["C"] // hd,
                                                hd ** -0.5, s["ws"], s["shift"], dtype=DTYPES[case["dtype"]])]
    dtype = DTYPES[case["dtype"]]
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16 if dtype == torch.float32 else dtype,
                                         enabled=dtype != torch.float32):
        return s["model"](s["x"])


# ---- what a pass cannot do without -----------------------------------------


def work(case):
    es = 4 if case["dtype"] == "fp32" else 2
    if case["kind"] == "gather":
        ws, grid = _triple(case, "ws_"), _triple(case, "n")
        size = case["B"] * math.prod(ws) * math.prod(grid) * case["C"] * es
        return {"bytes": (8 if case["grad"] else 4) * size, "flops": 0}
    if case["kind"] == "attention":
        _, _, _, nw, n = _attention_geometry(case)
        B, H, hd = case["B"] * nw, case["heads"], case["hd"]
        masks = nw * n * n * es if case["mode"] in ("kept", "new") else 0
        return {"bytes": 4 * B * H * n * hd * es + H * n * n * 4 + masks, "flops": 4 * B * H * n * n * hd}
    if case["kind"] == "block":
        return _block_work(case["B"], tuple(case[a] for a in "dhw"), _triple(case, "ws_"), case["C"],
                           4 if case["x_dtype"] == "fp32" else 2, es)
    dims = tuple(-(-case[a] // 2) for a in "dhw")
    C, B = case["feature"], case["B"]
    tokens = B * math.prod(dims)
    # outputs in the types that autocast leaves them in, weights read once
    total = {"bytes": 4 * 8 * tokens + 4 * tokens * C, "flops": 2 * 8 * tokens * C}
    for _ in range(4):
        ws = tuple(min(7, d) for d in dims)
        block = _block_work(B, dims, ws, C, 4, es)
        tokens = B * math.prod(dims)
        total["flops"] += 2 * (block["flops"] + 16 * tokens * C * C)
        dims = tuple(-(-d // 2) for d in dims)
        tokens = B * math.prod(dims)
        total["flops"] += 2 * tokens * 8 * C * 2 * C
        total["bytes"] += 4 * (2 * 12 * C * C + 16 * C * C) + es * tokens * 2 * C
        C *= 2
    return total


def _block_work(B, dims, ws, C, x_size, es):
    tokens = B * math.prod(dims)
    padded = B * math.prod(-(-d // w) * w for d, w in zip(dims, ws))
    n = math.prod(ws)
    return {"bytes": tokens * C * (x_size + es) + 4 * C * C * es,
            "flops": 8 * tokens * C * C + 4 * padded * n * C}


# ---- how far another correct implementation may be -------------------------


def tolerance(case):
    if case["kind"] == "gather":
        return "exact"
    return _TOLERANCE[case["kind"]][case["dtype"]]


# about four times the largest error against 64 bits seen over the ranges
# above: the rounding of the inputs' products, of the probabilities and of the
# results in the data type (fp32: sums in another order)
_TOLERANCE = {
    "attention": {"fp32": {"rel": 2e-6, "max": 3e-5}, "fp16": {"rel": 1.4e-3, "max": 1.3e-2},
                  "bf16": {"rel": 1e-2, "max": 1e-1}},
    "block": {"fp32": {"rel": 2e-6, "max": 2e-5}, "fp16": {"rel": 2e-3, "max": 2e-2},
              "bf16": {"rel": 1.6e-2, "max": 1.2e-1}},
    "encoder": {"fp32": {"rel": 5e-6, "max": 5e-5}, "fp16": {"rel": 5e-3, "max": 2.5e-2},
                "bf16": {"rel": 3e-2, "max": 1.6e-1}},
}


# ---- the same in 64 bits, in plain torch -----------------------------------


def _windows(x, ws, shift):
    """Cyclic shift and window partition: [B, D, H, W, C] -> [B * nW, N, C]."""
    B, D, H, W, C = x.shape
    x = torch.roll(x, tuple(-v for v in shift), (1, 2, 3))
    x = x.reshape(B, D // ws[0], ws[0], H // ws[1], ws[1], W // ws[2], ws[2], C)
    return x.permute(0, 1, 3, 5, 2, 4, 6, 7).reshape(-1, ws[0] * ws[1] * ws[2], C)


def _volume(windows, B, dims, ws, shift):
    D, H, W = dims
    x = windows.reshape(B, D // ws[0], H // ws[1], W // ws[2], *ws, -1)
    x = x.permute(0, 1, 4, 2, 5, 3, 6, 7).reshape(B, D, H, W, -1)
    return torch.roll(x, tuple(shift), (1, 2, 3))


def _labels(dims, ws, shift):
    """[nW, N] shift-region label of every window token."""
    ax = [torch.where(i < d - w, 0, torch.where(i < d - s, 1, 2)) if s else torch.zeros_like(i)
          for d, w, s, i in ((d, w, s, torch.arange(d, device="cuda")) for d, w, s in zip(dims, ws, shift))]
    ids = (ax[0][:, None, None] * 3 + ax[1][None, :, None]) * 3 + ax[2][None, None, :]
    return _windows(ids[None, ..., None], ws, (0, 0, 0))[..., 0]


def _attend(q, k, v, bias, labels, scale):
    """softmax(q k^T scale + bias + mask) v in 64 bits; labels [nW, N] or None."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    step = max(1, (1 << 27) // (q.shape[1] * q.shape[2] ** 2))
    bias = bias.double()
    for b in range(0, q.shape[0], step):
        at = slice(b, min(q.shape[0], b + step))
        s = (q[at].double() * scale).contiguous() @ k[at].double().transpose(-2, -1).contiguous() + bias
        if labels is not None:
            w = labels[torch.arange(at.start, at.stop, device=q.device) % labels.shape[0]]
            s = s + (w[:, :, None] != w[:, None, :])[:, None] * -100.0
        out[at] = torch.softmax(s, -1) @ v[at].double().contiguous()
    return out


def _msa(x, ln_w, ln_b, eps, wq, bq, wp, bp, bias, hd, ws, shift):
    """The attention half of a Swin block: [B, D, H, W, C] in 64 bits."""
    B, D, H, W, C = x.shape
    a = F.layer_norm(x, (C,), ln_w.double(), ln_b.double(), eps)
    pad = [-n % w for n, w in zip((D, H, W), ws)]
    a = F.pad(a, (0, 0, 0, pad[2], 0, pad[1], 0, pad[0]))
    dims = a.shape[1:4]
    t = _windows(a, ws, shift) @ wq.double().t() + bq.double()
    n = t.shape[1]
    t = t.reshape(-1, n, 3, C // hd, hd).permute(2, 0, 3, 1, 4)
    labels = _labels(dims, ws, shift) if any(shift) else None
    o = _attend(t[0], t[1], t[2], bias, labels, hd ** -0.5)
    o = o.permute(0, 2, 1, 3).reshape(-1, n, C) @ wp.double().t() + bp.double()
    return _volume(o, B, dims, ws, shift)[:, :D, :H, :W]


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "gather":
        windows = _windows(s["x"].detach(), s["ws"], s["shift"]).double()
        out = [windows, s["x"].detach().double()]
        return out + [s["g"].double()] if case["grad"] else out
    if case["kind"] == "attention":
        dims, ws, shift = s["geometry"]
        labels = _labels(dims, ws, shift) if case["mode"] != "none" else None
        out = _attend(s["q"], s["k"], s["v"], s["bias"], labels, case["hd"] ** -0.5)
        return [None, out] if case["mode"] == "new" else [out]
    if case["kind"] == "block":
        norm = s["norm"]
        return [_msa(s["x"].double(), norm.weight, norm.bias, norm.eps, *s["qkv"], *s["proj"], s["bias"], case["hd"],
                     s["ws"], s["shift"])]
    return _encode(s["model"], s["x"].double())


def _encode(model, x):
    """The five features of the Swin encoder (patch 2, windows of 7) in 64 bits."""
    conv = model.patch_embed.proj
    B, _, D, H, W = x.shape
    x = x.reshape(B, D // 2, 2, H // 2, 2, W // 2, 2).permute(0, 1, 3, 5, 2, 4, 6).reshape(B, D // 2, H // 2, W // 2, 8)
    x = x @ conv.weight.double().reshape(conv.weight.shape[0], 8).t() + conv.bias.double()
    outs = [x]
    for i in range(4):
        layer = getattr(model, f"layers{i + 1}")[0]
        dims = x.shape[1:4]
        ws = tuple(min(7, d) for d in dims)
        for j, block in enumerate(layer.blocks):
            shift = tuple(3 if j % 2 and d > 7 else 0 for d in dims)
            a = block.attn
            n = ws[0] * ws[1] * ws[2]
            index = a.relative_position_index[:n, :n].reshape(-1)
            bias = a.relative_position_bias_table.double()[index].reshape(n, n, -1).permute(2, 0, 1)
            C = x.shape[-1]
            x = x + _msa(x, block.norm1.weight, block.norm1.bias, block.norm1.eps, a.qkv.weight, a.qkv.bias,
                         a.proj.weight, a.proj.bias, bias, C // a.num_heads, ws, shift)
            h = F.layer_norm(x, (C,), block.norm2.weight.double(), block.norm2.bias.double(), block.norm2.eps)
            h = F.gelu(h @ block.mlp.linear1.weight.double().t() + block.mlp.linear1.bias.double())
            x = x + h @ block.mlp.linear2.weight.double().t() + block.mlp.linear2.bias.double()
        merge = layer.downsample
        x = F.pad(x, (0, 0, 0, x.shape[3] % 2, 0, x.shape[2] % 2, 0, x.shape[1] % 2))
        order = ((0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (0, 1, 0), (0, 0, 1), (1, 1, 1))
        x = torch.cat([x[:, d::2, h::2, w::2] for d, h, w in order], -1)
        x = F.layer_norm(x, (x.shape[-1],), merge.norm.weight.double(), merge.norm.bias.double(), merge.norm.eps)
        x = x @ merge.reduction.weight.double().t()
        outs.append(x)
    return [F.layer_norm(o, (o.shape[-1],)).permute(0, 4, 1, 2, 3) for o in outs]
