"""The window permutations' native op against their Python autograd function:
values and gradients bit for bit, for contiguous, strided and expanded inputs
and gradients, second derivatives, hooks, empty batches, and the function
transforms that keep the Python path."""

from __future__ import annotations

import pytest
import torch

import crumpet_amd
from crumpet_amd import _WindowPermute, _grid

pytestmark = pytest.mark.gpu

WS, SS, DIMS = (2, 4, 3), (1, 2, 0), (4, 8, 6)


def _volume(B, C, dtype, layout):
    g = torch.Generator(device="cuda").manual_seed(B + C)
    if layout == "strided":
        return torch.randn((B, C, *DIMS), generator=g, device="cuda").to(dtype).permute(0, 2, 3, 4, 1)
    if layout == "expanded":
        return torch.randn((1, *DIMS, C), generator=g, device="cuda").to(dtype).expand(B, *DIMS, C)
    return torch.randn((B, *DIMS, C), generator=g, device="cuda").to(dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,C", [(1, 1), (2, 12), (3, 33), (0, 4)])
@pytest.mark.parametrize("layout", ["contiguous", "strided", "expanded"])
def test_values_and_gradients(dev, dtype, B, C, layout):
    grid = _grid(*DIMS, WS, SS)
    x = _volume(B, C, dtype, layout).detach().requires_grad_()
    w = crumpet_amd.fused_shift_partition_3d(x, WS, SS)
    w_py = _WindowPermute.apply(x, grid, True, B)
    assert torch.equal(w, w_py) and w.requires_grad and w.stride() == w_py.stride()
    y = crumpet_amd.fused_unshift_unpartition_3d(w, B, *DIMS, C, WS, SS)
    assert torch.equal(y, x)
    for out, ref in ((w, w_py), (y, _WindowPermute.apply(w_py, grid, False, B))):
        gout = torch.randn(out.shape[:-1] + (1,), device="cuda").to(dtype).expand(out.shape)
        (gx,) = torch.autograd.grad(out, x, gout, retain_graph=True)
        (gr,) = torch.autograd.grad(ref, x, gout, retain_graph=True)
        assert torch.equal(gx, gr) and gx.stride() == gr.stride()
    with torch.no_grad():
        assert not crumpet_amd.fused_shift_partition_3d(x, WS, SS).requires_grad


def test_second_derivative_hooks_and_streams(dev):
    x = _volume(2, 8, torch.float32, "contiguous").requires_grad_()
    seen = []
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s), torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(1) or t, lambda t: t):
        w = crumpet_amd.fused_shift_partition_3d(x, WS, SS)
        assert not seen  # nothing is saved
        w.register_hook(lambda g: 2 * g)
        (gx,) = torch.autograd.grad((w ** 3).sum(), x, create_graph=True)
        (gg,) = torch.autograd.grad(gx.sum(), x)
    torch.cuda.current_stream().wait_stream(s)
    assert torch.allclose(gx, 6 * x ** 2) and torch.allclose(gg, 24 * x)


def test_function_transforms_as_before(dev):
    x = _volume(2, 8, torch.float32, "contiguous")
    with pytest.raises(RuntimeError):  # no vmap, jvp or grad rule: refused, not wrong
        torch.func.grad(lambda t: crumpet_amd.fused_shift_partition_3d(t, WS, SS).sum())(x)
    with torch.autograd.forward_ad.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        d = torch.autograd.forward_ad.make_dual(x.clone().requires_grad_(), torch.ones_like(x))
        crumpet_amd.fused_shift_partition_3d(d, WS, SS)
