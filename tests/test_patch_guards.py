"""When the patched encoder leaves its fused second half, patch merging and
channels-last chain for the eager modules (no GPU needed to decide that)."""

from __future__ import annotations

import pytest
import torch

from crumpet_amd import monai_patch


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
