"""The natively computed coarse-to-fine window is the tensor expression it stands for, bit for bit."""
import math

import pytest
import torch

import permutohedral_encoding_amd as pe


@pytest.mark.parametrize("levels", [1, 7, 16, 24, 65])
def test_native_window_is_the_tensor_expression(levels):
    for k in range(200):
        alpha = (k / 150.0) * levels - 0.25
        x = torch.clip(alpha - torch.arange(levels, dtype=torch.float32), 0.0, 1.0)
        assert torch.equal(pe.cosine_easing_window(levels, alpha), 0.5 * (1 + torch.cos(math.pi * x + math.pi)))
    assert torch.equal(pe.cosine_easing_window(levels, torch.tensor(2.5)), pe.cosine_easing_window(levels, 2.5))


def test_window_is_made_on_the_default_device():
    with torch.device("meta"):
        assert pe.cosine_easing_window(8, 2.5).device.type == "meta"
    assert pe.cosine_easing_window(8, 2.5).device.type == "cpu"
