"""The natively computed coarse-to-fine window is the tensor expression it stands for, bit for bit."""
import math

import numpy as np
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


def expression(levels, alpha):
    x = torch.clip(alpha - torch.arange(levels, dtype=torch.float32), 0.0, 1.0)
    return 0.5 * (1 + torch.cos(math.pi * x + math.pi))


class Scheduled(torch.nn.Module):
    def __init__(self):
        super().__init__()
        self.window = pe.Coarse2Fine(8)

    def forward(self, x):
        return x * self.window(0.4)


def test_window_in_a_trace():
    want = expression(8, 0.4 * 8)
    assert torch.equal(torch.jit.trace(Scheduled(), torch.ones(8))(torch.ones(8)), want)
    assert torch.equal(torch.fx.experimental.proxy_tensor.make_fx(Scheduled())(torch.ones(8))(torch.ones(8)), want)


def test_window_under_fake_tensors():
    from torch._subclasses import FakeTensor, FakeTensorMode
    with FakeTensorMode():
        window = pe.Coarse2Fine(24)(0.5)
        assert isinstance(window, FakeTensor) and window.shape == (24,) and window.dtype == torch.float32


def test_window_in_a_compiled_module():
    module = torch.compile(Scheduled(), backend="eager", fullgraph=True)
    assert torch.equal(module(torch.ones(8)), expression(8, 0.4 * 8))


def test_window_under_a_dispatch_mode_and_transforms():
    from torch.utils._python_dispatch import TorchDispatchMode

    class Doubling(TorchDispatchMode):  # stands for any mode that computes something else than the operation
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            out = func(*args, **(kwargs or {}))
            return 2 * out if func is torch.ops.aten.cos.default else out

    with Doubling():
        window, want = pe.cosine_easing_window(8, 3.25), expression(8, 3.25)
    assert torch.equal(window, want) and not torch.equal(want, expression(8, 3.25))
    seen = torch.func.functionalize(Scheduled())(torch.ones(8))
    assert torch.equal(seen, expression(8, 0.4 * 8))
    assert torch.equal(torch.vmap(Scheduled())(torch.ones(3, 8)), expression(8, 0.4 * 8).expand(3, 8))


def test_window_without_the_built_library(monkeypatch):
    from permutohedral_encoding_amd import _native
    monkeypatch.setattr(_native, "_lib", None)
    monkeypatch.setattr(_native, "_bridge", None)
    monkeypatch.setattr(_native, "LIB_PATH", _native.LIB_PATH + ".missing")
    assert torch.equal(pe.Coarse2Fine(8)(0.4), expression(8, 0.4 * 8))


@pytest.mark.parametrize("alpha", [0, 3, -2, 1e300, -1e300, math.inf, math.nan, np.float64(2.5), np.float32(2.5), True, 10 ** 30, torch.tensor(1.5), None])
def test_window_takes_and_refuses_what_the_expression_does(alpha):
    try:
        want = expression(6, alpha)
    except Exception as e:
        with pytest.raises(type(e)):
            pe.cosine_easing_window(6, alpha)
    else:
        got = pe.cosine_easing_window(6, alpha)
        assert got.dtype == want.dtype and torch.equal(torch.nan_to_num(got, nan=7.0), torch.nan_to_num(want, nan=7.0))
