"""Groups along the last axis are quantized and dequantized in the input's own
shape, without views: codes, scales and values equal those of the 2-D binding on
x.reshape(-1, group_size), and results are plain contiguous tensors also for a
subclass, a parameter, or size-1 dims with odd strides. What the 2-D binding
refuses stays refused."""
from __future__ import annotations

import pytest
import torch

from cublade_amd.bindings.hip.dequantize_int8 import dequantize_per_group_int8
from cublade_amd.bindings.hip.quantize_int8 import quantize_per_group_int8
from cublade_amd.quantization import dequantize_tensor, quantize_tensor

pytestmark = pytest.mark.gpu


class Sub(torch.Tensor):
    pass


@pytest.mark.parametrize("shape,gs", [((7, 96), 32), ((3, 5, 64), 64), ((24,), 8), ((), 1),
                                      ((0, 64), 32), ((4, 0), 32), ((2, 3, 4096), 4096)])
@pytest.mark.parametrize("kind", ["plain", "subclass", "parameter"])
def test_group_last_axis(shape, gs, kind):
    x = torch.randn(shape, device="cuda").bfloat16()
    given = {"plain": lambda: x, "subclass": lambda: x.as_subclass(Sub),
             "parameter": lambda: torch.nn.Parameter(x.clone())}[kind]()
    qt = quantize_tensor(given, mode="group", group_size=gs, ch_axis=-1 if shape else 0)
    q, s = quantize_per_group_int8(x.reshape(-1, gs), gs)
    assert type(qt.data) is torch.Tensor and type(qt.scale) is torch.Tensor
    assert qt.data.shape == x.shape and qt.data.is_contiguous() and not qt.data.requires_grad
    assert torch.equal(qt.data.reshape(-1, gs), q) and torch.equal(qt.scale, s)
    y = dequantize_tensor(qt)
    assert type(y) is torch.Tensor and y.shape == x.shape and y.dtype == torch.bfloat16
    assert torch.equal(y.reshape(-1, gs), dequantize_per_group_int8(q, s, gs))


def test_strides_of_size_one_dims():
    x = torch.randn(64, device="cuda").as_strided((1, 64), (7, 1))
    assert x.is_contiguous()
    for mode, axis in (("tensor", 0), ("channel", 0), ("group", 1)):
        qt = quantize_tensor(x, mode=mode, ch_axis=axis)
        assert qt.data.stride() == (64, 1)


@pytest.mark.parametrize("gs,err", [(8192, RuntimeError), (-32, RuntimeError), (32.0, TypeError),
                                    (48, ValueError), (0, ZeroDivisionError)])
def test_group_last_axis_refuses(gs, err):
    x = torch.randn(2, 8192, device="cuda")
    with pytest.raises(err):
        quantize_tensor(x, mode="group", group_size=gs, ch_axis=1)
