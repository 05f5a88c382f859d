"""Rows of a multiple of 4 elements that 16-byte loads cannot take, in units of
four (k_rows_sub_any1 / k_deq_rows_sub_any1 with E = 4), against the oracle, bit for
bit: lengths around each lane and slot count, row counts around a workgroup's, the
maximum in the first and the last element, NaN and infinities, and buffers off the
unit's alignment (pairs and single elements there)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from cublade_amd.bindings.hip.dequantize_int8 import dequantize_per_channel_int8
from cublade_amd.bindings.hip.quantize_int8 import quantize_per_channel_int8
from tests._util import (
    CODE_OF, assert_array_equal, assert_bits_equal_16, assert_scales_equal, bits,
)

pytestmark = pytest.mark.gpu
LENGTHS = [4, 12, 20, 36, 60, 68, 100, 124, 132, 252, 260, 508, 516, 1020, 1028, 2044]


def check(x: torch.Tensor, q_offset: int = 0):
    code = CODE_OF[x.dtype]
    qo, so = oracle.quant_int8_channel(bits(x), code, axis=0)
    q, s = quantize_per_channel_int8(x)
    assert_array_equal(bits(q), qo, str(tuple(x.shape)))
    assert_scales_equal(bits(s), so, str(tuple(x.shape)))
    if q_offset:
        buf = torch.empty(q.numel() + q_offset, dtype=torch.int8, device="cuda")
        buf[q_offset:].copy_(q.reshape(-1))
        q = buf[q_offset:].view(q.shape)
    for out in (torch.float16, torch.bfloat16):
        y = dequantize_per_channel_int8(q, s, out)
        assert_bits_equal_16(bits(y), oracle.dequant_int8_channel(qo, so, CODE_OF[out], axis=0),
                             CODE_OF[out], str(tuple(x.shape)))


@pytest.mark.parametrize("L", LENGTHS)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_rows_quad(L, dtype):
    for rows in (1, 33, 1025):
        x = torch.randn(rows, L, generator=torch.Generator().manual_seed(L + rows))
        x[0, 0] = 9.0
        x[-1, -1] = -11.0
        if rows > 5:
            x[1, L // 2] = float("nan")
            x[2, L - 1] = float("inf")
            x[3] = 0.0
        check(x.to(dtype).cuda())


@pytest.mark.parametrize("L", [64, 100, 512, 2044])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_rows_quad_alignment(L, dtype):
    rows = 67
    for offset in (1, 2, 4):
        buf = torch.randn(rows * L + offset, device="cuda").to(dtype)
        check(buf[offset:].view(rows, L), q_offset=offset)
