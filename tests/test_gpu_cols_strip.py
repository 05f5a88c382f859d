"""The one-launch per-column quant for any row length that is a multiple of 8
(k_quant_cols_strip), against the oracle, bit for bit.

Shapes sit at the edges of its geometry on 256 CUs: strips of 64, 32 and 16
chunks of 8 columns with a partial last strip, rows of less than one strip, one
row block (no exchange), blocks of less than one 64-byte step, and x past what
the registers (five steps) and LDS (two steps) of the workgroups hold. Random
data puts the column maxima in random rows, so across the columns each part of
a block holds some maximum.

A workgroup that gives up waiting for the others takes its strip's maxima from
x itself, so with a spin limit of 0 (every workgroup that does not find all the
others at its first poll gives up; every kernel still ends normally) results
stay exact, also on the calls after it.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from cublade_amd import _abi
from tests._util import (
    assert_array_equal, assert_scales_equal, bits, from_bits, set_suspect_word, suspect_word,
)

pytestmark = pytest.mark.gpu

F32, F16, BF16 = oracle.F32, oracle.F16, oracle.BF16
CASES = [
    (1, 8, BF16), (5, 8, F32), (3, 16, F16), (1, 4096, BF16), (2, 264, F16),     # no exchange
    (31, 512, BF16), (32, 512, BF16), (33, 512, F16), (64, 520, BF16), (65, 1000, F32),
    (127, 5120, F16), (128, 5128, BF16), (342, 4736, F32), (1000, 1000, BF16), (777, 40, F16),
    (4099, 64, F32), (3, 131064, BF16), (70, 131072, F16),
    (11008, 4096, BF16), (4096, 11008, F16), (2751, 11008, F32), (20011, 3080, BF16),
    (9000, 8200, F16),                                                           # re-read
]


def make(rows, cols, code, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, cols, generator=g) * torch.exp(torch.randn(1, cols, generator=g))
    x = x.to({F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}[code])
    return bits(x)


def check(xb, rows, cols, code, xt=None):
    from cublade_amd.quantization import quantize_tensor
    qo, so = oracle.quant_int8_channel(xb.reshape(rows, cols), code, axis=1)
    if xt is None:
        xt = from_bits(xb.reshape(-1), code, "cuda").view(rows, cols)
    qt = quantize_tensor(xt, dtype=torch.int8, mode="channel", ch_axis=1)
    assert_array_equal(bits(qt.data), qo, f"codes {rows}x{cols}")
    assert_scales_equal(bits(qt.scale), so, f"scales {rows}x{cols}")


@pytest.mark.parametrize("rows,cols,code", CASES)
def test_cols_strip(rows, cols, code):
    print(f"[strip] {rows}x{cols} code={code}", flush=True)
    check(make(rows, cols, code, rows * 7 + cols), rows, cols, code)


def test_cols_strip_special_values():
    """NaN is ignored and quantizes to 0, infinities saturate, all-zero and
    subnormal columns take eps."""
    rows, cols = 2000, 1544
    x = torch.randn(rows, cols, generator=torch.Generator().manual_seed(3))
    x[5, 3] = float("nan")
    x[:, 9] = float("nan")
    x[1999, 63], x[0, 64] = float("inf"), -float("inf")
    x[:, 512] = 0.0
    x[:, 1543] = 1e-40
    xb = bits(x.to(torch.bfloat16))
    check(xb, rows, cols, BF16)


@pytest.mark.parametrize("rows,cols,code", [(2048, 2048, BF16), (700, 1000, F32),
                                            (11008, 512, F16), (20011, 72, BF16)])
def test_cols_strip_gives_up_exact(rows, cols, code):
    """The control block's suspect word tells that a workgroup gave up (shapes whose
    strips have several row blocks; others need no exchange)."""
    xb = make(rows, cols, code, 17)
    xt = from_bits(xb.reshape(-1), code, "cuda").view(rows, cols)
    dev = xt.device
    check(xb, rows, cols, code, xt)
    default = _abi.set_tensor_spin_limit(0)
    try:
        gave_up = 0
        for i in range(20):
            set_suspect_word(dev, 0)
            check(xb, rows, cols, code, xt)
            gave_up += suspect_word(dev) != 0
            _abi.clear_tensor_quant_status(dev)
    finally:
        _abi.set_tensor_spin_limit(default)
    print("calls in which a workgroup gave up:", gave_up, flush=True)
    assert gave_up > 0
    for _ in range(3):
        check(xb, rows, cols, code, xt)
    assert _abi.tensor_quant_status(dev) == 0
