"""The one-launch per-tensor quant of x up to 2^19 elements
(k_quant_tensor_small), against the oracle, bit for bit: one workgroup up to 2^15
elements, then one per 8192, with every kind of tail and the maximum in the first,
the last and the trailing elements; and under a spin limit of 0 (a workgroup that
gives up waiting takes the maximum from x itself, so results stay exact)."""
from __future__ import annotations

import os

import numpy as np
import pytest
import torch

import oracle
from cublade_amd import _abi
from cublade_amd.bindings.hip.quantize_fp8 import quantize_per_tensor_fp8
from cublade_amd.bindings.hip.quantize_int8 import (
    quantize_per_channel_int8, quantize_per_tensor_int8,
)
from tests._util import (
    assert_array_equal, assert_fp8_equal, assert_scales_equal, bits, from_bits, set_suspect_word,
    suspect_word,
)

pytestmark = pytest.mark.gpu
F32, F16, BF16 = oracle.F32, oracle.F16, oracle.BF16
SIZES = [1, 7, 8, 9, 1000, 8191, 8192, 8193, 32767, 32768, 32769, 40960, 65536, 100003,
         (1 << 19) - 1, 1 << 19, (1 << 19) + 1, (1 << 20) - 1]


def check(n, code, fp8, at, seed=0):
    x = torch.randn(n, generator=torch.Generator().manual_seed(n + seed)) * 0.5
    x[at] = 20.0
    xb = bits(x.to({F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}[code]))
    xt = from_bits(xb, code, "cuda")
    if fp8:
        qo, so = oracle.quant_fp8_tensor(xb, code)
        q, s = quantize_per_tensor_fp8(xt)
        assert_fp8_equal(bits(q), qo, f"n={n}")
    else:
        qo, so = oracle.quant_int8_tensor(xb, code)
        q, s = quantize_per_tensor_int8(xt)
        assert_array_equal(bits(q), qo, f"n={n}")
    assert_scales_equal(bits(s).reshape(-1), np.asarray(so, np.float32).reshape(-1), f"n={n}")


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("code,fp8", [(BF16, True), (F16, True), (BF16, False), (F32, False)])
def test_tensor_small(n, code, fp8):
    for at in {0, n // 2, n - 1}:
        check(n, code, fp8, at)


def test_tensor_small_gives_up_exact():
    """With CUBLADE_CHECK_EXCHANGE=1 as well: an exact call never raises, also
    after a column quant that set the status word. The control block's suspect word
    tells that a workgroup gave up."""
    dev = torch.device("cuda", torch.cuda.current_device())
    default = _abi.set_tensor_spin_limit(0)
    os.environ["CUBLADE_CHECK_EXCHANGE"] = "1"
    try:
        check(65536, BF16, True, 3)
        gave_up = 0
        for i in range(24):
            set_suspect_word(dev, 0)
            check([40960, 65536, 100003, (1 << 19) - 1][i % 4], BF16, i % 2 == 0, 5 + i, seed=i)
            gave_up += suspect_word(dev) != 0
        print("calls in which a workgroup gave up:", gave_up, flush=True)
        assert gave_up > 0
        assert _abi.tensor_quant_status(dev) == 0
        quantize_per_channel_int8(torch.randn(4096, 512, device=dev), axis=1)
        check(65536, BF16, True, 3)
    finally:
        del os.environ["CUBLADE_CHECK_EXCHANGE"]
        _abi.set_tensor_spin_limit(default)
    _abi.clear_tensor_quant_status(dev)
    check(1 << 18, F16, False, 77)
    check(3 << 20, F16, False, 77)          # the large path on the same control block
    assert _abi.tensor_quant_status(dev) == 0
