"""W8A16 weight streaming at small M (k_decode) against a float64 product of the
same operands: one, two, three, four, six and eight row tiles per workgroup, each
x chunk width (M <= 4, 8, 16, 32), one and several chunks, a last chunk and a last
128-k block that are not whole, waves without a last block, row and column
tails, outlier columns. The bound: one rounding of the output to its type plus K
fp32 additions."""
from __future__ import annotations

import pytest
import torch

from tests._util import assert_within, w8a16_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N,n_out", [
    (1, 2064, 4090, 0), (4, 11008, 4096, 0), (4, 8208, 1100, 2), (3, 40016, 230, 0),   # one tile
    (8, 4096, 2100, 1), (7, 4112, 4096, 0), (5, 14336, 600, 0), (16, 4096, 4096, 0),
    (9, 2048, 4100, 0), (13, 7296, 2969, 3),
    (2, 1040, 8190, 0), (8, 13824, 5120, 0), (16, 10256, 5000, 6), (32, 2064, 6000, 0),   # two
    (1, 5440, 8832, 0), (6, 3000 // 16 * 16, 11000, 1), (15, 944, 9000, 0), (24, 1040, 12000, 0),
    (1, 4096, 14336, 0), (16, 2048, 13001, 0), (17, 4096, 14336, 2), (32, 592, 16000, 0),  # four
    (4, 512, 20000, 0), (12, 2176, 20000, 0), (31, 432, 24000, 1),                        # six
    (2, 320, 32000, 0), (16, 4096, 32000, 6), (32, 512, 40000, 0), (1, 16, 600000, 0)])  # eight
def test_decode(M, K, N, n_out, dt):
    from cublade_amd.bindings.hip.w8a16 import w8a16_linear
    assert N * K >= 8 << 20
    print(f"[w8a16 decode] M={M} K={K} N={N} n_out={n_out} {dt}", flush=True)
    (x, w, s, b, oc, wo), ref, bound = w8a16_case(M, K, N, n_out, dt, M + K + N)
    y = w8a16_linear(x, w, s, b, oc, wo)
    assert_within(y, ref, bound)
    assert torch.equal(w8a16_linear(x, w, s, b, oc, wo), y)
