"""W8A16 tile kernels with a short last k-step (K % 16 == 0, K % 64 != 0,
M > 64): every tile shape, whole and split over K, the short step alone, among
the first three and after the unrolled loop, with and without outlier columns,
against a float64 product of the same operands. The bound: one rounding of the
output to its type plus K fp32 additions."""
from __future__ import annotations

import pytest
import torch

from tests._util import assert_within, w8a16_case

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N,n_out", [
    (65, 16, 40, 0), (130, 48, 300, 2), (65, 80, 520, 0), (200, 144, 130, 3), (70, 208, 1000, 0),
    (256, 272, 700, 0), (256, 4000, 11008, 6), (334, 3312, 12288, 6), (128, 4080, 1024, 0),
    (96, 8208, 512, 1), (700, 1040, 11008, 0), (1536, 464, 11008, 0), (2753, 3440, 421, 0),
    (3415, 560, 1673, 0), (40, 8240, 1024, 0)])
def test_short_last_step(M, K, N, n_out, dt):
    from cublade_amd.bindings.hip.w8a16 import w8a16_linear
    print(f"[w8a16 k tail] M={M} K={K} N={N} n_out={n_out} {dt}", flush=True)
    (x, w, s, b, oc, wo), ref, bound = w8a16_case(M, K, N, n_out, dt, M + K + N)
    y = w8a16_linear(x, w, s, b, oc, wo)
    assert_within(y, ref, bound)
    # rows past the end of x must not matter: the same rows inside a larger batch
    xl = torch.cat([x, torch.full((3, K), float("inf"), dtype=dt, device=DEV)])
    assert torch.equal(w8a16_linear(xl[:M].contiguous(), w, s, b, oc, wo), y)
