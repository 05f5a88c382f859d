"""W8A16 weight streaming at small M (k_decode) against a float64 product of the
same operands: one, two, three, four, six and eight row tiles per workgroup, each
x chunk width (M <= 4, 8, 16, 32), one and several chunks, a last chunk and a last
128-k block that are not whole, waves without a last block, row and column
tails, outlier columns. The bound: one rounding of the output to its type plus K
fp32 additions."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


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
    g = torch.Generator(device=DEV).manual_seed(M + K + N)
    print(f"[w8a16 decode] M={M} K={K} N={N} n_out={n_out} {dt}", flush=True)
    x = torch.randn(M, K, generator=g, device=DEV).to(dt)
    w = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int16).to(torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) * 1e-3 + 1e-4).to(dt)
    b = torch.randn(N, generator=g, device=DEV).to(dt)
    oc = wo = None
    if n_out:
        oc = torch.randperm(K, generator=g, device=DEV)[:n_out].sort().values
        w[:, oc] = 0
        wo = (0.1 * torch.randn(N, n_out, generator=g, device=DEV)).to(dt)
    ref = torch.empty(M, N, dtype=torch.float64, device=DEV)
    mag = torch.empty_like(ref)
    for n0 in range(0, N, 65536):                     # float64 copies of the weight in parts
        wt = w[n0:n0 + 65536].double().t().contiguous()
        ref[:, n0:n0 + 65536] = x.double() @ wt
        mag[:, n0:n0 + 65536] = x.double().abs() @ wt.abs()
    ref = ref * s.double() + b.double()
    mag = mag * s.double() + b.double().abs()
    if n_out:
        ref = ref + x[:, oc].double() @ wo.double().t().contiguous()
        mag = mag + x[:, oc].double().abs() @ wo.double().abs().t().contiguous()
    y = w8a16_linear(x, w, s, b, oc, wo)
    ulp = 2.0 ** (-11 if dt == torch.float16 else -8)
    bound = ref.abs() * ulp * 1.01 + mag * (K + 8) * 2.0 ** -24 + 1e-6
    err = (y.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
    assert torch.equal(w8a16_linear(x, w, s, b, oc, wo), y)
