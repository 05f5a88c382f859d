"""W8A16 tile kernels with a short last k-step (K % 16 == 0, K % 64 != 0,
M > 64): every tile shape, whole and split over K, the short step alone, among
the first three and after the unrolled loop, with and without outlier columns,
against a float64 product of the same operands. The bound: one rounding of the
output to its type plus K fp32 additions."""
from __future__ import annotations

import pytest
import torch

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
    g = torch.Generator(device=DEV).manual_seed(M + K + N)
    print(f"[w8a16 k tail] M={M} K={K} N={N} n_out={n_out} {dt}", flush=True)
    x = torch.randn(M, K, generator=g, device=DEV).to(dt)
    w = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int16).to(torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) * 1e-3 + 1e-4).to(dt)
    b = torch.randn(N, generator=g, device=DEV).to(dt)
    oc = wo = None
    ref = (x.double() @ w.double().t().contiguous()) * s.double() + b.double()
    mag = (x.double().abs() @ w.double().abs().t().contiguous()) * s.double() + b.double().abs()
    if n_out:
        oc = torch.randperm(K, generator=g, device=DEV)[:n_out].sort().values
        w[:, oc] = 0
        wo = (0.1 * torch.randn(N, n_out, generator=g, device=DEV)).to(dt)
        ref = (x.double() @ w.double().t().contiguous()) * s.double() + b.double() \
            + x[:, oc].double() @ wo.double().t().contiguous()
        mag = mag + x[:, oc].double().abs() @ wo.double().abs().t().contiguous()
    y = w8a16_linear(x, w, s, b, oc, wo)
    ulp = 2.0 ** (-11 if dt == torch.float16 else -8)
    bound = ref.abs() * ulp * 1.01 + mag * (K + 8) * 2.0 ** -24 + 1e-6
    err = (y.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
    # rows past the end of x must not matter: the same rows inside a larger batch
    xl = torch.cat([x, torch.full((3, K), float("inf"), dtype=dt, device=DEV)])
    assert torch.equal(w8a16_linear(xl[:M].contiguous(), w, s, b, oc, wo), y)
