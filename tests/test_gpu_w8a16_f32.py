"""The fp32-activation W8A16 linear on the matrix cores (cbq_w8a16_f32.hip) against
a float64 product of the same codes.

Shapes reach each tile (64 rows x 128 / 256 / 384 columns, 128 x 64 / 128 / 192),
whole and split over K, with partial tiles in M and N, rows that a workgroup does
not hold in registers (K > 16384), and calls of several row chunks. The bound per
output: an element of these rows keeps 21 significant bits or more (two fp16 planes
down to 2^-29 of the row's largest, three bf16 ones for elements outside the row's
band), and the fp32 sums add a few 2^-24 of sum |x w s|; 2^-20 of that sum in all.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def check(x, seed, N, bias=True):
    from cublade_amd.bindings.hip.w8a16 import w8a16_linear
    M, K = x.shape
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int16).to(torch.int8)
    s = torch.rand(N, generator=g, device=DEV) * 1e-2 + 1e-3
    b = torch.randn(N, generator=g, device=DEV) if bias else None
    print(f"[w8a16 f32] M={M} K={K} N={N}", flush=True)
    y = w8a16_linear(x, w, s, b)
    y2 = w8a16_linear(x, w, s, b)
    assert torch.equal(torch.nan_to_num(y), torch.nan_to_num(y2)), "not repeatable"
    ref = (x.double() @ w.double().t().contiguous()) * s.double()
    if b is not None:
        ref = ref + b.double()
    fin = torch.where(torch.isfinite(x.double()), x.double(), torch.zeros((), dtype=torch.float64, device=DEV))
    wa = w.double().abs().t().contiguous()
    bound = (fin.abs() @ wa) * s.double() * 2.0 ** -20 + 1e-6
    ok = torch.isfinite(ref)
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(y.double()[inf], ref[inf])
    err = (y.double() - ref).abs()
    assert bool((err[ok] <= bound[ok]).all()), float((err[ok] / bound[ok]).max())


@pytest.mark.parametrize("M,K,N", [
    (1, 4096, 2100), (16, 11008, 1024), (33, 2048, 4200), (64, 4096, 11008), (64, 8192, 16500),
    (65, 64, 40), (65, 128, 130), (66, 192, 70), (128, 4096, 11008), (129, 1280, 12096),
    (250, 11008, 1024), (500, 1024, 333), (500, 4096, 11008), (1300, 512, 577),
    (70, 16384, 200), (70, 16448, 200), (130, 40000, 64), (2100, 128, 9000)])
def test_f32_tiles(M, K, N):
    x = torch.randn(M, K, generator=torch.Generator(device=DEV).manual_seed(M + K), device=DEV)
    check(x, M * 3 + N, N)


def test_f32_spikes_and_special_rows():
    """Rows of special values and of every range, K = 4096 and M > 64."""
    M, K, N = 150, 4096, 200
    g = torch.Generator(device=DEV).manual_seed(9)
    x = torch.randn(M, K, generator=g, device=DEV)
    x[0] = 0.0
    x[1] = 0.0
    x[1, 77] = 3.5                                  # one-hot
    x[2, 5] = float("nan")
    x[3, 9] = float("inf")
    x[4, 0], x[4, K - 1] = -float("inf"), 1e30
    x[5, 2] = 2.0e36                                # times 127 still an fp32 number
    x[6] = 1e-40                                    # subnormal
    x[7] = 1e30
    x[8] = torch.where(torch.arange(K, device=DEV) % 160 == 0, 1e3, 1e-3)
    x[9, :200] = float("inf")
    x[10] = 1.0
    x[11] = -1.0
    x[12] = torch.exp(4 * torch.randn(K, generator=g, device=DEV))          # heavy tail
    x[13, 4000] = 200.0
    x[149, 1] = -1e6
    check(x, 5, N)
    check(x, 5, N, bias=False)
    check(x[:64].contiguous(), 6, 2048 + 24)        # the 64-row tiles
    xl = torch.randn(70, 16384 * 2 + 64, generator=g, device=DEV)           # rows past the registers
    xl[0, 20000], xl[1, 5], xl[2] = 1e6, float("inf"), 0.0
    check(xl, 8, 60)


@pytest.mark.parametrize("M", [1080, 1500, 2110])
def test_f32_row_chunks(M):
    """K = 40000: 1024 rows per chunk. One chunk with the remainder merged, two, and
    two of which the second is longer; a row with elements outside its band and one
    without in the second; a workspace of exactly the size asked for."""
    from cublade_amd import _abi
    K, N, guard = 40000, 64, 4096
    L = _abi.lib()
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=DEV)
    x[1030, 11], x[1031, 12] = 1e20, 1e6
    w = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int16).to(torch.int8)
    s = torch.rand(N, generator=g, device=DEV) * 1e-2 + 1e-3
    need = L.cbq_w8a16_ws_bytes(M, N, K, 0, _abi.F32)
    ws = torch.zeros(need + guard, dtype=torch.uint8, device=DEV)
    ws[need:] = 0x5a
    y = torch.empty(M, N, device=DEV)
    print(f"[w8a16 f32 chunks] M={M}", flush=True)
    _abi.check(L.cbq_w8a16_linear(_abi.ptr(x), _abi.F32, _abi.ptr(w), _abi.ptr(s), None, None, 0,
                                  None, M, N, K, _abi.ptr(ws), need, _abi.ptr(y),
                                  _abi.stream_handle(x.device)), "chunks")
    assert bool((ws[need:] == 0x5a).all())
    wt = w.double().t().contiguous()
    ref, mag = (x.double() @ wt) * s.double(), (x.double().abs() @ wt.abs()) * s.double()
    # 21 bits per element; K / 16 additions to a sum of one sign (the 1e6 and 1e20
    # rows), each rounded by up to 2^-24 of it, as a random walk with a factor of 4
    bound = mag * (2.0 ** -21 + 4 * (K / 16) ** 0.5 * 2.0 ** -24)
    assert bool(((y.double() - ref).abs() <= bound).all())


def test_f32_distance_from_64_bits():
    """2-norm distance for N(0, 1) rows: the two bf16 planes this replaced were
    4.9e-6 away."""
    from cublade_amd.bindings.hip.w8a16 import w8a16_linear
    M, K, N = 500, 4096, 1000
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(M, K, generator=g, device=DEV)
    w = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int16).to(torch.int8)
    s = torch.ones(N, device=DEV)
    ref = x.double() @ w.double().t().contiguous()
    assert float((w8a16_linear(x, w, s).double() - ref).norm() / ref.norm()) < 5e-7
