"""fp16 / bf16 W8A16 with rows that are no multiple of 16 (K % 16 != 0): x padded
in the workspace, the weight read unaligned (k_decode, M <= 32 and 8 MB or more)
or padded too, against a float64 product of the same operands; the weight ends at
the end of its buffer, so that nothing may be read past it; and the same call with
a control-block-only workspace (the fp32 FMA kernel). The bound: one rounding of
the output to its type plus K fp32 additions."""
from __future__ import annotations

import pytest
import torch

from tests._util import assert_within, w8a16_case

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N,n_out", [
    (1, 3, 5, 0), (5, 17, 33, 1), (2, 5908, 832, 0), (16, 1458, 700, 2), (40, 1001, 300, 0),
    (1, 4097, 2100, 0), (4, 11002, 4096, 3), (16, 5000, 9000, 0), (32, 4090, 11008, 6),
    (24, 1030, 14001, 0), (9, 515, 33000, 0), (3, 16401, 520, 0), (8, 4111, 2049, 0),
    (70, 4570, 1000, 0), (108, 4570, 7386, 6), (300, 1002, 500, 0), (1500, 250, 1100, 1)])
def test_ragged_rows(M, K, N, n_out, dt):
    from cublade_amd import _abi
    from cublade_amd.bindings.hip.w8a16 import w8a16_linear
    print(f"[w8a16 ragged] M={M} K={K} N={N} n_out={n_out} {dt}", flush=True)
    (x, w, s, b, oc, wo), ref, bound = w8a16_case(M, K, N, n_out, dt, M + K + N, last_outlier=True)
    y = w8a16_linear(x, w, s, b, oc, wo)
    assert_within(y, ref, bound)
    # a workspace without room for the padded rows
    L = _abi.lib()
    ws = torch.zeros(_abi.WS_CTRL_BYTES, dtype=torch.uint8, device=DEV)
    yg = torch.empty_like(y)
    _abi.check(L.cbq_w8a16_linear(_abi.ptr(x), _abi.DTYPE_CODE[dt], _abi.ptr(w), _abi.ptr(s),
                                  _abi.ptr(b), _abi.ptr(oc), n_out, _abi.ptr(wo), M, N, K,
                                  _abi.ptr(ws), ws.numel(), _abi.ptr(yg),
                                  _abi.stream_handle(x.device)), "w8a16")
    assert_within(yg, ref, bound)


@pytest.mark.parametrize("M,K,N,n_out", [(70001, 1002, 67, 2), (40, 1002, 300001, 3)])
def test_ragged_rows_in_parts(M, K, N, n_out):
    """Padded copies past their caps are made in parts: rows of x (66560 and 3441 of
    them), and rows of the weight (266240 and 33761, columns of y), with a workspace
    of exactly the size asked for."""
    from cublade_amd import _abi
    dt, L, guard = torch.float16, _abi.lib(), 4096
    g = torch.Generator(device=DEV).manual_seed(M + N)
    print(f"[w8a16 ragged parts] M={M} K={K} N={N}", flush=True)
    x = torch.randn(M, K, generator=g, device=DEV).to(dt)
    w = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int16).to(torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) * 1e-3 + 1e-4).to(dt)
    b = torch.randn(N, generator=g, device=DEV).to(dt)
    oc = torch.tensor([0, K // 2, K - 1][:n_out], device=DEV)
    w[:, oc] = 0
    wo = (0.1 * torch.randn(N, n_out, generator=g, device=DEV)).to(dt)
    need = L.cbq_w8a16_ws_bytes(M, N, K, n_out, _abi.F16)
    assert need < 400 << 20
    ws = torch.zeros(need + guard, dtype=torch.uint8, device=DEV)
    ws[need:] = 0x5a
    y = torch.empty(M, N, dtype=dt, device=DEV)
    _abi.check(L.cbq_w8a16_linear(_abi.ptr(x), _abi.F16, _abi.ptr(w), _abi.ptr(s), _abi.ptr(b),
                                  _abi.ptr(oc), n_out, _abi.ptr(wo), M, N, K, _abi.ptr(ws), need,
                                  _abi.ptr(y), _abi.stream_handle(x.device)), "w8a16")
    assert bool((ws[need:] == 0x5a).all())
    for n0 in range(0, N, 60000):                    # float64 copies in parts
        p = slice(n0, n0 + 60000)
        wt, wot = w[p].double().t().contiguous(), wo[p].double().t().contiguous()
        ref = (x.double() @ wt) * s[p].double() + b[p].double() + x[:, oc].double() @ wot
        mag = (x.double().abs() @ wt.abs()) * s[p].double() + b[p].double().abs() \
            + x[:, oc].double().abs() @ wot.abs()
        bound = ref.abs() * 2.0 ** -11 * 1.01 + mag * (K + 8) * 2.0 ** -24 + 1e-6
        err = (y[:, p].double() - ref).abs()
        assert bool((err <= bound).all()), float((err / bound).max())
