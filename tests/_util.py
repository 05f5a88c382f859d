"""Helpers shared by the test modules: bit views, device upload, NaN-aware
bit comparisons."""
from __future__ import annotations

import numpy as np
import torch

import oracle

CODE_OF = {torch.float32: oracle.F32, torch.float16: oracle.F16, torch.bfloat16: oracle.BF16}
DTYPE_OF = {v: k for k, v in CODE_OF.items()}


def bits(t: torch.Tensor) -> np.ndarray:
    """Raw bit pattern of a tensor as numpy (uint16 for 16-bit floats, uint8
    for FP8, the native type otherwise)."""
    t = t.detach().cpu().contiguous()
    if t.dtype in (torch.float16, torch.bfloat16):
        return t.view(torch.int16).numpy().view(np.uint16).copy()
    if t.dtype == torch.float8_e4m3fn:
        return t.view(torch.uint8).numpy().copy()
    return t.numpy().copy()


def from_bits(a: np.ndarray, code: int, device="cpu") -> torch.Tensor:
    """Tensor of dtype DTYPE_OF[code] holding the bit pattern ``a``."""
    if code == oracle.F32:
        return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(device)
    t = torch.from_numpy(np.ascontiguousarray(a, np.uint16).view(np.int16))
    return t.view(DTYPE_OF[code]).to(device)


def f16_nan_mask(b: np.ndarray, code: int) -> np.ndarray:
    b = np.asarray(b, np.uint16)
    if code == oracle.BF16:
        return (b & 0x7FFF) > 0x7F80
    return (b & 0x7FFF) > 0x7C00


def assert_bits_equal_16(got: np.ndarray, want: np.ndarray, code: int, what: str = ""):
    """16-bit float outputs equal bit for bit, except that any NaN matches any
    NaN (the NaN payload of a conversion is not part of the contract)."""
    got = np.asarray(got, np.uint16).reshape(-1)
    want = np.asarray(want, np.uint16).reshape(-1)
    assert got.shape == want.shape, what
    nan_w = f16_nan_mask(want, code)
    nan_g = f16_nan_mask(got, code)
    bad = (got != want) & ~(nan_w & nan_g)
    if bad.any():
        i = np.flatnonzero(bad)[:8]
        raise AssertionError(f"{what}: {bad.sum()} of {got.size} differ; first at {i.tolist()}: "
                             f"got {[hex(v) for v in got[i]]} want {[hex(v) for v in want[i]]}")


def assert_fp8_equal(got: np.ndarray, want: np.ndarray, what: str = ""):
    got = np.asarray(got, np.uint8).reshape(-1)
    want = np.asarray(want, np.uint8).reshape(-1)
    assert got.shape == want.shape, what
    nan = ((want & 0x7F) == 0x7F) & ((got & 0x7F) == 0x7F)
    bad = (got != want) & ~nan
    if bad.any():
        i = np.flatnonzero(bad)[:8]
        raise AssertionError(f"{what}: {bad.sum()} of {got.size} FP8 codes differ; first at "
                             f"{i.tolist()}: got {[hex(v) for v in got[i]]} "
                             f"want {[hex(v) for v in want[i]]}")


def assert_array_equal(got, want, what: str = ""):
    got = np.asarray(got).reshape(-1)
    want = np.asarray(want).reshape(-1)
    assert got.shape == want.shape, what
    bad = got != want
    if bad.any():
        i = np.flatnonzero(bad)[:8]
        raise AssertionError(f"{what}: {bad.sum()} of {got.size} differ; first at {i.tolist()}: "
                             f"got {got[i].tolist()} want {want[i].tolist()}")


def assert_scales_equal(got: np.ndarray, want: np.ndarray, what: str = ""):
    assert_array_equal(np.asarray(got, np.float32).view(np.uint32),
                       np.asarray(want, np.float32).view(np.uint32), what + " scale bits")


def _suspect_view(dev: torch.device) -> torch.Tensor:
    """The control block's word at byte 520 (the tag of the last call in which a
    workgroup gave up waiting for the others, or 0) in the stream's workspace."""
    from cublade_amd import _abi
    return _abi._tensor_ws(dev)[520:524].view(torch.int32)


def suspect_word(dev: torch.device) -> int:
    return int(_suspect_view(dev).item())


def set_suspect_word(dev: torch.device, value: int) -> None:
    _suspect_view(dev).fill_(value)


def w8a16_case(M, K, N, n_out, dt, seed, last_outlier=False):
    """Random operands (x, w, s, b, oc, wo) of a W8A16 linear on the GPU, its float64
    result, and a bound on the error per output: one rounding of the output to its
    type plus K fp32 additions. The float64 copies of the weight are made in parts."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K, generator=g, device="cuda").to(dt)
    w = torch.randint(-127, 128, (N, K), generator=g, device="cuda", dtype=torch.int16).to(torch.int8)
    s = (torch.rand(N, generator=g, device="cuda") * 1e-3 + 1e-4).to(dt)
    b = torch.randn(N, generator=g, device="cuda").to(dt)
    oc = wo = None
    if n_out:
        oc = torch.randperm(K, generator=g, device="cuda")[:n_out].sort().values
        if last_outlier:
            oc[-1] = K - 1
        w[:, oc] = 0
        wo = (0.1 * torch.randn(N, n_out, generator=g, device="cuda")).to(dt)
    ref = torch.empty(M, N, dtype=torch.float64, device="cuda")
    mag = torch.empty_like(ref)
    for n0 in range(0, N, 65536):
        p = slice(n0, n0 + 65536)
        wt = w[p].double().t().contiguous()
        ref[:, p] = (x.double() @ wt) * s[p].double() + b[p].double()
        mag[:, p] = (x.double().abs() @ wt.abs()) * s[p].double() + b[p].double().abs()
        if n_out:
            wot = wo[p].double().t().contiguous()
            ref[:, p] += x[:, oc].double() @ wot
            mag[:, p] += x[:, oc].double().abs() @ wot.abs()
    ulp = 2.0 ** (-11 if dt == torch.float16 else -8)
    return (x, w, s, b, oc, wo), ref, ref.abs() * ulp * 1.01 + mag * (K + 8) * 2.0 ** -24 + 1e-6


def assert_within(y, ref, bound):
    err = (y.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
