"""fp32 activations whose elements lie far apart, through the W8A16 linear with
weights that are zero at the large features: every element of a row counts with at
least 16 significant bits, whatever else the row holds, against a float64 product.

The bound per output: 2^-16 |x| per element (two 16-bit planes of x), and the fp32
sums, a few units of 2^-24 of the sum of magnitudes, within 2^-14 sum |x w s| in all,
plus one rounding of the output.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
ROWS = 70          # more than the 64 rows below which small weights take another kernel


def _one(K, big, small=1.0):
    """One feature of magnitude big, the others N(0, small)."""
    def make(g):
        x = small * torch.randn(ROWS, K, generator=g, device=DEV)
        x[:, K // 3] = big
        return x, torch.arange(K, device=DEV) == K // 3
    return make


def _all_but_one(K, big):
    """One N(0, 1) feature among large ones."""
    def make(g):
        x = big * (1 + torch.rand(ROWS, K, generator=g, device=DEV))
        x[:, 5] = torch.randn(ROWS, generator=g, device=DEV)
        return x, torch.arange(K, device=DEV) != 5
    return make


def _some(K, n, big):
    def make(g):
        x = torch.randn(ROWS, K, generator=g, device=DEV)
        cols = torch.randperm(K, generator=g, device=DEV)[:n]
        x[:, cols] *= big
        large = torch.zeros(K, dtype=torch.bool, device=DEV)
        large[cols] = True
        return x, large
    return make


def _spread(K, sigma):
    """Log-normal magnitudes; the weights are zero at the features of the upper half."""
    def make(g):
        mag = torch.exp(sigma * torch.randn(K, generator=g, device=DEV))
        x = mag * torch.randn(ROWS, K, generator=g, device=DEV)
        return x, mag > mag.median()
    return make


def _sparse(K, n, small):
    """n features of magnitude small among N(0, 1) ones: few far elements per row."""
    def make(g):
        x = torch.randn(ROWS, K, generator=g, device=DEV)
        cols = torch.randperm(K, generator=g, device=DEV)[:n]
        x[:, cols] *= small
        large = torch.ones(K, dtype=torch.bool, device=DEV)
        large[cols] = False
        return x, large
    return make


CASES = {
    "k64_one_1e8": _one(64, 1e8), "k64_one_1e5": _one(64, 1e5), "k64_one_1e18": _one(64, 1e18),
    "k64_all_but_one": _all_but_one(64, 1e8), "k4096_all_but_one": _all_but_one(4096, 1e12),
    "k4096_40_at_1e6": _some(4096, 40, 1e6), "k4096_half_1e5": _some(4096, 2048, 1e5),
    "k4096_half_1e12": _some(4096, 2048, 1e12), "k4096_half_1e20": _some(4096, 2048, 1e20),
    "k1024_lognormal_4": _spread(1024, 4.0), "k1024_lognormal_12": _spread(1024, 12.0),
    "k64_small_1e-15": _sparse(64, 1, 1e-15), "k4096_small_1e-20": _sparse(4096, 3, 1e-20),
    "k20032_small_1e-12": _sparse(20032, 5, 1e-12), "k4096_subnormal": _sparse(4096, 9, 1e-39),
    "k4096_tiny_rows": _one(4096, 1e-20, 1e-27), "k20032_half_1e9": _some(20032, 10016, 1e9),
}


def reference(x, w, s):
    x, w, s = x.double(), w.double().t().contiguous(), s.double()
    return (x @ w) * s, (x.abs() @ w.abs()) * s


def weights(K, N, g):
    w = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int16).to(torch.int8)
    return w, torch.rand(N, generator=g, device=DEV) * 1e-2 + 1e-3


@pytest.mark.parametrize("name", list(CASES))
def test_small_elements_keep_their_bits(name):
    from cublade_amd.bindings.hip.w8a16 import w8a16_linear
    g = torch.Generator(device=DEV).manual_seed(11)
    x, large = CASES[name](g)
    K, N = x.size(1), 200
    w, s = weights(K, N, g)
    w[:, large] = 0
    w[-1] = 0                                   # weight rows of a single code
    w[-1, int((~large).nonzero()[0])] = 127
    print(f"[w8a16 f32 range] {name}", flush=True)
    y = w8a16_linear(x, w, s)
    ref, mag = reference(x, w, s)
    err = (y.double() - ref).abs()
    bound = mag * 2.0 ** -14 + ref.abs() * 2.0 ** -23 + 3e-45   # of subnormal results: their spacing
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("M,N", [(150, 200), (48, 2100)])
def test_rows_of_every_kind_in_one_tile(M, N):
    """Rows with and without far elements, of zeros, of tiny and huge values and with
    infinities and NaN side by side: none changes another's result."""
    from cublade_amd.bindings.hip.w8a16 import w8a16_linear
    K = 4096
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(M, K, generator=g, device=DEV)
    w, s = weights(K, N, g)
    w[:, 100:200] = 0
    x[1::7, 100:200] *= 1e20                     # beside zero codes
    x[2::7] *= 1e-38
    x[3::7, 9] = float("inf")
    x[4::7, 10] = float("nan")
    x[5::7] = 0.0
    x[6::7, 100:200] *= 1e7
    x[1, 7], x[8, 8] = float("inf"), float("nan")
    y = w8a16_linear(x, w, s)
    ref, mag = reference(x, w, s)
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(y.double()[inf], ref[inf])
    ok = torch.isfinite(ref)
    err = (y.double() - ref).abs()[ok]
    bound = mag[ok] * 2.0 ** -14 + ref.abs()[ok] * 2.0 ** -23 + 1e-44
    assert bool((err <= bound).all()), float((err / bound).max())
    for r in (0, 1, 2, 3, 6, 8, 13):
        alone = w8a16_linear(x[r:r + 1].expand(M, K).contiguous(), w, s)[0]
        assert torch.equal(torch.nan_to_num(alone), torch.nan_to_num(y[r])), r
