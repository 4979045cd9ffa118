"""The fp32 GEMM on fp16 pairs (gemm_f32_split.hip) through jc_linear, against float64.

Bound per element, S = sum |a w|: each operand is held within 2^-22 of itself, or within 2^-25 of its
row's scale (2^-27 of the row's first nonzero stage's maximum M, which the scale brings to 4 to 8), the
lo.lo products left out are at most 2^-22 of S, and fp32 accumulation rounds at most 3k/16 + 3 times.
"""
import numpy as np
import pytest
import torch

from jitcast_amd import chronos2

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _first_stage_max(x):
    """Per row: the maximum of the first 32-column stage that holds a nonzero finite value."""
    m = torch.zeros(x.shape[0], dtype=torch.float64, device=DEV)
    for c in x.double().abs().split(32, dim=1):
        m = torch.where(m == 0, torch.nan_to_num(c, nan=0.0, posinf=0.0).amax(1), m)
    return m


def _bound(a, w, k):
    aa, ww = torch.nan_to_num(a.double().abs(), posinf=0.0), torch.nan_to_num(w.double().abs(), posinf=0.0)
    s = aa @ ww.t()
    return (2.0 ** -20 + (3 * k / 16 + 3) * 2.0 ** -24) * s + 2.0 ** -27 * (
        _first_stage_max(a)[:, None] * ww.sum(1)[None, :] + _first_stage_max(w)[None, :] * aa.sum(1)[:, None])


def _own(monkeypatch):
    monkeypatch.setenv("JITCAST_HIP_GEMM", "own")


# 64-, 128- and 256-row tiles, whole and ragged; k of one half stage, one stage, odd halves, many stages
SHAPES = [(1, 1, 16), (63, 65, 32), (64, 64, 48), (130, 70, 16), (665, 300, 768), (2000, 1100, 48), (2048, 1152, 80),
          (4200, 2100, 48), (4352, 2304, 64), (4353, 2305, 112)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("flags,bias", [(0, True), (chronos2.GEMM_RELU | chronos2.GEMM_ACCUMULATE, False)])
def test_matches_float64(gpu, monkeypatch, m, n, k, flags, bias):
    print(f"case m={m} n={n} k={k} flags={flags}", flush=True)
    _own(monkeypatch)
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a, w = torch.randn(m, k, generator=g, device=DEV), torch.randn(n, k, generator=g, device=DEV)
    b = torch.randn(n, generator=g, device=DEV) if bias else None
    c0 = torch.randn(m, n, generator=g, device=DEV)
    c = c0.clone()
    chronos2.linear(a, w, c, bias=b, flags=flags)
    exp = a.double() @ w.double().t() + (b.double() if bias else 0.0)
    if flags & chronos2.GEMM_RELU:
        exp = exp.relu()
    if flags & chronos2.GEMM_ACCUMULATE:
        exp = exp + c0.double()
    # and the roundings of the bias and accumulate additions
    assert bool(((c.double() - exp).abs() <= _bound(a, w, k) + 2.0 ** -22 * (exp.abs() + 4)).all())


@pytest.mark.parametrize("m,n,k", [(70, 70, 96), (2000, 1100, 64), (4200, 2100, 64)])
def test_rows_of_any_magnitude(gpu, monkeypatch, m, n, k):
    """Rows from 1e-18 to 1e18, some zero throughout and some zero in their first stage, each at its own scale."""
    print(f"case m={m} n={n} k={k}", flush=True)
    _own(monkeypatch)
    g = torch.Generator(device=DEV).manual_seed(k)
    u = lambda r: 10.0 ** (36 * torch.rand(r, 1, generator=g, device=DEV) - 18)  # noqa: E731
    a, w = torch.randn(m, k, generator=g, device=DEV) * u(m), torch.randn(n, k, generator=g, device=DEV) * u(n)
    a[3] = 0
    w[5] = 0
    a[7::50, :32] = 0
    w[9::50, :32] = 0
    c = torch.empty(m, n, device=DEV)
    chronos2.linear(a, w, c)
    exp = a.double() @ w.double().t()
    tiny = 2.0 ** -126  # fp32's own underflow
    assert bool(((c.double() - exp).abs() <= _bound(a, w, k) + tiny).all())
    assert not bool(c[3].any()) and not bool(c[:, 5].any())


@pytest.mark.parametrize("m,n,k", [(70, 70, 96), (2000, 1100, 64), (4200, 2100, 96)])
def test_values_past_the_scale_and_not_finite(gpu, monkeypatch, m, n, k):
    """Rows whose later values pass 2^13 times their first stage (computed again on fp32 MFMA), infinities
    and NaN: every element is what float64 gives, and rows without such values are untouched by them."""
    print(f"case m={m} n={n} k={k}", flush=True)
    _own(monkeypatch)
    g = torch.Generator(device=DEV).manual_seed(k + 1)
    a, w = torch.randn(m, k, generator=g, device=DEV), torch.randn(n, k, generator=g, device=DEV)
    plain = torch.empty(m, n, device=DEV)
    chronos2.linear(a, w, plain)
    a[11, k - 1] = 1e7
    a[12, 40:] *= 3e20
    w[13, k - 2] = -5e8
    a[20, 3], a[21, k - 3], a[22, 5] = float("inf"), float("nan"), -float("inf")
    w[23, k - 5] = float("inf")
    w[24] = 0
    w[24, 0] = 1.0
    c = torch.empty(m, n, device=DEV)
    chronos2.linear(a, w, c)
    exp = (a.double() @ w.double().t()).float()
    assert torch.equal(torch.isnan(c), torch.isnan(exp))
    inf = torch.isinf(exp)
    assert torch.equal(c[inf], exp[inf])
    ok = torch.isfinite(exp)
    # the recomputed elements sum in fp32, one rounding per value of k
    lim = _bound(a, w, k) + k * 2.0 ** -24 * (torch.nan_to_num(a.double().abs(), posinf=0.0) @ torch.nan_to_num(
        w.double().abs(), posinf=0.0).t())
    assert bool(((c.double() - exp.double()).abs()[ok] <= lim[ok] + 2.0 ** -22 * exp.double().abs()[ok]).all())
    rows = [i for i in range(64) if i not in (11, 12, 20, 21, 22)]
    cols = [i for i in range(64) if i not in (13, 23, 24)]
    assert torch.equal(c[rows][:, cols], plain[rows][:, cols])


def test_tile_size_does_not_change_a_row(gpu, monkeypatch):
    """The same rows in a call of 64-row tiles and of 256-row tiles: equal bit for bit."""
    _own(monkeypatch)
    g = torch.Generator(device=DEV).manual_seed(5)
    a, w = torch.randn(4352, 768, generator=g, device=DEV), torch.randn(2304, 768, generator=g, device=DEV)
    big, small = torch.empty(4352, 2304, device=DEV), torch.empty(100, 2304, device=DEV)
    chronos2.linear(a, w, big)
    chronos2.linear(a[1000:1100], w, small)
    assert torch.equal(big[1000:1100], small)


def test_strides(gpu, monkeypatch):
    """lda > k and ldc > n on ragged tiles, and the last row ending where its buffer ends."""
    _own(monkeypatch)
    g = torch.Generator(device=DEV).manual_seed(6)
    buf = torch.randn(299 * 116 + 80, generator=g, device=DEV)
    a = buf.as_strided((300, 80), (116, 1))
    w, c = torch.randn(130, 80, generator=g, device=DEV), torch.full((300, 144), 7.0, device=DEV)
    chronos2.linear(a, w, c, m=300, n=130, k=80, lda=116, ldc=144)
    exp = a.double() @ w.double().t()
    assert bool(((c[:, :130].double() - exp).abs() <= _bound(a, w, 80)).all())
    assert bool((c[:, 130:] == 7.0).all())
