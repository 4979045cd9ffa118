"""The fp32 time attention on fp16 pairs (time_attention_f32_split.hip, 64-wide heads) against float64:
the scales of the pairs, the recomputation of what leaves their range, infinities and NaN."""
import numpy as np
import pytest
import torch

from jitcast_amd import chronos2, timestral
from tests.test_gpu_stage import _run_layer
from tests.test_oracle_ops import _layer_weights

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
DH = 64
# (2-norm of the error) / (2-norm of the result): a few roundings of fp32 (2^-24) on the scores, which
# reach some 10 in these cases, and on the sums
TOL = 2e-6


def _qkv(seed, rows, n, heads, std=0.55):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(rows, n, 3, heads, DH, generator=g, device=DEV) * std


def _c2(qkv, live):
    rows, n, _, heads, _ = qkv.shape
    out = torch.full((rows, n, heads, DH), float("nan"), device=DEV)
    chronos2.time_attention(qkv.contiguous(), out, live.int().contiguous(), rows, n, heads, DH, heads * DH, None)
    return out


def _ref(qkv, mask, scale=1.0):
    """qkv [rows, n, 3, heads, dh], mask [rows, n, n] (query, key), in float64."""
    q, k, v = (t.transpose(1, 2).contiguous() for t in qkv.double().unbind(2))
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    p = torch.softmax(s.masked_fill(~mask[:, None], -torch.inf), -1)
    return torch.matmul(p, v).transpose(1, 2)


def _c2_ref(qkv, live):
    return _ref(qkv, (live != 0)[:, None, :].expand(-1, qkv.shape[1], -1))


def _err(got, exp):
    return float((got.double() - exp).norm() / exp.norm())


@pytest.mark.parametrize("n", [1, 31, 33, 64, 128, 129, 133, 161, 513])
@pytest.mark.parametrize("qs,ks,vs", [(1, 1, 1), (1e-14, 1e14, 1e-20), (1e16, 1e-16, 1e20), (3e-8, 3e7, 1e-36)])
def test_scales(gpu, n, qs, ks, vs):
    """Queries, keys and values of any magnitude (their product's fixed): the pairs scale with them."""
    print(f"case n={n} scales {qs} {ks} {vs}", flush=True)
    qkv = _qkv(n, 2, n, 3)
    live = torch.ones(2, n, device=DEV)
    live[0, : n // 3] = 0
    x = qkv * torch.tensor([qs, ks, vs], device=DEV)[:, None, None]
    got = _c2(x, live)
    assert _err(got.double() / vs, _c2_ref(x, live) / vs) <= TOL


@pytest.mark.parametrize("n,zero", [(70, 32), (133, 64), (300, 40)])
def test_leading_zero_blocks(gpu, n, zero):
    """Keys and values that are zero in the first blocks: the scales are set by the first that are not."""
    qkv = _qkv(n, 2, n, 2)
    qkv[0, :zero, 1] = 0
    qkv[1, :zero, 2] = 0
    live = torch.ones(2, n, device=DEV)
    assert _err(_c2(qkv, live), _c2_ref(qkv, live)) <= TOL
    qkv[:, :, 1] = 0  # no key anywhere: the mean of the values
    assert _err(_c2(qkv, live), _c2_ref(qkv, live)) <= TOL
    qkv[:, :, 2] = 0
    assert not bool(_c2(qkv, live).any())


@pytest.mark.parametrize("part,at,factor", [(1, 100, 1e6), (2, 100, 1e7), (2, 132, -1e9), (0, 50, 1e6)])
def test_values_past_the_scale(gpu, part, at, factor):
    """One token's key, value or query far past what its (row, head)'s first block sets: those queries are
    computed again on fp32 MFMA; the other heads and rows come out as without it."""
    n = 133
    qkv, live = _qkv(7, 3, n, 2), torch.ones(3, n, device=DEV)
    plain = _c2(qkv, live)
    qkv[1, at, part, 1] *= factor
    got, exp = _c2(qkv, live), _c2_ref(qkv, live)
    assert bool(torch.isfinite(got).all())
    # scores of 1e6 lose 20 bits of a float's 24 to their size: the softmax of that head is one key's
    tol = TOL if part == 2 else 1e-2
    assert _err(got[1, :, 1], exp[1, :, 1]) <= tol
    others = torch.ones(3, n, 2, dtype=torch.bool, device=DEV)
    others[1, :, 1] = False
    assert torch.equal(got[others], plain[others])


def test_not_finite(gpu):
    """An infinity or NaN in a value reaches the dims it stands in, in a key or query its head; masked keys
    take no part in the scores, whatever they hold."""
    n = 133
    qkv, live = _qkv(9, 4, n, 2), torch.ones(4, n, device=DEV)
    live[3, :40] = 0
    plain = _c2(qkv, live)
    qkv[0, 90, 2, 0, 5] = float("inf")
    qkv[1, 20, 2, 1, 7] = float("nan")
    qkv[2, 60, 0, 1, 3] = float("nan")
    qkv[3, 10, 1, 0, 9] = float("inf")  # a masked key, in a block that live keys share
    got = _c2(qkv, live)
    exp = plain.clone()
    exp[0, :, 0, 5] = float("inf")
    exp[1, :, 1, 7] = float("nan")
    exp[2, 60, 1] = float("nan")
    assert torch.equal(torch.isnan(got), torch.isnan(exp))
    assert torch.equal(torch.isinf(got), torch.isinf(exp))
    ok = torch.isfinite(exp)
    assert float((got[ok].double() - exp[ok].double()).norm() / exp[ok].double().norm()) <= TOL


@pytest.mark.parametrize("enc,h,gate", [(31, 1, True), (128, 5, True), (300, 3, False), (640, 0, True)])
@pytest.mark.parametrize("factor", [1.0, 1e8])
def test_timestral(gpu, enc, h, gate, factor):
    """The causal mask, known rows, decoder queries and the gate; factor: one late value past the scale."""
    print(f"case enc={enc} h={h} gate={gate} factor={factor}", flush=True)
    rows, n, heads = 3, enc + h, 2
    d = heads * DH
    qkv = _qkv(enc, rows, n, heads)
    qkv[1, enc - 3, 2, 1] *= factor
    start = torch.tensor([0, enc // 4, enc // 2], device=DEV)
    kv = torch.arange(enc, device=DEV)[None, :] >= start[:, None]
    known = torch.tensor([0, 1, 0], dtype=torch.int32, device=DEV)
    g = torch.randn(rows, n, heads, DH, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV) if gate else None
    out = torch.full((rows, n, heads, DH), float("nan"), device=DEV)
    timestral.time_attention(qkv, out, kv.int().contiguous(), known, None, None, g, rows, enc, enc, n, heads, DH, d)
    t = torch.arange(n, device=DEV)
    q, k = t[:, None], t[None, :]
    valid = torch.zeros(rows, n, dtype=torch.bool, device=DEV)
    valid[:, :enc] = kv
    ctx = (k < enc) & ((k == q) | (valid[:, None, :] & ((k <= q) | (known[:, None, None] != 0))))
    mask = torch.where(q < enc, ctx, torch.where(k < enc, valid[:, None, :], k <= q))
    exp = _ref(qkv, mask, DH ** -0.5)
    if gate:
        exp = exp * torch.sigmoid(g.double())
    for r in range(rows):
        for hh in range(heads):
            assert _err(out[r, :, hh], exp[r, :, hh]) <= TOL


@pytest.mark.parametrize("n,quiet", [(37, 0), (129, 0), (37, 32), (133, 33), (260, 40)])
def test_split_output(gpu, n, quiet):
    """The split rows that the f16x3 layer's O projection reads, against the fp32 layer. The `quiet` first tokens
    are so small that the scales they set overflow at the others: those queries come from the recomputation."""
    print(f"case f16x3 layer n={n} quiet={quiet}", flush=True)
    rows, heads, d, dff = 3, 2, 64, 128
    r = np.random.default_rng(n + quiet)
    w = _layer_weights(n, d, heads * DH, dff, False)
    x = r.standard_normal((rows, n, d)).astype(np.float32)
    x[:, :quiet] *= 1e-9  # rms norm's eps leaves them at 1e-6 of the others
    live = np.ones((rows, n), np.int32)
    live[1, : n // 4] = 0
    group = np.array([0, 0, 1], np.int32)
    out = [_run_layer(x.reshape(-1, d), w, live, group, rows, n, heads, DH, dff, 1e-6, t).astype(np.float64)
           for t in ("f16x3", None)]
    assert np.isfinite(out[0]).all()
    # three terms of fp16 pairs leave 2^-22 of a product, and at most 2^-25 absolute of a value below fp16's range
    assert np.linalg.norm(out[0] - out[1]) <= 1e-5 * np.linalg.norm(out[1])
