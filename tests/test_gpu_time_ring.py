"""The ring kernel of the bf16/fp16 time attention (time_attention_lpr.hip, 64-wide heads): against float64 at the
edges of its tiles, blocks and workgroups, and against the streaming kernel (JITCAST_HIP_LP_KERNEL=stream) over the
forms the two share: table rows in any order, gates, masks, padded rows of qkv, infinities."""
import numpy as np
import pytest
import torch

from jitcast_amd import chronos2, timestral

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
DH = 64
DTYPES = {"bf16": (torch.bfloat16, 2.0 ** -9), "fp16": (torch.float16, 2.0 ** -12)}  # half an ulp of 1 .. 2


def _qkv(seed, rows, n, inner, dtype):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(rows, n, 3, inner, generator=g, device=DEV) * 0.55).to(dtype)


def _c2(qkv, live, heads, table=None):
    rows, n, _, inner = qkv.shape
    out = torch.full((rows, n, inner), float("nan"), dtype=qkv.dtype, device=DEV)
    chronos2.time_attention(qkv, out, live, rows, n, heads, DH, inner, table)
    torch.cuda.synchronize()
    return out[..., : heads * DH].double()


@pytest.mark.parametrize("dt", sorted(DTYPES))
@pytest.mark.parametrize("n", [33, 63, 64, 65, 128, 129, 200, 256, 257, 288, 290, 320, 385, 513, 545, 577])
def test_edges_against_float64(gpu, n, dt, monkeypatch):
    """4 and 8 waves per workgroup, full and ragged tiles, blocks and halves, a last part of one tile (257, 288, 513,
    545) whose keys six waves share; a left-padded row, one of a single live key, and one without."""
    monkeypatch.setenv("JITCAST_HIP_LP_KERNEL", "wide")
    print(f"case ring {dt} n={n}", flush=True)
    dtype, u = DTYPES[dt]
    rows, heads, inner = 4, 2, 2 * DH + 8
    qkv = _qkv(n, rows, n, inner, dtype)
    live = torch.ones(rows, n, dtype=torch.int32, device=DEV)
    live[1, : n // 2] = 0
    live[2] = 0
    live[2, n - 1] = 1
    live[3] = 0
    got = _c2(qkv, live, heads)
    q, k, v = (t[..., : heads * DH].double().reshape(rows, n, heads, DH).transpose(1, 2).contiguous()
               for t in qkv.unbind(2))
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()).masked_fill(live[:, None, None, :] == 0, -torch.inf)
    exp = torch.nan_to_num(torch.matmul(torch.softmax(s, -1), v)).transpose(1, 2).reshape(rows, n, heads * DH)
    # roundings to the storage type: q times log2(e) (u of scores of some 2.5), P and the result (u each)
    assert float((got[:3] - exp[:3]).norm() / exp[:3].norm()) <= 4.5 * u
    assert (got[3] == 0).all()


@pytest.mark.parametrize("dt", sorted(DTYPES))
@pytest.mark.parametrize("enc,h,gate,shuffled", [(20, 3, False, False), (64, 1, True, True), (190, 9, True, False),
                                                 (256, 1, True, True), (256, 40, False, False), (500, 21, True, True),
                                                 (1024, 1, True, False)])
def test_timestral_against_the_streaming_kernel(gpu, enc, h, gate, shuffled, dt, monkeypatch):
    dtype, u = DTYPES[dt]
    print(f"case ring ts {dt} enc={enc} h={h} gate={gate} shuffled={shuffled}", flush=True)
    rows, heads, n = 3, 2, enc + h
    inner = heads * DH
    r = np.random.default_rng(enc + h)
    qkv = _qkv(enc + h, rows, n, inner, dtype)
    kv = torch.from_numpy((r.random((rows, enc)) < 0.8).astype(np.int32)).to(DEV)
    kv[0, : enc // 3] = 0
    known = torch.tensor([0, 1, 0], dtype=torch.int32, device=DEV)
    pos = np.tile(np.arange(enc, enc + n, dtype=np.int32), (rows, 1))
    if shuffled:
        pos = r.permutation(pos.reshape(-1)).astype(np.int32) - enc // 2
    pos = torch.from_numpy(np.ascontiguousarray(pos.reshape(-1))).to(DEV)
    table = torch.from_numpy(timestral.rope_table(enc, n, DH, 32)).to(DEV)
    g = _qkv(7, rows, n, inner, dtype)[:, :, 0].contiguous() * 4 if gate else None
    outs = []
    for kernel in ("wide", "stream"):
        monkeypatch.setenv("JITCAST_HIP_LP_KERNEL", kernel)
        out = torch.full((rows, n, inner), float("nan"), dtype=dtype, device=DEV)
        timestral.time_attention(qkv, out, kv, known, pos, table, g, rows, enc, enc, n, heads, DH, inner)
        torch.cuda.synchronize()
        outs.append(out.double())
    assert torch.isfinite(outs[0]).all()
    # the same operands; each side rounds its P (against its own reference) and its result
    assert float((outs[0] - outs[1]).norm() / outs[1].norm()) <= 3 * u


@pytest.mark.parametrize("n", [40, 130, 257, 300])
def test_infinities_stay_where_they_are(gpu, n, monkeypatch):
    """An infinite value in the row's last key reaches every query of its row and dim only, and neither a dead key's
    large values nor the next row's first tokens (NaN here) reach any."""
    print(f"case ring infinities n={n}", flush=True)
    rows, heads = 3, 2
    qkv = _qkv(n, rows, n, heads * DH, torch.bfloat16)
    qkv[0, n - 1, 2, 5] = float("inf")
    qkv[1] = float("nan")
    qkv[2, 0, 1] = 1e6  # a dead key's mask is -2^100, added to a score of at most 1e6 * 64 * some 3 * log2(e)
    live = torch.ones(rows, n, dtype=torch.int32, device=DEV)
    live[2, 0] = 0
    outs = []
    for kernel in ("wide", "stream"):  # "wide" is the ring kernel for 64-wide heads
        monkeypatch.setenv("JITCAST_HIP_LP_KERNEL", kernel)
        outs.append(_c2(qkv, live, heads))
    for got in outs:
        assert torch.isinf(got[0, :, 5]).all()
        rest = got[0].clone()
        rest[:, 5] = 0
        assert torch.isfinite(rest).all() and torch.isfinite(got[2]).all()
