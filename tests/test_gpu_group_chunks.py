"""Groups of more than 64 rows in the group kernel: their further 64-row query chunks are taken by the
waves of the tiles where the chunks begin. Against the C oracle, at the fp32 bar of 1e-4 (its metric)."""
import numpy as np
import pytest
import torch

from jitcast_amd import chronos2, timestral
from tests import cases

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _i32(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.int32).reshape(-1)).to(DEV)


# the long group first, last, alone, after rows that shift its chunks inside the tiles; a last chunk of one
# row; groups that end where a tile does, with small groups behind the last chunk
SIZES = [(65,), (7, 129), (3, 64, 5, 5), (1, 193, 2, 2, 1), (300,), (16, 128, 16, 4), (5, 5, 6, 257, 3, 1)]


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("dh", [64, 24])
def test_chronos2(gpu, oracle, sizes, dh):
    print(f"case sizes={sizes} dh={dh}", flush=True)
    rows, n, heads = sum(sizes), 3, 5
    inner = heads * dh
    qkv = cases.qkv(61, rows * n, inner)
    live = cases.random_live(61, rows, n, 0.9)
    group = np.repeat(np.arange(len(sizes)), sizes).astype(np.int32)
    s, e = chronos2.group_bounds(group)
    out = torch.full((rows * n, inner), float("nan"), device=DEV)
    chronos2.group_attention(torch.from_numpy(qkv).to(DEV), out, _i32(live), _i32(s), _i32(e), rows, n, heads, dh, inner)
    exp = oracle.c2_group_attention(qkv, live, group, rows, n, heads, dh, inner)
    assert oracle.rel_max_error(out.cpu().numpy(), exp) <= 1e-4


@pytest.mark.parametrize("sizes", [(7, 129), (40, 300, 9)])
@pytest.mark.parametrize("dh", [64, 128])
def test_timestral(gpu, oracle, sizes, dh):
    """128-wide heads take chunks of 32 rows."""
    print(f"case sizes={sizes} dh={dh}", flush=True)
    rows, enc, n, heads = sum(sizes), 2, 3, 2
    d = heads * dh
    qkv = cases.qkv(63, rows * n, d)
    kv = cases.random_live(63, rows, enc, 0.8)
    role = np.random.default_rng(63).integers(0, 3, rows).astype(np.int32)
    group = np.repeat(np.arange(len(sizes)), sizes).astype(np.int32)
    s, e = chronos2.group_bounds(group)
    out = torch.full((rows * n, d), float("nan"), device=DEV)
    timestral.variate_attention(torch.from_numpy(qkv).to(DEV), out, _i32(kv), _i32(s), _i32(e), _i32(role), True, None,
                                rows, enc, n, heads, dh, d)
    exp = oracle.ts_variate_attention(qkv, kv, group, role, 1, rows, enc, n, heads, dh, d)
    assert oracle.rel_max_error(out.cpu().numpy(), exp) <= 1e-4


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_lowp(gpu, oracle, dt):
    sizes = (5, 130, 20, 70)
    rows, n, heads, dh = sum(sizes), 2, 3, 64
    inner = heads * dh
    qkv = torch.from_numpy(cases.qkv(65, rows * n, inner)).to(DEV).to(dt)
    live = cases.random_live(65, rows, n, 0.9)
    group = np.repeat(np.arange(len(sizes)), sizes).astype(np.int32)
    s, e = chronos2.group_bounds(group)
    out = torch.full((rows * n, inner), float("nan"), dtype=dt, device=DEV)
    chronos2.group_attention(qkv, out, _i32(live), _i32(s), _i32(e), rows, n, heads, dh, inner)
    exp = oracle.c2_group_attention(qkv.float().cpu().numpy(), live, group, rows, n, heads, dh, inner)
    assert oracle.rel_max_error(out.float().cpu().numpy(), exp) <= 2 ** -8  # the output's own rounding
