"""jc_c2_layer in JC_F16X3 where its GEMMs split their fp32 A operand themselves (gemm_f32_split.hip with W as
jc_split_f16x3's rows; JITCAST_HIP_GEMM=own takes that path at every size), against the oracle's fp32 layer.

Bar 1e-4 (max relative error), the fp32 layer's: a product is within 2^-20 |a w| + 2^-25 |a| of fp32's, so with
weights of standard deviation 0.02 a GEMM's result is within about 3e-6 of its size.
"""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_stage import MATRICES, TOL, _run_layer
from tests.test_oracle_ops import _layer_weights

pytestmark = pytest.mark.gpu


def _weights(d, inner, dff, bias):
    w = _layer_weights(61 + d, d, inner, dff, bias)
    r = np.random.default_rng(62)
    for k in MATRICES:
        w[k] = (0.02 * r.standard_normal(w[k].shape)).astype(np.float32)
    return w


def _check(oracle, w, x, rows, n, heads, dh, dff):
    live = cases.left_pad_live(63, rows, n, n // 3)
    group = np.sort(np.random.default_rng(64).integers(0, max(1, rows // 2), rows)).astype(np.int32)
    got = _run_layer(x, w, live, group, rows, n, heads, dh, dff, 1e-6, "f16x3")
    exp = oracle.c2_layer(x, w, live, group, rows, n, heads, dh, 1e-6)
    err = oracle.rel_max_error(got, exp)
    print(f"  rel err {err:.3e}", flush=True)
    assert np.isfinite(got).all()
    assert err <= TOL


# tokens around the tiles of 64 and 128 rows, k of 16 mod 32 (a half last stage), n past and below a tile
@pytest.mark.parametrize("rows,n,heads,dh,d,dff,bias", [
    (1, 17, 3, 16, 48, 80, True),
    (5, 13, 5, 16, 80, 144, False),
    (3, 43, 3, 16, 272, 80, True),
    (2, 129, 4, 64, 256, 272, False),
    (16, 129, 12, 64, 768, 3072, True),
])
def test_tile_edges(gpu, oracle, monkeypatch, rows, n, heads, dh, d, dff, bias):
    print(f"case rows={rows} n={n} heads={heads} dh={dh} d={d} dff={dff} bias={bias}", flush=True)
    monkeypatch.setenv("JITCAST_HIP_GEMM", "own")
    x = np.random.default_rng(65).standard_normal((rows * n, d)).astype(np.float32)
    _check(oracle, _weights(d, heads * dh, dff, bias), x, rows, n, heads, dh, dff)


def test_activations_past_the_scale(gpu, oracle, monkeypatch):
    """Normed values that grow by 2^18 after a row's first 32, past what its scale leaves fp16: those tiles are
    computed again from fp32 A and hi + lo of W."""
    monkeypatch.setenv("JITCAST_HIP_GEMM", "own")
    rows, n, heads, dh, d, dff = 3, 33, 4, 16, 64, 128
    w = _weights(d, heads * dh, dff, False)
    w["mlp_norm"] = np.where(np.arange(d) < 32, 1.0, 2.0**18).astype(np.float32)
    x = np.random.default_rng(66).standard_normal((rows * n, d)).astype(np.float32)
    _check(oracle, w, x, rows, n, heads, dh, dff)
