"""The performance cases: what a program that embeds this framework has it do, through the public
entry points of jitcast_amd, at the sizes such programs run.

Kinds of case (a case is a dict of plain values):

  c2_time      chronos2.time_attention: one Chronos-2 time-attention stage (RoPE, padding mask)
  c2_group     chronos2.group_attention: one Chronos-2 cross-series stage
  c2_layer     chronos2.layer: one Chronos-2 encoder layer, as an engine's layer loop calls it
  c2_forecast  HipChronos2Model.forecast: one forward call, raw series in, quantiles out
  ts_time      timestral.time_attention with its output gate
  ts_variate   timestral.variate_attention with roles and its output gate
  ts_block     HipTimestralModel.predict_block: one block, raw series in, quantiles out

The references in exact() are plain torch in 64 bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from jitcast_amd import _lib, chronos2, timestral
from jitcast_amd.chronos2_model import Chronos2Config, HipChronos2Model
from jitcast_amd.timestral_model import HipTimestralModel, TimestralConfig

DEV = "cuda:0"
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
CODE = {"f32": _lib.JC_F32, "bf16": _lib.JC_BF16, "fp16": _lib.JC_F16, "f16x3": _lib.JC_F16X3}
DH, EPS, THETA, PATCH = 64, 1e-6, 10000.0, 16
# a standard deviation of q, k and v: N(0, 1) activations through N(0, 0.02) projections of width 768
QKV_STD = 0.55


def listed() -> list:
    return [
        # 8192-step contexts (512 patches and [REG]) of 256 series, padded on the left by up to half:
        # the attention stage of the longest context the models take, in full and in half precision
        {"name": "time_f32_long", "kind": "c2_time", "dtype": "f32", "rows": 256, "n": 513, "heads": 12, "pad": 0.5},
        {"name": "time_bf16_long", "kind": "c2_time", "dtype": "bf16", "rows": 256, "n": 513, "heads": 12, "pad": 0.5},
        # a middling batch of 3000-step series of uneven age with an 8-patch horizon
        {"name": "time_fp16_mid", "kind": "c2_time", "dtype": "fp16", "rows": 90, "n": 197, "heads": 12, "pad": 0.3},
        # cross-series attention over a large batch of groups of all sizes (one series to sixty-four)
        {"name": "group_f32_mixed", "kind": "c2_group", "dtype": "f32", "rows": 4096, "n": 129, "heads": 12, "lo": 1,
         "hi": 64, "pad": 0.0},
        # the same stage for small groups: four targets and a covariate each
        {"name": "group_bf16_fives", "kind": "c2_group", "dtype": "bf16", "rows": 1300, "n": 133, "heads": 12, "lo": 5,
         "hi": 5, "pad": 0.1},
        # 64 series of 1024 patches and one forecast patch: causal targets with some known covariates
        {"name": "ts_time_bf16", "kind": "ts_time", "dtype": "bf16", "rows": 64, "enc": 1024, "h": 1, "known": 0.25,
         "pad": 0.25},
        # cross-variate attention of a multivariate request: groups of one to six rows with roles
        {"name": "ts_variate_f32", "kind": "ts_variate", "dtype": "f32", "rows": 96, "enc": 256, "h": 4, "lo": 1,
         "hi": 6, "pad": 0.25},
        # one encoder layer of an ordinary forecast call (52 groups of five rows, 2048 steps), by type
        {"name": "layer_f32", "kind": "c2_layer", "dtype": "f32", "rows": 260, "n": 133, "heads": 12, "per": 5},
        {"name": "layer_bf16", "kind": "c2_layer", "dtype": "bf16", "rows": 260, "n": 133, "heads": 12, "per": 5},
        {"name": "layer_f16x3", "kind": "c2_layer", "dtype": "f16x3", "rows": 99, "n": 133, "heads": 12, "per": 3},
        # the smallest request: four univariate series of 512 steps through the 28M-class model
        {"name": "forecast_small_f32", "kind": "c2_forecast", "dtype": "f32", "rows": 4, "steps": 512, "h": 4, "per": 1,
         "heads": 8, "layers": 6},
        # the largest: a block of 64 series of 16,368 steps through the 123M-class model
        {"name": "ts_block_bf16", "kind": "ts_block", "dtype": "bf16", "rows": 64, "patches": 1023, "h": 1, "per": 1,
         "layers": 12},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(["c2_time", "c2_time", "c2_group", "c2_layer", "c2_layer", "c2_forecast", "ts_time", "ts_variate",
                       "ts_block"])
    pad = round(rng.uniform(0.0, 0.5), 2)
    heads = rng.choice([8, 12, 12])
    if kind == "c2_time":
        n = _log(rng, 17, 577)
        return {"kind": kind, "dtype": rng.choice(["f32", "bf16", "fp16"]), "rows": _log(rng, 4, 130000 // n), "n": n,
                "heads": heads, "pad": pad}
    if kind == "c2_group":
        n = _log(rng, 17, 513)
        lo = rng.choice([1, 2, 5])
        return {"kind": kind, "dtype": rng.choice(["f32", "bf16", "fp16"]), "rows": _log(rng, 16, 500000 // n), "n": n,
                "heads": heads, "lo": lo, "hi": _log(rng, lo, 64), "pad": pad}
    if kind == "c2_layer":
        n = _log(rng, 34, 513)
        return {"kind": kind, "dtype": rng.choice(["f32", "f32", "bf16", "fp16", "f16x3"]), "rows": _log(rng, 4, 40000 // n),
                "n": n, "heads": heads, "per": rng.randint(1, 9)}
    if kind == "c2_forecast":
        steps = _log(rng, 256, 8192)
        return {"kind": kind, "dtype": rng.choice(["f32", "f32", "bf16"]), "rows": _log(rng, 1, 12000 // (steps // PATCH)),
                "steps": steps, "h": rng.randint(1, 8), "per": rng.randint(1, 5), "heads": heads,
                "layers": rng.choice([4, 6, 12])}
    if kind == "ts_time":
        enc = _log(rng, 33, 1100)
        return {"kind": kind, "dtype": rng.choice(["f32", "bf16", "fp16"]), "rows": _log(rng, 2, 66000 // enc), "enc": enc,
                "h": rng.randint(0, 8), "known": round(rng.uniform(0.0, 1.0), 2), "pad": pad}
    if kind == "ts_variate":
        enc = _log(rng, 33, 1100)
        lo = rng.choice([1, 1, 3])
        return {"kind": kind, "dtype": rng.choice(["f32", "bf16"]), "rows": _log(rng, 2, 66000 // enc), "enc": enc,
                "h": rng.randint(0, 8), "lo": lo, "hi": _log(rng, lo, 24), "pad": pad}
    patches = _log(rng, 32, 1000)
    dtype = rng.choice(["f32", "bf16"])
    return {"kind": kind, "dtype": dtype, "rows": _log(rng, 1, (12000 if dtype == "f32" else 60000) // patches),
            "patches": patches, "h": rng.randint(1, 4), "per": rng.choice([1, 1, 3]), "layers": rng.choice([2, 6, 12])}


# ---- inputs -------------------------------------------------------------------------------------


def _gen(seed: int, k: int = 0) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed * 1000 + k)


def _normal(g, *shape, std: float = 1.0) -> torch.Tensor:
    return torch.randn(*shape, generator=g, device=DEV) * std


def _i32(a) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32).reshape(-1)).to(DEV)


def _pads(r, rows: int, n: int, share: float) -> np.ndarray:
    """Each row's count of leading padding tokens: uniform up to `share` of the row."""
    return r.integers(0, int(share * n) + 1, rows)


def _groups(r, rows: int, lo: int, hi: int) -> np.ndarray:
    return np.repeat(np.arange(rows), r.integers(lo, hi + 1, rows))[:rows].astype(np.int32)


def _ts_masks(case: dict, seed: int) -> dict:
    """A Timestral block's masks on the host: key validity, known rows, positions, groups and roles."""
    r = np.random.default_rng(seed)
    rows, enc, h = case["rows"], case["enc"], case["h"]
    start = _pads(r, rows, enc, case["pad"])
    kv = (np.arange(enc)[None, :] >= start[:, None]).astype(np.int32)
    pos = np.arange(enc + h)[None, :] - start[:, None]
    m = {"kv": kv, "pos": pos, "known": (r.random(rows) < case.get("known", 0.0)).astype(np.int32)}
    if case["kind"] == "ts_variate":
        m["group"] = _groups(r, rows, case["lo"], case["hi"])
        first = np.r_[True, m["group"][1:] != m["group"][:-1]]
        m["role"] = np.where(first, 0, r.integers(1, 3, rows)).astype(np.int32)
    return m


def _layer_inputs(case: dict, seed: int):
    """x and the fp32 weights of one encoder layer (d_model = heads * 64, d_ff = 4 d_model)."""
    g = _gen(seed)
    d = case["heads"] * DH
    x = _normal(g, case["rows"] * case["n"], d)
    w = {k: _normal(g, o, i, std=0.02) for k, (o, i) in {
        "time_qkv": (3 * d, d), "time_o": (d, d), "group_qkv": (3 * d, d), "group_o": (d, d), "wi": (4 * d, d),
        "wo": (d, 4 * d)}.items()}
    for k in ("time_norm", "group_norm", "mlp_norm"):
        w[k] = 1.0 + _normal(g, d, std=0.1)
    r = np.random.default_rng(seed)
    live = np.arange(case["n"])[None, :] >= _pads(r, case["rows"], case["n"], 0.1)[:, None]
    group = (np.arange(case["rows"]) // case["per"]).astype(np.int32)
    return x, w, live.astype(np.int32), group


def _c2_config(case: dict) -> Chronos2Config:
    d = case["heads"] * DH
    return Chronos2Config(d_model=d, d_kv=DH, d_ff=4 * d, num_layers=case["layers"], num_heads=case["heads"])


def _c2_weights(c: Chronos2Config, seed: int) -> dict:
    g = _gen(seed, 1)
    m = lambda *s: _normal(g, *s, std=0.02)  # noqa: E731
    d, ff, p = c.d_model, c.d_ff, c.patch_size
    w = {"shared": m(2, d), "final_norm": torch.ones(d, device=DEV)}
    for pre, din, dout in (("in", 3 * p, d), ("out", d, c.num_quantiles * p)):
        for part, o, i in (("hidden", ff, din), ("output", dout, ff), ("residual", dout, din)):
            w[f"{pre}_{part}_w"], w[f"{pre}_{part}_b"] = m(o, i), m(o)
    w["layers"] = [{"time_norm": torch.ones(d, device=DEV), "time_qkv": m(3 * d, d), "time_o": m(d, d),
                    "group_norm": torch.ones(d, device=DEV), "group_qkv": m(3 * d, d), "group_o": m(d, d),
                    "mlp_norm": torch.ones(d, device=DEV), "wi": m(ff, d), "wo": m(d, ff)} for _ in range(c.num_layers)]
    return w


def _ts_config(case: dict) -> TimestralConfig:
    return TimestralConfig(layers=((True, False),) * case["layers"])


def _ts_weights(c: TimestralConfig, seed: int) -> dict:
    g = _gen(seed, 2)
    m = lambda *s: _normal(g, *s, std=0.02)  # noqa: E731
    d, p, f = c.d_model, c.patch_size, c.mlp_hidden_dim
    w = {"query": m(d), "out_norm": 1.0 + m(d)}
    for pre, din, dout, bias in (("embed", 2 * p, d, True), ("head", d, p * c.num_quantiles, False)):
        for part, o, i in (("hidden", 4 * d, din), ("output", dout, 4 * d), ("residual", dout, din)):
            w[f"{pre}_{part}_w"] = m(o, i)
            if bias:
                w[f"{pre}_{part}_b"] = m(o)
    w["layers"] = [{"attentions": [{"time": t, "norm": 1.0 + m(d), "qkv": m(3 * d, d), "gate": m(d, d), "wo": m(d, d)}
                                   for t in axes], "mlp_norm": 1.0 + m(d), "up": m(2 * f, d), "down": m(d, f)}
                   for axes in c.layers]
    return w


def _host(w):
    """The weights as numpy arrays, the form a checkpoint loads into."""
    if isinstance(w, dict):
        return {k: _host(v) for k, v in w.items()}
    if isinstance(w, list):
        return [_host(v) for v in w]
    return w.cpu().numpy() if isinstance(w, torch.Tensor) else w


def _series(seed: int, rows: int, steps: int) -> np.ndarray:
    """Daily and weekly cycles, a slow trend and noise, per series."""
    r = np.random.default_rng(seed)
    t = np.arange(steps, dtype=np.float64)
    a = r.uniform(0.5, 2.0, (rows, 2))
    x = a[:, :1] * np.sin(2 * np.pi * t / 24) + a[:, 1:] * np.sin(2 * np.pi * t / 168)
    return (x + r.uniform(-0.01, 0.01, (rows, 1)) * t + r.normal(0, 0.1, (rows, steps))).astype(np.float32)


def _c2_request(case: dict, seed: int):
    """A forecast call's raw rows: NaN before each series began, and one known covariate per group."""
    r = np.random.default_rng(seed + 1)
    rows, steps, per, h = case["rows"], case["steps"], case["per"], case["h"]
    x = _series(seed, rows, steps)
    x[np.arange(steps)[None, :] < _pads(r, rows, steps, 0.2)[:, None]] = np.nan
    group = (np.arange(rows) // per).astype(np.int32)
    fut = None
    if per > 1:
        fut = np.full((rows, h * PATCH), np.nan, np.float32)
        last = np.r_[group[1:] != group[:-1], True]
        fut[last] = r.normal(0, 1, (int(last.sum()), h * PATCH))
    return x, group, fut


def _ts_request(case: dict, seed: int):
    """A block's raw rows: leading patches unobserved, a few steps missing, rows of one series together
    (its target, a past covariate, a known covariate)."""
    r = np.random.default_rng(seed + 1)
    rows, per, h = case["rows"], case["per"], case["h"]
    t = case["patches"] * PATCH
    x = _series(seed, rows, t)
    obs = np.arange(t)[None, :] >= (_pads(r, rows, case["patches"], 0.25) * PATCH)[:, None]
    obs &= r.random((rows, t)) >= 0.02
    x = np.where(obs, x, np.float32(0))
    group = (np.arange(rows) // per).astype(np.int32)
    if per == 1 or rows == 1:
        return x, obs, group, None, None, None
    role = (np.arange(rows) % per).astype(np.int32)
    fut = r.normal(0, 1, (rows, h * PATCH)).astype(np.float32) * (role == 2)[:, None]
    return x, obs, group, role, fut.astype(np.float32), np.broadcast_to((role == 2)[:, None], fut.shape).copy()


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    s = {"case": case}
    if kind in ("c2_time", "c2_group"):
        rows, n, d = case["rows"], case["n"], case["heads"] * DH
        r = np.random.default_rng(seed)
        std = QKV_STD if kind == "c2_time" else 1.0
        s["qkv"] = _normal(_gen(seed), rows * n, 3 * d, std=std).to(TORCH[case["dtype"]])
        live = np.arange(n)[None, :] >= _pads(r, rows, n, case["pad"])[:, None]
        live[:, n - 1] = True
        s["live"] = _i32(live)
        s["out"] = torch.empty(rows * n, d, dtype=s["qkv"].dtype, device=DEV)
        if kind == "c2_time":
            s["table"] = torch.from_numpy(chronos2.rope_table(n, DH)).to(DEV)
        else:
            s["group"] = _groups(r, rows, case["lo"], case["hi"])
            s["gs"], s["ge"] = (_i32(b) for b in chronos2.group_bounds(s["group"]))
    elif kind == "c2_layer":
        x, w, live, group = _layer_inputs(case, seed)
        rows, n, d = case["rows"], case["n"], case["heads"] * DH
        for k in ("time_qkv", "time_o", "group_qkv", "group_o", "wi", "wo"):
            if case["dtype"] == "f16x3":
                t = torch.empty(w[k].shape[0], 3 * w[k].shape[1], dtype=torch.float16, device=DEV)
                chronos2.split_f16x3(w[k], t, weights=True)
                w[k] = t
            elif case["dtype"] != "f32":
                t = torch.empty(w[k].shape, dtype=TORCH[case["dtype"]], device=DEV)
                chronos2.to_lp(w[k], t)
                w[k] = t
        s.update(x0=x, x=torch.empty_like(x), w=w, live=_i32(live), table=torch.from_numpy(chronos2.rope_table(n, DH)).to(DEV))
        s["gs"], s["ge"] = (_i32(b) for b in chronos2.group_bounds(group))
        s["ws"] = torch.empty(chronos2.layer_workspace_bytes(rows, n, d, d, 4 * d, CODE[case["dtype"]]) // 4 + 64, device=DEV)
    elif kind in ("ts_time", "ts_variate"):
        rows, enc, n, d = case["rows"], case["enc"], case["enc"] + case["h"], 768
        m = _ts_masks(case, seed)
        dt = TORCH[case["dtype"]]
        s["qkv"] = _normal(_gen(seed), rows * n, 3 * d, std=QKV_STD).to(dt)
        s["gate"] = _normal(_gen(seed, 3), rows * n, d, std=QKV_STD).to(dt)
        s["out"] = torch.empty(rows * n, d, dtype=dt, device=DEV)
        s["kv"] = _i32(m["kv"])
        if kind == "ts_time":
            s["known"], s["pos"] = _i32(m["known"]), _i32(m["pos"] + enc)
            s["table"] = torch.from_numpy(timestral.rope_table(enc, n, DH, DH // 2)).to(DEV)
        else:
            s["role"] = _i32(m["role"])
            s["gs"], s["ge"] = (_i32(b) for b in chronos2.group_bounds(m["group"]))
    elif kind == "c2_forecast":
        c = _c2_config(case)
        s["model"] = HipChronos2Model(c, _host(_c2_weights(c, seed)), dtype=case["dtype"], max_plans=8)
        s["request"] = _c2_request(case, seed)
    else:
        c = _ts_config(case)
        s["model"] = HipTimestralModel(c, _host(_ts_weights(c, seed)), dtype=case["dtype"])
        s["request"] = _ts_request(case, seed)
    return s


def run(s: dict):
    c = s["case"]
    kind = c["kind"]
    if kind == "c2_time":
        d = c["heads"] * DH
        chronos2.time_attention(s["qkv"], s["out"], s["live"], c["rows"], c["n"], c["heads"], DH, d, s["table"])
        return s["out"]
    if kind == "c2_group":
        d = c["heads"] * DH
        chronos2.group_attention(s["qkv"], s["out"], s["live"], s["gs"], s["ge"], c["rows"], c["n"], c["heads"], DH, d)
        return s["out"]
    if kind == "c2_layer":  # in place on the residual stream, which the stage before has just written
        d = c["heads"] * DH
        s["x"].copy_(s["x0"])
        chronos2.layer(s["x"], s["w"], s["live"], s["table"], s["gs"], s["ge"], s["ws"], c["rows"], c["n"], d, c["heads"],
                       DH, 4 * d, EPS, CODE[c["dtype"]])
        return s["x"]
    if kind == "ts_time":
        timestral.time_attention(s["qkv"], s["out"], s["kv"], s["known"], s["pos"], s["table"], s["gate"], c["rows"],
                                 c["enc"], c["enc"], c["enc"] + c["h"], 12, DH, 768)
        return s["out"]
    if kind == "ts_variate":
        timestral.variate_attention(s["qkv"], s["out"], s["kv"], s["gs"], s["ge"], s["role"], True, s["gate"], c["rows"],
                                    c["enc"], c["enc"] + c["h"], 12, DH, 768)
        return s["out"]
    if kind == "c2_forecast":
        x, group, fut = s["request"]
        return s["model"].forecast(x, group, fut, h=c["h"])
    x, obs, group, role, fut, fut_obs = s["request"]
    return s["model"].predict_block(x, obs, group, c["h"], role, fut, fut_obs)


# ---- the work a pass cannot do without ------------------------------------------------------------


def work(case: dict) -> dict:
    kind = case["kind"]
    size = 4 if case["dtype"] in ("f32", "f16x3") else 2
    if kind in ("c2_time", "c2_group"):
        rows, n, d = case["rows"], case["n"], case["heads"] * DH
        keys = n * (1 - case["pad"] / 2) if kind == "c2_time" else (case["lo"] + case["hi"]) / 2
        return {"bytes": 4.0 * rows * n * d * size + 4.0 * rows * n, "flops": 4.0 * rows * n * d * keys}
    if kind in ("ts_time", "ts_variate"):
        rows, n, d = case["rows"], case["enc"] + case["h"], 768
        live = n * (1 - case["pad"] / 2)
        keys = live * (0.5 + 0.5 * case.get("known", 0)) if kind == "ts_time" else (case["lo"] + case["hi"]) / 2
        return {"bytes": 5.0 * rows * n * d * size + 8.0 * rows * n, "flops": 4.0 * rows * n * d * keys}
    if kind == "c2_layer":
        tokens, d = case["rows"] * case["n"], case["heads"] * DH
        return {"bytes": 8.0 * tokens * d + 16.0 * d * d * size,
                "flops": tokens * (2.0 * 16 * d * d + 4.0 * d * (case["n"] * 0.95 + case["per"]))}
    if kind == "c2_forecast":
        c = _c2_config(case)
        nc, h, d = -(-case["steps"] // PATCH), case["h"], c.d_model
        n, q = nc + 1 + h, c.num_quantiles * PATCH
        flops = case["rows"] * c.num_layers * n * (2.0 * 16 * d * d + 4.0 * d * (n + case["per"]))
        flops += 2.0 * case["rows"] * ((nc + h) * (4 * d * (48 + d) + 48 * d) + h * (4 * d * (d + q) + d * q))
        weights = 16.0 * d * d * c.num_layers * size + 16.0 * d * (48 + 2 * d + q) + 4.0 * d * (48 + q)
        return {"bytes": weights + 4.0 * case["rows"] * (case["steps"] + h * q), "flops": flops}
    c = _ts_config(case)
    d, f, q = c.d_model, c.mlp_hidden_dim, c.num_quantiles * PATCH
    cov = case["per"] > 1 and case["rows"] > 1
    enc = case["patches"] + (case["h"] if cov else 0)
    n = enc + case["h"]
    flops = case["rows"] * len(c.layers) * n * (2.0 * (10 * d * d + 3 * f * d) + 4.0 * d * (n * 0.44 + case["per"]))
    flops += 2.0 * case["rows"] * (enc * (4 * d * (32 + d) + 32 * d) + case["h"] * (4 * d * (d + q) + d * q))
    weights = (10.0 * d * d + 3 * f * d) * len(c.layers) * size + 16.0 * d * (32 + 2 * d + q) + 4.0 * d * (32 + q)
    return {"bytes": weights + 5.0 * case["rows"] * case["patches"] * PATCH + 4.0 * case["rows"] * case["h"] * q,
            "flops": flops}


# (rel, max) per kind and type: about four times what the outputs of seeded cases over these ranges
# were off from exact() (f32 kinds 1e-7 to 1.6e-6; 16-bit outputs their type's rounding of the scores'
# operands and the result; the whole calls what twelve such layers add up to)
TOLERANCE = {
    "c2_time": {"f32": (4e-6, 1e-4), "bf16": (2e-2, 0.4), "fp16": (2.5e-3, 5e-2)},
    "c2_group": {"f32": (2e-6, 1e-4), "bf16": (6e-3, 2e-2), "fp16": (8e-4, 2.5e-3)},
    "ts_time": {"f32": (2e-6, 4e-5), "bf16": (1e-2, 0.1), "fp16": (1.2e-3, 1.5e-2)},
    "ts_variate": {"f32": (6e-7, 1e-5), "bf16": (6e-3, 2e-2)},
    "c2_layer": {"f32": (2e-6, 2e-5), "f16x3": (3.5e-6, 3e-5), "bf16": (8e-3, 5e-2), "fp16": (1e-3, 8e-3)},
    "c2_forecast": {"f32": (3.5e-6, 3e-5), "bf16": (1.5e-2, 0.15)},
    "ts_block": {"f32": (6.4e-6, 3e-5), "bf16": (1.5e-2, 0.1)},
}


def tolerance(case: dict) -> dict:
    rel, most = TOLERANCE[case["kind"]][case["dtype"]]
    return {"rel": rel, "max": most}


# ---- the same in 64 bits --------------------------------------------------------------------------


def _rope64(x: torch.Tensor, pos: np.ndarray, rope_dim: int) -> torch.Tensor:
    """x [rows, n, heads, dh] rotated at pos [rows or 1, n]: the angles round to float, as the models define."""
    e = np.zeros(DH // 2, np.float32)
    for i in range(rope_dim // 2):
        e[i] = np.float32(1.0) / np.float32(float(THETA) ** float(np.float32(2 * i) / np.float32(rope_dim)))
    ang = torch.from_numpy((pos.astype(np.float32)[..., None] * e).astype(np.float64)).to(x.device)[:, :, None, :]
    a, b = x[..., : DH // 2], x[..., DH // 2:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], dim=-1)


def _attend64(q, k, v, mask, scale: float) -> torch.Tensor:
    """q, k, v [..., L, dh]; mask [..., L, L] (query, key); rows without a key give zeros."""
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    p = torch.softmax(s.masked_fill(~mask, -torch.inf), dim=-1)
    return torch.matmul(torch.nan_to_num(p, nan=0.0), v)


def _split64(qkv: torch.Tensor, rows: int, n: int):
    return qkv.double().view(rows, n, 3, -1, DH).unbind(2)


def _time64(qkv, mask_of, pos: np.ndarray, rope_dim: int, scale: float, rows: int, n: int) -> torch.Tensor:
    out = []
    step = max(1, int(3e8 // (n * n * qkv.shape[1] // (3 * DH))))
    for r in range(0, rows, step):
        m = min(step, rows - r)
        q, k, v = _split64(qkv[r * n:(r + m) * n], m, n)
        ps = pos[r:r + m] if pos.shape[0] > 1 else pos
        q, k = (_rope64(t, ps, rope_dim).transpose(1, 2).contiguous() for t in (q, k))
        out.append(_attend64(q, k, v.transpose(1, 2).contiguous(), mask_of(r, r + m)[:, None], scale).transpose(1, 2)
                   .reshape(m * n, -1))
    return torch.cat(out)


def _c2_time64(qkv, live: torch.Tensor, rows: int, n: int) -> torch.Tensor:
    mask = lambda a, b: (live.view(rows, 1, n)[a:b] != 0).expand(b - a, n, n)  # noqa: E731
    return _time64(qkv, mask, np.arange(n)[None, :], DH, 1.0, rows, n)


def _group64(qkv, group: np.ndarray, mask_of, scale: float, rows: int, n: int) -> torch.Tensor:
    """Attention across the rows of each (contiguous) group at every slot, groups of one size together.
    mask_of(rows [G, s]) -> bool [G, n, s, s]."""
    q, k, v = _split64(qkv, rows, n)
    out = torch.zeros(rows, n, q.shape[2], DH, dtype=torch.float64, device=DEV)
    starts = np.flatnonzero(np.r_[True, group[1:] != group[:-1]])
    sizes = np.diff(np.r_[starts, rows])
    for s in np.unique(sizes):
        st = starts[sizes == s]
        step = max(1, int(5e7 // (s * n * q.shape[2] * DH)))
        for i in range(0, len(st), step):
            idx = torch.from_numpy(st[i:i + step, None] + np.arange(s)[None, :]).to(DEV)
            pick = lambda t: t[idx].permute(0, 2, 3, 1, 4).contiguous()  # noqa: E731
            o = _attend64(pick(q), pick(k), pick(v), mask_of(idx)[:, :, None], scale)
            out[idx] = o.permute(0, 3, 1, 2, 4)
    return out.view(rows * n, -1)


def _c2_group64(qkv, live: torch.Tensor, group: np.ndarray, rows: int, n: int) -> torch.Tensor:
    lv = live.view(rows, n) != 0
    return _group64(qkv, group, lambda i: lv[i].permute(0, 2, 1)[:, :, None, :].expand(-1, -1, i.shape[1], -1), 1.0, rows, n)


def _ts_time64(qkv, kv, known, pos: np.ndarray, rows: int, enc: int, ll: int, n: int) -> torch.Tensor:
    t = torch.arange(n, device=DEV)
    q, k = t[:, None], t[None, :]
    valid = torch.zeros(rows, n, dtype=torch.bool, device=DEV)
    valid[:, :enc] = kv.view(rows, enc) != 0

    def mask(a, b):
        val, kn = valid[a:b, None, :], known[a:b, None, None] != 0
        ctx = (k < enc) & ((k == q) | (val & ((k <= q) | kn)))
        return torch.where(q < enc, ctx, torch.where(k < enc, (k < ll) & val, k <= q))

    return _time64(qkv, mask, pos, DH // 2, DH ** -0.5, rows, n)


def _ts_variate64(qkv, kv, group: np.ndarray, role, rows: int, enc: int, n: int) -> torch.Tensor:
    valid = torch.ones(rows, n, dtype=torch.bool, device=DEV)
    valid[:, :enc] = kv.view(rows, enc) != 0

    def mask(i):
        m = valid[i].permute(0, 2, 1)[:, :, None, :].expand(-1, -1, i.shape[1], -1)
        if role is not None:
            rq, rk = role[i][:, :, None], role[i][:, None, :]
            m = m & ~(((rq != 0) & (rk == 0)) | ((rq == 2) & (rk != 2)))[:, None]
        return m | torch.eye(i.shape[1], dtype=torch.bool, device=DEV)

    return _group64(qkv, group, mask, DH ** -0.5, rows, n)


def _rms64(x, w, eps: float = EPS):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _lin64(x, w, b=None):
    y = torch.cat([p @ w.double().t() for p in x.split(65536)])
    return y if b is None else y + b.double()


def _c2_layer64(x, w: dict, live, group: np.ndarray, rows: int, n: int) -> torch.Tensor:
    x = x + _lin64(_c2_time64(_lin64(_rms64(x, w["time_norm"]), w["time_qkv"]), live, rows, n), w["time_o"])
    x = x + _lin64(_c2_group64(_lin64(_rms64(x, w["group_norm"]), w["group_qkv"]), live, group, rows, n), w["group_o"])
    return x + _lin64(torch.relu(_lin64(_rms64(x, w["mlp_norm"]), w["wi"])), w["wo"])


def _residual64(x, w: dict, pre: str, act) -> torch.Tensor:
    g = lambda k: (w[f"{pre}_{k}_w"], w.get(f"{pre}_{k}_b"))  # noqa: E731
    return _lin64(act(_lin64(x, *g("hidden"))), *g("output")) + _lin64(x, *g("residual"))


def _c2_forecast64(case: dict, seed: int) -> torch.Tensor:
    c = _c2_config(case)
    w = _c2_weights(c, seed)
    x, group, fut = _c2_request(case, seed)
    rows, steps, h = case["rows"], case["steps"], case["h"]
    nc = -(-steps // PATCH)
    n = nc + 1 + h
    win = torch.full((rows, nc * PATCH), torch.nan, dtype=torch.float64, device=DEV)
    win[:, nc * PATCH - steps:] = torch.from_numpy(x).to(DEV).double()
    fu = torch.full((rows, h * PATCH), torch.nan, dtype=torch.float64, device=DEV)
    if fut is not None:
        fu[:] = torch.from_numpy(fut).to(DEV).double()
    obs = ~win.isnan()
    cnt = obs.sum(1, keepdim=True).clamp(min=1)
    loc = torch.nan_to_num(win).sum(1, keepdim=True) / cnt
    scale = (torch.where(obs, win - loc, 0.0).square().sum(1, keepdim=True) / cnt).sqrt()
    seq = torch.cat([win, fu], 1)
    time = (torch.arange((nc + h) * PATCH, device=DEV) - nc * PATCH).double() / c.time_encoding_scale
    val = torch.nan_to_num(torch.asinh((seq - loc) / scale), nan=0.0)
    tok = torch.stack([time.expand(rows, -1), val, (~seq.isnan()).double()], 1).view(rows, 3, nc + h, PATCH)
    emb = _residual64(tok.permute(0, 2, 1, 3).reshape(rows * (nc + h), 3 * PATCH), w, "in", torch.relu)
    emb = emb.view(rows, nc + h, -1)
    reg = w["shared"][1].double().expand(rows, 1, -1)
    live = torch.ones(rows, n, dtype=torch.int32, device=DEV)
    live[:, :nc] = obs.view(rows, nc, PATCH).any(-1).int()
    y = torch.cat([emb[:, :nc], reg, emb[:, nc:]], 1).reshape(rows * n, -1)
    for lw in w["layers"]:
        y = _c2_layer64(y, lw, live, group, rows, n)
    dec = _rms64(y, w["final_norm"]).view(rows, n, -1)[:, nc + 1:].reshape(rows * h, -1)
    raw = _residual64(dec, w, "out", torch.relu).view(rows, h, c.num_quantiles, PATCH)
    return torch.sinh(raw).permute(0, 2, 1, 3).reshape(rows, c.num_quantiles, h * PATCH) * scale[..., None] + loc[..., None]


def _ts_block64(case: dict, seed: int) -> torch.Tensor:
    c = _ts_config(case)
    w = _ts_weights(c, seed)
    x, obs, group, role, fut, fut_obs = _ts_request(case, seed)
    rows, t, h = case["rows"], x.shape[1], case["h"]
    ll = t // PATCH
    win, ob = torch.from_numpy(x).to(DEV).double(), torch.from_numpy(obs).to(DEV)
    if role is not None:
        win = torch.cat([win, torch.from_numpy(fut).to(DEV).double()], 1)
        ob = torch.cat([ob, torch.from_numpy(fut_obs).to(DEV)], 1)
    enc = win.shape[1] // PATCH
    n = enc + h
    known = torch.zeros(rows, dtype=torch.int32, device=DEV) if role is None else (_i32(role) == 2).int()
    # the causal scaler: a running mean and Welford's sum of squares, read at each patch's last step
    wt = ob.double()
    cum = wt.cumsum(1)
    mean = (wt * win).cumsum(1) / cum.clamp(min=1.0)
    prev = torch.cat([torch.zeros(rows, 1, dtype=torch.float64, device=DEV), mean[:, :-1]], 1)
    m2 = ((win - prev) * (win - mean) * wt).cumsum(1)
    std = (m2 / (cum.clamp(min=1.0) - 1.0).clamp(min=1.0)).sqrt().clamp(min=c.minimum_scale)
    ends = torch.arange(enc, device=DEV) * PATCH + PATCH - 1
    loc, scale = (v[:, ends].repeat_interleave(PATCH, 1) for v in (mean, std))
    cnt = wt.sum(1, keepdim=True).clamp(min=1.0)
    row_loc = (wt * win).sum(1, keepdim=True) / cnt
    row_scale = ((wt * (win - row_loc)).square().sum(1, keepdim=True) / cnt).sqrt().clamp(min=c.minimum_scale)
    is_known = known[:, None] != 0
    loc, scale = torch.where(is_known, row_loc, loc), torch.where(is_known, row_scale, scale)
    val = torch.where(ob, torch.asinh((win - loc) / scale.clamp(min=float(np.finfo(np.float32).eps))), 0.0)
    tok = torch.cat([val.view(rows, enc, PATCH), (~ob).double().view(rows, enc, PATCH)], 2).view(rows * enc, 2 * PATCH)
    seen = ob.view(rows, enc, PATCH).any(-1)
    kv = (seen.int().cumsum(1) > 0).int()
    first = torch.where(seen.any(1), seen.int().argmax(1), enc).cpu().numpy()
    at = np.array([first[group == g].min() for g in group])
    at = np.where(at == enc, 0, at)
    base = np.r_[np.arange(enc), ll + np.arange(h)]
    pos = base[None, :] - at[:, None]
    silu = torch.nn.functional.silu
    emb = _residual64(tok, w, "embed", silu).view(rows, enc, -1)
    y = torch.cat([emb, w["query"].double().expand(rows, h, -1)], 1).reshape(rows * n, -1)
    rl = None if role is None else _i32(role)
    for lw in w["layers"]:
        for a in lw["attentions"]:
            hn = _rms64(y, a["norm"], c.norm_eps)
            qkv = _lin64(hn, a["qkv"])
            att = (_ts_time64(qkv, kv, known, pos, rows, enc, ll, n) if a["time"]
                   else _ts_variate64(qkv, kv, group, rl, rows, enc, n))
            del qkv
            y = y + _lin64(att * torch.sigmoid(_lin64(hn, a["gate"])), a["wo"])
        up, gate = _rms64(y, lw["mlp_norm"], c.norm_eps), c.mlp_hidden_dim
        y = torch.cat([p + _lin64(silu(_lin64(u, lw["up"][:gate])) * _lin64(u, lw["up"][gate:]), lw["down"])
                       for p, u in zip(y.split(16384), up.split(16384))])
    dec = _rms64(y, w["out_norm"], c.norm_eps).view(rows, n, -1)[:, enc:].reshape(rows * h, -1)
    raw = _residual64(dec, w, "head", silu).view(rows, h * PATCH, c.num_quantiles)
    med, width = c.median_index, np.abs(np.diff(np.asarray(c.quantiles)))
    out = raw.clone()
    sp = torch.nn.functional.softplus(raw)
    step = torch.zeros_like(raw[..., 0])
    for i in range(med + 1, c.num_quantiles):
        step = step + c.quantile_width_factor * width[i - 1] * sp[..., i]
        out[..., i] = raw[..., med] + step
    step = torch.zeros_like(step)
    for i in range(med - 1, -1, -1):
        step = step + c.quantile_width_factor * width[i] * sp[..., i]
        out[..., i] = raw[..., med] - step
    anchor = (ll - 1) * PATCH
    return torch.sinh(out) * scale[:, anchor, None, None] + loc[:, anchor, None, None]


def exact(case: dict, seed: int):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "c2_forecast":
            return _c2_forecast64(case, seed).cpu().numpy()
        if kind == "ts_block":
            return _ts_block64(case, seed).cpu().numpy()
        s = prepare(case, seed)
        if kind == "c2_time":
            return _c2_time64(s["qkv"], s["live"], case["rows"], case["n"])
        if kind == "c2_group":
            return _c2_group64(s["qkv"], s["live"], s["group"], case["rows"], case["n"])
        if kind == "c2_layer":
            _, w, _, group = _layer_inputs(case, seed)
            if case["dtype"] in ("bf16", "fp16"):  # the weights the caller holds
                w = s["w"]
            return _c2_layer64(s["x0"].double(), w, s["live"], group, case["rows"], case["n"])
        rows, enc, n = case["rows"], case["enc"], case["enc"] + case["h"]
        m = _ts_masks(case, seed)
        if kind == "ts_time":
            o = _ts_time64(s["qkv"], s["kv"], s["known"], m["pos"], rows, enc, enc, n)
        else:
            o = _ts_variate64(s["qkv"], s["kv"], m["group"], s["role"], rows, enc, n)
        return o * torch.sigmoid(s["gate"].double())
