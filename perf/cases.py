"""The work this library is used for, as cases that can be timed and checked.

Every case is one pass through the public entry points (kvcache_amd.ops, kvcache_amd.model)
as a serving program calls them: decode attention of one sequence, of ragged batches (device
lengths, paged and contiguous, fp16 and fp32, one query head per KV head and grouped), of
few long contexts, the planned decode of all layers of a serving step with its new K/V rows;
prompt attention with the K/V write before it (host and device position); the linear layers
of a decode step; the output head; and a whole prompt through the decoder.

listed() holds one case per use, draw() gives more of the same ranges.  K, V and q are
N(0, 1), blocks lie in the pool in random order, weights are N(0, 0.02) as in the model.
Lengths belong to the case (so that its bytes are known), values and block order to the seed.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from kvcache_amd import KVC_F16, KVC_F32, ops
from kvcache_amd import workloads as wl
from kvcache_amd.model import QwenConfig, QwenModel

DEV = "cuda"
EPS, THETA = 1e-6, 1e6
VOCAB = 151936  # the decoder's vocabulary (QwenConfig)


# ---- the cases ---------------------------------------------------------------------------

def listed():
    return [
        # one request at a time, the smallest call: fp32 as the reference, 8 heads, 1024 tokens
        {"name": "single-f32-1024", "kind": "single", "dtype": "f32", "h": 8, "d": 64, "length": 1024, "block": 16},
        # the headline workload: 128 ragged sequences, lengths skewed short in [16, 2048), fp16, MHA
        {"name": "ragged-mha-f16-128", "kind": "ragged", "dtype": "f16", "layout": "paged", "n": 128, "hq": 8,
         "hkv": 8, "d": 64, "block": 16, "dist": "skew", "lo": 16, "hi": 2048, "lens_seed": 12345},
        # the reference's data type and its contiguous caches, an odd batch
        {"name": "ragged-mha-f32-contig-61", "kind": "ragged", "dtype": "f32", "layout": "contig", "n": 61, "hq": 8,
         "hkv": 8, "d": 64, "block": 16, "dist": "skew", "lo": 16, "hi": 2048, "lens_seed": 99},
        # four long contexts, grouped heads, splits of 512 tokens
        {"name": "gqa-long-split512", "kind": "long", "dtype": "f16", "hq": 14, "hkv": 2, "d": 64, "block": 16,
         "lens": "8192,16384,32768,32768", "split": 512},
        # a wide batch with head_dim 128 and four query heads per KV head, lengths over two decades
        {"name": "gqa-d128-log-200", "kind": "ragged", "dtype": "f16", "layout": "paged", "n": 200, "hq": 32,
         "hkv": 8, "d": 128, "block": 16, "dist": "log", "lo": 32, "hi": 4096, "lens_seed": 7},
        # the attention of a serving step: every layer appends its new row and attends, on one host plan
        {"name": "step-append-64x12", "kind": "step", "n": 64, "layers": 12, "hq": 14, "hkv": 2, "d": 64,
         "block": 16, "dist": "log", "lo": 128, "hi": 4096, "lens_seed": 5},
        # a prompt of 2048 tokens: its K/V written, then causal attention
        {"name": "prompt-2048", "kind": "prompt", "pos": "host", "nq": 2048, "base": 0, "hq": 14, "hkv": 2, "d": 64,
         "block": 16},
        # a piece of a long prompt behind 6000 tokens that are already cached, head_dim 128
        {"name": "prompt-1000-at-6000-d128", "kind": "prompt", "pos": "host", "nq": 1000, "base": 6000, "hq": 32,
         "hkv": 8, "d": 128, "block": 16},
        # a few new tokens of one sequence, position in device memory (the form that can be captured)
        {"name": "prompt-device-96-at-1500", "kind": "prompt", "pos": "device", "nq": 96, "base": 1500, "hq": 14,
         "hkv": 2, "d": 64, "block": 16},
        # the linear layers of a decode step, 8 layers with weights of their own, 32 running sequences
        {"name": "rows-32x8", "kind": "rows", "m": 32, "layers": 8, "hidden": 896, "hq": 14, "hkv": 2, "d": 64,
         "inter": 4864},
        # final norm, output head and greedy token of 32 running sequences
        {"name": "head-32", "kind": "head", "m": 32, "hidden": 896, "vocab": VOCAB},
        # a whole prompt through the 24-layer decoder, to the logits of its last position
        {"name": "model-prefill-700", "kind": "model", "tokens": 700, "layers": 24},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng: random.Random):
    kind = rng.choice(["single", "ragged", "ragged", "long", "step", "prompt", "prompt", "prompt", "rows", "head",
                       "model"])
    if kind == "single":
        return {"kind": kind, "dtype": rng.choice(["f32", "f16"]), "h": rng.choice([4, 8, 16]),
                "d": rng.choice([64, 128]), "length": _log_int(rng, 100, 8192), "block": 16}
    if kind == "ragged":
        grouped = rng.random() < 0.5
        d = rng.choice([64, 64, 128])
        if grouped:
            hkv = rng.choice([2, 4, 8])
            hq, dtype = hkv * rng.choice([4, 7, 8]), "f16"
        else:
            hkv = hq = rng.choice([8, 12, 16])
            dtype = rng.choice(["f16", "f32"])
        lo, hi = 16, rng.choice([1024, 2048, 3000])
        return {"kind": kind, "dtype": dtype, "layout": rng.choice(["paged", "paged", "contig"]),
                "n": _log_int(rng, 5, 200), "hq": hq, "hkv": hkv, "d": d, "block": 16,
                "dist": rng.choice(["skew", "log"]), "lo": lo, "hi": hi, "lens_seed": rng.randrange(1, 1 << 20)}
    if kind == "long":
        lens = [_log_int(rng, 5000, 40000) for _ in range(rng.randint(1, 5))]
        return {"kind": kind, "dtype": "f16", "hq": 14, "hkv": 2, "d": 64, "block": 16,
                "lens": ",".join(map(str, lens)), "split": rng.choice([0, 512, 1024])}
    if kind == "step":
        hkv = rng.choice([2, 4])
        return {"kind": kind, "n": _log_int(rng, 4, 96), "layers": 12, "hq": hkv * 7, "hkv": hkv, "d": 64,
                "block": 16, "dist": "log", "lo": 32, "hi": rng.choice([1000, 4096]),
                "lens_seed": rng.randrange(1, 1 << 20)}
    if kind == "prompt":
        hkv = rng.choice([2, 8])
        hq, d = (14, 64) if hkv == 2 else (32, 128)
        if rng.random() < 0.25:
            return {"kind": kind, "pos": "device", "nq": _log_int(rng, 1, 400), "base": rng.randrange(0, 4000),
                    "hq": 14, "hkv": 2, "d": 64, "block": 16}
        return {"kind": kind, "pos": "host", "nq": _log_int(rng, 20, 2500),
                "base": rng.choice([0, 0, rng.randrange(1, 6000)]), "hq": hq, "hkv": hkv, "d": d, "block": 16}
    if kind == "rows":
        return {"kind": kind, "m": rng.randint(1, 32), "layers": 8, "hidden": rng.choice([512, 896, 1024]), "hq": 14,
                "hkv": 2, "d": 64, "inter": rng.choice([2816, 4864])}
    if kind == "head":
        return {"kind": kind, "m": rng.randint(1, 32), "hidden": rng.choice([512, 896, 1024]),
                "vocab": rng.choice([32000, 100352, VOCAB])}
    return {"kind": "model", "tokens": _log_int(rng, 16, 700), "layers": 24}


# ---- inputs ------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, dtype=torch.float16, std=1.0):
    t = torch.empty(shape, device=DEV, dtype=dtype)
    t.normal_(0.0, std, generator=g)
    return t


def _torch_dtype(case):
    return torch.float16 if case.get("dtype", "f16") == "f16" else torch.float32


def _kvc_dtype(case):
    return KVC_F16 if case.get("dtype", "f16") == "f16" else KVC_F32


def _lens(case):
    if "lens" in case:
        return np.array([int(x) for x in case["lens"].split(",")], np.int32)
    if case["dist"] == "skew":
        return wl.ref_lengths(case["n"], case["hi"], case["lens_seed"])
    return wl.loguniform_lengths(case["n"], case["lo"], case["hi"], case["lens_seed"])


def _paged(g, lens, block):
    """Block tables of the sequences over a pool of exactly their blocks, in random order."""
    nblk = (lens + block - 1) // block
    off = np.concatenate([[0], np.cumsum(nblk)]).astype(np.int32)
    nb = int(off[-1])
    table = torch.randperm(nb, device=DEV, generator=g).to(torch.int32)
    return nb, table, torch.from_numpy(off).to(DEV), off


def _bytes_of(t):
    return t.numel() * t.element_size()


def _ws(nbytes):
    return torch.zeros(max(int(nbytes), 256), dtype=torch.uint8, device=DEV)


def _attention_inputs(case, seed):
    g = _gen(seed)
    dt, kind = _torch_dtype(case), case["kind"]
    s = {}
    if kind == "single":
        h, d, n, b = case["h"], case["d"], case["length"], case["block"]
        nb = (n + b - 1) // b
        s["q"] = _normal(g, (1, h, d), dt)
        s["k"], s["v"] = _normal(g, (nb, h, b, d), dt), _normal(g, (nb, h, b, d), dt)
        s["table"] = torch.randperm(nb, device=DEV, generator=g).to(torch.int32)
        s["off"], s["lens"] = np.array([0, nb], np.int32), np.array([n], np.int32)
        return s
    hq, hkv, d, b = case["hq"], case["hkv"], case["d"], case["block"]
    if kind == "prompt":
        n, base = case["nq"], case["base"]
        nb = (base + n + b - 1) // b
        s["q"] = _normal(g, (n, hq, d))
        s["k_new"], s["v_new"] = _normal(g, (n, hkv, d)), _normal(g, (n, hkv, d))
        s["k"], s["v"] = _normal(g, (nb, hkv, b, d)), _normal(g, (nb, hkv, b, d))
        s["table"] = torch.randperm(nb, device=DEV, generator=g).to(torch.int32)
        s["start"] = torch.tensor([base], dtype=torch.int32, device=DEV)
        return s
    lens = _lens(case)
    n = len(lens)
    s["lens"] = lens
    s["lens_dev"] = torch.from_numpy(lens).to(DEV)
    if case.get("layout") == "contig":
        maxs = int(lens.max())
        s["q"] = _normal(g, (n, hq, d), dt)
        s["k"], s["v"] = _normal(g, (n, hkv, maxs, d), dt), _normal(g, (n, hkv, maxs, d), dt)
        return s
    nb, s["table"], s["off_dev"], s["off"] = _paged(g, lens, b)
    if kind == "step":
        lay = case["layers"]
        s["q"] = _normal(g, (lay, n, hq, d))
        s["k_new"], s["v_new"] = _normal(g, (lay, n, hkv, d)), _normal(g, (lay, n, hkv, d))
        s["k"], s["v"] = _normal(g, (lay, nb, hkv, b, d)), _normal(g, (lay, nb, hkv, b, d))
    else:
        s["q"] = _normal(g, (n, hq, d), dt)
        s["k"], s["v"] = _normal(g, (nb, hkv, b, d), dt), _normal(g, (nb, hkv, b, d), dt)
    return s


def _rows_inputs(case, seed):
    g = _gen(seed)
    m, h, lay, inter = case["m"], case["hidden"], case["layers"], case["inter"]
    qd, kd = case["hq"] * case["d"], case["hkv"] * case["d"]
    s = {"embed": _normal(g, (1000, h)),
         "ids": torch.randint(0, 1000, (m,), device=DEV, generator=g).to(torch.int32),
         "pos": torch.randint(0, 4096, (m,), device=DEV, generator=g).to(torch.int32),
         "att": _normal(g, (lay, m, qd), std=0.3),
         "ln1": 1 + _normal(g, (lay, h), std=0.1), "ln2": 1 + _normal(g, (lay, h), std=0.1),
         "wqkv": _normal(g, (lay, qd + 2 * kd, h), std=0.02), "bqkv": _normal(g, (lay, qd + 2 * kd), std=0.02),
         "wo": _normal(g, (lay, h, qd), std=0.02), "wgu": _normal(g, (lay, 2 * inter, h), std=0.02),
         "wd": _normal(g, (lay, h, inter), std=0.02)}
    return s


def _head_inputs(case, seed):
    g = _gen(seed)
    return {"x": _normal(g, (case["m"], case["hidden"])), "norm": 1 + _normal(g, (case["hidden"],), std=0.1),
            "w": _normal(g, (case["vocab"], case["hidden"]), std=0.02)}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "model":
        t = case["tokens"]
        m = QwenModel(QwenConfig(layers=case["layers"], max_batch=4, max_rows=max(t, 16), prefill_rows=max(t, 16),
                                 num_blocks=(t + 15) // 16 + 16, seed=1 + int(seed) % (1 << 30)))
        toks = np.random.default_rng(int(seed)).integers(0, VOCAB, t).astype(np.int32)
        return {"case": case, "model": m, "tokens": toks}
    if kind == "rows":
        s = _rows_inputs(case, seed)
        m, h, lay, inter = case["m"], case["hidden"], case["layers"], case["inter"]
        qd, kd = case["hq"] * case["d"], case["hkv"] * case["d"]
        z = lambda *sh: torch.zeros(sh, dtype=torch.float16, device=DEV)  # noqa: E731
        s.update(x=z(m, h), q=z(lay, m, qd), kk=z(lay, m, kd), vv=z(lay, m, kd), act=z(lay, m, inter))
        s["ws"] = _ws(max(ops.rows_workspace_size(h, qd), ops.rows_workspace_size(h, inter)))
    elif kind == "head":
        s = _head_inputs(case, seed)
        m, v = case["m"], case["vocab"]
        s["logits"] = torch.zeros((m, v), dtype=torch.float32, device=DEV)
        s["tokens"] = torch.zeros((m,), dtype=torch.int32, device=DEV)
        s["ws"] = _ws(ops.rows_workspace_size(v, case["hidden"]))
    else:
        s = _attention_inputs(case, seed)
        s["out"] = torch.zeros_like(s["q"])
        d = case["d"]
        s["scale"] = 1.0 / math.sqrt(d)
        if kind == "ragged" or kind == "long":
            block = 0 if case.get("layout") == "contig" else case["block"]
            s["cap"] = int(s["lens"].max())
            s["ws"] = _ws(ops.decode_workspace_size(len(s["lens"]), case["hq"], case["hkv"], d, block, s["cap"],
                                                    case.get("split", 0), _kvc_dtype(case)))
        elif kind == "step":
            # the step's plan: the scheduler makes it once, every layer's launch uses it
            table = s["table"].cpu().numpy()
            work, nu, nr = ops.decode_plan(s["lens"], case["hq"], case["hkv"], d, case["block"], tab_off=s["off"],
                                           table=table)
            s["work"], s["units"], s["records"] = torch.from_numpy(np.ascontiguousarray(work)).to(DEV), nu, nr
            s["wpos"] = s["lens_dev"] - 1
            s["ws"] = _ws(ops.planned_workspace_size(case["hq"], case["hkv"], d, nr, BLOCK=case["block"]))
        elif kind == "prompt":
            from kvcache_amd import lib
            if case["pos"] == "host":
                need = lib().kvc_paged_causal_attn_workspace_size(case["base"], case["nq"], case["hq"], case["hkv"], d,
                                                                  case["block"], KVC_F16)
            else:
                need = lib().kvc_paged_causal_attn_dev_workspace_size(case["nq"], case["hq"], case["hkv"], d,
                                                                      case["block"], KVC_F16)
            s["ws"] = _ws(need)
    s["case"] = case
    # the addresses a C caller would hold
    s["p"] = {k: t.data_ptr() for k, t in s.items() if isinstance(t, torch.Tensor)}
    if "ws" in s:
        s["wsp"] = (s["ws"].data_ptr(), _bytes_of(s["ws"]))
    torch.cuda.synchronize()
    return s


# ---- one pass ----------------------------------------------------------------------------

def run(s):
    c = s["case"]
    return _RUN[c["kind"]](c, s)


def _run_single(c, s):
    p = s["p"]
    ops.launch_paged(p["q"], p["k"], p["v"], p["table"], p["out"], c["length"], c["h"], c["d"], c["block"],
                     s["scale"], dtype=_kvc_dtype(c))
    return s["out"]


def _run_ragged(c, s):
    p, n = s["p"], len(s["lens"])
    if c.get("layout") == "contig":
        ops.launch_batched_decode(p["q"], p["k"], p["v"], p["lens_dev"], p["out"], n, c["hq"], c["d"], s["cap"],
                                  s["cap"], s["scale"], Hkv=c["hkv"], dtype=_kvc_dtype(c), workspace=s["wsp"])
    else:
        ops.launch_batched_paged(p["q"], p["k"], p["v"], p["table"], p["off_dev"], p["lens_dev"], p["out"], n, c["hq"],
                                 c["d"], c["block"], s["cap"], s["scale"], Hkv=c["hkv"], dtype=_kvc_dtype(c),
                                 split=c.get("split", 0), workspace=s["wsp"])
    return s["out"]


def _run_step(c, s):
    p, n, d = s["p"], c["n"], c["d"]
    qs, ks = n * c["hq"] * d * 2, n * c["hkv"] * d * 2
    pool = s["k"][0].numel() * 2
    for i in range(c["layers"]):
        ops.launch_batched_paged_append_planned(p["q"] + i * qs, p["k_new"] + i * ks, p["v_new"] + i * ks, p["wpos"],
                                                p["k"] + i * pool, p["v"] + i * pool, p["table"], len(s["table"]),
                                                p["out"] + i * qs, n, c["hq"], c["hkv"], d, c["block"], s["scale"],
                                                p["work"], s["units"], s["records"], workspace=s["wsp"])
    return {"out": s["out"], "k": s["k"], "v": s["v"]}


def _run_prompt(c, s):
    p = s["p"]
    if c["pos"] == "host":
        ops.qk_write_kv(p["k_new"], p["v_new"], p["k"], p["v"], p["table"], c["base"], c["nq"], c["hkv"], c["d"],
                        c["block"])
        ops.qk_paged_causal_attn(p["q"], p["out"], p["k"], p["v"], p["table"], c["base"], c["nq"], c["hq"], c["hkv"],
                                 c["d"], c["block"], s["scale"], workspace=s["wsp"])
    else:
        ops.qkcuda_write_kv(p["k_new"], p["v_new"], p["k"], p["v"], p["table"], p["start"], c["nq"], c["hkv"], c["d"],
                            c["block"])
        ops.qkcuda_paged_causal_attn(p["q"], p["out"], p["k"], p["v"], p["table"], p["start"], c["nq"], c["hq"],
                                     c["hkv"], c["d"], c["block"], s["scale"], workspace=s["wsp"])
    return {"out": s["out"], "k": s["k"], "v": s["v"]}


def _run_rows(c, s):
    p, m, h, inter = s["p"], c["m"], c["hidden"], c["inter"]
    qd, kd = c["hq"] * c["d"], c["hkv"] * c["d"]
    ops.qk_embed_gather(p["x"], p["embed"], p["ids"], m, h, 1000)
    for i in range(c["layers"]):
        ops.rows_qkv(p["q"] + i * m * qd * 2, p["kk"] + i * m * kd * 2, p["vv"] + i * m * kd * 2, p["x"],
                     p["wqkv"] + i * (qd + 2 * kd) * h * 2, p["bqkv"] + i * (qd + 2 * kd) * 2, p["pos"], m, h, c["hq"],
                     c["hkv"], c["d"], THETA, norm_w=p["ln1"] + i * h * 2, eps=EPS)
        ops.rows_linear(p["x"], p["att"] + i * m * qd * 2, p["wo"] + i * h * qd * 2, m, h, qd, residual=True,
                        workspace=s["wsp"])
        ops.rows_swiglu(p["act"] + i * m * inter * 2, p["x"], p["wgu"] + i * 2 * inter * h * 2, m, inter, h,
                        norm_w=p["ln2"] + i * h * 2, eps=EPS)
        ops.rows_linear(p["x"], p["act"] + i * m * inter * 2, p["wd"] + i * h * inter * 2, m, h, inter, residual=True,
                        workspace=s["wsp"])
    return {"x": s["x"], "q": s["q"], "k": s["kk"], "v": s["vv"]}


def _run_head(c, s):
    p = s["p"]
    ops.rows_lm_head(p["logits"], p["tokens"], p["x"], p["w"], c["m"], c["vocab"], c["hidden"], norm_w=p["norm"],
                     eps=EPS, workspace=s["wsp"])
    return {"logits": s["logits"], "tokens": s["tokens"]}


def _run_model(c, s):
    return s["model"].prefill_logits(s["tokens"])[1]


_RUN = {"single": _run_single, "ragged": _run_ragged, "long": _run_ragged, "step": _run_step, "prompt": _run_prompt,
        "rows": _run_rows, "head": _run_head, "model": _run_model}


# ---- what a pass cannot do without --------------------------------------------------------

def work(case):
    c, kind = case, case["kind"]
    es = 2 if c.get("dtype", "f16") == "f16" else 4
    if kind == "single":
        return {"bytes": 2 * c["length"] * c["h"] * c["d"] * es + 2 * c["h"] * c["d"] * es,
                "flops": 4 * c["length"] * c["h"] * c["d"]}
    if kind in ("ragged", "long", "step"):
        lens, lay = _lens(c), c.get("layers", 1)
        tok, n = int(lens.sum()), len(lens)
        # (a step's new rows are read from the inputs and written once, in place of a read of the pool)
        extra = 2 * n * c["hkv"] * c["d"] * es if kind == "step" else 0
        return {"bytes": lay * (2 * tok * c["hkv"] * c["d"] * es + 2 * n * c["hq"] * c["d"] * es + extra),
                "flops": lay * 4 * tok * c["hq"] * c["d"]}
    if kind == "prompt":
        n, base, d = c["nq"], c["base"], c["d"]
        keys = n * base + n * (n + 1) // 2
        return {"bytes": 2 * (base + n) * c["hkv"] * d * 2 + 2 * n * c["hkv"] * d * 2 + 2 * n * c["hq"] * d * 2,
                "flops": 4 * keys * c["hq"] * d}
    if kind == "rows":
        m, h, inter = c["m"], c["hidden"], c["inter"]
        qd, kd = c["hq"] * c["d"], c["hkv"] * c["d"]
        w = (qd + 2 * kd) * h + h * qd + 3 * inter * h
        act = m * (qd + 2 * kd + qd)  # q|k|v out, attention in
        return {"bytes": c["layers"] * (w + act) * 2 + 2 * m * h * 2, "flops": c["layers"] * 2 * m * w}
    if kind == "head":
        m, h, v = c["m"], c["hidden"], c["vocab"]
        return {"bytes": v * h * 2 + m * v * 4 + m * h * 2, "flops": 2 * m * v * h}
    t, h, inter, qd, kd = c["tokens"], 896, 4864, 896, 128
    w = (qd + 2 * kd) * h + h * qd + 3 * inter * h
    return {"bytes": c["layers"] * w * 2 + VOCAB * h * 2,
            "flops": c["layers"] * (2 * t * w + 4 * (t * (t + 1) // 2) * qd) + 2 * VOCAB * h}


def tolerance(case):
    kind = case["kind"]
    if kind in ("single", "ragged", "long", "step", "prompt"):
        return {"rel": 2e-6} if case.get("dtype") == "f32" else {"rel": 1.5e-3}
    if kind == "rows":
        return {"rel": 4e-3}
    if kind == "head":
        return {"rel": 1e-3}
    return {"rel": 1e-2}


# ---- the same in 64 bits ------------------------------------------------------------------

def _attend64(q, k, v, scale, first=None):
    """q [n, Hq, D] against k, v [S, Hkv, D]; query i sees keys 0 .. first + i (all if first is None)."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    out = torch.empty((n, hq, d), dtype=torch.float64, device=q.device)
    for h in range(hkv):
        kd, vd = k[:, h].double(), v[:, h].double()
        for j in range(h * (hq // hkv), (h + 1) * (hq // hkv)):
            sc = (q[:, j].double() @ kd.T.contiguous()) * scale
            if first is not None:
                seen = torch.arange(k.shape[0], device=q.device)[None, :] <= first + torch.arange(n, device=q.device)[:, None]
                sc = sc.masked_fill(~seen, -math.inf)
            out[:, j] = torch.softmax(sc, dim=1) @ vd
    return out


def _rows_of(pool, table, n):
    """[nb, H, B, D] pool blocks of a table -> [n, H, D] token rows."""
    x = pool[table.long()]
    return x.permute(0, 2, 1, 3).reshape(-1, pool.shape[1], pool.shape[3])[:n]


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + EPS) * w.double()


def _rope64(x, pos, d):
    m = x.shape[0]
    y = x.reshape(m, -1, 2, d // 2)
    ang = pos.double()[:, None] * THETA ** (-2.0 * torch.arange(d // 2, device=x.device, dtype=torch.float64) / d)
    co, si = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    return torch.stack([y[:, :, 0] * co - y[:, :, 1] * si, y[:, :, 1] * co + y[:, :, 0] * si], dim=2).reshape(m, -1)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "model":
        return None  # the weights are the library's own random fill
    if kind == "rows":
        s = _rows_inputs(c, seed)
        m, h, inter = c["m"], c["hidden"], c["inter"]
        qd, kd = c["hq"] * c["d"], c["hkv"] * c["d"]
        x = s["embed"][s["ids"].long()].double()
        q, k, v = [], [], []
        for i in range(c["layers"]):
            y = _rms64(x, s["ln1"][i]) @ s["wqkv"][i].double().T + s["bqkv"][i].double()
            q.append(_rope64(y[:, :qd], s["pos"], c["d"]))
            k.append(_rope64(y[:, qd:qd + kd], s["pos"], c["d"]))
            v.append(y[:, qd + kd:])
            x = x + s["att"][i].double() @ s["wo"][i].double().T
            gu = _rms64(x, s["ln2"][i]) @ s["wgu"][i].double().T
            gate, up = gu[:, :inter], gu[:, inter:]
            x = x + (gate / (1 + torch.exp(-gate)) * up) @ s["wd"][i].double().T
        return {"x": x, "q": torch.stack(q), "k": torch.stack(k), "v": torch.stack(v)}
    if kind == "head":
        s = _head_inputs(c, seed)
        return {"logits": _rms64(s["x"].double(), s["norm"]) @ s["w"].double().T, "tokens": None}
    s = _attention_inputs(c, seed)
    scale = 1.0 / math.sqrt(c["d"])
    if kind == "prompt":
        n, base, d = c["nq"], c["base"], c["d"]
        k, v = (_rows_of(s[a], s["table"], base + n) for a in ("k", "v"))
        k = torch.cat([k[:base], s["k_new"]])
        v = torch.cat([v[:base], s["v_new"]])
        return {"out": _attend64(s["q"], k, v, scale, base), "k": None, "v": None}
    if c.get("layout") == "contig":
        return torch.cat([_attend64(s["q"][i:i + 1], s["k"][i, :, :n].transpose(0, 1), s["v"][i, :, :n].transpose(0, 1),
                                    scale) for i, n in enumerate(s["lens"].tolist())])
    off, lens = s["off"].tolist(), s["lens"].tolist()

    def layer(q, kp, vp, kn=None, vn=None):
        out = []
        for i, n in enumerate(lens):
            t = s["table"][off[i]:off[i + 1]]
            k, v = _rows_of(kp, t, n), _rows_of(vp, t, n)
            if kn is not None:
                k, v = torch.cat([k[:n - 1], kn[i:i + 1]]), torch.cat([v[:n - 1], vn[i:i + 1]])
            out.append(_attend64(q[i:i + 1], k, v, scale))
        return torch.cat(out)

    if kind == "step":
        out = [layer(s["q"][i], s["k"][i], s["v"][i], s["k_new"][i], s["v_new"][i]) for i in range(c["layers"])]
        return {"out": torch.stack(out), "k": None, "v": None}
    return layer(s["q"], s["k"], s["v"])
