"""Performance cases of the draft library: the calls that a drafting program makes, each
through the package's public entry points, from the smallest (the soft-anchor embedding of
one block) to the largest (a 4096-row prompt through every layer, eight stacked sequences).

A case names a shape of ``config.workload`` and the sizes of one call.  Its ``kind`` is the
entry point:

  anchor    ``embed_block``: a block's noise embedding with the soft anchor in row 0;
  layer     ``model(noise, target_hidden, cache)`` and the caller's ``trim``: a decode step
            that hands the hidden states on (new context rows ingested, then the block), of
            one sequence or of several in lockstep, in a full or a sink + window cache;
  draft     ``draft(ids, target_hidden, cache)``: the same step down to logits and ids;
  batch     ``draft_batch(ids)``: one block for each of several sequences of ragged contexts;
  ingest    ``ingest_seq``: a prompt's rows (or a long step's) into the K/V caches, from one
            tensor or from the tapped layers' own tensors;
  quantize  ``quantize_w8``: one projection of a checkpoint to int8 rows and scales.

Most cases run one decoder layer (``num_hidden_layers`` is the caller's to choose), so that
a rounding does not travel through others before it is compared; ``draft``, ``batch`` and one
``ingest`` case run the workloads' five.
"""

from __future__ import annotations

import copy
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_ROOT, "mirror-sd_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_ROOT, "mirror-sd_amd"))

from mirror_sd_amd.config import workload  # noqa: E402
from mirror_sd_amd.dflash import DFlashDraftModel  # noqa: E402

PROJ = ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj")
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}


def listed():
    return [
        # The parallel caller embeds the next block before every draft, with the verify
        # logits of the rejected position as a soft anchor: the smallest call, per step.
        {"name": "anchor_8b", "kind": "anchor", "shape": "qwen3_8b_draft", "block": 16,
         "dtype": "bfloat16"},
        # A small draft layer early in a conversation, four accepted rows: launches count.
        {"name": "layer_4b_ctx64", "kind": "layer", "shape": "qwen3_4b_layer", "layers": 1,
         "seqs": 1, "block": 16, "new": 4, "ctx": 64, "window": False},
        # The cache that make_cache() gives by default (64 sink rows, a window of 1024), full,
        # in the steady state of a long generation: 7 accepted rows and a block of 32.
        {"name": "layer_27b_window", "kind": "layer", "shape": "dflash_27b", "layers": 1,
         "seqs": 1, "block": 32, "new": 7, "ctx": 1088, "window": True},
        # A long document resident in the cache: attention over 32768 rows.
        {"name": "layer_27b_ctx32768", "kind": "layer", "shape": "dflash_27b", "layers": 1,
         "seqs": 1, "block": 32, "new": 5, "ctx": 32768, "window": False},
        # A few users drafted in lockstep with short blocks: 3 x 16 = 48 stacked rows.
        {"name": "layer_8b_3x16", "kind": "layer", "shape": "qwen3_8b_draft", "layers": 1,
         "seqs": 3, "block": 16, "new": 5, "ctx": 1500, "window": False},
        # The decode step of the 8B draft down to its tokens and logits, all layers.
        {"name": "draft_8b", "kind": "draft", "shape": "qwen3_8b_draft", "layers": 5,
         "block": 16, "new": 6, "ctx": 2048},
        # The benchmark's headline shape as its caller runs it: 16 accepted rows, then the
        # block of 32 against 4096 resident rows, all layers and the lm_head.
        {"name": "draft_27b", "kind": "draft", "shape": "dflash_27b", "layers": 5, "block": 32,
         "new": 16, "ctx": 4096},
        # Eight sequences of ragged contexts, 256 stacked rows: the batched benchmark shape.
        {"name": "batch_llama8b_8x32", "kind": "batch", "shape": "llama8b_batch", "layers": 5,
         "seqs": 8, "block": 32,
         "ctx": "4146 4443 6312 7812 779 1619 6833 7798"},
        # A long acceptance or a short follow-up turn: 45 rows in one step, tapped tensors.
        {"name": "ingest_27b_45", "kind": "ingest", "shape": "dflash_27b", "layers": 5,
         "rows": 45, "features": True},
        # An ordinary prompt of ragged length, from the tapped layers' tensors.
        {"name": "ingest_8b_777", "kind": "ingest", "shape": "qwen3_8b_draft", "layers": 5,
         "rows": 777, "features": True},
        # A long prompt in one call, concatenated hidden states: the benchmark's context.
        {"name": "ingest_27b_4096", "kind": "ingest", "shape": "dflash_27b", "layers": 5,
         "rows": 4096, "features": False},
        # Loading a checkpoint: the largest projection of the 27B draft to W8A16.
        {"name": "quantize_27b_down", "kind": "quantize", "shape": "dflash_27b",
         "proj": "down_proj", "rows": 5120},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["anchor", "layer", "layer", "layer", "draft", "batch", "ingest",
                       "ingest", "quantize"])
    if kind == "anchor":
        return {"kind": kind, "shape": rng.choice(["qwen3_8b_draft", "dflash_27b",
                                                   "llama8b_batch"]),
                "block": rng.randint(2, 32), "dtype": rng.choice(sorted(DTYPES))}
    if kind == "layer":
        shape = rng.choice(["qwen3_4b_layer", "qwen3_8b_draft", "dflash_27b"])
        seqs = rng.choice([1, 1, 1, 2, 3, 4] if shape == "dflash_27b" else [1, 1, 1, 2, 3, 4, 6, 8])
        window = rng.random() < 0.3
        ctx = _log_int(rng, 16, 32768 // seqs if not window else 1088)
        return {"kind": kind, "shape": shape, "layers": 1, "seqs": seqs, "block": rng.randint(4, 32), "new": _log_int(rng, 1, 64 if seqs == 1 else 20),
                "ctx": ctx, "window": window}
    if kind == "draft":
        return {"kind": kind, "shape": rng.choice(["qwen3_8b_draft", "dflash_27b"]),
                "layers": rng.randint(1, 5), "block": rng.randint(4, 32),
                "new": _log_int(rng, 1, 33), "ctx": _log_int(rng, 64, 4096)}
    if kind == "batch":
        seqs = rng.randint(2, 8)
        return {"kind": kind, "shape": "llama8b_batch", "layers": rng.randint(1, 5),
                "seqs": seqs, "block": rng.randint(4, 32),
                "ctx": " ".join(str(_log_int(rng, 64, 4096)) for _ in range(seqs))}
    if kind == "ingest":
        return {"kind": kind, "shape": rng.choice(["qwen3_8b_draft", "dflash_27b"]),
                "layers": rng.randint(1, 5), "rows": _log_int(rng, 17, 4096),
                "features": rng.random() < 0.5}
    # a tensor-parallel checkpoint's shard holds some of a projection's rows
    shape, proj = rng.choice(["qwen3_4b_layer", "qwen3_8b_draft", "dflash_27b"]), rng.choice(PROJ)
    rows = _proj_shapes(workload(shape).cfg)[proj][0]
    return {"kind": kind, "shape": shape, "proj": proj, "rows": _log_int(rng, 512, rows)}


# ------------------------------------------------------------------------------- inputs

def _cfg(case):
    cfg = copy.deepcopy(workload(case["shape"]).cfg)
    cfg.num_hidden_layers = case.get("layers", 1)
    return cfg


def _contexts(case):
    """Resident rows of each sequence (``ctx``: one count for all, or a text of counts)."""
    ctx = case.get("ctx", "")
    return [int(c) for c in ctx.split()] if isinstance(ctx, str) else [ctx] * case.get("seqs", 1)


def _proj_shapes(cfg):
    H, D, F = cfg.hidden_size, cfg.head_dim, cfg.intermediate_size
    q, kv = cfg.num_attention_heads * D, cfg.num_key_value_heads * D
    return {"q_proj": (q, H), "k_proj": (kv, H), "v_proj": (kv, H), "o_proj": (H, q),
            "gate_proj": (F, H), "up_proj": (F, H), "down_proj": (H, F)}


def _proj_name(layer, proj):
    part = "mlp" if proj in ("gate_proj", "up_proj", "down_proj") else "self_attn"
    return f"layers.{layer}.{part}.{proj}.weight"


class _Source:
    """Seeded tensors on the GPU: the n-th draw depends on the seed and n alone."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, shape, std=1.0, dtype=torch.float16):
        t = torch.randn(shape, generator=self.g, dtype=torch.float32, device="cuda")
        return t.mul_(std).to(dtype)

    def gain(self, n):   # norm gains as the package's synthetic weights have them
        return torch.ones((n,), dtype=torch.float16, device="cuda")

    def ids(self, shape, V):
        return torch.randint(0, V, shape, generator=self.g, dtype=torch.int32, device="cuda")

    def int8_rows(self, shape):
        """A projection as a W8A16 checkpoint holds it: int8 rows and fp16 row scales."""
        w = self.normal(shape, 0.02, torch.float32)
        s = w.abs().amax(1, keepdim=True) / 127.0
        return torch.round(w / s).to(torch.int8), s.reshape(-1).to(torch.float16)


def _weights(src, cfg, fc, head):
    """Draft weights: plain tensors by name, and the W8A16 projections (rows, scales)."""
    H, D = cfg.hidden_size, cfg.head_dim
    t, q = {}, {}
    for i in range(cfg.num_hidden_layers):
        for p, shape in _proj_shapes(cfg).items():
            q[_proj_name(i, p)] = src.int8_rows(shape)
        t[f"layers.{i}.input_layernorm.weight"] = src.gain(H)
        t[f"layers.{i}.post_attention_layernorm.weight"] = src.gain(H)
        t[f"layers.{i}.self_attn.q_norm.weight"] = src.gain(D)
        t[f"layers.{i}.self_attn.k_norm.weight"] = src.gain(D)
    t["norm.weight"] = src.gain(H)
    if fc:
        t["fc.weight"] = src.normal((H, cfg.num_target_features * H), 0.02)
        t["hidden_norm.weight"] = src.gain(H)
    if head:
        t["embed_tokens.weight"] = src.normal((cfg.vocab_size, H), 0.02)
        t["lm_head.weight"] = src.normal((cfg.vocab_size, H), 0.02)
    return t, q


def _block_ids(src, cfg, shape):
    """A block's ids: the anchor token, then masks."""
    ids = torch.full(shape, cfg.mask_token_id, dtype=torch.int32, device="cuda")
    ids[..., 0] = src.ids(shape[:-1], cfg.vocab_size)
    return ids


def _resident_rows(src, cfg, seqs, ctx):
    """K/V rows [seqs, NKV, ctx, D] of one layer as a cache holds them: keys normed and
    rotated, values of the spread that the v projection gives a normed row."""
    shape = (seqs, cfg.num_key_value_heads, ctx, cfg.head_dim)
    return src.normal(shape), src.normal(shape, 0.02 * math.sqrt(cfg.hidden_size))


def _inputs(case, seed):
    """Everything prepare() hands to the library and exact() computes from."""
    src = _Source(seed)
    kind, cfg = case["kind"], _cfg(case)
    H, d = cfg.hidden_size, {"cfg": cfg}
    if kind == "quantize":
        d["w"] = src.normal((case["rows"], _proj_shapes(cfg)[case["proj"]][1]), 0.02,
                            torch.float32)
        return d
    if kind == "anchor":
        d["t"] = {"norm.weight": src.gain(H),
                  "embed_tokens.weight": src.normal((cfg.vocab_size, H), 0.02)}
        d["ids"] = _block_ids(src, cfg, (case["block"],))
        d["logits"] = src.normal((cfg.vocab_size,), 3.0, DTYPES[case["dtype"]])
        return d
    d["t"], d["q"] = _weights(src, cfg, fc=kind != "batch", head=kind in ("draft", "batch"))
    nf = cfg.num_target_features
    if kind in ("layer", "draft"):
        n = case.get("seqs", 1)
        d["kv"] = [_resident_rows(src, cfg, n, case["ctx"]) for _ in range(cfg.num_hidden_layers)]
        d["th"] = src.normal((n, case["new"], nf * H))
        if kind == "layer":
            d["noise"] = src.normal((n, case["block"], H), 0.02)
        else:
            d["ids"] = _block_ids(src, cfg, (case["block"],))
    elif kind == "batch":
        d["ctx"] = [src.normal((c, H)) for c in _contexts(case)]
        d["ids"] = _block_ids(src, cfg, (case["seqs"], case["block"]))
    else:
        d["th"] = src.normal((case["rows"], nf * H))
    return d


# -------------------------------------------------------------------------- the call itself

SINK, WINDOW = 64, 1024   # make_cache()'s defaults


def prepare(case, seed):
    kind, d = case["kind"], _inputs(case, seed)
    cfg = d["cfg"]
    st = {"kind": kind, "case": case}
    if kind == "quantize":
        model = DFlashDraftModel(cfg, max_ctx=64)
        st.update(model=model, w=d["w"])
        return st
    if kind == "anchor":
        model = DFlashDraftModel(cfg, max_ctx=64)
        model.load_head(d["t"]["norm.weight"], d["t"]["embed_tokens.weight"])
        st.update(model=model, ids=d["ids"], logits=d["logits"])
        return st
    seqs, block = case.get("seqs", 1), case.get("block", 32)
    ctx = max(_contexts(case), default=0)
    rows = max(ctx + case.get("new", 0) + case.get("rows", 0),
               SINK + WINDOW if case.get("window") else 0)
    model = DFlashDraftModel(cfg, max_ctx=rows, max_block=max(block, 32), max_seqs=seqs)
    model.load_weights(d["t"], quantized=d["q"])
    st["model"] = model
    if kind in ("layer", "draft"):
        cache = model.make_cache(SINK, WINDOW) if case.get("window") else model.make_cache(0, 0)
        for c, (k, v) in zip(cache, d["kv"]):
            c.keys, c.values, c.offset = k, v, case["ctx"]
        st.update(cache=cache, th=d["th"], noise=d.get("noise"), ids=d.get("ids"))
        run(st)   # the resident rows settle in the device cache with the first step
    elif kind == "batch":
        for i, rows in enumerate(d["ctx"]):
            model.ingest_seq(i, rows, fused_context=True)
        st["ids"] = d["ids"]
    else:
        rows, H = case["rows"], cfg.hidden_size
        th = d["th"]
        if case["features"]:
            th = [th[:, j * H:(j + 1) * H].contiguous() for j in range(cfg.num_target_features)]
        st["th"] = th
        st["kv"] = [(k[:, :rows], vt[:, :, :rows]) for k, vt in model.cache_tensors(0)]
        for view in [v for pair in st["kv"] for v in pair]:
            view.owner = model   # a view of the model's memory, which lives as long as it does
    torch.cuda.synchronize()
    return st


def run(st):
    kind, model, case = st["kind"], st["model"], st["case"]
    if kind == "quantize":
        return model.quantize_w8(st["w"])
    if kind == "anchor":
        return model.embed_block(st["ids"], correction_logits=st["logits"])
    if kind == "layer":
        hidden = model(st["noise"], st["th"], cache=st["cache"])
        # the block's rows and, so that every pass meets the same cache, the step's own
        for c in st["cache"]:
            c.trim(case["block"] + case["new"])
        return hidden
    if kind == "draft":
        ids, logits = model.draft(st["ids"], st["th"], cache=st["cache"], return_logits=True)
        for c in st["cache"]:
            c.trim(case["new"])
        return ids, logits
    if kind == "batch":
        return model.draft_batch(ids=st["ids"], return_logits=True)
    model.ingest_seq(0, st["th"])
    return st["kv"]


# ----------------------------------------------------------------- what it cannot do without

def work(case):
    cfg, kind = _cfg(case), case["kind"]
    H, V, D = cfg.hidden_size, cfg.vocab_size, cfg.head_dim
    if kind == "quantize":
        n, k = case["rows"], _proj_shapes(cfg)[case["proj"]][1]
        return {"bytes": n * k * 5 + n * 2, "flops": 3 * n * k}
    if kind == "anchor":
        b = V * torch.finfo(DTYPES[case["dtype"]]).bits // 8
        return {"bytes": b + (8 + 2 * case["block"]) * H * 2, "flops": 2 * V}
    NL, NKV, NH = cfg.num_hidden_layers, cfg.num_key_value_heads, cfg.num_attention_heads
    shapes = _proj_shapes(cfg)
    w = sum(n * k + 2 * n for n, k in shapes.values())
    wkv = sum(shapes[p][0] * (shapes[p][1] + 2) for p in ("k_proj", "v_proj"))
    row_bytes = 2 * NKV * D * 2                      # one cached row of one layer
    seqs = case.get("seqs", 1)
    M = seqs * case.get("block", 0)
    new = case.get("rows", 0) + seqs * case.get("new", 0)   # rows through the fc
    fc_k = cfg.num_target_features * H
    flops = 2 * new * (H * fc_k + NL * 2 * NKV * D * H) + 2 * M * NL * w
    bytes_ = new * (fc_k * 2 + NL * row_bytes)
    if new:
        bytes_ += H * fc_k * 2
    if kind == "ingest":
        return {"bytes": bytes_ + NL * wkv, "flops": flops}
    ctxs = [c + case.get("new", 0) for c in _contexts(case)]
    if case.get("window"):
        ctxs = [min(c, SINK + WINDOW - case["block"]) for c in ctxs]
    keys = sum(c + case["block"] for c in ctxs)
    bytes_ += NL * (w + keys * row_bytes)
    flops += NL * 4 * NH * D * case["block"] * keys
    if kind == "layer":
        return {"bytes": bytes_ + 2 * M * H * 2, "flops": flops}
    return {"bytes": bytes_ + M * H * 2 + V * H * 2 + M * V * 4, "flops": flops + 2 * M * V * H}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind == "anchor":
        # gathered rows are copies; the anchor row is an fp32 sum rounded to fp16 once
        return {"rel": 1e-4}
    if kind == "ingest":
        return {"rel": 2e-3}       # K/V rows in fp16: a Linear, a norm and a rotation
    if kind == "layer":
        return {"rel": 4e-3}       # one layer and the final norm, fp16 between the steps
    # five layers, fp16 between the steps, and the argmax of logits that may all but tie
    return {"rel": 1e-2, "differ": 0.15}


# --------------------------------------------------------------------------- in 64 bits

def _rms64(x, g, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * g.double()


def _lin64(x, qs):
    q, s = qs
    return (x @ q.double().t()) * s.double()


def _rope64(x, pos0, theta):
    """x [rows, heads, D] at positions pos0 .. pos0 + rows - 1, halves rotated."""
    half = x.shape[-1] // 2
    f = theta ** (-torch.arange(half, dtype=torch.float64, device=x.device) / half)
    a = (pos0 + torch.arange(x.shape[0], dtype=torch.float64, device=x.device))[:, None] * f
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    x0, x1 = x[..., :half], x[..., half:]
    return torch.cat([x0 * c - x1 * s, x1 * c + x0 * s], -1)


def _kv64(cfg, t, q, i, h, pos0):
    """Layer i's K (normed, rotated) and V of the rows h, [NKV, rows, D]."""
    shape = (h.shape[0], cfg.num_key_value_heads, cfg.head_dim)
    k = _lin64(h, q[_proj_name(i, "k_proj")]).reshape(shape)
    k = _rms64(k, t[f"layers.{i}.self_attn.k_norm.weight"], cfg.rms_norm_eps)
    v = _lin64(h, q[_proj_name(i, "v_proj")]).reshape(shape)
    return (_rope64(k, pos0, cfg.rope_theta).transpose(0, 1), v.transpose(0, 1))


def _layer64(cfg, t, q, i, x, K, V, pos0, window):
    """Layer i over the block rows x; K / V [NKV, L, D] are the context's rows."""
    D, NH, eps = cfg.head_dim, cfg.num_attention_heads, cfg.rms_norm_eps
    h = _rms64(x, t[f"layers.{i}.input_layernorm.weight"], eps)
    qh = _lin64(h, q[_proj_name(i, "q_proj")]).reshape(-1, NH, D)
    qh = _rope64(_rms64(qh, t[f"layers.{i}.self_attn.q_norm.weight"], eps), pos0, cfg.rope_theta)
    kb, vb = _kv64(cfg, t, q, i, h, pos0)
    K, V = torch.cat([K, kb], 1), torch.cat([V, vb], 1)
    if window and K.shape[1] > SINK + WINDOW:
        K = torch.cat([K[:, :SINK], K[:, -WINDOW:]], 1)
        V = torch.cat([V[:, :SINK], V[:, -WINDOW:]], 1)
    out = torch.empty_like(qh)
    per = NH // cfg.num_key_value_heads
    for g in range(cfg.num_key_value_heads):
        for j in range(g * per, (g + 1) * per):
            p = torch.softmax((qh[:, j] @ K[g].t()) / math.sqrt(D), -1)
            out[:, j] = p @ V[g]
    x = x + _lin64(out.reshape(x.shape[0], NH * D), q[_proj_name(i, "o_proj")])
    h = _rms64(x, t[f"layers.{i}.post_attention_layernorm.weight"], eps)
    act = torch.nn.functional.silu(_lin64(h, q[_proj_name(i, "gate_proj")]))
    act = act * _lin64(h, q[_proj_name(i, "up_proj")])
    return x + _lin64(act, q[_proj_name(i, "down_proj")])


def _fused64(cfg, t, th):
    return _rms64(th.double() @ t["fc.weight"].double().t(), t["hidden_norm.weight"],
                  cfg.rms_norm_eps)


def exact(case, seed):
    kind, d = case["kind"], _inputs(case, seed)
    cfg, t = d["cfg"], d.get("t")
    if kind == "quantize":
        w = d["w"].double()
        s = w.abs().amax(1, keepdim=True) / 127.0
        return torch.round(w / s).clamp_(-127, 127), s.reshape(-1)
    if kind == "anchor":
        e = t["embed_tokens.weight"]
        out = e[d["ids"].long()].double()
        # ties among 16-bit logits go to the lower id: a stable descending order
        top = torch.sort(d["logits"].double(), descending=True, stable=True)
        p = torch.softmax(top.values[:8], 0)
        out[0] = p @ e[top.indices[:8]].double()
        return out[None]
    q, eps = d["q"], cfg.rms_norm_eps
    if kind == "ingest":
        h = _fused64(cfg, t, d["th"])
        res = []
        for i in range(cfg.num_hidden_layers):
            k, v = _kv64(cfg, t, q, i, h, 0)
            res.append((k, v.transpose(1, 2)))
        return res
    if kind == "batch":
        rows = []
        for s, c in enumerate(d["ctx"]):
            x = t["embed_tokens.weight"][d["ids"][s].long()].double()
            h = c.double()
            for i in range(cfg.num_hidden_layers):
                K, V = _kv64(cfg, t, q, i, h, 0)
                x = _layer64(cfg, t, q, i, x, K, V, h.shape[0], False)
            rows.append(_rms64(x, t["norm.weight"], eps))
        logits = torch.stack(rows) @ t["lm_head.weight"].double().t()
        return None, logits
    window, outs = bool(case.get("window")), []
    for s in range(case.get("seqs", 1)):
        if kind == "layer":
            x = d["noise"][s].double()
        else:
            x = t["embed_tokens.weight"][d["ids"].long()].double()
        h = _fused64(cfg, t, d["th"][s])
        for i in range(cfg.num_hidden_layers):
            k, v = _kv64(cfg, t, q, i, h, case["ctx"])
            K = torch.cat([d["kv"][i][0][s].double(), k], 1)
            V = torch.cat([d["kv"][i][1][s].double(), v], 1)
            x = _layer64(cfg, t, q, i, x, K, V, case["ctx"] + case["new"], window)
        outs.append(_rms64(x, t["norm.weight"], eps))
    hidden = torch.stack(outs)
    if kind == "layer":
        return hidden
    return None, hidden[0] @ t["lm_head.weight"].double().t()
