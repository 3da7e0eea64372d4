"""What is timed and compared when this framework's speed is measured: the calls that a
gemma.c-style program makes, from one decode layer to a whole decode step, from a chat turn's
short prefill chunk to a 2048-row prompt, through the entry points of `gemma_kv`.

A case is a dict of plain values:

  kind "decode"   one layer's append + attention for `batch` sequences of min_len..max_len keys
                  (the new token included); `raw`: from the raw q/k/v projections (RMSNorm + RoPE
                  inside the call), otherwise from prepared rows
  kind "step"     a whole 48-layer decode step (40 sliding layers, 8 global ones)
  kind "chunk"    causal attention of a prefill chunk over `prior` cached keys and itself
  kind "prompt"   a prompt's self-attention from raw projections (the norm + RoPE launchers)
  kind "project"  the attention output projection with its post-attention norm and residual

Geometries: 8 KV heads x 256 ("8x256") and the model's global one, 1 KV head x 512 ("1x512"),
16 query heads; bf16 inputs ~ N(0, 1), softmax scale 1 / sqrt(head_dim).
"""
from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "gemma.c_amd"))
import gemma_kv as gk  # noqa: E402

LAYERS = 48
QUERY_HEADS = 16
HIDDEN = 3840
WINDOW = 1024
SLIDING, GLOBAL = "8x256", "1x512"
EPS = 1e-6


def _heads_dim(geometry):
    return (8, 256) if geometry == "8x256" else (1, 512)


def _is_global(layer):
    return layer == LAYERS - 1 or (layer + 1) % 6 == 0


# ---- the cases ---------------------------------------------------------------------------------

def listed():
    return [
        # A sliding layer of one conversation: the smallest call, a full 1024-slot ring.
        {"name": "decode_sliding_b1", "kind": "decode", "geometry": "8x256", "window": WINDOW,
         "page": 1, "batch": 1, "min_len": 8193, "max_len": 8193, "lengths": 0, "raw": False},
        # A global layer of the model, one conversation of 8192 tokens, as the fused layer call.
        {"name": "decode_global512_b1", "kind": "decode", "geometry": "1x512", "window": 0,
         "page": 64, "batch": 1, "min_len": 8193, "max_len": 8193, "lengths": 0, "raw": True},
        # The same layer served to 24 conversations of ragged lengths.
        {"name": "decode_global512_b24", "kind": "decode", "geometry": "1x512", "window": 0,
         "page": 64, "batch": 24, "min_len": 200, "max_len": 12001, "lengths": 1, "raw": True},
        # A full-length cache of 8 KV heads under a serving batch: 64 sequences of 512-32768 keys.
        {"name": "decode_global256_b64", "kind": "decode", "geometry": "8x256", "window": 0,
         "page": 64, "batch": 64, "min_len": 512, "max_len": 32768, "lengths": 64, "raw": False},
        # A whole decode step in one call, prepared rows, 8 x 256 everywhere.
        {"name": "step_256_b1", "kind": "step", "geometry": "8x256", "batch": 1, "min_len": 8193,
         "max_len": 8193, "lengths": 0, "raw": False},
        # The model's own step: 1 x 512 global layers, from the raw projections.
        {"name": "step_model_b1", "kind": "step", "geometry": "1x512", "batch": 1,
         "min_len": 8193, "max_len": 8193, "lengths": 0, "raw": True},
        # A 2048-row chunk of a long prompt on a sliding layer, ring already wrapped.
        {"name": "chunk_sliding_2048", "kind": "chunk", "window": WINDOW, "page": 1, "batch": 1,
         "chunk": 2048, "prior": 1536},
        # The same on a global layer after 6144 tokens, with the balancing workspace.
        {"name": "chunk_global_2048", "kind": "chunk", "window": 0, "page": 64, "batch": 1,
         "chunk": 2048, "prior": 6144},
        # The next message of a long chat: a short, odd chunk behind a long cached context.
        {"name": "chunk_turn_93", "kind": "chunk", "window": 0, "page": 64, "batch": 1,
         "chunk": 93, "prior": 7401},
        # Two short first prompts on a sliding layer, from raw projections.
        {"name": "prompt_sliding_333x2", "kind": "prompt", "geometry": "8x256", "batch": 2,
         "seq": 333},
        # A 2048-token prompt on the model's global layer, from raw projections.
        {"name": "prompt_global512_2048", "kind": "prompt", "geometry": "1x512", "batch": 1,
         "seq": 2048},
        # The projection behind a global layer for a serving batch.
        {"name": "project_8192_b24", "kind": "project", "rows": 24, "width": 8192},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["step"] * 2 + ["chunk"] * 3 + ["prompt"] * 2 + ["project"])
    if kind == "decode":
        which = rng.choice(["sliding", "global512", "global512", "global256"])
        batch = _log_int(rng, 1, 64)
        longest = {"sliding": 16384, "global512": min(32768, 288_000 // batch),
                   "global256": min(131072, 1_000_000 // batch)}[which]
        max_len = _log_int(rng, 64, longest)
        return {"kind": "decode", "geometry": GLOBAL if which == "global512" else SLIDING,
                "window": WINDOW if which == "sliding" else 0,
                "page": rng.choice([1, 16, 64]) if which == "sliding" else rng.choice([16, 64]),
                "batch": batch, "min_len": _log_int(rng, 1, max_len), "max_len": max_len,
                "lengths": rng.randrange(1 << 20), "raw": rng.random() < 0.5}
    if kind == "step":
        batch = rng.choice([1, 1, 2, 3, 4, 8])
        max_len = _log_int(rng, 128, 12288 // batch)
        return {"kind": "step", "geometry": rng.choice([SLIDING, GLOBAL]), "batch": batch,
                "min_len": _log_int(rng, 32, max_len), "max_len": max_len,
                "lengths": rng.randrange(1 << 20), "raw": rng.random() < 0.5}
    if kind == "chunk":
        batch = rng.choice([1, 1, 1, 2, 3])
        chunk = _log_int(rng, 16, 2048 // batch)
        window = rng.choice([WINDOW, 0, 0])
        return {"kind": "chunk", "window": window, "page": rng.choice([1, 16]) if window else 64,
                "batch": batch, "chunk": chunk, "prior": _log_int(rng, 1, 12288 // batch)}
    if kind == "prompt":
        batch = rng.choice([1, 1, 2, 4])
        return {"kind": "prompt", "geometry": rng.choice([SLIDING, GLOBAL]), "batch": batch,
                "seq": _log_int(rng, 16, 2048 // batch)}
    return {"kind": "project", "rows": _log_int(rng, 1, 256), "width": rng.choice([4096, 8192])}


# ---- inputs, from the case and the seed alone --------------------------------------------------

DEVICE = "cuda"


class _Inputs:
    def __init__(self, case, seed):
        self.case = case
        self.gen = torch.Generator(device=DEVICE)
        self.gen.manual_seed(seed * 1_000_003 + 17)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.gen, device=DEVICE, dtype=torch.bfloat16)

    def norm_weight(self, *shape):
        return (1.0 + 0.1 * torch.randn(shape, generator=self.gen, device=DEVICE)).bfloat16()


def _lengths(case):
    rng = random.Random(case["lengths"])
    lens = [rng.randint(case["min_len"], case["max_len"]) for _ in range(case["batch"])]
    lens[rng.randrange(case["batch"])] = case["max_len"]
    return lens


def _rope_tables(positions, rotary, theta):
    half = rotary // 2
    freq = theta ** (-torch.arange(half, dtype=torch.float64, device=DEVICE) / half)
    angle = torch.arange(positions, dtype=torch.float64, device=DEVICE)[:, None] * freq
    return angle.cos().float(), angle.sin().float()


def _rope_of(geometry, positions):
    return _rope_tables(positions, 256, 1e4) if geometry == "8x256" else _rope_tables(positions, 128, 1e6)


def _ring_pages(window, page):
    return (window + 2 * page - 2) // page


def _cache_shape(case, window, page, longest):
    """Pages per sequence of a cache that holds `longest` positions, or a window's ring."""
    return _ring_pages(window, page) if window else -(-longest // page)


def _page_table(config, lengths):
    table = np.full(config.batch_size * config.max_pages_per_seq, -1, dtype=np.int32)
    slots = table.copy()
    for b, n in enumerate(lengths):
        if n:
            gk.check(gk.kv_cache_ensure_range(table, slots, config, b, 0, n), "ensure_range")
    return torch.from_numpy(table).to(DEVICE)


def _int32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEVICE)


def _make_decode(case, seed):
    i = _Inputs(case, seed)
    heads, dim = _heads_dim(case["geometry"])
    pages = _cache_shape(case, case["window"], case["page"], case["max_len"])
    b, rows = case["batch"], case["batch"] * pages * case["page"]
    got = {"pages": pages, "k_cache": i.normal(rows, heads, dim), "v_cache": i.normal(rows, heads, dim),
           "q": i.normal(b, QUERY_HEADS, dim), "k": i.normal(b, heads, dim), "v": i.normal(b, heads, dim)}
    if case["raw"]:
        got["wq"], got["wk"] = i.norm_weight(dim), i.norm_weight(dim)
        got["cos"], got["sin"] = _rope_of(case["geometry"], case["max_len"])
    return got


def _make_step(case, seed):
    i = _Inputs(case, seed)
    b = case["batch"]
    gh, gd = _heads_dim(case["geometry"])
    g_pages = -(-case["max_len"] // 64)
    got = {"g_pages": g_pages,
           "sk": i.normal(40 * b * WINDOW, 8, 256), "sv": i.normal(40 * b * WINDOW, 8, 256),
           "gk": i.normal(8 * b * g_pages * 64, gh, gd), "gv": i.normal(8 * b * g_pages * 64, gh, gd)}
    dims = [(gh, gd) if _is_global(n) else (8, 256) for n in range(LAYERS)]
    got["q"] = i.normal(sum(b * QUERY_HEADS * d for _, d in dims))
    got["k"] = i.normal(sum(b * h * d for h, d in dims))
    got["v"] = i.normal(sum(b * h * d for h, d in dims))
    if case["raw"]:
        got["wq"], got["wk"] = (i.norm_weight(sum(d for _, d in dims)) for _ in range(2))
        got["s_cos"], got["s_sin"] = _rope_of("8x256", case["max_len"])
        got["g_cos"], got["g_sin"] = _rope_of(case["geometry"], case["max_len"])
    return got


def _make_chunk(case, seed):
    i = _Inputs(case, seed)
    pages = _cache_shape(case, case["window"], case["page"], case["prior"] + case["chunk"])
    b, n, rows = case["batch"], case["chunk"], case["batch"] * pages * case["page"]
    return {"pages": pages, "k_cache": i.normal(rows, 8, 256), "v_cache": i.normal(rows, 8, 256),
            "q": i.normal(b, n, QUERY_HEADS, 256), "k": i.normal(b, n, 8, 256), "v": i.normal(b, n, 8, 256)}


def _make_prompt(case, seed):
    i = _Inputs(case, seed)
    heads, dim = _heads_dim(case["geometry"])
    b, n = case["batch"], case["seq"]
    got = {"q": i.normal(b, n, QUERY_HEADS, dim), "k": i.normal(b, n, heads, dim),
           "v": i.normal(b, n, heads, dim), "wq": i.norm_weight(dim), "wk": i.norm_weight(dim)}
    got["cos"], got["sin"] = _rope_of(case["geometry"], n)
    return got


def _make_project(case, seed):
    i = _Inputs(case, seed)
    # Weights of a trained projection's size: outputs of the order of the residual stream's.
    return {"a": i.normal(case["rows"], case["width"]),
            "w": i.normal(HIDDEN, case["width"]) * (case["width"] ** -0.5),
            "norm": i.norm_weight(HIDDEN), "x": i.normal(case["rows"], HIDDEN)}


_MAKE = {"decode": _make_decode, "step": _make_step, "chunk": _make_chunk, "prompt": _make_prompt,
         "project": _make_project}


# ---- the program's side: what it holds, and one pass ------------------------------------------

def prepare(case, seed):
    s = _MAKE[case["kind"]](case, seed)
    s["case"] = case
    kind = case["kind"]
    if kind == "decode":
        heads, dim = _heads_dim(case["geometry"])
        b, lens = case["batch"], _lengths(case)
        s["config"] = gk.make_config(1, b * s["pages"], case["page"], s["pages"], b, heads, dim, case["window"])
        s["table"] = _page_table(s["config"], lens)
        s["len"], s["pos"] = _int32(lens), _int32([n - 1 for n in lens])
        live = min(max(lens), case["window"] or max(lens))
        s["split"], s["splits"] = gk.decode_split_plan(s["config"], b, live)
        n = b * QUERY_HEADS * s["splits"]
        s["pm"], s["pl"] = torch.empty(n, device=DEVICE), torch.empty(n, device=DEVICE)
        s["pa"] = torch.empty(n * dim, device=DEVICE)
        s["out"] = torch.empty_like(s["q"])
    elif kind == "step":
        b, lens = case["batch"], _lengths(case)
        gh, gd = _heads_dim(case["geometry"])
        s["s_config"] = gk.make_config(40, b * WINDOW, 1, WINDOW, b, 8, 256, WINDOW)
        s["g_config"] = gk.make_config(8, b * s["g_pages"], 64, s["g_pages"], b, gh, gd, 0)
        s["s_table"], s["g_table"] = _page_table(s["s_config"], lens), _page_table(s["g_config"], lens)
        s["len"], s["pos"] = _int32(lens), _int32([n - 1 for n in lens])
        s["ws"] = torch.empty(gk.decode_step_workspace_bytes(b) // 4, dtype=torch.int32, device=DEVICE)
        gk.check(gk.decode_step_workspace_init(s["ws"], b), "decode_step_workspace_init")
        s["out"] = torch.empty_like(s["q"])
    elif kind == "chunk":
        b = case["batch"]
        s["config"] = gk.make_config(1, b * s["pages"], case["page"], s["pages"], b, 8, 256, case["window"])
        s["table"] = _page_table(s["config"], [case["prior"]] * b)
        s["prior"] = _int32([case["prior"]] * b)
        if not case["window"]:
            s["bytes"] = gk.flash_attention_prefill_chunk_workspace_bytes(b, case["chunk"], s["config"])
            s["ws"] = torch.zeros(max(s["bytes"], 256), dtype=torch.uint8, device=DEVICE)
        s["out"] = torch.empty_like(s["q"])
    elif kind == "prompt":
        b, n = case["batch"], case["seq"]
        s["pos"] = torch.arange(n, dtype=torch.int32, device=DEVICE).repeat(b)
        for name in ("q", "k", "v"):
            s[name + "_prepared"] = torch.empty_like(s[name])
        s["out"] = torch.empty_like(s["q"])
    else:
        s["outs"] = [torch.empty_like(s["x"]) for _ in range(3)]
    return s


def _bits(t):
    return t.view(torch.int16)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        scale = 1.0 / math.sqrt(s["q"].shape[-1])
        if case["raw"]:
            gk.check(gk.flash_attention_prep_append_decode_paged_bf16(
                s["out"], s["pm"], s["pl"], s["pa"], s["q"], s["k_cache"], s["v_cache"], s["table"],
                s["len"], s["pos"], s["k"], s["v"] if case["geometry"] == "8x256" else None, s["wq"], s["wk"],
                s["cos"], s["sin"], s["config"], 0, scale, s["split"], s["splits"], case["batch"]))
            return {"out": s["out"], "k": s["k_cache"], "v": s["v_cache"]}
        gk.check(gk.flash_attention_append_decode_paged_bf16(
            s["out"], s["pm"], s["pl"], s["pa"], s["q"], s["k_cache"], s["v_cache"], s["table"], s["len"],
            s["pos"], s["k"], s["v"], s["config"], 0, scale, s["split"], s["splits"], case["batch"]))
        return {"out": s["out"], "k": _bits(s["k_cache"]), "v": _bits(s["v_cache"])}
    if kind == "step":
        caches = (s["sk"], s["sv"], s["s_table"], s["s_config"], s["gk"], s["gv"], s["g_table"], s["g_config"])
        if case["raw"]:
            gk.check(gk.decode_step_layers_prep_bf16(
                s["out"], s["q"], s["k"], s["v"], *caches, s["len"], s["pos"], s["wq"], s["wk"], s["s_cos"],
                s["s_sin"], s["g_cos"], s["g_sin"], 0, LAYERS, 1.0 / 16, case["batch"], s["ws"]))
            return {"out": s["out"], "caches": [s["sk"], s["sv"], s["gk"], s["gv"]]}
        gk.check(gk.decode_step_layers_bf16(
            s["out"], s["q"], s["k"], s["v"], *caches, s["len"], s["pos"], 0, LAYERS, 1.0 / 16,
            case["batch"], s["ws"]))
        return {"out": s["out"], "caches": [_bits(s[n]) for n in ("sk", "sv", "gk", "gv")]}
    if kind == "chunk":
        args = (s["out"], s["q"], s["k"], s["v"], s["k_cache"], s["v_cache"], s["table"], s["prior"],
                s["config"], 0, case["batch"], case["chunk"], 1.0 / 16)
        if case["window"]:
            gk.check(gk.flash_attention_prefill_chunk_paged_bf16(*args))
        else:
            gk.check(gk.flash_attention_prefill_chunk_paged_bf16_ws(*args, s["ws"], s["bytes"]))
        return s["out"]
    if kind == "prompt":
        n, b = case["seq"], case["batch"]
        if case["geometry"] == "8x256":
            gk.check(gk.flash_attention_sliding_fwd_bf16_norm_rope(
                s["out"], s["q_prepared"], s["k_prepared"], s["v_prepared"], s["q"], s["k"], s["v"], s["wq"],
                s["wk"], s["cos"], s["sin"], s["pos"], b, n, n, WINDOW, 1.0 / 16))
        else:
            gk.check(gk.flash_attention_global_fwd_bf16_norm_rope(
                s["out"], s["q_prepared"], s["k_prepared"], s["v_prepared"], s["q"], s["k"], s["wq"],
                s["wk"], s["cos"], s["sin"], s["pos"], b, n, n, 1.0 / math.sqrt(512)))
        return {"out": s["out"], "q": s["q_prepared"], "k": s["k_prepared"], "v": s["v_prepared"]}
    gk.check(gk.attention_o_projection_post_norm_bf16(
        *s["outs"], s["a"], s["w"], s["norm"], s["x"], case["rows"], case["width"]))
    return s["outs"]


# ---- what a pass cannot do without -------------------------------------------------------------

def _decode_work(keys, batch, heads, dim):
    """(bytes, flops): K and V of every live key, the appended rows in and out, q and out."""
    return (4 * heads * dim * keys + 8 * heads * dim * batch + 4 * QUERY_HEADS * dim * batch,
            4 * QUERY_HEADS * dim * keys)


def work(case):
    kind = case["kind"]
    if kind == "decode":
        keys = sum(min(n, case["window"] or n) for n in _lengths(case))
        nbytes, flops = _decode_work(keys, case["batch"], *_heads_dim(case["geometry"]))
    elif kind == "step":
        lens = _lengths(case)
        sliding = _decode_work(sum(min(n, WINDOW) for n in lens), case["batch"], 8, 256)
        full = _decode_work(sum(lens), case["batch"], *_heads_dim(case["geometry"]))
        nbytes, flops = (40 * a + 8 * b for a, b in zip(sliding, full))
    elif kind == "chunk":
        n, p, w = case["chunk"], case["prior"], case["window"]
        pairs = sum(min(p + r + 1, w or p + r + 1) for r in range(n))
        rows = n + min(p, w - 1 if w else p)
        nbytes = case["batch"] * (4 * QUERY_HEADS * 256 * n + 4 * 8 * 256 * rows)
        flops = case["batch"] * pairs * 4 * QUERY_HEADS * 256
    elif kind == "prompt":
        n = case["seq"]
        heads, dim = _heads_dim(case["geometry"])
        w = WINDOW if case["geometry"] == "8x256" else n
        pairs = sum(min(r + 1, w) for r in range(n))
        read = (QUERY_HEADS + (2 if heads == 8 else 1) * heads) * dim
        written = (2 * QUERY_HEADS + 2 * heads) * dim
        nbytes = case["batch"] * n * 2 * (read + written)
        flops = case["batch"] * pairs * 4 * QUERY_HEADS * dim
    else:
        r, w = case["rows"], case["width"]
        nbytes = 2 * (HIDDEN * w + HIDDEN + r * w + 4 * r * HIDDEN)
        flops = 2 * r * w * HIDDEN
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # bf16 results of 32-bit sums, with bf16 probabilities in most of the kernels: 0.0016 to 0.0026
    # off the 64-bit result (rel) and at most 0.023 at one value, from raw prompts (whose first rows,
    # of a few keys each, are the large ones) 0.0033 and 0.083. Four times that. Appended cache rows
    # that are copies are compared as bits ("differ").
    if case["kind"] == "prompt":
        return {"rel": 1.3e-2, "max": 0.33}
    return {"rel": 1e-2, "max": 0.1, "differ": 0.0}


# ---- the same in 64 bits -----------------------------------------------------------------------

def _norm(x, weight=None):
    y = x.double()
    y = y / torch.sqrt(y.square().mean(-1, keepdim=True) + EPS)
    return y if weight is None else y * weight.double()


def _rope(x, cos, sin):
    """Split-half rotation of the first 2 * cos.shape[-1] dims; cos / sin [..., half]."""
    half = cos.shape[-1]
    a, b, rest = x[..., :half], x[..., half:2 * half], x[..., 2 * half:]
    cos, sin = cos.double(), sin.double()
    return torch.cat([a * cos - b * sin, b * cos + a * sin, rest], -1)


def _rows_of(first, end, page, pages, batch_index, base, device):
    """Cache rows of positions first..end-1 of a sequence whose ring slots map to its own pages."""
    pos = torch.arange(first, end, device=device)
    return base + (batch_index * pages + (pos // page) % pages) * page + pos % page


def _attend(q, k, v, scale):
    """q [16, D], k and v [n, heads, D], all in 64 bits: [16, D]."""
    heads, dim = k.shape[1], k.shape[2]
    qh = q.reshape(heads, QUERY_HEADS // heads, dim)
    p = torch.softmax(torch.matmul(qh, k.permute(1, 2, 0).contiguous()) * scale, -1)
    return torch.matmul(p, v.permute(1, 0, 2).contiguous()).reshape(QUERY_HEADS, dim)


def _decode_layer(x, q, k, v, kc, vc, lens, window, page, pages, base, scale, wq=None, wk=None, cos=None,
                  sin=None):
    """One layer's append and attention: the outputs, and the appended (row, k, v) of each sequence."""
    outs, new = [], []
    for b, n in enumerate(lens):
        qb, kb, vb = q[b].double(), k[b].double(), v[b].double()
        if wq is not None:
            c, s = cos[n - 1], sin[n - 1]
            vb = _norm(kb if kc.shape[1] == 1 else vb)
            qb, kb = _rope(_norm(qb, wq), c, s), _rope(_norm(kb, wk), c, s)
        first = max(0, n - window) if window else 0
        rows = _rows_of(first, n, page, pages, b, base, q.device)
        new.append((int(rows[-1]), kb, vb))
        ks, vs = kc[rows].double(), vc[rows].double()
        ks[-1], vs[-1] = kb, vb
        outs.append(_attend(qb, ks, vs, scale))
    return torch.stack(outs), new


def exact(case, seed):
    i = _MAKE[case["kind"]](case, seed)
    kind = case["kind"]
    if kind == "decode":
        more = {n: i[n] for n in ("wq", "wk", "cos", "sin")} if case["raw"] else {}
        out, new = _decode_layer(case, i["q"], i["k"], i["v"], i["k_cache"], i["v_cache"], _lengths(case),
                                 case["window"], case["page"], i["pages"], 0,
                                 1.0 / math.sqrt(i["q"].shape[-1]), **more)
        if not case["raw"] or i["k_cache"].numel() > 1 << 29:
            return {"out": out, "k": None, "v": None}
        k, v = i["k_cache"].double(), i["v_cache"].double()
        for row, kb, vb in new:
            k[row], v[row] = kb, vb
        return {"out": out, "k": k, "v": v}
    if kind == "step":
        return _exact_step(case, i)
    if kind == "chunk":
        outs = []
        for b in range(case["batch"]):
            n, p, w = case["chunk"], case["prior"], case["window"]
            first = max(0, p - w + 1) if w else 0
            rows = _rows_of(first, p, case["page"], i["pages"], b, 0, DEVICE)
            ks = torch.cat([i["k_cache"][rows], i["k"][b]]).double()
            vs = torch.cat([i["v_cache"][rows], i["v"][b]]).double()
            outs.append(_causal(i["q"][b].double(), ks, vs, p - first, w, 1.0 / 16))
        return torch.stack(outs)
    if kind == "prompt":
        heads = i["k"].shape[2]
        cos, sin = i["cos"][:, None], i["sin"][:, None]
        q, k = _rope(_norm(i["q"], i["wq"]), cos, sin), _rope(_norm(i["k"], i["wk"]), cos, sin)
        v = _norm(i["k"] if heads == 1 else i["v"])
        w = WINDOW if heads == 8 else 0
        out = torch.stack([_causal(q[b], k[b], v[b], 0, w, 1.0 / math.sqrt(q.shape[-1]))
                           for b in range(case["batch"])])
        return {"out": out, "q": q, "k": k, "v": v}
    res = i["a"].double() @ i["w"].double().T
    normed = _norm(res, i["norm"])
    return [res, normed, i["x"].double() + normed]


def _causal(q, k, v, offset, window, scale):
    """q [n, 16, D]; k, v [m, heads, D]; row r sees keys (r + offset - window, r + offset]."""
    n, heads = q.shape[0], k.shape[1]
    r = torch.arange(n, device=q.device)[:, None] + offset
    c = torch.arange(k.shape[0], device=q.device)[None]
    hidden = (c > r) | ((c <= r - window) if window else False)
    out = torch.empty_like(q)
    for h in range(QUERY_HEADS):
        kh = h * heads // QUERY_HEADS
        s = (q[:, h] @ k[:, kh].T * scale).masked_fill_(hidden, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, kh]
    return out


def _exact_step(case, i):
    b, lens = case["batch"], _lengths(case)
    g_rows, g_pages = b * i["g_pages"] * 64, i["g_pages"]
    outs, kinds, at = [], {False: [], True: []}, {"q": 0, "k": 0, "w": 0}
    seen = {False: 0, True: 0}
    for layer in range(LAYERS):
        g = _is_global(layer)
        heads, dim = _heads_dim(case["geometry"]) if g else (8, 256)

        def take(name, key, count):
            return i[name][at[key]:at[key] + count]

        q = take("q", "q", b * QUERY_HEADS * dim).reshape(b, QUERY_HEADS, dim)
        k, v = (take(n, "k", b * heads * dim).reshape(b, heads, dim) for n in ("k", "v"))
        more = {}
        if case["raw"]:
            more = {"wq": take("wq", "w", dim), "wk": take("wk", "w", dim),
                    "cos": i["g_cos" if g else "s_cos"], "sin": i["g_sin" if g else "s_sin"]}
        kc, vc, window, page, pages, rows = (
            (i["gk"], i["gv"], 0, 64, g_pages, g_rows) if g else (i["sk"], i["sv"], WINDOW, 1, WINDOW, b * WINDOW))
        out, new = _decode_layer(case, q, k, v, kc, vc, lens, window, page, pages, seen[g] * rows, 1.0 / 16, **more)
        outs.append(out.reshape(-1))
        kinds[g] += new
        seen[g] += 1
        at["q"] += q.numel()
        at["k"] += k.numel()
        at["w"] += dim
    if not case["raw"]:
        return {"out": torch.cat(outs), "caches": [None] * 4}
    caches = []
    for g, names in ((False, ("sk", "sv")), (True, ("gk", "gv"))):
        for n, name in enumerate(names):
            c = i[name].double()
            for entry in kinds[g]:
                c[entry[0]] = entry[1 + n]
            caches.append(c)
    return {"out": torch.cat(outs), "caches": caches}
