"""The work that users of chunkkv_amd have it do, as measurable cases.

Kinds of case (each through the entry points that a program calls):

attention  ops.attention_active, the attention of a layer over its cache in the three forms a
           request meets it: "blend" (the recomputed rows of a blend prefill over the whole cache),
           "causal" (every row: layers 0-1, chunk prefills) and "decode" (one new row).
repair     one request's KV repair as the engine issues it: layer 0's fresh rows, layer 1's repair
           with the base cache of the other layers, the fresh rows of layers 2..
gather     ops.rerope_gather of every layer: plain reuse of cached chunks without recompute.
extract    ops.extract_chunks: the store-put of a finished prefill's segments.
layer      the steps between a decoder layer's GEMMs: residual add + RMSNorm twice, RoPE of q/k with
           the cache write, the SiLU-gated product.
prefill    HipEngine.prefill of a whole request on a random-init model, logits and caches returned.

Model shapes: "7b" is Qwen2.5-7B's (28 layers, 28 query / 4 KV heads of 128, hidden 3584,
intermediate 18944), "0.5b" Qwen2.5-0.5B's (24 layers, 14 / 2 heads of 64, hidden 896,
intermediate 4864); theta 1e6 for both.
"""

import math

import numpy as np
import torch
from torch import nn

from chunkkv_amd import ops
from chunkkv_amd.engine import HipEngine
from chunkkv_amd.planner import local_index, plan_request
from chunkkv_amd.types import BlendConfig, ChunkKV, Placement

THETA = 1e6
VOCAB = 151936
SHAPES = {
    "7b": {"layers": 28, "hq": 28, "hkv": 4, "d": 128, "hidden": 3584, "inter": 18944},
    "0.5b": {"layers": 24, "hq": 14, "hkv": 2, "d": 64, "hidden": 896, "inter": 4864},
}
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
DEV = "cuda"


def listed():
    return [
        # layers 2.. of an 8k-token blend request: 24 chunks of 320 tokens at 30 % recompute + 4
        # sinks each, a 576-token uncached tail: 2976 query rows over 8256 cache rows
        {"name": "attention_blend_8k", "kind": "attention", "form": "blend", "shape": "7b", "chunks": 24,
         "chunk_len": 320, "tail": 576, "ratio": 0.3, "n_sink": 4},
        # layers 0-1 of the same request: every position active
        {"name": "attention_causal_8k", "kind": "attention", "form": "causal", "shape": "7b", "n": 8256},
        # a chunk prefilled on its own before it enters the store
        {"name": "attention_chunk_320", "kind": "attention", "form": "causal", "shape": "7b", "n": 320},
        # a short RAG request on the small model (about 1.1k tokens), ragged sizes
        {"name": "attention_blend_1k", "kind": "attention", "form": "blend", "shape": "0.5b", "chunks": 4,
         "chunk_len": 253, "tail": 91, "ratio": 0.15, "n_sink": 2},
        # one decoded token after the 8k request (cache rows for 32 more tokens allocated)
        {"name": "attention_decode_8k", "kind": "attention", "form": "decode", "shape": "7b", "n": 8256},
        # long-context request: 128 chunks of 256 tokens + a 64-token query at 15 % recompute
        {"name": "repair_32k", "kind": "repair", "shape": "7b", "dtype": "bf16", "chunks": 128, "chunk_len": 256,
         "tail": 64, "ratio": 0.15, "n_sink": 4, "exact": False},
        # the 8k request
        {"name": "repair_8k", "kind": "repair", "shape": "7b", "dtype": "bf16", "chunks": 24, "chunk_len": 320,
         "tail": 576, "ratio": 0.3, "n_sink": 4, "exact": False},
        # the short request in fp32, its first chunk (a system prompt) reused under its own prefix
        {"name": "repair_1k_f32", "kind": "repair", "shape": "0.5b", "dtype": "f32", "chunks": 4, "chunk_len": 253,
         "tail": 91, "ratio": 0.15, "n_sink": 2, "exact": True},
        # plain reuse: 16 chunks of 256 tokens into every layer's cache
        {"name": "gather_4k", "kind": "gather", "shape": "7b", "dtype": "bf16", "chunks": 16, "chunk_len": 256},
        # the store-put of the 8k request's 24 segments
        {"name": "extract_8k", "kind": "extract", "shape": "7b", "dtype": "bf16", "chunks": 24, "chunk_len": 320,
         "tail": 576},
        # the steps between the GEMMs of layers 2.. of the 8k request
        {"name": "layer_8k", "kind": "layer", "shape": "7b", "dtype": "bf16", "rows": 2976, "cache": 8256},
        # the short request through the whole engine
        {"name": "prefill_1k", "kind": "prefill", "shape": "0.5b", "chunks": 4, "chunk_len": 253, "tail": 91,
         "ratio": 0.15, "n_sink": 2},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _request_sizes(rng, most):
    """A request's layout: chunk length and count, uncached tail, recompute ratio, sinks."""
    chunk_len = _log_int(rng, 24, min(512, most))
    chunks = _log_int(rng, 1, max(1, min(128, most // chunk_len)))
    return {"chunks": chunks, "chunk_len": chunk_len, "tail": _log_int(rng, 8, min(576, max(8, most // 4))),
            "ratio": rng.choice([0.05, 0.15, 0.3, 0.5]), "n_sink": rng.choice([2, 4])}


def draw(rng):
    kind = rng.choice(["attention", "attention", "repair", "repair", "gather", "extract", "layer", "prefill"])
    shape = rng.choice(["7b", "7b", "0.5b"])
    c = {"kind": kind, "shape": shape}
    if kind == "attention":
        c["form"] = rng.choice(["blend", "blend", "causal", "decode"])
        if c["form"] == "blend":
            c.update(_request_sizes(rng, _log_int(rng, 64, 7680)))
        else:
            c["n"] = _log_int(rng, 33, 8256 if c["form"] == "causal" else 32832)
        return c
    if kind == "prefill":
        c["shape"] = "0.5b"
        c.update(_request_sizes(rng, _log_int(rng, 128, 2048)))
        return c
    c["dtype"] = "bf16" if shape == "7b" else rng.choice(["bf16", "f32"])
    if kind == "layer":
        c["rows"] = _log_int(rng, 1, 8256)
        c["cache"] = _log_int(rng, c["rows"], 8256)
        return c
    # sizes up to the long request for the repair, up to the 8k request for the copies
    c.update(_request_sizes(rng, _log_int(rng, 128, 32768 if kind == "repair" else 7680)))
    if kind == "repair":
        c["exact"] = c["chunks"] > 1 and rng.random() < 0.25
    else:
        del c["ratio"], c["n_sink"]
    if kind == "gather":
        del c["tail"]
    if kind == "extract":
        c["chunks"] = min(c["chunks"], 64)
    return c


# ---- inputs ---------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _randn(gen, shape, dtype=torch.bfloat16):
    return torch.randn(shape, generator=gen, device=DEV, dtype=dtype)


def _inv_freq(d):
    """fp32 inverse frequencies theta ** (-2i / d) (the exponent in fp32, one rounding)."""
    e = (-np.arange(0, d, 2, dtype=np.float32) / np.float32(d)).astype(np.float64)
    return torch.from_numpy((THETA ** e).astype(np.float32)).to(DEV)


def _rotate(x, pos, inv):
    """Half-split rotation of x (..., n, d) by fp32 angles pos * inv, in fp64."""
    ang = (pos.to(torch.float32)[:, None] * inv[None, :]).double()
    cos, sin = ang.cos(), ang.sin()
    a, b = x.double().chunk(2, dim=-1)
    return torch.cat((a * cos - b * sin, a * sin + b * cos), dim=-1)


def _layout(case, seed):
    """Host side of a request: the starts at which its chunks were computed, their order, per-chunk
    deviation levels (log-normal: some chunks move a lot under their new prefix, most little)."""
    rs = np.random.RandomState(seed % (1 << 31))
    n = case["chunks"]
    return {"orig": rs.randint(0, 8192, n), "order": rs.permutation(n), "sigma": np.exp(rs.randn(n) - 3.0), "rs": rs}


def _n_tokens(case):
    return case["chunks"] * case["chunk_len"] + case.get("tail", 0)


def _store(case, gen, lay):
    """Cached chunks as the store holds them: per layer contiguous (1, H, L, D) keys and values."""
    s = SHAPES[case["shape"]]
    dims = (s["layers"], 1, s["hkv"], case["chunk_len"], s["d"])
    chunks = []
    for i in range(case["chunks"]):
        k, v = (_randn(gen, dims, DTYPES[case["dtype"]]) for _ in range(2))
        chunks.append(ChunkKV(list(k.unbind(0)), list(v.unbind(0)), int(lay["orig"][i])))
    return chunks


def _placements(case, chunks, lay):
    L = case["chunk_len"]
    pl = [Placement(chunks[c], i * L) for i, c in enumerate(lay["order"])]
    if case.get("exact"):  # the first chunk was computed here, under this prefix
        pl[0].chunk.start = 0
        pl[0].exact = True
    return pl


def _tables(case, plan):
    """Device descriptors of a planned request (what the engine uploads)."""
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    tab = np.array([[[k.data_ptr(), v.data_ptr()] for k, v in zip(c.keys, c.values)] for c in plan.chunks],
                   dtype=np.uint64)
    return {"tab": up(tab.reshape(-1).view(np.int64)), "segs": up(plan.segments.reshape(-1)),
            "flags": up(plan.flags), "local": up(local_index(plan.n_tokens, plan.layer0_idx)),
            "spans": up(plan.spans.reshape(-1)), "layer0": up(plan.layer0_idx.astype(np.int64))}


def _base_rows(placements, layer, n, hkv, d, dtype):
    """One layer's base cache (1, H, n, d): re-rotated cached keys and values, zero elsewhere."""
    inv = _inv_freq(d)
    k = torch.zeros((1, hkv, n, d), dtype=dtype, device=DEV)
    v = torch.zeros_like(k)
    for p in placements:
        at = slice(p.start, p.start + p.chunk.length)
        delta = torch.full((p.chunk.length,), float(p.start - p.chunk.start), device=DEV)
        k[:, :, at] = _rotate(p.chunk.keys[layer], delta, inv).to(dtype)
        v[:, :, at] = p.chunk.values[layer]
    return k, v


def _kept_positions(case, seed):
    """Sorted positions a blend recomputes: the tail, each chunk's sinks, and the positions of
    largest deviation, which gather in the chunks that moved most."""
    lay = _layout(case, seed)
    L, C, n = case["chunk_len"], case["chunks"], _n_tokens(case)
    score = (np.repeat(lay["sigma"], L) * (1.0 + 0.1 * lay["rs"].randn(C * L))).reshape(C, L)
    sinks = min(L, case["n_sink"])
    score[:, :sinks] = -1.0
    budget = min(C * int(round(case["ratio"] * L)), C * (L - sinks))
    keep = np.zeros(n, dtype=bool)
    keep[C * L :] = True
    keep[: C * L].reshape(C, L)[:, :sinks] = True
    keep[np.argsort(-score.reshape(-1), kind="stable")[:budget]] = True
    return np.flatnonzero(keep)


def _attention_sizes(case):
    """(query rows, cache rows, visible pairs) of an attention case."""
    if case["form"] == "decode":
        return 1, case["n"] + 32, case["n"] + 1
    if case["form"] == "causal":
        return case["n"], case["n"], case["n"] * (case["n"] + 1) // 2
    pos = _kept_positions(case, 0)
    return len(pos), _n_tokens(case), int((pos + 1).sum())


def _prepare_attention(case, seed):
    s, gen = SHAPES[case["shape"]], _gen(seed)
    nq, n, _ = _attention_sizes(case)
    pos = {"blend": lambda: _kept_positions(case, seed), "causal": lambda: np.arange(n),
           "decode": lambda: np.array([case["n"]])}[case["form"]]()
    # q as ckv_rope_qkv leaves it (token-major), scores of a standard deviation of two
    q = (2.0 * _randn(gen, (1, nq, s["hq"], s["d"]))).transpose(1, 2)
    K, V = (_randn(gen, (1, s["hkv"], n, s["d"])) for _ in range(2))
    return {"q": q, "K": K, "V": V, "pos": torch.from_numpy(pos.astype(np.int64)).to(DEV)}


def _prepare_repair(case, seed):
    s, gen, lay = SHAPES[case["shape"]], _gen(seed), _layout(case, seed)
    dtype, n, L = DTYPES[case["dtype"]], _n_tokens(case), case["chunk_len"]
    placements = _placements(case, _store(case, gen, lay), lay)
    plan = plan_request(n, placements, case["n_sink"], case["ratio"])
    row, n0 = s["hkv"] * s["d"], len(plan.layer0_idx)
    # layer 1's fresh rows: the cached rows moved by each chunk's level, random where uncached
    bk, bv = _base_rows(placements, 1, n, s["hkv"], s["d"], dtype)
    level = np.ones(n, dtype=np.float32)
    level[: case["chunks"] * L] = np.repeat(lay["sigma"][lay["order"]], L)
    level = torch.from_numpy(level).to(DEV)[:, None]
    at = torch.from_numpy(plan.layer0_idx).to(DEV)
    k1, v1 = ((b.float() + level * _randn(gen, b.shape, torch.float32)).to(dtype)[:, :, at] for b in (bk, bv))
    # projections of the other layers, token-major, before RoPE
    proj = [None if li == 1 else tuple(_randn(gen, (1, n0 if li == 0 else plan.n_keep, row), dtype) for _ in range(2))
            for li in range(s["layers"])]
    slab = (s["layers"], 1, s["hkv"], n, s["d"])
    return {"case": case, "plan": plan, "placements": placements, **_tables(case, plan), "k1": k1,
            "v1": v1.transpose(1, 2).contiguous().transpose(1, 2),  # token-major, as the projection leaves it
            "proj": proj, "K": torch.zeros(slab, dtype=dtype, device=DEV), "V": torch.zeros(slab, dtype=dtype, device=DEV),
            "ws": ops.layer1_repair_workspace(DEV), "err": torch.zeros(1, dtype=torch.int32, device=DEV)}


def _prepare_gather(case, seed):
    s, gen, lay = SHAPES[case["shape"]], _gen(seed), _layout(case, seed)
    placements = _placements(case, _store(case, gen, lay), lay)
    plan = plan_request(_n_tokens(case), placements, 0, 0.0)
    slab = (s["layers"], 1, s["hkv"], plan.n_tokens, s["d"])
    return {"plan": plan, "placements": placements, **_tables(case, plan),
            "K": torch.zeros(slab, dtype=DTYPES[case["dtype"]], device=DEV),
            "V": torch.zeros(slab, dtype=DTYPES[case["dtype"]], device=DEV),
            "err": torch.zeros(1, dtype=torch.int32, device=DEV)}


def _prepare_extract(case, seed):
    s, gen, L = SHAPES[case["shape"]], _gen(seed), case["chunk_len"]
    slab = (s["layers"], 1, s["hkv"], _n_tokens(case), s["d"])
    K, V = (_randn(gen, slab, DTYPES[case["dtype"]]) for _ in range(2))
    return {"K": K, "V": V, "spans": [(i * L, (i + 1) * L) for i in range(case["chunks"])]}


def _prepare_layer(case, seed):
    s, gen, dtype, n = SHAPES[case["shape"]], _gen(seed), DTYPES[case["dtype"]], case["rows"]
    hid, qd, kd = s["hidden"], s["hq"] * s["d"], s["hkv"] * s["d"]
    rs = np.random.RandomState(seed % (1 << 31))
    rows = np.sort(rs.choice(case["cache"], n, replace=False)).astype(np.int64)
    cache = (1, s["hkv"], case["cache"], s["d"])
    return {"shape": s, "h": 3.0 * _randn(gen, (1, n, hid), dtype), "mlp_out": _randn(gen, (1, n, hid), dtype),
            "attn_out": _randn(gen, (1, n, hid), dtype),
            "w_in": 1.0 + 0.1 * _randn(gen, (hid,), dtype), "w_post": 1.0 + 0.1 * _randn(gen, (hid,), dtype),
            "qkv": _randn(gen, (1, n, qd + 2 * kd), dtype), "gate_up": _randn(gen, (1, n, 2 * s["inter"]), dtype),
            "pos": torch.from_numpy(rows).to(DEV), "K": torch.zeros(cache, dtype=dtype, device=DEV),
            "V": torch.zeros(cache, dtype=dtype, device=DEV)}


class Qwen2RMSNorm(nn.Module):
    def __init__(self, hidden, eps=1e-6):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(hidden, device=DEV, dtype=torch.bfloat16))
        self.variance_epsilon = eps

    def forward(self, h):
        x = h.float()
        x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + self.variance_epsilon)
        return self.weight * x.to(h.dtype)


def _linear(i, o, bias, gen, std=0.02):
    m = nn.utils.skip_init(nn.Linear, i, o, bias=bias, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        m.weight.normal_(0.0, std, generator=gen)
        if bias:
            m.bias.normal_(0.0, 0.02, generator=gen)
    return m


class _Layer(nn.Module):
    def __init__(self, s, gen):
        super().__init__()
        hid, qd, kd = s["hidden"], s["hq"] * s["d"], s["hkv"] * s["d"]
        self.input_layernorm, self.post_attention_layernorm = Qwen2RMSNorm(hid), Qwen2RMSNorm(hid)
        self.self_attn, self.mlp = nn.Module(), nn.Module()
        a, m = self.self_attn, self.mlp
        a.q_proj, a.k_proj, a.v_proj = _linear(hid, qd, True, gen), _linear(hid, kd, True, gen), _linear(hid, kd, True, gen)
        out_std = 0.02 / math.sqrt(2 * s["layers"])  # the products that add to the residual stream
        a.o_proj = _linear(qd, hid, False, gen, out_std)
        m.gate_proj, m.up_proj = _linear(hid, s["inter"], False, gen), _linear(hid, s["inter"], False, gen)
        m.down_proj = _linear(s["inter"], hid, False, gen, out_std)


class _Config:
    hidden_act, rope_theta, rope_scaling, eos_token_id = "silu", THETA, None, 0

    def __init__(self, s):
        self.hidden_size, self.head_dim = s["hidden"], s["d"]
        self.num_attention_heads, self.num_key_value_heads = s["hq"], s["hkv"]


class _Model(nn.Module):
    """A random-init causal language model with the modules HipEngine reads: weights of standard
    deviation 0.02 (those that add to the residual stream smaller by the root of twice the layers),
    tied embeddings of deviation one: the layers add to the residual stream, as a trained model's
    do, instead of replacing it."""

    def __init__(self, s, gen):
        super().__init__()
        self.config = self.generation_config = _Config(s)
        self.model = nn.Module()
        self.model.embed_tokens = nn.utils.skip_init(nn.Embedding, VOCAB, s["hidden"], device=DEV, dtype=torch.bfloat16)
        with torch.no_grad():
            self.model.embed_tokens.weight.normal_(0.0, 1.0, generator=gen)
        self.model.layers = nn.ModuleList(_Layer(s, gen) for _ in range(s["layers"]))
        self.model.norm = Qwen2RMSNorm(s["hidden"])
        self.lm_head = nn.utils.skip_init(nn.Linear, s["hidden"], VOCAB, bias=False, device=DEV, dtype=torch.bfloat16)
        self.lm_head.weight = self.model.embed_tokens.weight


class _Tokenizer:
    eos_token_id = 0


@torch.inference_mode()
def _chunk_kv(model, s, tokens):
    """Keys and values of each chunk (rows of tokens) computed on its own at positions 0.., in
    plain torch fp32 (rounded to bf16 as stored)."""
    C, L = tokens.shape
    hq, hkv, d = s["hq"], s["hkv"], s["d"]
    pos, inv = torch.arange(L, device=DEV), _inv_freq(d)
    lin = lambda m, x: x @ m.weight.float().t() + (m.bias.float() if m.bias is not None else 0.0)  # noqa: E731
    norm = lambda m, x: m.weight.float() * x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + m.variance_epsilon)  # noqa: E731
    heads = lambda x, h: x.view(C, L, h, d).transpose(1, 2).contiguous()  # noqa: E731
    mask = torch.full((L, L), float("-inf"), device=DEV).triu(1)
    h = model.model.embed_tokens(tokens).float()
    keys, values = [], []
    for layer in model.model.layers:
        a, m = layer.self_attn, layer.mlp
        x = norm(layer.input_layernorm, h)
        q, k, v = heads(lin(a.q_proj, x), hq), heads(lin(a.k_proj, x), hkv), heads(lin(a.v_proj, x), hkv)
        q, k = (_rotate(t, pos, inv).float() for t in (q, k))
        keys.append(k.bfloat16())
        values.append(v.bfloat16())
        kt = k.repeat_interleave(hq // hkv, 1).transpose(2, 3).contiguous()
        w = torch.softmax(torch.matmul(q, kt) / math.sqrt(d) + mask, -1)
        o = torch.matmul(w, v.repeat_interleave(hq // hkv, 1).contiguous())
        h = h + lin(a.o_proj, o.transpose(1, 2).reshape(C, L, hq * d))
        x = norm(layer.post_attention_layernorm, h)
        h = h + lin(m.down_proj, torch.nn.functional.silu(lin(m.gate_proj, x)) * lin(m.up_proj, x))
    return [ChunkKV([k[c : c + 1].contiguous() for k in keys], [v[c : c + 1].contiguous() for v in values], 0)
            for c in range(C)]


def _prepare_prefill(case, seed):
    s, gen, lay = SHAPES[case["shape"]], _gen(seed), _layout(case, seed)
    model = _Model(s, gen).eval()
    L = case["chunk_len"]
    toks = torch.randint(1, VOCAB, (case["chunks"], L), generator=gen, device=DEV)
    tail = torch.randint(1, VOCAB, (case["tail"],), generator=gen, device=DEV).tolist()
    chunks = _chunk_kv(model, s, toks)
    toks = toks.tolist()
    tokens = [t for c in lay["order"] for t in toks[c]] + tail
    placements = [Placement(chunks[c], i * L) for i, c in enumerate(lay["order"])]
    return {"engine": HipEngine(model, _Tokenizer()), "tokens": tokens, "placements": placements,
            "config": BlendConfig(recompute_ratio=case["ratio"], n_sink=case["n_sink"])}


_PREPARE = {"attention": _prepare_attention, "repair": _prepare_repair, "gather": _prepare_gather,
            "extract": _prepare_extract, "layer": _prepare_layer, "prefill": _prepare_prefill}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    state["kind"] = case["kind"]
    return state


# ---- one pass -------------------------------------------------------------------------------


def _run_attention(st):
    return ops.attention_active(st["q"], st["K"], st["V"], st["pos"])


def _run_repair(st):
    s, plan, K, V, err = SHAPES[st["case"]["shape"]], st["plan"], st["K"], st["V"], st["err"]
    n_seg, most, hkv, d, layers = len(plan.segments), plan.max_seg_tokens, s["hkv"], s["d"], s["layers"]
    Ks, Vs = K.unbind(0), V.unbind(0)
    ops.rope_qkv(None, *st["proj"][0], st["layer0"], 0, hkv, d, THETA, k_out=Ks[0], v_out=Vs[0], rows=st["layer0"],
                 err=err)
    if st["case"]["exact"]:  # layer 0's rows of the chunk reused under its own prefix
        ops.rerope_gather(K, V, st["tab"], st["segs"], n_seg, most, THETA, err, layers=(0, 1), skip=st["local"])
    diff, norm, sel = ops.layer1_repair_gather(K, V, st["tab"], 1, (2, layers), st["segs"], n_seg, most, st["k1"],
                                               st["v1"], st["flags"], st["local"], st["spans"], None, THETA, st["ws"],
                                               err)
    kept = sel.keep_abs[: plan.n_keep]
    for li in range(2, layers):
        ops.rope_qkv(None, *st["proj"][li], kept, 0, hkv, d, THETA, k_out=Ks[li], v_out=Vs[li], rows=kept, err=err)
    return {"K": K, "V": V, "kept": kept, "local": sel.keep_local[: plan.n_keep], "rank": sel.keep_rank, "diff": diff,
            "norm": norm, "rel_dev": sel.rel_dev, "escalated": sel.escalated, "err": err}


def _run_gather(st):
    ops.rerope_gather(st["K"], st["V"], st["tab"], st["segs"], len(st["plan"].segments), st["plan"].max_seg_tokens,
                      THETA, st["err"])
    return [st["K"], st["V"]]


def _run_extract(st):
    return ops.extract_chunks(st["K"], st["V"], st["spans"])


def _run_layer(st):
    s = st["shape"]
    qd, kd = s["hq"] * s["d"], s["hkv"] * s["d"]
    h, x = ops.add_rmsnorm(st["h"], st["mlp_out"], st["w_in"], 1e-6)
    qkv = st["qkv"]
    q, _ = ops.rope_qkv(qkv[..., :qd], qkv[..., qd : qd + kd], qkv[..., qd + kd :], st["pos"], s["hq"], s["hkv"],
                        s["d"], THETA, k_out=st["K"], v_out=st["V"], rows=st["pos"])
    h2, y = ops.add_rmsnorm(h, st["attn_out"], st["w_post"], 1e-6)
    gu = st["gate_up"]
    return {"h": h, "x": x, "q": q, "K": st["K"], "V": st["V"], "h2": h2, "y": y,
            "act": ops.silu_mul(gu[..., : s["inter"]], gu[..., s["inter"] :])}


def _run_prefill(st):
    r = st["engine"].prefill(st["tokens"], st["placements"], st["config"])
    return {"logits": r.logits, "keys": r.keys, "values": r.values}


_RUN = {"attention": _run_attention, "repair": _run_repair, "gather": _run_gather, "extract": _run_extract,
        "layer": _run_layer, "prefill": _run_prefill}


def run(state):
    return _RUN[state["kind"]](state)


# ---- what a pass cannot do without ----------------------------------------------------------


def work(case):
    s, kind = SHAPES[case["shape"]], case["kind"]
    eb = 4 if case.get("dtype") == "f32" else 2
    row = s["hkv"] * s["d"] * eb  # one token's keys (or values) of one layer
    if kind == "attention":
        nq, n, pairs = _attention_sizes(case)
        used = case["n"] + 1 if case["form"] == "decode" else n
        return {"bytes": 2 * nq * s["hq"] * s["d"] * 2 + 2 * used * row + 8 * nq, "flops": 4 * pairs * s["hq"] * s["d"]}
    if kind == "layer":
        n, qkv = case["rows"], (s["hq"] + 2 * s["hkv"]) * s["d"]
        # h, mlp_out, attn_out in; h, x, h2, y out; qkv in and out; gate, up in, product out
        return {"bytes": n * eb * (7 * s["hidden"] + 2 * qkv + 3 * s["inter"]),
                "flops": n * (12 * s["hidden"] + 3 * qkv + 8 * s["inter"])}
    C, L, n = case["chunks"], case["chunk_len"], _n_tokens(case)
    if kind in ("gather", "extract"):
        return {"bytes": 4 * s["layers"] * C * L * row, "flops": 3 * s["layers"] * C * L * row // eb if kind == "gather" else 0}
    first = L if case.get("exact") else 0  # positions reused as they are
    pooled = (C * L - first) // L
    sinks = min(L, case["n_sink"])
    kept = min(pooled * int(round(case["ratio"] * L)), pooled * (L - sinks)) + pooled * sinks + case["tail"]
    if kind == "repair":
        # written: every row of every layer. Read: layer 0's and 1's computed rows, the other
        # layers' kept rows; the cached rows that stay, and at layer 1 (the deviation) all.
        reads = 2 * (n - first) + (s["layers"] - 2) * kept + first + C * L + (s["layers"] - 2) * (n - kept)
        moved = 2 * row * (reads + s["layers"] * n) + n * (8 + 4 + 4 + 5) + 16 * kept
        return {"bytes": moved, "flops": 3 * s["layers"] * n * row // eb + 8 * n * row // eb}
    hid, qkv = s["hidden"], (s["hq"] + 2 * s["hkv"]) * s["d"]
    per_row = 2 * (hid * qkv + s["hq"] * s["d"] * hid + 3 * hid * s["inter"])
    weights = s["layers"] * per_row + 2 * VOCAB * hid
    pos = _kept_positions(case, 0)
    pairs = 2 * n * (n + 1) // 2 + (s["layers"] - 2) * int((pos + 1).sum())
    return {"bytes": weights + 2 * row * s["layers"] * (n + C * L) + 2 * VOCAB,
            "flops": per_row * (2 * n + (s["layers"] - 2) * kept) + 4 * pairs * s["hq"] * s["d"] + 2 * hid * VOCAB}


def tolerance(case):
    kind = case["kind"]
    if kind == "attention":
        # bf16 weights and outputs: two correct kernels differ by their roundings (2.4e-3 measured
        # against 64 bits)
        return {"rel": 8e-3, "max": 0.1}
    if kind == "layer":
        # another order of the fp32 sum of squares, another exp: a few results round the other way
        return {"rel": 2e-3, "max": 0.04} if case["dtype"] == "bf16" else {"rel": 1e-5, "max": 1e-4}
    if kind == "prefill":
        # the logits with the attention in fp32 or fp64 instead: 5.4e-3 (rel), caches 3e-3; max 0.1
        return {"rel": 0.02, "max": 0.4}
    # copies, rotations of correctly rounded tables and sums in a stated order: bit for bit
    return "exact"


# ---- the same results in 64 bits ------------------------------------------------------------


def _exact_attention(case, st):
    s = SHAPES[case["shape"]]
    group, n = s["hq"] // s["hkv"], st["K"].shape[2]
    out = torch.empty((1, st["q"].shape[2], s["hq"], s["d"]), dtype=torch.float64, device=DEV)
    hide = torch.arange(n, device=DEV)[None, :] > st["pos"][:, None]
    for h in range(s["hq"]):
        k, v = st["K"][0, h // group].double(), st["V"][0, h // group].double()
        w = st["q"][0, h].double() @ k.t().contiguous() / math.sqrt(s["d"])
        out[0, :, h] = torch.softmax(w.masked_fill_(hide, float("-inf")), -1) @ v
    return out


def _exact_repair(case, st):
    s, plan, n = SHAPES[case["shape"]], st["plan"], st["plan"].n_tokens
    hkv, d, inv = s["hkv"], s["d"], _inv_freq(s["d"])
    dtype = st["k1"].dtype
    # deviation of the stored rows (a difference is taken in the cache's type), sums in 64 bits
    bk, bv = _base_rows(st["placements"], 1, n, hkv, d, dtype)
    at = st["layer0"]
    sq = lambda t: t.double().square().sum((0, 1, 3))  # noqa: E731
    diff, norm = torch.zeros(n, dtype=torch.float64, device=DEV), torch.zeros(n, dtype=torch.float64, device=DEV)
    diff[at] = sq(st["k1"] - bk[:, :, at]) + sq(st["v1"] - bv[:, :, at])
    norm[at] = sq(st["k1"]) + sq(st["v1"])
    host = diff.cpu().numpy()
    keep = ~plan.cached | plan.sink
    cand = np.zeros(n, dtype=bool)
    for a, length, _, pooled in plan.spans:
        cand[a : a + length] |= bool(pooled)
    cand = np.flatnonzero(cand & ~keep)
    keep[cand[np.argsort(-host[cand], kind="stable")[: plan.budget]]] = True
    kept_np = np.flatnonzero(keep)
    kept, local = torch.from_numpy(kept_np).to(DEV), torch.from_numpy(plan.layer0_idx.searchsorted(kept_np)).to(DEV)
    rank = torch.full((n,), -1, dtype=torch.int64, device=DEV)
    rank[kept] = torch.arange(len(kept_np), device=DEV)
    rel = torch.stack([diff[a : a + length].sum() / norm[a : a + length].sum() for a, length, _, _ in plan.spans.tolist()])
    K, V = (torch.zeros(t.shape, dtype=torch.float64, device=DEV) for t in (st["K"], st["V"]))
    for p in st["placements"]:
        to = slice(p.start, p.start + p.chunk.length)
        delta = torch.full((p.chunk.length,), float(p.start - p.chunk.start), device=DEV)
        K[:, :, :, to] = _rotate(torch.stack(p.chunk.keys), delta, inv)
        V[:, :, :, to] = torch.stack(p.chunk.values).double()
    heads = lambda t: t[0].view(t.shape[1], hkv, d).transpose(0, 1)  # noqa: E731
    for li in range(s["layers"]):
        if li == 1:
            K[1, 0][:, kept], V[1, 0][:, kept] = st["k1"][0][:, local].double(), st["v1"][0][:, local].double()
            continue
        rows = at if li == 0 else kept
        k, v = (heads(t) for t in st["proj"][li])
        K[li, 0][:, rows], V[li, 0][:, rows] = _rotate(k, rows, inv), v.double()
    return {"K": K, "V": V, "kept": None, "local": None, "rank": None, "diff": diff, "norm": norm, "rel_dev": rel,
            "escalated": None, "err": None}


def _exact_gather(case, st):
    inv = _inv_freq(SHAPES[case["shape"]]["d"])
    K, V = (torch.zeros(t.shape, dtype=torch.float64, device=DEV) for t in (st["K"], st["V"]))
    for p in st["placements"]:
        to = slice(p.start, p.start + p.chunk.length)
        delta = torch.full((p.chunk.length,), float(p.start - p.chunk.start), device=DEV)
        K[:, :, :, to] = _rotate(torch.stack(p.chunk.keys), delta, inv)
        V[:, :, :, to] = torch.stack(p.chunk.values).double()
    return [K, V]


def _exact_layer(case, st):
    s = st["shape"]
    inv, n, rows = _inv_freq(s["d"]), case["rows"], st["pos"]
    qd, kd = s["hq"] * s["d"], s["hkv"] * s["d"]

    def norm(h, w):
        return w.double() * h * torch.rsqrt(h.square().mean(-1, keepdim=True) + 1e-6)

    h = st["h"].double() + st["mlp_out"].double()
    h2 = h + st["attn_out"].double()
    qkv = st["qkv"].double()
    heads = lambda t, k: t[0].view(n, k, s["d"]).transpose(0, 1)  # noqa: E731
    K, V = (torch.zeros(t.shape, dtype=torch.float64, device=DEV) for t in (st["K"], st["V"]))
    K[0][:, rows] = _rotate(heads(qkv[..., qd : qd + kd], s["hkv"]), rows, inv)
    V[0][:, rows] = heads(qkv[..., qd + kd :], s["hkv"])
    gate, up = st["gate_up"].double().chunk(2, -1)
    return {"h": h, "x": norm(h, st["w_in"]), "q": _rotate(heads(qkv[..., :qd], s["hq"]), rows, inv).transpose(0, 1)[None],
            "K": K, "V": V, "h2": h2, "y": norm(h2, st["w_post"]), "act": gate * torch.sigmoid(gate) * up}


def exact(case, seed):
    """What run() returns, in 64 bits. None for the extraction (a copy) and for the whole prefill:
    which positions it recomputes follows from 16-bit activations, so another precision is another
    request."""
    kind = case["kind"]
    if kind in ("extract", "prefill"):
        return None
    made = {"attention": _exact_attention, "repair": _exact_repair, "gather": _exact_gather, "layer": _exact_layer}
    return made[kind](case, prepare(case, seed))
