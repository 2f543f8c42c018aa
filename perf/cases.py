"""The work that programs on this framework have it do, as cases to be timed.

A serving program runs a Llama-shaped model step by step, each step through the
tensor-core path (bf16, stride_amd.harness and stride_amd.engine) or the exact path
(fp32, stride_amd.exact). A step is made of blocks, and each case is one pass of one
block through the public operators, or one whole step:

  attn  RMSNorm, fused QKV with RoPE and paged-KV append, paged attention, O
        projection with residual. "decode": each row is the next token of a sequence
        of its own, at ragged positions; "prefill": the rows are consecutive prompt
        positions of a few sequences, after `past` positions that are cached already.
  mlp   RMSNorm, gate/up with SiLU, down projection with residual.
  head  final RMSNorm and the LM head: greedy argmax (serving), or full logits.
  step  a whole decode step of the engine, from the host's row list to logits.

The shapes are those of the repository's benchmark and tests: hidden 2048, 32 query
and 8 KV heads of 64, FFN 8192, vocabulary 128256, 16-token KV pages (64 on the exact
path), weights ~N(0, 0.02), contexts of up to 2048 positions; draw() adds other widths.
"""
import math

import numpy as np
import torch

from stride_amd import exact as ex
from stride_amd import engine, harness, layout, tc
from stride_amd._lib import (AttentionParams, GemmResidualParams, KvRef, LmFullParams, LmGreedyParams, Mlp13Params,
                             NormParams, QkvParams)
from stride_amd.weights import ModelConfig, Weights

DEV = "cuda:0"
EPS = 1e-5
THETA = 500000.0
BASE = dict(hidden=2048, heads=32, head_dim=64, mlp=8192, vocab=128256)


# ---------------------------------------------------------------------------
# The cases.

def listed():
    def attn(name, path, phase, rows, seqs, ctx, past=0, page=16):
        return dict(name=name, path=path, block="attn", phase=phase, rows=rows, seqs=seqs, ctx=ctx, past=past,
                    page=page if path == "tc" else 64, **BASE)

    def mlp(name, path, rows):
        return dict(name=name, path=path, block="mlp", rows=rows, **BASE)

    def head(name, path, rows, full):
        return dict(name=name, path=path, block="head", rows=rows, full=full, **BASE)

    return [
        # One user: a single token per step, where latency and launches count.
        attn("tc_attn_decode_1", "tc", "decode", 1, 1, 384),
        # The benchmark's serving batch, 256-token prompts part way through 256 new tokens.
        attn("tc_attn_decode_128", "tc", "decode", 128, 128, 512),
        # Prompts of about 256 tokens prefilled together, a ragged 1000-row chunk.
        attn("tc_attn_prefill_1000", "tc", "prefill", 1000, 4, 256),
        # One prompt of the longest context the reference serves.
        attn("tc_attn_prefill_2048", "tc", "prefill", 2048, 1, 2048, page=64),
        # A medium decode batch.
        mlp("tc_mlp_32", "tc", 32),
        # The benchmark's prefill size.
        mlp("tc_mlp_2048", "tc", 2048),
        # The greedy head of a decode step.
        head("tc_head_greedy_64", "tc", 64, False),
        # A whole decode step of the 16-layer model, rows described on the host.
        dict(name="tc_step_64", path="tc", block="step", rows=64, ctx=384, layers=16, page=16, **BASE),
        # The exact path: one user's token, a decode batch, a prompt, full logits.
        mlp("exact_mlp_1", "exact", 1),
        attn("exact_attn_decode_32", "exact", "decode", 32, 32, 384),
        attn("exact_attn_prefill_256", "exact", "prefill", 256, 1, 256),
        head("exact_head_full_8", "exact", 8, True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    # Mostly the benchmark's model; else another width, with its own head size and FFN.
    if rng.random() < 0.6:
        m = dict(BASE)
    else:
        hidden, head_dim = rng.choice([(1024, 64), (1024, 32), (1536, 64), (2048, 128), (3072, 128)])
        mlp = rng.choice([2816, 4096, 5632, 8192])
        m = dict(hidden=hidden, heads=hidden // head_dim, head_dim=head_dim, mlp=mlp, vocab=rng.choice([32000, 50257, 128256]))
    most = 2048 * 2048 // max(2048, m["hidden"])  # rows of a prefill chunk: wider models take fewer
    path = "tc" if rng.random() < 0.6 else "exact"
    block = rng.choice(["attn", "attn", "attn", "mlp", "mlp", "head"])
    if block == "attn":
        page = rng.choice([16, 64]) if path == "tc" else 64
        if rng.random() < 0.5:
            rows = _log_int(rng, 1, 128 if path == "tc" else 64)
            ctx = _log_int(rng, 40, min(2048, 65536 // rows))
            return dict(path=path, block=block, phase="decode", rows=rows, seqs=rows, ctx=ctx, past=0, page=page, **m)
        rows = _log_int(rng, 17, most if path == "tc" else most // 8)
        seqs = rng.randint(1, min(8, max(1, rows // 16)))
        each = -(-rows // seqs)
        past = min(rng.choice([0, 0, rng.randint(1, 512)]), 2048 - each)
        ctx = past + each
        return dict(path=path, block=block, phase="prefill", rows=rows, seqs=seqs, ctx=ctx, past=past, page=page, **m)
    if block == "mlp":
        return dict(path=path, block=block, rows=_log_int(rng, 1, most if path == "tc" else most // 8), **m)
    full = rng.random() < 0.4
    return dict(path=path, block=block, rows=_log_int(rng, 1, 64 if path == "tc" else 12), full=full, **m)


# ---------------------------------------------------------------------------
# Inputs, row-major, from the seed alone.

def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed(seed * 1000 + salt)


def _w(g, n, k):
    """bf16 weights ~N(0, 0.02)."""
    return (torch.randn(n, k, generator=g, device=DEV) * 0.02).to(torch.bfloat16)


def _gain(g, n):
    return 1.0 + 0.1 * torch.randn(n, generator=g, device=DEV)


def _rope(positions, head_dim):
    """[positions][head_dim/2][cos, sin] fp32."""
    inv = 1.0 / THETA ** (np.arange(0, head_dim, 2) / head_dim)
    ang = (np.arange(positions)[:, None] * inv[None, :]).astype(np.float32).astype(np.float64)
    return torch.from_numpy(np.stack([np.cos(ang), np.sin(ang)], -1).astype(np.float32)).to(DEV)


def _rows(case, seed):
    """(slot, position) of every row."""
    r = np.random.default_rng(seed)
    n, seqs = case["rows"], case["seqs"]
    order = r.permutation(seqs)
    if case["phase"] == "decode":
        lo = max(1, case["ctx"] // 2)
        return [(int(order[i]), int(p) - 1) for i, p in enumerate(r.integers(lo, case["ctx"] + 1, n))]
    out, left = [], n
    for i in range(seqs):
        take = -(-left // (seqs - i))
        out += [(int(order[i]), case["past"] + p) for p in range(take)]
        left -= take
    return out


def _attn_inputs(case, seed):
    g = _gen(seed, 1)
    H, heads, D, n = case["hidden"], case["heads"], case["head_dim"], case["rows"]
    kvh = heads // 4
    blocks = -(-case["ctx"] // case["page"])
    dense_t = torch.bfloat16 if case["path"] == "tc" else torch.float32
    cap = blocks * case["page"]
    return dict(
        q=_w(g, heads * D, H), k=_w(g, kvh * D, H), v=_w(g, kvh * D, H), o=_w(g, H, heads * D), gain=_gain(g, H),
        h=torch.randn(n, H, generator=g, device=DEV), rope=_rope(case["ctx"], D), rows=_rows(case, seed),
        # cached K and V [2][slot][KV head][position][dim], and where their pages lie
        kv=torch.randn(2, case["seqs"], kvh, cap, D, generator=g, device=DEV).to(dense_t),
        table=torch.from_numpy(np.random.default_rng(seed + 7).permutation(case["seqs"] * blocks).astype(np.int32)
                               .reshape(case["seqs"], blocks)).to(DEV))


def _arena(kv, table, page):
    """Paged arena [block][layer 0][K|V][KV head][token][dim] of dense K and V."""
    _, slots, kvh, cap, D = kv.shape
    blocks = cap // page
    a = torch.empty(slots * blocks, 2, kvh, page, D, dtype=kv.dtype, device=DEV)
    a[table.long().reshape(-1)] = (kv.reshape(2, slots, kvh, blocks, page, D).permute(1, 3, 0, 2, 4, 5)
                                   .reshape(slots * blocks, 2, kvh, page, D))
    return a


def _mlp_inputs(case, seed):
    g = _gen(seed, 2)
    H, F = case["hidden"], case["mlp"]
    return dict(w1=_w(g, F, H), w3=_w(g, F, H), w2=_w(g, H, F), gain=_gain(g, H),
                h=torch.randn(case["rows"], H, generator=g, device=DEV))


def _head_inputs(case, seed):
    g = _gen(seed, 3)
    return dict(w=_w(g, case["vocab"], case["hidden"]), gain=_gain(g, case["hidden"]),
                h=torch.randn(case["rows"], case["hidden"], generator=g, device=DEV))


# ---------------------------------------------------------------------------
# States: the buffers and packed weights an engine keeps.

def _i16(w):
    return w.view(torch.int16)


def _int(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _items(rows):
    """Every 64-position page of every row, as the engine lists them."""
    return _int([x for j, (_, p) in enumerate(rows) for page in range((p >> 6) + 1) for x in (j, page)])


def prepare(case, seed):
    return globals()["_prepare_%s_%s" % (case["path"], case["block"])](case, seed)


def _prepare_tc_attn(case, seed):
    i = _attn_inputs(case, seed)
    n, D, heads = case["rows"], case["head_dim"], case["heads"]
    kvh, page, lt = heads // 4, case["page"], -(-n // 16)
    arena = _i16(_arena(i["kv"], i["table"], page)).reshape(-1)
    group = page * D
    ref = KvRef(tc.ptr(arena), tc.ptr(i["table"]), group * kvh * 2, group * kvh * 2, group * kvh, group,
                int(i["table"].shape[1]), D)
    max_pages = -(-case["ctx"] // 64)
    pack = lambda name, rope: layout.pack_tiles(_i16(i[name]), layout.rope_rows(i[name].shape[0], D) if rope else None)  # noqa: E731
    zeros = lambda cols: torch.zeros((lt, cols // 16, 16, 16), dtype=torch.int16, device=DEV)  # noqa: E731
    return dict(case=case, q=pack("q", True), k=pack("k", True), v=pack("v", True), o=pack("o", False), gain=i["gain"],
                h=layout.lane_tiles(i["h"]), rope=i["rope"], kv=harness.PagedKv(arena, i["table"], ref, page, ref.max_blocks),
                slot=_int([r[0] for r in i["rows"]]), pos=_int([r[1] for r in i["rows"]]), items=_items(i["rows"]),
                x=zeros(case["hidden"]), attn=zeros(heads * D), max_pages=max_pages,
                q_out=torch.zeros((n, heads * D), dtype=torch.float32, device=DEV),
                scratch=torch.zeros(n * kvh * max_pages * (4 * D + 8), dtype=torch.float32, device=DEV))


def _prepare_exact_attn(case, seed):
    i = _attn_inputs(case, seed)
    n, D, heads = case["rows"], case["head_dim"], case["heads"]
    kvh, page = heads // 4, case["page"]
    stride = ex.lane_shape(n)[2]
    arena = _arena(i["kv"], i["table"], page).reshape(-1)
    group = page * D
    max_pages = -(-case["ctx"] // 64)
    pack = lambda name, rope: ex.pack_groups(_i16(i[name]), ex.rope_group_rows(i[name].shape[0], D) if rope else None)  # noqa: E731
    zeros = lambda cols: torch.zeros((cols, stride), dtype=torch.float32, device=DEV)  # noqa: E731
    return dict(case=case, q=pack("q", True), k=pack("k", True), v=pack("v", True), o=pack("o", False), gain=i["gain"],
                h=ex.dim_major(i["h"], stride), rope=i["rope"], arena=arena, table=i["table"],
                kv=KvRef(tc.ptr(arena), tc.ptr(i["table"]), group * kvh * 2, group * kvh * 2, group * kvh, group,
                         int(i["table"].shape[1]), D),
                slot=_int([r[0] for r in i["rows"]]), pos=_int([r[1] for r in i["rows"]]), items=_items(i["rows"]),
                x=zeros(case["hidden"]), attn=zeros(heads * D), max_pages=max_pages,
                q_out=torch.zeros((stride, heads * D), dtype=torch.float32, device=DEV),
                scratch=torch.zeros(n * kvh * max_pages * (4 * D + 8), dtype=torch.float32, device=DEV))


def _prepare_tc_mlp(case, seed):
    i = _mlp_inputs(case, seed)
    lt = -(-case["rows"] // 16)
    zeros = lambda cols: torch.zeros((lt, cols // 16, 16, 16), dtype=torch.int16, device=DEV)  # noqa: E731
    return dict(case=case, gain=i["gain"], h=layout.lane_tiles(i["h"]), x=zeros(case["hidden"]), z=zeros(case["mlp"]),
                **{k: layout.pack_tiles(_i16(i[k])) for k in ("w1", "w3", "w2")})


def _prepare_exact_mlp(case, seed):
    i = _mlp_inputs(case, seed)
    stride = ex.lane_shape(case["rows"])[2]
    zeros = lambda cols: torch.zeros((cols, stride), dtype=torch.float32, device=DEV)  # noqa: E731
    return dict(case=case, gain=i["gain"], h=ex.dim_major(i["h"], stride), x=zeros(case["hidden"]), z=zeros(case["mlp"]),
                **{k: ex.pack_groups(_i16(i[k])) for k in ("w1", "w3", "w2")})


def _prepare_tc_head(case, seed):
    i = _head_inputs(case, seed)
    n, lt, rt = case["rows"], -(-case["rows"] // 16), -(-case["vocab"] // 16)
    return dict(case=case, gain=i["gain"], h=layout.lane_tiles(i["h"]), w=layout.pack_tiles(_i16(i["w"]), None, rt),
                x=torch.zeros((lt, case["hidden"] // 16, 16, 16), dtype=torch.int16, device=DEV),
                best=harness.best_init(n, DEV),
                logits=torch.zeros((rt, lt, 16, 16), dtype=torch.float32, device=DEV) if case["full"] else None)


def _prepare_exact_head(case, seed):
    i = _head_inputs(case, seed)
    n, stride = case["rows"], ex.lane_shape(case["rows"])[2]
    w = ex.pack_groups(_i16(i["w"]))
    return dict(case=case, gain=i["gain"], h=ex.dim_major(i["h"], stride), w=w,
                x=torch.zeros((case["hidden"], stride), dtype=torch.float32, device=DEV), best=harness.best_init(n, DEV),
                logits=torch.zeros((w.shape[0] * 4, stride), dtype=torch.float32, device=DEV) if case["full"] else None)


def _step_config(case):
    return ModelConfig(hidden=case["hidden"], mlp=case["mlp"], layers=case["layers"], heads=case["heads"],
                       kv_heads=case["heads"] // 4, head_dim=case["head_dim"], vocab=case["vocab"], rms_eps=EPS)


def _step_layers(case, seed):
    """The layers' row-major weights, one after the other."""
    H, F, A = case["hidden"], case["mlp"], case["heads"] * case["head_dim"]
    for li in range(case["layers"]):
        g = _gen(seed, 100 + li)
        yield dict(q=_w(g, A, H), k=_w(g, A // 4, H), v=_w(g, A // 4, H), o=_w(g, H, A), w1=_w(g, F, H), w3=_w(g, F, H),
                   w2=_w(g, H, F), norm_attn=_gain(g, H), norm_mlp=_gain(g, H))


def _step_rows(case, seed):
    r = np.random.default_rng(seed)
    slots = r.permutation(case["rows"])
    pos = r.integers(case["ctx"] // 2, case["ctx"], case["rows"])
    tok = r.integers(0, case["vocab"], case["rows"])
    return [(int(s), int(p), int(t)) for s, p, t in zip(slots, pos, tok)]


def _step_arena(case, seed):
    """Cached K and V of every layer, and the page table."""
    blocks = -(-case["ctx"] // case["page"])
    n = case["rows"] * blocks
    a = torch.empty(n, case["layers"], 2, case["heads"] // 4, case["page"], case["head_dim"], dtype=torch.bfloat16, device=DEV)
    g = _gen(seed, 90)
    for li in range(case["layers"]):
        a[:, li] = torch.randn(a[:, li].shape, generator=g, device=DEV).to(torch.bfloat16)
    table = np.random.default_rng(seed + 7).permutation(n).astype(np.int32).reshape(case["rows"], blocks)
    return a, torch.from_numpy(table).to(DEV)


def _prepare_tc_step(case, seed):
    cfg, D = _step_config(case), case["head_dim"]
    g = _gen(seed, 4)
    pack = lambda w, rope: layout.pack_tiles(_i16(w), layout.rope_rows(w.shape[0], D) if rope else None)  # noqa: E731
    embed = layout.pack_tiles(_i16(_w(g, cfg.vocab, cfg.hidden)), None, -(-cfg.vocab // 16))
    layers = [{k: w if k.startswith("norm") else pack(w, k in "qkv") for k, w in L.items()} for L in _step_layers(case, seed)]
    weights = Weights(cfg, embed, embed, layers, _gain(g, cfg.hidden), _rope(case["ctx"], D))
    eng = engine.Engine(weights, case["rows"], case["ctx"], case["rows"], case["page"])
    arena, table = _step_arena(case, seed)
    eng.kv.arena.copy_(_i16(arena).reshape(-1))
    eng.kv.table.copy_(table)
    return dict(case=case, eng=eng, rows=_step_rows(case, seed),
                logits=torch.zeros((embed.shape[0], -(-case["rows"] // 16), 16, 16), dtype=torch.float32, device=DEV))


# ---------------------------------------------------------------------------
# Passes.

def run(state):
    case = state["case"]
    return globals()["_run_%s_%s" % (case["path"], case["block"])](state, case)


def _run_tc_attn(s, c):
    n, D = c["rows"], c["head_dim"]
    harness.norm(s["h"], n, s["gain"], EPS, x_out=s["x"])
    harness.qkv(s["q"], s["k"], s["v"], s["x"], n, D, s["rope"], s["slot"], s["pos"], s["kv"], q_out=s["q_out"])
    harness.attention(s["q_out"], s["kv"], s["slot"], s["pos"], c["heads"] // 4, D, float(D ** -0.5),
                      max_pages=s["max_pages"], out_tiles=s["attn"], items=s["items"], scratch=s["scratch"])
    harness.gemm_residual(s["o"], s["attn"], s["h"], n)
    return dict(h=s["h"], q=s["q_out"], attn=s["attn"].view(torch.bfloat16), kv=s["kv"].arena.view(torch.bfloat16))


def _run_exact_attn(s, c):
    n, D, H, A = c["rows"], c["head_dim"], c["hidden"], c["heads"] * c["head_dim"]
    J, lanes = ex.lane_shape(n)[0], ex.lanes(n)
    P = tc.ptr
    ex.k_norm(NormParams(lanes, P(s["h"]), P(s["x"]), P(s["gain"]), H, EPS), J)
    ex.k_qkv(QkvParams(lanes, P(s["x"]), ex.mat(s["q"], H), ex.mat(s["k"], H), ex.mat(s["v"], H), P(s["q_out"]), A,
                       s["kv"], P(s["rope"]), P(s["slot"]), P(s["pos"]), 0, D), J)
    a = AttentionParams()
    a.l = lanes
    a.q, a.q_stride, a.out, a.out_cols, a.kv = P(s["q_out"]), A, P(s["attn"]), A, s["kv"]
    a.row_slot, a.row_pos, a.items, a.item_count = P(s["slot"]), P(s["pos"]), P(s["items"]), s["items"].numel() // 2
    a.scratch, a.max_pages, a.rec_floats = P(s["scratch"]), s["max_pages"], 4 * D + 8
    a.layer, a.n_kv, a.n_q, a.head_dim, a.scale = 0, c["heads"] // 4, 4, D, float(D ** -0.5)
    ex.k_attention(a)
    ex.k_gemm_residual(GemmResidualParams(lanes, P(s["attn"]), ex.mat(s["o"], A), P(s["h"])), J)
    return dict(h=s["h"], q=s["q_out"], attn=s["attn"], kv=s["arena"])


def _run_tc_mlp(s, c):
    n = c["rows"]
    harness.norm(s["h"], n, s["gain"], EPS, x_out=s["x"])
    harness.mlp13(s["w1"], s["w3"], s["x"], n, out=s["z"])
    harness.gemm_residual(s["w2"], s["z"], s["h"], n)
    return dict(h=s["h"], z=s["z"].view(torch.bfloat16))


def _run_exact_mlp(s, c):
    n, H, F = c["rows"], c["hidden"], c["mlp"]
    J, lanes = ex.lane_shape(n)[0], ex.lanes(n)
    P = tc.ptr
    ex.k_norm(NormParams(lanes, P(s["h"]), P(s["x"]), P(s["gain"]), H, EPS), J)
    ex.k_mlp13(Mlp13Params(lanes, P(s["x"]), ex.mat(s["w1"], H), ex.mat(s["w3"], H), P(s["z"])), J)
    ex.k_gemm_residual(GemmResidualParams(lanes, P(s["z"]), ex.mat(s["w2"], F), P(s["h"])), J)
    return dict(h=s["h"], z=s["z"])


def _best(best):
    return dict(value=best.view(torch.float32)[:, 0], index=best[:, 1])


def _run_tc_head(s, c):
    n = c["rows"]
    harness.norm(s["h"], n, s["gain"], EPS, x_out=s["x"])
    if c["full"]:
        return dict(x=s["x"].view(torch.bfloat16), logits=harness.lm_full(s["w"], s["x"], n, out=s["logits"]))
    harness.best_reset(s["best"])
    harness.lm_greedy(s["w"], s["x"], n, c["vocab"], best=s["best"])
    return dict(x=s["x"].view(torch.bfloat16), **_best(s["best"]))


def _run_exact_head(s, c):
    n, H = c["rows"], c["hidden"]
    J, lanes = ex.lane_shape(n)[0], ex.lanes(n)
    P = tc.ptr
    ex.k_norm(NormParams(lanes, P(s["h"]), P(s["x"]), P(s["gain"]), H, EPS), J)
    if c["full"]:
        ex.k_lm_full(LmFullParams(lanes, P(s["x"]), ex.mat(s["w"], H), P(s["logits"])), J)
        return dict(x=s["x"], logits=s["logits"])
    harness.best_reset(s["best"])
    ex.k_lm_greedy(LmGreedyParams(lanes, P(s["x"]), ex.mat(s["w"], H), c["vocab"], P(s["best"])), J)
    return dict(x=s["x"], **_best(s["best"]))


def _run_tc_step(s, c):
    eng, n = s["eng"], c["rows"]
    slot, pos, tok, items = eng.device_rows(s["rows"])
    best = torch.empty((n, 2), dtype=torch.int32, device=DEV)
    eng.launch(n, slot, pos, tok, items, best=best)
    harness.lm_full(eng.w.lm, eng.x, n, out=s["logits"])
    return dict(logits=s["logits"], **_best(best))


# ---------------------------------------------------------------------------
# What a pass cannot do without.

def _visible(case, seed=0):
    if case["block"] == "step":
        return [p + 1 for _, p, _ in _step_rows(case, seed)]
    return [p + 1 for _, p in _rows(case, seed)]


def work(case):
    n, H, F, V = case["rows"], case["hidden"], case["mlp"], case["vocab"]
    A = case["heads"] * case["head_dim"]
    kv_size = 2 if case["path"] == "tc" else 4

    def attn():
        vis = _visible(case)
        if case.get("phase") == "prefill":  # each sequence's cached positions once
            cached = case["rows"] + case["seqs"] * case["past"]
        else:
            cached = sum(vis)
        nbytes = 2 * (A + A // 2) * H + 2 * H * A + 8 * n * H + cached * (A // 4) * 2 * kv_size + n * (A // 2) * kv_size
        return nbytes, 2 * n * H * (A + A // 2) + 2 * n * A * H + 4 * A * sum(vis)

    def mlp():
        return 2 * 3 * H * F + 8 * n * H, 2 * n * 3 * H * F

    def head(full):
        return 2 * V * H + 4 * n * H + (4 * n * V if full else 8 * n), 2 * n * V * H

    if case["block"] == "attn":
        b, f = attn()
    elif case["block"] == "mlp":
        b, f = mlp()
    elif case["block"] == "head":
        b, f = head(case["full"])
    else:
        (ab, af), (mb, mf), (hb, hf) = attn(), mlp(), head(True)
        b, f = case["layers"] * (ab + mb) + hb, case["layers"] * (af + mf) + hf
    return {"bytes": b, "flops": f}


def tolerance(case):
    # The exact path's contract is the reference's bits.
    if case["path"] == "exact":
        return "exact"
    # bf16 roundings of activations, K and V; measured against 64 bits, times four.
    if case["block"] == "step":
        return {"rel": 3e-2, "max": 0.3, "differ": 0.01}
    if case["block"] == "attn":
        return {"rel": 1.2e-2, "max": 0.15}
    if case["block"] == "mlp":
        return {"rel": 1.2e-2, "max": 0.15}
    return {"rel": 8e-3, "max": 0.05, "differ": 0.01}


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch.

def _norm64(h, gain):
    h = h.double()
    return gain.double() * (h / torch.sqrt((h * h).mean(1, keepdim=True) + EPS))


def _mm(x, w):
    return x @ w.double().t()


def _rope64(y, pos, rope, D):
    """Rotated [rows][heads][D]."""
    y = y.reshape(y.shape[0], -1, D)
    c, s = rope[pos].double()[:, None, :, 0], rope[pos].double()[:, None, :, 1]
    a, b = y[..., : D // 2], y[..., D // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attention64(q, kv, rows, D):
    """q [rows][heads][D], kv [2][slot][KV head][position][D] holding every position."""
    out = torch.empty_like(q)
    by_slot = {}
    for j, (s, p) in enumerate(rows):
        by_slot.setdefault(s, []).append((j, p))
    for s, members in by_slot.items():
        js = torch.tensor([j for j, _ in members], device=DEV)
        ps = torch.tensor([p for _, p in members], device=DEV)
        top = int(ps.max()) + 1
        hidden = torch.arange(top, device=DEV)[None, :] > ps[:, None]
        for g in range(kv.shape[2]):
            k, v = kv[0, s, g, :top].double(), kv[1, s, g, :top].double()
            for h in range(4 * g, 4 * g + 4):
                sc = (q[js, h] @ k.t()) * D ** -0.5
                out[js, h] = torch.softmax(sc.masked_fill(hidden, -math.inf), 1) @ v
    return out


def _attn64(x, w, rows, rope, kv, D):
    """(q, attention output, K and V with the rows' own entries) of one layer."""
    n = x.shape[0]
    pos = torch.tensor([p for _, p in rows], device=DEV)
    slot = torch.tensor([s for s, _ in rows], device=DEV)
    q = _rope64(_mm(x, w["q"]), pos, rope, D)
    kv = kv.double()
    kv[0, slot, :, pos] = _rope64(_mm(x, w["k"]), pos, rope, D)
    kv[1, slot, :, pos] = _mm(x, w["v"]).reshape(n, -1, D)
    return q.reshape(n, -1), _attention64(q, kv, rows, D).reshape(n, -1), kv


def _mlp64(x, w):
    a = _mm(x, w["w1"])
    return a * torch.sigmoid(a) * _mm(x, w["w3"])


def _tiles64(a):
    """[rows][cols] as lane tiles, zeros in the lanes past the last row."""
    n, cols = a.shape
    p = torch.zeros((-(-n // 16) * 16, cols), dtype=a.dtype, device=DEV)
    p[:n] = a
    return p.reshape(-1, 16, cols // 16, 16).permute(0, 2, 1, 3).contiguous()


def _lanes64(case, a):
    if case["path"] == "tc":
        return _tiles64(a)
    stride = 1 if case["rows"] == 1 else -(-case["rows"] // 4) * 4
    p = torch.zeros((a.shape[1], stride), dtype=a.dtype, device=DEV)
    p[:, : a.shape[0]] = a.t()
    return p


def _logits64(case, x, w):
    """Logits in the path's layout, zeros for the padded vocabulary rows and lanes."""
    n, V = case["rows"], case["vocab"]
    y = _mm(x, w)
    if case["path"] == "tc":
        lt, rt = -(-n // 16), -(-V // 16)
        p = torch.zeros((rt * 16, lt * 16), dtype=y.dtype, device=DEV)
        p[:V, :n] = y.t()
        return p.reshape(rt, 16, lt, 16).permute(0, 2, 1, 3).contiguous(), y
    stride = 1 if n == 1 else -(-n // 4) * 4
    p = torch.zeros((-(-V // 4) * 4, stride), dtype=y.dtype, device=DEV)
    p[:V, :n] = y.t()
    return p, y


def exact(case, seed):
    if case["block"] == "attn":
        i = _attn_inputs(case, seed)
        q, attn, kv = _attn64(_norm64(i["h"], i["gain"]), i, i["rows"], i["rope"], i["kv"], case["head_dim"])
        h = i["h"].double() + _mm(attn, i["o"])
        if case["path"] == "exact" and case["rows"] > 1:
            q = torch.cat([q, torch.zeros(-case["rows"] % 4, q.shape[1], dtype=q.dtype, device=DEV)])
        return dict(h=_lanes64(case, h), q=q, attn=_lanes64(case, attn), kv=_arena(kv, i["table"], case["page"]).reshape(-1))
    if case["block"] == "mlp":
        i = _mlp_inputs(case, seed)
        z = _mlp64(_norm64(i["h"], i["gain"]), i)
        return dict(h=_lanes64(case, i["h"].double() + _mm(z, i["w2"])), z=_lanes64(case, z))
    if case["block"] == "head":
        i = _head_inputs(case, seed)
        x = _norm64(i["h"], i["gain"])
        logits, y = _logits64(case, x, i["w"])
        if case["full"]:
            return dict(x=_lanes64(case, x), logits=logits)
        return dict(x=_lanes64(case, x), value=y.max(1).values, index=None)
    return _step64(case, seed)


def _step64(case, seed):
    D, kvh = case["head_dim"], case["heads"] // 4
    rows = _step_rows(case, seed)
    g = _gen(seed, 4)
    embed = _w(g, case["vocab"], case["hidden"])
    final = _gain(g, case["hidden"])
    arena, table = _step_arena(case, seed)
    rope = _rope(case["ctx"], D)
    h = embed[torch.tensor([t for _, _, t in rows], device=DEV)].double()
    where = [(s, p) for s, p, _ in rows]
    for li, L in enumerate(_step_layers(case, seed)):
        # [slot][page][K|V][KV head][token][dim] -> [K|V][slot][KV head][position][dim]
        kv = arena[:, li][table.long().reshape(-1)].reshape(*table.shape, 2, kvh, case["page"], D)
        kv = kv.permute(2, 0, 3, 1, 4, 5).reshape(2, case["rows"], kvh, -1, D)
        _, attn, _ = _attn64(_norm64(h, L["norm_attn"]), L, where, rope, kv, D)
        h = h + _mm(attn, L["o"])
        h = h + _mm(_mlp64(_norm64(h, L["norm_mlp"]), L), L["w2"])
    logits, y = _logits64(case, _norm64(h, final), embed)
    return dict(logits=logits, value=y.max(1).values, index=None)
