"""The calls that a serving program makes on this library, at the sizes it makes them.

A program that serves a decoder with a paged KV cache appends prompts to the
pools, prefills them in chunks, then decodes token by token, over 2-byte, FP8
or KIVI pages, with the norms and activations at the edges of each layer.
Every case is one such call (or the calls of one step) through tl_attn.

A case is a dict of plain values; lengths that differ over a batch are drawn
from the case's own values, so that two states of a case do the same work on
other data.
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "truellm-engine_amd"))

import tl_attn as tla  # noqa: E402

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
PAGE = 32                # tokens of a KIVI page
FP8_MAX = 448.0
EPS = 1e-5
ROPE_BASE = 10000.0


def listed():
    return [
        # One user's next token, through every attention layer of a model: 32
        # layers with pools of their own, append and decode in each.
        dict(name="decode_one_user", kind="decode", batch=1, ctx=4096, heads=32, kv_heads=8, head=128, block=16,
             dtype="f16", kv="same", ragged=False, append=True, layers=32),
        # A full batch at one context length: the repository's headline decode
        # step, append included.
        dict(name="decode_batch", kind="decode", batch=64, ctx=4096, heads=32, kv_heads=8, head=128, block=16,
             dtype="bf16", kv="same", ragged=False, append=True, layers=1),
        # A batch as it stands in service: few sequences, lengths of every
        # size, the 64-head shape (8 query heads for each KV head).
        dict(name="decode_ragged", kind="decode", batch=24, ctx=8192, heads=64, kv_heads=8, head=128, block=32,
             dtype="bf16", kv="same", ragged=True, append=True, layers=1),
        # Long contexts over an FP8 pool.
        dict(name="decode_fp8_long", kind="decode", batch=16, ctx=32768, heads=32, kv_heads=8, head=128, block=16,
             dtype="f16", kv="fp8", ragged=False, append=True, layers=1),
        # The KIVI INT4 step of a full batch whose sequences are at different
        # places in their pages.
        dict(name="kivi_int4_step", kind="kivi_step", batch=64, ctx=4096, heads=32, kv_heads=8, bits=4, residual=128,
             pre_rope=False, style=1, block=16),
        # The default KIVI configuration (INT8, keys held before RoPE, the
        # engine's adjacent pairs) at a smaller batch.
        dict(name="kivi_default_step", kind="kivi_step", batch=16, ctx=2900, heads=32, kv_heads=8, bits=8,
             residual=128, pre_rope=True, style=0, block=16),
        # Prompts that have been prefilled go into KIVI pages.
        dict(name="kivi_build", kind="kivi_build", batch=8, ctx=4096, heads=32, kv_heads=8, bits=4, residual=128,
             block=16),
        # A scheduler's mixed batch: the last 512-token chunk of eight
        # 2048-token prompts, with 32 decode rows beside them.
        dict(name="prefill_mixed", kind="prefill", prompts=8, chunk=512, ctx=2048, decodes=32, heads=64, kv_heads=8,
             block=16, dtype="bf16", kv="same"),
        # One user's prompt, nothing else in the batch: what time to first
        # token is made of.
        dict(name="prefill_one_user", kind="prefill", prompts=1, chunk=500, ctx=1500, decodes=0, heads=32, kv_heads=8,
             block=16, dtype="f16", kv="same"),
        # A prompt's keys and values into the pools, rotated on the way, with
        # its queries: prompts of 700 tokens that begin in the middle of a block.
        dict(name="append_prompts", kind="append", prompts=6, tokens=700, heads=32, kv_heads=8, block=16,
             dtype="bf16", kv="same", style=1),
        # The edges of a layer over one prompt chunk: residual add with norm,
        # and the gated activation.
        dict(name="layer_edges", kind="edges", rows=512, hidden=4096, inter=14336, dtype="bf16", norm="fused_add",
             act=tla.ACT_SILU),
        # A sequence's cache through the vector codec and back: 2048 tokens of
        # 8 KV heads.
        dict(name="kivi_codec", kind="codec", vectors=16384, head=128, outliers=8, group=16),
    ]


def log_int(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "kivi_step", "kivi_build", "prefill", "prefill", "append", "edges",
                       "codec"])
    heads, kv_heads = rng.choice([(32, 8), (64, 8), (32, 8), (32, 32)])
    dtype = rng.choice(["f16", "bf16"])
    block = rng.choice([16, 16, 16, 32, 64])
    kv = rng.choice(["same", "same", "fp8"])
    if kind == "decode":
        batch = log_int(rng, 1, 64)
        # at most the tokens of the largest batch, over all KV heads
        most = min(32768, 64 * 4096 * 8 // (batch * kv_heads))
        ctx = log_int(rng, 100, most)
        head = 128
        if block == 16 and kv == "same" and rng.random() < 0.15:
            head = 64
        return dict(kind=kind, batch=batch, ctx=ctx, heads=heads, kv_heads=kv_heads, head=head, block=block,
                    dtype=dtype, kv=kv, ragged=rng.random() < 0.6, append=rng.random() < 0.6, layers=1)
    if kind == "kivi_step":
        batch = log_int(rng, 1, 64)
        return dict(kind=kind, batch=batch, ctx=log_int(rng, 200, min(8192, 64 * 4096 // batch)), heads=heads,
                    kv_heads=8, bits=rng.choice([4, 8]), residual=rng.choice([128, 128, 64]),
                    pre_rope=rng.random() < 0.4, style=rng.choice([0, 1]), block=block)
    if kind == "kivi_build":
        batch = log_int(rng, 1, 8)
        return dict(kind=kind, batch=batch, ctx=log_int(rng, 200, 8 * 4096 // batch), heads=heads, kv_heads=8,
                    bits=rng.choice([4, 8]), residual=rng.choice([128, 128, 64]), block=block)
    if kind == "prefill":
        prompts = log_int(rng, 1, 8)
        chunk = log_int(rng, 16, 4096 // prompts)
        ctx = chunk if rng.random() < 0.4 else min(chunk + log_int(rng, 16, 6000), 8192 * 2048 // (prompts * chunk))
        return dict(kind=kind, prompts=prompts, chunk=chunk, ctx=max(ctx, chunk), decodes=rng.choice([0, 0, 3, 17]),
                    heads=heads, kv_heads=8, block=block, dtype=dtype, kv=kv)
    if kind == "append":
        prompts = log_int(rng, 1, 8)
        return dict(kind=kind, prompts=prompts, tokens=log_int(rng, 1, 4200 // prompts), heads=heads, kv_heads=8,
                    block=block, dtype=dtype, kv=kv, style=rng.choice([0, 1]))
    if kind == "edges":
        hidden, inter = rng.choice([(4096, 14336), (4096, 11008), (8192, 28672), (2048, 5632)])
        return dict(kind=kind, rows=log_int(rng, 1, 2048), hidden=hidden, inter=inter, dtype=dtype,
                    norm=rng.choice(["fused_add", "rms", "layer"]),
                    act=rng.choice([tla.ACT_SILU, tla.ACT_GELU, tla.ACT_GELU_TANH]))
    head, outliers, group = rng.choice([(128, 8, 16), (64, 4, 16), (128, 0, 32), (96, 13, 8), (128, 4, 16)])
    return dict(kind=kind, vectors=log_int(rng, 8, 16384), head=head, outliers=outliers, group=group)


# ---------------------------------------------------------------------------
# what the cases are made of
# ---------------------------------------------------------------------------

def case_rng(case):
    return random.Random("|".join("%s=%s" % (k, case[k]) for k in sorted(case) if k != "name"))


def lengths(case):
    """Sequence lengths of a batch: all of ctx, or spread from ctx / 16 to ctx."""
    n, ctx = case["batch"], case["ctx"]
    if case["kind"] == "kivi_step":              # each sequence at its own place in a page
        return [ctx + s % 32 for s in range(n)]
    if case["kind"] == "kivi_build" or not case["ragged"]:
        return [ctx] * n
    rng = case_rng(case)
    return [ctx] + [rng.randint(max(1, ctx // 16), ctx) for _ in range(n - 1)]


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def normal(shape, dtype, g):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, 1.0, generator=g)


def tables_for(blocks, total, g):
    """Block tables over a pool of `total` blocks in a free list's order: row s holds blocks[s] ids."""
    order = torch.randperm(total, generator=g, device="cuda").to(torch.int32)
    t = torch.full((len(blocks), max(blocks)), -1, dtype=torch.int32, device="cuda")
    at = 0
    for s, n in enumerate(blocks):
        t[s, :n] = order[at:at + n]
        at += n
    return t


def pool_blocks(blocks):
    return math.ceil(1.25 * sum(blocks)) + 1


def block_counts(lens, bs):
    return [(n + bs - 1) // bs for n in lens]


def fp8_pool(shape, scale, g):
    """E4M3 codes of N(0, 1) values under a per-tensor scale."""
    pool = torch.empty(shape, dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 26) // math.prod(shape[1:]))
    for i in range(0, shape[0], step):
        x = normal(pool[i:i + step].shape, torch.float32, g)
        pool[i:i + step] = (x / scale).clamp_(-FP8_MAX, FP8_MAX).to(torch.float8_e4m3fn).view(torch.uint8)
    return pool


def make_pool(shape, case, g):
    if case["kv"] == "fp8":
        return fp8_pool(shape, case_scale(case), g)
    return normal(shape, DTYPES[case["dtype"]], g)


def case_scale(case):
    """Scale of an FP8 pool of N(0, 1) values (absmax / 448 of a few million of them), 1 otherwise."""
    return 5.5 / FP8_MAX if case.get("kv") == "fp8" else 1.0


def slots_at(tables, positions, bs):
    """Pool slot of position positions[s] of sequence s."""
    pos = torch.tensor(positions, device="cuda")
    blk = tables[torch.arange(len(positions), device="cuda"), pos // bs].long()
    return (blk * bs + pos % bs).to(torch.int32)


def rope_tables(n, head):
    inv = ROPE_BASE ** (-torch.arange(0, head, 2, device="cuda", dtype=torch.float64) / head)
    a = torch.outer(torch.arange(n, device="cuda", dtype=torch.float64), inv)
    return a.cos().float().contiguous(), a.sin().float().contiguous()


def int32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------

def prepare(case, seed):
    return {"decode": prepare_decode, "kivi_step": prepare_kivi, "kivi_build": prepare_kivi,
            "prefill": prepare_prefill, "append": prepare_append, "edges": prepare_edges,
            "codec": prepare_codec}[case["kind"]](case, seed)


def prepare_decode(case, seed):
    g = generator(seed)
    lens, bs, H, n_kv, D = lengths(case), case["block"], case["heads"], case["kv_heads"], case["head"]
    S, layers, dtype = case["batch"], case["layers"], DTYPES[case["dtype"]]
    blocks = block_counts(lens, bs)
    total = pool_blocks(blocks)
    tables = tables_for(blocks, total, g)
    kpools = make_pool((layers * total, n_kv, D, bs), case, g).view(layers, total, n_kv, D, bs)
    vpools = make_pool((layers * total, n_kv, D, bs), case, g).view(layers, total, n_kv, D, bs)
    q = normal((layers, S, H, D), dtype, g)
    key, value = normal((layers, S, n_kv, D), dtype, g), normal((layers, S, n_kv, D), dtype, g)
    out = torch.empty_like(q)
    scale = case_scale(case)
    desc = tla.make_decode_desc(q[0], kpools[0], tables, n_kv, 1.0 / math.sqrt(D),
                                gqa_map=tla.GQA_GROUPED, k_scale=scale, v_scale=scale)
    ws = torch.empty(max(16, tla.workspace_bytes(desc, max(lens))), dtype=torch.uint8, device="cuda")
    return dict(case=case, desc=desc, q=q, key=key, value=value, out=out, kpools=kpools, vpools=vpools,
                tables=tables, lens=int32(lens), max_ctx=max(lens), ws=ws,
                slots=slots_at(tables, [n - 1 for n in lens], bs),
                layers=[(out[i], q[i], key[i], value[i], kpools[i], vpools[i]) for i in range(layers)])


def prepare_kivi(case, seed):
    g = generator(seed)
    lens, bs, H, n_kv, D = lengths(case), case["block"], case["heads"], case["kv_heads"], 128
    S = case["batch"]
    blocks = block_counts(lens, bs)
    total = pool_blocks(blocks)
    tables = tables_for(blocks, total, g)
    k, v = normal((total, n_kv, D, bs), torch.float16, g), normal((total, n_kv, D, bs), torch.float16, g)
    # a few key channels of each head are larger than the rest, which is what
    # per-channel quantisation is for
    loud = torch.ones((n_kv, D), dtype=torch.float16, device="cuda")
    for h in range(n_kv):
        loud[h, torch.randperm(D, generator=g, device="cuda")[:4]] = 8.0
    k *= loud[None, :, :, None]
    pages_of = [max(1, (n + PAGE - 1) // PAGE) for n in lens]
    n_pages = pool_blocks(pages_of)
    page_tables = tables_for(pages_of, n_pages, g)
    pages = torch.zeros((n_pages, n_kv, tla.kivi_page_bytes(case["bits"])), dtype=torch.uint8, device="cuda")
    q = normal((S, H, D), torch.float16, g)
    key, value = normal((S, n_kv, D), torch.float16, g) * loud, normal((S, n_kv, D), torch.float16, g)
    desc = tla.make_kivi_desc(q, k, tables, page_tables, n_pages, n_kv, 1.0 / math.sqrt(D),
                              residual_length=case["residual"], bits=case["bits"],
                              pre_rope_keys=case.get("pre_rope", False))
    state = dict(case=case, desc=desc, q=q, out=torch.empty_like(q), key=key, value=value, k=k, v=v, tables=tables,
                 pages=pages, page_tables=page_tables, lens=int32(lens), max_ctx=max(lens))
    if case["kind"] == "kivi_step":
        before = int32([n - 1 for n in lens])
        tla.kivi_build_pages(desc, k, v, tables, before, page_tables, pages, max(lens))
        state["slots"] = slots_at(tables, [n - 1 for n in lens], bs)
        ws = max(16, tla.kivi_workspace_bytes(desc, max(lens)))
        state["ws"] = torch.empty(ws, dtype=torch.uint8, device="cuda")
        state["cos"], state["sin"] = rope_tables(max(lens), D)
    return state


def prefill_lengths(case):
    """(query tokens, context) of each prompt, then of each decode row."""
    rng = case_rng(case)
    rows = []
    for i in range(case["prompts"]):
        cut = 0 if i == 0 or case["prompts"] == 8 else rng.randint(0, case["chunk"] // 2)
        rows.append((max(2, case["chunk"] - cut), max(2, case["ctx"] - cut)))
    return rows + [(1, case["ctx"])] * case["decodes"]


def prepare_prefill(case, seed):
    g = generator(seed)
    rows, bs, H, n_kv, D = prefill_lengths(case), case["block"], case["heads"], case["kv_heads"], 128
    dtype = DTYPES[case["dtype"]]
    lens = [c for _, c in rows]
    blocks = block_counts(lens, bs)
    total = pool_blocks(blocks)
    tables = tables_for(blocks, total, g)
    k, v = make_pool((total, n_kv, D, bs), case, g), make_pool((total, n_kv, D, bs), case, g)
    starts = [0]
    for n, _ in rows:
        starts.append(starts[-1] + n)
    q = normal((starts[-1], H, D), dtype, g)
    scale = case_scale(case)
    desc = tla.make_prefill_desc(q, k, tables, len(rows), n_kv, 1.0 / math.sqrt(D), gqa_map=tla.GQA_GROUPED,
                                 num_prefill_seqs=case["prompts"],
                                 kv_dtype=tla.FP8_E4M3 if case["kv"] == "fp8" else None, k_scale=scale,
                                 v_scale=scale)
    return dict(case=case, desc=desc, q=q, out=torch.empty_like(q), k=k, v=v, tables=tables, lens=int32(lens),
                cu=int32(starts), max_q=max(n for n, _ in rows), rows=rows)


def append_spans(case):
    """(first position, tokens) of each prompt: a chunk that begins anywhere in a block."""
    rng = case_rng(case)
    return [(rng.randint(0, 3 * case["block"]), max(1, case["tokens"] - (rng.randint(0, 7) if i else 0)))
            for i in range(case["prompts"])]


def prepare_append(case, seed):
    g = generator(seed)
    spans, bs, H, n_kv, D = append_spans(case), case["block"], case["heads"], case["kv_heads"], 128
    dtype = DTYPES[case["dtype"]]
    blocks = block_counts([a + n for a, n in spans], bs)
    total = pool_blocks(blocks)
    tables = tables_for(blocks, total, g)
    T = sum(n for _, n in spans)
    positions = torch.cat([torch.arange(a, a + n, device="cuda") for a, n in spans])
    seq = torch.cat([torch.full((n,), i, device="cuda") for i, (_, n) in enumerate(spans)])
    slots = (tables[seq, positions // bs].long() * bs + positions % bs).to(torch.int32)
    k, v = make_pool((total, n_kv, D, bs), case, g), make_pool((total, n_kv, D, bs), case, g)
    q = normal((T, H, D), dtype, g)
    cos, sin = rope_tables(max(a + n for a, n in spans), D)
    return dict(case=case, q=q, q_out=torch.empty_like(q), key=normal((T, n_kv, D), dtype, g),
                value=normal((T, n_kv, D), dtype, g), k=k, v=v, slots=slots, positions=positions.to(torch.int32),
                cos=cos, sin=sin)


def prepare_edges(case, seed):
    g = generator(seed)
    dtype, rows, hidden, inter = DTYPES[case["dtype"]], case["rows"], case["hidden"], case["inter"]
    return dict(case=case, x=normal((rows, hidden), dtype, g), residual=normal((rows, hidden), dtype, g),
                weight=(1.0 + 0.1 * normal((hidden,), torch.float32, g)).to(dtype),
                bias=(0.1 * normal((hidden,), torch.float32, g)).to(dtype),
                gate=normal((rows, inter), dtype, g), up=normal((rows, inter), dtype, g),
                out=torch.empty((rows, hidden), dtype=dtype, device="cuda"),
                act=torch.empty((rows, inter), dtype=dtype, device="cuda"))


def prepare_codec(case, seed):
    g = generator(seed)
    n, D, O, G = case["vectors"], case["head"], case["outliers"], case["group"]
    x = normal((n, D), torch.float16, g)
    stride = tla.kivi_compressed_bytes(D, O, G)
    return dict(case=case, x=x, rec=torch.zeros((n, stride), dtype=torch.uint8, device="cuda"),
                back=torch.empty_like(x))


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        if not case["append"]:
            for out, q, _, _, k, v in s["layers"]:
                tla.paged_attention_decode(s["desc"], out, q, k, v, s["tables"], s["lens"], s["max_ctx"], s["ws"])
            return [s["out"]]
        for out, q, key, value, k, v in s["layers"]:
            tla.paged_attention_decode_step(s["desc"], out, q, key, value, s["slots"], k, v, s["tables"], s["lens"],
                                            s["max_ctx"], s["ws"])
        return [s["out"], s["kpools"], s["vpools"]]
    if kind == "kivi_step":
        if case["pre_rope"]:
            tla.kivi_decode_step_pre_rope(s["desc"], s["out"], s["q"], s["key"], s["value"], s["slots"], s["pages"],
                                          s["page_tables"], s["k"], s["v"], s["tables"], s["lens"], s["max_ctx"],
                                          s["cos"], s["sin"], case["style"], s["ws"])
        else:
            tla.kivi_decode_step(s["desc"], s["out"], s["q"], s["key"], s["value"], s["slots"], s["pages"],
                                 s["page_tables"], s["k"], s["v"], s["tables"], s["lens"], s["max_ctx"], s["ws"])
        return [s["out"], s["k"], s["v"], s["pages"]]
    if kind == "kivi_build":
        tla.kivi_build_pages(s["desc"], s["k"], s["v"], s["tables"], s["lens"], s["page_tables"], s["pages"],
                             s["max_ctx"])
        return [s["pages"]]
    if kind == "prefill":
        tla.chunked_prefill(s["desc"], s["out"], s["q"], s["cu"], s["k"], s["v"], s["tables"], s["lens"], s["max_q"])
        return [s["out"]]
    if kind == "append":
        if case["kv"] == "fp8":
            scale = case_scale(case)
            tla.reshape_and_cache_fp8(s["key"], s["value"], s["k"], s["v"], s["slots"], scale, scale)
            return [s["k"], s["v"]]
        tla.rope_reshape_and_cache(s["q"], s["key"], s["value"], s["k"], s["v"], s["slots"], s["positions"],
                                   s["cos"], s["sin"], case["style"], q_out=s["q_out"])
        return [s["k"], s["v"], s["q_out"]]
    if kind == "edges":
        if case["norm"] == "fused_add":
            tla.fused_add_rms_norm(s["out"], s["residual"], s["x"], s["weight"], EPS)
        elif case["norm"] == "rms":
            tla.rms_norm(s["out"], s["x"], s["weight"], EPS)
        else:
            tla.layer_norm(s["out"], s["x"], s["weight"], s["bias"], EPS)
        tla.act_and_mul(s["act"], s["gate"], s["up"], case["act"])
        return [s["out"], s["residual"], s["act"]]
    n, D, O, G = case["vectors"], case["head"], case["outliers"], case["group"]
    tla.kivi_compress(s["x"], s["rec"], n, D, O, G)
    tla.kivi_decompress(s["rec"], s["back"], n, D, O, G)
    return [s["rec"], s["back"]]


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------

def quantised(n, residual):
    return 0 if n <= residual else (n - residual) // PAGE * PAGE


def work(case):
    kind = case["kind"]
    if kind == "decode":
        S, H, n_kv, D, lens = case["batch"], case["heads"], case["kv_heads"], case["head"], lengths(case)
        e = 1 if case["kv"] == "fp8" else 2
        b = sum(lens) * n_kv * D * 2 * e + 2 * S * H * D * 2 + 4 * (sum(block_counts(lens, case["block"])) + S)
        if case["append"]:
            b += S * n_kv * D * 2 * (2 + e)
        return {"bytes": b * case["layers"], "flops": 4 * sum(lens) * H * D * case["layers"]}
    if kind in ("kivi_step", "kivi_build"):
        S, H, n_kv, D, R, lens = case["batch"], case["heads"], case["kv_heads"], 128, case["residual"], lengths(case)
        page = n_kv * (5120 if case["bits"] == 4 else 9216)
        if kind == "kivi_build":
            n = sum(quantised(x, R) for x in lens)
            return {"bytes": n * n_kv * D * 4 + n // PAGE * page, "flops": 8 * n * n_kv * D}
        b = 2 * S * H * D * 2 + S * n_kv * D * 8
        for x in lens:
            lq = quantised(x, R)
            b += lq // PAGE * page + (x - lq) * n_kv * D * 4 + 4 * (lq // PAGE + (x - lq) // case["block"] + 2)
            if lq != quantised(x - 1, R):
                b += PAGE * n_kv * D * 4 + page
        return {"bytes": b, "flops": 4 * sum(lens) * H * D}
    if kind == "prefill":
        H, n_kv, D, rows = case["heads"], case["kv_heads"], 128, prefill_lengths(case)
        e = 1 if case["kv"] == "fp8" else 2
        pairs = sum(n * (c - n) + n * (n + 1) // 2 for n, c in rows)
        b = sum(c for _, c in rows) * n_kv * D * 2 * e + 2 * sum(n for n, _ in rows) * H * D * 2
        return {"bytes": b, "flops": 4 * pairs * H * D}
    if kind == "append":
        T, H, n_kv, D = sum(n for _, n in append_spans(case)), case["heads"], case["kv_heads"], 128
        if case["kv"] == "fp8":
            return {"bytes": T * n_kv * D * 2 * 3 + 4 * T, "flops": 2 * T * n_kv * D}
        return {"bytes": T * (2 * H * D * 2 + n_kv * D * 8 + D * 4 + 8), "flops": 3 * T * (H + n_kv) * D}
    if kind == "edges":
        rows, hidden, inter = case["rows"], case["hidden"], case["inter"]
        moved = 4 if case["norm"] == "fused_add" else 2
        return {"bytes": 2 * rows * (moved * hidden + 3 * inter), "flops": rows * (5 * hidden + 6 * inter)}
    n, D = case["vectors"], case["head"]
    stride = tla.kivi_compressed_bytes(D, case["outliers"], case["group"])
    return {"bytes": n * (2 * D * 2 + 2 * stride), "flops": 8 * n * D}


def tolerance(case):
    # About four times the distance from the 64-bit results.  The 2-byte
    # outputs are rounded once from fp32 sums: 2e-4 to 3e-4 of the result in
    # f16 and 1.7e-3 to 2.4e-3 in bf16, weights in 2 bytes for the matrix
    # products included.  The KIVI step is 2e-3 (8 bits) to 3e-3 (4 bits) off,
    # as the quantisation's steps are folded into 2-byte operands.  Rotated
    # keys and queries are one fixed fp32 expression; pages, records and
    # copied values are bytes.
    if case["kind"] in ("kivi_build", "append", "codec"):
        return "exact"
    if case["kind"] == "kivi_step":
        return {"rel": 1e-2}
    return {"rel": 8e-3 if case["dtype"] == "bf16" else 1.2e-3}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def exact(case, seed):
    with torch.no_grad():
        return {"decode": exact_decode, "kivi_step": exact_kivi, "kivi_build": lambda c, s: None,
                "prefill": exact_prefill, "append": exact_append, "edges": exact_edges,
                "codec": lambda c, s: None}[case["kind"]](case, seed)


def widen(pool, case):
    if case.get("kv") == "fp8":
        return pool.view(torch.float8_e4m3fn).float().double() * case_scale(case)
    return pool.double()


def gathered(pool, row, n):
    """[kv_heads, n, head] of one sequence from a pool [blocks, kv_heads, head, block]."""
    bs = pool.shape[3]
    b = pool[row[:(n + bs - 1) // bs].long()]
    return b.permute(1, 0, 3, 2).reshape(b.shape[1], -1, b.shape[2])[:, :n].contiguous()


def attention(q, k, v, first):
    """q [n, H, D] at positions first, first + 1, ... over k, v [kv_heads, L, D], causal, in 64 bits."""
    n, H, D = q.shape
    n_kv, L = k.shape[0], k.shape[1]
    group = H // n_kv
    qq = q.double().view(n, n_kv, group, D).permute(1, 0, 2, 3).reshape(n_kv, n * group, D)
    out = torch.empty_like(qq)
    pos = torch.arange(L, device=q.device)
    at = (first + torch.arange(n, device=q.device)).repeat_interleave(group)
    for h in range(n_kv):
        sc = (qq[h] @ k[h].t().contiguous()) / math.sqrt(D)
        sc.masked_fill_(pos[None, :] > at[:, None], -math.inf)
        out[h] = torch.softmax(sc, -1) @ v[h]
    return out.view(n_kv, n, group, D).permute(1, 0, 2, 3).reshape(n, H, D)


def put(pool, slots, rows):
    """rows [T, kv_heads, head] into a copy of pool [blocks, kv_heads, head, block] at slots, in 64 bits."""
    p, bs = pool.double(), pool.shape[3]
    s = slots.long()
    p[s // bs, :, :, s % bs] = rows.double()
    return p


def exact_decode(case, seed):
    s = prepare(case, seed)
    lens, bs = lengths(case), case["block"]
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    for i in range(case["layers"]):
        kp, vp = s["kpools"][i], s["vpools"][i]
        for j, n in enumerate(lens):
            k = widen(gathered(kp, s["tables"][j], n), case)
            v = widen(gathered(vp, s["tables"][j], n), case)
            if case["append"]:
                new = s["key"][i, j].double(), s["value"][i, j].double()
                if case["kv"] == "fp8":
                    new = [fp8_rounded(x, case_scale(case)) for x in new]
                k[:, n - 1], v[:, n - 1] = new
            out[i, j] = attention(s["q"][i, j:j + 1], k, v, n - 1)[0]
    # the pools hold copied values, which have no 64-bit value of their own
    return [out, None, None] if case["append"] else [out]


def fp8_rounded(x, scale):
    return (x / scale).clamp(-FP8_MAX, FP8_MAX).float().to(torch.float8_e4m3fn).float().double() * scale


def requantised(x, levels, dim):
    """What a group along `dim` reads back as: `levels` steps between its least and its greatest value,
    step and least value held in f16."""
    x = x.float()
    lo, hi = x.amin(dim, keepdim=True), x.amax(dim, keepdim=True)
    scale = torch.where(hi - lo > 1e-6, levels / (hi - lo), torch.zeros_like(lo))
    step = torch.where(scale > 0, 1.0 / scale, torch.zeros_like(lo)).half().double()
    code = torch.round((x - lo) * scale).clamp_(0, levels)
    return code.double() * step + lo.half().double()


def rotated(x, cos, sin, style):
    """Rows x [..., n, D] at positions 0 .. n - 1."""
    c, s = cos.double(), sin.double()
    if style == 0:
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack((a * c - b * s, a * s + b * c), -1).flatten(-2)
    a, b = x.chunk(2, -1)
    return torch.cat((a * c - b * s, a * s + b * c), -1)


def exact_kivi(case, seed):
    s = prepare(case, seed)
    levels = 15 if case["bits"] == 4 else 255
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    for j, n in enumerate(lengths(case)):
        k, v = gathered(s["k"], s["tables"][j], n).double(), gathered(s["v"], s["tables"][j], n).double()
        k[:, n - 1], v[:, n - 1] = s["key"][j].double(), s["value"][j].double()
        lq = quantised(n, case["residual"])
        if lq:
            h, D = k.shape[0], k.shape[2]
            k[:, :lq] = requantised(k[:, :lq].reshape(h, lq // PAGE, PAGE, D), levels, 2).reshape(h, lq, D)
            v[:, :lq] = requantised(v[:, :lq].reshape(h, lq, D // 32, 32), levels, 3).reshape(h, lq, D)
        if case["pre_rope"]:
            k = rotated(k, s["cos"][:n], s["sin"][:n], case["style"])
        out[j] = attention(s["q"][j:j + 1], k, v, n - 1)[0]
    return [out, None, None, None]


def exact_prefill(case, seed):
    s = prepare(case, seed)
    out = torch.empty(s["q"].shape, dtype=torch.float64, device="cuda")
    at = 0
    for j, (n, c) in enumerate(s["rows"]):
        k = widen(gathered(s["k"], s["tables"][j], c), case)
        v = widen(gathered(s["v"], s["tables"][j], c), case)
        out[at:at + n] = attention(s["q"][at:at + n], k, v, c - n)
        at += n
    return [out]


def exact_append(case, seed):
    s = prepare(case, seed)
    if case["kv"] == "fp8":
        return None
    c, sn = s["cos"][s["positions"].long()], s["sin"][s["positions"].long()]

    def rot(x):
        return rotated(x.double().transpose(0, 1), c, sn, case["style"]).transpose(0, 1)
    return [put(s["k"], s["slots"], rot(s["key"])), put(s["v"], s["slots"], s["value"]), rot(s["q"]).contiguous()]


def exact_edges(case, seed):
    s = prepare(case, seed)
    x, w, res = s["x"].double(), s["weight"].double(), s["residual"].double()
    if case["norm"] == "layer":
        out = torch.nn.functional.layer_norm(x, (case["hidden"],), w, s["bias"].double(), EPS)
    else:
        if case["norm"] == "fused_add":
            x = res = x + res
        out = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w
    gate, up = s["gate"].double(), s["up"].double()
    if case["act"] == tla.ACT_SILU:
        act = torch.nn.functional.silu(gate)
    else:
        act = torch.nn.functional.gelu(gate, approximate="tanh" if case["act"] == tla.ACT_GELU_TANH else "none")
    return [out, res, act * up]
