"""Measured cases of the attention path: what an engine step runs through ``femtovllm.ops``.

Each case is a dict of plain values.  ``kind`` names the entry point:

* ``decode``    ``ops.paged_attention_gemv``: one query token per sequence;
* ``prefill``   ``ops.paged_attention_gemm``: chunks of new tokens after cached
  prefixes, with or without decode rows in the same call;
* ``prologue``  ``ops.qk_norm_rope_cache_write`` of a chunked batch;
* ``layer``     the prologue and then the attention of the same step, as one
  decoder layer runs them;
* ``dense``     ``_C.FlashAttentionWarpCuda``: contiguous, non-causal.

A paged batch is ``seqs`` prefill chunks (``new_min..new_max`` tokens after
``prefix_min..prefix_max`` cached ones) followed by ``rows`` decode rows
(contexts ``ctx_min..ctx_max``); lengths are drawn from ``lens`` so that a
case's work does not depend on the seed.  ``chunks`` (text, "prefix+new ...")
gives the prefill chunks one by one instead.  The first ``shared`` blocks of
every second sequence are the same physical blocks (a prefix-cache hit).
Blocks are placed by a random permutation of a pool 1.2 times the used blocks.
"""

import math
import os
import random
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "nano-vllm-practice_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

PAGE = 16
DIM = 128
EPS = 1e-6
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}
MAX_POSITIONS = 40960  # rows of the rotary tables


def _case(kind, dtype, heads, kv_heads, **kw):
    c = {"kind": kind, "dtype": dtype, "heads": heads, "kv_heads": kv_heads}
    c.update(kw)
    return c


def listed():
    return [
        # One user's chat on a small model: the step is all launches and latency.
        _case("decode", "bf16", 16, 8, name="decode_one_user", rows=1, ctx_min=300, ctx_max=300, lens=1),
        # The float32 check that the reference runs without a GPU's 16-bit types: 4 short sequences.
        _case("decode", "f32", 16, 8, name="decode_f32_4", rows=4, ctx_min=17, ctx_max=511, lens=2),
        # The serving batch of the benchmark: 64 sequences of very different lengths.
        _case("decode", "bf16", 16, 8, name="decode_64", rows=64, ctx_min=256, ctx_max=4096, lens=1002),
        # A few long conversations at the context limit, in float16, on the 32/8 head shape.
        _case("decode", "f16", 32, 8, name="decode_f16_long", rows=6, ctx_min=6001, ctx_max=8192, lens=3),
        # One decoder layer of a decode step with short contexts: prologue, then attention.
        _case("layer", "bf16", 16, 8, name="layer_decode_short", rows=64, ctx_min=64, ctx_max=512, lens=1006),
        # A first prompt of one user, nothing cached.
        _case("prefill", "bf16", 16, 8, name="prefill_prompt", chunks="0+333", lens=0),
        # Chunked prefill of the benchmark: 8 chunks of 512 after prefixes of up to 2048.
        _case("prefill", "bf16", 16, 8, name="prefill_8x512", seqs=8, new_min=512, new_max=512,
              prefix_min=0, prefix_max=2048, lens=1003),
        # Chunked prefill of uneven sequences: long contexts among short ones.
        _case("prefill", "bf16", 16, 8, name="prefill_uneven", chunks="3000+512 200+512 4000+256 100+1024", lens=0),
        # The last chunk of a 32k prompt on the 32/8 head shape: the largest call.
        _case("prefill", "bf16", 32, 8, name="prefill_long", chunks="30720+2048", lens=0),
        # Unified batch: one prefill chunk beside 127 decode rows, half of them sharing a prefix.
        _case("prefill", "bf16", 32, 8, name="mixed_128", chunks="4096+1024", rows=127, ctx_min=512, ctx_max=8192,
              shared=64, lens=1005),
        # Dense attention of a 2048-token block over 8192 keys.
        _case("dense", "bf16", 32, 8, name="dense_2048x8192", batch=1, q_len=2048, kv_len=8192),
        # The prologue of the chunked prefill: q/k norm, rotary embedding and the cache write of 4096 tokens.
        _case("prologue", "bf16", 16, 8, name="prologue_8x512", seqs=8, new_min=512, new_max=512,
              prefix_min=0, prefix_max=2048, lens=1003),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


MAX_FLOPS, MAX_BYTES = 1.0e12, 2.0e9  # no drawn case costs more than the largest listed ones


def draw(rng):
    while True:
        kind = rng.choice(["decode", "decode", "prefill", "prefill", "mixed", "layer", "layer", "prologue", "dense"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16"])
        heads, kv_heads = rng.choice([(16, 8), (16, 8), (32, 8), (32, 8), (4, 1), (2, 1), (64, 8), (16, 16)])
        lens = rng.randrange(1 << 30)
        if kind == "dense":
            c = _case("dense", dtype, heads, kv_heads, batch=rng.choice([1, 1, 2, 4]), q_len=_log(rng, 1, 2048),
                      kv_len=_log(rng, 16, 16384))
        else:
            rows = dict(rows=_log(rng, 1, 256), ctx_max=_log(rng, 16, 8192))
            rows["ctx_min"] = max(1, int(rows["ctx_max"] * rng.uniform(0.03, 1.0)))
            pre = dict(seqs=_log(rng, 1, 16), new_max=_log(rng, 2, 2048), prefix_max=rng.choice([0, _log(rng, 16, 30720)]))
            pre["new_min"] = max(2, int(pre["new_max"] * rng.uniform(0.1, 1.0)))
            pre["prefix_min"] = int(pre["prefix_max"] * rng.uniform(0.0, 1.0))
            shared = rng.choice([0, 0, 16])
            if kind == "decode":
                if rng.random() < 0.15:
                    dtype = "f32"
                c = _case("decode", dtype, heads, kv_heads, shared=shared, lens=lens, **rows)
            elif kind == "mixed":
                c = _case("prefill", dtype, heads, kv_heads, shared=shared, lens=lens, **pre, **rows)
            elif kind == "prefill":
                c = _case("prefill", dtype, heads, kv_heads, lens=lens, **pre)
            elif kind == "prologue":
                c = _case("prologue", dtype, heads, kv_heads, lens=lens, **pre)
            else:
                c = _case("layer", dtype, heads, kv_heads, lens=lens, **(rows if rng.random() < 0.5 else pre))
        w = work(c)
        if w["flops"] <= MAX_FLOPS and _pool_bytes(c) <= MAX_BYTES:
            return c


# ---- the batch ------------------------------------------------------------


def _chunks(case):
    """(cached, new) tokens of every sequence: the prefill chunks, then the decode rows."""
    r = random.Random(case["lens"])
    out = []
    if case.get("chunks"):
        out += [tuple(int(x) for x in part.split("+")) for part in case["chunks"].split()]
    for _ in range(case.get("seqs", 0)):
        out.append((r.randint(case["prefix_min"], case["prefix_max"]), r.randint(case["new_min"], case["new_max"])))
    for _ in range(case.get("rows", 0)):
        out.append((r.randint(case["ctx_min"], case["ctx_max"]) - 1, 1))
    return out


def _pages(chunks):
    return [-(-(p + n) // PAGE) for p, n in chunks]


def _shared_pages(case, chunks):
    """Leading pages that every second sequence takes from the shared blocks: cached full pages only,
    so that no step writes a block that another sequence reads."""
    s = case.get("shared", 0)
    return [min(s, p // PAGE) if i % 2 == 0 else 0 for i, (p, _) in enumerate(chunks)]


def _unique_pages(case, chunks):
    sh = _shared_pages(case, chunks)
    return sum(_pages(chunks)) - sum(sh) + max(sh, default=0)


def _pool_bytes(case):
    if case["kind"] == "dense":
        return 0
    return 1.2 * _unique_pages(case, _chunks(case)) * PAGE * case["kv_heads"] * DIM * BYTES[case["dtype"]] * 2


def _tables(case, chunks, seed):
    pages, sh = _pages(chunks), _shared_pages(case, chunks)
    unique = _unique_pages(case, chunks)
    num_blocks = max(1, math.ceil(1.2 * unique))
    perm = torch.randperm(num_blocks, generator=torch.Generator().manual_seed(seed)).tolist()
    shared, cursor, tables = perm[: max(sh, default=0)], max(sh, default=0), []
    for n, s in zip(pages, sh):
        tables.append(shared[:s] + perm[cursor : cursor + n - s])
        cursor += n - s
    return tables, num_blocks


def _randn(shape, gen, dtype):
    return torch.randn(shape, generator=gen, dtype=dtype, device=gen.device)


def prepare(case, seed):
    from femtovllm.metadata import build_varlen_metadata

    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    H, KVH = case["heads"], case["kv_heads"]
    st = {"case": case}
    if case["kind"] == "dense":
        st["q"] = _randn((case["batch"], H, case["q_len"], DIM), gen, dt)
        st["k"] = _randn((case["batch"], KVH, case["kv_len"], DIM), gen, dt)
        st["v"] = _randn((case["batch"], KVH, case["kv_len"], DIM), gen, dt)
        return st
    chunks = _chunks(case)
    tables, num_blocks = _tables(case, chunks, seed)
    tokens = sum(n for _, n in chunks)
    st["chunks"], st["tables"] = chunks, tables
    st["meta"] = build_varlen_metadata(chunks, tables, device=dev)
    st["k_pool"] = _randn((num_blocks, KVH, PAGE, DIM), gen, dt)
    st["v_pool"] = _randn((num_blocks, KVH, PAGE, DIM), gen, dt)
    if case["kind"] in ("decode", "prefill"):
        # The engine passes the projection's (tokens, heads, dim) transposed.
        st["q"] = _randn((tokens, H, DIM), gen, dt).transpose(0, 1)
        return st
    from femtovllm.rope import rope_tables

    # The raw projections and the layer's norm weights.
    st["q"] = _randn((tokens, H, DIM), gen, dt)
    st["k"] = _randn((tokens, KVH, DIM), gen, dt)
    st["v"] = _randn((tokens, KVH, DIM), gen, dt)
    st["wq"] = (1.0 + 0.1 * _randn((DIM,), gen, torch.float32)).to(dt)
    st["wk"] = (1.0 + 0.1 * _randn((DIM,), gen, torch.float32)).to(dt)
    st["cos"], st["sin"] = rope_tables(MAX_POSITIONS, DIM, device=dev)
    return st


def _attention(st, q):
    from femtovllm import ops

    m = st["meta"]
    if m.max_q_len == 1:
        return ops.paged_attention_gemv(q, st["k_pool"], st["v_pool"], m.block_tables, m.kv_lens, m.max_kv_len)
    return ops.paged_attention_gemm(q, st["k_pool"], st["v_pool"], m.cu_seqlens, m.max_q_len, m.Q_TILE_SIZE,
                                    m.cu_q_tiles, m.q_tile_to_seq_idx, m.block_tables, m.kv_lens, m.positions)


def run(st):
    from femtovllm import _C, ops

    kind = st["case"]["kind"]
    if kind == "dense":
        return _C.FlashAttentionWarpCuda(st["q"], st["k"], st["v"])
    if kind in ("decode", "prefill"):
        return _attention(st, st["q"])
    m = st["meta"]
    decode = m.max_q_len == 1
    q = ops.qk_norm_rope_cache_write(st["q"], st["k"], st["v"], st["wq"], st["wk"], EPS, st["cos"], st["sin"],
                                     m.positions, st["k_pool"], st["v_pool"], m.block_tables,
                                     cu_seqlens=None if decode else m.cu_seqlens, max_q_len=m.max_q_len)
    if kind == "prologue":
        return {"q": q, "k_pool": st["k_pool"], "v_pool": st["v_pool"]}
    out = _attention(st, q.transpose(0, 1))
    return {"out": out, "k_pool": st["k_pool"], "v_pool": st["v_pool"]}


# ---- work, tolerance, 64-bit results ----------------------------------------


def work(case):
    """K and V of every visible key once per KV head (shared blocks once), q in and out once, the
    tables and lengths; 4 * dim flops per visible (query, key) pair and query head.  The prologue reads
    and writes every q, k and v row once and reads the rotary rows."""
    s, H, KVH = BYTES[case["dtype"]], case["heads"], case["kv_heads"]
    if case["kind"] == "dense":
        b, tq, tk = case["batch"], case["q_len"], case["kv_len"]
        return {"bytes": s * DIM * b * (2 * H * tq + 2 * KVH * tk), "flops": 4 * DIM * H * b * tq * tk}
    chunks = _chunks(case)
    sh = _shared_pages(case, chunks)
    tokens = sum(n for _, n in chunks)
    keys = sum(p + n for p, n in chunks) - PAGE * (sum(sh) - max(sh, default=0))
    attn_bytes = s * DIM * (2 * KVH * keys + 2 * H * tokens) + 4 * sum(_pages(chunks)) + 8 * len(chunks)
    attn_flops = 4 * DIM * H * sum(n * p + n * (n + 1) // 2 for p, n in chunks)
    pro_bytes = 2 * s * DIM * tokens * (H + 2 * KVH) + 8 * DIM * tokens
    if case["kind"] == "prologue":
        return {"bytes": pro_bytes, "flops": 0}
    if case["kind"] == "layer":
        return {"bytes": attn_bytes + pro_bytes, "flops": attn_flops}
    return {"bytes": attn_bytes, "flops": attn_flops}


def tolerance(case):
    # Four times the distance to the 64-bit results over the listed and 30 drawn cases: bf16 2.9e-3 (largest
    # difference 0.020 of the result's magnitude; 0.062 where the prologue's rounding of q and k comes before the
    # attention), f16 3.9e-4 (1.2e-3; 4e-3), f32 3.0e-7 (1.8e-6).
    layer = case["kind"] == "layer"
    return {"f32": {"rel": 1.2e-6, "max": 8e-6}, "f16": {"rel": 1.5e-3, "max": 1.6e-2 if layer else 5e-3},
            "bf16": {"rel": 1.2e-2, "max": 0.25 if layer else 0.08}}[case["dtype"]]


def _softmax_av(q, k, v, limit):
    """softmax(q k^T / sqrt(dim)) v in 64 bits; row i sees keys below limit[i]."""
    out = torch.empty_like(q)
    for a in range(0, q.shape[0], 4096):
        s = torch.mm(q[a : a + 4096], k.t().contiguous()) / math.sqrt(DIM)
        hidden = torch.arange(k.shape[0], device=q.device)[None, :] >= limit[a : a + 4096, None]
        s.masked_fill_(hidden, -math.inf)
        out[a : a + 4096] = torch.mm(torch.softmax(s, dim=-1), v)
    return out


def _gather(pool, table, n):
    """Logical (kv_heads, n, dim) rows of a paged sequence."""
    idx = torch.tensor(table, device=pool.device, dtype=torch.long)
    return pool[idx].permute(1, 0, 2, 3).reshape(pool.shape[1], -1, DIM)[:, :n].double()


def _exact_attention(case, st, q, k_pool, v_pool):
    """q (tokens, heads, dim) in 64 bits; returns (heads, tokens, dim)."""
    H, KVH = case["heads"], case["kv_heads"]
    rep = H // KVH
    out = torch.empty((H, q.shape[0], DIM), dtype=torch.float64, device=q.device)
    t0 = 0
    for (p, n), table in zip(st["chunks"], st["tables"]):
        k, v = _gather(k_pool, table, p + n), _gather(v_pool, table, p + n)
        limit = torch.arange(p + 1, p + n + 1, device=q.device).repeat(rep)
        for g in range(KVH):
            qg = q[t0 : t0 + n, g * rep : (g + 1) * rep].transpose(0, 1).reshape(rep * n, DIM).contiguous()
            o = _softmax_av(qg, k[g].contiguous(), v[g].contiguous(), limit)
            out[g * rep : (g + 1) * rep, t0 : t0 + n] = o.reshape(rep, n, DIM)
        t0 += n
    return out


def exact(case, seed):
    st = prepare(case, seed)
    H, KVH = case["heads"], case["kv_heads"]
    if case["kind"] == "dense":
        q, k, v = (st[x].double() for x in ("q", "k", "v"))
        out = torch.empty_like(q)
        rep = H // KVH
        limit = torch.full((q.shape[2],), k.shape[2], device=q.device)
        for b in range(q.shape[0]):
            for h in range(H):
                out[b, h] = _softmax_av(q[b, h].contiguous(), k[b, h // rep].contiguous(), v[b, h // rep].contiguous(), limit)
        return out
    if case["kind"] in ("decode", "prefill"):
        return _exact_attention(case, st, st["q"].transpose(0, 1).double(), st["k_pool"], st["v_pool"])

    pos = torch.cat([torch.arange(p, p + n) for p, n in st["chunks"]]).to(st["q"].device)
    cos, sin = st["cos"].double()[pos][:, None, :], st["sin"].double()[pos][:, None, :]

    def norm_rope(x, w):
        x = x.double()
        x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()
        a, b = x.chunk(2, dim=-1)
        return cos * x + sin * torch.cat((-b, a), dim=-1)

    q, k = norm_rope(st["q"], st["wq"]), norm_rope(st["k"], st["wk"])
    k_pool, v_pool = st["k_pool"].double(), st["v_pool"].double()
    blocks = torch.cat([torch.tensor(t, dtype=torch.long)[torch.arange(p, p + n) // PAGE]
                        for (p, n), t in zip(st["chunks"], st["tables"])]).to(pos.device)
    k_pool[blocks, :, pos % PAGE] = k
    v_pool[blocks, :, pos % PAGE] = st["v"].double()
    if case["kind"] == "prologue":
        return {"q": q, "k_pool": k_pool, "v_pool": v_pool}
    return {"out": _exact_attention(case, st, q, k_pool, v_pool), "k_pool": k_pool, "v_pool": v_pool}
