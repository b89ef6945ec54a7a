"""The work a serving engine gives this library, as cases that can be timed.

A case is a dict of plain values; its "kind" says which entry points it calls:

  decode   one decode step's attention over a paged cache: paged_attention
           (with or without shared_pages), paged_attention_v2 or
           paged_attention_v3
  prefill  chunked causal prefill: paged_attention_prefill_wmma and the ragged
           paged_attention_prefill_varlen on the matrix cores, or
           paged_attention_prefill in fp32 arithmetic
  write    new K/V rows into the cache: scatter_kv, append_kv or write_kv
  move     whole blocks: export_blocks_device and write_blocks_device (a
           migration), or gather_kv_batch
  step     an engine's decode step over all layers: block_table_tensor once,
           then append_kv and paged_attention per layer

Context and chunk lengths are quantiles of the case's distribution, dealt to
the sequences in an order that the seed gives, so a case's work is the same for
every seed.  Pages lie scattered over a pool twice as large as they need.
"""

import math
import os
import statistics
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.abspath("hetero-serve_amd"))

from heteroserve.kv import pack  # noqa: E402
from heteroserve.model.paged_attn import paged_attention  # noqa: E402
from heteroserve.model.paged_attn_prefill import (  # noqa: E402
    paged_attention_prefill, paged_attention_prefill_varlen)
from heteroserve.model.paged_attn_v2 import paged_attention_v2  # noqa: E402
from heteroserve.model.paged_attn_v3 import choose_num_splits, paged_attention_v3  # noqa: E402
from heteroserve.model.paged_attn_wmma import paged_attention_prefill_wmma  # noqa: E402

DEV = "cuda:0"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}

# (query heads, KV heads, head dim) of the configurations this repository has:
# GPT-2 small, the Llama-style benchmark batches, Llama-3-8B's grouped heads,
# and the wider groups and head dims the tests cover.
GEOMETRIES = [(12, 12, 64), (32, 32, 128), (32, 8, 128), (32, 8, 64), (32, 4, 128), (16, 16, 64),
              (16, 1, 128), (8, 8, 32), (8, 4, 256)]


def listed():
    return [
        # The CPU-reference configuration: a small GPT-2 batch, where a step is
        # a few microseconds and launches and host work count.
        decode("decode_small", "v1", 8, 12, 12, 64, "f16", 16, 512),
        # The headline batch: 64 ragged sequences, multi-head, bf16.
        decode("decode_ragged", "v1", 64, 32, 32, 128, "bf16", 64, 8192, median=2048),
        # The same batch at Llama-3-8B's geometry.
        decode("decode_ragged_gqa", "v1", 64, 32, 8, 128, "bf16", 64, 8192, median=2048),
        # A few interactive sequences with long contexts.
        decode("decode_long_few", "v1", 4, 32, 8, 128, "f16", 8192, 32768),
        # Explicit context splits over an fp32 cache, the split count chosen by
        # the library's heuristic.
        decode("decode_splits_f32", "v3", 8, 12, 12, 64, "f32", 256, 4096),
        # A large batch of which half shares a cached 1024-token prefix.
        decode("decode_shared_prefix", "shared", 255, 32, 32, 128, "bf16", 256, 4096, shared=1024),
        # Eight ragged chunks with cached prefixes in one call.
        prefill("prefill_ragged", "varlen", 8, 32, 32, 128, "bf16", 128, 2048, 0, 4096),
        # The engine's call: one sequence's chunk, grouped heads, fp16.
        prefill("prefill_chunk_gqa", "wmma", 1, 32, 8, 128, "f16", 512, 512, 1536, 1536),
        # One chunk of an fp32 cache (GPT-2 small), which the matrix-core entry
        # point does not take.
        prefill("prefill_f32", "rows", 1, 12, 12, 64, "f32", 512, 512, 512, 512),
        # A 1024-token chunk's K and V from the fused QKV output into the cache.
        write("write_chunk", "scatter", 1, 32, 128, "bf16", "f32", 1024),
        # A 2048-token prefix of a 32-layer model to another worker's pool.
        move("migrate_prefix", "migrate", 32, 8, 128, "bf16", 128),
        # A whole decode step of GPT-2 small: 12 layers, 32 sequences.
        step("engine_step", 12, 32, 12, 12, 64, "f16", 64, 1024),
    ]


# --- case constructors -------------------------------------------------------


def decode(name, entry, batch, heads, kv_heads, dim, dtype, lo, hi, median=0, shared=0, block=16):
    return {"name": name, "kind": "decode", "entry": entry, "batch": batch, "heads": heads,
            "kv_heads": kv_heads, "dim": dim, "dtype": dtype, "block": block, "ctx_lo": lo,
            "ctx_hi": hi, "ctx_median": median, "shared": shared}


def prefill(name, entry, batch, heads, kv_heads, dim, dtype, s_lo, s_hi, p_lo, p_hi, block=16):
    return {"name": name, "kind": "prefill", "entry": entry, "batch": batch, "heads": heads,
            "kv_heads": kv_heads, "dim": dim, "dtype": dtype, "block": block, "chunk_lo": s_lo,
            "chunk_hi": s_hi, "prefix_lo": p_lo, "prefix_hi": p_hi}


def write(name, entry, layers, kv_heads, dim, dtype, src, tokens, block=16):
    return {"name": name, "kind": "write", "entry": entry, "layers": layers,
            "kv_heads": kv_heads, "dim": dim, "dtype": dtype, "src": src, "tokens": tokens,
            "block": block}


def move(name, entry, layers, kv_heads, dim, dtype, blocks, batch=1, block=16):
    return {"name": name, "kind": "move", "entry": entry, "layers": layers, "kv_heads": kv_heads,
            "dim": dim, "dtype": dtype, "blocks": blocks, "batch": batch, "block": block}


def step(name, layers, batch, heads, kv_heads, dim, dtype, lo, hi, block=16):
    return {"name": name, "kind": "step", "layers": layers, "batch": batch, "heads": heads,
            "kv_heads": kv_heads, "dim": dim, "dtype": dtype, "block": block, "ctx_lo": lo,
            "ctx_hi": hi}


# --- drawn cases -------------------------------------------------------------


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def _dtype(rng):
    return rng.choice(["f16", "bf16", "bf16", "f32"])


def draw(rng):
    kind = rng.choice(["decode", "decode", "shared", "prefill", "prefill", "rows", "write",
                       "move", "step"])
    heads, kv_heads, dim = rng.choice(GEOMETRIES)
    while True:
        c = _draw(rng, kind, heads, kv_heads, dim)
        del c["name"]
        if _affordable(c):
            return c


def _draw(rng, kind, heads, kv_heads, dim):
    block = rng.choice([16, 16, 16, 16, 8, 32])
    if kind == "decode":
        entry = rng.choice(["v1", "v1", "v2", "v3"])
        hi = _log(rng, 16, 8192 if entry == "v2" else 32768)   # v2: one pass per row
        return decode("", entry, _log(rng, 1, 256), heads, kv_heads, dim, _dtype(rng),
                      max(1, hi // rng.choice([1, 4, 32])), hi, block=block)
    if kind == "shared":
        if dim == 256:
            dim = 128
        hi = _log(rng, 512, 4096)
        return decode("", "shared", _log(rng, 8, 255), heads, kv_heads, dim,
                      rng.choice(["f16", "bf16"]), max(1, hi // 8), hi,
                      shared=rng.randint(32, hi) // 32 * 32)
    if kind == "prefill":
        if dim == 256:
            dim = 128
        dtype, prefix = rng.choice(["f16", "bf16"]), rng.choice([0, _log(rng, 1, 4096)])
        chunk = _log(rng, 2, 2048)
        if rng.random() < 0.5:
            return prefill("", "wmma", 1, heads, kv_heads, dim, dtype, chunk, chunk, prefix, prefix)
        return prefill("", "varlen", _log(rng, 2, 16), heads, kv_heads, dim, dtype,
                       max(1, chunk // 8), chunk, prefix // 4, prefix)
    if kind == "rows":
        dtype = rng.choice(["f32", "f32", "bf16", "f16"])
        if dtype != "f32" and dim != 256 and block == 16:
            block = rng.choice([8, 32])   # what the matrix-core entry point does not take
        chunk, prefix = _log(rng, 2, 2048), rng.choice([0, _log(rng, 1, 4096)])
        return prefill("", "rows", rng.choice([1, 1, 3]), heads, kv_heads, dim, dtype, chunk,
                       chunk, prefix, prefix, block)
    if kind == "write":
        entry = rng.choice(["scatter", "append", "write_kv"])
        return write("", entry, rng.choice([12, 32]) if entry == "write_kv" else 1, kv_heads, dim,
                     _dtype(rng), rng.choice(["f32", "f32", "f16", "bf16"]),
                     _log(rng, 1, 255 if entry == "append" else 2048), block)
    if kind == "move":
        if rng.random() < 0.3:
            return move("", "gather", 2, kv_heads, dim, _dtype(rng), _log(rng, 1, 256),
                        _log(rng, 1, 64), block)
        return move("", "migrate", rng.choice([1, 12, 32]), kv_heads, dim, _dtype(rng),
                    _log(rng, 1, 4096), 1, block)
    hi = _log(rng, 32, 4096)
    return step("", rng.choice([4, 12, 24]), _log(rng, 1, 128), heads, kv_heads, dim, _dtype(rng),
                max(1, hi // 8), hi, block)


def _affordable(c):
    """No dearer than the largest listed cases, in bytes read or written and in
    operations (in fp32 arithmetic: at the rate of vector units)."""
    w = work(c)
    matrix = c.get("entry") in ("wmma", "varlen", "shared") or \
        (c.get("entry") == "v1" and c["dtype"] != "f32")
    return w["bytes"] <= (1.2e9 if c["kind"] in ("move", "step", "write") else 5e9) and \
        w.get("flops", 0) <= (2e11 if matrix else 5e9)


# --- sizes -------------------------------------------------------------------


def _spread(lo, hi, n):
    """n values spread evenly over [lo, hi]."""
    return np.rint(lo + (hi - lo) * (np.arange(n) + 0.5) / n).astype(np.int64)


def _contexts(c):
    """The context lengths of a decode batch, in no particular order."""
    n = c["batch"]
    if c.get("ctx_median"):
        z = [statistics.NormalDist().inv_cdf((i + 0.5) / n) for i in range(n)]
        ctx = np.rint(c["ctx_median"] * np.exp(0.8 * np.array(z)))
        return np.clip(ctx, c["ctx_lo"], c["ctx_hi"]).astype(np.int64)
    return _spread(c["ctx_lo"], c["ctx_hi"], n)


def _sharers(c, ctx):
    """Which sequences start with the shared prefix (every other one)."""
    return (np.arange(len(ctx)) % 2 == 0) if c.get("shared") else np.zeros(len(ctx), bool)


def _chunks(c):
    """(chunk, prefix) lengths of a prefill batch; long chunks have short prefixes."""
    return (_spread(c["chunk_lo"], c["chunk_hi"], c["batch"]),
            _spread(c["prefix_lo"], c["prefix_hi"], c["batch"])[::-1])


def work(case):
    c = case
    if c["kind"] == "move":
        page = c["block"] * c["kv_heads"] * c["dim"] * BYTES[c["dtype"]]
        if c["entry"] == "gather":    # one layer's K and V pages, read and written
            return {"bytes": c["batch"] * c["blocks"] * 2 * page * 2}
        # pool -> payload -> pool
        return {"bytes": c["layers"] * c["blocks"] * 2 * page * 4}
    row = 2 * c["kv_heads"] * c["dim"]        # K and V elements of one token
    if c["kind"] == "write":
        return {"bytes": c["layers"] * c["tokens"] * row * (BYTES[c["dtype"]] + BYTES[c["src"]])}
    hd = c["heads"] * c["dim"]
    kv = row * BYTES[c["dtype"]]
    if c["kind"] == "prefill":
        s, p = _chunks(c)
        return {"bytes": int((s + p).sum()) * kv + int(s.sum()) * hd * 8,
                "flops": 4 * hd * int((s * p + s * (s + 1) // 2).sum())}
    ctx = _contexts(c)
    tokens = int(ctx.sum())
    if c["kind"] == "step":
        return {"bytes": c["layers"] * (tokens * kv + c["batch"] * (hd * 8 + row * 4)),
                "flops": c["layers"] * 4 * hd * tokens}
    if c["shared"]:
        mine = np.minimum(ctx, c["shared"])[_sharers(c, ctx)]
        tokens += int(mine.max()) - int(mine.sum())
    return {"bytes": tokens * kv + c["batch"] * hd * 8, "flops": 4 * hd * int(ctx.sum())}


# --- states ------------------------------------------------------------------


def _pool(gen, layers, blocks, c):
    """[layers, 2, blocks, block, kv_heads, dim] of N(0, 1), made in slabs."""
    pool = torch.empty((layers, 2, blocks, c["block"], c["kv_heads"], c["dim"]),
                       dtype=DTYPES[c["dtype"]], device=DEV)
    flat = pool.view(-1)
    for i in range(0, flat.numel(), 1 << 28):
        part = flat[i:i + (1 << 28)]
        part.normal_(generator=gen)
    return pool


def _tables(rng, lengths, block, share=None, shared=0):
    """(block lists, blocks of the pool): scattered pages for every length; the
    sequences in `share` start with the same blocks for `shared` tokens."""
    need = [-(-int(n) // block) for n in lengths]
    lead = [min(k, -(-shared // block)) if share is not None and share[b] else 0
            for b, k in enumerate(need)]
    common = max(lead, default=0)
    total = common + sum(need) - sum(lead)
    ids = rng.permutation(2 * total)[:total].tolist()
    first, at, out = ids[:common], common, []
    for k, s in zip(need, lead):
        out.append(first[:s] + ids[at:at + k - s])
        at += k - s
    return out, 2 * total


def _table_tensor(tables):
    bt = np.full((len(tables), max(len(t) for t in tables)), -1, dtype=np.int32)
    for i, t in enumerate(tables):
        bt[i, :len(t)] = t
    return torch.from_numpy(bt).to(DEV)


def _int32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).to(DEV)


def prepare(case, seed):
    c = case
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=DEV).manual_seed(int(seed))

    def normal(*shape, dtype=torch.float32):
        return torch.randn(shape, generator=gen, device=DEV).to(dtype)

    s = {"case": c, "scale": 1.0 / math.sqrt(c["dim"])}
    if c["kind"] == "decode":
        ctx = _contexts(c)
        share = _sharers(c, ctx)
        order = rng.permutation(len(ctx))
        ctx, share = ctx[order], share[order]
        tables, blocks = _tables(rng, ctx, c["block"], share, c["shared"])
        s.update(pool=_pool(gen, 1, blocks, c), tables=_table_tensor(tables), ctx=_int32(ctx),
                 lengths=ctx, q=normal(c["batch"], c["heads"], c["dim"]))
    elif c["kind"] == "prefill":
        chunk, prefix = _chunks(c)
        order = rng.permutation(len(chunk))
        chunk, prefix = chunk[order], prefix[order]
        tables, blocks = _tables(rng, chunk + prefix, c["block"])
        shape = ((int(chunk.sum()),) if c["entry"] == "varlen" else (c["batch"], int(chunk[0])))
        s.update(pool=_pool(gen, 1, blocks, c), tables=_table_tensor(tables),
                 ctx=_int32(chunk + prefix), lengths=chunk + prefix, chunk=chunk,
                 cu=_int32(np.concatenate([[0], np.cumsum(chunk)])), longest=int(chunk.max()),
                 q=normal(*shape, c["heads"], c["dim"]))
    elif c["kind"] == "write":
        n, hkv, d = c["tokens"], c["kv_heads"], c["dim"]
        src = DTYPES[c["src"]]
        if c["entry"] == "append":     # one new token of each of n sequences
            pos = rng.permutation(_spread(0, 32 * c["block"] - 1, n))
            tables, blocks = _tables(rng, pos + 1, c["block"])
            s.update(tables=_table_tensor(tables), positions=_int32(pos))
        else:                          # n tokens of one sequence, from the middle of a block
            start = 3 * c["block"] + c["block"] // 2 - 1
            tables, blocks = _tables(rng, [start + n], c["block"])
            s.update(table=tables[0], start=start)
        s["pool"] = _pool(gen, c["layers"], blocks, c)
        if c["entry"] == "write_kv":
            s.update(k=normal(c["layers"], hkv, n, d, dtype=src),
                     v=normal(c["layers"], hkv, n, d, dtype=src))
        else:                          # K and V inside the fused QKV rows
            qkv = normal(n, 3 * hkv * d, dtype=src)
            s.update(k=qkv[:, hkv * d:2 * hkv * d].view(n, hkv, d),
                     v=qkv[:, 2 * hkv * d:].view(n, hkv, d))
        if c["entry"] == "scatter":
            s["slots"] = pack.slots_for(s["table"], range(s["start"], s["start"] + n),
                                        c["block"]).to(DEV)
    elif c["kind"] == "move":
        if c["entry"] == "gather":
            tables, blocks = _tables(rng, [c["blocks"] * c["block"]] * c["batch"], c["block"])
            s.update(pool=_pool(gen, c["layers"], blocks, c), tables=tables)
        else:
            n = c["blocks"]
            s.update(pool=_pool(gen, c["layers"], 2 * n, c), other=_pool(gen, c["layers"], 2 * n, c),
                     source=rng.permutation(2 * n)[:n].tolist(),
                     target=rng.permutation(2 * n)[:n].tolist())
    else:
        ctx = _contexts(c)[rng.permutation(c["batch"])]
        tables, blocks = _tables(rng, ctx, c["block"])
        hd, kvd = c["heads"] * c["dim"], c["kv_heads"] * c["dim"]
        qkv = [normal(c["batch"], hd + 2 * kvd) for _ in range(c["layers"])]
        s.update(pool=_pool(gen, c["layers"], blocks, c), tables=tables, ctx=_int32(ctx),
                 lengths=ctx, positions=_int32(ctx - 1),
                 q=[x[:, :hd].contiguous().view(-1, c["heads"], c["dim"]) for x in qkv],
                 k=[x[:, hd:hd + kvd].view(-1, c["kv_heads"], c["dim"]) for x in qkv],
                 v=[x[:, hd + kvd:].view(-1, c["kv_heads"], c["dim"]) for x in qkv])
    return s


# --- one pass ----------------------------------------------------------------


def run(state):
    s, c = state, state["case"]
    pool, scale, entry = s["pool"], s["scale"], c.get("entry")
    if c["kind"] == "decode":
        args = (s["q"], pool[0, 0], pool[0, 1], s["tables"], s["ctx"], scale)
        if entry == "v1":
            return paged_attention(*args)
        if entry == "shared":
            return paged_attention(*args, shared_pages=True)
        if entry == "v2":
            return paged_attention_v2(*args)
        splits = choose_num_splits(c["batch"], c["heads"], int(s["lengths"].max()))
        return paged_attention_v3(*args, num_splits=splits)
    if c["kind"] == "prefill":
        if entry == "varlen":
            return paged_attention_prefill_varlen(s["q"], s["cu"], s["longest"], pool[0, 0],
                                                  pool[0, 1], s["tables"], s["ctx"], scale)
        call = paged_attention_prefill_wmma if entry == "wmma" else paged_attention_prefill
        return call(s["q"], pool[0, 0], pool[0, 1], s["tables"], s["ctx"], scale)
    if c["kind"] == "write":
        if entry == "scatter":
            pack.scatter_kv(pool[0, 0], pool[0, 1], s["slots"], s["k"], s["v"])
        elif entry == "append":
            pack.append_kv(pool[0, 0], pool[0, 1], s["tables"], s["positions"], s["k"], s["v"])
        else:
            pack.write_kv(pool, s["table"], s["start"], s["k"], s["v"])
        return pool
    if c["kind"] == "move":
        if entry == "gather":
            return pack.gather_kv_batch(pool, s["tables"], c["blocks"] * c["block"], 1)
        payload = pack.export_blocks_device(pool, s["source"])
        pack.write_blocks_device(s["other"], s["target"], payload)
        return payload, s["other"]
    tables = pack.block_table_tensor(s["tables"], device=DEV)
    outs = []
    for layer in range(c["layers"]):
        k_cache, v_cache = pool[layer, 0], pool[layer, 1]
        pack.append_kv(k_cache, v_cache, tables, s["positions"], s["k"][layer], s["v"][layer])
        outs.append(paged_attention(s["q"][layer], k_cache, v_cache, tables, s["ctx"], scale))
    return {"attention": outs, "pool": pool}


# --- how far a correct result may be off -------------------------------------


def tolerance(case):
    c = case
    if c["kind"] in ("write", "move"):
        return "exact"
    if c["kind"] == "prefill" and c["entry"] != "rows":
        # queries and probabilities are fp16 operands: 2.9e-4 from fp64
        return {"rel": 1.2e-3}
    if c["dtype"] == "bf16" and (c.get("shared") or c["heads"] != c["kv_heads"]):
        # queries and probabilities are pairs of bf16 terms, 16 bits in all:
        # 3.4e-6 from fp64
        return {"rel": 1.5e-5}
    # fp32 sums of up to 32768 terms: 1.5e-7 to 7e-7 from fp64
    return {"rel": 5e-6}


def _attend(q, k, v, scale, first):
    """fp64 attention of q [S, H, D] over k, v [n, Hkv, D]; row i sees keys up
    to first + i."""
    S, H, D = q.shape
    n, hkv, _ = k.shape
    g = H // hkv
    q = q.double().view(S, hkv, g, D).permute(1, 2, 0, 3).reshape(hkv, g * S, D)
    k = k.double().permute(1, 2, 0).contiguous()
    v = v.double().permute(1, 0, 2).contiguous()
    p = torch.bmm(q, k).mul_(scale).view(hkv, g, S, n)
    if S > 1:
        hidden = torch.arange(n, device=q.device)[None] > first + torch.arange(
            S, device=q.device)[:, None]
        p.masked_fill_(hidden, -math.inf)
    p = torch.softmax(p, -1).view(hkv, g * S, n)
    return torch.bmm(p, v).view(hkv, g, S, D).permute(2, 0, 1, 3).reshape(S, H, D)


def _rows(cache, table, n):
    """The first n tokens' rows of one sequence."""
    pages = cache.index_select(0, table[:-(-n // cache.shape[1])].long())
    return pages.reshape(-1, *cache.shape[2:])[:n]


def exact(case, seed):
    c = case
    if c["kind"] in ("write", "move"):
        return None                    # copies and casts: compared bit for bit
    s = prepare(c, seed)
    scale, lengths = s["scale"], [int(n) for n in s["lengths"]]

    def batch(q, k_cache, v_cache, tables, rows):
        out = []
        for b, n in enumerate(lengths):
            k, v = _rows(k_cache, tables[b], n), _rows(v_cache, tables[b], n)
            out.append(_attend(q[rows[b]:rows[b + 1]], k, v, scale, n - (rows[b + 1] - rows[b])))
        return torch.cat(out)

    if c["kind"] == "decode":
        return batch(s["q"], s["pool"][0, 0], s["pool"][0, 1], s["tables"],
                     list(range(len(lengths) + 1)))
    if c["kind"] == "prefill":
        rows = [int(x) for x in np.concatenate([[0], np.cumsum(s["chunk"])])]
        out = batch(s["q"].view(-1, c["heads"], c["dim"]), s["pool"][0, 0], s["pool"][0, 1],
                    s["tables"], rows)
        return out.view(s["q"].shape)
    tables = _table_tensor(s["tables"])
    outs = []
    for layer in range(c["layers"]):
        k_cache, v_cache = s["pool"][layer, 0], s["pool"][layer, 1]
        for b, n in enumerate(lengths):
            blk = s["tables"][b][(n - 1) // c["block"]]
            k_cache[blk, (n - 1) % c["block"]] = s["k"][layer][b].to(k_cache.dtype)
            v_cache[blk, (n - 1) % c["block"]] = s["v"][layer][b].to(v_cache.dtype)
        outs.append(batch(s["q"][layer], k_cache, v_cache, tables, list(range(len(lengths) + 1))))
    return {"attention": outs, "pool": None}
