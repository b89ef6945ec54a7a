"""The fp32 prefill (use_mfma = 0) on the fp32 matrix cores, at the sizes where
its tiles can go wrong: row tiles of 16 and 32, key tiles of 16, waves that
get no tile, block sizes that are no power of two, grouped heads that share a
row tile, ragged and padded rows, and values that a row must not see.

Tolerance.  Nothing is rounded below fp32, so the error is that of fp32 sums:
a random walk of at most max(D, n / 8) = 256 roundings of 2^-24 relative to the
result, 16 * 6e-8 = 1e-6 in the 2-norm against fp64.
"""

from __future__ import annotations

import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle.attention import prefill_one  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
REL = 1e-6


def _case(chunks, ctxs, H, Hkv, D, BS, dtype, seed=0):
    rng = np.random.default_rng(seed)
    need = [max(1, -(-max(n, 1) // BS)) for n in ctxs]
    ids = rng.permutation(sum(need) + 3)
    bt = np.full((len(ctxs), max(need) + 1), -1, dtype=np.int32)
    at = 0
    for i, k in enumerate(need):
        bt[i, :k] = ids[at:at + k]
        at += k
    gen = torch.Generator().manual_seed(seed)
    k, v = (torch.randn((sum(need) + 3, BS, Hkv, D), generator=gen).to(dtype) for _ in range(2))
    q = torch.randn((sum(chunks), H, D), generator=gen)
    return q, k, v, torch.from_numpy(bt), torch.tensor(ctxs, dtype=torch.int32)


def _run(q, k, v, bt, ctx, chunks, longest=None):
    from heteroserve.model.paged_attn_prefill import paged_attention_prefill_varlen

    cu = torch.tensor(np.concatenate([[0], np.cumsum(chunks)]), dtype=torch.int32)
    got = paged_attention_prefill_varlen(
        q.to(DEV), cu.to(DEV), longest or max(chunks), k.to(DEV), v.to(DEV), bt.to(DEV),
        ctx.to(DEV), 1.0 / math.sqrt(q.shape[2]), use_mfma=False)
    return got.cpu()


def _want(q, k, v, bt, ctx, chunks):
    """prefill_one in fp64: same function, doubled operands."""
    out, row = [], 0
    for b, n in enumerate(chunks):
        S, H, D = n, q.shape[1], q.shape[2]
        m = min(int(ctx[b]), bt.shape[1] * k.shape[1])
        res = torch.zeros((S, H, D), dtype=torch.float64)
        if S and m > 0:
            pages = bt[b, :-(-m // k.shape[1])].long().clamp(min=0)
            g = H // k.shape[2]
            kk, vv = (x[pages].reshape(-1, *x.shape[2:])[:m].double().repeat_interleave(g, 1)
                      for x in (k, v))
            s = torch.einsum("shd,nhd->shn", q[row:row + S].double(), kk) / math.sqrt(D)
            pos = int(ctx[b]) - S + torch.arange(S)
            s = s.masked_fill((torch.arange(m)[None] > pos[:, None])[:, None], -math.inf)
            res = torch.einsum("shn,nhd->shd", torch.nan_to_num(torch.softmax(s, -1)), vv)
        out.append(res)
        row += n
    return torch.cat(out)


def _rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("H,Hkv,BS", [(4, 4, 16), (6, 2, 5), (16, 1, 32), (3, 3, 1)])
def test_edges_of_tiles(dtype, D, H, Hkv, BS):
    """Chunks and contexts on both sides of 16, 32 and 8 x 16, in one ragged call."""
    chunks = [1, 15, 16, 17, 33, 0, 64]
    ctxs = [1, 15, 129, 200, 33, 40, 321]
    args = _case(chunks, ctxs, H, Hkv, D, BS, dtype)
    got = _run(*args, chunks)
    assert _rel(got, _want(*args, chunks)) <= REL


@pytest.mark.parametrize("D", [64, 128])
def test_wide_row_tiles(D):
    """Enough rows for the 32-row tiles (2 workgroups a CU), a remainder of 9."""
    chunks, ctxs = [521, 300], [521, 333]
    args = _case(chunks, ctxs, 32, 32, D, 16, torch.float32, seed=1)
    assert _rel(_run(*args, chunks), _want(*args, chunks)) <= REL


def test_one_to_two_workgroups_per_cu():
    """The reversed first round: 12 heads x 25 row tiles = 300 workgroups."""
    chunks, ctxs = [400], [500]
    args = _case(chunks, ctxs, 12, 12, 64, 16, torch.float32, seed=2)
    assert _rel(_run(*args, chunks), _want(*args, chunks)) <= REL


def test_short_context_rows_and_understated_maximum():
    """Rows at negative positions are zero, contexts past the table are cut at
    its end, and rows past max_seqlen_q are still served."""
    chunks, ctxs = [40, 50], [10, 96]
    args = _case(chunks, ctxs, 4, 2, 64, 16, torch.float16, seed=3)
    got = _run(*args, chunks)
    assert torch.all(got[:30] == 0)
    assert _rel(got, _want(*args, chunks)) <= REL
    assert torch.equal(_run(*args, chunks, longest=20), got)
    q, k, v, bt, ctx = args
    long_ctx = ctx.clone()
    long_ctx[1] = 500      # the table holds 112 tokens
    want = torch.cat([prefill_one(q[:40], k, v, bt[0], 10, 0.125),
                      prefill_one(q[40:], k, v, bt[1], 500, 0.125)])
    assert _rel(_run(q, k, v, bt, long_ctx, chunks), want.double()) <= REL


@pytest.mark.parametrize("bad", [math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D,H,Hkv", [(64, 2, 2), (128, 8, 2), (256, 2, 1)])
def test_rows_do_not_see_later_values(bad, dtype, D, H, Hkv):
    """A non-finite V value reaches the rows at or after its position, in its
    own head and dim only; stale values after the context reach no row."""
    chunks, ctxs = [50], [70]
    q, k, v, bt, ctx = _case(chunks, ctxs, H, Hkv, D, 16, dtype, seed=4)
    clean = _run(q, k, v, bt, ctx, chunks)
    pos = 45
    v[bt[0, pos // 16], pos % 16, 0, 7] = bad
    v[bt[0, 4], 70 - 64:, :, :] = bad        # past the context, in its last page
    k[bt[0, 4], 70 - 64:, :, :] = bad
    got = _run(q, k, v, bt, ctx, chunks)
    G = H // Hkv
    first = pos - 20                         # row of that position
    hit = torch.zeros_like(got, dtype=torch.bool)
    hit[first:, :G, 7] = True
    if math.isnan(bad):
        assert torch.isnan(got[hit]).all()
    else:
        assert (got[hit] == bad).all()
    # the others: the same values, up to the order of the sums in that tile
    assert _rel(got[~hit], clean[~hit].double()) <= REL


def _fma(a, b, c):
    return (a.double() * b.double() + c.double()).float()


def _tree(parts):
    while len(parts) > 1:
        half = len(parts) // 2
        parts = [parts[i] + parts[i + half] for i in range(half)]
    return parts[0]


def _row_walk(q, k, v):
    """One query row against its keys in fp32, summed as the VALU kernel sums:
    scores in chains of the elements of a 16-byte load and a tree over the
    lanes of a token, values in chains over the tokens of a lane group and a
    tree over the groups.  q [R, D], k and v [R, n, D]."""
    D = q.shape[1]
    vec = 16 // k.element_size()
    k, v = k.float(), v.float()
    qs = q * (math.log2(math.e) / math.sqrt(D))
    parts = []
    for c in range(D // vec):
        x = torch.zeros(k.shape[:2])
        for e in range(c * vec, (c + 1) * vec):
            x = _fma(qs[:, None, e], k[..., e], x)
        parts.append(x)
    s = _tree(parts)
    p = torch.exp2(s.double() - s.amax(1, keepdim=True).double()).float()
    tokens = 64 // (D // vec)
    accs, sums = [], []
    for r in range(tokens):
        acc, total = torch.zeros_like(q), torch.zeros(q.shape[0])
        for t in range(r, k.shape[1], tokens):
            acc, total = _fma(p[:, t, None], v[:, t], acc), total + p[:, t]
        accs.append(acc)
        sums.append(total)
    return _tree(accs) * (1.0 / _tree(sums))[:, None]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D,H,Hkv,batch,keys", [
    (128, 32, 32, 32, 17), (128, 32, 32, 8, 64), (128, 32, 8, 128, 17), (128, 32, 8, 96, 40),
    (256, 8, 4, 16, 17), (64, 12, 12, 64, 33), (32, 8, 8, 128, 33)])
def test_sums_no_further_off_than_the_row_walk(dtype, D, H, Hkv, batch, keys):
    """With few keys the error is that of the scores' sums.  It must not exceed
    the VALU kernel's order of sums (its error is computed here): both are
    random walks over at least 500 rows of D values, so a tenth between their
    2-norms is more than chance gives."""
    q, k, v, bt, ctx = _case([1] * batch, [keys] * batch, H, Hkv, D, 8, dtype, seed=keys + D)
    q = torch.randn(q.shape, generator=torch.Generator().manual_seed(D))
    want = _want(q, k, v, bt, ctx, [1] * batch)
    pages = bt[:, :-(-keys // 8)].long()
    kk, vv = (x[pages].reshape(batch, -1, Hkv, D)[:, :keys].repeat_interleave(H // Hkv, 2)
              .permute(0, 2, 1, 3).reshape(batch * H, keys, D) for x in (k, v))
    walk = _row_walk(q.reshape(-1, D), kk, vv).view(q.shape)
    got = _run(q, k, v, bt, ctx, [1] * batch)
    assert _rel(got, want) <= 1.1 * _rel(walk, want)
    from heteroserve import _hip

    got = _hip.decode(q.to(DEV), k.to(DEV), v.to(DEV), bt.to(DEV), ctx.to(DEV),
                      1.0 / math.sqrt(D), num_splits=1).cpu()
    assert _rel(got, want) <= 1.1 * _rel(walk, want)


@pytest.mark.parametrize("dtype,D", [(torch.float32, 128), (torch.bfloat16, 64),
                                     (torch.bfloat16, 32), (torch.float32, 64)])
@pytest.mark.parametrize("rows", [1, 16, 17, 32, 33])
def test_few_rows_of_many_sequences(dtype, D, rows):
    """A row tile or two of each of 64 sequences, 8 heads: grids of 512
    workgroups, on both sides of the rule for the 32-row tile."""
    chunks = [rows] * 64
    ctxs = [rows + 3 * i for i in range(64)]
    args = _case(chunks, ctxs, 8, 8, D, 16, dtype, seed=rows)
    assert _rel(_run(*args, chunks), _want(*args, chunks)) <= REL


def test_uniform_chunks_on_long_prefixes():
    """32-row tiles of an fp32 cache: uniform chunks of 17 to 32 rows on tables of
    1024 tokens or more."""
    from heteroserve.model.paged_attn_prefill import paged_attention_prefill

    for S, n in ((17, 1024), (32, 1040), (32, 1008)):
        chunks, ctxs = [S] * 64, [n - (i % 7) for i in range(64)]
        q, k, v, bt, ctx = _case(chunks, ctxs, 8, 8, 32, 16, torch.float32, seed=S)
        bt = bt[:, :-(-n // 16)].contiguous()
        got = paged_attention_prefill(q.view(64, S, 8, 32).to(DEV), k.to(DEV), v.to(DEV),
                                      bt.to(DEV), ctx.to(DEV), 1.0 / math.sqrt(32)).cpu()
        assert _rel(got.view(q.shape), _want(q, k, v, bt, ctx, chunks)) <= REL


@pytest.mark.parametrize("H,Hkv,D,dtype", [(4, 4, 64, torch.float32), (8, 2, 128, torch.bfloat16),
                                           (16, 1, 128, torch.float32), (4, 2, 256, torch.float16)])
@pytest.mark.parametrize("batch", [3, 200])
@pytest.mark.parametrize("keys", [16, 32, 48, 64, 96, 112, 160, 176])
def test_both_kernels_of_short_tables(H, Hkv, D, dtype, batch, keys):
    """Tables of 16 to 176 tokens, on both sides of the lines below which a wave
    per row serves the chunks: few sequences and a full device, ragged rows."""
    chunks = [1 + (5 * i) % min(13, keys) for i in range(batch)]
    ctxs = [max(n, keys - 3 * (i % 5)) for i, n in enumerate(chunks)]
    q, k, v, bt, ctx = _case(chunks, ctxs, H, Hkv, D, 16, dtype, seed=keys)
    bt = bt[:, :-(-max(ctxs) // 16)].contiguous()
    assert _rel(_run(q, k, v, bt, ctx, chunks), _want(q, k, v, bt, ctx, chunks)) <= REL
