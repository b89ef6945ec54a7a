"""Decode paths that give a (row, head) or a KV head's group a workgroup: plain
multi-head attention in one pass and by splits (8 waves a row, rows dealt
longest first, several slices taken together), and grouped heads on the fp32
matrix cores (default partitions, one pass, splits), at the edges of their
key tiles, slices and partitions.

Tolerance.  fp32 throughout: as in test_prefill_rows_gpu.py, 1e-6 in the
2-norm against fp64.
"""

from __future__ import annotations

import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
REL = 1e-6


def _case(ctxs, H, Hkv, D, BS, dtype, seed=0):
    rng = np.random.default_rng(seed)
    need = [-(-max(n, 0) // BS) for n in ctxs]
    width = max(max(need), 1) + 1
    ids = rng.permutation(sum(need) + 2)
    bt = np.full((len(ctxs), width), -1, dtype=np.int32)
    at = 0
    for i, k in enumerate(need):
        bt[i, :k] = ids[at:at + k]
        at += k
    gen = torch.Generator().manual_seed(seed)
    k, v = (torch.randn((sum(need) + 2, BS, Hkv, D), generator=gen).to(dtype) for _ in range(2))
    return (torch.randn((len(ctxs), H, D), generator=gen), k, v, torch.from_numpy(bt),
            torch.tensor(ctxs, dtype=torch.int32), 1.0 / math.sqrt(D))


def _want(q, k, v, bt, ctx, scale):
    out = torch.zeros(q.shape, dtype=torch.float64)
    g = q.shape[1] // k.shape[2]
    for b, n in enumerate(ctx.tolist()):
        n = min(n, bt.shape[1] * k.shape[1])
        if n <= 0:
            continue
        pages = bt[b, :-(-n // k.shape[1])].long()
        kk, vv = (x[pages].reshape(-1, *x.shape[2:])[:n].double().repeat_interleave(g, 1)
                  for x in (k, v))
        p = torch.softmax(torch.einsum("hd,nhd->hn", q[b].double(), kk) * scale, -1)
        out[b] = torch.einsum("hn,nhd->hd", p, vv)
    return out


def _runs(case, splits=(0, 1, 2, 7, 64)):
    from heteroserve import _hip

    dev = [x.to(DEV) if torch.is_tensor(x) else x for x in case]
    want = _want(*case)
    for s in splits:
        got = _hip.decode(*dev, num_splits=s).cpu().double()
        err = ((got - want).norm() / want.norm()).item()
        assert err <= REL, (s, err)
        assert torch.equal(got[case[4] <= 0], torch.zeros_like(got[case[4] <= 0])), s


EDGES = [0, 1, 15, 16, 17, 127, 128, 129, -3, 300, 1031]


@pytest.mark.parametrize("dtype,H,Hkv,D,BS", [
    (torch.float32, 8, 2, 64, 16), (torch.float32, 6, 2, 128, 5), (torch.float32, 4, 2, 256, 16),
    (torch.float32, 3, 1, 32, 8), (torch.bfloat16, 10, 2, 128, 8), (torch.float16, 40, 2, 64, 32),
    (torch.float16, 16, 1, 256, 16), (torch.bfloat16, 8, 2, 64, 3), (torch.float16, 4, 2, 256, 16)])
def test_grouped_heads(dtype, H, Hkv, D, BS):
    """fp32 caches, groups above 4 or of 3 (one or several row tiles), and 16-bit
    groups of 2 and 4, which leave the VALU kernel in one pass only."""
    _runs(_case(EDGES, H, Hkv, D, BS, dtype))


@pytest.mark.parametrize("dtype,H,Hkv,D,BS", [
    (torch.float16, 8, 2, 128, 8), (torch.bfloat16, 4, 2, 64, 32), (torch.float16, 8, 4, 256, 16),
    (torch.float32, 32, 8, 128, 16), (torch.float32, 8, 4, 256, 16)])
@pytest.mark.parametrize("ctxs", [[0, 1, 15, 16, 17, 127, 128, 129, -3, 200],
                                  [0, 1, 15, 16, 17, 127, 128, 129, -3, 300, 975],
                                  [(29 * i) % 250 for i in range(32)]])
def test_grouped_short_rows(dtype, H, Hkv, D, BS, ctxs):
    """Groups of 2 and 4 whose tables hold at most 1024 tokens, in the default
    partitions: one or several, with and without a workgroup for every CU."""
    _runs(_case(ctxs, H, Hkv, D, BS, dtype, seed=4), splits=(0,))


@pytest.mark.parametrize("dtype,D,BS", [(torch.float16, 64, 16), (torch.float32, 128, 16),
                                        (torch.bfloat16, 256, 5), (torch.float32, 32, 3)])
def test_multi_head_rows(dtype, D, BS):
    """A workgroup per row: slices that start inside a load group, empty waves."""
    _runs(_case(EDGES, 5, 5, D, BS, dtype))


def test_longest_rows_first():
    """More workgroups than CUs: rows are dealt by rank, equal lengths and empty
    rows among them (64 sequences is the most that are ranked)."""
    ctxs = [(37 * i) % 200 for i in range(60)] + [77, 77, 0, 512]
    _runs(_case(ctxs, 6, 6, 64, 16, torch.float16, seed=1), splits=(0, 1, 3))
    _runs(_case(ctxs + [9], 6, 6, 64, 16, torch.float16, seed=2), splits=(0, 1, 3))


@pytest.mark.parametrize("splits", [0, 1, 5])
def test_values_past_the_context(splits):
    """Stale infinities and NaN in the last page reach no row."""
    from heteroserve import _hip

    case = _case([21, 40], 8, 2, 64, 16, torch.float32, seed=3)
    q, k, v, bt, ctx, scale = case
    want = _want(*case)
    for b, n in enumerate((21, 40)):
        for x in (k, v):
            x[bt[b, n // 16], n % 16:] = math.nan if b else math.inf
    got = _hip.decode(*(x.to(DEV) for x in (q, k, v, bt, ctx)), scale, num_splits=splits).cpu()
    assert ((got.double() - want).norm() / want.norm()).item() <= REL


def _fma(a, b, c):
    return (a.double() * b.double() + c.double()).float()


def _tree(parts):
    while len(parts) > 1:
        half = len(parts) // 2
        parts = [parts[i] + parts[i + half] for i in range(half)]
    return parts[0]


def _sliced_walk(q, k, v, splits):
    """One query row against its keys in fp32, a state per slice, summed as the
    VALU kernel sums a slice (chains over the elements of a 16-byte load and the
    tokens of a lane group, trees over lanes and groups) and the merge adds the
    slices up.  q [R, D], k and v [R, n, D]."""
    n, D = k.shape[1:]
    vec = 16 // k.element_size()
    tokens = 64 // (D // vec)
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
    acc, total = torch.zeros_like(q), torch.zeros(q.shape[0])
    size = -(-n // splits)
    for lo in range(0, n, size):
        accs, sums = [], []
        for r in range(tokens):
            a, t_sum = torch.zeros_like(q), torch.zeros(q.shape[0])
            for t in range(lo + r, min(lo + size, n), tokens):
                a, t_sum = _fma(p[:, t, None], v[:, t], a), t_sum + p[:, t]
            accs.append(a)
            sums.append(t_sum)
        acc, total = acc + _tree(accs), total + _tree(sums)
    return acc * (1.0 / total)[:, None]


@pytest.mark.parametrize("dtype,H,Hkv,D,batch,n,splits", [
    (torch.float32, 32, 32, 128, 128, 200, 7), (torch.float32, 8, 4, 256, 128, 64, 7),
    (torch.bfloat16, 8, 4, 256, 16, 200, 7), (torch.float32, 32, 8, 128, 128, 64, 7),
    (torch.float32, 12, 12, 64, 32, 500, 16), (torch.bfloat16, 32, 8, 64, 8, 700, 64)])
def test_splits_no_further_off_than_their_slices(dtype, H, Hkv, D, batch, n, splits):
    """Slices that are taken together add up no longer chains than one state per
    slice does: the error of that order, computed here, is not exceeded (both are
    random walks over at least 96 rows of D values; a tenth is more than chance
    gives)."""
    from heteroserve import _hip

    case = _case([n] * batch, H, Hkv, D, 8, dtype, seed=splits + n)
    q, k, v, bt, _, scale = case
    want = _want(*case)
    pages = bt[:, :-(-n // 8)].long()
    kk, vv = (x[pages].reshape(batch, -1, Hkv, D)[:, :n].repeat_interleave(H // Hkv, 2)
              .permute(0, 2, 1, 3).reshape(batch * H, n, D) for x in (k, v))
    rows = slice(0, 512)
    walk = _sliced_walk(q.reshape(-1, D)[rows], kk[rows], vv[rows], splits)
    exact = want.reshape(-1, D)[rows]
    limit = 1.1 * ((walk.double() - exact).norm() / exact.norm()).item()
    got = _hip.decode(*(x.to(DEV) for x in case[:5]), scale, num_splits=splits).cpu().double()
    assert ((got - want).norm() / want.norm()).item() <= limit


@pytest.mark.parametrize("dtype,H,Hkv,D,BS", [
    (torch.float32, 4, 2, 64, 16), (torch.bfloat16, 4, 2, 32, 8), (torch.float16, 6, 2, 128, 8),
    (torch.float32, 8, 2, 128, 16), (torch.bfloat16, 8, 2, 128, 8), (torch.float16, 4, 2, 256, 16),
    (torch.float32, 8, 2, 256, 16)])
@pytest.mark.parametrize("batch,longest", [(3, 64), (3, 250), (70, 250), (70, 500), (140, 130),
                                           (300, 40)])
def test_grouped_rows_around_the_rules(dtype, H, Hkv, D, BS, batch, longest):
    """Groups of 2, 3 and 4: few rows and a full device, short rows and longer
    ones, in the default partitions, in one pass and by splits."""
    ctxs = [(longest - 7 * i) % longest + (i % 2) for i in range(batch)]
    ctxs[0] = longest
    _runs(_case(ctxs, H, Hkv, D, BS, dtype, seed=longest), splits=(0, 1, 5))


def test_own_partitions_of_grouped_heads():
    """Partitions that the caller names, of one tile and of several."""
    from heteroserve import _hip

    for H, dtype in ((8, torch.float32), (16, torch.bfloat16)):
        case = _case([0, 1, 15, 16, 17, 100, 300], H, 2, 64, 8, dtype)
        want = _want(*case)
        for tokens in (16, 48, 512):
            got = _hip.decode(*(x.to(DEV) for x in case[:5]), case[5], num_splits=0,
                              partition_tokens=tokens)
            assert ((got.cpu().double() - want).norm() / want.norm()).item() <= REL, tokens


@pytest.mark.parametrize("H,D", [(8, 64), (8, 32)])
@pytest.mark.parametrize("batch", [32, 33, 65, 97, 129])
def test_one_pass_around_the_rules(H, D, batch):
    """Multi-head rows by a workgroup and by a wave: one to four rows a CU, tables
    on both sides of 128 and 256 tokens."""
    for longest in (128, 144, 272):
        ctxs = [longest - (5 * i) % 90 for i in range(batch)]
        case = _case(ctxs, H, H, D, 16, torch.float16, seed=batch)
        bt = case[3][:, :-(-longest // 16)].contiguous()
        _runs((*case[:3], bt, *case[4:]), splits=(1,))


@pytest.mark.parametrize("H,D,dtype,batch", [
    (32, 128, torch.bfloat16, 32), (32, 128, torch.bfloat16, 33), (32, 128, torch.bfloat16, 128),
    (16, 256, torch.float16, 66), (16, 64, torch.float32, 65), (16, 64, torch.float16, 65)])
def test_one_pass_of_many_long_rows(H, D, dtype, batch):
    """More than four rows a CU, up to sixteen, tables on both sides of 512 tokens."""
    for longest in (496, 512):   # tables of 512 and 528 tokens
        case = _case([longest] + [1 + (7 * i) % 40 for i in range(1, batch)], H, H, D, 16, dtype,
                     seed=batch)
        _runs(case, splits=(1,))
