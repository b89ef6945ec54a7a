"""KV writes of several layers in one launch (write_kv) and the wrap of negative
slots in the kernel (scatter_kv with device slots): bit-exact against the
oracle at odd sizes, layouts and alignments."""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

from oracle import kvpack as kvp  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _bits(x):
    return x.cpu().view(torch.int32 if x.element_size() == 4 else torch.int16)


@pytest.mark.parametrize("src", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("cache", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L,H,T,D,BS,start", [(3, 2, 1, 64, 16, 5), (2, 3, 33, 32, 8, 7),
                                              (1, 1, 50, 128, 5, 0), (2, 2, 9, 36, 16, 30)])
def test_write_kv_layers(src, cache, L, H, T, D, BS, start):
    """Rows of 8-element groups and of others; a token-major view, a slice that
    starts off a 16-byte boundary, and table entries counted from the end."""
    from heteroserve.kv import pack

    nb = -(-(start + T) // BS) + 3
    gen = torch.Generator().manual_seed(T)
    table = torch.randperm(nb, generator=gen)[:-(-(start + T) // BS)].tolist()
    table[0] -= nb
    wide = torch.randn(L, H, T, D + 1, generator=gen).to(src)
    layouts = {
        "contiguous": wide[..., :D].contiguous(),
        "token-major": wide[..., :D].permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3),
        "off a boundary": wide[..., 1:],
    }
    for name, k in layouts.items():
        v = -k
        want = torch.zeros(L, 2, nb, BS, H, D, dtype=cache)
        kvp.write_kv(want, [t % nb for t in table], start, k, v)
        pool = torch.zeros_like(want, device=DEV)
        # the slice keeps its strides on the device
        kd = wide.to(DEV)[..., 1:] if name == "off a boundary" else k.to(DEV)
        pack.write_kv(pool, table, start, kd, -kd if name != "off a boundary" else v.to(DEV))
        assert torch.equal(_bits(pool), _bits(want)), name


def _random_bits(shape, dtype, gen):
    """Every bit pattern, NaN payloads and signs of NaN among them; at least one
    element in sixteen is a NaN."""
    size = torch.empty(0, dtype=dtype).element_size()
    word = torch.int32 if size == 4 else torch.int16
    low, high = torch.iinfo(word).min, torch.iinfo(word).max
    bits = torch.randint(low, high + 1, shape, generator=gen, dtype=torch.int64)
    nan = {torch.float32: 0x7F800001, torch.float16: 0x7C01, torch.bfloat16: 0x7F81}[dtype]
    bits = torch.where(torch.randint(0, 16, shape, generator=gen) == 0, bits | nan, bits)
    return bits.to(word).view(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L,H,T,D", [(2, 2, 9, 36), (2, 2, 9, 64), (1, 3, 5, 32), (1, 1, 4, 7)])
def test_equal_types_keep_every_bit(dtype, L, H, T, D):
    """Sources of the cache's type are copied word for word in every layout,
    also where a head's rows are no 16-byte groups: write_kv, scatter_kv and
    append_kv."""
    from heteroserve.kv import pack

    gen = torch.Generator().manual_seed(D)
    wide = _random_bits((L, H, T, D + 1), dtype, gen)
    nb, table = 4, [2, 0]
    for x in (wide[..., :D], wide[..., 1:], wide[..., :D].contiguous()):
        xd = wide.to(DEV)[..., 1:] if x.storage_offset() else x.to(DEV)
        want = torch.zeros(L, 2, nb, 8, H, D, dtype=dtype)
        kvp.write_kv(want, table, 3, x, x)
        pool = torch.zeros_like(want, device=DEV)
        pack.write_kv(pool, table, 3, xd, xd)
        assert torch.equal(_bits(pool), _bits(want))
        if L > 1:
            continue
        rows = xd[0].transpose(0, 1).contiguous()
        slots = pack.slots_for(table, range(3, 3 + T), 8)
        pool.zero_()
        pack.scatter_kv(pool[0, 0], pool[0, 1], slots, rows, rows)
        assert torch.equal(_bits(pool), _bits(want))
        pool.zero_()
        pack.append_kv(pool[0, 0], pool[0, 1], torch.tensor([table], dtype=torch.int32),
                       torch.arange(3, 3 + T, dtype=torch.int32), rows, rows,
                       torch.zeros(T, dtype=torch.int32))
        assert torch.equal(_bits(pool), _bits(want))


def test_write_kv_refuses_what_does_not_fit():
    from heteroserve.kv import pack

    pool = torch.zeros(2, 2, 4, 16, 2, 32, device=DEV)
    k = torch.ones(2, 2, 5, 32, device=DEV)
    pack.write_kv(pool, [1], 0, k[:, :, :0], k[:, :, :0])
    with pytest.raises(IndexError):
        pack.write_kv(pool, [1], 0, k[:1], k[:1])
    with pytest.raises(RuntimeError):
        pack.write_kv(pool, [1], 0, k[:, :1], k[:, :1])
    with pytest.raises(RuntimeError):
        pack.write_kv(pool, [1], 0, k, k[:, :, :4])
    with pytest.raises(RuntimeError):
        pack.write_kv(pool, [1], 0, k, k.half())
    with pytest.raises(IndexError):
        pack.write_kv(pool, [1], 12, k, k)      # past the table
    assert not pool.any()


@pytest.mark.parametrize("n", [1, 37])
def test_device_slots_wrap_and_skip(n):
    """Device slots: -1 is the last slot, those outside [-slots, slots) are left."""
    from heteroserve.kv import pack

    gk = torch.zeros(6, 8, 2, 32, dtype=torch.bfloat16, device=DEV)
    gv = torch.zeros_like(gk)
    rows = torch.randn(n + 2, 2, 32, device=DEV)
    slots = torch.cat([torch.arange(n) - n, torch.tensor([48, -49])])
    pack.scatter_kv(gk, gv, slots.to(DEV), rows, -rows)
    want = torch.zeros(48, 2, 32, dtype=torch.bfloat16)
    want[48 - n:] = rows[:n].cpu().to(torch.bfloat16)
    assert torch.equal(gk.view(48, 2, 32).cpu(), want)
    assert torch.equal(gv.view(48, 2, 32).cpu(), -want)


@pytest.mark.parametrize("L", [0, 32767, 32768, 65536])
def test_any_number_of_layers(L):
    """No layers, and one more than a launch's grid holds (strided K, one head)."""
    from heteroserve.kv import pack

    pool = torch.zeros(L, 2, 2, 1, 1, 8, dtype=torch.float16, device=DEV)
    k = torch.arange(L * 16, device=DEV).remainder(2039).to(torch.float16).view(L, 1, 1, 16)
    pack.write_kv(pool, [1], 0, k[..., :8], k[..., 8:])
    assert torch.equal(pool[:, 0, 1, 0], k[:, 0, :, :8]) and not pool[:, :, 0].any()
    assert torch.equal(pool[:, 1, 1, 0], k[:, 0, :, 8:])
