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
