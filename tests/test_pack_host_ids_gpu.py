"""Pack and unpack around the number of ids that a kernel's arguments hold, of
16-byte and of odd pages, with repeated ids and under capture: byte for byte."""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("shape", [(2, 3, 32), (1, 1, 3)])
@pytest.mark.parametrize("n", [1, 895, 896, 897])
def test_round_trip(n, shape):
    from heteroserve import _hip
    from heteroserve.kv import pack

    assert _hip.HOST_IDS == 896
    BS, H, D = shape
    rng = np.random.default_rng(n)
    pool = torch.randint(0, 2 ** 15, (2, 2, 1000, BS, H, D), dtype=torch.int16).view(torch.bfloat16)
    ids = rng.permutation(1000)[:n]
    ids[0] -= 1000                      # counts from the end
    dev = pool.to(DEV)
    got = pack.export_blocks_device(dev, ids.tolist())
    want = pool[:, :, ids].permute(2, 0, 1, 3, 4, 5).contiguous()
    assert torch.equal(got.cpu().view(torch.int16), want.view(torch.int16))
    other = torch.zeros_like(dev)
    target = rng.permutation(1000)[:n]
    pack.write_blocks_device(other, target.tolist(), got)
    ref = torch.zeros_like(pool)
    ref[:, :, target] = want.permute(1, 2, 0, 3, 4, 5)
    assert torch.equal(other.cpu().view(torch.int16), ref.view(torch.int16))


def test_capture_holds_the_ids():
    from heteroserve.kv import pack

    pool = torch.randn(2, 2, 50, 16, 2, 32, device=DEV)
    ids = [7, 3, 49]
    want = pool[:, :, ids].permute(2, 0, 1, 3, 4, 5).contiguous()
    pack.export_blocks_device(pool, ids)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = pack.export_blocks_device(pool, ids)
    ids[:] = [1, 1, 1]
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        want.add_(1)
        pool.add_(1)
