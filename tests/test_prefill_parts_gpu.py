"""Matrix-core prefill of short chunks on long prefixes: each query tile's keys
over up to 16 workgroups, and fewer where the workspace holds no more.

Tolerance: fp16 operands, 2e-3 as in test_prefill_gpu.py.
"""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle.attention import prefill_one  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("prefix,chunk,H,Hkv,D,dtype", [
    ([4000], [16], 8, 2, 64, torch.float16),            # 16 parts of 4 tiles
    ([2300], [257], 3, 3, 128, torch.bfloat16),         # two query tiles; H * D / 4 = 96
    ([1000, 0, 1999], [3, 200, 1], 10, 5, 32, torch.bfloat16),
    ([300], [20], 12, 12, 64, torch.float16),           # 5 tiles: 4 parts, the last empty
])
def test_many_parts(prefix, chunk, H, Hkv, D, dtype):
    """The call's own workspace, and one that holds 5 parts."""
    from heteroserve import _hip
    from hsbench.cases import build_prefill

    need = int(sum(-(-(p + s) // 16) for p, s in zip(prefix, chunk)))
    case = build_prefill("t", np.array(prefix), np.array(chunk), H, Hkv, D, need + 8, dtype, DEV,
                         seed=sum(chunk) + D)
    lib, B, rows = _hip.lib(), len(prefix), max(chunk)
    full = lib.hs_prefill_workspace_bytes(B, rows, H, D, 1)
    five = 5 * B * rows * H * (D + 2) * 4 + 256
    cu = case.cu_seqlens.cpu().numpy()
    for nbytes in (full, min(full, five)):
        ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
        out = torch.empty_like(case.q)
        _hip.check(lib.hs_prefill_varlen(
            case.q.data_ptr(), case.cu_seqlens.data_ptr(), rows, case.k_cache.data_ptr(),
            case.v_cache.data_ptr(), _hip.dtype_code(dtype), case.k_cache.shape[0],
            case.block_tables.data_ptr(), case.context_lens.data_ptr(), out.data_ptr(), B, H, Hkv,
            D, 16, case.block_tables.shape[1], case.scale, 1, ws.data_ptr(), nbytes,
            _hip.stream_of(case.q.device)))
        for b in range(B):
            want = prefill_one(case.q[cu[b]:cu[b + 1]].cpu(), case.k_cache.cpu(),
                               case.v_cache.cpu(), case.block_tables[b].cpu(), int(case.ctx[b]),
                               case.scale)
            got = out[cu[b]:cu[b + 1]].cpu()
            assert (got - want).abs().max().item() <= 2e-3, (nbytes, b)
