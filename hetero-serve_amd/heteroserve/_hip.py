"""Loader and tensor marshalling for libhsattn.so (the gfx950 C-ABI library).

This module is the only place that touches ctypes.  It keeps the reference's
module-state contract (heteroserve/model/paged_attn.py:197-252): the library is
loaded once, on first use, and a failure is recorded with a reason rather than
raised at import.  Unlike the reference there is no compute fallback: an entry
point called while the library is unavailable raises RuntimeError.

Environment:
  HETEROSERVE_DISABLE_CUDA_KERNEL  treat the library as unavailable (reference flag)
  HETEROSERVE_HIP_LIB              path of libhsattn.so (default: next to this file)
  HETEROSERVE_PREFILL_GRID=1       keep the MFMA prefill on its grid kernel (one workgroup
                                   per query tile) where the persistent one would run;
                                   read at each call, for comparisons

PyTorch provides device memory and the current stream; every kernel launches
on ``torch.cuda.current_stream(device)`` of the input's device.
"""

from __future__ import annotations

import ctypes
import os
import threading
from pathlib import Path
from typing import Optional

try:
    import torch
except ImportError as _exc:   # reported by _load()
    torch = None
    _torch_error = str(_exc)

ABI_VERSION = 5
DTYPE_F32, DTYPE_F16, DTYPE_BF16 = 0, 1, 2

_lock = threading.Lock()
_lib: Optional[ctypes.CDLL] = None
_state = "unloaded"          # "unloaded" | "ready" | "unavailable"
_error: Optional[str] = None

_c_int, _c_i64, _c_size, _c_float, _c_vp = (
    ctypes.c_int, ctypes.c_int64, ctypes.c_size_t, ctypes.c_float, ctypes.c_void_p)

# name -> (restype, argtypes); must match include/hsattn.h
_SIGNATURES = {
    "hs_abi_version": (_c_int, []),
    "hs_last_error": (ctypes.c_char_p, []),
    "hs_profile_next_launch": (_c_int, [_c_vp, _c_vp]),
    "hs_device_cu_count": (_c_int, [_c_int]),
    "hs_choose_num_splits": (_c_i64, [_c_i64, _c_i64, _c_i64]),
    "hs_decode_workspace_bytes": (_c_size, [_c_int] * 8),
    "hs_decode": (_c_int, [_c_vp, _c_vp, _c_vp, _c_int, _c_int, _c_vp, _c_vp, _c_vp,
                           _c_int, _c_int, _c_int, _c_int, _c_int, _c_int, _c_float,
                           _c_int, _c_int, _c_vp, _c_size, _c_vp]),
    "hs_decode_noalloc": (_c_int, [_c_vp, _c_vp, _c_vp, _c_int, _c_int, _c_vp, _c_vp, _c_vp,
                                   _c_int, _c_int, _c_int, _c_int, _c_int, _c_int, _c_float,
                                   _c_int, _c_int, _c_vp]),
    "hs_decode_shared_workspace_bytes": (_c_size, [_c_int] * 7),
    "hs_decode_shared": (_c_int, [_c_vp, _c_vp, _c_vp, _c_int, _c_int, _c_vp, _c_vp, _c_vp,
                                  _c_int, _c_int, _c_int, _c_int, _c_int, _c_int, _c_float,
                                  _c_int, _c_vp, _c_size, _c_vp]),
    "hs_prefill_workspace_bytes": (_c_size, [_c_int] * 5),
    "hs_prefill": (_c_int, [_c_vp, _c_vp, _c_vp, _c_int, _c_int, _c_vp, _c_vp, _c_vp,
                            _c_int, _c_int, _c_int, _c_int, _c_int, _c_int, _c_int,
                            _c_float, _c_int, _c_vp, _c_size, _c_vp]),
    "hs_prefill_varlen": (_c_int, [_c_vp, _c_vp, _c_int, _c_vp, _c_vp, _c_int, _c_int,
                                   _c_vp, _c_vp, _c_vp, _c_int, _c_int, _c_int, _c_int,
                                   _c_int, _c_int, _c_float, _c_int, _c_vp, _c_size, _c_vp]),
    "hs_kv_pack": (_c_int, [_c_vp, _c_int, _c_int, _c_i64, _c_vp, _c_int, _c_vp, _c_vp]),
    "hs_kv_unpack": (_c_int, [_c_vp, _c_int, _c_int, _c_i64, _c_vp, _c_int, _c_vp, _c_vp]),
    "hs_kv_gather": (_c_int, [_c_vp, _c_int, _c_int, _c_i64, _c_vp, _c_int, _c_int, _c_int,
                              _c_vp, _c_vp]),
    "hs_block_tables": (_c_int, [_c_vp, _c_int, _c_int, _c_vp, _c_vp]),
    "hs_kv_scatter": (_c_int, [_c_vp, _c_vp, _c_int, _c_i64, _c_int, _c_int, _c_vp, _c_i64,
                               _c_vp, _c_vp, _c_int, _c_i64, _c_vp]),
    "hs_kv_append": (_c_int, [_c_vp, _c_vp, _c_int, _c_int, _c_int, _c_int, _c_int, _c_vp,
                              _c_int, _c_int, _c_vp, _c_vp, _c_i64, _c_vp, _c_vp, _c_int, _c_i64,
                              _c_vp]),
}

EXPORTED_SYMBOLS = tuple(_SIGNATURES)

# entry points of this layer's own; must match csrc/hs_private.h
_PRIVATE = {
    "hs_kv_pack_host_ids": (_c_int, [_c_vp, _c_int, _c_int, _c_i64, _c_vp, _c_int, _c_vp, _c_vp]),
    "hs_kv_unpack_host_ids": (_c_int, [_c_vp, _c_int, _c_int, _c_i64, _c_vp, _c_int, _c_vp, _c_vp]),
    "hs_kv_scatter_layers": (_c_int, [_c_vp, _c_vp, _c_int, _c_i64, _c_int, _c_int, _c_int, _c_i64,
                                      _c_vp, _c_i64, _c_vp, _c_vp, _c_int, _c_i64, _c_i64, _c_i64,
                                      _c_vp]),
}


def lib_path() -> Path:
    env = os.environ.get("HETEROSERVE_HIP_LIB")
    return Path(env) if env else Path(__file__).resolve().parent / "libhsattn.so"


def open_library(path: Optional[Path] = None) -> ctypes.CDLL:
    """dlopen libhsattn.so and bind its signatures.  Needs no GPU.  OSError when the
    library is of another ABI, or was built without an entry point that this
    layer calls."""
    path = path or lib_path()
    lib = ctypes.CDLL(str(path))

    def bind(name, res, args):
        fn = getattr(lib, name, None)
        if fn is None:
            raise OSError(f"no {name} in {path}: rebuild it")
        fn.restype = res
        fn.argtypes = args
        return fn

    got = bind("hs_abi_version", *_SIGNATURES["hs_abi_version"])()
    if got != ABI_VERSION:
        raise OSError(f"libhsattn ABI version {got}, expected {ABI_VERSION}")
    for name, (res, args) in {**_SIGNATURES, **_PRIVATE}.items():
        bind(name, res, args)
    return lib


def _load() -> None:
    global _lib, _state, _error
    if _state != "unloaded":
        return
    with _lock:
        if _state != "unloaded":
            return
        if os.environ.get("HETEROSERVE_DISABLE_CUDA_KERNEL"):
            _state, _error = "unavailable", "disabled by HETEROSERVE_DISABLE_CUDA_KERNEL"
            return
        if torch is None:
            _state, _error = "unavailable", f"torch unavailable: {_torch_error}"
            return
        if not torch.cuda.is_available():
            _state, _error = "unavailable", "no HIP device"
            return
        arch = getattr(torch.cuda.get_device_properties(0), "gcnArchName", "").split(":")[0]
        if arch != "gfx950":
            _state, _error = "unavailable", (
                f"libhsattn.so is built for gfx950 only; device 0 is {arch or 'unknown'}")
            return
        path = lib_path()
        if not path.exists():
            _state, _error = "unavailable", (
                f"{path} is missing -- build it with python hetero-serve_amd/build.py")
            return
        try:
            _lib = open_library(path)
        except OSError as exc:
            _state, _error = "unavailable", f"OSError: {str(exc)[:200]}"
            return
        _state = "ready"


def ready() -> bool:
    _load()
    return _state == "ready"


def error() -> Optional[str]:
    _load()
    return _error


def lib(what: str = "paged attention HIP kernel") -> ctypes.CDLL:
    """The loaded library, or RuntimeError naming why it is unavailable."""
    if _state == "ready":
        return _lib
    _load()
    if _state != "ready":
        raise RuntimeError(f"{what} unavailable: {_error}")
    return _lib


def check(rc: int) -> None:
    if rc != 0:
        raise RuntimeError(_lib.hs_last_error().decode(errors="replace"))


# ---------------------------------------------------------------------------
# marshalling helpers
#
# A small decode step is a few microseconds on the GPU, so the calls below are
# what such a step costs: they compare device indexes (an int from one C call)
# instead of device objects, convert only what needs converting, ask torch for
# the raw stream, and remember workspace sizes.  A decode call of 8 sequences
# took 16.2 us of host time before.
# ---------------------------------------------------------------------------

_DTYPE_CODES = {} if torch is None else {
    torch.float32: DTYPE_F32, torch.float16: DTYPE_F16, torch.bfloat16: DTYPE_BF16}
_raw_stream = getattr(getattr(torch, "_C", None), "_cuda_getCurrentRawStream", None)


def dtype_code(dt) -> int:
    code = _DTYPE_CODES.get(dt)
    if code is None:
        raise RuntimeError(f"unsupported KV cache dtype {dt} (float32, float16 or bfloat16)")
    return code


def stream_of(device) -> int:
    if _raw_stream is not None:
        return _raw_stream(torch.cuda.current_device() if device.index is None else device.index)
    return torch.cuda.current_stream(device).cuda_stream


def _stream_at(index: int) -> int:
    """The current stream of device `index`."""
    if _raw_stream is not None:
        return _raw_stream(index)
    return torch.cuda.current_stream(index).cuda_stream


def _int32_on(t, device):
    if not torch.is_tensor(t):
        t = torch.as_tensor(t)
    if t.dtype is torch.int32 and t.get_device() == device.index and t.is_contiguous():
        return t
    return t.to(device=device, dtype=torch.int32).contiguous()


def _check_device(q, k_cache, v_cache) -> int:
    """The device index that all three tensors are on."""
    index = q.get_device()
    if index < 0 or not q.is_cuda:
        raise RuntimeError("q must be on CUDA")
    if k_cache.get_device() != index or v_cache.get_device() != index:
        if not (k_cache.is_cuda and v_cache.is_cuda):
            raise RuntimeError("kv cache must be on CUDA")
        raise RuntimeError("q and the kv cache must be on the same device")
    return index


def _check_q(q):
    if q.dtype is not torch.float32:
        raise RuntimeError(f"q must be float32, got {q.dtype}")
    return q.contiguous()


def _check_kv(k_cache, v_cache, D):
    """(k_cache, v_cache) contiguous, and their shape."""
    shape = k_cache.shape
    if len(shape) != 4:
        raise RuntimeError("k_cache must be [NB, BS, H, D]")
    if v_cache.shape != shape:
        raise RuntimeError("v_cache must have the shape of k_cache")
    if k_cache.dtype is not v_cache.dtype:
        raise RuntimeError("k_cache and v_cache must have the same dtype")
    if shape[3] != D:
        raise RuntimeError(f"head_dim mismatch: q has {D}, cache has {shape[3]}")
    return k_cache.contiguous(), v_cache.contiguous(), shape


class _DeviceGuard:
    """Make device `index` current for the duration of a library call."""

    __slots__ = ("_index", "_prev")

    def __init__(self, index: int):
        self._index = index
        self._prev = None

    def __enter__(self):
        cur = torch.cuda.current_device()
        if cur != self._index:
            self._prev = cur
            torch.cuda.set_device(self._index)

    def __exit__(self, *exc):
        if self._prev is not None:
            torch.cuda.set_device(self._prev)


# Workspace sizes of decode calls by their arguments and device.  The sizes are
# fixed for a device and a library; the table is emptied when it grows past
# what a server's batch sizes and table widths make.
_WS_SIZES: dict = {}
_WS_SIZES_MAX = 4096


def _decode_workspace(query, index: int, *sizes: int) -> int:
    """query(*sizes), with device `index` current (only sizes above 0 are kept:
    0 may also be a failed query)."""
    key = (query.__name__, index, sizes)
    n = _WS_SIZES.get(key)
    if n is None:
        n = query(*sizes)
        if n:
            if len(_WS_SIZES) >= _WS_SIZES_MAX:
                _WS_SIZES.clear()
            _WS_SIZES[key] = n
    return n


def decode(q, k_cache, v_cache, block_tables, context_lens, scale: float,
           num_splits: int, partition_tokens: int = 0, shared_pages: bool = False):
    """out[B, H, D] fp32 = paged decode attention via hs_decode.

    shared_pages=True (fixed partitions only, num_splits == 0) runs
    hs_decode_shared: partitions whose block ids several sequences share are
    read once for all of them."""
    L = lib()
    index = _check_device(q, k_cache, v_cache)
    if q.dim() != 3:
        raise RuntimeError("q must be [B, H, D]")
    q = _check_q(q)
    B, H, D = q.shape
    k_cache, v_cache, (NB, BS, Hkv, _) = _check_kv(k_cache, v_cache, D)
    dev = q.device
    bt = _int32_on(block_tables, dev)
    ctx = _int32_on(context_lens, dev)
    if bt.dim() != 2 or bt.shape[0] != B:
        raise RuntimeError("block_tables must be [B, max_blocks]")
    if ctx.numel() != B:
        raise RuntimeError("context_lens must have one entry per sequence")
    MB = bt.shape[1]
    out = q.new_empty(q.shape)
    if B == 0:
        return out
    scale, num_splits, partition_tokens = float(scale), int(num_splits), int(partition_tokens)
    if shared_pages and num_splits != 0:
        raise RuntimeError("shared_pages needs fixed partitions (num_splits == 0)")
    with _DeviceGuard(index):
        if shared_pages:
            ws_bytes = _decode_workspace(L.hs_decode_shared_workspace_bytes, index, B, H, Hkv, D,
                                         BS, max(MB, 1), partition_tokens)
        else:
            ws_bytes = _decode_workspace(L.hs_decode_workspace_bytes, index, B, H, Hkv, D, BS,
                                         max(MB, 1), num_splits, partition_tokens)
        ws = q.new_empty((ws_bytes + 3) // 4) if ws_bytes else None
        wsp = ws.data_ptr() if ws is not None else None
        if shared_pages:
            rc = L.hs_decode_shared(
                q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), dtype_code(k_cache.dtype),
                NB, bt.data_ptr(), ctx.data_ptr(), out.data_ptr(), B, H, Hkv, D, BS, MB,
                scale, partition_tokens, wsp, ws_bytes, _stream_at(index))
        else:
            rc = L.hs_decode(
                q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), dtype_code(k_cache.dtype),
                NB, bt.data_ptr(), ctx.data_ptr(), out.data_ptr(), B, H, Hkv, D, BS, MB,
                scale, num_splits, partition_tokens, wsp, ws_bytes, _stream_at(index))
        check(rc)
    return out


def _prefill_workspace(L, B: int, rows: int, H: int, D: int, use_mfma: bool, split: bool,
                       device):
    """(tensor or None, bytes): the key-range split's scratch, when it applies."""
    nbytes = L.hs_prefill_workspace_bytes(B, rows, H, D, int(bool(use_mfma))) if split else 0
    if not nbytes:
        return None, 0
    return torch.empty(nbytes, dtype=torch.uint8, device=device), nbytes


def prefill(q, k_cache, v_cache, block_tables, context_lens, scale: float, use_mfma: bool,
            split: bool = True):
    """out[B, S, H, D] fp32 = causal chunked prefill via hs_prefill.

    split=False passes no workspace, so the matrix-core kernel runs without
    the key-range split (for tests of that launch shape)."""
    L = lib()
    index = _check_device(q, k_cache, v_cache)
    if q.dim() != 4:
        raise RuntimeError("q must be [B, S, H, D]")
    q = _check_q(q)
    B, S, H, D = q.shape
    k_cache, v_cache, (NB, BS, Hkv, _) = _check_kv(k_cache, v_cache, D)
    bt = _int32_on(block_tables, q.device)
    ctx = _int32_on(context_lens, q.device)
    if bt.dim() != 2 or bt.shape[0] != B:
        raise RuntimeError("block_tables must be [B, max_blocks]")
    if ctx.numel() != B:
        raise RuntimeError("context_lens must have one entry per sequence")
    out = q.new_empty(q.shape)
    if B == 0 or S == 0:
        return out
    with _DeviceGuard(index):
        ws, ws_bytes = _prefill_workspace(L, B, S, H, D, use_mfma, split, q.device)
        check(L.hs_prefill(
            q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), dtype_code(k_cache.dtype),
            NB, bt.data_ptr(), ctx.data_ptr(), out.data_ptr(), B, S, H, Hkv, D, BS,
            bt.shape[1], float(scale), int(bool(use_mfma)),
            ws.data_ptr() if ws is not None else None, ws_bytes, _stream_at(index)))
    return out


def prefill_varlen(q, cu_seqlens_q, max_seqlen_q: int, k_cache, v_cache, block_tables,
                   context_lens, scale: float, use_mfma: bool, split: bool = True):
    """out[T, H, D] fp32 for ragged chunks via hs_prefill_varlen (split as for
    prefill)."""
    L = lib()
    index = _check_device(q, k_cache, v_cache)
    if q.dim() != 3:
        raise RuntimeError("q must be [total_tokens, H, D]")
    q = _check_q(q)
    T, H, D = q.shape
    k_cache, v_cache, (NB, BS, Hkv, _) = _check_kv(k_cache, v_cache, D)
    bt = _int32_on(block_tables, q.device)
    ctx = _int32_on(context_lens, q.device)
    cu = _int32_on(cu_seqlens_q, q.device)
    B = bt.shape[0]
    if cu.numel() != B + 1 or ctx.numel() != B:
        raise RuntimeError("cu_seqlens_q must be [B + 1] and context_lens [B]")
    out = q.new_empty(q.shape)
    if B == 0 or T == 0:
        return out
    with _DeviceGuard(index):
        ws, ws_bytes = _prefill_workspace(L, B, int(max_seqlen_q), H, D, use_mfma, split,
                                          q.device)
        check(L.hs_prefill_varlen(
            q.data_ptr(), cu.data_ptr(), int(max_seqlen_q), k_cache.data_ptr(),
            v_cache.data_ptr(), dtype_code(k_cache.dtype), NB, bt.data_ptr(), ctx.data_ptr(),
            out.data_ptr(), B, H, Hkv, D, BS, bt.shape[1], float(scale),
            int(bool(use_mfma)), ws.data_ptr() if ws is not None else None, ws_bytes,
            _stream_at(index)))
    return out


def choose_num_splits(num_seqs: int, num_heads: int, max_context: int) -> int:
    L = lib("v3 kernel")
    s = L.hs_choose_num_splits(int(num_seqs), int(num_heads), int(max_context))
    if s < 0:
        raise RuntimeError(L.hs_last_error().decode(errors="replace"))
    return int(s)


HOST_IDS = 896   # most block ids that fit a kernel's arguments (csrc/hs_private.h)


def _pages(pool):
    """(layers, blocks, bytes of one page) of pool [L, 2, NB, BS, Hkv, D]."""
    Ls, _, NB, BS, H, D = pool.shape
    return Ls, NB, BS * H * D * pool.element_size()


def kv_pack(pool, ids_dev, out) -> None:
    """out[n, L, 2, page] = pool[L, 2, NB, page][:, :, ids]  (bitwise)."""
    L = lib("KV pack HIP kernel")
    index = pool.get_device()
    with _DeviceGuard(index):
        check(L.hs_kv_pack(pool.data_ptr(), *_pages(pool), ids_dev.data_ptr(), ids_dev.numel(),
                           out.data_ptr(), _stream_at(index)))


def kv_unpack(pool, ids_dev, src) -> None:
    """pool[:, :, ids[i]] = src[i]  (bitwise; ids must not repeat)."""
    L = lib("KV unpack HIP kernel")
    index = pool.get_device()
    with _DeviceGuard(index):
        check(L.hs_kv_unpack(pool.data_ptr(), *_pages(pool), ids_dev.data_ptr(),
                             ids_dev.numel(), src.data_ptr(), _stream_at(index)))


def kv_pack_host_ids(pool, ids, out) -> None:
    """kv_pack with at most HOST_IDS ids in a contiguous int64 numpy array."""
    L = lib("KV pack HIP kernel")
    index = pool.get_device()
    with _DeviceGuard(index):
        check(L.hs_kv_pack_host_ids(pool.data_ptr(), *_pages(pool), ids.ctypes.data, ids.size,
                                    out.data_ptr(), _stream_at(index)))


def kv_unpack_host_ids(pool, ids, src) -> None:
    """kv_unpack with at most HOST_IDS ids in a contiguous int64 numpy array."""
    L = lib("KV unpack HIP kernel")
    index = pool.get_device()
    with _DeviceGuard(index):
        check(L.hs_kv_unpack_host_ids(pool.data_ptr(), *_pages(pool), ids.ctypes.data, ids.size,
                                      src.data_ptr(), _stream_at(index)))


def kv_gather(cache, block_tables_dev, length: int, out) -> None:
    """out[B, length, Hkv, D] = cache[NB, BS, Hkv, D] gathered through the tables."""
    L = lib("KV gather HIP kernel")
    NB, BS = cache.shape[:2]
    row = cache[0, 0].numel() * cache.element_size()
    B, MB = block_tables_dev.shape
    with _DeviceGuard(cache.get_device()):
        check(L.hs_kv_gather(cache.data_ptr(), NB, BS, row, block_tables_dev.data_ptr(), MB,
                             B, int(length), out.data_ptr(), _stream_at(cache.get_device())))


def _rows(x, Hkv: int, D: int):
    """(tensor, row stride in elements) of new K or V rows [n, Hkv, D].

    Accepts [n, Hkv, D] or [n, Hkv * D]; the rows may be strided (a slice of
    the fused QKV output) but each row's Hkv * D elements must be contiguous.
    """
    if x.dim() == 3:
        if tuple(x.shape[1:]) != (Hkv, D):
            raise RuntimeError(f"K/V rows must be [n, {Hkv}, {D}], got {tuple(x.shape)}")
        row_ok = x.stride(2) == 1 and x.stride(1) == D
    elif x.dim() == 2:
        if x.shape[1] != Hkv * D:
            raise RuntimeError(f"K/V rows must be [n, {Hkv * D}], got {tuple(x.shape)}")
        row_ok = x.stride(1) == 1
    else:
        raise RuntimeError(f"K/V rows must be [n, Hkv, D], got {tuple(x.shape)}")
    if not row_ok:
        x = x.contiguous()
    stride = x.stride(0) if x.shape[0] > 1 else Hkv * D
    return x, stride


def _check_write(k_cache, v_cache, k, v):
    """The caches are written in place: CUDA, contiguous, same shape/dtype.
    Returns their shape and device index."""
    shape = k_cache.shape
    if len(shape) != 4:
        raise RuntimeError("k_cache must be [NB, BS, Hkv, D]")
    if v_cache.shape != shape or v_cache.dtype is not k_cache.dtype:
        raise RuntimeError("k_cache and v_cache must have the same shape and dtype")
    index = k_cache.get_device()
    if (index < 0 or v_cache.get_device() != index or k.get_device() != index
            or v.get_device() != index):
        if not (k_cache.is_cuda and v_cache.is_cuda and k.is_cuda and v.is_cuda):
            raise RuntimeError("kv cache and new rows must be on CUDA")
        raise RuntimeError("kv cache and new rows must be on the same device")
    if not (k_cache.is_contiguous() and v_cache.is_contiguous()):
        raise RuntimeError("kv cache must be contiguous (it is written in place)")
    return shape, index


def _same_rows(k, v, Hkv: int, D: int):
    k, ks = _rows(k, Hkv, D)
    v, vs = _rows(v, Hkv, D)
    if k.shape[0] != v.shape[0] or k.dtype != v.dtype:
        raise RuntimeError("k and v rows must have the same count and dtype")
    if ks != vs:
        k, v = k.contiguous(), v.contiguous()
        ks = vs = Hkv * D
    return k, v, ks


def kv_scatter(k_cache, v_cache, slots, k, v, wrap: bool = False) -> None:
    """k_cache.view(-1, Hkv, D)[slots] = k.to(cache dtype); same for v.  wrap:
    negative slots count from the end (otherwise they are skipped)."""
    L = lib("KV scatter HIP kernel")
    (NB, BS, Hkv, D), index = _check_write(k_cache, v_cache, k, v)
    k, v, stride = _same_rows(k, v, Hkv, D)
    n = k.shape[0]
    if slots.numel() != n:
        raise RuntimeError(f"{slots.numel()} slots for {n} rows")
    slots = torch.as_tensor(slots).to(device=k_cache.device, dtype=torch.int64).contiguous()
    with _DeviceGuard(index):
        head = (k_cache.data_ptr(), v_cache.data_ptr(), dtype_code(k_cache.dtype), NB * BS, Hkv, D)
        rows = (slots.data_ptr(), n, k.data_ptr(), v.data_ptr(), dtype_code(k.dtype))
        if wrap:
            check(L.hs_kv_scatter_layers(*head, 1, 0, *rows, 0, D, stride, _stream_at(index)))
        else:
            check(L.hs_kv_scatter(*head, *rows, stride, _stream_at(index)))


def kv_scatter_layers(pool, slots, k, v) -> None:
    """pool[l, 0].view(-1, Hkv, D)[slots] = k[l].transpose(0, 1) for every layer of
    pool [L, 2, NB, BS, Hkv, D] and k, v [>= L, Hkv, T, D], in one launch;
    negative slots count from the end."""
    lib_ = lib("KV scatter HIP kernel")
    L, _, NB, BS, Hkv, D = pool.shape
    if L == 0:
        return
    (_, _, _, _), index = _check_write(pool[0, 0], pool[0, 1], k, v)
    T = slots.numel()
    for x in (k, v):
        if x.shape[0] < L:
            raise IndexError(f"index {x.shape[0]} is out of bounds for dimension 0 with size "
                             f"{x.shape[0]}")
        if tuple(x.shape[1:]) != (Hkv, T, D):
            raise RuntimeError(f"K/V must be [{L}, {Hkv}, {T}, {D}], got {tuple(x.shape)}")
    if k.dtype != v.dtype:
        raise RuntimeError("k and v rows must have the same count and dtype")
    if k.stride() != v.stride() or k.stride(3) != 1:
        k, v = k.contiguous(), v.contiguous()
    # a dim of one index has no stride of its own
    sl, sh, st = (k.stride(i) if k.shape[i] > 1 else n for i, n in
                  enumerate((Hkv * T * D, T * D, D)))
    slots = slots.to(device=pool.device, dtype=torch.int64).contiguous()
    with _DeviceGuard(index):
        check(lib_.hs_kv_scatter_layers(
            pool.data_ptr(), pool[0, 1].data_ptr(), dtype_code(pool.dtype), NB * BS, Hkv, D, L,
            2 * NB * BS * Hkv * D, slots.data_ptr(), T, k.data_ptr(), v.data_ptr(),
            dtype_code(k.dtype), sl, sh, st, _stream_at(index)))


def kv_append(k_cache, v_cache, block_tables, positions, k, v, seq_ids=None) -> None:
    """Row i -> slot block_tables[s][pos // BS] * BS + pos % BS of sequence
    s = seq_ids[i] (or i), pos = positions[i]; cast as kv_scatter."""
    L = lib("KV append HIP kernel")
    (NB, BS, Hkv, D), index = _check_write(k_cache, v_cache, k, v)
    k, v, stride = _same_rows(k, v, Hkv, D)
    n = k.shape[0]
    dev = k_cache.device
    bt = _int32_on(block_tables, dev)
    pos = _int32_on(positions, dev)
    if pos.numel() != n:
        raise RuntimeError(f"{pos.numel()} positions for {n} rows")
    sid = None if seq_ids is None else _int32_on(seq_ids, dev)
    if sid is not None and sid.numel() != n:
        raise RuntimeError(f"{sid.numel()} sequence ids for {n} rows")
    if sid is None and n > bt.shape[0]:
        raise RuntimeError("without seq_ids, row i uses table row i: more rows than tables")
    with _DeviceGuard(index):
        check(L.hs_kv_append(k_cache.data_ptr(), v_cache.data_ptr(), dtype_code(k_cache.dtype), NB,
                             BS, Hkv, D, bt.data_ptr(), bt.shape[0], bt.shape[1], pos.data_ptr(),
                             None if sid is None else sid.data_ptr(), n, k.data_ptr(),
                             v.data_ptr(), dtype_code(k.dtype), stride, _stream_at(index)))


def block_tables(packed_dev, B: int, width: int, out) -> None:
    """out[B, width] int32 from the packed [off[0..B], ids...] device buffer."""
    L = lib("block table HIP kernel")
    with _DeviceGuard(out.get_device()):
        check(L.hs_block_tables(packed_dev.data_ptr(), B, width, out.data_ptr(),
                                _stream_at(out.get_device())))
