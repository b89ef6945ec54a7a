/*
 * Entry points that libhsattn.so exports for the Python layer beside it
 * (heteroserve/_hip.py).  They are not part of the C ABI (include/hsattn.h),
 * whose conventions they share, and may change with the layer.
 */
#ifndef HS_PRIVATE_H
#define HS_PRIVATE_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/*
 * hs_kv_scatter over L layers in one launch, for sources of any layout:
 *   k_cache[l][slots[i], h] = cast(k_src[l, h, i])      (v the same)
 * where layer l of a cache starts cache_layer_stride elements after layer
 * l - 1 and the source's layers, heads and rows are src_layer_stride,
 * src_head_stride and src_row_stride elements apart (D elements of a head are
 * contiguous).  Negative slots count from the end of the cache, as in torch
 * indexing; slots outside [-num_slots, num_slots) are skipped; slots must not
 * repeat.
 * Replaces: TorchBlockAllocator.write_kv, heteroserve/kv/torch_blocks.py:89-106
 *           (a cast and an index_put per layer), and the index arithmetic
 *           before the scatter at heteroserve/model/torch_engine.py:306-308.
 */
int hs_kv_scatter_layers(void* k_cache, void* v_cache, int kv_dtype, int64_t num_slots, int Hkv,
                         int D, int L, int64_t cache_layer_stride, const int64_t* slots, int64_t n,
                         const void* k_src, const void* v_src, int src_dtype,
                         int64_t src_layer_stride, int64_t src_head_stride,
                         int64_t src_row_stride, void* stream);

/*
 * hs_kv_pack and hs_kv_unpack with at most HS_KV_HOST_IDS block ids in host
 * memory, which are read before the call returns and travel in the kernel's
 * arguments (of at most 4 KiB): nothing to upload, and a capture holds the ids.
 */
#define HS_KV_HOST_IDS 896
int hs_kv_pack_host_ids(const void* pool, int L, int NB, int64_t page_bytes,
                        const int64_t* host_ids, int n, void* out, void* stream);
int hs_kv_unpack_host_ids(void* pool, int L, int NB, int64_t page_bytes, const int64_t* host_ids,
                          int n, const void* in, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* HS_PRIVATE_H */
