// Writing new K/V rows into the paged cache: the step just before attention.
//
// Reference: the engine's `fk[slots] = k.to(pool dtype)` / `fv[slots] = ...`
// (heteroserve/model/torch_engine.py:239-240 for decode, :306-308 for a
// prefill chunk) and TorchBlockAllocator.write_kv (kv/torch_blocks.py:89-106,
// the same scatter per layer), with slots from slots_for (:68-73):
//   slot = table[pos // BS] * BS + pos % BS.
//
// One token row is Hkv * D elements.  A thread converts and moves 8
// elements (16 bytes of a 16-bit cache), so a D = 128 head row is one
// 16-lane group and a wave covers 4 heads; K and V, and the layers of a call
// that writes several, are the y index of one launch.  The source may be a
// strided view (rows of the fused QKV output, or a [layers, heads, tokens, D]
// array), so its strides are parameters.  Casts round like torch's
// `.to()`: fp32 -> bf16 and -> fp16 to nearest even, NaN to the canonical
// quiet NaN torch produces; equal types are copied bit for bit.
//
// A row whose slot is outside the cache (or whose table entry / position is
// invalid in the append form) is skipped: the kernel never writes outside
// the cache.  Rows must not share a slot (the engine never writes two tokens
// to one slot in a step; which of two duplicates survives is unspecified, as
// for torch's index_put).
#include "hs_kernels.h"

#include <algorithm>
#include <type_traits>

namespace hs {

namespace {

constexpr int kWriteThreads = 256;
constexpr int kMaxLayers = 32767;   // of one launch: K and V of each are the grid's y index

// ---- element codecs: 8 elements <-> 8 fp32 ------------------------------
template <typename T>
struct Codec;

template <>
struct Codec<float> {
  static constexpr int kBytes = 4;
  __device__ static void load8(const uint8_t* p, float* x) {
    const uint4 a = load16(p), b = load16(p + 16);
    x[0] = __uint_as_float(a.x); x[1] = __uint_as_float(a.y);
    x[2] = __uint_as_float(a.z); x[3] = __uint_as_float(a.w);
    x[4] = __uint_as_float(b.x); x[5] = __uint_as_float(b.y);
    x[6] = __uint_as_float(b.z); x[7] = __uint_as_float(b.w);
  }
  __device__ static void store8(uint8_t* p, const float* x) {
    *reinterpret_cast<uint4*>(p) = make_uint4(__float_as_uint(x[0]), __float_as_uint(x[1]),
                                              __float_as_uint(x[2]), __float_as_uint(x[3]));
    *reinterpret_cast<uint4*>(p + 16) = make_uint4(__float_as_uint(x[4]), __float_as_uint(x[5]),
                                                   __float_as_uint(x[6]), __float_as_uint(x[7]));
  }
  __device__ static float load1(const uint8_t* p) { return *reinterpret_cast<const float*>(p); }
  __device__ static void store1(uint8_t* p, float x) { *reinterpret_cast<float*>(p) = x; }
};

// fp32 -> bf16 bits, round to nearest even; NaN -> 0x7FC0 (c10::BFloat16).
__device__ inline uint32_t f32_to_bf16_bits(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0u;
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// fp32 -> fp16 bits, round to nearest even (v_cvt_f16_f32); NaN -> sign | 0x7E00
// as torch's CPU conversion gives.
__device__ inline uint32_t f32_to_f16_bits(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return ((u >> 16) & 0x8000u) | 0x7e00u;
  return __builtin_bit_cast(uint16_t, (_Float16)f);
}

template <>
struct Codec<Bf16> {
  static constexpr int kBytes = 2;
  __device__ static void load8(const uint8_t* p, float* x) {
    const uint4 a = load16(p);
    const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = __uint_as_float(w[i] << 16);
      x[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
  __device__ static void store8(uint8_t* p, const float* x) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = f32_to_bf16_bits(x[2 * i]) | (f32_to_bf16_bits(x[2 * i + 1]) << 16);
    *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
  }
  __device__ static float load1(const uint8_t* p) {
    return __uint_as_float((uint32_t)*reinterpret_cast<const uint16_t*>(p) << 16);
  }
  __device__ static void store1(uint8_t* p, float x) {
    *reinterpret_cast<uint16_t*>(p) = (uint16_t)f32_to_bf16_bits(x);
  }
};

template <>
struct Codec<_Float16> {
  static constexpr int kBytes = 2;
  __device__ static void load8(const uint8_t* p, float* x) {
    const uint4 a = load16(p);
    const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[i] & 0xffffu));
      x[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[i] >> 16));
    }
  }
  __device__ static void store8(uint8_t* p, const float* x) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = f32_to_f16_bits(x[2 * i]) | (f32_to_f16_bits(x[2 * i + 1]) << 16);
    *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
  }
  __device__ static float load1(const uint8_t* p) {
    return (float)*reinterpret_cast<const _Float16*>(p);
  }
  __device__ static void store1(uint8_t* p, float x) {
    *reinterpret_cast<uint16_t*>(p) = (uint16_t)f32_to_f16_bits(x);
  }
};

// Where row i goes: an explicit slot, or the slot of (sequence, position)
// through the block table.  Returns -1 for a row that must be skipped.
struct RowMap {
  const int64_t* slots;        // scatter form (null in the append form)
  const int32_t* bt;           // append form: [B, MB] tables
  const int32_t* positions;    //              [n] absolute positions
  const int32_t* seq_ids;      //              [n] row -> sequence, or null (row i = sequence i)
  int64_t num_slots;           // NB * BS
  int NB, BS, B, MB;           // B: table rows; a sequence index must be below it
  int wrap;                    // scatter form: negative slots count from the end

  __device__ int64_t slot(int64_t i) const {
    if (slots) {
      int64_t s = slots[i];
      if (wrap && s < 0) s += num_slots;
      return (s >= 0 && s < num_slots) ? s : -1;
    }
    const int64_t b = seq_ids ? seq_ids[i] : i;
    const int pos = positions[i];
    if (b < 0 || b >= B || pos < 0 || pos / BS >= MB) return -1;
    const int blk = bt[b * MB + pos / BS];
    if (blk < 0 || blk >= NB) return -1;
    return (int64_t)blk * BS + pos % BS;
  }
};

// What one launch writes: n rows of heads * dim elements into each of the
// layers' K and V caches (a row that is contiguous in the source counts as one
// head).
struct WriteArgs {
  uint8_t *k_cache, *v_cache;
  const uint8_t *k_src, *v_src;
  int64_t cache_layer, src_layer, src_head, src_row;   // bytes
  int64_t n;
  int heads, dim;
  RowMap map;
};

// Row i and element e of it, of the flat index g over rows of `per` units of
// kUnit elements: 32-bit division where the index fits, since a 64-bit one is
// most of this kernel's instructions.
template <int kUnit>
__device__ inline void split_index(int64_t g, int64_t total, uint32_t per, int64_t& i, int& e) {
  if (total <= 0xffffffffLL) {   // uniform
    const uint32_t r = (uint32_t)g / per;
    i = r;
    e = (int)((uint32_t)g - r * per) * kUnit;
  } else {
    i = g / per;
    e = (int)(g - i * per) * kUnit;
  }
}

// Element e of a row lies in head e / dim; its byte offset in the source row.
__device__ inline int64_t src_offset(const WriteArgs& a, int e, int elem_bytes) {
  if (a.heads == 1) return (int64_t)e * elem_bytes;
  const uint32_t h = (uint32_t)e / (uint32_t)a.dim;
  return h * a.src_head + (int64_t)(e - (int)h * a.dim) * elem_bytes;
}

// grid.x covers n rows x (row / 8) chunks; grid.y = 2 * layer + (0: K, 1: V).
template <typename S, typename C>
__global__ __launch_bounds__(kWriteThreads) void kv_write_kernel(WriteArgs a) {
  const uint32_t chunks = (uint32_t)(a.heads * a.dim / 8);
  const int64_t g = (int64_t)blockIdx.x * kWriteThreads + threadIdx.x;
  if (g >= a.n * chunks) return;
  int64_t i;
  int e;
  split_index<8>(g, a.n * chunks, chunks, i, e);
  const int64_t slot = a.map.slot(i);
  if (slot < 0) return;
  const int layer = blockIdx.y >> 1;
  const uint8_t* src = ((blockIdx.y & 1) ? a.v_src : a.k_src) + layer * a.src_layer +
                       i * a.src_row + src_offset(a, e, Codec<S>::kBytes);
  uint8_t* dst = ((blockIdx.y & 1) ? a.v_cache : a.k_cache) + layer * a.cache_layer +
                 (slot * ((int64_t)a.heads * a.dim) + e) * Codec<C>::kBytes;
  if constexpr (std::is_same<S, C>::value) {   // a bit copy (NaN payloads included)
#pragma unroll
    for (int b = 0; b < 8 * Codec<C>::kBytes; b += 16)
      *reinterpret_cast<uint4*>(dst + b) = load16(src + b);
  } else {
    float x[8];
    Codec<S>::load8(src, x);
    Codec<C>::store8(dst, x);
  }
}

// Any alignment: one element per thread.
template <typename S, typename C>
__global__ __launch_bounds__(kWriteThreads) void kv_write_scalar_kernel(WriteArgs a) {
  const uint32_t row = (uint32_t)(a.heads * a.dim);
  const int64_t g = (int64_t)blockIdx.x * kWriteThreads + threadIdx.x;
  if (g >= a.n * row) return;
  int64_t i;
  int e;
  split_index<1>(g, a.n * row, row, i, e);
  const int64_t slot = a.map.slot(i);
  if (slot < 0) return;
  const int layer = blockIdx.y >> 1;
  const uint8_t* src = ((blockIdx.y & 1) ? a.v_src : a.k_src) + layer * a.src_layer +
                       i * a.src_row + src_offset(a, e, Codec<S>::kBytes);
  uint8_t* dst = ((blockIdx.y & 1) ? a.v_cache : a.k_cache) + layer * a.cache_layer +
                 (slot * (int64_t)row + e) * Codec<C>::kBytes;
  if constexpr (std::is_same<S, C>::value) {   // a bit copy here too
    using Word = std::conditional_t<Codec<C>::kBytes == 4, uint32_t, uint16_t>;
    *reinterpret_cast<Word*>(dst) = *reinterpret_cast<const Word*>(src);
  } else {
    Codec<C>::store1(dst, Codec<S>::load1(src));
  }
}

template <typename S, typename C>
void launch_pair(const WriteArgs& a, int layers, bool vec, hipStream_t stream) {
  const int64_t work = a.n * ((int64_t)a.heads * a.dim / (vec ? 8 : 1));
  const dim3 grid((unsigned)((work + kWriteThreads - 1) / kWriteThreads), 2 * layers);
  if (vec)
    hipLaunchKernelGGL((kv_write_kernel<S, C>), grid, dim3(kWriteThreads), 0, stream, a);
  else
    hipLaunchKernelGGL((kv_write_scalar_kernel<S, C>), grid, dim3(kWriteThreads), 0, stream, a);
}

template <typename S>
int launch_src(int kv_dtype, const WriteArgs& a, int layers, bool vec, hipStream_t stream) {
  switch (kv_dtype) {
    case HS_DTYPE_F32: launch_pair<S, float>(a, layers, vec, stream); break;
    case HS_DTYPE_F16: launch_pair<S, _Float16>(a, layers, vec, stream); break;
    case HS_DTYPE_BF16: launch_pair<S, Bf16>(a, layers, vec, stream); break;
    default: return fail(HS_EINVAL, "unsupported KV cache dtype code " + std::to_string(kv_dtype));
  }
  return HS_OK;
}

int dtype_bytes(int code) { return code == HS_DTYPE_F32 ? 4 : 2; }

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Strides in elements.
int launch_kv_write(const KvWrite& w, const RowMap& map, hipStream_t stream) {
  if (w.n == 0) return HS_OK;
  const int64_t sb = dtype_bytes(w.src_dtype), cb = dtype_bytes(w.kv_dtype);
  const int64_t row_elems = (int64_t)w.Hkv * w.D;
  const int64_t row_b = sat_mul(w.src_row, sb), head_b = sat_mul(w.src_head, sb),
                layer_b = sat_mul(w.src_layer, sb), cache_b = sat_mul(w.cache_layer, cb);
  if (sat_add(sat_add(sat_mul(w.n, row_b), sat_mul(w.Hkv, head_b)), sat_mul(w.layers, layer_b)) ==
          INT64_MAX ||
      sat_add(sat_mul(map.num_slots, row_elems, cb), sat_mul(w.layers, cache_b)) == INT64_MAX)
    return fail(HS_EUNSUPPORTED, "KV write sizes too large for 64-bit offsets");
  const bool one_head = w.src_head == w.D || w.Hkv == 1;   // the row is contiguous in the source
  // the vector kernel needs 16-byte aligned 8-element groups on both sides
  const bool vec = (one_head ? row_elems : w.D) % 8 == 0 && aligned16(w.k_src) &&
                   aligned16(w.v_src) && aligned16(w.k_cache) && aligned16(w.v_cache) &&
                   row_b % 16 == 0 && (one_head || head_b % 16 == 0) && layer_b % 16 == 0 &&
                   cache_b % 16 == 0 && (row_elems * cb) % 16 == 0;
  const int64_t work = sat_mul(w.n, row_elems);
  if (row_elems > 0x7fffffffLL || ceil_div(work, kWriteThreads) > 0x7fffffffLL)
    return fail(HS_EUNSUPPORTED, "KV write too large for one launch");
  WriteArgs a;
  a.k_cache = static_cast<uint8_t*>(w.k_cache);
  a.v_cache = static_cast<uint8_t*>(w.v_cache);
  a.k_src = static_cast<const uint8_t*>(w.k_src);
  a.v_src = static_cast<const uint8_t*>(w.v_src);
  a.cache_layer = cache_b;
  a.src_layer = layer_b;
  a.src_head = head_b;
  a.src_row = row_b;
  a.n = w.n;
  a.heads = one_head ? 1 : w.Hkv;
  a.dim = one_head ? (int)row_elems : w.D;
  a.map = map;
  int rc = HS_OK;
  profile_begin(stream);
  for (int left = w.layers; left > 0 && rc == HS_OK; left -= kMaxLayers) {
    const int layers = std::min(left, kMaxLayers);
    switch (w.src_dtype) {
      case HS_DTYPE_F32: rc = launch_src<float>(w.kv_dtype, a, layers, vec, stream); break;
      case HS_DTYPE_F16: rc = launch_src<_Float16>(w.kv_dtype, a, layers, vec, stream); break;
      case HS_DTYPE_BF16: rc = launch_src<Bf16>(w.kv_dtype, a, layers, vec, stream); break;
      default: rc = fail(HS_EINVAL, "unsupported source dtype code " + std::to_string(w.src_dtype));
    }
    if (left <= kMaxLayers) break;   // (the products below fit where those layers exist)
    a.k_cache += kMaxLayers * cache_b;
    a.v_cache += kMaxLayers * cache_b;
    a.k_src += kMaxLayers * layer_b;
    a.v_src += kMaxLayers * layer_b;
  }
  profile_end(stream);
  if (rc != HS_OK) return rc;
  return check_launch("KV write");
}

}  // namespace

// out[b, j] = ids[off[b] + j] for j < off[b+1] - off[b] (capped at width), else
// -1; packed = [off[0..B], ids...] uploaded in one copy.
__global__ __launch_bounds__(kWriteThreads) void block_tables_kernel(const int32_t* packed, int B,
                                                                    int width, int32_t* out) {
  const int64_t g = (int64_t)blockIdx.x * kWriteThreads + threadIdx.x;
  if (g >= (int64_t)B * width) return;
  const int b = (int)(g / width);
  const int j = (int)(g - (int64_t)b * width);
  const int off = packed[b];
  const int len = packed[b + 1] - off;
  out[g] = j < len ? packed[B + 1 + off + j] : -1;
}

int launch_block_tables(const int32_t* packed, int B, int width, int32_t* out,
                        hipStream_t stream) {
  const int64_t work = (int64_t)B * width;   // both are int: no overflow
  if (work == 0) return HS_OK;
  if (ceil_div(work, kWriteThreads) > 0x7fffffffLL)
    return fail(HS_EUNSUPPORTED, "block table too large for one launch");
  hipLaunchKernelGGL(block_tables_kernel, dim3((unsigned)((work + kWriteThreads - 1) / kWriteThreads)),
                     dim3(kWriteThreads), 0, stream, packed, B, width, out);
  return check_launch("block table build");
}

int launch_kv_scatter(const KvWrite& w, int64_t num_slots, const int64_t* slots, bool wrap,
                      hipStream_t stream) {
  RowMap map{};
  map.slots = slots;
  map.num_slots = num_slots;
  map.wrap = wrap;
  return launch_kv_write(w, map, stream);
}

int launch_kv_append(const KvWrite& w, int NB, int BS, const int32_t* bt, int B, int MB,
                     const int32_t* positions, const int32_t* seq_ids, hipStream_t stream) {
  RowMap map{};
  map.bt = bt;
  map.positions = positions;
  map.seq_ids = seq_ids;
  map.num_slots = (int64_t)NB * BS;
  map.NB = NB;
  map.BS = BS;
  map.B = B;
  map.MB = MB;
  return launch_kv_write(w, map, stream);
}

}  // namespace hs
