// Causal chunked prefill in fp32 arithmetic on gfx950's fp32 matrix cores.
//
// Reference: paged_attention_prefill_kernel,
// heteroserve/model/paged_attn_prefill.py:72-157 (query s of a chunk sits at
// position ctx - S + s and attends to keys [0, that position]; rows at
// negative positions are zero).  This is hs_prefill*'s use_mfma = 0 path: any
// cache dtype, any block size, head dims 32 to 256, nothing rounded below
// fp32 anywhere.  A decode with grouped heads whose cache the split-operand
// kernel does not take (hs_decode_splitmm.hip) is the same thing with one query
// and its heads as rows; there a workgroup serves one partition of the keys
// and writes its state for the merge (hs_decode.hip).
//
// What bounds it.  The products run on v_mfma_f32_16x16x4_f32 (64 FLOPs a
// cycle and SIMD, 157 TFLOP/s over the device at 2.4 GHz), whose 32 cycles
// each leave room for everything else: the softmax, the LDS reads and the
// loads of a 16-key tile take a fraction of its products' time.  The VALU
// kernel (hs_decode.hip) gives every row and up to 8 of its heads a wave of their
// own, which reads all the keys of its row again and reduces every score over
// the lanes; it keeps the short tables (rows_prefill_pays) and some decodes
// (grouped_on_matrix_cores in hs_api.hip).
//
// Work decomposition.  A workgroup owns 16 * NT rows of one (sequence, KV
// head), a row being a (query, head of the group) pair with the queries
// outermost, so a short chunk of grouped heads still fills the tiles.  Its W
// waves take the 16-key tiles in turn and combine their softmax states
// through LDS at the end: the key split, and not a second query tile, is what
// gives a small chunk enough waves.  Per tile and wave:
//   S^T = K . Q^T    K staged in the wave's own LDS as fp32 (coalesced loads,
//                    one tile ahead), lane (row j = l % 16, group g = l / 16)
//                    reading dims g D/4 .. of key j; Q^T from LDS the same way
//   O^T += V^T . P^T V^T straight from global memory: lane (j, g) loads the
//                    D/16 values of key 4 g + i that are rows j of the
//                    output tiles, 16 lanes a whole head row, and the S^T
//                    accumulator is P^T's operand layout as it stands
// The waves share nothing in the loop, so it has no barriers.  Rows of one
// (sequence, KV head) are dealt heaviest first.
//
// Masked keys.  A score that a row does not see is -inf and its probability
// 0, but 0 times an infinite or NaN value is NaN in a matrix product, and a
// row must not see values past its own position.  Tiles in which some row
// masks some key therefore look at their V values, and one with a non-finite
// value adds its keys one by one, to the rows that see them.
#include <algorithm>

#include "hs_kernels.h"

namespace hs {

namespace {

typedef float float4x __attribute__((ext_vector_type(4)));

constexpr int kKeys = 16;            // keys of a tile (MFMA M), and rows of a row tile (MFMA N)
constexpr float kRowsSlack = 8.0f;   // lazy raise of the running max, log2 units

struct RowsArgs {
  RowAttnArgs a;
  int n_tiles;    // row tiles per (sequence, KV head) in the grid
  int bs_shift;   // log2(BS), or -1
  int reversed;   // the first workgroups, taken in reverse
};

// N 32-bit words of consecutive bytes, loaded at once.
template <int N>
struct Words {
  uint32_t w[N];
};

template <int N>
__device__ inline Words<N> load_words(const void* p) {
  typedef unsigned int vec __attribute__((ext_vector_type(N)));
  typedef vec vec_u __attribute__((aligned(4)));
  const vec x = *reinterpret_cast<const vec_u*>(p);
  Words<N> r;
#pragma unroll
  for (int i = 0; i < N; ++i) r.w[i] = x[i];
  return r;
}

template <>
__device__ inline Words<1> load_words<1>(const void* p) {
  return Words<1>{{*reinterpret_cast<const uint32_t*>(p)}};
}

// Element e of the words, widened to fp32 (exact).
template <typename T, int N>
__device__ inline float word_elem(const Words<N>& x, int e) {
  if constexpr (sizeof(T) == 4) {
    return __uint_as_float(x.w[e]);
  } else {
    float f[2];
    Elem<T>::pair(x.w[e >> 1], f);
    return f[e & 1];
  }
}

__device__ inline float max_over_groups(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ inline float sum_over_groups(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Orders a wave's LDS writes before its later LDS reads for the compiler (the
// hardware keeps a wave's LDS operations in order).
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Scheduling barrier mask: everything but matrix instructions may cross it.
constexpr int kAllButProducts = 0x3F6;

// acc plus the products of 4 dims or keys.
__device__ inline float4x product4(float a, float b, float4x acc = float4x{0.0f, 0.0f, 0.0f, 0.0f}) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
}

// Dot products over the lane's 4 N dims (16 N in all) of NT row tiles, row
// tiles `step` floats apart: chains of kChain matrix instructions (4 kChain
// products), added as a tree.  A row with few keys has the error of its scores,
// and in chains of 16 to 64 products it was up to 1.6 times that of the VALU
// kernel's chains of 4 (fp32 caches) or 8 (16-bit ones) and trees over the lanes:
// 2-norm against fp64, head dim 128, 17 keys, bf16, 1.79e-7, 1.12e-7 there, 1.07e-7
// in chains of 8.  These cost head dim 64, bf16, 4% of its speed, chains of 4 22%.
// kHold: the results of at most two groups of products at once, without which
// an fp32 cache at head dim 64 takes 162 VGPRs and half the waves (15% slower;
// with 16-bit caches, which fit either way, the barrier costs 3%).
template <int N, int NT, int kChain, bool kHold>
__device__ inline void dot_tree(const float* k, const float* q, int step, float4x (&s)[NT]) {
  if constexpr (N == 1) {
    const float4 kf = *reinterpret_cast<const float4*>(k);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float4 qf = *reinterpret_cast<const float4*>(q + t * step);
      s[t] = (product4(kf.x, qf.x) + product4(kf.y, qf.y)) +
             (product4(kf.z, qf.z) + product4(kf.w, qf.w));
      if constexpr (kHold) __builtin_amdgcn_sched_barrier(kAllButProducts);
    }
  } else if constexpr (N == kChain) {
    const float4 k0 = *reinterpret_cast<const float4*>(k);
    const float4 k1 = *reinterpret_cast<const float4*>(k + 4);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float4 q0 = *reinterpret_cast<const float4*>(q + t * step);
      const float4 q1 = *reinterpret_cast<const float4*>(q + t * step + 4);
      s[t] = (product4(k1.x, q1.x, product4(k0.x, q0.x)) +
              product4(k1.y, q1.y, product4(k0.y, q0.y))) +
             (product4(k1.z, q1.z, product4(k0.z, q0.z)) +
              product4(k1.w, q1.w, product4(k0.w, q0.w)));
    }
  } else {
    float4x r[NT];
    dot_tree<N / 2, NT, kChain, kHold>(k, q, step, s);
    dot_tree<N / 2, NT, kChain, kHold>(k + 2 * N, q + 2 * N, step, r);
#pragma unroll
    for (int t = 0; t < NT; ++t) s[t] += r[t];
  }
}

// The rows of row tile `tile` of (sequence b, KV head kvh) against the keys of
// partition p (decode; prefill has one partition, all keys); every thread of
// the workgroup calls it (it holds barriers).
template <typename T, int D, int NT, int W>
__device__ inline void rows_tile(const RowsArgs& ra, int b, int kvh, int tile, int p) {
  const RowAttnArgs& a = ra.a;
  constexpr int kRows = kKeys * NT;
  constexpr int kRow = D + 4;                    // floats of a staged row: 16-byte reads of 16
                                                 // rows fall on 16 different bank quads
  constexpr int kVec = Elem<T>::kVec;            // elements of a 16-byte load
  constexpr int kLpr = D / kVec;                 // K loads: lanes per token
  constexpr int kTpl = 64 / kLpr;                // tokens per load
  constexpr int kLi = kKeys / kTpl;              // loads per tile
  constexpr int kDT = D / 16;                    // output tiles, and V values per lane and key
  constexpr int kVE = kDT < kVec ? kDT : kVec;   // V values of one load
  constexpr int kNV = kDT / kVE;                 // V loads per key
  constexpr int kVW = kVE * (int)sizeof(T) / 4;  // words of one V load
  static_assert(kLi >= 1 && kTpl * kLi == kKeys && kVW >= 1, "head_dim");

  __shared__ __align__(16) float ks[W][kKeys][kRow];
  __shared__ __align__(16) float qs[kRows][kRow];
  __shared__ float wave_m[W][kRows], wave_l[W][kRows], row_l[kKeys];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);   // scalar: the tile loop is too
  const int j = lane & 15;
  const int g = lane >> 4;

  // ---- the rows of this workgroup (everything here is workgroup-uniform) ----
  const int G = a.H / a.Hkv;
  const int row0 = a.cu_q ? a.cu_q[b] : b * a.S;
  const int S_b = a.cu_q ? a.cu_q[b + 1] - row0 : a.S;
  const int n_rows = S_b * G;                     // the launcher keeps S * G within 31 bits
  const int r_first = tile * kRows;
  const int64_t cap = (int64_t)a.MB * a.BS;
  const int64_t base = (int64_t)a.ctx[b] - S_b;   // position of query 0
  auto query_of = [&](int r) { return G == 1 ? r : (int)((uint32_t)r / (uint32_t)G); };
  auto row_end = [&](int r) -> int {              // keys row r sees: [0, row_end)
    const int64_t e = base + query_of(r) + 1;
    return (int)max((int64_t)0, min(e, cap));
  };
  auto out_row = [&](int r) -> int64_t {          // element offset of row r in q and out
    const int s = query_of(r);
    return (((int64_t)row0 + s) * a.H + kvh * G + (r - s * G)) * D;
  };
  const int end = row_end(min(r_first + kRows, n_rows) - 1);   // rows see more keys as r grows
  const int seen_by_all = row_end(r_first);
  int lo = 0, hi = end, nparts = 1;
  if (a.P > 1 && end > 0 && !partition_range(a, end, p, lo, hi, nparts)) return;
  if (end <= 0) {
    if (p > 0) return;
    for (int i = tid; i < kRows * (D / 4); i += 64 * W) {
      const int r = r_first + i / (D / 4);
      if (r < n_rows)
        *reinterpret_cast<float4*>(a.out + out_row(r) + 4 * (i % (D / 4))) =
            make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    return;
  }

  // ---- the tiles of this wave: wv, wv + W, ... ------------------------------
  const int n_kt = (hi - lo + kKeys - 1) / kKeys;
  const int32_t* bt = a.bt + (int64_t)b * a.MB;
  const uint32_t tok_units = (uint32_t)(a.Hkv * (D * (int)sizeof(T) / 64));   // 64-byte units
  const char* kbase = static_cast<const char*>(a.k) + (int64_t)kvh * D * (int)sizeof(T) +
                      (lane % kLpr) * 16;
  const char* vbase = static_cast<const char*>(a.v) +
                      ((int64_t)kvh * D + kVE * j) * (int)sizeof(T);
  // Where key lo + 16 n + j lies in the cache, in 64-byte units (a key past the
  // last is read as the last).  The launcher keeps the cache within 32 bits of them.
  auto slot_of = [&](int n) -> uint32_t {
    const int t = min(lo + n * kKeys + j, hi - 1);
    const int blk = ra.bs_shift >= 0 ? t >> ra.bs_shift : t / a.BS;
    return ((uint32_t)safe_block(bt[blk], a.NB) * (uint32_t)a.BS + (uint32_t)(t - blk * a.BS)) *
           tok_units;
  };
  uint4 kr[kLi];
  Words<kVW> vr[4][kNV];
  auto load_k = [&](uint32_t slots) {
#pragma unroll
    for (int u = 0; u < kLi; ++u) {
      const uint32_t s = __shfl(slots, u * kTpl + lane / kLpr);
      kr[u] = load16(kbase + ((uint64_t)s << 6));
    }
  };
  auto load_v = [&](uint32_t slots) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t s = __shfl(slots, 4 * g + i);
      const char* p = vbase + ((uint64_t)s << 6);
#pragma unroll
      for (int u = 0; u < kNV; ++u)
        vr[i][u] = load_words<kVW>(p + u * 16 * kVE * (int)sizeof(T));
    }
  };

  uint32_t next_slots = 0;
  if (wv < n_kt) {
    const uint32_t slots = slot_of(wv);
    next_slots = slot_of(wv + W);
    load_k(slots);
    load_v(slots);
  }

  // ---- queries into LDS, scaled; rows past the last are zero ----------------
  for (int i = tid; i < kRows * (D / 4); i += 64 * W) {
    const int r = r_first + i / (D / 4);
    float4 x = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (r < n_rows) {
      x = *reinterpret_cast<const float4*>(a.q + out_row(r) + 4 * (i % (D / 4)));
      x = make_float4(x.x * a.qscale, x.y * a.qscale, x.z * a.qscale, x.w * a.qscale);
    }
    *reinterpret_cast<float4*>(&qs[i / (D / 4)][4 * (i % (D / 4))]) = x;
  }
  int lim[NT];   // keys that row j of each row tile sees
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int r = r_first + t * kKeys + j;
    lim[t] = r < n_rows ? min(row_end(r), hi) : 0;
  }
  __syncthreads();

  float m[NT], l[NT];
  float4x o[NT][kDT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    m[t] = kNegBig;
    l[t] = 0.0f;
#pragma unroll
    for (int d = 0; d < kDT; ++d) o[t][d] = float4x{0.0f, 0.0f, 0.0f, 0.0f};
  }

  for (int n = wv; n < n_kt; n += W) {
#pragma unroll
    for (int u = 0; u < kLi; ++u) {
      float f[kVec];
      Elem<T>::to_f32(kr[u], f);
      float* dst = &ks[wv][u * kTpl + lane / kLpr][(lane % kLpr) * kVec];
#pragma unroll
      for (int e = 0; e < kVec; e += 4)
        *reinterpret_cast<float4*>(dst + e) = make_float4(f[e], f[e + 1], f[e + 2], f[e + 3]);
    }
    wave_lds_fence();
    // The slots two tiles ahead are asked for before the loads of the next
    // tile, so that no later wait for them waits for those loads; and past
    // the last tile the loads go on (one token's rows again), because a load
    // under a condition makes the compiler wait for every load at the join.
    const uint32_t slots = next_slots;
    next_slots = slot_of(n + 2 * W);
    load_k(slots);

    // S^T: lane (j, g) gets keys 4 g + i of row j of each row tile.
    float4x s[NT];
    dot_tree<D / 16, NT, (sizeof(T) == 2 && D > 32 ? 2 : 1), (sizeof(T) == 4 && D <= 64)>(
        &ks[wv][j][g * (D / 4)], &qs[j][g * (D / 4)], kKeys * kRow, s);
    wave_lds_fence();

    const int t0 = lo + n * kKeys;
    const bool masked = t0 + kKeys > min(seen_by_all, hi);   // wave-uniform
    float p[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        x[i] = !masked || t0 + 4 * g + i < lim[t] ? s[t][i] : -INFINITY;
      const float mx = max_over_groups(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
      const float m_new = mx > m[t] + kRowsSlack ? mx : m[t];
      if (__builtin_amdgcn_ballot_w64(m_new != m[t]) != 0) {
        const float corr = fast_exp2(m[t] - m_new);
        l[t] *= corr;
#pragma unroll
        for (int d = 0; d < kDT; ++d)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[t][d][i] *= corr;
        m[t] = m_new;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[t][i] = fast_exp2(x[i] - m[t]);   // masked: exp2(-inf) = 0
        l[t] += p[t][i];
      }
    }

    bool one_by_one = false;
    if (masked) {
      float chk = 0.0f;   // 0 unless some V value is infinite or NaN
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int u = 0; u < kNV; ++u)
#pragma unroll
          for (int e = 0; e < kVE; ++e) chk = fmaf(word_elem<T>(vr[i][u], e), 0.0f, chk);
      one_by_one = __builtin_amdgcn_ballot_w64(chk != 0.0f) != 0;   // NaN != 0
    }
    if (!one_by_one) {
      // O^T += V^T . P^T: output tile (u, e) holds dims 16 kVE u + kVE row + e.
      // The 16 keys are summed by themselves first, as a tree over their
      // products of 4: a wave's sum over its keys then has one rounding per
      // tile and not one per key.
#pragma unroll
      for (int u = 0; u < kNV; ++u)
#pragma unroll
        for (int e = 0; e < kVE; ++e)
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            float4x x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
              x[i] = product4(word_elem<T>(vr[i][u], e), p[t][i]);
            o[t][u * kVE + e] += (x[0] + x[1]) + (x[2] + x[3]);
          }
    } else {
#pragma unroll 1
      for (int gk = 0; gk < 4; ++gk) {   // keys 4 gk + i, the other groups' values zero
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int u = 0; u < kNV; ++u)
#pragma unroll
            for (int e = 0; e < kVE; ++e) {
              const float vf = g == gk ? word_elem<T>(vr[i][u], e) : 0.0f;
#pragma unroll
              for (int t = 0; t < NT; ++t) {
                const float4x with = __builtin_amdgcn_mfma_f32_16x16x4f32(
                    vf, p[t][i], o[t][u * kVE + e], 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  if (t0 + 4 * gk + i < lim[t]) o[t][u * kVE + e][r] = with[r];
              }
              __builtin_amdgcn_sched_barrier(0);   // one product at a time: registers
            }
      }
    }
    load_v(slots);
  }

  // ---- combine the waves' states and write the rows -------------------------
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    l[t] = sum_over_groups(l[t]);
    if (g == 0) {
      wave_m[wv][t * kKeys + j] = m[t];
      wave_l[wv][t * kKeys + j] = l[t];
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    float mm = wave_m[0][t * kKeys + j];
#pragma unroll
    for (int w = 1; w < W; ++w) mm = fmaxf(mm, wave_m[w][t * kKeys + j]);
    float ll = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w)
      ll += wave_l[w][t * kKeys + j] * fast_exp2(wave_m[w][t * kKeys + j] - mm);
    const float sc = fast_exp2(m[t] - mm);
    // row j of the tile, this wave's part; its K rows are no longer needed
#pragma unroll
    for (int u = 0; u < kNV; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < kVE; ++e)
          ks[wv][j][16 * kVE * u + kVE * (4 * g + i) + e] = o[t][u * kVE + e][i] * sc;
    if (wv == 0 && g == 0) {
      row_l[j] = nparts > 1 || ll == 0.0f ? 1.0f : ll;   // a row without keys: 0 / 1
      const int r = r_first + t * kKeys + j;
      if (nparts > 1 && r < n_rows)   // decode: one query, row r is head r of the group
        reinterpret_cast<float2*>(a.part_ml)[((int64_t)b * a.H + kvh * G + r) * a.P + p] =
            make_float2(mm, ll);
    }
    __syncthreads();
    for (int i = tid; i < kKeys * (D / 4); i += 64 * W) {
      const int rr = i / (D / 4), c = 4 * (i % (D / 4));
      float4 x = *reinterpret_cast<const float4*>(&ks[0][rr][c]);
#pragma unroll
      for (int w = 1; w < W; ++w) {
        const float4 y = *reinterpret_cast<const float4*>(&ks[w][rr][c]);
        x = make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w);
      }
      const float f = row_l[rr];
      const int r = r_first + t * kKeys + rr;
      if (r < n_rows) {
        float* dst = nparts > 1
                         ? a.part_acc + (((int64_t)b * a.H + kvh * G + r) * a.P + p) * D + c
                         : a.out + out_row(r) + c;
        *reinterpret_cast<float4*>(dst) = make_float4(x.x / f, x.y / f, x.z / f, x.w / f);
      }
    }
    __syncthreads();
  }
}

template <typename T, int D, int NT, int W>
__global__ __launch_bounds__(64 * W) void rows_prefill_kernel(RowsArgs ra) {
  const RowAttnArgs& a = ra.a;
  const int n_pairs = a.B * a.Hkv;
  const int wg = (int)blockIdx.x < ra.reversed ? ra.reversed - 1 - (int)blockIdx.x : (int)blockIdx.x;
  const int pair = wg % n_pairs;
  const int b = pair / a.Hkv;
  const int kvh = pair - b * a.Hkv;
  const int rows = (a.cu_q ? a.cu_q[b + 1] - a.cu_q[b] : a.S) * (a.H / a.Hkv);
  const int tp = wg / n_pairs;
  const int p = tp % a.P;
  // heaviest first; the step is for a ragged sequence of more than a.S rows
  for (int tile = ra.n_tiles - 1 - tp / a.P; tile * kKeys * NT < rows; tile += ra.n_tiles)
    rows_tile<T, D, NT, W>(ra, b, kvh, tile, p);
}

// ---------------------------------------------------------------------------
// host launch
// ---------------------------------------------------------------------------

template <typename T, int D, int NT, int W>
void launch_shape(const RowAttnArgs& a, int64_t rows_per_pair, int cus, hipStream_t stream) {
  RowsArgs ra;
  ra.a = a;
  ra.n_tiles = (int)ceil_div(rows_per_pair, kKeys * NT);
  ra.bs_shift = (a.BS & (a.BS - 1)) == 0 ? __builtin_ctz((unsigned)a.BS) : -1;
  const int64_t n_wg = (int64_t)ra.n_tiles * a.B * a.Hkv * a.P;
  // More than one workgroup per CU but not two: the hardware deals the first
  // round out to all CUs and the second to the first of them again, so with
  // the first round reversed those hold its lightest workgroups (and not its
  // heaviest) beside the second's.  Only where two workgroups fit a CU
  // together (their registers, up to head dim 64).  GPT-2's 512-token chunk,
  // 384 workgroups: 26.4 -> 23.7 us.
  ra.reversed = D <= 64 && a.P == 1 && n_wg > cus && n_wg <= 2 * (int64_t)cus ? cus : 0;
  const dim3 grid((unsigned)n_wg), block(64 * W);
  hipLaunchKernelGGL((rows_prefill_kernel<T, D, NT, W>), grid, block, 0, stream, ra);
}

// The workgroup's shape: 8 waves of 16 rows, and 4 at head dim 256, where the
// registers hold one wave a SIMD.  Measured on MI355X (us, rows x waves 16 x 4 /
// 16 x 8 with an earlier order of sums, 5 to 20% cheaper than this one; one
// sequence):
//   12 heads, D 64, fp32, 512 rows on 512 tokens     27 / 24
//   the same, 16 rows on 1000                         20 / 17
//   32 / 8 heads, D 128, bf16, 256 rows on 512        38 / 39
//   32 / 8 heads, D 128, fp16, 9 rows on 3000         87 / 72
//   8 / 4 heads, D 256, fp32, 700 rows on 1000        142 / 170
//
// 32 rows halve what is read of K and V but hold twice the state, which at
// head dim 128 spills.  16 / 32 rows, us, 64 sequences unless said:
//   8 heads, D 32, bf16, 128 rows on 64 / on 1024     49 / 38, 175 / 136
//   the same, fp32, 128 rows on 64                    0.93 of the time with 16
//   12 heads, D 64, fp32, 32 rows on 512 / on 1024    77 / 72, 151 / 115
//   the same, bf16                                    0.90 to 0.94
//   16 sequences, 12 heads, D 64, fp32, 512 rows      136 / 153
//   3 sequences, 32 heads, D 128, fp32, 512 rows      157 / 309
// So 32 rows, where there are more than 16 and every CU gets two workgroups
// either way: with 16-bit caches at head dim 32; and with fp32 ones where every
// sequence has one row tile instead of two and long rows of K and V to read.
template <typename T, int D>
void launch_d(const RowAttnArgs& a, int64_t rows_per_pair, int cus, hipStream_t stream) {
  if constexpr (D == 256) {
    launch_shape<T, D, 1, 4>(a, rows_per_pair, cus, stream);
  } else {
    if constexpr (D == 32 || (D == 64 && sizeof(T) == 4)) {
      const int64_t wide = sat_mul(ceil_div(rows_per_pair, 2 * kKeys), a.B, a.Hkv, a.P);
      const bool pays = sizeof(T) == 2
                            ? D == 32
                            : !a.cu_q && rows_per_pair <= 2 * kKeys && (int64_t)a.MB * a.BS >= 1024;
      if (pays && rows_per_pair > kKeys && wide >= 2 * (int64_t)cus) {
        launch_shape<T, D, 2, 8>(a, rows_per_pair, cus, stream);
        return;
      }
    }
    launch_shape<T, D, 1, 8>(a, rows_per_pair, cus, stream);
  }
}

template <typename T>
void launch_t(const RowAttnArgs& a, int D, int64_t rows_per_pair, int cus, hipStream_t stream) {
  switch (D) {
    case 32: launch_d<T, 32>(a, rows_per_pair, cus, stream); break;
    case 64: launch_d<T, 64>(a, rows_per_pair, cus, stream); break;
    case 128: launch_d<T, 128>(a, rows_per_pair, cus, stream); break;
    default: launch_d<T, 256>(a, rows_per_pair, cus, stream); break;
  }
}

}  // namespace

bool rows_serves(const RowAttnArgs& a, int kv_dtype, int D) {
  const int elem = kv_dtype == HS_DTYPE_F32 ? 4 : 2;
  const int64_t tiles = sat_mul(ceil_div(sat_mul(a.S, a.H / a.Hkv), kKeys), a.B, a.Hkv, a.P);
  return tiles > 0 && tiles <= 0x7fffffffLL && sat_mul(a.S, a.H / a.Hkv) <= (1LL << 30) &&
         sat_mul(a.NB, a.BS, (int64_t)a.Hkv * (D * elem / 64)) <= 0xffffffffLL &&
         sat_mul(a.MB, a.BS) <= (1LL << 30);
}

// A workgroup here costs its set-up (8 us alone, 22 to 40 ns each in a full
// device) whatever its keys are; the VALU kernel costs each row its keys.  us,
// VALU / here, chunks of rows x keys of the table:
//   1 chunk,  32 heads of 8 groups, D 128, fp32    8 x 8 7.2 / 8.5, 8 x 24 11.6 / 8.6
//   1 chunk,  8 heads of 4 groups, D 256, bf16     8 x 8 6.7 / 12.6, 8 x 40 11.3 / 12.7
//   64 chunks, 32 heads, D 128, fp32               2 x 66 37 / 73, 2 x 258 128 / 124,
//                                                  8 x 8 24 / 48, 8 x 72 107 / 75
//   64 chunks, 32 heads of 8 groups, D 128, bf16   8 x 72 29 / 36, 8 x 264 76 / 62
// With one head a group the rows of a tile are what the VALU kernel repeats; with
// grouped heads a wave there serves up to 8 of them.  Ragged chunks have tiles
// that are empty here.  Over 22000 shapes (1 to 128 chunks of 1 to 128 rows, tables
// of 16 to 640 tokens) the rule is within 2% of the better kernel in the mean.
bool rows_prefill_pays(const RowAttnArgs& a, int kv_dtype, int D, int cus) {
  const bool half = kv_dtype != HS_DTYPE_F32;
  const int G = a.H / a.Hkv;
  const int64_t rows = (int64_t)a.S * G;
  int keys;   // up to here the VALU kernel
  const int64_t wgs = sat_mul(ceil_div(rows, kKeys), a.B, a.Hkv);
  if (wgs < 2 * (int64_t)cus) {
    keys = D == 256 ? (half ? 64 : 32) : G < 4 || wgs >= cus ? 32 : 16;
  } else if (G == 1) {
    keys = 640 / (int)std::min<int64_t>(rows, kKeys);
    if (D >= 128 && half) keys *= rows <= 4 ? 4 : 2;
    if (D == 32) keys /= 2;
  } else {
    keys = G > 4 ? (half ? 48 : 32) : D >= 128 ? (half ? 112 : 86) : 64;
    if (a.cu_q) keys = keys * 3 / 2;
  }
  return (int64_t)a.MB * a.BS > keys;
}

int launch_rows(const RowAttnArgs& a, int kv_dtype, int D, int cus, hipStream_t stream) {
  const int64_t rows_per_pair = (int64_t)a.S * (a.H / a.Hkv);
  profile_begin(stream);
  if (kv_dtype == HS_DTYPE_F32) launch_t<float>(a, D, rows_per_pair, cus, stream);
  else if (kv_dtype == HS_DTYPE_F16) launch_t<_Float16>(a, D, rows_per_pair, cus, stream);
  else launch_t<Bf16>(a, D, rows_per_pair, cus, stream);
  profile_end(stream);
  return check_launch(a.mma ? "paged attention" : "paged prefill");
}

}  // namespace hs
