// Per-item work of the fused RoPE + ring-slot K/V store kernel (rope_kv_store.hip, gfx950): one
// item = N = 16 or 8 consecutive input elements of one (tensor, batch, head, token) row.
#pragma once
#include <type_traits>

#include "we_common.h"
#include "we_kernels.h"
#include "../../include/we_attn.h"

namespace we {

struct Bf16Tag {
  typedef uint16_t store_t;
  static constexpr int kBytes = 2;
  __device__ static float to_f32(uint16_t b) { return bf16_bits_to_f32(b); }
  // v_cvt_pk_bf16_f32 (round-to-nearest-even) with c10::BFloat16's NaN (0x7FC0) patched in
  __device__ static uint16_t from_f32(float f) {
    const uint16_t r = __builtin_bit_cast(uint16_t, (__bf16)f);
    return f != f ? (uint16_t)0x7fc0 : r;
  }
};
struct F16Tag {
  typedef uint16_t store_t;
  static constexpr int kBytes = 2;
  __device__ static float to_f32(uint16_t b) { return f16_bits_to_f32(b); }
  __device__ static uint16_t from_f32(float f) { return f32_to_f16_bits(f); }
};
struct F32Tag {
  typedef float store_t;
  static constexpr int kBytes = 4;
  __device__ static float to_f32(float b) { return b; }
  __device__ static float from_f32(float f) { return f; }
};

// N elements of a row as raw storage.
template <typename Tag, int N>
struct Chunk {
  typedef typename Tag::store_t values_t __attribute__((ext_vector_type(N)));
  values_t e;
};

template <typename Tag, int N>
struct ChunkWords {   // what a chunk is loaded and stored as
  static constexpr int kBytes = N * Tag::kBytes;
  typedef typename std::conditional<kBytes % 16 == 0, uint4, uint2>::type word_t;
  static constexpr int kWords = kBytes / (int)sizeof(word_t);
};
template <typename Tag, int N>
__device__ __forceinline__ void load_chunk(Chunk<Tag, N>& c, const void* p) {
  typedef ChunkWords<Tag, N> W;
#pragma unroll
  for (int i = 0; i < W::kWords; ++i)
    reinterpret_cast<typename W::word_t*>(&c.e)[i] = reinterpret_cast<const typename W::word_t*>(p)[i];
}
template <typename Tag, int N>
__device__ __forceinline__ void store_chunk(void* p, const Chunk<Tag, N>& c) {
  typedef ChunkWords<Tag, N> W;
#pragma unroll
  for (int i = 0; i < W::kWords; ++i)
    reinterpret_cast<typename W::word_t*>(p)[i] = reinterpret_cast<const typename W::word_t*>(&c.e)[i];
}

// Weightless RMS norm of a row held N = 16 or 8 elements per lane by `cpr` consecutive lanes (a power of
// two, at most 64): x * rsqrt(mean(x^2) + eps) in fp32, rounded to the element type, as
// F.rms_norm on a low-precision tensor does (src/model/nn.py:55-56).  The squares are added in the order
// that torch 2.10's norm shows on this GPU - four neighbours one after the other, then halves onto halves:
// half-precision squares are exact in fp32, so the order is all that decides a sum's bits, and of the orders
// tried (groups of 1 to 16, neighbouring or strided, sequential or as trees) this one, with this reciprocal
// root, gives every bit of 2*10^5 rows of 64 and of 128.
template <typename Tag, int N>
__device__ __forceinline__ void rms_norm_chunk(Chunk<Tag, N>& c, int cpr, int Dh, float eps) {
  float x[N], part[N / 4];
#pragma unroll
  for (int j = 0; j < N / 4; ++j) {
    part[j] = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[4 * j + i] = Tag::to_f32(c.e[4 * j + i]);
      part[j] += x[4 * j + i] * x[4 * j + i];
    }
  }
  for (int m = cpr >> 1; m > 0; m >>= 1)
#pragma unroll
    for (int j = 0; j < N / 4; ++j) part[j] += __shfl_xor(part[j], m);
  const float sum = N == 16 ? (part[0] + part[N / 4 - 2]) + (part[1] + part[N / 4 - 1]) : part[0] + part[1];
  const float r = rsqrtf(sum / (float)Dh + eps);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    float y = x[i] * r;
    asm("" : "+v"(y));  // (fused with the conversion to f16 the product of a negative value and 0 loses its sign)
    c.e[i] = Tag::from_f32(y);
  }
}

// torch.lerp(v, v1, w) on N elements: fp32 arithmetic, the formula switches at |w| = 0.5
// (ATen/native/Lerp.h), result rounded to the element type.
template <typename Tag, int N>
__device__ __forceinline__ void lerp_chunk(Chunk<Tag, N>& v, const Chunk<Tag, N>& v1, float w) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float a = Tag::to_f32(v.e[i]), b = Tag::to_f32(v1.e[i]);
    const float d = b - a;
    v.e[i] = Tag::from_f32(fabsf(w) < 0.5f ? a + w * d : b - d * (1.f - w));
  }
}

// Row of the cos / sin tables for token t of batch element b (src/model/attn.py:33-36): the
// three position ids select one row of the flattened [frames, height, width] table.
__device__ __forceinline__ int64_t rope_table_row(const StoreParams& p, int64_t t_id, int64_t y_id, int64_t x_id) {
  const int64_t pos = t_id * p.grid_hw + y_id * p.grid_w + x_id;
  return pos < 0 ? 0 : (pos >= p.table_rows ? p.table_rows - 1 : pos);
}
__device__ __forceinline__ int64_t rope_table_row(const StoreParams& p, int b, int t) {
  const int64_t at = b * p.pos_stride_b + t;
  return rope_table_row(p, p.t_pos[at], p.y_pos[at], p.x_pos[at]);
}

// cos / sin of the N / 2 pairs of chunk `chunk` of a table row.
template <int N>
__device__ __forceinline__ void load_cos_sin(const float* cos_row, const float* sin_row, int chunk, float (&c)[N / 2],
                                             float (&s)[N / 2]) {
#pragma unroll
  for (int i = 0; i < N / 2; i += 4) {
    *reinterpret_cast<float4*>(c + i) = *reinterpret_cast<const float4*>(cos_row + chunk * (N / 2) + i);
    *reinterpret_cast<float4*>(s + i) = *reinterpret_cast<const float4*>(sin_row + chunk * (N / 2) + i);
  }
}

// Rotation of the N / 2 (even, odd) pairs of one N-element chunk: lo gets x0*cos - x1*sin (elements
// [N / 2 * chunk, N / 2 * (chunk + 1)) of the output row), hi gets x1*cos + x0*sin (the same range of the second
// half; the reference concatenates the rotated halves, attn.py:38-40).  Every product and sum is
// rounded separately, as eager fp32 tensor ops do: contraction into fused multiply-adds is
// switched off for this function (plain operators; the pragma does not govern inlined intrinsics).
template <typename Tag, int N>
__device__ __forceinline__ void rotate_values(const Chunk<Tag, N>& in, const float (&c)[N / 2], const float (&s)[N / 2],
                                              Chunk<Tag, N / 2>& lo, Chunk<Tag, N / 2>& hi) {
#pragma clang fp contract(off)
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    const float x0 = Tag::to_f32(in.e[2 * i]);
    const float x1 = Tag::to_f32(in.e[2 * i + 1]);
    const float p0 = x0 * c[i], p1 = x1 * s[i], p2 = x1 * c[i], p3 = x0 * s[i];
    const float y0 = p0 - p1;
    const float y1 = p2 + p3;
    lo.e[i] = Tag::from_f32(y0);
    hi.e[i] = Tag::from_f32(y1);
  }
}
// What an item needs besides its own N elements: the N / 2 cos / sin values of its pairs (rotated
// items) and the value residual's N elements with the blend weight (V items of a layer that has
// one).  Separate from the arithmetic so that a caller can request them long before it has the
// item's own values.  EXTRAS: whether a norm or a blend can be asked for at all.
template <typename Tag, int N>
struct ItemSide {
  float c[N / 2], s[N / 2];
  Chunk<Tag, N> res;
  float lamb;
  bool rotate;
};
template <typename Tag, int N, bool EXTRAS = true>
__device__ __forceinline__ void load_item_side(const StoreParams& p, int which, int b, int h, int t, int chunk,
                                               ItemSide<Tag, N>& sd) {
  typedef typename Tag::store_t st_t;
  sd.rotate = which != 2 && p.cos_t != nullptr;
  sd.lamb = 0.f;
  if (sd.rotate) {
    const int64_t pos = rope_table_row(p, b, t);
    const int half = p.Dh >> 1;
    load_cos_sin<N>(p.cos_t + pos * half, p.sin_t + pos * half, chunk, sd.c, sd.s);
  }
  if (EXTRAS && which == 2 && p.v1 != nullptr) {
    load_chunk(sd.res, (const st_t*)p.v1 + b * p.v1s_b + h * p.v1s_h + t * p.v1s_t + chunk * N);
    sd.lamb = Tag::to_f32(*reinterpret_cast<const st_t*>(p.v_lamb));
  }
}

// An item's two halves for the output row: rotated, or as they are.
template <typename Tag, int N>
__device__ __forceinline__ void item_halves(const Chunk<Tag, N>& in, const ItemSide<Tag, N>& sd, Chunk<Tag, N / 2>& lo, Chunk<Tag, N / 2>& hi) {
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    lo.e[i] = in.e[i];
    hi.e[i] = in.e[N / 2 + i];
  }
  if (sd.rotate) rotate_values(in, sd.c, sd.s, lo, hi);
}
// Into the row `to`: into its two halves, or next to each other (no branch: small launches wait for their code).
template <typename Tag, int N>
__device__ __forceinline__ void store_halves(typename Tag::store_t* to, int Dh, int chunk, bool rotated, const Chunk<Tag, N>& lo,
                                             const Chunk<Tag, N>& hi) {
  store_chunk(to + (rotated ? chunk * N : chunk * 2 * N), lo);
  store_chunk(to + (rotated ? (Dh >> 1) + chunk * N : chunk * 2 * N + N), hi);
}

// Destination rows of a K/V item: tail always, ring slot on an unfrozen persisting frame.
template <typename Tag, int N>
__device__ __forceinline__ void store_kv_rows(const StoreParams& p, int which, int b, int h, int t, int chunk,
                                              const SlotInfo& si, bool rotated, const Chunk<Tag, N>& lo,
                                              const Chunk<Tag, N>& hi) {
  typedef typename Tag::store_t st_t;
  const int64_t cap = p.L + p.T;
  const int plane = which - 1;
  st_t* plane_base = (st_t*)p.kv + (((int64_t)plane * p.B + b) * p.Hkv + h) * cap * p.Dh;
  const bool to_ring = (!p.frozen) && si.write_step;
  const int64_t tail_row = p.L + t;
  const int64_t ring_row = (int64_t)si.slot * p.T + t;
  store_halves(plane_base + tail_row * p.Dh, p.Dh, chunk, rotated, lo, hi);
  if (to_ring) store_halves(plane_base + ring_row * p.Dh, p.Dh, chunk, rotated, lo, hi);
  // written[dst] = True for the rows the unfrozen write went to (kv_cache.py:149-151).
  if (!p.frozen && which == 1 && b == 0 && h == 0 && chunk == 0) p.written[to_ring ? ring_row : tail_row] = 1;
}

// Everything after the load of a K (which = 1) or V (which = 2) item: K is normalised (optional)
// and rotated, V is blended with the value residual (optional); the tail row is written always
// and the ring-slot row when this is an unfrozen persisting frame; `written` is marked
// (src/model/attn.py:105-110, src/model/kv_cache.py:138,147-151).
template <typename Tag, int N, bool EXTRAS = true>
__device__ __forceinline__ void finish_kv_chunk(const StoreParams& p, int which, int b, int h, int t, int chunk,
                                                const SlotInfo& si, Chunk<Tag, N>& in, const ItemSide<Tag, N>& sd) {
  if (EXTRAS && which == 1 && p.norm_eps > 0.f) rms_norm_chunk(in, (int)((unsigned)p.Dh / (unsigned)N), p.Dh, p.norm_eps);
  if (EXTRAS && which == 2 && p.v1 != nullptr) lerp_chunk(in, sd.res, sd.lamb);
  Chunk<Tag, N / 2> lo, hi;
  item_halves(in, sd, lo, hi);
  store_kv_rows(p, which, b, h, t, chunk, si, sd.rotate, lo, hi);
}

// Everything after the load of a Q item: optional norm, rotation (or plain copy when there is no
// table), store into the contiguous [B, H, T, Dh] output.
template <typename Tag, int N, bool EXTRAS = true>
__device__ __forceinline__ void finish_q_chunk(const StoreParams& p, int b, int h, int t, int chunk,
                                               Chunk<Tag, N>& in, const ItemSide<Tag, N>& sd) {
  if (EXTRAS && p.norm_eps > 0.f) rms_norm_chunk(in, (int)((unsigned)p.Dh / (unsigned)N), p.Dh, p.norm_eps);
  Chunk<Tag, N / 2> lo, hi;
  item_halves(in, sd, lo, hi);
  store_halves((typename Tag::store_t*)p.q_out + (((int64_t)b * p.H + h) * p.T + t) * p.Dh, p.Dh, chunk, sd.rotate, lo, hi);
}

// Whether the position ids of token i (0 .. B * T) break one of the rules asked for: the frame index
// non-negative and the same over the frame (src/model/kv_cache.py:112-124), the table position
// inside the table (src/model/attn.py:25-30).  Free of branches, so that an unrolled loop has the
// ids of several tokens in flight (without table rules y_pos and x_pos stand for t_pos).
__device__ __forceinline__ bool pos_id_bad(const StoreParams& p, int i) {
  const int b = p.B == 1 ? 0 : (int)((unsigned)i / (unsigned)p.T);
  const int64_t row0 = b * p.pos_stride_b, at = row0 + (i - b * p.T);
  const int64_t t = p.t_pos[at], t0 = p.t_pos[row0], y = p.y_pos[at], x = p.x_pos[at];
  const int64_t row = t * p.grid_hw + y * p.grid_w + x;
  const bool frame = (t < 0) | (t != t0);
  const bool table = (x >= p.grid_w) | (y >= p.grid_h) | (row < 0) | (row >= p.table_rows);
  return (frame & ((p.check & WE_CHECK_FRAME) != 0)) | (table & ((p.check & WE_CHECK_TABLE) != 0));
}

// The verdict goes to the waiting host as soon as it is known: one relaxed word to host-coherent
// memory (no fence - the host reads nothing else of this kernel's).
__device__ __forceinline__ void report_verdict(const StoreParams& p, bool bad) {
  __hip_atomic_store(p.report, (p.ticket << 1) | (bad ? 1u : 0u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Whether the call's position ids were refused: uniform over the workgroup, which must reach both
// halves as a whole.  Without a verdict from the check kernel every workgroup looks at all ids itself
// (so that none of them writes a row of a refused frame) and the first one reports.  The first half
// requests the ids, ahead of everything else of the call (loads return in order, and the host waits
// for the report); the second has the verdict.
__device__ __forceinline__ bool own_ids_bad(const StoreParams& p) {
  if (p.guard != nullptr) return false;
  bool bad = false;
  for (int i = threadIdx.x; i < p.B * p.T; i += blockDim.x) bad = pos_id_bad(p, i) | bad;
  return bad;
}
__device__ __forceinline__ bool frame_refused(const StoreParams& p, bool bad) {
  if (p.guard != nullptr) return *p.guard != 0u;
  bad = __syncthreads_or(bad) != 0;
  if (threadIdx.x == 0 && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0) report_verdict(p, bad);
  return bad;
}

}  // namespace we
