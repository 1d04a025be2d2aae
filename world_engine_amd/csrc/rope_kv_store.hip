// Fused RoPE + ring-slot K/V store for one frame (gfx950).
//
// One launch replaces, for a single attention layer, the reference's RoPE on q and k
// (src/model/attn.py:33-40), torch.stack([k, v]) (src/model/kv_cache.py:192), the tail
// index_copy_ (:138), the unfrozen ring index_copy_ and the `written` update (:147-151).
// The ring slot is derived on the device from t_pos[0] (:126-131,:140).
//
// Work item: one thread per 16 consecutive input elements of one (tensor, b, head, token)
// row; a workgroup covers 256 consecutive (token, chunk) pairs of one head.  For a rotated row those are 8 (even, odd) pairs; the thread writes 8 contiguous
// elements into the first half of the output row and 8 into the second half (the reference
// concatenates the rotated halves, attn.py:40).  Threads are ordered chunk-fastest, then
// token, so a wavefront reads whole 256-byte input rows and writes contiguous cache rows.
// HBM-bound: bytes = elements read once + written once (twice for K/V on a persisting call).
#include "rope_kv_store.h"

namespace we {

// CHECK: the call's position ids are checked (a variant of its own: the check's code in front of the
// stores costs an unchecked call 0.5 us).
template <typename Tag, bool CHECK>
__global__ void __launch_bounds__(256) rope_kv_store_kernel(StoreParams p) {
  touch_args<StoreParams>();
  typedef typename Tag::store_t st_t;
  // grid: x = 256-thread slices of the (token, chunk) pairs of one row block, y = head among
  // [q heads | k heads | v heads], z = batch; everything below the block level is 32-bit math
  const int cpr = p.Dh >> 4;  // 16-element chunks per row
  const int hq = p.q ? p.H : 0;
  const int hkv = p.k ? p.Hkv : 0;  // rotation-only launches carry no k/v
  const int idx = blockIdx.x * 256 + threadIdx.x;
  const bool live = idx < p.T * cpr;
  const int t = p.cpr_shift >= 0 ? idx >> p.cpr_shift : idx / cpr;  // head dims are powers of two in practice
  const int chunk = idx - t * cpr;
  const int head_all = blockIdx.y;
  const int b = blockIdx.z;
  const int which = head_all < hq ? 0 : (head_all < hq + hkv ? 1 : 2);
  const int h = head_all - (which == 0 ? 0 : (which == 1 ? hq : hq + hkv));

  const bool bad = CHECK && own_ids_bad(p);
  const int64_t frame_t = p.t_pos[0];
  Chunk16<Tag> in;
  ItemSide<Tag> sd;
  if (live) {
    const st_t* src = which == 0   ? (const st_t*)p.q + b * p.qs_b + h * p.qs_h + t * p.qs_t
                      : which == 1 ? (const st_t*)p.k + b * p.ks_b + h * p.ks_h + t * p.ks_t
                                   : (const st_t*)p.v + b * p.vs_b + h * p.vs_h + t * p.vs_t;
    load16<Tag>(in, src + chunk * 16);
    load_item_side<Tag>(p, which, b, h, t, chunk, sd);
  }
  if (CHECK && frame_refused(p, bad)) return;
  if (!live) return;
  if (which == 0) {  // rotate (or copy when there is no table) into the contiguous output
    finish_q_chunk<Tag>(p, b, h, t, chunk, in, sd.rotate, sd.c, sd.s);
  } else {
    const SlotInfo si = ring_slot(frame_t, p.dilation, p.num_buckets);
    finish_kv_chunk<Tag>(p, which, b, h, t, chunk, si, in, sd.rotate, sd.c, sd.s, sd.res, sd.lamb);
  }
}

// The same with 8 elements a thread (EXTRAS: a norm or a blend too): bound by its trips to memory where the launch is small, and of fp32
// rows by the requests, each of which takes a quarter of every 64 bytes with 16 elements a thread (us, 16 / 8
// elements, persisting calls in a graph: fp32, 16 heads of 128, 256 tokens 5.94 / 4.42, 8 heads, 1024 tokens 9.50 / 7.28, 8 heads
// of 64, 64 tokens 3.02 / 2.45; bf16, 16 heads of 128, 256 tokens 3.53 / 3.39, 16 of 64, 64 tokens 2.74 / 2.53).
template <typename Tag, bool CHECK, bool EXTRAS>
__global__ void __launch_bounds__(256) rope_kv_store_8_kernel(StoreParams p) {
  touch_args<StoreParams>();
  typedef typename Tag::store_t st_t;
  typedef st_t four_t __attribute__((ext_vector_type(4)));
  typedef st_t eight_t __attribute__((ext_vector_type(8)));
  const int cpr = p.Dh >> 3;
  const int hq = p.q ? p.H : 0;
  const int hkv = p.k ? p.Hkv : 0;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  const bool live = idx < p.T * cpr;
  const int t = p.cpr_shift >= 0 ? idx >> (p.cpr_shift + 1) : idx / cpr;
  const int chunk = idx - t * cpr;
  const int b = blockIdx.z;
  const int which = (int)blockIdx.y < hq ? 0 : ((int)blockIdx.y < hq + hkv ? 1 : 2);
  const int h = (int)blockIdx.y - (which == 0 ? 0 : (which == 1 ? hq : hq + hkv));

  const bool bad = CHECK && own_ids_bad(p);
  const int64_t frame_t = p.t_pos[0];
  const bool rotate = which != 2 && p.cos_t != nullptr;
  const bool blend = EXTRAS && which == 2 && p.v1 != nullptr;
  eight_t in, res;
  float lamb = 0.f;
  f32x4_t c, s;
  if (live) {
    const st_t* src = which == 0   ? (const st_t*)p.q + b * p.qs_b + h * p.qs_h + t * p.qs_t
                      : which == 1 ? (const st_t*)p.k + b * p.ks_b + h * p.ks_h + t * p.ks_t
                                   : (const st_t*)p.v + b * p.vs_b + h * p.vs_h + t * p.vs_t;
#pragma unroll
    for (int i = 0; i < Tag::kBytes / 2; ++i)
      reinterpret_cast<uint4*>(&in)[i] = reinterpret_cast<const uint4*>(src + chunk * 8)[i];
    if (rotate) {
      const int64_t at = rope_table_row(p, b, t) * (p.Dh >> 1) + chunk * 4;
      c = *reinterpret_cast<const f32x4_t*>(p.cos_t + at);
      s = *reinterpret_cast<const f32x4_t*>(p.sin_t + at);
    }
    if (blend) {
      const st_t* from = (const st_t*)p.v1 + b * p.v1s_b + h * p.v1s_h + t * p.v1s_t + chunk * 8;
#pragma unroll
      for (int i = 0; i < Tag::kBytes / 2; ++i) reinterpret_cast<uint4*>(&res)[i] = reinterpret_cast<const uint4*>(from)[i];
      lamb = Tag::to_f32(*reinterpret_cast<const st_t*>(p.v_lamb));
    }
  }
  if (CHECK && frame_refused(p, bad)) return;
  if (!live) return;
  if (EXTRAS && which != 2 && p.norm_eps > 0.f) rms_norm_chunk<Tag, 8>(in, cpr, p.Dh, p.norm_eps);
  if (blend) lerp_chunk<Tag, 8>(in, res, lamb);
  four_t lo = __builtin_shufflevector(in, in, 0, 1, 2, 3), hi = __builtin_shufflevector(in, in, 4, 5, 6, 7);
  if (rotate) {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // (every product and sum rounded by itself: rotate_values)
      const float x0 = Tag::to_f32(in[2 * i]), x1 = Tag::to_f32(in[2 * i + 1]);
      const float p0 = x0 * c[i], p1 = x1 * s[i], p2 = x1 * c[i], p3 = x0 * s[i];
      const float y0 = p0 - p1, y1 = p2 + p3;
      lo[i] = Tag::from_f32(y0);
      hi[i] = Tag::from_f32(y1);
    }
  }
  // the two quarters of 4 elements: of the halves of the row, or neighbours
  const int at_lo = rotate ? chunk * 4 : chunk * 8, at_hi = rotate ? (p.Dh >> 1) + chunk * 4 : chunk * 8 + 4;
  auto put = [&](st_t* row) __attribute__((always_inline)) {
    *reinterpret_cast<four_t*>(row + at_lo) = lo;
    *reinterpret_cast<four_t*>(row + at_hi) = hi;
  };
  if (which == 0) {
    put((st_t*)p.q_out + (((int64_t)b * p.H + h) * p.T + t) * p.Dh);
    return;
  }
  const SlotInfo si = ring_slot(frame_t, p.dilation, p.num_buckets);
  st_t* plane = (st_t*)p.kv + (((int64_t)(which - 1) * p.B + b) * p.Hkv + h) * (p.L + p.T) * p.Dh;
  const bool to_ring = !p.frozen && si.write_step;
  const int64_t tail_row = p.L + t, ring_row = (int64_t)si.slot * p.T + t;
  put(plane + tail_row * p.Dh);
  if (to_ring) put(plane + ring_row * p.Dh);
  if (!p.frozen && which == 1 && b == 0 && h == 0 && chunk == 0) p.written[to_ring ? ring_row : tail_row] = 1;
}

// The check alone, for frames whose ids are too many for every workgroup of the store to look at.
__global__ void __launch_bounds__(1024) pos_check_kernel(StoreParams p, uint32_t* guard) {
  bool bad = false;
#pragma unroll 4
  for (int i = threadIdx.x; i < p.B * p.T; i += 1024) bad = pos_id_bad(p, i) | bad;
  bad = __syncthreads_or(bad) != 0;
  if (threadIdx.x == 0) {
    *guard = bad ? 1u : 0u;
    report_verdict(p, bad);
  }
}

hipError_t launch_pos_check(const StoreParams& p, uint32_t* guard, hipStream_t stream) {
  hipLaunchKernelGGL(pos_check_kernel, dim3(1), dim3(1024), 0, stream, p, guard);
  return hipGetLastError();
}

template <typename Tag>
static void launch_store(const StoreParams& p, hipStream_t stream) {
  const int heads = (p.q ? p.H : 0) + 2 * (p.k ? p.Hkv : 0);
  const auto grid = [&](int elements) {
    return dim3((unsigned)((p.T * (p.Dh / elements) + 255) / 256), (unsigned)heads, (unsigned)p.B);
  };
  // (16 elements of half precision are what one request takes in whole.  A frame's store, attention and second pass, 16 / 8
  // elements, by the launch's workgroups of 16: up to 720 of them 0.2 to 0.3 us less with 8, none of 60 shapes slower by more than its
  // runs differ; from 738 on as much lost as gained and up to 2.7 us more a pass: 810 34.0 / 35.1, 1008 24.9 / 25.6, 1276 45.3 /
  // 46.3, 1386 229 / 241, 3536 72.5 / 74.7 - twice the workgroups, which no longer find room at once.  fp32 calls 3 to 8 % less at
  // 405 to 1170.  With a norm or a blend the same 0.3 us: 34 module passes of 24 to 1188 1.009 times as fast, 0.99 at worst with
  // runs 1 % apart.  A rotation alone: 360 3.25 / 3.05, 456 3.35 / 3.48, 720 4.06 / 4.36; half the line also because a layer that
  // rotates q and k and then stores both should find one kernel: 24 heads, 588 tokens, four layers of five passes 735 us with 16
  // elements in all three launches, 742 with 8, 763 with 8 in one kind only.)
  const dim3 whole = grid(16);
  const int64_t most = p.k == nullptr ? 360 : 720;
  const bool large = Tag::kBytes == 2 && (int64_t)whole.x * whole.y * whole.z > most;
  const bool extras = p.norm_eps > 0.f || p.v1 != nullptr;
  const auto run = [&](auto kernel, int elements) {
    hipLaunchKernelGGL(kernel, grid(elements), dim3(256), 0, stream, p);
  };
  if (large) {
    p.check != 0 ? run(rope_kv_store_kernel<Tag, true>, 16) : run(rope_kv_store_kernel<Tag, false>, 16);
  } else if (extras) {
    p.check != 0 ? run(rope_kv_store_8_kernel<Tag, true, true>, 8) : run(rope_kv_store_8_kernel<Tag, false, true>, 8);
  } else {
    p.check != 0 ? run(rope_kv_store_8_kernel<Tag, true, false>, 8) : run(rope_kv_store_8_kernel<Tag, false, false>, 8);
  }
}

hipError_t launch_rope_kv_store(const StoreParams& p, int dtype, hipStream_t stream) {
  if (dtype == 0) launch_store<Bf16Tag>(p, stream);
  else if (dtype == 1) launch_store<F16Tag>(p, stream);
  else launch_store<F32Tag>(p, stream);
  return hipGetLastError();
}

}  // namespace we
