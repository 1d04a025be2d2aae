// Fused RoPE + ring-slot K/V store for one frame (gfx950).
//
// One launch replaces, for a single attention layer, the reference's RoPE on q and k
// (src/model/attn.py:33-40), torch.stack([k, v]) (src/model/kv_cache.py:192), the tail
// index_copy_ (:138), the unfrozen ring index_copy_ and the `written` update (:147-151).
// The ring slot is derived on the device from t_pos[0] (:126-131,:140).
//
// Work item: one thread per N = 16 or 8 consecutive input elements of one (tensor, b, head, token)
// row; a workgroup covers 256 consecutive (token, chunk) pairs of one head.  For a rotated row those are N / 2 (even, odd) pairs; the
// thread writes N / 2 contiguous elements into the first half of the output row and as many into the second half (the reference
// concatenates the rotated halves, attn.py:40).  Threads are ordered chunk-fastest, then
// token, so a wavefront reads whole input rows and writes contiguous cache rows.
// HBM-bound: bytes = elements read once + written once (twice for K/V on a persisting call); small launches by their
// trips to memory, and fp32 rows by the requests, each of which takes a quarter of every 64 bytes with 16 elements a thread (us, 16 / 8
// elements, persisting calls in a graph: fp32, 16 heads of 128, 256 tokens 5.94 / 4.42, 8 heads, 1024 tokens 9.50 / 7.28, 8 heads
// of 64, 64 tokens 3.02 / 2.45; bf16, 16 of 64, 64 tokens 2.74 / 2.53).
#include "rope_kv_store.h"

namespace we {

// CHECK: the call's position ids are checked (a variant of its own: the check's code in front of the
// stores costs an unchecked call 0.5 us).  EXTRAS: a norm or a blend may be asked for.
template <typename Tag, int N, bool CHECK, bool EXTRAS>
__global__ void __launch_bounds__(256) rope_kv_store_kernel(StoreParams p) {
  touch_args<StoreParams>();
  typedef typename Tag::store_t st_t;
  // grid: x = 256-thread slices of the (token, chunk) pairs of one row block, y = head among
  // [q heads | k heads | v heads], z = batch; everything below the block level is 32-bit math
  const int cpr = (int)((unsigned)p.Dh / (unsigned)N);  // chunks per row
  const int hq = p.q ? p.H : 0;
  const int hkv = p.k ? p.Hkv : 0;  // rotation-only launches carry no k/v
  const int idx = blockIdx.x * 256 + threadIdx.x;
  const bool live = idx < p.T * cpr;
  const int t = p.cpr_shift >= 0 ? idx >> (p.cpr_shift + (N == 8 ? 1 : 0)) : idx / cpr;  // head dims are powers of two in practice
  const int chunk = idx - t * cpr;
  const int head_all = blockIdx.y;
  const int b = blockIdx.z;
  const int which = head_all < hq ? 0 : (head_all < hq + hkv ? 1 : 2);
  const int h = head_all - (which == 0 ? 0 : (which == 1 ? hq : hq + hkv));

  const bool bad = CHECK && own_ids_bad(p);
  const int64_t frame_t = p.t_pos[0];
  Chunk<Tag, N> in;
  ItemSide<Tag, N> sd;
  if (live) {
    const st_t* src = which == 0   ? (const st_t*)p.q + b * p.qs_b + h * p.qs_h + t * p.qs_t
                      : which == 1 ? (const st_t*)p.k + b * p.ks_b + h * p.ks_h + t * p.ks_t
                                   : (const st_t*)p.v + b * p.vs_b + h * p.vs_h + t * p.vs_t;
    load_chunk(in, src + chunk * N);
    load_item_side<Tag, N, EXTRAS>(p, which, b, h, t, chunk, sd);
  }
  if (CHECK && frame_refused(p, bad)) return;
  if (!live) return;
  if (which == 0) {  // rotate (or copy when there is no table) into the contiguous output
    finish_q_chunk<Tag, N, EXTRAS>(p, b, h, t, chunk, in, sd);
  } else {
    const SlotInfo si = ring_slot(frame_t, p.dilation, p.num_buckets);
    finish_kv_chunk<Tag, N, EXTRAS>(p, which, b, h, t, chunk, si, in, sd);
  }
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
  // (16 elements of half precision are what one request takes in whole; 8 are twice the workgroups, which beyond some number no
  // longer find room at once.  A frame's store, attention and second pass, us with 16 / 8 elements, by the launch's workgroups
  // of 16: 384 24.57 / 24.37, 480 42.07 / 41.97, 700 35.64 / 35.75, 720 25.48 / 25.71, 810 30.13 / 29.98, 1008 32.5 / 33.2 and 35.8 /
  // 36.35, 1276 30.5 / 30.8, 1536 34.9 / 34.7, 2592 75.4 / 74.5; the store alone from 360 on as fast or faster with 16, 1008 5.68 /
  // 6.09.  The line is from 100 drawn passes with kernels of 16 that held more registers: 0.2 to 0.3 us less with 8 up to 720
  // workgroups, with a norm or a blend too, as much lost as gained beyond.  fp32 calls 3 to 8 % less at 405 to 1170.  A rotation
  // alone: 128 2.86 / 2.72, 360 3.37 / 3.33, 456 3.52 / 3.68, 512 3.56 / 3.78, 720 4.18 / 4.45; half the line also because a layer that
  // rotates q and k and then stores both should find one kernel: 24 heads, 588 tokens, four layers of five passes 735 us with 16
  // elements in all three launches, 742 with 8, 763 with 8 in one kind only.)
  const dim3 whole = grid(16);
  const int64_t most = p.k == nullptr ? 360 : 720;
  const bool extras = p.norm_eps > 0.f || p.v1 != nullptr;
  const auto run = [&](auto kernel, int elements) {
    hipLaunchKernelGGL(kernel, grid(elements), dim3(256), 0, stream, p);
  };
  if constexpr (Tag::kBytes == 2) {
    if ((int64_t)whole.x * whole.y * whole.z > most) {
      p.check != 0 ? run(rope_kv_store_kernel<Tag, 16, true, true>, 16) : run(rope_kv_store_kernel<Tag, 16, false, true>, 16);
      return;
    }
  }
  if (extras) p.check != 0 ? run(rope_kv_store_kernel<Tag, 8, true, true>, 8) : run(rope_kv_store_kernel<Tag, 8, false, true>, 8);
  else p.check != 0 ? run(rope_kv_store_kernel<Tag, 8, true, false>, 8) : run(rope_kv_store_kernel<Tag, 8, false, false>, 8);
}

hipError_t launch_rope_kv_store(const StoreParams& p, int dtype, hipStream_t stream) {
  if (dtype == 0) launch_store<Bf16Tag>(p, stream);
  else if (dtype == 1) launch_store<F16Tag>(p, stream);
  else launch_store<F32Tag>(p, stream);
  return hipGetLastError();
}

}  // namespace we
