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
static void launch_store(const StoreParams& p, dim3 grid, hipStream_t stream) {
  if (p.check != 0) hipLaunchKernelGGL((rope_kv_store_kernel<Tag, true>), grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((rope_kv_store_kernel<Tag, false>), grid, dim3(256), 0, stream, p);
}

hipError_t launch_rope_kv_store(const StoreParams& p, int dtype, hipStream_t stream) {
  const int hq = p.q ? p.H : 0;
  const int hkv = p.k ? p.Hkv : 0;
  const dim3 grid((unsigned)((p.T * (p.Dh >> 4) + 255) / 256), (unsigned)(hq + 2 * hkv), (unsigned)p.B);
  if (dtype == 0) launch_store<Bf16Tag>(p, grid, stream);
  else if (dtype == 1) launch_store<F16Tag>(p, grid, stream);
  else launch_store<F32Tag>(p, grid, stream);
  return hipGetLastError();
}

}  // namespace we
