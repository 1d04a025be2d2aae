// Merged q/k/v projection of one frame with RoPE + ring-slot K/V store as its epilogue (gfx950).
//
// One launch replaces the module's qkv_proj GEMM (src/patch_model.py:116-122) and everything the
// store kernel does after it (src/model/attn.py:105-110, src/model/kv_cache.py:138,147-151,192):
// the projected rows never travel through HBM as a [B, T, (H + 2 Hkv) Dh] tensor.  Meant for
// frames of a few hundred tokens, where the projection is a skinny GEMM (tokens x features x
// d_model = 256 x 6144 x 2048) whose cost is streaming the weight matrix once.
//
// One workgroup = 8 wavefronts = one CU computes a 64-token x 128-feature tile of x W^T, i.e. one
// head of 64 tokens (two heads when Dh = 64).  x and W tiles of 128 contraction elements travel
// HBM/L2 -> LDS by DMA (global_load_lds_dwordx4) into a ring of 3 slots, two ahead; rows are 256
// bytes, 16-byte chunks XOR-swizzled with (row & 15) on the global side of the DMA.  Wavefront w
// takes feature half (w & 1) and the contraction steps (w >> 1) and (w >> 1) + 4 of every slot:
// per slot 8 fragment reads (ds_read_b128) feed 8 v_mfma_f32_32x32x16 (A = W rows, B = x rows, so
// a lane owns one token and registers run along features).  The four partial sums of a tile go
// through LDS; every thread adds those of one 16-element item in a fixed order, rounds them to the
// element type as the GEMM's output tensor would be, and goes on exactly like a thread of the store
// kernel (same functions, same bits): RMS norm, rotation, value blend, tail / ring-slot rows,
// `written`.
//
// What runs outside the loop is a third of the time, so it waits for as little as it can: the position
// ids come by DMA ahead of the first slot, cos / sin values and the value residual of a thread's item
// are requested behind the second one, and the sums reach the items without a staging tile (256 x 6144
// x 2048, weights out of HBM: 18.96 -> 18.36 us; 11.2 of it is the tiles' intake alone).
//
// The grid is 1-D: workgroup id % 8 is the XCD, and the token tiles of one feature tile follow
// each other on one XCD, so a weight slab is fetched from HBM once and re-read from that L2; the CUs left without a
// tile fetch weights into it as well (fetch_ahead).
// Roofline: the weight matrix once (2 K N bytes) + x once; 2 T N K flops.
#include "attn_mma.h"
#include "rope_kv_store.h"
#include "device_state.h"
#include "we_kernels.h"

namespace we {

namespace {
constexpr int PM = 64;                       // tokens per tile
constexpr int PN = 128;                      // features per tile
constexpr int PK = 128;                      // contraction elements per ring slot
constexpr int P_ROW_B = PK * 2;              // bytes per tile row
constexpr int X_TILE_B = PM * P_ROW_B;       // 16 KB
constexpr int W_TILE_B = PN * P_ROW_B;       // 32 KB
constexpr int SLOT_B = X_TILE_B + W_TILE_B;  // 48 KB
constexpr int NSLOT = 3;
constexpr int IDS_OFF = NSLOT * SLOT_B;      // position ids: [wavefront][t, y, x][8 tokens], padded to 256 bytes each
constexpr int PROJ_LDS_B = IDS_OFF + 8 * 256;
static_assert(2 * 4 * 4 * (32 * 32 * 4) <= IDS_OFF, "the exchange area (4 shares of 8 fp32 blocks) reuses the ring");
}  // namespace

template <typename M, typename Tag>
__global__ void __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2)))
qkv_rope_store_kernel(ProjParams p) {
  touch_args<ProjParams>();
  typedef typename M::frag_t frag_t;
  typedef typename Tag::store_t st_t;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  const StoreParams& s = p.s;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, hh = lane >> 5;
  const int nh = wave & 1;     // feature half of the tile
  const int kg = wave >> 1;    // contraction group

  // ---- which tile ----
  const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
  const int mt_all = p.m_tiles * s.B;
  const int own = (int)((unsigned)(p.n_tiles + 7) / 8u) * mt_all;
  if (j >= own) {
    fetch_ahead<PN>(p.w, p.ws_n, p.n_tiles, p.K, xcd, j - own, p.helpers, wave, lane, lds0);
    return;
  }
  const int ng = j / mt_all;
  const int mi = j - ng * mt_all;
  const int nt = ng * 8 + xcd;
  if (nt >= p.n_tiles) return;
  const int b = mi / p.m_tiles;
  const int m0 = (mi - b * p.m_tiles) * PM;
  const int n0 = nt * PN;

  // ---- this thread's item of the epilogue: 16 features of one token ----
  const int e_row = tid >> 3;
  const int e_t = m0 + e_row;
  const bool e_live = e_t < s.T;
  const int e_tc = e_live ? e_t : s.T - 1;
  const int f0 = n0 + (tid & 7) * 16;
  const int q_feats = s.H * s.Dh, k_end = q_feats + s.Hkv * s.Dh;
  const int which = f0 < q_feats ? 0 : (f0 < k_end ? 1 : 2);
  const int f_in = f0 - (which == 0 ? 0 : (which == 1 ? q_feats : k_end));
  const int dh_shift = s.Dh == 128 ? 7 : 6;
  const int e_h = f_in >> dh_shift;
  const int e_chunk = (f_in & (s.Dh - 1)) >> 4;
  int64_t frame_t = s.t_pos[0];

  // ---- DMA plumbing: instruction q of a tile moves its rows 4q .. 4q+3 ----
  uint32_t xvo[2], wvo[4];
  {
    const int phys = lane & 15;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = 4 * (wave + 8 * i) + (lane >> 4);
      int tok = m0 + row;
      tok = tok < s.T ? tok : s.T - 1;  // rows past the frame repeat its last token; never stored
      xvo[i] = (uint32_t)tok * (uint32_t)(p.xs_t * 2) + (uint32_t)((phys ^ (row & 15)) << 4);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * (wave + 8 * i) + (lane >> 4);
      wvo[i] = (uint32_t)row * (uint32_t)(p.ws_n * 2) + (uint32_t)((phys ^ (row & 15)) << 4);
    }
  }
  const uint64_t xbase = uniform64((uint64_t)(uintptr_t)p.x + (uint64_t)((int64_t)b * p.xs_b * 2));
  const uint64_t wbase = uniform64((uint64_t)(uintptr_t)p.w + (uint64_t)((int64_t)n0 * p.ws_n * 2));
  const uint32_t wave_lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + wave * 1024));
  auto dma_slot = [&](int c, int slot) __attribute__((always_inline)) {
    const uint64_t kb = (uint64_t)c * P_ROW_B;
#pragma unroll
    for (int i = 0; i < 2; ++i) dma16(xbase + kb, xvo[i], wave_lds + slot * SLOT_B + i * 8 * 1024);
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16(wbase + kb, wvo[i], wave_lds + slot * SLOT_B + X_TILE_B + i * 8 * 1024);
  };
  constexpr int NDMA = 6;  // DMA instructions per wavefront and slot

  const int nc = p.K / PK;
  // Contraction chunks are taken in groups of G, and within a group token tile i starts at chunk
  // i mod G: the tiles that share a weight slab then ask for different lines at any one time, each
  // line comes from HBM at one tile's request and is an L2 hit for the others a slot or two later.
  // (A CU streams from HBM at less than half the rate it reads L2 at, so tiles asking for the same
  // lines together move the slab at a fraction of what they could.  Groups longer than 8 slots
  // keep more of the slab alive in L2 than pays.)
  const int G = mt_all >= 8 ? 8 : (mt_all >= 4 ? 4 : (mt_all >= 2 ? 2 : 1));
  const int rot = mi & (G - 1), ncg = nc & ~(G - 1);
  auto chunk = [&](int c) __attribute__((always_inline)) { return c < ncg ? (c & ~(G - 1)) | ((c + rot) & (G - 1)) : c; };
  // the position ids of this wavefront's 8 items' tokens: lane 16 a + 2 k + half takes 4 bytes of array a's
  // id of token k (the last lanes repeat lane 47)
  {
    const int l = lane < 48 ? lane : 47, a = l >> 4;
    int tok = m0 + wave * 8 + ((l & 15) >> 1);
    tok = tok < s.T ? tok : s.T - 1;
    const int64_t* ids = a == 0 ? s.t_pos : (a == 1 ? s.y_pos : s.x_pos);
    dma4(reinterpret_cast<const uint32_t*>(ids + b * s.pos_stride_b + tok) + (l & 1),
         (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + IDS_OFF + wave * 256)));
  }
  dma_slot(chunk(0), 0);
  if (nc > 1) dma_slot(chunk(1), 1);

  // ---- fragment read addresses: row l32 of a 32-row block, logical chunk 2 * step + hh ----
  uint32_t a_rd[2], b_rd[2];
#pragma unroll
  for (int h2 = 0; h2 < 2; ++h2) {
    const int phys = (2 * (kg + 4 * h2) + hh) ^ (l32 & 15);
    b_rd[h2] = (uint32_t)(l32 * P_ROW_B + phys * 16);
    a_rd[h2] = (uint32_t)(X_TILE_B + (nh * 64 + l32) * P_ROW_B + phys * 16);
  }

  f32x16_t acc[2][2];  // [feature block][token block]
#pragma unroll
  for (int nb = 0; nb < 2; ++nb)
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[nb][mb][i] = 0.f;

  // ---- what the item needs besides the projection (as it comes: a conversion here would wait for it) ----
  ItemSide<Tag, 16> side;
  u32x4_t res_raw[2];
  st_t lamb_raw;
  uint32_t guard;
  side.rotate = which != 2;
  const bool blend = which == 2 && s.v1 != nullptr;
  auto request_side = [&]() __attribute__((always_inline)) {
    if (side.rotate) {
      const int64_t* ids = reinterpret_cast<const int64_t*>(smem + IDS_OFF + wave * 256) + (e_row & 7);
      const int64_t at = rope_table_row(s, ids[0], ids[8], ids[16]) * (s.Dh >> 1);
      load_cos_sin<16>(s.cos_t + at, s.sin_t + at, e_chunk, side.c, side.s);
    }
    if (blend) {
      const u32x4_t* src = reinterpret_cast<const u32x4_t*>((const st_t*)s.v1 + b * s.v1s_b + e_h * s.v1s_h + e_tc * s.v1s_t + e_chunk * 16);
      res_raw[0] = src[0];
      res_raw[1] = src[1];
    }
    // (requested whether there are any or not - a value merged with another is waited for on the spot - and
    // by a lane's own load, for the same reason)
    int zero = 0;
    asm volatile("" : "+v"(zero));
    lamb_raw = *(reinterpret_cast<const st_t*>(blend ? s.v_lamb : p.w) + zero);
    guard = *((s.guard != nullptr ? s.guard : reinterpret_cast<const uint32_t*>(s.t_pos)) + zero);
  };

  // ---- main loop: one barrier per slot ----
  uint32_t slot_off = 0;   // byte offset of the slot being consumed
  int fill = 2 % NSLOT;    // slot the next DMA goes to
  auto consume = [&](int c, auto with_side) __attribute__((always_inline)) {
    if (c + 1 < nc) dma_wait<NDMA>(); else dma_wait<0>();  // this wavefront's part of slot c has landed
    // every wavefront's part has landed, and everybody is done with the slot refilled next
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // (in front of the next slot's request: the counter wait for the slot after this one covers it)
    if (decltype(with_side)::value) request_side();
    if (c + 2 < nc) dma_slot(chunk(c + 2), fill);
    fill = fill + 1 == NSLOT ? 0 : fill + 1;
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      const unsigned char* ab = smem + slot_off + a_rd[h2];
      const unsigned char* bb = smem + slot_off + b_rd[h2];
      const frag_t a0 = *reinterpret_cast<const frag_t*>(ab);
      const frag_t a1 = *reinterpret_cast<const frag_t*>(ab + 32 * P_ROW_B);
      const frag_t b0 = *reinterpret_cast<const frag_t*>(bb);
      const frag_t b1 = *reinterpret_cast<const frag_t*>(bb + 32 * P_ROW_B);
      acc[0][0] = M::mma(a0, b0, acc[0][0]);
      acc[0][1] = M::mma(a0, b1, acc[0][1]);
      acc[1][0] = M::mma(a1, b0, acc[1][0]);
      acc[1][1] = M::mma(a1, b1, acc[1][1]);
    }
    slot_off = slot_off + SLOT_B == (uint32_t)(NSLOT * SLOT_B) ? 0u : slot_off + SLOT_B;
  };
  int c0 = 0;
  if (nc > 1) consume(c0++, std::false_type());
  consume(c0++, std::true_type());
  for (int c = c0; c < nc; ++c) consume(c, std::false_type());

  // ---- the four contraction groups add their partial sums through LDS ----
  // Vector g (features 8 g + 4 hh + 0..3 of the lane's token) of lane l of block (nb, mb) of feature half nh,
  // group k, sits at ((((nh * 4 + k) * 4 + 2 * nb + mb) * 4 + g) * 64 + (l ^ 2 * item)) * 16, item being the
  // 16-feature item of the tile that it belongs to: a quarter wavefront then reads 16 bank groups below.
  __syncthreads();  // everybody is done with the ring
  f32x4_t* xch = reinterpret_cast<f32x4_t*>(smem);
#pragma unroll
  for (int nb = 0; nb < 2; ++nb)
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        xch[(((nh * 4 + kg) * 4 + 2 * nb + mb) * 4 + g) * 64 + (lane ^ (2 * (nh * 4 + nb * 2 + (g >> 1))))] =
            f32x4_t{acc[nb][mb][4 * g], acc[nb][mb][4 * g + 1], acc[nb][mb][4 * g + 2], acc[nb][mb][4 * g + 3]};
  __syncthreads();
  Chunk<Tag, 16> in;
  {
    const int item = tid & 7, blk = (item & 2) + (e_row >> 5);
    const f32x4_t* src = xch + ((item >> 2) * 16 + blk) * 256 + (item & 1) * 128;
#pragma unroll
    for (int v = 0; v < 4; ++v) {   // features 4 v .. 4 v + 3 of the item
      const int at = (v >> 1) * 64 + (((v & 1) * 32 + (e_row & 31)) ^ (2 * item));
      f32x4_t r = src[at];
#pragma unroll
      for (int k = 1; k < 4; ++k) r += src[k * 1024 + at];
#pragma unroll
      for (int e = 0; e < 4; ++e) in.e[4 * v + e] = Tag::from_f32(r[e]);
    }
  }

  // ---- epilogue: the store kernel's work on this thread's item ----
  // (the slot's arithmetic belongs here: the compiler puts it, and the wait for the frame index, in front of the first
  // slot's requests otherwise: 8 layers of 256 tokens 812 against 805 us)
  asm volatile("" : "+v"(frame_t));
  if (!e_live || (s.guard != nullptr && guard != 0u)) return;  // (refused position ids: nothing is written)
  if (blend) {
    reinterpret_cast<u32x4_t*>(&side.res.e)[0] = res_raw[0];
    reinterpret_cast<u32x4_t*>(&side.res.e)[1] = res_raw[1];
    side.lamb = Tag::to_f32(lamb_raw);
  }
  if (which == 0) {
    finish_q_chunk(s, b, e_h, e_t, e_chunk, in, side);
  } else {
    if (which == 2 && p.v_out != nullptr)
      store_chunk((st_t*)p.v_out + b * p.vo_b + e_h * p.vo_h + e_t * p.vo_t + e_chunk * 16, in);
    const SlotInfo si = ring_slot((int64_t)uniform64((uint64_t)frame_t), s.dilation, s.num_buckets);
    finish_kv_chunk(s, which, b, e_h, e_t, e_chunk, si, in, side);
  }
}

template <typename M, typename Tag>
static hipError_t launch_proj(ProjParams p, int cus, hipStream_t stream) {
  const unsigned groups = (unsigned)((p.n_tiles + 7) / 8), per_xcd = groups * (unsigned)(p.m_tiles * p.s.B);
  p.helpers = helpers_of((int)per_xcd, cus, p.K / PK, NSLOT - 1);
  const dim3 grid(8u * (per_xcd + (unsigned)p.helpers));
  hipLaunchKernelGGL((qkv_rope_store_kernel<M, Tag>), grid, dim3(512), PROJ_LDS_B, stream, p);
  return hipGetLastError();
}

hipError_t launch_qkv_rope_store(const ProjParams& p, int dtype, int cus, hipStream_t stream) {
  if (dtype == 0) return launch_proj<Bf16Mma, Bf16Tag>(p, cus, stream);
  return launch_proj<F16Mma, F16Tag>(p, cus, stream);
}

// The kernel's LDS ring exceeds the default per-launch limit: raised once per device by the
// library's set-up (device_state.hip).
hipError_t configure_qkv_rope_store() {
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&qkv_rope_store_kernel<Bf16Mma, Bf16Tag>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, PROJ_LDS_B);
  if (e == hipSuccess)
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&qkv_rope_store_kernel<F16Mma, F16Tag>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, PROJ_LDS_B);
  return e;
}

}  // namespace we
