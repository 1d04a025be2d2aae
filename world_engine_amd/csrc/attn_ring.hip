// Frame-block-causal flash attention over the KV ring buffer: 8-wavefront workgroups fed by
// LDS-DMA (gfx950, wave64, MFMA).
//
// Replaces the reference's make_block_mask + flex_attention pair (src/model/kv_cache.py:12-61,
// :141-144; src/model/attn.py:116).  A key row is visible iff it is in the tail [L, L+T) or in
// a ring slot s with written[s*T] set that is not the slot the current frame replaces on a
// persisting frame.  Visibility is per slot and identical for every batch element, head and
// query, so the kernel builds a short list of visible slots and walks those slots of the
// cache buffer in place, 64 keys at a time; no mask tensor and no gathered context exist.
//
// One workgroup = 8 wavefronts = one CU (2 wavefronts per SIMD, so one wavefront's vector work
// overlaps the other's matrix work).  Two shapes:
//   KSPLIT = 1: 256 queries; each wavefront owns 32 queries and handles both 32-key blocks of
//               every tile (large frames).
//   KSPLIT = 2: 128 queries; two wavefronts share a block of 32 queries, each taking one of the
//               two 32-key blocks of every tile, and merge their (reference, sum, O) through LDS
//               at the end.  Twice the parallelism per query without more split-context
//               partials (256-token frames, where the grid alone cannot fill the chip).
// K/V tiles travel HBM -> LDS directly (global_load_lds_dwordx4, no VGPR staging) into rings
// of 4 slots per operand, issued two to three tiles ahead.  LDS tiles are unpadded; bank
// conflicts are avoided by XOR-swizzling 16-byte chunks, applied on the global side of the DMA
// (lane i always lands at LDS offset 16*i) and undone in the fragment addresses.
// Per 32-key block and wavefront:
//   S^T = K Q^T        v_mfma_f32_32x32x16, A = K rows (ds_read_b128), B = Q in registers as
//                      loaded (no scaling, so nothing is rounded in front of the matrix core).
//   P = 2^((S-m) c)    one fused multiply-add per logit applies the softmax scale (c = scale *
//                      log2 e) and the running reference m, then v_exp_f32 + v_cvt_pk and the row sum
//                      (v_dot2c, or a small product); each lane owns one query column.
//   O^T += V^T P^T     A = V^T via ds_read_b64_tr_b16, B = P straight from registers.
// The three are software-pipelined across blocks (logits of block i+1 and product of block i-1
// run on the matrix cores while the VALU handles block i); LDS fragment reads are stated up to 15
// reads ahead of their MFMAs, also across steps and barriers, and the order is pinned with
// sched_barrier.  When the workgroup count leaves a partial last round of CUs, only that round's
// (batch, kv head) units are context-split (see the planner in attn_plan.h); split workgroups leave
// normalised partial outputs that a second kernel merges (attn_combine.hip).
//
// The grid is 3-D (8 * query tiles, heads with tiles of their own, rounds of 8 units): no division by
// run-time values is needed to find a workgroup's unit, and blockIdx.x % 8 is the XCD it runs on,
// so the workgroups that share one K/V stream share an L2.  Start-up code is kept short on purpose:
// a 256-token frame runs 8 tiles per workgroup and start-up is a third of the kernel.
//
// Frame lengths that are not a multiple of 64 (KEYS_PACKED, 64 tokens and more): the visible keys
// count through - slot after slot without padding - and a tile is 64 consecutive ones of them, in at
// most two pieces of memory: the rows behind a slot boundary that is not contiguous (the hidden slot,
// the step to the tail) get that gap added to their address.  Only the very last tile can be short;
// the split that owns it takes it first, so that clamped rows and masked keys stay in the prologue and
// in a peeled first step.  (Before, every slot's last tile was short and every step of the loop
// carried the masking and some 20 spilled registers; same plan, us: 24 heads of 128, 3600 tokens, 8
// slots 1395 -> 1338; 24 heads of 64 on 8, 720 tokens, f16 59.7 -> 51.2; 16 heads, 225 tokens, 16 slots
// 22.2 -> 20.1, in one part 55.1 -> 43.6.)  Frames below 64 tokens
// (KEYS_SLOT) take a tile per slot, every one of them equally short.
//
// Roofline: 4*T*N_vis*Dh flops and 4*N_vis*Dh bytes of K/V per (batch, kv head).
#include "attn_mma.h"
#include "device_state.h"
#include "ring_tiles.h"
#include "we_kernels.h"
#include "../../include/we_attn.h"

#include <type_traits>

namespace we {

template <int DH>
struct RingLds {
  static constexpr int CPR = DH / 8;          // 16-byte chunks per row
  static constexpr int ROW_B = DH * 2;        // bytes per K/V row
  static constexpr int TILE_B = BN * ROW_B;   // bytes per K or V tile
  static constexpr int SLOTS = 4;             // ring slots per operand over all wave groups
  static constexpr int V_OFF = SLOTS * TILE_B;
  static constexpr int MISC_OFF = 2 * SLOTS * TILE_B;
  static constexpr int kBytes = MISC_OFF + 8 * (WE_MAX_SLOTS + 64) * 4;  // + a slot-list strip per wavefront
};

// chunk swizzles: physical 16-byte chunk = logical chunk ^ swz(row)
template <int DH>
__device__ __forceinline__ int k_swz(int row) {
  return DH == 128 ? (row & 15) : ((row >> 1) & 7);
}
template <int DH>
__device__ __forceinline__ int v_swz(int row) {
  return DH == 128 ? ((row & 3) << 2) : (((row >> 1) & 1) << 2);
}

template <int V>
struct IntC {
  static constexpr int value = V;
};

// ---- LDS fragment reads ---------------------------------------------------------------------
// Left alone, the compiler keeps a single fragment read in flight ahead of the MFMA that needs
// it, which exposes the full LDS latency on every MFMA.  The hot loop therefore states its reads
// early in program order, several fragments ahead of their MFMAs, and pins that order with
// sched_barrier; the reads stay ordinary loads, so the compiler still places the (counted)
// lgkmcnt waits itself and knows the registers are in flight.
template <int OFF>
__device__ __forceinline__ u32x4_t lds_read128(const unsigned char* smem, uint32_t off) {
  return *reinterpret_cast<const u32x4_t*>(smem + off + OFF);
}
template <int OFF>
__device__ __forceinline__ u32x2_t lds_read_tr(const unsigned char* smem, uint32_t off) {
  const s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(smem + off + OFF));
  return __builtin_bit_cast(u32x2_t, v);
}

// The kernel's argument, read anew: what only the epilogue needs then takes no scalar registers through the
// tile loop.  Short frames and shared query tiles need more of those than there are (70 moved to vector lanes
// and back, 21 with this; 24 heads of 36 tokens, 64 slots: 18.1 -> 17.7 us).
template <typename P>
__device__ __forceinline__ const P& reread_args() {
  uint64_t at = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(at));
  return *(const P*)(const __attribute__((address_space(4))) P*)at;
}

// How tiles are laid over the visible keys (a separate instantiation each: the ragged ones' few extra
// instructions and registers are nothing the common case could spare).
constexpr int KEYS_TILED = 0;   // T % 64 == 0: whole tiles of one slot
constexpr int KEYS_PACKED = 1;  // T > 64: 64 consecutive visible keys, the last tile short
constexpr int KEYS_SLOT = 2;    // T < 64: one slot, short
constexpr int KEYS_SHARED = 3;  // as KEYS_PACKED, any T > 64, and grouped heads share query tiles
// CLOCKED: measurement library only - every workgroup reports its duration (p.clock_out).
template <typename M, int DH, int KSPLIT, int KEYS, bool CLOCKED>
__global__ void __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2)))
attn_ring_kernel(AttnParams p) {
  touch_args<AttnParams>();
  constexpr bool SHARED = KEYS == KEYS_SHARED, RUN = KEYS == KEYS_PACKED || SHARED;
  constexpr bool PARTS_F32 = std::is_same<M, F16Mma>::value;
  typedef typename M::frag_t frag_t;
  typedef RingLds<DH> L;
  constexpr int KS = DH / 16;               // contraction steps of K Q^T
  constexpr int DB = DH / 32;               // 32-row blocks of O^T
  constexpr int NV = 2 * DB;                // V^T fragments of one 32-key block
  constexpr int QW = 8 / KSPLIT;            // wavefronts with distinct query blocks
  constexpr int BM = 32 * QW;               // queries per workgroup
  constexpr int NST = 4;                    // ring slots per operand
  constexpr int CPR = L::CPR, ROW_B = L::ROW_B, TILE_B = L::TILE_B;
  constexpr int KB_B = 32 * ROW_B;          // bytes of one 32-key block of a tile
  constexpr int RPI = 1024 / ROW_B;         // rows moved by one DMA instruction
  constexpr int NDMA = TILE_B / 1024 / 8;   // DMA instructions per wavefront and tile operand

  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const uint32_t lds0 =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, hh = lane >> 5;
  // shader-clock and constant-rate (100 MHz) counters at the workgroup's start
  const uint64_t clk0 = CLOCKED ? (uint64_t)__builtin_readcyclecounter() : 0;
  const uint64_t wall0 = CLOCKED ? (uint64_t)__builtin_amdgcn_s_memrealtime() : 0;
  // CLOCKED: thread 0 also leaves the time (100 MHz ticks since the start) at which it passed each
  // stage, at [kClockSlots * workgroup + 2 + stage]
  const uint64_t wg_id = blockIdx.x + (uint64_t)gridDim.x * (blockIdx.y + (uint64_t)gridDim.y * blockIdx.z);
  auto stamp = [&](int stage) __attribute__((always_inline)) {
    if (CLOCKED && tid == 0)
      p.clock_out[kClockSlots * wg_id + 2 + stage] = (uint64_t)__builtin_amdgcn_s_memrealtime() - wall0;
  };
  const int qb = wave % QW;   // query block of this wavefront
  const int hb = wave / QW;   // key block of every tile it handles when KSPLIT == 2 (else 0)

  // ---- frame index and slot flags: they need nothing but the kernel arguments ----
  const int64_t frame_t = p.t_pos[0];
  uint8_t flag = lane < p.n_slots ? p.written[(int64_t)lane * p.T] : (uint8_t)0;

  // ---- which (batch, head, query tile, split) this workgroup owns ----
  // The grid is (8 * query tiles, heads with tiles of their own, rounds): workgroups are dispatched
  // to XCDs round-robin in linear order, so XCD = blockIdx.x % 8, and the workgroups that share
  // one K/V stream (the x * y of one round) all land on the same XCD and its L2.
  const int xcd = blockIdx.x & 7, qtile = blockIdx.x >> 3, hq_in = blockIdx.y;
  const int us_raw = blockIdx.z * 8 + xcd;
  // a workgroup past the end computes the addresses of the last one and leaves further down, so
  // that the requests above and below do not wait behind a branch
  const int us = us_raw < p.unit_splits ? us_raw : p.unit_splits - 1;
  // leading units run unsplit; the rest are cut into n_splits context parts each
  int unit, split, nsp;
  if (us < p.units_whole) {
    unit = us; split = 0; nsp = 1;
  } else {
    const int r = us - p.units_whole;
    unit = p.units_whole + r / p.n_splits; split = r % p.n_splits; nsp = p.n_splits;
  }
  const int b = unit / p.Hkv, hkv = unit - b * p.Hkv;
  // Query rows of this workgroup's heads.  Where grouped heads share tiles the rows count
  // through all of them: row r is token r % T of head r / T of the group.  Rows past the last token are
  // computed and not stored.
  const int row0 = qtile * BM;
  const int h0 = hkv * p.group + hq_in;

  // ---- raw Q fragments ----
  // A lane's fragment loads touch 32 rows x 32 bytes each: 512 small requests per wavefront, which
  // the 256-query shape (long loops) does not notice and the 128-query shape does: the tile DMAs
  // below cannot go out before Q is back.  There the workgroup's 128 x Dh tile comes by DMA - 16
  // lanes per row, whole cache lines - into the V ring's slots 2 and 3, laid out and swizzled like
  // two K tiles, while the slot flags are on their way; the fragments are read from there once the
  // first K tile is in (the V stream's first request for those slots goes out after the next barrier).
  constexpr int Q_OFF = L::V_OFF + 2 * TILE_B;
  const bool q_dma = KSPLIT == 2 && p.q_dma != 0;
  frag_t qf[KS];
  const unsigned qrow = (unsigned)(row0 + qb * 32 + l32);
  if (!q_dma) {
    int hq = SHARED ? (int)(qrow / (unsigned)p.T) : 0, qr = (int)qrow - hq * p.T;
    if (SHARED && hq >= p.group) { hq = p.group - 1; qr = p.T - 1; }
    qr = qr < p.T ? qr : p.T - 1;
    const uint16_t* src = reinterpret_cast<const uint16_t*>(p.q) + b * p.qs_b + (h0 + hq) * p.qs_h + (int64_t)qr * p.qs_t + hh * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const frag_t*>(src + ks * 16);
  }
  if (us_raw >= p.unit_splits) return;
  if (KSPLIT == 2 && q_dma) {
    const int limit = SHARED ? p.group * p.T : p.T;
    const uint64_t qplane = uniform64((uint64_t)(uintptr_t)p.q + (uint64_t)(((int64_t)b * p.qs_b + (int64_t)h0 * p.qs_h) * 2));
    const uint32_t q_lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + Q_OFF + wave * 1024));
#pragma unroll
    for (int i = 0; i < 2 * NDMA; ++i) {
      const int row = (wave + i * 8) * RPI + lane / CPR;   // row of the 128-query tile
      int qr = row0 + row;
      qr = qr < limit ? qr : limit - 1;
      dma16(qplane, (uint32_t)qr * (uint32_t)(p.qs_t * 2) + (uint32_t)(((lane % CPR) ^ k_swz<DH>(row)) << 4), q_lds + i * 8 * 1024);
    }
  }

  // ---- list of visible slots (the tail is pseudo-slot n_slots) ----
  // Every wavefront builds it for itself (no barrier, no serial section) in a private strip of
  // LDS: lane i of round k looks at slot 64*k + i.
  int* vis = reinterpret_cast<int*>(smem + L::MISC_OFF) + wave * (WE_MAX_SLOTS + 64);
  int nvis = 0;
  {
    const SlotInfo si = ring_slot(frame_t, p.dilation, p.num_buckets);
    for (int base = 0; base < p.n_slots; base += 64) {
      const int sl = base + lane;
      const bool f = flag != 0 && !(si.write_step && sl == si.slot);
      if (base + 64 < p.n_slots) flag = sl + 64 < p.n_slots ? p.written[(int64_t)(sl + 64) * p.T] : (uint8_t)0;
      const unsigned long long m = __ballot(f);
      if (f) vis[nvis + __popcll(m & ((1ull << lane) - 1ull))] = sl;
      nvis += __popcll(m);
    }
    if (lane == 0) vis[nvis] = p.n_slots;
    ++nvis;
  }
  stamp(0);  // slot list built
  // tiles of the visible keys; last_keys: keys of the last one
  const int tps = KEYS == KEYS_TILED ? p.T / BN : 1;
  const int nt = RUN ? (nvis * p.T + BN - 1) / BN : nvis * tps;
  const int last_keys = nvis * p.T - (nt - 1) * BN;  // (RUN)
  int t_begin = 0, t_end = nt;
  if (nsp > 1) {  // nt <= 257 * T / 64 and nsp <= 64: the products fit 32 bits
    t_begin = (int)((unsigned)split * (unsigned)nt / (unsigned)nsp);
    t_end = (int)((unsigned)(split + 1) * (unsigned)nt / (unsigned)nsp);
  }
  const int ntile = t_end - t_begin;
  // this split owns a short last tile (and takes it first)
  const bool shorted = RUN && t_end == nt && last_keys < BN && ntile > 0;

  const int64_t cap = p.L + p.T;
  const uint64_t kbase = (uint64_t)(uintptr_t)p.kv + (uint64_t)(((int64_t)b * p.Hkv + hkv) * cap) * ROW_B;
  const uint64_t vbase = kbase + (uint64_t)((int64_t)p.B * p.Hkv * cap) * ROW_B;

  // ---- DMA plumbing ----
  // Instruction i of this wavefront moves rows [q*RPI, (q+1)*RPI) of a tile, q = wave + 8*i.
  uint32_t kvoff[NDMA], vvoff[NDMA];
#pragma unroll
  for (int i = 0; i < NDMA; ++i) {
    const int row = (wave + i * 8) * RPI + lane / CPR;
    const int phys = lane % CPR;
    // (a short slot must not read rows of the next one: its missing rows repeat its last)
    const int src = KEYS == KEYS_SLOT && row >= p.T ? p.T - 1 : row;
    kvoff[i] = src * ROW_B + ((phys ^ k_swz<DH>(row)) << 4);
    vvoff[i] = src * ROW_B + ((phys ^ v_swz<DH>(row)) << 4);
  }
  // The split's visible tiles, 64 at a time: lane i of toff holds the byte offset, inside the
  // (batch, kv head) plane, of tile 64*k + i of the split (fits 32 bits, checked on the host).
  // RUN: its low 7 bits (row starts are multiples of 128 bytes) hold the tile row at which
  // the next slot begins (64: none does), tgap the bytes between the two slots.  The tile loop then
  // needs one v_readlane (two) per tile instead of walking slots and tiles with scalar code.
  // The workgroups that share this K/V stream (query tiles x grouped query heads) take the tiles
  // in groups of rot_g = 2 or 4, member m starting at tile m of every group: they then ask for
  // different lines at any one time, each line comes from HBM at one member's request and is an
  // L2 hit for the others a tile later.  (Asking together, every member waits the whole way to
  // HBM for every tile; a model's layers each bring their own ring, so K/V is never cache-warm:
  // 24 rings of 4096 tokens, 256-token frames: 757 -> 719 us per frame-step.)  The order of the
  // keys does not matter to a softmax.
  int rot_g = 1;
  while (rot_g * 2 <= p.members && rot_g < 4) rot_g *= 2;
  const SplitTiles split_tiles = {(unsigned)t_begin, (unsigned)t_end, shorted, (unsigned)rot_g,
                                  (unsigned)(qtile * p.q_heads + hq_in) & (unsigned)(rot_g - 1)};
  uint32_t toff = 0, tgap = 0;
  struct TileAt { uint32_t off, gap; };
  auto load_offsets = [&](int first) __attribute__((always_inline)) {
    const unsigned ti = split_tiles.at((unsigned)(first + lane));
    if (RUN) {
      const unsigned v0 = ti * BN, T = (unsigned)p.T;
      const unsigned sidx = v0 / T, in = v0 - sidx * T;
      const unsigned brk = T - in < BN ? T - in : BN;
      const int sl = vis[sidx];
      const int nx = brk < BN && (int)sidx + 1 < nvis ? vis[sidx + 1] : sl + 1;
      toff = ((uint32_t)sl * T + in) * (uint32_t)ROW_B | brk;
      tgap = (uint32_t)(nx - sl - 1) * T * (uint32_t)ROW_B;
    } else {
      const unsigned sidx = ti / (unsigned)tps;
      const unsigned sub = ti - sidx * (unsigned)tps;
      toff = ((uint32_t)vis[sidx] * (uint32_t)p.T + sub * BN) * (uint32_t)ROW_B;
    }
  };
  int kc = 0;  // tile the K stream requests next; it stays on the last one
  auto next_off = [&]() __attribute__((always_inline)) {
    if ((kc & 63) == 0) load_offsets(kc);
    TileAt t;
    t.off = (uint32_t)__builtin_amdgcn_readlane((int)toff, kc & 63);
    t.gap = RUN ? (uint32_t)__builtin_amdgcn_readlane((int)tgap, kc & 63) : 0u;
    kc = split_tiles.next(kc);
    return t;
  };
  const uint64_t kplane = uniform64(kbase), vplane = uniform64(vbase);
  const uint32_t wave_lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + wave * 1024));
  // the tile offset is uniform: it goes into the scalar base address, not into every lane's offset
  const int dma_row = wave * RPI + lane / CPR;  // tile row of this lane's first instruction
  auto dma_tile = [&](uint64_t plane, const uint32_t(&voff)[NDMA], TileAt t, uint32_t lds) __attribute__((always_inline)) {
    const uint64_t base = plane + (RUN ? t.off & ~127u : t.off);
    const int brk = (int)(t.off & 127u);
#pragma unroll
    for (int i = 0; i < NDMA; ++i)
      dma16(base, RUN && dma_row >= brk - i * 8 * RPI ? voff[i] + t.gap : voff[i], lds + i * 8 * 1024);
  };
  // the split's first tile: rows past the keys of a short one repeat its last
  auto dma_tile0 = [&](uint64_t plane, const uint32_t(&voff)[NDMA], TileAt t, uint32_t lds) __attribute__((always_inline)) {
    if (!RUN || !shorted) { dma_tile(plane, voff, t, lds); return; }
    const uint64_t base = plane + (t.off & ~127u);
    const int brk = (int)(t.off & 127u);
#pragma unroll
    for (int i = 0; i < NDMA; ++i) {
      const int row = dma_row + i * 8 * RPI, src = row < last_keys ? row : last_keys - 1;
      dma16(base, voff[i] - (uint32_t)(row - src) * ROW_B + (src >= brk ? t.gap : 0u), lds + i * 8 * 1024);
    }
  };
  auto dma_k = [&](TileAt t, int slot) __attribute__((always_inline)) { dma_tile(kplane, kvoff, t, wave_lds + slot * TILE_B); };
  auto dma_v = [&](TileAt t, int slot) __attribute__((always_inline)) { dma_tile(vplane, vvoff, t, wave_lds + L::V_OFF + slot * TILE_B); };
  // keys that exist in 32-key block blk of the split's first tile (KEYS_SLOT: of every tile)
  auto block_keys = [&](int blk) __attribute__((always_inline)) {
    if (KEYS == KEYS_TILED) return 32;
    const int n = (KEYS == KEYS_SLOT ? p.T : (shorted ? last_keys : BN)) - 32 * blk;
    return n < 0 ? 0 : (n > 32 ? 32 : n);
  };
  // logits of keys that do not exist become -inf (register i of a lane is key row
  // (i / 4) * 8 + 4 * hh + i % 4 of the block)
  auto mask_keys = [&](f32x16_t& sv, int nkeys) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if ((i / 4) * 8 + 4 * hh + (i % 4) >= nkeys) sv[i] = -INFINITY;
  };

  // ---- fragment read addresses (byte offsets into smem) ----
  // K row l32 of a key block, logical chunk 2*ks + hh: physical chunk bits [3:1] are
  // ks ^ (swz >> 1), so the address for step ks is the step-0 address with bits 5.. flipped.
  uint32_t k_rd;
  {
    const int x = k_swz<DH>(l32);
    k_rd = hb * KB_B + l32 * ROW_B + ((((x >> 1) << 1) | (hh ^ (x & 1))) << 4);
  }
  // V rows 4*hh + r (r = lane bits 3:2) of each 8-row group, logical chunk 4*db + c.
  uint32_t v_rd;
  {
    const int r = 4 * hh + ((lane & 15) >> 2);
    const int y = v_swz<DH>(r) >> 2;
    const int c = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    v_rd = L::V_OFF + hb * KB_B + r * ROW_B + ((y * 4 + c) << 4) + (lane & 1) * 8;
  }

  f32x16_t o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  float m_ref = -INFINITY, l_run = 0.f;

  const f32x16_t zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // Softmax scale and reference: the logits are the exact products' sums of the element-type q
  // and k (nothing is rounded before the matrix core); the scale c = softmax scale * log2(e) and
  // the running reference m_ref of this lane's query (every lane owns one query column of the
  // transposed scores) are applied by one fused multiply-add per logit in front of its
  // exponential: p = 2^(s * c + msc), msc = -m_ref * c.
  // Row sums of P (of the rounded values).  256-query shape: on the matrix cores; a 16x16x32 product reads P's registers
  // as 32 keys by 16 columns whose contraction groups are the lane groups, so rows of ones on the even groups, or on the
  // odd ones, leave every lane its own query's sum, both half-waves' keys in it.  (What is not finite in another
  // query's P meets a zero there and makes the sum NaN: that takes the rare path, which adds lane by lane.)  A
  // v_dot2c_f32_bf16 behind another wavefront's products waits for them (16 products and a block's softmax on two
  // wavefronts of a SIMD: 722 cycles each with eight of them, 606 with two 16x16x32, 556 without); in the kernel, at its
  // power limit, 24 heads of 64 on 8, 720 tokens 42.9 -> 41.9 us, 4 x 24 heads, 1024 tokens 352 -> 349, 10 heads of 64,
  // 1500 tokens 55.2 -> 54.4, 24 heads, 3600 tokens 1074 -> 1071 (once more with the present loops: 1600 tokens, 24 heads
  // of 64 140.0 against 136.7, 4 x 40 heads, 256 tokens 32.4 / 30.4).  The 128-query shape keeps the dot products, whose
  // result a step has sooner: 2 x 16 heads of 64, 1000 tokens 0.6 to 1.4 % faster with them (8 slots 74.4 against 75.3 us),
  // 13 heads of 64, 209 tokens, 2 slots 8.83 / 8.97, 56 shapes of heads of 64 off the key tile 0.25 % in the mean; 16 heads
  // of 128, 256 tokens 19.9 either way, 32 on 8, 64 slots 68.6 / 68.9.
  constexpr bool SUMS_MMA = KSPLIT == 1;
  frag_t sum_rows;
#pragma unroll
  for (int i = 0; i < 8; ++i) sum_rows[i] = (typename M::elem_t)((((lane >> 2) ^ (lane >> 4)) & 1) == 0 ? 1.f : 0.f);
  const float lmul = p.scale_log2;
  float msc = 0.f;
  auto set_shift = [&]() __attribute__((always_inline)) { msc = -m_ref * lmul; };

  // probabilities of one 32-key block from its logits: p = 2^((s - sub) * lmul), packed to the
  // element type; returns this half-wave's share of the row sum (of the rounded values)
  auto probabilities = [&](frag_t(&pf)[2], const f32x16_t& s, float sub) __attribute__((always_inline)) {
    float rs = 0.f;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      float e[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) e[j] = __builtin_amdgcn_exp2f((s[8 * m + j] - sub) * lmul);
      pf[m] = M::pack8(e[0], e[1], e[2], e[3], e[4], e[5], e[6], e[7]);
#pragma unroll
      for (int j = 0; j < 4; ++j) rs = M::add_pair(rs, pf[m], j);
    }
    return rs;
  };
  auto block_max = [&](const f32x16_t& s) __attribute__((always_inline)) {
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    float lo, up;
    half_wave_pair(mx, lo, up);
    return fmaxf(lo, up);
  };

  // The pipeline runs on 32-key blocks.  One step computes, for this wavefront,
  //   matrix cores: the logits of the block read at K offset KOFF (-> s_next) and the
  //                 product of the previous block's probabilities with the V block at VOFF;
  //   VALU:         the probabilities of the current block (s_cur -> p_cur).
  // LDS reads are issued in consumption order - K fragments 0..KS-1, then the NV V^T fragments
  // (two transposing reads each) - running up to 15 reads ahead of the MFMAs.
  frag_t p_prev[2];
  f32x16_t s_cur;
  // Fragment registers live across steps: every step starts with its first PRE reads (all K
  // fragments and the first V^T fragment) already in flight, issued during the previous step.
  constexpr int PRE = KS + 2;
  u32x4_t kf[KS];
  u32x2_t v0[NV], v1[NV];
  auto read_k = [&](auto koff_c, int ks) __attribute__((always_inline)) {
    kf[ks] = lds_read128<decltype(koff_c)::value>(smem, k_rd ^ (ks << 5));
  };
  auto read_v = [&](auto voff_c, int i) __attribute__((always_inline)) {  // fragment i = (m, db) = (i / DB, i % DB)
    constexpr int VOFF = decltype(voff_c)::value;
    const uint32_t a = v_rd ^ ((i % DB) << 6);
    if (i / DB == 0) {
      v0[i] = lds_read_tr<VOFF>(smem, a);
      v1[i] = lds_read_tr<VOFF + 8 * ROW_B>(smem, a);
    } else {
      v0[i] = lds_read_tr<VOFF + 16 * ROW_B>(smem, a);
      v1[i] = lds_read_tr<VOFF + 24 * ROW_B>(smem, a);
    }
  };
  auto prefetch = [&](auto koff_c, auto voff_c) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) read_k(koff_c, ks);
    read_v(voff_c, 0);
  };
  // nkeys: keys that exist in the block whose logits this step computes, where mask_c says that it
  // may be short
  // (the K fragments at koff_c were requested by the previous step; the offset documents the call)
  // first_c (128-query shape only): the workgroup's very first step has no previous block, so it
  // skips the product and its V reads instead of multiplying a zeroed tile by zeros.
  auto step = [&](auto /*koff_c*/, auto voff_c, auto nkoff_c, auto nvoff_c, auto mask_c, int nkeys, auto&& mid, auto first_c) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first_c)::value;
    // (logits of a block past the end of the split are never consumed)
    // next own V fragment to request / next-step read pairs requested so far
    int vnext = 1, npair = 0;
    constexpr int NPAIR = PRE / 2;            // the next step's first reads go out two at a time
    constexpr int I0 = NV - 1 - NPAIR;        // ... after the product MFMAs I0, I0+1, ...
    auto next_pair = [&]() __attribute__((always_inline)) {
      if (2 * npair < KS) {
        read_k(nkoff_c, 2 * npair);
        read_k(nkoff_c, 2 * npair + 1);
      } else {
        read_v(nvoff_c, 0);
      }
      ++npair;
    };

    // From here to the end of the product the issue order is pinned statement by statement
    // (sched_barrier): MFMA, the reads that refill the queue, a slice of the VALU work.
    __builtin_amdgcn_sched_barrier(0);
    frag_t p_cur[2];
    float e[16];
    float rs = 0.f;
    f32x4_t sums;  // (SUMS_MMA)
    // VALU slices: the 16 exponentials of the current block are spread evenly over the MFMAs of
    // the step.  The two wavefronts of a SIMD run in phase, so bunching them under the logits
    // would saturate the quarter-rate unit there and leave it idle under the product.
    constexpr int EPS = 16 / (KS + NV);
    static_assert(EPS * (KS + NV) == 16, "exponentials per slot");
    auto exp_slot = [&](int g) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < EPS; ++t)
        if (g * EPS + t < 16) {
          e[g * EPS + t] = __builtin_amdgcn_exp2f(__builtin_fmaf(s_cur[g * EPS + t], lmul, msc));
          // an exponential has no side effect, so nothing else keeps it in its slot: left alone the
          // compiler sinks the first nine of a step below the tile DMAs
          asm volatile("" : "+v"(e[g * EPS + t]));
        }
    };
    f32x16_t s_next;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      s_next = M::mma(__builtin_bit_cast(frag_t, kf[ks]), qf[ks], ks == 0 ? zero16 : s_next);
      // keep the read queue full without exceeding the 15 reads the counter can track
      if (!FIRST && vnext < NV && ks <= 12 - KS) {
        read_v(voff_c, vnext);
        ++vnext;
        }
      exp_slot(ks);
      __builtin_amdgcn_sched_barrier(0);
    }
    mid();  // the tile DMAs of this iteration go out here, under the MFMAs already queued
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if (!FIRST) {
        if (vnext < NV) {  // reads 0..KS+2i-1 have completed: room for one more fragment
          read_v(voff_c, vnext);
          ++vnext;
        }
        typedef unsigned int u32x4v __attribute__((ext_vector_type(4)));
        const u32x4v a4 = __builtin_shufflevector(v0[i], v1[i], 0, 1, 2, 3);
        o[i % DB] = M::mma(__builtin_bit_cast(frag_t, a4), p_prev[i / DB], o[i % DB]);
      }
      if (i >= I0 && npair < NPAIR) next_pair();
      // VALU slices: the last exponentials; packing of the two 16-key halves and their row sums
      exp_slot(KS + i);
      if (i == 1) p_cur[0] = M::pack8(e[0], e[1], e[2], e[3], e[4], e[5], e[6], e[7]);
      if (i == 2) {
        if (SUMS_MMA) {
          sums = M::mma16(sum_rows, p_cur[0], f32x4_t{0.f, 0.f, 0.f, 0.f});
        } else {
#pragma unroll
          for (int t = 0; t < 4; ++t) rs = M::add_pair(rs, p_cur[0], t);
        }
      }
      if (i == NV - 1) p_cur[1] = M::pack8(e[8], e[9], e[10], e[11], e[12], e[13], e[14], e[15]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (SUMS_MMA) {
      rs = M::mma16(sum_rows, p_cur[1], sums)[0];
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) rs = M::add_pair(rs, p_cur[1], t);
    }

    if (__ballot(!(rs <= 256.f)) != 0ull) {
      // Rare: some probability of this block may exceed 2^8.  Raise the reference of the rows
      // that need it, redo the block's probabilities exactly and rescale the accumulators: they
      // hold the blocks before this one (the last of those products was issued above).
      const float mx = block_max(s_cur);
      const float m_new = mx > m_ref ? mx : m_ref;
      const float alpha = __builtin_amdgcn_exp2f((m_ref - m_new) * lmul);
      rs = probabilities(p_cur, s_cur, m_new);
      if (SUMS_MMA) {
        float lo, up;
        half_wave_pair(rs, lo, up);
        rs = lo + up;
      }
      l_run *= alpha;
      m_ref = m_new;
      set_shift();
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
    }
    l_run += rs;
    p_prev[0] = p_cur[0];
    p_prev[1] = p_cur[1];
    if (decltype(mask_c)::value && nkeys < 32) mask_keys(s_next, nkeys);
    s_cur = s_next;
  };

  // A wavefront whose 32 rows all lie behind the last token only fetches: its products would be thrown away, and they
  // cost the others clock (the board runs these kernels at its power limit).  24 heads, 3600 tokens, 8 slots (15 tiles
  // of 256 rows, the last with 16 of them) 1102 -> 1074 us; 12 heads on 6, 920 tokens 50.9 -> 49.5; 32 heads, 130
  // tokens, 16 slots 20.0 -> 19.3.  Not in the 128-query shape of whole tiles, whose frames leave no wavefront idle or
  // half of them: there the branch cost 256-token frames 1 to 2 % (32 slots 28.6 -> 29.1).
  constexpr bool MAY_IDLE = RUN || KSPLIT == 1;
  const bool idle = MAY_IDLE && __builtin_amdgcn_readfirstlane(row0 + qb * 32) >= (SHARED ? p.group * p.T : p.T);
  if (ntile > 0) {
    // 256-query shape: zero V slot 3, which stands in for "tile -1", and P, so that the first
    // product adds zeros (the 128-query shape skips the product of its first step instead)
    if (KSPLIT == 1) {
      const u32x4_t z = {0u, 0u, 0u, 0u};
      unsigned char* vz = smem + L::V_OFF + 3 * TILE_B;
      for (int i = tid; i < TILE_B / 16; i += 512) *reinterpret_cast<u32x4_t*>(vz + i * 16) = z;
    }
    {
      const u32x4_t z = {0u, 0u, 0u, 0u};
      p_prev[0] = __builtin_bit_cast(frag_t, z);
      p_prev[1] = __builtin_bit_cast(frag_t, z);
    }
    // Iteration j issues K(j+KA) and V(j+2) (KA = 3, or 4 when every wavefront handles one key
    // block per tile and prefetches its next fragments across the barrier); the prologue issues
    // what the iterations before 0 would have.
    constexpr int KA = KSPLIT == 1 ? 3 : 4;
    // The V stream trails the K stream by KA - 2 tiles, so it reuses the K stream's offsets.
    TileAt off1, off2;  // offsets of the last and the last-but-one tile the K stream visited
    // Q was requested before the slot flags and loads return in order, so it is here; stating a
    // use now keeps the wait for it from landing behind the tile DMAs issued next.
    if (!q_dma) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) asm volatile("" ::"v"(qf[ks]));
    }
    {
      const TileAt o0 = next_off();
      const TileAt o1 = next_off();
      const TileAt o2 = next_off();
      dma_tile0(kplane, kvoff, o0, wave_lds);
      dma_k(o1, 1);
      if (KSPLIT == 2) dma_k(o2, 2);
      dma_tile0(vplane, vvoff, o0, wave_lds + L::V_OFF);
      if (KSPLIT == 1) {
        dma_k(o2, 2);
        off1 = o2; off2 = o1;
      } else {
        const TileAt o3 = next_off();
        dma_k(o3, 3);
        off1 = o3; off2 = o2;
      }
      dma_v(o1, 1);
    }
    dma_wait<(KA + 1) * NDMA>();
    __syncthreads();  // K(0) and the zeroed V slot (128-query shape: the Q tile, requested long before K(0)) are in LDS
    stamp(1);  // first K tile landed
    if (idle) {
      // (the same requests and barriers as the wavefronts that have queries)
      dma_wait<2 * NDMA>();
      __syncthreads();
      for (int j = 0; j < ntile; ++j) {
        const TileAt o = next_off();
        dma_k(o, (j + KA) % NST);
        dma_v(KA == 3 ? off1 : off2, (j + 2) % NST);
        off2 = off1;
        off1 = o;
        dma_wait<2 * NDMA>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      if (KSPLIT == 2 && DH == 64) {
        // Nothing of it is merged, stored or kept, and the two ways need not meet again: bf16, 8 heads, 100 tokens, 2
        // slots 7.70 -> 7.57 us, 13 heads, 209 tokens 8.97 -> 8.88, 2 x 24 heads, 150 tokens 8.15 -> 8.03; f16 the same to 1 %
        // slower (7.71 / 7.72, 9.00 / 9.01, 8.10 / 8.19).  The other shapes gain nothing (16 heads of 128, 225 tokens, 2 slots
        // 12.72 / 12.74, 6 heads, 150 tokens 9.91 / 9.99; 256 queries: 24 heads of 64 on 8, 720 tokens 42.9 / 43.2).
        dma_wait<0>();
        __syncthreads();
        __syncthreads();
        return;
      }
      m_ref = 0.f;
    } else {
    if (KSPLIT == 2 && q_dma) {
      // row qb*32 + l32 of the tile, logical chunk 2*ks + hh: the K fragment's address arithmetic
      const int x = k_swz<DH>(l32);
      const uint32_t q_rd = (uint32_t)(Q_OFF + qb * KB_B + l32 * ROW_B + ((((x >> 1) << 1) | (hh ^ (x & 1))) << 4));
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const frag_t*>(smem + (q_rd ^ (ks << 5)));
    }
    // (Q stays in registers for the rest of the kernel)
    // first block: reference = its row max
    {
      s_cur = zero16;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const frag_t a = *reinterpret_cast<const frag_t*>(smem + (k_rd ^ (ks << 5)));
        s_cur = M::mma(a, qf[ks], s_cur);
      }
      const int nk0 = block_keys(hb);
      if (KEYS != KEYS_TILED && nk0 < 32) mask_keys(s_cur, nk0);
      const float mx0 = block_max(s_cur);
      // An empty block has no reference to give: one far below any logit makes the first block with
      // keys exceed every bound and take the rare path, which finds the right one (sums and
      // accumulators are still zero then).
      m_ref = mx0 > -INFINITY ? mx0 : (KEYS == KEYS_TILED ? 0.f : -1e30f);
      set_shift();
    }
    // (every wavefront has read its Q fragments before it passes the barrier below: the staging area
    // becomes V slots again)
    dma_wait<2 * NDMA>();
    __syncthreads();  // everything but the last K and V tile issued so far has landed
    // first reads of the first step
    if (KSPLIT == 1) {
      prefetch(IntC<KB_B>(), IntC<3 * TILE_B + KB_B>());
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) read_k(IntC<TILE_B>(), ks);
    }

    // one tile iteration with compile-time ring positions (JM = j mod 4)
    auto iteration = [&](int j, auto jm_c, auto first_c) __attribute__((always_inline)) {
      constexpr int JM = decltype(jm_c)::value;
      constexpr bool FIRST = decltype(first_c)::value;
      auto issue_dma = [&]() __attribute__((always_inline)) {
        const TileAt o = next_off();
        dma_k(o, (JM + KA) % NST);                       // K(j+KA)
        dma_v(KA == 3 ? off1 : off2, (JM + 2) % NST);    // V(j+2)
        off2 = off1;
        off1 = o;
      };
      auto nothing = [&]() __attribute__((always_inline)) {};
      typedef std::integral_constant<bool, KEYS == KEYS_SLOT> short_slots;
      if (KSPLIT == 1) {
        // block (j, 0) -> probabilities; logits of (j, 1); product of (j-1, 1)
        step(IntC<JM * TILE_B + KB_B>(), IntC<((JM + 3) % NST) * TILE_B + KB_B>(),
             IntC<((JM + 1) % NST) * TILE_B>(), IntC<JM * TILE_B>(),
             std::integral_constant<bool, KEYS == KEYS_SLOT || (RUN && FIRST)>(), block_keys(1), issue_dma,
             std::false_type());
        // block (j, 1) -> probabilities; logits of (j+1, 0); product of (j, 0)
        step(IntC<((JM + 1) % NST) * TILE_B>(), IntC<JM * TILE_B>(),
             IntC<((JM + 1) % NST) * TILE_B + KB_B>(), IntC<JM * TILE_B + KB_B>(),
             short_slots(), block_keys(0), nothing, std::false_type());
      } else {
        // block (j, hb) -> probabilities; logits of (j+1, hb); product of (j-1, hb)
        step(IntC<((JM + 1) % NST) * TILE_B>(), IntC<((JM + 3) % NST) * TILE_B>(),
             IntC<((JM + 2) % NST) * TILE_B>(), IntC<JM * TILE_B>(),
             short_slots(), block_keys(__builtin_amdgcn_readfirstlane(hb)), issue_dma, first_c);
      }
      dma_wait<2 * NDMA>();  // all but this iteration's two tiles have landed (this wavefront's part)
      // A bare barrier: __syncthreads() would also wait for every LDS read in flight, i.e. for the
      // next step's fragments requested a moment ago.  Nothing needs that: the tiles arrive by DMA,
      // whose completion the counter wait above tracks, fragment reads are awaited where they are
      // used, and the reads still in flight here target ring slots that no DMA overwrites before
      // the barrier after next.  The empty asm keeps the compiler from moving memory accesses across.
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };

    int j = 0;
    const std::false_type not_first;
    if (KSPLIT == 2 || RUN) {
      // the first tile's step has no product to do (128 queries) or may have keys to mask: peeled,
      // with the three iterations that bring the ring position back to zero
      iteration(0, IntC<0>(), std::true_type());
      j = 1;
      if (j < ntile) { iteration(j, IntC<1>(), not_first); ++j; }
      if (j < ntile) { iteration(j, IntC<2>(), not_first); ++j; }
      if (j < ntile) { iteration(j, IntC<3>(), not_first); ++j; }
    }
    for (; j + 4 <= ntile; j += 4) {
      iteration(j, IntC<0>(), not_first);
      iteration(j + 1, IntC<1>(), not_first);
      iteration(j + 2, IntC<2>(), not_first);
      iteration(j + 3, IntC<3>(), not_first);
    }
    if (j < ntile) { iteration(j, IntC<0>(), not_first); ++j; }
    if (j < ntile) { iteration(j, IntC<1>(), not_first); ++j; }
    if (j < ntile) { iteration(j, IntC<2>(), not_first); ++j; }

    stamp(2);  // tile loop left
    // product of the last block: (ntile-1, 1) for full-tile wavefronts, (ntile-1, hb) otherwise
    {
      const int last = (ntile - 1) % NST;
      const unsigned char* vt = smem + v_rd + last * TILE_B + (KSPLIT == 1 ? KB_B : 0);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const unsigned char* va = smem + ((uint32_t)(vt - smem) ^ (db << 6)) + 16 * m * ROW_B;
          const s16x4_t a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(va));
          const s16x4_t a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(va + 8 * ROW_B));
          typedef short s16x8_t __attribute__((ext_vector_type(8)));
          const s16x8_t a8 = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
          o[db] = M::mma(__builtin_bit_cast(frag_t, a8), p_prev[m], o[db]);
        }
      }
    }
    }
    dma_wait<0>();  // no DMA may still be writing LDS when the rings are reused or the CU is freed
  } else if (q_dma) {
    dma_wait<0>();  // (a split without visible keys: the Q tile it asked for must not land after the merge below)
  }

  float l_tot = l_run;
  if (!SUMS_MMA) {
    float lo, up;
    half_wave_pair(l_run, lo, up);
    l_tot = lo + up;
  }
  m_ref *= lmul;  // from raw logits to the log2 domain the merges work in

  if (KSPLIT == 2) {
    // ---- the two wavefronts of a query block merge their (m, l, O) through LDS ----
    // 16-byte accesses: vector k of lane l sits at ((qb * (DB * 4 + 1) + k) * 64 + l) * 16.
    __syncthreads();  // every wavefront is done with the rings
    f32x4_t* mb = reinterpret_cast<f32x4_t*>(smem) + (qb * (DB * 4 + 1)) * 64 + lane;
    if (hb == 1) {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          mb[(db * 4 + c) * 64] = f32x4_t{o[db][4 * c], o[db][4 * c + 1], o[db][4 * c + 2], o[db][4 * c + 3]};
      mb[(DB * 4) * 64] = f32x4_t{m_ref, l_tot, 0.f, 0.f};
    }
    __syncthreads();
    if (hb == 1) return;
    const f32x4_t ml1 = mb[(DB * 4) * 64];
    // a wavefront whose sum is zero saw no key (or only keys that vanish against its reference):
    // its reference must not take part in the maximum
    const float m1 = ml1[1] > 0.f ? ml1[0] : -INFINITY, l1 = ml1[1];
    if (!(l_tot > 0.f)) m_ref = -INFINITY;
    const float mm = fmaxf(m_ref, m1);
    if (mm > -INFINITY) {
      const float a0 = __builtin_amdgcn_exp2f(m_ref - mm), a1 = __builtin_amdgcn_exp2f(m1 - mm);
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const f32x4_t other = mb[(db * 4 + c) * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) o[db][4 * c + e] = a0 * o[db][4 * c + e] + a1 * other[e];
        }
      l_tot = a0 * l_tot + a1 * l1;
      m_ref = mm;
    }
  }

  stamp(3);  // pair merged
  // ---- epilogue ----
  const AttnParams& ep = KEYS != KEYS_SLOT && !SHARED ? p : reread_args<AttnParams>();
  const int64_t rows = (int64_t)ep.B * ep.H * ep.T - ep.ws_row0;  // rows in the workspace
  const int hq = SHARED ? (int)(qrow / (unsigned)ep.T) : 0, qt = (int)qrow - hq * ep.T;
  const int h = h0 + hq;
  const bool valid = qt < ep.T && (!SHARED || hq < ep.group);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  const int64_t row = ((int64_t)b * ep.H + h) * ep.T + qt;
  float gate_v = 1.f;
  const bool gated = ep.gate != nullptr || ep.gate_w != nullptr;
  if (gated && nsp == 1 && valid) gate_v = head_gate<typename M::elem_t>(ep, b, h, qt);
  // A split leaves its partial output as values in [-1, 1] plus one fp32 scale per row (the row's
  // largest normalised magnitude).  For a bf16 output they are fp16: 11 significant bits for the bytes
  // of a bf16 row, three more than the output has, and no overflow for any finite V.  For an f16 output
  // that would be its own precision once more per part, so they are fp32 (PARTS_F32; ws_f32 is off only
  // where a caller's workspace is too short for it).  A row that holds an infinity keeps the
  // plain normalised values (scale 1), so that only the columns concerned turn non-finite, as in a
  // single pass; a row whose largest magnitude is too small for its reciprocal is scaled by 2^100.
  float mul = inv;
  if (nsp > 1) {
    float amax = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(o[db][i]));
    float alo, aup;
    half_wave_pair(amax, alo, aup);
    amax = fmaxf(alo, aup);
    float row_scale;
    if (amax < INFINITY) {
      const float a = fmaxf(amax, 0x1p-100f);
      mul = 1.f / a;
      row_scale = a * inv;
    } else {
      mul = inv;
      row_scale = 1.f;
    }
    if (valid && hh == 0)
      *reinterpret_cast<f32x4_t*>(ep.ws_ml + ((int64_t)split * rows + (row - ep.ws_row0)) * 4) =
          f32x4_t{l_tot > 0.f ? m_ref : -INFINITY, l_tot, row_scale, 0.f};
  }
#pragma unroll
  for (int db = 0; db < DB; ++db) {
#pragma unroll
    for (int c = 0; c < 4; c += 2) {
      // register quad c holds head-dim rows 8c + 4*half + 0..3; after the swap a lane of the
      // lower half owns rows 8c..8c+7 and a lane of the upper half rows 8(c+1)..8(c+1)+7.
      float f[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(o[db][4 * c + e] * mul),
                                                  __float_as_uint(o[db][4 * c + 4 + e] * mul), false, false);
        f[e] = __uint_as_float(r[0]);
        f[4 + e] = __uint_as_float(r[1]);
      }
      const int d0 = 32 * db + 8 * (c + hh);
      if (valid) {
        if (nsp == 1) {
          uint16_t* dst = reinterpret_cast<uint16_t*>(ep.out) + b * ep.os_b + h * ep.os_h +
                          (int64_t)qt * ep.os_t + d0;
          frag_t y = M::pack8(f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7]);
          if (gated) {  // y * gate on element-type values, as the module's own multiply
            y = M::pack8((float)y[0] * gate_v, (float)y[1] * gate_v, (float)y[2] * gate_v, (float)y[3] * gate_v,
                         (float)y[4] * gate_v, (float)y[5] * gate_v, (float)y[6] * gate_v, (float)y[7] * gate_v);
          }
          *reinterpret_cast<frag_t*>(dst) = y;
        } else {
          const int64_t at = ((int64_t)split * rows + (row - ep.ws_row0)) * DH + d0;
          if (PARTS_F32 && ep.ws_f32 != 0) {
            f32x4_t* dst = reinterpret_cast<f32x4_t*>(static_cast<float*>(ep.ws_o) + at);
            dst[0] = f32x4_t{f[0], f[1], f[2], f[3]};
            dst[1] = f32x4_t{f[4], f[5], f[6], f[7]};
          } else {
            *reinterpret_cast<f16x8_t*>(static_cast<uint16_t*>(ep.ws_o) + at) = F16Mma::pack8(f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7]);
          }
        }
      }
    }
  }
  stamp(4);  // results / partial results stored (requests issued)
  if (CLOCKED && tid == 0) {
    p.clock_out[kClockSlots * wg_id] = (uint64_t)__builtin_readcyclecounter() - clk0;
    p.clock_out[kClockSlots * wg_id + 1] = (uint64_t)__builtin_amdgcn_s_memrealtime() - wall0;
  }
}

// WE_WITH_PROBES (the measurement library's build) adds the CLOCKED instantiations; the product's
// objects hold none of their code.
#ifdef WE_WITH_PROBES
constexpr bool kWithProbes = true;
#else
constexpr bool kWithProbes = false;
#endif

template <typename M, int DH, int KSPLIT, int KEYS, bool CLOCKED>
static hipError_t launch_ring_c(const AttnParams& p, hipStream_t stream) {
  const int rounds = (p.unit_splits + 7) / 8;
  const dim3 grid((unsigned)(8 * (p.members / p.q_heads)), (unsigned)p.q_heads, (unsigned)rounds);
  hipLaunchKernelGGL((attn_ring_kernel<M, DH, KSPLIT, KEYS, CLOCKED>), grid, dim3(512), RingLds<DH>::kBytes, stream, p);
  return hipGetLastError();
}
template <typename M, int DH, int KSPLIT, int KEYS>
static hipError_t launch_ring_r(const AttnParams& p, hipStream_t stream) {
  if constexpr (kWithProbes) {
    if (p.clock_out != nullptr) return launch_ring_c<M, DH, KSPLIT, KEYS, true>(p, stream);
  }
  return launch_ring_c<M, DH, KSPLIT, KEYS, false>(p, stream);
}
template <typename M, int DH, int KSPLIT>
static hipError_t launch_ring_t(const AttnParams& p, hipStream_t stream) {
  return p.T % BN == 0 ? launch_ring_r<M, DH, KSPLIT, KEYS_TILED>(p, stream) : launch_ring_r<M, DH, KSPLIT, KEYS_PACKED>(p, stream);
}

// The kernels use more LDS than a launch may ask for by default; the limit is a per-device
// setting of each kernel, raised once per device by the library's set-up (device_state.hip).
template <typename M, int DH, int KSPLIT, int KEYS, bool CLOCKED>
static hipError_t configure_one() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_ring_kernel<M, DH, KSPLIT, KEYS, CLOCKED>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, RingLds<DH>::kBytes);
}
template <typename M, int DH, int KEYS>
static hipError_t configure_keys() {
  hipError_t e = configure_one<M, DH, 1, KEYS, false>();
  if (e == hipSuccess) e = configure_one<M, DH, 2, KEYS, false>();
  if constexpr (kWithProbes) {
    if (e == hipSuccess) e = configure_one<M, DH, 1, KEYS, true>();
    if (e == hipSuccess) e = configure_one<M, DH, 2, KEYS, true>();
  }
  return e;
}
template <typename M, int DH>
static hipError_t configure_family() {
  const hipError_t e = configure_keys<M, DH, KEYS_TILED>();
  return e == hipSuccess ? configure_keys<M, DH, KEYS_PACKED>() : e;
}
// frames below one tile, and grouped heads that share query tiles
template <typename M, int KEYS>
static hipError_t launch_keys(const AttnParams& p, int Dh, int ksplit, hipStream_t stream) {
  if (Dh == 128) return ksplit == 2 ? launch_ring_r<M, 128, 2, KEYS>(p, stream) : launch_ring_r<M, 128, 1, KEYS>(p, stream);
  return ksplit == 2 ? launch_ring_r<M, 64, 2, KEYS>(p, stream) : launch_ring_r<M, 64, 1, KEYS>(p, stream);
}
template <typename M, int KEYS>
static hipError_t configure_both() {
  const hipError_t e = configure_keys<M, 128, KEYS>();
  return e == hipSuccess ? configure_keys<M, 64, KEYS>() : e;
}

// The four (element type, head dim) families (parts 0 to 3) and the short frames' and the shared tiles'
// instantiations (4 to 7) are compiled as separate objects, one per WE_RING_PART, so that they build in
// parallel.  Without it this translation unit holds parts 0 to 3.
#if !defined(WE_RING_PART) || WE_RING_PART == 0
hipError_t launch_attn_ring_bf16_128(const AttnParams& p, int ksplit, hipStream_t stream) {
  return ksplit == 2 ? launch_ring_t<Bf16Mma, 128, 2>(p, stream) : launch_ring_t<Bf16Mma, 128, 1>(p, stream);
}
hipError_t configure_attn_ring_bf16_128() { return configure_family<Bf16Mma, 128>(); }
#endif
#if !defined(WE_RING_PART) || WE_RING_PART == 1
hipError_t launch_attn_ring_bf16_64(const AttnParams& p, int ksplit, hipStream_t stream) {
  return ksplit == 2 ? launch_ring_t<Bf16Mma, 64, 2>(p, stream) : launch_ring_t<Bf16Mma, 64, 1>(p, stream);
}
hipError_t configure_attn_ring_bf16_64() { return configure_family<Bf16Mma, 64>(); }
#endif
#if !defined(WE_RING_PART) || WE_RING_PART == 2
hipError_t launch_attn_ring_f16_128(const AttnParams& p, int ksplit, hipStream_t stream) {
  return ksplit == 2 ? launch_ring_t<F16Mma, 128, 2>(p, stream) : launch_ring_t<F16Mma, 128, 1>(p, stream);
}
hipError_t configure_attn_ring_f16_128() { return configure_family<F16Mma, 128>(); }
#endif
#if !defined(WE_RING_PART) || WE_RING_PART == 3
hipError_t launch_attn_ring_f16_64(const AttnParams& p, int ksplit, hipStream_t stream) {
  return ksplit == 2 ? launch_ring_t<F16Mma, 64, 2>(p, stream) : launch_ring_t<F16Mma, 64, 1>(p, stream);
}
hipError_t configure_attn_ring_f16_64() { return configure_family<F16Mma, 64>(); }
#endif

#if defined(WE_RING_PART) && WE_RING_PART == 4
hipError_t launch_attn_ring_short_bf16(const AttnParams& p, int Dh, int ksplit, hipStream_t stream) {
  return launch_keys<Bf16Mma, KEYS_SLOT>(p, Dh, ksplit, stream);
}
hipError_t configure_attn_ring_short_bf16() { return configure_both<Bf16Mma, KEYS_SLOT>(); }
#endif
#if defined(WE_RING_PART) && WE_RING_PART == 5
hipError_t launch_attn_ring_short_f16(const AttnParams& p, int Dh, int ksplit, hipStream_t stream) {
  return launch_keys<F16Mma, KEYS_SLOT>(p, Dh, ksplit, stream);
}
hipError_t configure_attn_ring_short_f16() { return configure_both<F16Mma, KEYS_SLOT>(); }
#endif
#if defined(WE_RING_PART) && WE_RING_PART == 6
hipError_t launch_attn_ring_shared_bf16(const AttnParams& p, int Dh, int ksplit, hipStream_t stream) {
  return launch_keys<Bf16Mma, KEYS_SHARED>(p, Dh, ksplit, stream);
}
hipError_t configure_attn_ring_shared_bf16() { return configure_both<Bf16Mma, KEYS_SHARED>(); }
#endif
#if defined(WE_RING_PART) && WE_RING_PART == 7
hipError_t launch_attn_ring_shared_f16(const AttnParams& p, int Dh, int ksplit, hipStream_t stream) {
  return launch_keys<F16Mma, KEYS_SHARED>(p, Dh, ksplit, stream);
}
hipError_t configure_attn_ring_shared_f16() { return configure_both<F16Mma, KEYS_SHARED>(); }
#endif

}  // namespace we
