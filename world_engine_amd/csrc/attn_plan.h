// Host side of an attention call: argument validation, the choice of kernel shape and context
// splitting, and the kernel parameter block.  Shared by the C ABI (capi.hip) and by the
// measurement library's entry points (probe_capi.hip), so that both plan a call identically.
#pragma once
#include "../../include/we_attn.h"
#include "f32_parts.h"
#include "short_parts.h"
#include "we_kernels.h"

namespace we {
namespace host {

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline int elem_bytes(int dtype) { return dtype == WE_DTYPE_F32 ? 4 : 2; }

// element strides whose byte value keeps every row start 16-byte aligned
inline bool strides_ok(const int64_t s[3], int dtype) {
  const int per16 = 16 / elem_bytes(dtype);
  return s[0] % per16 == 0 && s[1] % per16 == 0 && s[2] % per16 == 0;
}

inline int ring_shape_ok(int B, int H, int Hkv, int T, int Dh, int64_t L, int dilation) {
  if (B <= 0 || H <= 0 || Hkv <= 0 || T <= 0 || Dh <= 0 || L <= 0 || dilation <= 0) return WE_ERR_BAD_SHAPE;
  if (H % Hkv != 0 || L % T != 0 || (L / T) % dilation != 0) return WE_ERR_BAD_SHAPE;
  return WE_OK;
}

struct AttnPlan {
  int variant;      // 1: 128 queries per workgroup, 2: 256
  int block_m;      // queries per workgroup
  int n_splits;     // context splits of the units that are split (1: none)
  int units_whole;  // leading (batch, kv head) units that are not split
  int64_t ws_rows;  // query rows that go through the split-context workspace
  int cus;          // compute units planned for
  int f32_groups = 1;   // fp32 calls: groups of 16 queries per workgroup, for the parts in AttnParams
};

inline int variant_of(int q_tile) {
  switch (q_tile) {
    case 0: return 0;
    case 128: return 1;
    case 256: return 2;
    default: return -1;
  }
}

// Workgroups of a (batch, kv head) unit, which share its K/V stream: the query tiles of its heads.  The heads of
// a group fill the tiles together where that saves one (3 heads of 143 queries: four tiles of 128 where each by
// itself takes two) and tiles are what takes the time: not in frames of up to 128 tokens, nor in calls whose rows
// fill less than a quarter of the CUs with tiles of 128, from 257 tokens an eighth.  (28 heads of 64 on 7, 374
// tokens, 16 slots 32.8 -> 29.3 us; 24 of 128 on 12, 180 tokens, batch 2 28.0 -> 23.8; 60 on 15, 308 tokens,
// batch 2 69.0 -> 59.  16 on 4, 192 tokens would be 18.1 -> 18.6, 6 on 2, 320 tokens 11.4 -> 11.9.)
inline int64_t members_of(int units, int group, int T, int block_m, int cus, bool* shared = nullptr) {
  const int64_t apart = group * (((int64_t)T + block_m - 1) / block_m);
  const int64_t together = ((int64_t)group * T + block_m - 1) / block_m;
  const bool share = together < apart && T > 128 && (int64_t)units * group * T >= (int64_t)cus * (T > 256 ? 16 : 32);
  if (shared != nullptr) *shared = share;
  return share ? together : apart;
}

// The basic choice of kernel shape and context splitting for a part with `cus` compute units (256 on an
// MI355X; every count below was measured there and is carried to other sizes as a fraction).
//  * Shape: 256 queries per workgroup when that alone gives at least one workgroup per CU, else
//    128 queries (two wavefronts share each query block and split every tile's keys).
//  * Few workgroups (256-token frames): every unit is split into the same number of context
//    parts - as many as fit the CUs in one round up to four parts, then as many as give 5/8 to
//    15/16 of the CUs a workgroup (more for long contexts, fewer for many parts) - but never fewer
//    than two 64-key tiles per part.
//  * Many workgroups that do not divide into whole rounds of CUs (e.g. 384 on 256): only the units
//    of the last, partial round are split, so that round finishes in a fraction of the time.
inline AttnPlan plan_basic(int B, int H, int Hkv, int T, int64_t L, int n_splits, int variant, int cus) {
  AttnPlan pl;
  if (cus < 8) cus = 8;
  pl.cus = cus;
  const int64_t wg256 = (int64_t)B * Hkv * members_of(B * Hkv, H / Hkv, T, 256, cus);
  const int64_t wg128 = (int64_t)B * Hkv * members_of(B * Hkv, H / Hkv, T, 128, cus);
  // 256 queries per workgroup when that alone fills the CUs - or when 128 would spill into a
  // second round that 256 avoids (136 to 256 heads of a 256-token frame: one round of fat
  // workgroups beats one and a bit rounds of thin ones by 5 to 17 %)
  pl.variant = variant ? variant : ((T >= 256 && (wg256 >= cus || wg128 > cus)) ? 2 : 1);
  pl.block_m = pl.variant == 2 ? 256 : 128;
  const int units = B * Hkv;
  const int group = H / Hkv;
  const int members = (int)members_of(units, group, T, pl.block_m, cus);
  const int64_t wgs = (int64_t)units * members;
  const int64_t tiles = L / 64;  // visible 64-key tiles at steady state
  const int64_t max_s = tiles / 2 > 0 ? tiles / 2 : 1;
  pl.units_whole = 0;
  pl.n_splits = 1;
  if (n_splits > 0) {
    pl.n_splits = n_splits;
  } else if (wgs < cus) {
    // Never more workgroups than CUs (a second, nearly empty round costs a whole kernel's
    // time); and when the context is cut four ways or more, fewer workgroups than CUs: a part's
    // fixed costs do not shrink with its length, the partial results grow with the number of
    // parts, and the board clocks the kernel lower the more CUs are busy (16 heads of a 256-token
    // frame over 16 slots: 6 parts 25.1 us per frame-step, 8 parts 27.2; 24 such rings: 653
    // against 717).  Measured over 8 to 160 workgroups per call: the best count is about 15/16 of
    // the CUs for up to six parts and about 3/4 for more.
    // Long contexts (32 slots of a 256-token frame and more) amortise the extra parts and the lower
    // clock over longer loops: about 15/16 there too (32 slots: 7 parts 32.0 us per frame-step,
    // 6 parts 32.8), and all CUs when that is exactly four parts (a quarter of the CUs unsplit:
    // 4 parts beat 3 by 2 to 7 %).
    // Beyond sixteen parts every part's own cost weighs more: about 5/8 of the CUs (4 heads: 20
    // parts 21.2 to 27.2 us per frame-step over 16 to 64 slots, 24 parts 21.7 to 27.4).
    const int64_t c15 = (int64_t)cus * 15 / 16, c34 = (int64_t)cus * 3 / 4, c58 = (int64_t)cus * 5 / 8;
    int64_t s = cus / wgs;
    if (s > 4) s = ((wgs * 32 >= (int64_t)cus * 5 || (tiles >= 96 && c15 / wgs <= 16)) ? c15 : (c34 / wgs > 16 ? c58 : c34)) / wgs;
    if (s > max_s) s = max_s;
    if (s > 64) s = 64;
    if (s < 1) s = 1;
    pl.n_splits = (int)s;
  } else if (wgs < 4 * (int64_t)cus && members <= cus) {
    const int whole_units = (int)((wgs / cus) * cus / members);
    const int64_t rem_wgs = (int64_t)(units - whole_units) * members;
    if (rem_wgs > 0 && rem_wgs <= cus / 2) {
      int64_t s = cus / rem_wgs;
      if (s > 8) s = 8;
      if (s > max_s / 2) s = max_s / 2;
      if (s > 1) {
        pl.n_splits = (int)s;
        pl.units_whole = whole_units;
      }
    }
  }
  const int split_units = units - pl.units_whole;
  pl.ws_rows = pl.n_splits > 1 ? (int64_t)split_units * group * T : 0;
  return pl;
}

// What a plan takes, us on an MI355X: every XCD works off its share of the (batch, kv head) unit parts
// - a unit's workgroups all run on one - in rounds of a workgroup per CU; then the second pass over the
// partial rows.  Per 64-key tile, per round and per call, with the partial rows' traffic at 3 to 5 TB/s;
// fitted to 860 timings over 46 shapes (2 to 124 heads, 153 to 3600 tokens, 2 to 64 slots, both tile
// sizes, 1 to 24 parts), which it met to 3 to 7 %.  The kernels have become faster since: over 1322 timings
// of 30 shapes the estimate is 3 to 4.5 % high for either tile size and head dim alike, and the choices, which hang
// on its ratios, are as good as they were: 0.8 to 1 % behind the best uniform split on average for bf16.  The
// rows counted are 16-bit ones; an f16 call's are fp32, and its best plan differs little: 1.3 to 1.6 % behind.
inline double plan_cost(const AttnPlan& pl, int B, int H, int Hkv, int T, int Dh, int64_t L) {
  struct Fit { double tile, round, call, comb, comb_mb; };
  static constexpr Fit kFit[2][2] = {{{0.484, 3.94, 2.21, 2.79, 0.215}, {0.733, 3.01, 2.39, 3.39, 0.331}},
                                     {{0.872, 2.64, 3.47, 2.61, 0.208}, {1.307, 1.67, 3.41, 3.57, 0.289}}};
  const Fit& f = kFit[pl.variant == 2][Dh > 64];
  const int64_t units = (int64_t)B * Hkv, members = members_of((int)units, H / Hkv, T, pl.block_m, pl.cus);
  const int64_t nt = (L + 63) / 64, per_xcd = pl.cus / 8 > 0 ? pl.cus / 8 : 1;
  auto rounds = [&](int64_t parts) { return ((parts + 7) / 8 * members + per_xcd - 1) / per_xcd; };
  const int64_t split_units = units - pl.units_whole;
  double c = f.call;
  if (pl.units_whole > 0) c += (double)rounds(pl.units_whole) * (f.tile * (double)nt + f.round);
  c += (double)rounds(split_units * pl.n_splits) * (f.tile * (double)((nt + pl.n_splits - 1) / pl.n_splits) + f.round);
  if (pl.n_splits > 1) c += f.comb + f.comb_mb * 2e-6 * (double)(pl.n_splits * pl.ws_rows) * (Dh * 2 + 16);
  return c;
}

// The plan of a call: the basic choice, or parts for every unit or for the last ones at either tile size
// where the cost above puts that 5 % lower - the basic rules know neither how units fall on the
// XCDs (9 units are two rounds on one of them) nor that a context in three parts can fill two rounds of
// CUs better than one part fills one (144 workgroups).  Against the best of the timings above the basic
// choice was 11 % slower on average (up to 67 %), this one 2 %.  Frames of up to 256 tokens keep to one
// round and ask for 15 %: there the parts' fixed costs are most of the time and the basic rules' finer
// points decide.
inline AttnPlan plan_attn(int B, int H, int Hkv, int T, int Dh, int64_t L, int n_splits, int variant, int cus) {
  AttnPlan best = plan_basic(B, H, Hkv, T, L, n_splits, variant, cus);
  if (n_splits > 0) return best;
  const double basic = plan_cost(best, B, H, Hkv, T, Dh, L);
  // (one pass where every unit was split: no second launch, a saving the estimate is sure of)
  double low = (T <= 256 ? 0.85 : 0.95) * basic, low_single = best.units_whole == 0 ? 0.97 * basic : low;
  const int64_t nt = (L + 63) / 64;
  for (int v = 1; v <= 2; ++v) {
    if (variant != 0 && v != variant) continue;
    if (v == 2 && T <= 128) continue;
    const int block_m = v == 2 ? 256 : 128;
    const int64_t members = members_of(B * Hkv, H / Hkv, T, block_m, best.cus), wgs = (int64_t)B * Hkv * members, per_xcd = best.cus / 8;
    auto consider = [&](int whole, int s) {
      AttnPlan pl;
      pl.variant = v; pl.block_m = block_m; pl.n_splits = s; pl.units_whole = whole; pl.cus = best.cus;
      pl.ws_rows = s > 1 ? ((int64_t)B * Hkv - whole) * (H / Hkv) * T : 0;
      const double c = plan_cost(pl, B, H, Hkv, T, Dh, L);
      if (c < (s == 1 ? low_single : low)) {
        low_single = c;
        low = c < low ? c : low;
        best = pl;
      }
    };
    for (int s = 1; s <= 24 && (s == 1 || nt / s >= 2); ++s) {
      if (s > 1 && wgs * s > (T <= 256 ? best.cus : 8 * (int64_t)best.cus)) break;
      consider(0, s);
    }
    // or only the units behind the last whole round (of every XCD) in parts: fewer partial rows
    for (int r = 1; r <= 3 && T > 256 && members <= r * per_xcd; ++r) {
      const int64_t whole = r * per_xcd / members * 8;
      if (whole >= (int64_t)B * Hkv) break;
      for (int s = 2; s <= 8 && nt / s >= 4; ++s) consider((int)whole, s);
    }
  }
  return best;
}

// plan_attn for callers that ask again and again: a thread keeps its last plans (each layer and frame of
// a model asks twice, and a plan is some fifty cost estimates).  row_bytes: of a partial row, for a call that takes fewer
// parts where that is the faster plan (short_parts.h; it needs less workspace than the plan without, which the sizing
// helpers go by); 0: the plan without.
inline AttnPlan plan_cached(int B, int H, int Hkv, int T, int Dh, int64_t L, int n_splits, int variant, int cus, int row_bytes = 0) {
  struct Entry { int64_t key[10]; AttnPlan plan; };
  static thread_local Entry kept[16] = {};
  const int64_t key[10] = {B, H, Hkv, T, Dh, L, n_splits, variant, cus, row_bytes};
  uint64_t h = 0;
  for (int64_t k : key) h = (h ^ (uint64_t)k) * 0x9e3779b97f4a7c15ull;
  Entry& e = kept[h >> 60];
  for (int i = 0; i < 10; ++i)
    if (e.key[i] != key[i]) {
      e.plan = plan_attn(B, H, Hkv, T, Dh, L, n_splits, variant, cus);
      AttnPlan& pl = e.plan;
      if (row_bytes > 0 && n_splits == 0 && T >= 64 && T <= 256 && pl.variant == 1 && pl.units_whole == 0 && pl.n_splits > 1) {
        const ShortCall call = {(int64_t)B * Hkv, members_of(B * Hkv, H / Hkv, T, pl.block_m, pl.cus), (L + 63) / 64,
                                (int64_t)B * H * T, row_bytes, Dh > 64, pl.cus};
        pl.n_splits = call.parts(pl.n_splits);
        if (pl.n_splits == 1) pl.ws_rows = 0;
      }
      for (int j = 0; j < 10; ++j) e.key[j] = key[j];
      break;
    }
  return e.plan;
}

// Partial rows of 16-bit values, or of fp32 ones (`wide`).
inline size_t workspace_bytes_of(const AttnPlan& pl, int Dh, bool wide = false) {
  if (pl.n_splits <= 1 || pl.ws_rows <= 0) return 0;
  return (size_t)pl.n_splits * (size_t)pl.ws_rows * ((size_t)Dh * (wide ? 4 : 2) + 4 * sizeof(float));
}

// Validation of a we_attn_ring_fwd call, its plan and its kernel parameters.  `cus`: compute units
// of the device the call will run on.  `workspace_limit`: a plan that needs more gives way to the basic one.
inline int prepare_attn(const void* q, const int64_t* q_strides, const void* kv, const uint8_t* written,
                        const int64_t* t_pos, void* out, const int64_t* out_strides, void* workspace,
                        size_t workspace_bytes, int B, int H, int Hkv, int T, int Dh, int64_t L, int dilation,
                        float scale, int n_splits, int q_tile, int dtype, int cus, AttnParams& p, AttnPlan& pl,
                        size_t workspace_limit = SIZE_MAX) {
  if (!q || !q_strides || !kv || !written || !t_pos || !out || !out_strides) return WE_ERR_NULL_POINTER;
  int rc = ring_shape_ok(B, H, Hkv, T, Dh, L, dilation);
  if (rc != WE_OK) return rc;
  if (dtype != WE_DTYPE_BF16 && dtype != WE_DTYPE_F16 && dtype != WE_DTYPE_F32) return WE_ERR_UNSUPPORTED;
  if (Dh != 64 && Dh != 128) return WE_ERR_UNSUPPORTED;
  if (L / T > WE_MAX_SLOTS) return WE_ERR_UNSUPPORTED;
  if ((uint64_t)(L + T) * (uint64_t)Dh * 2u >= (1ull << 32)) return WE_ERR_UNSUPPORTED;  // 32-bit tile offsets
  if (!(scale > 0.f) || n_splits < 0 || n_splits > 64) return WE_ERR_BAD_SHAPE;
  if (variant_of(q_tile) < 0) return WE_ERR_UNSUPPORTED;
  int f32_parts = 1, f32_groups = 1;
  if (dtype == WE_DTYPE_F32) {
    // fp32 caches take a kernel of their own: no given number of parts, no tile choice
    if (n_splits > 1 || H > 65535 || B > 65535) return WE_ERR_UNSUPPORTED;
    // (into parts where the caller leaves that to the library and has given memory for them; not in the library's own,
    // which calls that overlap would share)
    const bool room = n_splits == 0 && workspace && aligned16(workspace) && workspace_limit == SIZE_MAX;
    F32Call call = {(int64_t)B * H, T, L / T / dilation, Dh, cus};
    call.plan(!room ? 0 : (int64_t)(workspace_bytes > (size_t)INT64_MAX ? (size_t)INT64_MAX : workspace_bytes));
    f32_parts = call.parts;
    f32_groups = call.groups;
    n_splits = 1;
  }
  if (!aligned16(q) || !aligned16(kv) || !aligned16(out) || !strides_ok(q_strides, dtype) ||
      !strides_ok(out_strides, dtype))
    return WE_ERR_ALIGNMENT;

  pl = plan_cached(B, H, Hkv, T, Dh, L, n_splits, variant_of(q_tile), cus);
  int64_t keys = L;   // that the plan is for
  if (dilation > 1 && n_splits == 0) {
    // a dilated ring holds frames in one of `dilation` slots only; the sizing helpers do not know of it,
    // so the plan for the keys there are is taken where it needs no more workspace
    const AttnPlan short_ring = plan_cached(B, H, Hkv, T, Dh, L / dilation, 0, variant_of(q_tile), cus);
    if (workspace_bytes_of(short_ring, Dh) <= workspace_bytes_of(pl, Dh)) {
      pl = short_ring;
      keys = L / dilation;
    }
  }
  const size_t given = workspace_bytes < workspace_limit ? workspace_bytes : workspace_limit;
  if (n_splits == 0 && workspace_bytes_of(pl, Dh) > workspace_limit)
    pl = plan_basic(B, H, Hkv, T, L, 0, variant_of(q_tile), cus);
  else if (n_splits == 0 && workspace && aligned16(workspace) && workspace_bytes_of(pl, Dh) <= given)
    // (a workspace that is too short for the plan of the sizing helpers stays too short)
    pl = plan_cached(B, H, Hkv, T, Dh, keys, 0, variant_of(q_tile), cus, Dh * (dtype == WE_DTYPE_F16 ? 4 : 2) + 4 * (int)sizeof(float));
  // An f16 output has the 11 significant bits of a 16-bit partial row itself, which would round it once
  // more: its partial rows are fp32.  (24 heads of 64 on 8, 720 tokens, 16 slots, dilation 2, relative
  // error against 64 bits: one pass 2.93e-4; three parts with fp16 rows 3.50e-4, with fp32 rows 2.93e-4.
  // A bf16 output has 8 bits: 2.347e-3 in one pass, 2.352e-3 with fp16 rows.)  A workspace that holds
  // 16-bit rows only gets the basic plan, which splits less, where it holds that one's.
  bool wide = false;
  if (dtype == WE_DTYPE_F16 && workspace_bytes_of(pl, Dh) > 0 && workspace_bytes_of(pl, Dh) <= given) {
    wide = workspace_bytes_of(pl, Dh, true) <= given;
    if (!wide) {
      const AttnPlan basic = plan_basic(B, H, Hkv, T, L, n_splits, variant_of(q_tile), cus);
      if (workspace_bytes_of(basic, Dh) <= given) {
        pl = basic;
        wide = workspace_bytes_of(pl, Dh, true) <= given;
      }
    }
  }
  const size_t ws_need = workspace_bytes_of(pl, Dh, wide);
  if (ws_need > 0) {
    if (!workspace || !aligned16(workspace)) return WE_ERR_WORKSPACE;
    if (workspace_bytes < ws_need) return WE_ERR_WORKSPACE;
  }

  p.q = q; p.kv = kv; p.written = written; p.t_pos = t_pos; p.out = out;
  p.ws_o = ws_need ? workspace : nullptr;
  p.ws_ml = ws_need ? reinterpret_cast<float*>(static_cast<char*>(workspace) + (size_t)pl.n_splits * (size_t)pl.ws_rows * Dh * (wide ? 4 : 2)) : nullptr;
  p.ws_f32 = wide ? 1 : 0;
  p.qs_b = q_strides[0]; p.qs_h = q_strides[1]; p.qs_t = q_strides[2];
  p.os_b = out_strides[0]; p.os_h = out_strides[1]; p.os_t = out_strides[2];
  p.L = L;
  p.B = B; p.H = H; p.Hkv = Hkv; p.T = T;
  p.n_slots = (int)(L / T); p.dilation = dilation; p.num_buckets = p.n_slots / dilation;
  p.n_splits = pl.n_splits;
  p.units_whole = pl.units_whole;
  p.ws_row0 = (int64_t)B * H * T - pl.ws_rows;
  p.group = H / Hkv;
  bool shared = false;
  p.members = (int)members_of(B * Hkv, p.group, T, pl.block_m, pl.cus, &shared);
  p.q_heads = shared ? 1 : p.group;
  p.unit_splits = pl.units_whole + (B * Hkv - pl.units_whole) * pl.n_splits;
  p.scale_log2 = scale * 1.4426950408889634f;
  pl.f32_groups = f32_groups;
  if (f32_parts > 1) {
    p.n_splits = f32_parts;
    p.ws_o = workspace;
    p.ws_ml = reinterpret_cast<float*>(static_cast<char*>(workspace) + (size_t)f32_parts * (size_t)B * H * T * Dh * 4);
  }
  p.gate = nullptr; p.gs_b = p.gs_h = p.gs_t = 0;
  p.gate_x = nullptr; p.gate_w = nullptr; p.gx_b = p.gx_t = 0;
  p.clock_out = nullptr;
  // the Q tile by DMA: 32-bit row offsets, and rows one stride apart throughout the tile
  p.q_dma = (q_strides[2] > 0 && (uint64_t)T * (shared ? p.group : 1) * (uint64_t)q_strides[2] * 2u < (1ull << 31) &&
             (!shared || q_strides[1] == (int64_t)T * q_strides[2])) ? 1 : 0;

  if ((p.unit_splits + 7) / 8 > 65535 || p.q_heads > 65535 || 8ll * p.members > 0x7fffffff || (int64_t)B * H - (int64_t)pl.units_whole * p.group > 65535)
    return WE_ERR_UNSUPPORTED;  // grid y / z limits of the two launches
  return WE_OK;
}

// The launches of one planned attention call.
inline int launch_attn(const AttnParams& p, const AttnPlan& pl, int Dh, int dtype, hipStream_t st) {
  if (dtype == WE_DTYPE_F32) return launch_attn_ring_f32(p, Dh, pl.f32_groups, pl.cus, st) == hipSuccess ? WE_OK : WE_ERR_LAUNCH;
  const int ksplit = pl.variant == 1 ? 2 : 1;
  hipError_t e;
  if (p.T < 64) e = dtype == WE_DTYPE_BF16 ? launch_attn_ring_short_bf16(p, Dh, ksplit, st) : launch_attn_ring_short_f16(p, Dh, ksplit, st);
  else if (p.q_heads != p.group) e = dtype == WE_DTYPE_BF16 ? launch_attn_ring_shared_bf16(p, Dh, ksplit, st) : launch_attn_ring_shared_f16(p, Dh, ksplit, st);
  else if (dtype == WE_DTYPE_BF16) e = Dh == 128 ? launch_attn_ring_bf16_128(p, ksplit, st) : launch_attn_ring_bf16_64(p, ksplit, st);
  else e = Dh == 128 ? launch_attn_ring_f16_128(p, ksplit, st) : launch_attn_ring_f16_64(p, ksplit, st);
  if (e != hipSuccess) return WE_ERR_LAUNCH;
  if (pl.n_splits > 1 && launch_attn_combine(p, Dh, dtype, st) != hipSuccess) return WE_ERR_LAUNCH;
  return WE_OK;
}

}  // namespace host
}  // namespace we
