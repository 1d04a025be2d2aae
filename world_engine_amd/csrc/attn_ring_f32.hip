// fp32 attention over the KV ring buffer (gfx950): the same visibility rule and ring walk as the
// half-precision kernel (attn_ring.hip), scores, softmax and P V as exact as fp32 products and sums make them
// (src/model/attn.py:116 in eager mode).
//
// One workgroup = one or two groups of 16 queries of one (batch, head) and NW wavefronts that share out its keys: blocks
// of 16 keys go round the wavefronts, each keeps its own running (reference, sum, O) and they merge
// through LDS at the end.  A wavefront's keys are nobody else's, so K and V go from memory straight
// into registers, one block ahead, without a barrier in the loop.
//
// Most products go through the f16 matrix instructions, sixteen times the fp32 ones' rate, as sums of two
// halves (x = hi + lo, 22 bits; four products per pair).  S^T = K Q^T: K comes row by row - whole lines; read
// in the operands' layout every request touches 64 of them - and changes places between the lanes through the
// wavefront's own 8 KB of LDS, halved.  O^T += V^T P^T: the S^T accumulators are the B operand as they are (lane
// group g, register i = key 4 g + i), and one instruction's 32 places take 16 keys' hi and lo of V.  What a
// product of these instructions adds is cut off at the last bit of the largest one in its group of eight, and
// so is the sum it is carried into where that is smaller: the large products of S start from zero each and
// O's are added by the vector unit, so that no chain of products loses more than its own size.  f16 numbers
// have a smallest step: what is halved is scaled so that its halves are 22 bits (2^-21 at worst) of every single key,
// value and probability that counts, or goes through fp32 products (queries, values and probabilities below).
// Relative error against 64 bits, fp32 products / halves, normal inputs: 16 heads of 128, 2048 keys 3.9e-7 / 2.3e-7, 8 heads,
// 4096 keys 6.3e-7 / 2.7e-7, 4 heads, 128 keys 2.5e-7 / 1.8e-7; heads of 64, 2880 keys 5.2e-7 / 2.6e-7, 1024 keys 2.9e-7 / 2.1e-7.
//
// Blocks through v_mfma_f32_16x16x4_f32: the contraction of S is taken in an order that lets a lane load four of its
// head-dim values at once (lane group g of step (j, i) has value 16 j + 4 g + i of both operands), and output rows
// are numbered so that a lane's four values of V are consecutive: one 16-byte load per key and 64 head-dim values.
//
// Bound by the vector unit and the trips through LDS: at 16 queries a workgroup every CU halves all of its unit's keys and
// values itself, half of a block's vector instructions.  Where that is more than a workgroup a CU, two groups share what is
// halved (some 370 instructions a block for both, which issue 60 % of the time of 8 heads, 1024 queries, 4096 keys, beside 64
// f16 MFMAs of 16 cycles, 33 %).  us in one pass, fp32 products / halves: 16 heads of 128, 256 queries, 2048 keys 44.9 / 36.1 (119
// TFLOP/s), 8 heads of 128, 64 queries, 512 keys 17.0 / 13.5, 4 heads, 128 keys 9.0 / 8.7; of two groups: 8 heads, 1024 queries, 4096
// keys 151 / 94 (183 TFLOP/s, where a large fp32 matrix product reaches 153), 24 heads of 64 on 8, 720 queries, 2880 keys 136 / 99,
// 16 heads, 272 queries, 2176 keys 83 / 50.7.  Other inputs, first and fourth shape: values of standard deviation 0.05 36.9 and
// 96, queries of 30 37.1 and 96; queries of 1e4 in one channel, which take fp32 products, 46.9 and 156; values above 65504,
// for which a wavefront does everything a second time, 71 and 225.
#include <type_traits>

#include "attn_mma.h"
#include "device_state.h"
#include "f32_parts.h"
#include "we_kernels.h"
#include "../../include/we_attn.h"

namespace we {

namespace {
constexpr int F_Q = 16;   // queries of a group
constexpr int F_K = 16;   // keys per block
constexpr int K_UP = 5;          // exponent of the scale for the keys of large queries
constexpr float Q_MOST = 4.f;    // 2-norm of a query, times scale * log2(e) (normalised queries: 1.44)
constexpr int P_UP = 15;         // exponent of the scale for a block's probabilities
constexpr float M_SLACK = 8.f;   // how far above the running reference a logit may be

// NQ: groups of queries per workgroup
template <int DH, int NW, int NQ, bool SPLIT>
struct F32Lds {
  static constexpr int OROW = DH + 4;   // floats per row of a wavefront's O (the odd 16 bytes spread the banks)
  static constexpr int NOUT = NW / 2;   // wavefronts whose O is there at a time
  static constexpr int KROW = DH * 2 + 16;                  // bytes per key, halved (the odd 16 spread the banks)
  static constexpr int kWave = SPLIT ? 2 * F_K * KROW : 0;  // a wavefront's block of keys: [hi, lo][key][value]
  static constexpr int kOut = NOUT * NQ * F_Q * OROW * 4;
  static constexpr int kMl = NW * kWave > kOut ? NW * kWave : kOut;                        // references, sums
  static constexpr int kQ = kMl + 2 * NW * NQ * F_Q * 4;                                   // queries: [group][hi, lo][step][lane] 16 bytes,
  static constexpr int kBack = kQ + (SPLIT && NQ > 1 ? NQ * F_Q * DH * 4 : 0);             // what undoes their scaling
  static constexpr int kVis = kBack + (SPLIT && NQ > 1 ? NQ * F_Q * 4 : 0);
  static constexpr int kBytes = kVis + (WE_MAX_SLOTS + 2) * 4;
};
}  // namespace

struct F32Params {
  AttnParams a;
  int halves_from;   // blocks of visible keys from which on they go in halves
};

// maximum / sum over the four 16-lane groups of a wavefront, for each lane position in a group
__device__ __forceinline__ float groups_max(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float y = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  float lo, up;
  half_wave_pair(y, lo, up);
  return fmaxf(lo, up);
}
__device__ __forceinline__ float groups_sum(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float y = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  float lo, up;
  half_wave_pair(y, lo, up);
  return lo + up;
}

typedef float float2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t f16_pair(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2_t{a, b}), f16x2_t));
}
// Four fp32 values as sums of two f16 ones: rounded (hi), and what that leaves, rounded; or both `up` times as large (a power of
// two, f16_pow2).  All at the full rate, which conversions to one half of a register (v_fma_mixlo_f16) do not have: 36.9 -> 42
// us for the first shape above.
struct Halves4 {
  u32x2_t hi, lo;
  __device__ __forceinline__ Halves4(float a, float b, float c, float d) : Halves4(a, b, c, d, f16_pair(a, b), f16_pair(c, d), 1.f) {}
  __device__ __forceinline__ Halves4(float a, float b, float c, float d, float up, uint32_t up16)
      : Halves4(a, b, c, d, times(f16_pair(a, b), up16), times(f16_pair(c, d), up16), up) {}

 private:
  static __device__ __forceinline__ uint32_t times(uint32_t h, uint32_t by) {
    uint32_t y;
    asm("v_pk_mul_f16 %0, %1, %2" : "=v"(y) : "v"(h), "s"(by));
    return y;
  }
  __device__ __forceinline__ Halves4(float a, float b, float c, float d, uint32_t h0, uint32_t h1, float up) : hi{h0, h1} {
    float r[4];
    asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(r[0]) : "v"(a), "s"(up), "v"(h0));
    asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(r[1]) : "v"(b), "s"(up), "v"(h0));
    asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(r[2]) : "v"(c), "s"(up), "v"(h1));
    asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(r[3]) : "v"(d), "s"(up), "v"(h1));
    lo = u32x2_t{f16_pair(r[0], r[1]), f16_pair(r[2], r[3])};
  }
};
// eight f16 values: the four of `a` and the four of `b`
__device__ __forceinline__ f16x8_t f16x8_of(u32x2_t a, u32x2_t b) {
  return __builtin_bit_cast(f16x8_t, (u32x4_t{a[0], a[1], b[0], b[1]}));
}
// 2^e, -126 <= e <= 127
__device__ __forceinline__ float pow2(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }
// twice in f16, -14 <= e <= 15
__device__ __forceinline__ uint32_t f16_pow2(int e) { return (uint32_t)(e + 15) * 0x04000400u; }
__device__ __forceinline__ float max_abs3(float m, float a, float b) {
  asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(a), "v"(b));
  return m;
}
__device__ __forceinline__ float min_abs3(float m, float a, float b) {
  asm("v_min3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(a), "v"(b));
  return m;
}
// the largest x >= 0 of a wavefront
template <int ROR>
__device__ __forceinline__ float max_ror(float x) {
  return fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x120 | ROR, 0xf, 0xf, false)));
}
__device__ __forceinline__ float wave_max(float x) {
  x = max_ror<1>(max_ror<2>(max_ror<4>(max_ror<8>(groups_max(x)))));
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

// WHOLE: T % 16 == 0, every block has 16 keys (a separate instance: what the others work out per request is a tenth of a
// block's vector instructions).
template <int DH, int NW, int NQ, bool SPLIT, bool WHOLE>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2)))
attn_ring_f32_kernel(F32Params fp) {
  const AttnParams& p = fp.a;
  constexpr int NJ = DH / 16;    // 16-byte loads of K per lane and block
  constexpr int NH = DH / 64;    // 16-byte loads of V per lane and key
  constexpr int OROW = F32Lds<DH, NW, NQ, SPLIT>::OROW, NOUT = F32Lds<DH, NW, NQ, SPLIT>::NOUT;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  typedef F32Lds<DH, NW, NQ, SPLIT> Lds;
  constexpr int BQ = NQ * F_Q;   // queries per workgroup
  float(*osh)[BQ][OROW] = reinterpret_cast<float(*)[BQ][OROW]>(smem);   // (behind the loops: where the wavefronts' keys were)
  float(*msh)[BQ] = reinterpret_cast<float(*)[BQ]>(smem + Lds::kMl);
  float(*lsh)[BQ] = msh + NW;
  f16x8_t* qsh = reinterpret_cast<f16x8_t*>(smem + Lds::kQ);
  float* back = reinterpret_cast<float*>(smem + Lds::kBack);
  int* vis = reinterpret_cast<int*>(smem + Lds::kVis);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;

  // ---- which queries, which part of the keys ----
  // (spread over the XCDs by unit part where every XCD gets the same number: its workgroups share an L2)
  const int q_tiles = (p.T + BQ - 1) / BQ;
  unsigned up, member;
  const int n_parts = SPLIT ? p.n_splits : 1;   // (F32Call::plan: parts in halves only)
  if (((p.B * p.Hkv * n_parts) & 7) == 0) {
    const unsigned j = blockIdx.x >> 3;
    const unsigned u8 = j / (unsigned)p.members;
    up = u8 * 8 + (blockIdx.x & 7);
    member = j - u8 * (unsigned)p.members;
  } else {
    up = blockIdx.x / (unsigned)p.members;
    member = blockIdx.x - up * (unsigned)p.members;
  }
  int unit = (int)up, part = 0;
  if (n_parts > 1) {
    unit = (int)(up / (unsigned)n_parts);
    part = (int)(up - (unsigned)unit * (unsigned)n_parts);
  }
  const int b = unit / p.Hkv, hkv = unit - b * p.Hkv;
  const int hq_in = (int)member / q_tiles, h = hkv * p.group + hq_in;
  const int q0 = ((int)member - hq_in * q_tiles) * BQ;

  // ---- list of visible slots; the tail is pseudo-slot n_slots ----
  if (wave == 0) {
    const SlotInfo si = ring_slot(p.t_pos[0], p.dilation, p.num_buckets);
    int count = 0;
    for (int base = 0; base < p.n_slots; base += 64) {
      const int s = base + lane;
      bool f = false;
      if (s < p.n_slots) f = (p.written[(int64_t)s * p.T] != 0) && !(si.write_step && s == si.slot);
      const unsigned long long m = __ballot(f);
      if (f) vis[count + __popcll(m & ((1ull << lane) - 1ull))] = s;
      count += __popcll(m);
    }
    if (lane == 0) {
      vis[count] = p.n_slots;
      vis[WE_MAX_SLOTS + 1] = count + 1;
    }
  }

  auto query = [&](int qi) __attribute__((always_inline)) {
    const int qr = q0 + qi * F_Q + c < p.T ? q0 + qi * F_Q + c : p.T - 1;
    return reinterpret_cast<const float*>(p.q) + b * p.qs_b + h * p.qs_h + (int64_t)qr * p.qs_t;
  };
  // ---- query c of a group, values 16 j + 4 g + i, pre-multiplied by scale * log2(e) ----
  f32x4_t qf[NJ];
  auto load_q = [&](int qi) __attribute__((always_inline)) {
    const float* row = query(qi);
#pragma unroll
    for (int j = 0; j < NJ; ++j) qf[j] = *reinterpret_cast<const f32x4_t*>(row + 16 * j + 4 * g) * p.scale_log2;
  };
  if (!SPLIT) load_q(0);
  // ---- or in halves, values 32 j + 8 g + i, and by a power of two that brings the row's largest value to 2^14 .. 2^15; in
  // registers, or where there are several groups in LDS ----
  // A key's halves are off by up to 2^-22 of it and by up to 2^-25 (half the smallest f16 number).  Under a query of norm Q_MOST
  // the latter moves a logit by 2^-24 or so, as far as an exponential is off.  For larger queries keys are halved 2^K_UP times
  // as large, and beyond that there are fp32 products: q x 1e3 and k / 1e3 in one channel gave errors of 2e-6, 1e6 of 2e-3,
  // while the largest key of a few channels and keys stood for all (3 to 5e-7 now, as with fp32 products).
  f16x8_t q_hi[NJ / 2], q_lo[NJ / 2];
  float q_back[NQ];    // what undoes the queries' and the keys' scales
  bool split = false, scale_keys = false;
  auto halve_q = [&](int qi, float& undo) __attribute__((always_inline)) {
    const float* row = query(qi);
    float top = 0.f, square = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) qf[j] = *reinterpret_cast<const f32x4_t*>(row + 32 * (j / 2) + 8 * g + 4 * (j & 1)) * p.scale_log2;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      top = max_abs3(max_abs3(top, qf[j][0], qf[j][1]), qf[j][2], qf[j][3]);
      square += (qf[j][0] * qf[j][0] + qf[j][1] * qf[j][1]) + (qf[j][2] * qf[j][2] + qf[j][3] * qf[j][3]);
    }
    top = groups_max(top);
    int e = 15 - __builtin_amdgcn_frexp_expf(top);
    e = e < 100 ? e : 100;
    square = groups_sum(square);
    undo = __builtin_amdgcn_ldexpf(1.f, -e);
    if (!(square <= Q_MOST * Q_MOST)) undo = square <= Q_MOST * Q_MOST * pow2(2 * K_UP) ? -undo : INFINITY;   // (NaN: not halved)
#pragma unroll
    for (int j = 0; j < NJ; ++j) qf[j] *= __builtin_amdgcn_ldexpf(1.f, e);
#pragma unroll
    for (int j = 0; j < NJ / 2; ++j) {
      const Halves4 a(qf[2 * j][0], qf[2 * j][1], qf[2 * j][2], qf[2 * j][3]);
      const Halves4 b(qf[2 * j + 1][0], qf[2 * j + 1][1], qf[2 * j + 1][2], qf[2 * j + 1][3]);
      q_hi[j] = f16x8_of(a.hi, b.hi);
      q_lo[j] = f16x8_of(a.lo, b.lo);
    }
  };
  if (SPLIT && NQ == 1) halve_q(0, q_back[0]);
  if (SPLIT && NQ > 1 && wave >= 1 && wave <= NQ) {
    float undo;
    halve_q(wave - 1, undo);
    if (g == 0) back[(wave - 1) * F_Q + c] = undo;
#pragma unroll
    for (int j = 0; j < NJ / 2; ++j) {
      qsh[((wave - 1) * NJ + j) * 64 + lane] = q_hi[j];
      qsh[((wave - 1) * NJ + NJ / 2 + j) * 64 + lane] = q_lo[j];
    }
  }
  __syncthreads();
  const int nvis = vis[WE_MAX_SLOTS + 1];
  if (SPLIT) {
    float most = -INFINITY, least = INFINITY;
#pragma unroll
    for (int qi = 0; qi < NQ; ++qi) {
      if (NQ > 1) q_back[qi] = back[qi * F_Q + c];
      most = fmaxf(most, q_back[qi]);
      least = fminf(least, q_back[qi]);
    }
    split = __ballot(!(most < INFINITY)) == 0ull;
    scale_keys = __ballot(least < 0.f) != 0ull;
#pragma unroll
    for (int qi = 0; qi < NQ; ++qi) q_back[qi] = __builtin_fabsf(q_back[qi]) * (scale_keys ? pow2(-K_UP) : 1.f);
  }

  f32x4_t o[NQ][NH][4];  // o[qi][hh][e] register i: query c of group qi, value 64 hh + 16 g + 4 i + e
  float m_run[NQ], l_run[NQ];  // (l_run: this lane group's keys only)
  auto nothing_yet = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int qi = 0; qi < NQ; ++qi) {
      m_run[qi] = -INFINITY;
      l_run[qi] = 0.f;
#pragma unroll
      for (int hh = 0; hh < NH; ++hh)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[qi][hh][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
  };
  nothing_yet();

  const int64_t cap = p.L + p.T;
  const float* kplane = reinterpret_cast<const float*>(p.kv) + (((int64_t)b * p.Hkv + hkv) * cap) * DH;
  const float* vplane = kplane + (int64_t)p.B * p.Hkv * cap * DH;

  // Blocks go round the wavefronts in rounds of NW.  The workgroups that share a K/V stream take the
  // rounds in groups of rot_g, member m starting at round m of every group: they then ask for
  // different lines at any one time, and each line comes from memory at one member's request (184
  // against 192 us for 8 heads, 1024 queries, 4096 keys when they took 184; groups of 8 or 16: the same, then and now).
  const int bps = (p.T + F_K - 1) / F_K;  // blocks per slot; the last one may be short
  const int all_blk = nvis * bps;
  int blk0 = 0, nblk = all_blk;
  if (n_parts > 1) {
    blk0 = (int)((unsigned)part * (unsigned)all_blk / (unsigned)n_parts);
    nblk = (int)((unsigned)(part + 1) * (unsigned)all_blk / (unsigned)n_parts) - blk0;
  }
  const int rounds = (nblk + NW - 1) / NW;
  int rot_g = 1;
  while (rot_g * 2 <= p.members && rot_g < 4) rot_g *= 2;
  const int rot_end = (nblk / NW) & ~(rot_g - 1);
  auto block_of = [&](int k) __attribute__((always_inline)) {
    const int kk = k < rot_end ? (k & ~(rot_g - 1)) | ((k + (int)member) & (rot_g - 1)) : k;
    return blk0 + kk * NW + wave;
  };

  // (uniform base and 32-bit lane offsets; rows past the frame repeat its last one)
  struct Place {
    int64_t row0;
    int last;   // its last key
  };
  auto place = [&](int k) __attribute__((always_inline)) {
    const int at = block_of(k), vi = (int)((unsigned)at / (unsigned)bps), sub = at - vi * bps;
    return Place{(int64_t)__builtin_amdgcn_readfirstlane(vis[vi]) * p.T + sub * F_K, p.T - 1 - sub * F_K};
  };
  auto load_k = [&](f32x4_t(&kf)[NJ], Place at) __attribute__((always_inline)) {
    const char* kb = reinterpret_cast<const char*>(kplane + at.row0 * DH);
    const uint32_t ko = (uint32_t)((c < at.last ? c : at.last) * DH + 4 * g) * 4u;
#pragma unroll
    for (int j = 0; j < NJ; ++j) kf[j] = *reinterpret_cast<const f32x4_t*>(kb + ko + 64 * j);
  };
  auto load_v = [&](f32x4_t(&vf)[4][NH], Place at) __attribute__((always_inline)) {
    const char* vb = reinterpret_cast<const char*>(vplane + at.row0 * DH);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t vo = (uint32_t)((4 * g + i < at.last ? 4 * g + i : at.last) * DH + 4 * c) * 4u;
#pragma unroll
      for (int hh = 0; hh < NH; ++hh) vf[i][hh] = *reinterpret_cast<const f32x4_t*>(vb + vo + 256 * hh);
    }
  };
  auto block = [&](auto group, const f32x4_t(&kf)[NJ], f32x4_t(&vf)[4][NH], int keys) __attribute__((always_inline)) {
    constexpr int qi = decltype(group)::value;
    f32x4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NJ; j += 2)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][i], qf[j][i], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j + 1][i], qf[j + 1][i], s1, 0, 0, 0);
      }
    // (the next block's loads go out between these products: together they keep a wavefront from issuing anything
    // else while the CU's address path takes them, 45.5 against 47.0 us for 16 heads of 128, 256 queries, 2048 keys)
#pragma unroll
    for (int i = 0; i < NJ + 4 * NH; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x8, 4 * NJ / (NJ + 4 * NH), 0);
    }
    f32x4_t s = s0 + s1;
    if (keys < F_K) {  // missing keys: no weight, and nothing for a zero weight to meet but zeros
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (4 * g + i >= keys) {
          s[i] = -INFINITY;
#pragma unroll
          for (int hh = 0; hh < NH; ++hh) vf[i][hh] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    }
    const float mx = fmaxf(m_run[qi], groups_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
    if (__ballot(mx != m_run[qi]) != 0ull) {
      const float alpha = __builtin_amdgcn_exp2f(m_run[qi] - mx);  // 0 on the first block
      l_run[qi] *= alpha;
#pragma unroll
      for (int hh = 0; hh < NH; ++hh)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[qi][hh][e] *= alpha;
      m_run[qi] = mx;
    }
    f32x4_t pr;
#pragma unroll
    for (int i = 0; i < 4; ++i) pr[i] = __builtin_amdgcn_exp2f(s[i] - mx);
    l_run[qi] += (pr[0] + pr[1]) + (pr[2] + pr[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int hh = 0; hh < NH; ++hh)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[qi][hh][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][hh][e], pr[i], o[qi][hh][e], 0, 0, 0);
    // (two blocks in a row are not scheduled as one: 44.4 against 46.8 us for the same shape)
    __builtin_amdgcn_sched_barrier(0);
  };
  const int mine_n = rounds - (nblk - (rounds - 1) * NW > wave ? 0 : 1);  // rounds this wavefront takes part in
  auto fetch = [&](f32x4_t(&kf)[NJ], f32x4_t(&vf)[4][NH], int k) __attribute__((always_inline)) {
    const Place at = place(k);
    load_k(kf, at);
    load_v(vf, at);
    return at.last + 1;  // keys of the block (16 or more: a whole one)
  };

  // ---- blocks whose values two f16 halves hold ----
  int k = 0;
  if (SPLIT && split && all_blk >= fp.halves_from && mine_n > 0) {
    // The keys come row by row, whole cache lines a request, and change places with the other lanes' through LDS, halved.
    constexpr int CPR = DH / 4, RPL = 64 / CPR;   // 16-byte chunks per row, rows per request
    unsigned char* const k_to = smem + wave * Lds::kWave + (lane / CPR) * Lds::KROW + (lane % CPR) * 8;
    const unsigned char* const k_from = smem + wave * Lds::kWave + c * Lds::KROW + g * 16;
    f32x4_t kf[NJ], vf[4][NH];
    // (offsets of the lanes that are known here only: a uniform base and these, no vector addresses kept)
    auto load_rows = [&](Place at) __attribute__((always_inline)) {
      typedef const __attribute__((address_space(1))) char* bytes_t;
      bytes_t kb = (bytes_t)(kplane + at.row0 * DH), kb4 = kb + 4096;
      uint32_t l = (uint32_t)lane;
      asm volatile("" : "+v"(l), "+s"(kb4));
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        if (WHOLE) {
          kf[j] = *reinterpret_cast<const __attribute__((address_space(1))) f32x4_t*>((j < 4 ? kb + 1024 * j : kb4 + 1024 * (j - 4)) + l * 16u);
        } else {
          const int r = RPL * j + (int)(l / CPR);
          kf[j] = *reinterpret_cast<const __attribute__((address_space(1))) f32x4_t*>(kb + (uint32_t)((r < at.last ? r : at.last) * DH + 4 * (int)(l % CPR)) * 4u);
        }
      }
    };
    auto load_values = [&](Place at) __attribute__((always_inline)) {
      const char* vb = reinterpret_cast<const char*>(vplane + at.row0 * DH);
      uint32_t l = (uint32_t)lane;
      asm volatile("" : "+v"(l));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 4 * (int)(l >> 4) + i;
#pragma unroll
        for (int hh = 0; hh < NH; ++hh) {
          if (WHOLE) vf[i][hh] = *reinterpret_cast<const f32x4_t*>(vb + DH * 4 * i + 256 * hh + ((l >> 4) * (DH * 16) + (l & 15) * 16));
          else vf[i][hh] = *reinterpret_cast<const f32x4_t*>(vb + (uint32_t)((r < at.last ? r : at.last) * (DH * 4) + (int)(l & 15) * 16) + 256 * hh);
        }
      }
    };
    Place at = place(0);
    load_rows(at);
    load_values(at);
    // Values are halved 2^e times as large, which brings the largest of a wavefront's first block to 2^12 .. 2^13 (e up to 13:
    // should that block be empty, the next may have values of 8).  Halves are then off by up to 2^-22 of a value and by up to
    // 2^-25, which is 2^-21 of 2^-4.  Tiles of 16 keys and 16 channels with a smaller value take fp32 products, one block in twenty of
    // normal values has one.  By value: an output channel is a sum over keys only, and nearly all weight may be on one of them.
    // While the largest of a lane's values stood for all, a channel times 1e-4 was off by 3e-4 of itself, a row that looks at
    // one key with values times 1e-4 by 2e-4 (4e-7 to 1e-6 and 5e-7 to 2e-6 now, as with fp32 products).
    // (Keys and values too large for f16 are infinite and their rest the other infinity: what they meet is no number, at the end.)
    float v_up = 0.f, v_back = 0.f, v_low = 0.f;
    uint32_t v_up16 = 0;
    auto scale_values = [&]() __attribute__((always_inline)) {
      float top = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int hh = 0; hh < NH; ++hh) top = max_abs3(max_abs3(top, vf[i][hh][0], vf[i][hh][1]), vf[i][hh][2], vf[i][hh][3]);
      int e = 139 - (int)(__float_as_uint(wave_max(top)) >> 23);
      e = e < -14 ? -14 : (e > 13 ? 13 : e);
      v_up = pow2(e);
      v_up16 = f16_pow2(e);
      v_back = pow2(-e - P_UP);
      v_low = pow2(-e - 4);
    };
    auto values_fit = [&]() __attribute__((always_inline)) {
      float least = INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int hh = 0; hh < NH; ++hh) least = min_abs3(min_abs3(least, vf[i][hh][0], vf[i][hh][1]), vf[i][hh][2], vf[i][hh][3]);
      return __ballot(least < v_low) == 0ull;
    };
    f32x4_t s[NQ];   // logits / q_back
    int keys = 0;
    auto logits = [&](auto more) __attribute__((always_inline)) {
      auto to_lds = [&](int j, auto scaled) __attribute__((always_inline)) {
        const f32x4_t r = kf[j];
        const Halves4 x = decltype(scaled)::value ? Halves4(r[0], r[1], r[2], r[3], pow2(K_UP), f16_pow2(K_UP))
                                                  : Halves4(r[0], r[1], r[2], r[3]);
        *reinterpret_cast<u32x2_t*>(k_to + RPL * j * Lds::KROW) = x.hi;
        *reinterpret_cast<u32x2_t*>(k_to + (F_K + RPL * j) * Lds::KROW) = x.lo;
      };
      if (__builtin_expect(scale_keys, 0)) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) to_lds(j, std::true_type());
      } else {
#pragma unroll
        for (int j = 0; j < NJ; ++j) to_lds(j, std::false_type());
      }
      asm volatile("" ::: "memory");
      keys = at.last + 1;   // (16 or more: a whole block)
      // (the large products one by one, the others on top of each other: a sum that is carried from product to product
      // loses the bits that hang over the products')
      f32x4_t sh[NQ][NJ / 2], sl[NQ];
      int lane_q = lane;   // (the queries are read anew for every block: no registers to keep them in)
      if (NQ > 1) asm volatile("" : "+v"(lane_q));
#pragma unroll
      for (int qi = 0; qi < NQ; ++qi) sl[qi] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NJ / 2; ++j) {
        const f16x8_t k_hi = *reinterpret_cast<const f16x8_t*>(k_from + 64 * j);
        const f16x8_t k_lo = *reinterpret_cast<const f16x8_t*>(k_from + F_K * Lds::KROW + 64 * j);
#pragma unroll
        for (int qi = 0; qi < NQ; ++qi) {
          const f16x8_t qh = NQ > 1 ? qsh[(qi * NJ + j) * 64 + lane_q] : q_hi[j];
          const f16x8_t ql = NQ > 1 ? qsh[(qi * NJ + NJ / 2 + j) * 64 + lane_q] : q_lo[j];
          sh[qi][j] = F16Mma::mma16(k_hi, qh, f32x4_t{0.f, 0.f, 0.f, 0.f});
          sl[qi] = F16Mma::mma16(k_lo, ql, sl[qi]);
          sl[qi] = F16Mma::mma16(k_lo, qh, sl[qi]);
          sl[qi] = F16Mma::mma16(k_hi, ql, sl[qi]);
        }
        if (NQ > 1) __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("" ::: "memory");
      if (decltype(more)::value) {
        at = place(k + 1);
        load_rows(at);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[qi][i] = sh[qi][0][i] + sh[qi][1][i];
          if (NJ == 8) s[qi][i] += sh[qi][NJ / 2 - 2][i] + sh[qi][NJ / 2 - 1][i];
          s[qi][i] += sl[qi][i];
        }
    };
    auto outputs = [&]() __attribute__((always_inline)) {
      if (!WHOLE && keys < F_K) {  // missing keys: no weight (their values are the last key's)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int qi = 0; qi < NQ; ++qi) s[qi][i] = 4 * g + i < keys ? s[qi][i] : -INFINITY;
      }
      // Probabilities are relative to the block's largest (and near 1 lose nothing in the exponent's subtraction), of which their halves are off
      // by up to 2^-40: the keys next to one that has nearly all weight, but no value to speak of, keep their bits.  `part`
      // takes the block's sums to the running reference.
      const bool fit = values_fit();
      f32x4_t pr[NQ];
      float part[NQ];
#pragma unroll
      for (int qi = 0; qi < NQ; ++qi) {
        const float top = groups_max(fmaxf(fmaxf(s[qi][0], s[qi][1]), fmaxf(s[qi][2], s[qi][3]))) * q_back[qi];
        if (__ballot(top > m_run[qi] + M_SLACK) != 0ull) {
          const float mx = fmaxf(m_run[qi], top), alpha = __builtin_amdgcn_exp2f(m_run[qi] - mx);  // 0 on the first block
          l_run[qi] *= alpha;
#pragma unroll
          for (int hh = 0; hh < NH; ++hh)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[qi][hh][e] *= alpha;
          m_run[qi] = mx;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) pr[qi][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[qi][i], q_back[qi], -top));
        part[qi] = __builtin_amdgcn_exp2f(top - m_run[qi]);
        l_run[qi] += ((pr[qi][0] + pr[qi][1]) + (pr[qi][2] + pr[qi][3])) * part[qi];
      }
      if (__builtin_expect(!fit, 0)) {   // (then zeros to the products below: a branch around them would move o from registers to registers)
        f32x4_t w[NQ];
#pragma unroll
        for (int qi = 0; qi < NQ; ++qi) w[qi] = pr[qi] * part[qi];
#pragma unroll
        for (int hh = 0; hh < NH; ++hh)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float least = min_abs3(min_abs3(INFINITY, vf[0][hh][e], vf[1][hh][e]), vf[2][hh][e], vf[3][hh][e]);
            if (__ballot(least < v_low) != 0ull) {
#pragma unroll
              for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int qi = 0; qi < NQ; ++qi) o[qi][hh][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][hh][e], w[qi][i], o[qi][hh][e], 0, 0, 0);
                vf[i][hh][e] = 0.f;
              }
            }
          }
      }
      f16x8_t p_hi[NQ], p_lo[NQ];
#pragma unroll
      for (int qi = 0; qi < NQ; ++qi) {
        const Halves4 x(pr[qi][0], pr[qi][1], pr[qi][2], pr[qi][3], pow2(P_UP), f16_pow2(P_UP));
        p_hi[qi] = f16x8_of(x.hi, x.hi);
        p_lo[qi] = f16x8_of(x.lo, x.lo);
        part[qi] *= v_back;
      }
#pragma unroll
      for (int hh = 0; hh < NH; ++hh) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // value 64 hh + 4 c + e of the lane's four keys: rounded, and the rest
          const Halves4 x(vf[0][hh][e], vf[1][hh][e], vf[2][hh][e], vf[3][hh][e], v_up, v_up16);
          const f16x8_t v = f16x8_of(x.hi, x.lo);
#pragma unroll
          for (int qi = 0; qi < NQ; ++qi) {
            const f32x4_t d = F16Mma::mma16(v, p_hi[qi], F16Mma::mma16(v, p_lo[qi], f32x4_t{0.f, 0.f, 0.f, 0.f}));
#pragma unroll
            for (int i = 0; i < 4; ++i) o[qi][hh][e][i] += d[i] * part[qi];
          }
        }
      }
      // (the next block is not looked at, and waited for, in front of these products)
      __builtin_amdgcn_sched_barrier(0);
      ++k;
    };
    auto block_of_halves = [&](auto more) __attribute__((always_inline)) {
      logits(more);
      if (k == 0) scale_values();
      outputs();
      if (decltype(more)::value) load_values(at);
    };
    while (k + 1 < mine_n) block_of_halves(std::true_type());
    block_of_halves(std::false_type());
    float all = 0.f;
#pragma unroll
    for (int qi = 0; qi < NQ; ++qi) {
      all += l_run[qi];
#pragma unroll
      for (int hh = 0; hh < NH; ++hh)
#pragma unroll
        for (int e = 0; e < 4; ++e) all += (o[qi][hh][e][0] + o[qi][hh][e][1]) + (o[qi][hh][e][2] + o[qi][hh][e][3]);
    }
    if (__ballot(!(__builtin_fabsf(all) < INFINITY)) != 0ull) {  // all of it once more
      k = 0;
      nothing_yet();
    }
  }

  // ---- or all blocks through fp32 products ----
  auto others = [&](auto group) __attribute__((always_inline)) {
    if (SPLIT) load_q(decltype(group)::value);
    f32x4_t ka[NJ], va[4][NH], kb[NJ], vb[4][NH];
    // The loop always requests the next block - behind a branch the compiler counts the loads in flight as if it had
    // not been taken, and waits for the block just requested - and the last one or two blocks follow it.  (A last block
    // requested a second time, for nothing, costs wavefronts with one or two of them most: attention alone, 4 heads of 128,
    // 64 queries, 128 keys 9.8 -> 8.75 us, 8 heads, 256 keys 12.25 -> 11.4, 8 heads of 64, 256 keys 7.64 -> 7.40, 128 keys
    // 6.43 -> 6.11.)
    int k = 1;
    int keys_a = fetch(ka, va, 0);
    for (; k + 1 < mine_n; k += 2) {
      const int keys_b = fetch(kb, vb, k);
      block(group, ka, va, keys_a);
      keys_a = fetch(ka, va, k + 1);
      block(group, kb, vb, keys_b);
    }
    if (k < mine_n) {
      const int keys_b = fetch(kb, vb, k);
      block(group, ka, va, keys_a);
      block(group, kb, vb, keys_b);
    } else {
      block(group, ka, va, keys_a);
    }
  };
  if (k < mine_n) {
    others(std::integral_constant<int, 0>());
    if constexpr (NQ > 1) others(std::integral_constant<int, 1>());
  }

  // ---- the wavefronts merge ----
#pragma unroll
  for (int qi = 0; qi < NQ; ++qi) {
    l_run[qi] = groups_sum(l_run[qi]);
    if (g == 0) {
      msh[wave][qi * F_Q + c] = m_run[qi];
      lsh[wave][qi * F_Q + c] = l_run[qi];
    }
  }
  __syncthreads();   // (and everybody is done with the keys)
  float lt[NQ], mt[NQ];
#pragma unroll
  for (int qi = 0; qi < NQ; ++qi) {
    const int at = qi * F_Q + c;
    float& mm = mt[qi];
    mm = -INFINITY;
    lt[qi] = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w)
      if (lsh[w][at] != 0.f) mm = fmaxf(mm, msh[w][at]);  // (a wavefront without keys has no say)
#pragma unroll
    for (int w = 0; w < NW; ++w)
      if (lsh[w][at] != 0.f) lt[qi] += lsh[w][at] * __builtin_amdgcn_exp2f(msh[w][at] - mm);
    const float mine = l_run[qi] != 0.f ? __builtin_amdgcn_exp2f(m_run[qi] - mm) : 0.f;
#pragma unroll
    for (int hh = 0; hh < NH; ++hh)
#pragma unroll
      for (int e = 0; e < 4; ++e) o[qi][hh][e] *= mine;
  }
  auto row_of = [&](int w, int qi, int hh, int i) { return reinterpret_cast<f32x4_t*>(&osh[w][qi * F_Q + c][64 * hh + 16 * g + 4 * i]); };
  if (wave >= NOUT) {
#pragma unroll
    for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
      for (int hh = 0; hh < NH; ++hh)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *row_of(wave - NOUT, qi, hh, i) = f32x4_t{o[qi][hh][0][i], o[qi][hh][1][i], o[qi][hh][2][i], o[qi][hh][3][i]};
  }
  __syncthreads();
  if (wave < NOUT) {
#pragma unroll
    for (int qi = 0; qi < NQ; ++qi)
#pragma unroll
      for (int hh = 0; hh < NH; ++hh)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f32x4_t* r = row_of(wave, qi, hh, i);
          *r = f32x4_t{o[qi][hh][0][i], o[qi][hh][1][i], o[qi][hh][2][i], o[qi][hh][3][i]} + *r;
        }
  }
  if (wave == 0 && g == 0) {  // (every wavefront has read the sums before the barrier above)
#pragma unroll
    for (int qi = 0; qi < NQ; ++qi) {
      lsh[0][qi * F_Q + c] = lt[qi];
      msh[0][qi * F_Q + c] = mt[qi];
    }
  }
  __syncthreads();
  for (int item = tid; item < BQ * DH / 4; item += 64 * NW) {
    const int qi = item / (DH / 4), d = (item % (DH / 4)) * 4;
    const int qrow = q0 + qi;
    if (qrow >= p.T) continue;
    f32x4_t y = *reinterpret_cast<const f32x4_t*>(&osh[0][qi][d]);
#pragma unroll
    for (int w = 1; w < NOUT; ++w) y += *reinterpret_cast<const f32x4_t*>(&osh[w][qi][d]);
    if (n_parts > 1) {  // (a part: merged by the second pass)
      const int64_t row = ((int64_t)part * p.B * p.H + (int64_t)b * p.H + h) * p.T + qrow;
      *reinterpret_cast<f32x4_t*>(static_cast<float*>(p.ws_o) + row * DH + d) = y;
      if (d == 0) *reinterpret_cast<float2_t*>(p.ws_ml + row * 2) = float2_t{msh[0][qi], lsh[0][qi]};
      continue;
    }
    y *= 1.f / lsh[0][qi];
    // the gate multiplies the rounded attention output, as the module's own multiply does
    if (p.gate != nullptr) y *= reinterpret_cast<const float*>(p.gate)[b * p.gs_b + h * p.gs_h + (int64_t)qrow * p.gs_t];
    *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(p.out) + b * p.os_b + h * p.os_h + (int64_t)qrow * p.os_t + d) = y;
  }
}

// Second pass of a context in parts: one thread per four columns of a query row.
template <int DH>
__global__ void __launch_bounds__(256) f32_combine_kernel(AttnParams p) {
  const unsigned item = blockIdx.x * 256 + threadIdx.x, row = item / (DH / 4), d = item % (DH / 4) * 4;
  const unsigned rows = (unsigned)(p.B * p.H * p.T);
  if (row >= rows) return;
  float m = -INFINITY, l = 0.f;
  f32x4_t y = {0.f, 0.f, 0.f, 0.f};
#pragma nounroll
  for (int s0 = 0; s0 < p.n_splits; s0 += 4) {
    float2_t ml[4];
    f32x4_t o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (s0 + j < p.n_splits) {
        const int64_t at = (int64_t)(s0 + j) * rows + row;
        ml[j] = *reinterpret_cast<const float2_t*>(p.ws_ml + at * 2);
        o[j] = *reinterpret_cast<const f32x4_t*>(static_cast<const float*>(p.ws_o) + at * DH + d);
      } else {
        ml[j] = float2_t{-INFINITY, 0.f};
        o[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
    float mx = m;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (ml[j][1] != 0.f) mx = fmaxf(mx, ml[j][0]);  // (a part without keys has no say)
    const float carry = l != 0.f ? __builtin_amdgcn_exp2f(m - mx) : 0.f;
    l *= carry;
    y *= carry;
    m = mx;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (ml[j][1] != 0.f) {
        const float w = __builtin_amdgcn_exp2f(ml[j][0] - mx);
        l += w * ml[j][1];
        y += w * o[j];
      }
  }
  const int t = (int)(row % (unsigned)p.T), bh = (int)(row / (unsigned)p.T), b = bh / p.H, h = bh - b * p.H;
  y *= 1.f / l;
  if (p.gate != nullptr) y *= reinterpret_cast<const float*>(p.gate)[b * p.gs_b + h * p.gs_h + (int64_t)t * p.gs_t];
  *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(p.out) + b * p.os_b + h * p.os_h + (int64_t)t * p.os_t + d) = y;
}

template <int DH>
static hipError_t launch_f32(AttnParams p, int nq, int cus, hipStream_t stream) {
  const F32Call call = {(int64_t)p.B * p.H, p.T, p.num_buckets, DH, cus};
  const int64_t wgs = call.tiles(nq) * p.n_splits;
  if (wgs > 0x7fffffff) return hipErrorInvalidValue;
  p.members = p.group * ((p.T + nq * F_Q - 1) / (nq * F_Q));
  // eight wavefronts per workgroup (two per SIMD of a CU) while a CU gets one workgroup; two
  // workgroups of four beyond, which leave a smaller last round
  const int nw = wgs <= cus ? 8 : 4;
  const bool split = call.blocks() >= call.halves_from(), whole = p.T % F_K == 0;
  const void* kernel = nullptr;
  int lds = 0;
  auto pick = [&](auto waves, auto groups, auto halves) {
    constexpr int NW = decltype(waves)::value, NQ = decltype(groups)::value;
    constexpr bool SPLIT = decltype(halves)::value;
    kernel = SPLIT && whole ? reinterpret_cast<const void*>(&attn_ring_f32_kernel<DH, NW, NQ, SPLIT, SPLIT>)
                            : reinterpret_cast<const void*>(&attn_ring_f32_kernel<DH, NW, NQ, SPLIT, false>);
    lds = F32Lds<DH, NW, NQ, SPLIT>::kBytes;
  };
  const std::integral_constant<int, 8> w8; const std::integral_constant<int, 4> w4;
  const std::integral_constant<int, 1> one; const std::integral_constant<int, 2> two;
  if (nq == 2) nw == 8 ? pick(w8, two, std::true_type()) : pick(w4, two, std::true_type());
  else if (split) nw == 8 ? pick(w8, one, std::true_type()) : pick(w4, one, std::true_type());
  else nw == 8 ? pick(w8, one, std::false_type()) : pick(w4, one, std::false_type());
  F32Params fp = {p, (int)call.halves_from()};
  void* args[] = {&fp};
  const hipError_t e = hipLaunchKernel(kernel, dim3((unsigned)wgs), dim3(64 * nw), args, lds, stream);
  if (e != hipSuccess || p.n_splits == 1) return e;
  const int64_t items = (int64_t)p.B * p.H * p.T * (DH / 4);
  hipLaunchKernelGGL(f32_combine_kernel<DH>, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, stream, p);
  return hipGetLastError();
}

// The dynamic-LDS limit of the instances that may need more than the default.
template <int DH, int NQ, bool WHOLE>
static hipError_t configure_f32() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_ring_f32_kernel<DH, 8, NQ, true, WHOLE>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, F32Lds<DH, 8, NQ, true>::kBytes);
}
hipError_t configure_attn_ring_f32() {
  hipError_t e = configure_f32<128, 1, true>();
  if (e == hipSuccess) e = configure_f32<128, 1, false>();
  if (e == hipSuccess) e = configure_f32<128, 2, true>();
  if (e == hipSuccess) e = configure_f32<128, 2, false>();
  if (e == hipSuccess) e = configure_f32<64, 2, true>();
  return e == hipSuccess ? configure_f32<64, 2, false>() : e;
}

hipError_t launch_attn_ring_f32(const AttnParams& p, int Dh, int groups, int cus, hipStream_t stream) {
  if (Dh == 128) return launch_f32<128>(p, groups, cus, stream);
  if (Dh == 64) return launch_f32<64>(p, groups, cus, stream);
  return hipErrorInvalidValue;
}

}  // namespace we
