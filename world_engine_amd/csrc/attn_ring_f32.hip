// fp32 attention over the KV ring buffer (gfx950): the same visibility rule and ring walk as the
// half-precision kernel (attn_ring.hip), fp32 throughout (fp32 scores, softmax and P V,
// src/model/attn.py:116 in eager mode) on the fp32 matrix instructions.
//
// One workgroup = 16 queries of one (batch, head) and NW wavefronts that share out its keys: blocks
// of 16 keys go round the wavefronts, each keeps its own running (reference, sum, O) and they merge
// through LDS at the end.  A wavefront's keys are nobody else's, so K and V go from memory straight
// into the matrix operands' registers, one block ahead, without LDS and without a barrier in the loop:
//   S^T = K Q^T      v_mfma_f32_16x16x4_f32; the contraction is taken in an order that lets a lane
//                    load four of its head-dim values at once (lane group g of step (j, i) has value
//                    16 j + 4 g + i of both operands);
//   O^T += V^T P^T   the S^T accumulators are the B operand as they are (lane group g, register i =
//                    key 4 g + i), and output rows are numbered so that a lane's four values of V are
//                    consecutive: one 16-byte load per key and 64 head-dim values, 256 bytes a row.
//
// Bound by the matrix cores (64 MFMAs of 32 cycles per block of 16 keys at Dh = 128, against 16 loads
// and some 40 vector instructions) and, at 16 queries a workgroup, by the loads' way through the CU's
// address path beside them: 16 heads of 128, 256 queries, 2048 keys take 44.4 us = 97 TFLOP/s (a large
// fp32 matrix product reaches 153 here), 37 us without the loads; 8 heads, 1024 queries and 4096 keys
// 149 us = 115 TFLOP/s.  (54 and 185 us while the next block's loads stood behind a branch, below.)
#include "attn_mma.h"
#include "we_kernels.h"
#include "../../include/we_attn.h"

namespace we {

namespace {
constexpr int F_Q = 16;   // queries per workgroup
constexpr int F_K = 16;   // keys per block
}  // namespace

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

template <int DH, int NW>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2)))
attn_ring_f32_kernel(AttnParams p) {
  constexpr int NJ = DH / 16;    // 16-byte loads of K per lane and block
  constexpr int NH = DH / 64;    // 16-byte loads of V per lane and key
  constexpr int OROW = DH + 4;   // floats per row of a wavefront's O in LDS (the odd 16 bytes spread the banks)
  constexpr int NOUT = NW / 2;   // wavefronts whose O is in LDS at a time
  __shared__ __attribute__((aligned(16))) float osh[NOUT][F_Q][OROW];
  __shared__ float msh[NW][F_Q], lsh[NW][F_Q];
  __shared__ int vis[WE_MAX_SLOTS + 2];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;

  // ---- which queries ----
  // (spread over the XCDs by unit where every XCD gets the same number: a unit's workgroups share an L2)
  const int units = p.B * p.Hkv, q_tiles = (p.T + F_Q - 1) / F_Q;
  int unit, member;
  if ((units & 7) == 0) {
    const unsigned j = blockIdx.x >> 3;
    const unsigned u8 = j / (unsigned)p.members;
    unit = (int)(u8 * 8 + (blockIdx.x & 7));
    member = (int)(j - u8 * (unsigned)p.members);
  } else {
    unit = (int)(blockIdx.x / (unsigned)p.members);
    member = (int)(blockIdx.x - (unsigned)unit * (unsigned)p.members);
  }
  const int b = unit / p.Hkv, hkv = unit - b * p.Hkv;
  const int hq_in = member / q_tiles, h = hkv * p.group + hq_in;
  const int q0 = (member - hq_in * q_tiles) * F_Q;

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

  // ---- query c, values 16 j + 4 g + i, pre-multiplied by scale * log2(e) ----
  f32x4_t qf[NJ];
  {
    const int qr = q0 + c < p.T ? q0 + c : p.T - 1;
    const float* src = reinterpret_cast<const float*>(p.q) + b * p.qs_b + h * p.qs_h + (int64_t)qr * p.qs_t + 4 * g;
#pragma unroll
    for (int j = 0; j < NJ; ++j) qf[j] = *reinterpret_cast<const f32x4_t*>(src + 16 * j) * p.scale_log2;
  }
  __syncthreads();
  const int nvis = vis[WE_MAX_SLOTS + 1];

  f32x4_t o[NH][4];  // o[hh][e] register i: query c, value 64 hh + 16 g + 4 i + e
#pragma unroll
  for (int hh = 0; hh < NH; ++hh)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[hh][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;  // (l_run: this lane group's keys only)

  const int64_t cap = p.L + p.T;
  const float* kplane = reinterpret_cast<const float*>(p.kv) + (((int64_t)b * p.Hkv + hkv) * cap) * DH;
  const float* vplane = kplane + (int64_t)p.B * p.Hkv * cap * DH;

  // Blocks go round the wavefronts in rounds of NW.  The workgroups that share a K/V stream take the
  // rounds in groups of rot_g, member m starting at round m of every group: they then ask for
  // different lines at any one time, and each line comes from memory at one member's request (184
  // against 192 us for the 1024-query shape above when it took 184; groups of 8 or 16: the same, then and now).
  const int bps = (p.T + F_K - 1) / F_K;  // blocks per slot; the last one may be short
  const int nblk = nvis * bps, rounds = (nblk + NW - 1) / NW;
  int rot_g = 1;
  while (rot_g * 2 <= p.members && rot_g < 4) rot_g *= 2;
  const int rot_end = (nblk / NW) & ~(rot_g - 1);
  auto block_of = [&](int k) __attribute__((always_inline)) {
    const int kk = k < rot_end ? (k & ~(rot_g - 1)) | ((k + member) & (rot_g - 1)) : k;
    return kk * NW + wave;
  };

  // (uniform base and 32-bit lane offsets; rows past the frame repeat its last one)
  auto load = [&](f32x4_t(&kf)[NJ], f32x4_t(&vf)[4][NH], int vi_, int sub_) __attribute__((always_inline)) {
    const int64_t row0 = (int64_t)__builtin_amdgcn_readfirstlane(vis[vi_]) * p.T + sub_ * F_K;
    const int last = p.T - 1 - sub_ * F_K;
    const char* kb = reinterpret_cast<const char*>(kplane + row0 * DH);
    const char* vb = reinterpret_cast<const char*>(vplane + row0 * DH);
    const uint32_t ko = (uint32_t)((c < last ? c : last) * DH + 4 * g) * 4u;
#pragma unroll
    for (int j = 0; j < NJ; ++j) kf[j] = *reinterpret_cast<const f32x4_t*>(kb + ko + 64 * j);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t vo = (uint32_t)((4 * g + i < last ? 4 * g + i : last) * DH + 4 * c) * 4u;
#pragma unroll
      for (int hh = 0; hh < NH; ++hh) vf[i][hh] = *reinterpret_cast<const f32x4_t*>(vb + vo + 256 * hh);
    }
  };
  auto block = [&](const f32x4_t(&kf)[NJ], f32x4_t(&vf)[4][NH], int keys) __attribute__((always_inline)) {
    f32x4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NJ; j += 2)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][i], qf[j][i], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j + 1][i], qf[j + 1][i], s1, 0, 0, 0);
      }
    // (the next block's loads go out between these products: together they keep a wavefront from issuing anything
    // else while the CU's address path takes them, 47.0 against 45.5 us for the first shape above)
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
    const float mx = fmaxf(m_run, groups_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
    if (__ballot(mx != m_run) != 0ull) {
      const float alpha = __builtin_amdgcn_exp2f(m_run - mx);  // 0 on the first block
      l_run *= alpha;
#pragma unroll
      for (int hh = 0; hh < NH; ++hh)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[hh][e] *= alpha;
      m_run = mx;
    }
    f32x4_t pr;
#pragma unroll
    for (int i = 0; i < 4; ++i) pr[i] = __builtin_amdgcn_exp2f(s[i] - mx);
    l_run += (pr[0] + pr[1]) + (pr[2] + pr[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int hh = 0; hh < NH; ++hh)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[hh][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][hh][e], pr[i], o[hh][e], 0, 0, 0);
    // (two blocks in a row are not scheduled as one: 44.4 against 46.8 us for the first shape above)
    __builtin_amdgcn_sched_barrier(0);
  };
  const int mine_n = rounds - (nblk - (rounds - 1) * NW > wave ? 0 : 1);  // rounds this wavefront takes part in
  if (mine_n > 0) {
    f32x4_t ka[NJ], va[4][NH], kb[NJ], vb[4][NH];
    // The loop always requests the next block - behind a branch the compiler counts the loads in flight as if it had
    // not been taken, and waits for the block just requested - and the last one or two blocks follow it.  (A last block
    // requested a second time, for nothing, costs wavefronts with one or two of them most: attention alone, 4 heads of 128,
    // 64 queries, 128 keys 9.8 -> 8.75 us, 8 heads, 256 keys 12.25 -> 11.4, 8 heads of 64, 256 keys 7.64 -> 7.40, 128 keys
    // 6.43 -> 6.11.)
    auto fetch = [&](f32x4_t(&kf)[NJ], f32x4_t(&vf)[4][NH], int k) __attribute__((always_inline)) {
      const int at = block_of(k), vi = (int)((unsigned)at / (unsigned)bps), sub = at - vi * bps;
      load(kf, vf, vi, sub);
      return p.T - sub * F_K;  // keys of the block (16 or more: a whole one)
    };
    int keys_a = fetch(ka, va, 0), k = 1;
    for (; k + 1 < mine_n; k += 2) {
      const int keys_b = fetch(kb, vb, k);
      block(ka, va, keys_a);
      keys_a = fetch(ka, va, k + 1);
      block(kb, vb, keys_b);
    }
    if (k < mine_n) {
      const int keys_b = fetch(kb, vb, k);
      block(ka, va, keys_a);
      block(kb, vb, keys_b);
    } else {
      block(ka, va, keys_a);
    }
  }

  // ---- the wavefronts merge ----
  l_run = groups_sum(l_run);
  if (g == 0) {
    msh[wave][c] = m_run;
    lsh[wave][c] = l_run;
  }
  __syncthreads();
  float mm = -INFINITY, lt = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w)
    if (lsh[w][c] != 0.f) mm = fmaxf(mm, msh[w][c]);  // (a wavefront without keys has no say)
#pragma unroll
  for (int w = 0; w < NW; ++w)
    if (lsh[w][c] != 0.f) lt += lsh[w][c] * __builtin_amdgcn_exp2f(msh[w][c] - mm);
  const float mine = l_run != 0.f ? __builtin_amdgcn_exp2f(m_run - mm) : 0.f;
#pragma unroll
  for (int hh = 0; hh < NH; ++hh)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[hh][e] *= mine;
  auto row_of = [&](int w, int hh, int i) { return reinterpret_cast<f32x4_t*>(&osh[w][c][64 * hh + 16 * g + 4 * i]); };
  if (wave >= NOUT) {
#pragma unroll
    for (int hh = 0; hh < NH; ++hh)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *row_of(wave - NOUT, hh, i) = f32x4_t{o[hh][0][i], o[hh][1][i], o[hh][2][i], o[hh][3][i]};
  }
  __syncthreads();
  if (wave < NOUT) {
#pragma unroll
    for (int hh = 0; hh < NH; ++hh)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x4_t* r = row_of(wave, hh, i);
        *r = f32x4_t{o[hh][0][i], o[hh][1][i], o[hh][2][i], o[hh][3][i]} + *r;
      }
  }
  if (wave == 0 && g == 0) lsh[0][c] = lt;  // (every wavefront has read the sums before the barrier above)
  __syncthreads();
  for (int item = tid; item < F_Q * DH / 4; item += 64 * NW) {
    const int qi = item / (DH / 4), d = (item % (DH / 4)) * 4;
    const int qrow = q0 + qi;
    if (qrow >= p.T) continue;
    f32x4_t y = *reinterpret_cast<const f32x4_t*>(&osh[0][qi][d]);
#pragma unroll
    for (int w = 1; w < NOUT; ++w) y += *reinterpret_cast<const f32x4_t*>(&osh[w][qi][d]);
    y *= 1.f / lsh[0][qi];
    // the gate multiplies the rounded attention output, as the module's own multiply does
    if (p.gate != nullptr) y *= reinterpret_cast<const float*>(p.gate)[b * p.gs_b + h * p.gs_h + (int64_t)qrow * p.gs_t];
    *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(p.out) + b * p.os_b + h * p.os_h + (int64_t)qrow * p.os_t + d) = y;
  }
}

template <int DH>
static hipError_t launch_f32(AttnParams p, int cus, hipStream_t stream) {
  p.members = p.group * ((p.T + F_Q - 1) / F_Q);
  const int64_t wgs = (int64_t)p.B * p.Hkv * p.members;
  if (wgs > 0x7fffffff) return hipErrorInvalidValue;
  // eight wavefronts per workgroup (two per SIMD of a CU) while a CU gets one workgroup; two
  // workgroups of four beyond, which leave a smaller last round
  if (wgs <= cus) hipLaunchKernelGGL((attn_ring_f32_kernel<DH, 8>), dim3((unsigned)wgs), dim3(512), 0, stream, p);
  else hipLaunchKernelGGL((attn_ring_f32_kernel<DH, 4>), dim3((unsigned)wgs), dim3(256), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_attn_ring_f32(const AttnParams& p, int Dh, int cus, hipStream_t stream) {
  if (Dh == 128) return launch_f32<128>(p, cus, stream);
  if (Dh == 64) return launch_f32<64>(p, cus, stream);
  return hipErrorInvalidValue;
}

}  // namespace we
