// y = x W^T for a few hundred rows of x (gfx950): the attention module's projections of one frame,
// where the weight matrix is read once and a library GEMM is latency-bound.
//
// One workgroup = 8 wavefronts = one CU computes a 64-row x BN-feature tile.  x and W tiles of 128
// contraction elements travel HBM/L2 -> LDS by DMA (global_load_lds_dwordx4) into a ring as deep as
// LDS holds (BN = 32: six slots of 24 KB, 64: five of 32 KB, 128: three of 48 KB), all but one in
// flight; rows are 256 bytes, 16-byte chunks XOR-swizzled with (row & 15) on the global side of the
// DMA.  Wavefront w takes one 32-feature block, both 32-row blocks and one share of the contraction
// steps of every slot (A = W rows, B = x rows); the shares are added through LDS in a fixed order and
// rounded once.  Workgroup id % 8 is the XCD, the row tiles of one weight slab follow each other on
// one XCD and take the contraction chunks in rotated order (see qkv_proj_store.hip): a slab comes
// from HBM once and its lines are L2 hits for the other tiles; CUs without a tile fetch slabs into their L2 (fetch_ahead).
//
// Bound by what a CU takes in, (64 + BN) rows of K elements at some 90 GB/s, behind 3.5 us of launch,
// first slot and reduction.  Against the BLAS routine, us in a graph, 24 weight matrices with the last-level cache
// emptied in between (in brackets: eight matrices that stay in it), 256 rows: 2048 x 2048 10.0 / 14.1 (8.2 / 9.8), 4096
// x 2048 12.6 / 15.4 (10.5 / 11.3), 6144 x 2048 16.3 / 26.6 (14.3 / 19.3), 3072 x 3072 14.8 / 20.0 (12.3 / 14.2); 64 rows,
// 1536 x 512 5.4 / 9.5 (4.1 / 6.1), 2048 x 2048 8.6 / 13.9 (7.2 / 8.9), 3072 x 3072 13.0 / 18.4 (9.2 / 11.6).
#include "attn_mma.h"
#include "device_state.h"
#include "we_kernels.h"

namespace we {

namespace {
constexpr int LM = 64;            // rows of x per tile
constexpr int LK = 128;           // contraction elements per ring slot
constexpr int L_ROW_B = LK * 2;   // bytes per tile row

template <int BN>
struct LinLds {
  static constexpr int SLOT_B = (LM + BN) * L_ROW_B;
  static constexpr int NSLOT = BN == 32 ? 6 : (BN == 64 ? 5 : 3);
  static constexpr int kBytes = NSLOT * SLOT_B;
};
}  // namespace

template <typename M, int BN>
__global__ void __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2)))
linear_skinny_kernel(LinearParams p) {
  touch_args<LinearParams>();
  typedef typename M::frag_t frag_t;
  typedef LinLds<BN> L;
  constexpr int NF = BN / 32;              // feature blocks of the tile
  constexpr int KG = 8 / NF;               // contraction shares of a slot
  constexpr int STEPS = LK / 16 / KG;      // MFMA steps of a share
  constexpr int XQ = LM / 4 / 8;           // DMA instructions per wavefront and slot: x ...
  constexpr int WQ = BN / 4 / 8;           // ... and W
  constexpr int ND = XQ + WQ;
  constexpr int NSLOT = L::NSLOT;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, hh = lane >> 5;
  const int fb = wave % NF, kg = wave / NF;

  // ---- which tile ----
  const int xcd = blockIdx.x & 7;
  const unsigned j = blockIdx.x >> 3, own = (unsigned)(p.n_tiles + 7) / 8u * (unsigned)p.m_tiles;
  if (j >= own) {
    fetch_ahead<BN>(p.w, p.ws, p.n_tiles, p.K, xcd, (int)(j - own), p.helpers, wave, lane, lds0);
    return;
  }
  const int ng = (int)(j / (unsigned)p.m_tiles);
  const int mi = (int)j - ng * p.m_tiles;
  const int nt = ng * 8 + xcd;
  if (nt >= p.n_tiles) return;
  const int m0 = mi * LM, n0 = nt * BN;

  // ---- DMA plumbing: instruction i of this wavefront moves rows 4 (wave + 8 i) .. + 3 of a tile ----
  uint32_t xvo[XQ], wvo[WQ];
  {
    const int phys = lane & 15;
#pragma unroll
    for (int i = 0; i < XQ; ++i) {
      const int row = 4 * (wave + 8 * i) + (lane >> 4);
      const int r = m0 + row < p.M ? m0 + row : p.M - 1;  // rows past the end repeat the last one; never stored
      xvo[i] = (uint32_t)r * (uint32_t)(p.xs * 2) + (uint32_t)((phys ^ (row & 15)) << 4);
    }
#pragma unroll
    for (int i = 0; i < WQ; ++i) {
      const int row = 4 * (wave + 8 * i) + (lane >> 4);
      wvo[i] = (uint32_t)row * (uint32_t)(p.ws * 2) + (uint32_t)((phys ^ (row & 15)) << 4);
    }
  }
  const uint64_t xbase = uniform64((uint64_t)(uintptr_t)p.x);
  const uint64_t wbase = uniform64((uint64_t)(uintptr_t)p.w + (uint64_t)((int64_t)n0 * p.ws * 2));
  const uint32_t wave_lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + wave * 1024));
  auto dma_slot = [&](int c, int slot) __attribute__((always_inline)) {
    const uint64_t kb = (uint64_t)c * L_ROW_B;
    const uint32_t at = wave_lds + slot * L::SLOT_B;
#pragma unroll
    for (int i = 0; i < WQ; ++i) dma16(wbase + kb, wvo[i], at + LM * L_ROW_B + i * 8 * 1024);
#pragma unroll
    for (int i = 0; i < XQ; ++i) dma16(xbase + kb, xvo[i], at + i * 8 * 1024);
  };
  const int nc = p.K / LK;
  const int G = p.m_tiles >= 8 ? 8 : (p.m_tiles >= 4 ? 4 : (p.m_tiles >= 2 ? 2 : 1));
  const int rot = mi & (G - 1), ncg = nc & ~(G - 1);
  auto chunk = [&](int c) __attribute__((always_inline)) { return c < ncg ? (c & ~(G - 1)) | ((c + rot) & (G - 1)) : c; };
#pragma unroll
  for (int s = 0; s < NSLOT - 1; ++s)
    if (s < nc) dma_slot(chunk(s), s);

  // ---- fragment read addresses: row l32 of a 32-row block, logical chunk 2 * step + hh ----
  uint32_t a_rd[STEPS], b_rd[STEPS];
#pragma unroll
  for (int t = 0; t < STEPS; ++t) {
    const int phys = (2 * (kg * STEPS + t) + hh) ^ (l32 & 15);
    b_rd[t] = (uint32_t)(l32 * L_ROW_B + phys * 16);
    a_rd[t] = (uint32_t)((LM + fb * 32 + l32) * L_ROW_B + phys * 16);
  }
  f32x16_t acc[2];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[mb][i] = 0.f;

  // ---- main loop: one barrier per slot ----
  // slots requested behind slot c when it is waited for: as many as are left, at most NSLOT - 2
  auto wait_slot = [&](int left) __attribute__((always_inline)) {
    if (left >= NSLOT - 2) { dma_wait<(NSLOT - 2) * ND>(); return; }
    if (NSLOT > 5 && left == 3) { dma_wait<3 * ND>(); return; }
    if (NSLOT > 4 && left == 2) { dma_wait<2 * ND>(); return; }
    if (NSLOT > 3 && left == 1) { dma_wait<ND>(); return; }
    dma_wait<0>();
  };
  int use = 0, fill = NSLOT - 1;
  for (int c = 0; c < nc; ++c) {
    wait_slot(nc - 1 - c);  // this wavefront's part of slot c has landed
    // every wavefront's part has landed, and everybody is done with the slot refilled next
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (c + NSLOT - 1 < nc) dma_slot(chunk(c + NSLOT - 1), fill);
    fill = fill + 1 == NSLOT ? 0 : fill + 1;
    const unsigned char* sb = smem + use * L::SLOT_B;
    use = use + 1 == NSLOT ? 0 : use + 1;
#pragma unroll
    for (int t = 0; t < STEPS; ++t) {
      const frag_t a = *reinterpret_cast<const frag_t*>(sb + a_rd[t]);
      const frag_t b0 = *reinterpret_cast<const frag_t*>(sb + b_rd[t]);
      const frag_t b1 = *reinterpret_cast<const frag_t*>(sb + b_rd[t] + 32 * L_ROW_B);
      acc[0] = M::mma(a, b0, acc[0]);
      acc[1] = M::mma(a, b1, acc[1]);
    }
  }

  // ---- the contraction shares add up through LDS ----
  // Vector v of lane l of block (fb, mb) of share k - features 4 pc .. 4 pc + 3 of the tile, pc = 8 fb + 2 v + l / 32,
  // of row 32 mb + l % 32 - sits at ((((k * NF + fb) * 2 + mb) * 4 + v) * 64 + (l ^ swz(pc))) * 16: a quarter
  // wavefront of the readers, who take the vectors row by row as the output wants them, finds 16 bank groups.
  __syncthreads();  // everybody is done with the ring
  constexpr int PCR = BN / 4;                  // vectors per row
  auto swz = [](int pc) { return BN == 32 ? 2 * pc : pc & 15; };
  f32x4_t* xch = reinterpret_cast<f32x4_t*>(smem);
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int v = 0; v < 4; ++v)
      xch[(((kg * NF + fb) * 2 + mb) * 4 + v) * 64 + (lane ^ swz(fb * 8 + 2 * v + hh))] =
          f32x4_t{acc[mb][4 * v], acc[mb][4 * v + 1], acc[mb][4 * v + 2], acc[mb][4 * v + 3]};
  __syncthreads();
  constexpr int SHARE_V = NF * 2 * 4 * 64;     // vectors of one share
  static_assert(KG * SHARE_V * 16 <= L::kBytes && SHARE_V == LM * PCR, "the exchange area reuses the ring");
#pragma unroll
  for (int i = tid; i < SHARE_V; i += 512) {
    const int row = i / PCR, pc = i % PCR;
    const int at = (((pc >> 3) * 2 + (row >> 5)) * 4 + ((pc >> 1) & 3)) * 64 + ((((pc & 1) << 5) | (row & 31)) ^ swz(pc));
    f32x4_t r = xch[at];
#pragma unroll
    for (int k = 1; k < KG; ++k) r += xch[k * SHARE_V + at];
    typedef typename M::elem_t E;
    typedef E e4_t __attribute__((ext_vector_type(4)));
    if (m0 + row < p.M)
      *reinterpret_cast<e4_t*>(reinterpret_cast<uint16_t*>(p.y) + (int64_t)(m0 + row) * p.ys + n0 + pc * 4) =
          e4_t{(E)r[0], (E)r[1], (E)r[2], (E)r[3]};
  }
}

template <typename M, int BN>
static hipError_t launch_lin(LinearParams p, int cus, hipStream_t stream) {
  p.m_tiles = (p.M + LM - 1) / LM;
  p.n_tiles = p.N / BN;
  const unsigned per_xcd = (unsigned)((p.n_tiles + 7) / 8) * (unsigned)p.m_tiles;
  p.helpers = helpers_of((int)per_xcd, cus, p.K / LK, LinLds<BN>::NSLOT - 1);
  const dim3 grid(8u * (per_xcd + (unsigned)p.helpers));
  hipLaunchKernelGGL((linear_skinny_kernel<M, BN>), grid, dim3(512), LinLds<BN>::kBytes, stream, p);
  return hipGetLastError();
}

hipError_t launch_linear_skinny(const LinearParams& p, int bn, int dtype, int cus, hipStream_t stream) {
  if (dtype == 0) return bn == 32 ? launch_lin<Bf16Mma, 32>(p, cus, stream) : bn == 64 ? launch_lin<Bf16Mma, 64>(p, cus, stream) : launch_lin<Bf16Mma, 128>(p, cus, stream);
  return bn == 32 ? launch_lin<F16Mma, 32>(p, cus, stream) : bn == 64 ? launch_lin<F16Mma, 64>(p, cus, stream) : launch_lin<F16Mma, 128>(p, cus, stream);
}

template <typename M, int BN>
static hipError_t configure_lin() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&linear_skinny_kernel<M, BN>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, LinLds<BN>::kBytes);
}
hipError_t configure_linear_skinny() {
  hipError_t e = configure_lin<Bf16Mma, 32>();
  if (e == hipSuccess) e = configure_lin<Bf16Mma, 64>();
  if (e == hipSuccess) e = configure_lin<Bf16Mma, 128>();
  if (e == hipSuccess) e = configure_lin<F16Mma, 32>();
  if (e == hipSuccess) e = configure_lin<F16Mma, 64>();
  if (e == hipSuccess) e = configure_lin<F16Mma, 128>();
  return e;
}

}  // namespace we
