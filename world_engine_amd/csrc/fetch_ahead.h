// Which weights the helper workgroups of a projection fetch: plain arithmetic, apart from the kernels so that every
// case can be gone through on the host.
//
// A projection x W^T of a small frame is bound by what the CUs with a tile take in: 50 to 60 GB/s out of HBM whatever a CU
// has in flight, 120 out of L2.  The CUs that have no tile run a workgroup that asks for the weights of their XCD's tiles
// in steps of 128 contraction elements, as the tiles take them, and has no use for them: they are in the XCD's L2 when the
// tiles get there.  The first step is left to the tiles themselves.  us without / with them, weights out of HBM: linear of
// 64 x 2048 x 2048 11.2 / 8.7, 192 x 3072 x 3072 17.1 / 14.7; a layer of projection + store, attention and second pass (16
// heads of 128, d_model 2048, 4 slots) of 256 tokens 34.9 / 33.1, 64 tokens 33.6 / 27.4, 16 heads on 8, 256 tokens 33.7 /
// 31.6, 40 heads (5120), 64 tokens 62.5 / 59.3.  Weights that are in the last-level cache anyway gain nothing (7.24 / 7.28,
// 29.2 / 29.2), and the layer of 64 tokens loses 0.4 us (22.7 / 23.1).  Asking for x too, or for 1 KB of a row at a time: no
// better.
#pragma once

#ifdef __HIPCC__
#define WE_AHEAD_FN __host__ __device__ __forceinline__
#else
#define WE_AHEAD_FN inline
#endif

namespace we {

// Helpers per XCD: eight where tiles leave that many CUs idle (16 and more ask for the same lines no sooner and get in the
// tiles' way: the layer of 64 tokens above, its weights partly in that cache, with 8 / 16 / 32: 22.1 / 23.0 / 24.1 us; fewer
// beside more tiles are no help, 52 heads on 26, d_model 6656, 81 tokens with six: 49.4 -> 51.7); none where the tiles ask
// for half of the contraction's steps before their first wait (64 x 1536 x 512 4.04 -> 4.09 us with helpers).
inline int helpers_of(int tiles_per_xcd, int cus, int steps, int in_flight) {
  return cus / 8 - tiles_per_xcd < 8 || steps < 2 * in_flight ? 0 : 8;
}

// Weights of one XCD: tile t, of `rows` features, is XCD t % 8's.  Wavefront w of helper k takes the groups of four rows
// q = 8 k + w, 8 k + w + 8 helpers, ... of every every-th step.  A helper that cannot keep up is in the tiles' way (40 heads
// of 128, d_model 5120, 64 tokens, 20 MB of weights per XCD: 61.5 -> 63.3 us): it asks for no more rows per step than a
// tile takes in and leaves steps out for that (-> 56.7; 36 heads, d_model 4608 53.3 -> 49.5).
struct AheadOrder {
  int xcd, rows, quads, every;
  WE_AHEAD_FN AheadOrder(int n_tiles, int xcd_, int helpers, int rows_) : xcd(xcd_), rows(rows_) {
    quads = ((n_tiles - xcd + 7) >> 3) * (rows / 4);  // (none on an XCD without a tile)
    const int share = helpers * ((64 + rows) / 4);
    every = quads > share ? (quads + share - 1) / share : 1;
  }
  // first row of group q
  WE_AHEAD_FN int row(int q) const { return ((q / (rows / 4)) * 8 + xcd) * rows + (q % (rows / 4)) * 4; }
};

}  // namespace we
