// How many context parts a call of a frame of 64 to 256 tokens takes where the planner's count cuts it too fine: plain
// arithmetic, apart from the kernels so that it can be gone through on the host.
//
// The planner's count fills the CUs; a short context or a frame of 128 tokens is then cut into parts of two or three tiles,
// each with its own start-up and its partial rows, which for an f16 cache are fp32.  Estimated here, from 4330 timings of
// 454 shapes (48 to 256 tokens, 2 to 64 slots, 1 to 48 parts; a frame's store and attention in a graph, three
// rings; met to 5 % rms): us per round of CUs, per 64-key tile of a part, more so the more CUs are busy, and for the second
// pass and its rows.  The count with the lowest estimate is taken where that is 2 % below the planner's, never a
// larger one.  Over 150 other shapes bf16 calls take 0.993 of the planner's time and f16 ones 0.974 (us, before / after: f16,
// 24 heads of 64 on 6, 128 tokens, 5 slots 14.9 / 12.7, 8 of 128 on 4, 115 tokens, 28 slots 23.7 / 20.9; bf16, 8 of 128, 128
// tokens, 22 slots 20.3 / 17.9, 2 of 128, 132 tokens, 26 slots 18.6 / 17.5; at worst, f16, 56 on 28, 192 tokens, 8 slots 27.4 / 28.3).  Frames below 64 tokens,
// whose tiles are short, keep the planner's count: 3 x 17 heads of 64, 61 tokens, 11 slots would be 14.9 / 16.0.
#pragma once

#include <stdint.h>

namespace we {

struct ShortCall {
  int64_t units, members;   // (batch, kv head) units, workgroups per unit part
  int64_t tiles;            // key tiles of a full ring
  int64_t rows;             // query rows of all heads
  int row_bytes;            // of a partial row
  bool wide;                // heads of more than 64
  int cus;

  double cost(int64_t parts) const {
    const int64_t per_xcd = cus / 8 > 0 ? cus / 8 : 1;
    const int64_t rounds = ((units * parts + 7) / 8 * members + per_xcd - 1) / per_xcd;
    const double busy = (double)(units * parts * members) / (double)cus;
    const double tile = wide ? 0.577 + 0.110 * (busy < 1. ? busy : 1.) : 0.408 + 0.061 * (busy < 1. ? busy : 1.);
    double c = (wide ? 6.7 : 6.2) + (double)rounds * ((wide ? 3.53 : 2.99) + tile * (double)((tiles + parts - 1) / parts));
    if (parts > 1) c += 2.64 + (wide ? 0.68 : 0.77) * 1e-6 * (double)(parts * rows) * (double)row_bytes;
    return c;
  }
  int parts(int planned) const {
    int best = planned;
    double low = 0.98 * cost(planned);
    for (int s = planned - 1; s >= 1; --s) {
      const double c = cost(s);
      if (c < low) {
        low = c;
        best = s;
      }
    }
    return best;
  }
};

}  // namespace we
