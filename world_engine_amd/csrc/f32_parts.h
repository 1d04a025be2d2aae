// How an fp32 attention call is cut up: groups of 16 queries per workgroup and context parts.  Plain arithmetic, apart from the
// kernels so that it can be gone through on the host.
//
// A workgroup works off its keys in rounds of 128 (8 wavefronts, blocks of 16).  Where 16-query workgroups outnumber the CUs,
// two groups share what the rounds halve (attn_ring_f32.hip).  Where they do not, a context in parts fills the CUs - or the
// CUs take two groups of queries each and a part of the keys - at the price of a second pass over the parts' rows.
// The cost is a fit to single calls; parts are taken where it says 7 % less.  us, one pass / parts: 2 heads of 128, 64 tokens, 64
// slots 58.2 / 15.5 (16 parts), 2 heads, 256 tokens, 16 slots 58.8 / 20.3, 4 heads, 128 tokens, 16 slots 33.7 / 15.0, 8 heads,
// 256 tokens, 8 slots 33.2 / 23.6, 16 heads 36.1 / 34.8, 8 heads, 64 tokens, 8 slots 13.5 / 11.5; heads of 64: 3 of 100 tokens, 40
// slots 43.0 / 16.4, 8 of 64 tokens, 16 slots 13.3 / 10.5.  (The fit is from halves that took 3 to 6 % less.)
#pragma once

#include <stdint.h>

namespace we {

struct F32Call {
  int64_t heads;    // batch times query heads
  int T;            // queries per head, and keys per slot
  int64_t slots;    // of the ring that frames go to
  int dh, cus;

  int groups = 1, parts = 1;

  int64_t tiles(int g) const { return heads * ((T + 16 * g - 1) / (16 * g)); }
  int64_t blocks() const { return slots * ((T + 15) / 16); }
  // Blocks of keys from which on a call's products go in halves.  (The lines for heads of 64 are from halves that were less exact
  // than fp32 products in one short chain per wavefront, 512 keys 2.6e-7 against 2.45e-7.  The present ones are at 1.9e-7 there
  // and faster from some 24 blocks on, 512 keys 10.3 -> 9.6 us, but 128 keys 6.4 -> 6.75.)
  int64_t halves_from() const { return dh == 64 ? (tiles(1) > cus ? 32 : 64) : 1; }
  int64_t row_bytes() const { return (int64_t)dh * 4 + 8; }
  int64_t bytes(int p) const { return p > 1 ? heads * T * p * row_bytes() : 0; }
  double cost(int g, int p) const {
    const double rounds = (double)(((blocks() + p - 1) / p + 7) / 8);
    double c = dh == 64 ? (g == 1 ? 4.4 + 1.15 * rounds : 4.5 + 1.8 * rounds) : (g == 1 ? 3.3 + 2.32 * rounds : 5.0 + 2.85 * rounds);
    if (p > 1) c += 4.5 + 0.6e-6 * (double)bytes(p);
    return c;
  }
  // most bytes of partial rows: what the caller's workspace holds
  void plan(int64_t most) {
    const bool halves = blocks() >= halves_from();
    groups = tiles(1) > cus && halves ? 2 : 1;
    parts = 1;
    if (tiles(1) > cus || !halves) return;
    double low = 0.93 * cost(1, 1);
    for (int g = 1; g <= 2; ++g)
      for (int p = 2; p <= 16 && tiles(g) * p <= cus && blocks() / p >= 8 && bytes(p) <= most; ++p)
        if (cost(g, p) < low) {
          low = cost(g, p);
          groups = g;
          parts = p;
        }
  }
};

}  // namespace we
