// Which tile of its context a split asks for with each of its requests: plain arithmetic, apart from the kernel so
// that every case can be gone through on the host.
#pragma once

#ifdef __HIPCC__
#define WE_TILES_FN __host__ __device__ __forceinline__
#else
#define WE_TILES_FN inline
#endif

namespace we {

// A split owns the visible tiles [begin, end) of 64 consecutive keys.  `shorted`: the last of them has fewer and is
// taken first.  The others go in groups of rot_g (a power of two), starting rot_m into each group.
// Only the first request keeps to the keys that the short tile has: the rows behind the last one are nobody's.
// Where it is all there is, the requests that follow it go to the whole tile in front of it, and the tiles count from there.
// Bounds that do not depend on the place stand ready: lanes work places out before a workgroup's first request (selects
// for the first place and for a short tile alone: 24 heads of 128 on 8, 200 tokens, 2 slots 11.91 against 11.76 us, 6 heads,
// 150 tokens 10.04 / 9.92, 16 heads, 225 tokens, 2 slots 12.63 / 12.54).
struct SplitTiles {
  unsigned tiles;
  bool shorted;
  unsigned base, top;   // the tile that places count from, and the last one, counted from there
  unsigned rot_end, rot_mask, rot_m;

  WE_TILES_FN SplitTiles(unsigned begin, unsigned end, bool shorted_, unsigned rot_g, unsigned rot_m_)
      : tiles(end - begin), shorted(shorted_), rot_mask(rot_g - 1u), rot_m(rot_m_) {
    const unsigned alone = shorted && tiles == 1u ? 1u : 0u;
    base = begin - alone;
    top = tiles - 1u + alone;
    rot_end = (tiles - (shorted ? 1u : 0u)) & ~rot_mask;
  }
  WE_TILES_FN unsigned count() const { return tiles; }
  // tile of the split's k-th place (the short tile's, 0, wraps around to the largest number there is: the last tile)
  WE_TILES_FN unsigned at(unsigned k) const {
    k -= shorted ? 1u : 0u;
    const unsigned turned = (k & ~rot_mask) | ((k + rot_m) & rot_mask);
    k = k < rot_end ? turned : k;
    return base + (k < top ? k : top);
  }
  // place that the request after the one for place k is for: the last one again once there
  WE_TILES_FN int next(int k) const { return k < (int)top ? k + 1 : k; }
};

}  // namespace we
