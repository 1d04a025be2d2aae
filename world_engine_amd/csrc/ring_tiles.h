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
struct SplitTiles {
  unsigned begin, end;
  bool shorted;
  unsigned rot_g, rot_m;

  WE_TILES_FN unsigned count() const { return end - begin; }
  // tile of the split's k-th place
  WE_TILES_FN unsigned at(unsigned k) const {
    const unsigned rot_end = (count() - (shorted ? 1u : 0u)) & ~(rot_g - 1u);
    const bool head = shorted && k == 0;
    if (shorted && k > 0) --k;  // (the short tile stands in front of the others)
    if (k < rot_end) k = (k & ~(rot_g - 1u)) | ((k + rot_m) & (rot_g - 1u));
    // Only the first request keeps to the keys that the short tile has: the rows behind the last one are nobody's.
    // Where it is all there is, the requests that follow it go to the whole tile in front of it.
    const unsigned top = end - (shorted && count() == 1 ? 2u : 1u), t = begin + k;
    return head ? end - 1 : (t < top ? t : top);
  }
  // place that the request after the one for place k is for: the last one again once there (a short tile alone is
  // followed by the whole one in front of it; the bound is the same for every k)
  WE_TILES_FN int next(int k) const {
    const int last = shorted && count() == 1 ? 1 : (int)count() - 1;
    return k < last ? k + 1 : k;
  }
};

}  // namespace we
