// Bitonic sort of 64 NS composite keys {hi, lo} held by one wave, descending: after it slot
// NS l + s is in register s of lane l.  Strides below NS stay in a lane, the others exchange
// lanes.
#pragma once

#include "common.h"

namespace sgsa {

template <int NS>
__device__ __forceinline__ void wave_sort_desc(uint32_t (&hi)[NS], uint32_t (&lo)[NS], int lane) {
  // x is kept where it is the larger (max) or smaller of the pair
  auto keep = [](uint32_t& h, uint32_t& l, uint32_t oh, uint32_t ol, bool max) __attribute__((always_inline)) {
    const bool less = h < oh || (h == oh && l < ol);
    const bool take = less == max;
    h = take ? oh : h;
    l = take ? ol : l;
  };
#pragma unroll
  for (int size = 2; size <= 64 * NS; size <<= 1) {
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      if (stride >= NS) {
        const int m = stride / NS;
        const bool desc = (lane & (size / NS)) == 0;   // size = 64 NS: bit 6 of the lane is 0, descending
        const bool max = ((lane & m) == 0) == desc;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const uint32_t oh = lane_xor(hi[s], m, lane), ol = lane_xor(lo[s], m, lane);
          keep(hi[s], lo[s], oh, ol, max);
        }
      } else {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          if (s & stride) continue;
          const int y = s | stride;
          const bool desc = size >= NS ? (lane & (size / NS)) == 0 : (s & size) == 0;
          const bool less = hi[s] < hi[y] || (hi[s] == hi[y] && lo[s] < lo[y]);
          const bool swap = less == desc;
          const uint32_t h = hi[s], l = lo[s];
          hi[s] = swap ? hi[y] : h;
          lo[s] = swap ? lo[y] : l;
          hi[y] = swap ? h : hi[y];
          lo[y] = swap ? l : lo[y];
        }
      }
    }
  }
}

}  // namespace sgsa
