// Bitonic sort of 64 NS composite keys {hi, lo} held by one wave, descending: after it slot
// NS l + s is in register s of lane l.  Strides below NS stay in a lane, the others exchange
// lanes.
#pragma once

#include "common.h"

namespace sgsa {

// x of lane ^ M in VALU instructions: DPP within a row of 16 lanes, the row and half swaps across
// rows (a shuffle through LDS takes an address and a wait per word).
template <int M>
__device__ __forceinline__ uint32_t lane_xor(uint32_t x, int lane) {
  const int v = (int)x;
  if constexpr (M == 1) return (uint32_t)__builtin_amdgcn_update_dpp(v, v, 0xb1, 0xf, 0xf, false);         // quad_perm 1 0 3 2
  else if constexpr (M == 2) return (uint32_t)__builtin_amdgcn_update_dpp(v, v, 0x4e, 0xf, 0xf, false);    // quad_perm 2 3 0 1
  else if constexpr (M == 4) {   // lane ^ 7 (row_half_mirror), then ^ 3 (quad_perm 3 2 1 0)
    const int y = __builtin_amdgcn_update_dpp(v, v, 0x141, 0xf, 0xf, false);
    return (uint32_t)__builtin_amdgcn_update_dpp(y, y, 0x1b, 0xf, 0xf, false);
  } else if constexpr (M == 8) return (uint32_t)__builtin_amdgcn_update_dpp(v, v, 0x128, 0xf, 0xf, false);  // row_ror 8
  else if constexpr (M == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);   // even rows twice, odd rows twice
    return (lane & 16) ? r[0] : r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);   // low half twice, high half twice
    return (lane & 32) ? r[0] : r[1];
  }
}
__device__ __forceinline__ uint32_t lane_xor(uint32_t x, int m, int lane) {   // m a constant after unrolling
  switch (m) {
    case 1: return lane_xor<1>(x, lane);
    case 2: return lane_xor<2>(x, lane);
    case 4: return lane_xor<4>(x, lane);
    case 8: return lane_xor<8>(x, lane);
    case 16: return lane_xor<16>(x, lane);
    default: return lane_xor<32>(x, lane);
  }
}

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
