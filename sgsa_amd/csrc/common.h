// Shared device helpers for the SGSA gfx950 kernels: element types, bf16
// rounding, MFMA fragment wrappers and wave-level primitives.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sgsa {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

struct bf16_t {
  uint16_t bits;
};

// --- scalar conversions -------------------------------------------------

__device__ __forceinline__ float bf16_to_f32(uint16_t b) {
  return __uint_as_float(static_cast<uint32_t>(b) << 16);
}

// Round-to-nearest-even, the rounding torch uses for float -> bfloat16.
// Round to nearest even (v_cvt_pk_bf16_f32 on gfx950).
__device__ __forceinline__ uint16_t f32_to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

template <typename X> struct elem;
template <> struct elem<float> {
  __device__ __forceinline__ static float load(const float* p, long i) { return p[i]; }
  __device__ __forceinline__ static void store(float* p, long i, float v) { p[i] = v; }
};
template <> struct elem<bf16_t> {
  __device__ __forceinline__ static float load(const bf16_t* p, long i) { return bf16_to_f32(p[i].bits); }
  __device__ __forceinline__ static void store(bf16_t* p, long i, float v) { p[i].bits = f32_to_bf16(v); }
};

// The unsigned (bf16) or plain (fp32) element type of raw tiles.
template <typename X> struct elem_bits;
template <> struct elem_bits<float> { typedef float T; };
template <> struct elem_bits<bf16_t> { typedef uint16_t T; };

template <typename X>
__device__ __forceinline__ float ld(const X* p, long i) { return elem<X>::load(p, i); }
template <typename X>
__device__ __forceinline__ void st(X* p, long i, float v) { elem<X>::store(p, i, v); }

// Four consecutive elements as fp32.
__device__ __forceinline__ f4 vload4(const float* p) { return *reinterpret_cast<const f4*>(p); }
__device__ __forceinline__ f4 vload4(const bf16_t* p) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  return f4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
            __uint_as_float(u.y & 0xffff0000u)};
}

// Order-preserving map fp32 -> uint32 (larger float => larger key).  -0.0 is
// folded onto +0.0 first so the two compare equal, as IEEE comparison does.
__device__ __forceinline__ uint32_t f32_order_key(float f) {
  f = f + 0.0f;
  uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Inverse of f32_order_key.
__device__ __forceinline__ float key_to_f32(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Which of a head's n row blocks (0 the last, with the most keys under causality) workgroup
// position g of n takes, for grids of n * BH workgroups that differ in work.  Usually the heaviest
// go first.  Where the whole grid is resident at once, two workgroups to a CU (256 CUs), nothing is
// left to even that out, and the second 256 go lightest first: position i + 256 lands beside
// position i.  T = 4096 with 16 heads: K1 251 -> 246 us, K2 168 -> 160, block retrieval 376 -> 368;
// the heaviest workgroup's own chain of tiles bounds what is left.
__device__ __forceinline__ int causal_block(int g, int n, int BH) {
  const int g0 = (256 + BH - 1) / BH;
  return n * BH <= 512 && g >= g0 ? n - 1 - (g - g0) : g;
}

// --- MFMA fragments -------------------------------------------------------
// v_mfma_f32_16x16x4_f32 (one block): lane l supplies A[l%16][l/16] and
// B[l/16][l%16]; the accumulator holds C[4*(l/16)+i][l%16] in element i.
__device__ __forceinline__ f4 mma_f32(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// v_mfma_f32_16x16x32_bf16 (gfx950): lane l supplies A[l%16][8*(l/16)+j] and
// B[8*(l/16)+j][l%16], j=0..7; same accumulator layout as above.
__device__ __forceinline__ f4 mma_bf16(bf16x8 a, bf16x8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// fp32 score of an accumulated q.k product: acc * (1/scale), with -0.0 folded
// onto +0.0.  Every kernel that selects on scores or recomputes them goes
// through this one expression, so their scores agree bit for bit.
__device__ __forceinline__ f4 score_of(f4 acc, float mscale) {
#pragma clang fp contract(off)
  return acc * mscale + 0.0f;
}

// Smallest float above x (x finite or -inf; +inf stays +inf).  For scores s
// (never -0.0 or NaN): s > x  <=>  s >= next_up(x).
__device__ __forceinline__ float next_up(float x) {
  uint32_t u = __float_as_uint(x);
  if (u == 0x7f800000u) return x;
  if (u == 0x80000000u) u = 0u;
  return __uint_as_float((int32_t)u >= 0 ? u + 1u : u - 1u);
}

__device__ __forceinline__ f4 f4_zero() {
  f4 z = {0.f, 0.f, 0.f, 0.f};
  return z;
}

// --- wave primitives ------------------------------------------------------

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }
__device__ __forceinline__ int wave_id() { return threadIdx.x >> 6; }

// Between a wave's LDS stores and its lanes' reads of each other's words (a wave's LDS accesses stay in order; this
// keeps the compiler's order).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// x of lane ^ M in VALU instructions: DPP within a row of 16 lanes, the row and half swaps across
// rows.  A shuffle through LDS takes an address, a trip to LDS and a wait per
// word: block retrieval's gather (131072 rows of 16 slots, some 20 reductions each) 214 us with those,
// 204 so.
template <int M>
__device__ __forceinline__ uint32_t lane_xor(uint32_t x, int lane) {
  const int v = (int)x;
  if constexpr (M == 1) return (uint32_t)__builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, true);         // quad_perm 1 0 3 2
  else if constexpr (M == 2) return (uint32_t)__builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, true);    // quad_perm 2 3 0 1
  else if constexpr (M == 4) {   // lane ^ 7 (row_half_mirror), then ^ 3 (quad_perm 3 2 1 0)
    const int y = __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true);
    return (uint32_t)__builtin_amdgcn_update_dpp(0, y, 0x1b, 0xf, 0xf, true);
  } else if constexpr (M == 8) return (uint32_t)__builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, true);  // row_ror 8
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

// op(v, v of lane ^ o), op commutative: at 16 and 32 the two words of the swap are the pair.
template <typename Op>
__device__ __forceinline__ float xor_op(float v, int o, Op op) {
  const uint32_t x = __float_as_uint(v);
  if (o == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  if (o == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  return op(v, __uint_as_float(lane_xor(x, o, 0)));
}
__device__ __forceinline__ float xor_add(float v, int o) {
  return xor_op(v, o, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float xor_max(float v, int o) {
  return xor_op(v, o, [](float a, float b) { return fmaxf(a, b); });
}

__device__ __forceinline__ float xor_lane(float v, int o) {
  return __uint_as_float(lane_xor(__float_as_uint(v), o, lane_id()));
}

// Whole waves only (every lane active), as the two below.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = xor_add(v, o);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = xor_max(v, o);
  return v;
}

// Sum over the aligned group of `w` lanes containing this lane (w a constant power of 2, <= 64).
__device__ __forceinline__ float group_sum(float v, int w) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    if (o < w) v = xor_add(v, o);
  return v;
}

__device__ __forceinline__ int popc64(uint64_t x) { return __popcll(x); }

// Wave ballot straight from the predicate's lane mask (no int round trip).
__device__ __forceinline__ uint64_t ballot64(bool p) { return __builtin_amdgcn_ballot_w64(p); }
// Inclusive prefix sum over the 64 lanes: row_shr 1/2/4/8 within each row of 16
// lanes (lanes past the row edge read 0), then row_bcast 15 adds the last lane
// of rows 0 and 2 to rows 1 and 3 and row_bcast 31 adds lane 31 to rows 2 and 3.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
  int v = (int)x;
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return (uint32_t)v;
}
// Number of set bits of m below this lane.
__device__ __forceinline__ uint32_t lane_rank(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

}  // namespace sgsa
