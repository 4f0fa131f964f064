// Building blocks of the fp32 chunk kernels (chunk.hip: the fp32 forward and the
// per-chunk WY factors; chunk_bwd.hip: the backward), on v_mfma_f32_16x16x4_f32.
//
// The products of these kernels run column-owned: a wave owns 16 columns of the
// result (16 write samples, or 16 columns of the state) and holds every row of
// them, NR tiles of 16 rows, in accumulators.  The shared operand (A) is read
// from LDS; the wave's own columns (B) come from registers.  The accumulator
// layout of one product -- lane (lr, lg) holds rows 16r + 4lg + e of column lr --
// is the B operand of the next, with k = 16r + 4lg + e in its e-th MFMA, so
// chains such as R -> R G^T or d_nu -> S d_nu need no exchange between lanes or
// waves.  NR independent accumulators keep the matrix pipe fed at two waves per
// SIMD, and an A operand read once from LDS feeds one MFMA of 32 cycles: 32 of
// the LDS's 128 bytes per clock.
#pragma once

#include <initializer_list>

#include "common.h"
#include "kernels.h"

namespace sgsa {

namespace {

constexpr int L = 64;    // tokens of a chunk
constexpr int TLP = 20;  // row pitch (floats) of a 16x16 tile in LDS: 16-byte rows, and rows 4lg + e
                         // of one column fall into distinct banks
constexpr int TLS = 16 * TLP;

__device__ __host__ constexpr int tri(int I, int J) { return I * (I + 1) / 2 + J; }

// sample i of a chunk (M = 2L: i = 2t + r, r = 0 the local write, 1 the sparse one)
template <int M> __device__ __forceinline__ int samp_t(int i) { return M == 2 * L ? (i >> 1) : i; }
template <int M> __device__ __forceinline__ int samp_r(int i) { return M == 2 * L ? (i & 1) : 0; }

__device__ __forceinline__ void vstore4(float* p, f4 v) { *reinterpret_cast<f4*>(p) = v; }
__device__ __forceinline__ void vstore4(bf16_t* p, f4 v) {
  *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16),
                                            (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16));
}

// The rows of one (b, h) of a [B,T,H,D] tensor within one chunk: token tl in [0, nt),
// zero outside [0, nt) x [0, D).  FULL: D = DP and every row 4-element aligned, so rows
// are read and written four elements at a time; else element by element.
template <typename X, bool FULL>
struct ChunkRows {
  X* p;      // the chunk's first row
  long ts;   // elements from one token to the next
  int nt, D;
  __device__ __forceinline__ ChunkRows(const X* base, int b, int h, int t0, int T, int H, int D_)
      : p(const_cast<X*>(base) + ((long)(b * T + t0) * H + h) * D_), ts((long)H * D_), nt(min(L, T - t0)), D(D_) {}
  __device__ __forceinline__ f4 row4(int tl, int d) const {
    const bool ok = tl < nt;
    const X* r = p + (ok ? tl : 0) * ts;
    f4 v = f4_zero();
    if constexpr (FULL) {
      v = vload4(r + d);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (d + e < D) v[e] = ld(r, d + e);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = ok ? v[e] : 0.f;
    return v;
  }
  // The same where the rows are one tensor's for the whole wave (p in scalar registers):
  // FULL rows through a buffer resource that ends with the chunk's last row, so that rows
  // past it read zeros without a test and an address is one 32-bit offset.
  __device__ __forceinline__ int off(int tl, int d) const { return (tl * (int)ts + d) * (int)sizeof(X); }
  __device__ __forceinline__ auto rsrc() const {
    return __builtin_amdgcn_make_buffer_rsrc(p, 0, off(nt - 1, D), 0x00020000);
  }
  __device__ __forceinline__ f4 urow4(int tl, int d) const {
    if constexpr (!FULL) {
      return row4(tl, d);
    } else if constexpr (sizeof(X) == 4) {
      return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc(), off(tl, d), 0, 0));
    } else {
      const uint2 u = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rsrc(), off(tl, d), 0, 0));
      return f4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                __uint_as_float(u.y & 0xffff0000u)};
    }
  }
  __device__ __forceinline__ float uat(int tl, int d) const {
    if constexpr (!FULL) {
      const bool ok = tl < nt && d < D;
      const float x = ld((const X*)p, ok ? tl * ts + d : 0);
      return ok ? x : 0.f;
    } else if constexpr (sizeof(X) == 4) {
      return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc(), off(tl, d), 0, 0));
    } else {
      return bf16_to_f32((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rsrc(), off(tl, d), 0, 0));
    }
  }
  __device__ __forceinline__ void put4(int tl, int d, f4 v) const {
    if (tl >= nt) return;
    if constexpr (FULL) {
      vstore4(p + tl * ts + d, v);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (d + e < D) st(p, tl * ts + d + e, v[e]);
    }
  }
  __device__ __forceinline__ void put(int tl, int d, float v) const {
    if (tl < nt && (FULL || d < D)) st(p, tl * ts + d, v);
  }
};

// acc[r] += A[16r + .][k] b[k] over the 16 k of one block, A row-major in LDS at pitch P:
// `a` points at row lr, k offset 4lg of the block; b holds the lane's four k (4lg + e).
template <int NR, int P>
__device__ __forceinline__ void mm_row(f4 (&acc)[NR], const float* a, const f4& b) {
  f4 x[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) x[r] = *reinterpret_cast<const f4*>(a + 16 * r * P);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
#pragma unroll
    for (int r = 0; r < NR; ++r) acc[r] = mma_f32(x[r][e], b[e], acc[r]);
  }
}
// The same with A's transpose stored: `a` points at row 4lg of the block, column lr.
template <int NR, int P>
__device__ __forceinline__ void mm_col(f4 (&acc)[NR], const float* a, const f4& b) {
  float x[4][NR];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
#pragma unroll
    for (int r = 0; r < NR; ++r) x[e][r] = a[e * P + 16 * r];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
#pragma unroll
    for (int r = 0; r < NR; ++r) acc[r] = mma_f32(x[e][r], b[e], acc[r]);
  }
}

// 16x16 LDS tiles (row-major, pitch TLP): acc + X Y, and a store from the accumulator layout.
__device__ __forceinline__ f4 tile_mm(const float* X, const float* Y, f4 acc, int lr, int lg) {
  const f4 x = *reinterpret_cast<const f4*>(X + lr * TLP + 4 * lg);
#pragma unroll
  for (int e = 0; e < 4; ++e) acc = mma_f32(x[e], Y[(4 * lg + e) * TLP + lr], acc);
  return acc;
}
__device__ __forceinline__ void tile_put(float* Z, const f4& v, int lr, int lg) {
#pragma unroll
  for (int e = 0; e < 4; ++e) Z[(4 * lg + e) * TLP + lr] = v[e];
}

template <int N>
__device__ __forceinline__ void zero_tiles(f4 (&t)[N]) {
#pragma unroll
  for (int r = 0; r < N; ++r) t[r] = f4_zero();
}

// Sum over the 16 lanes of a row group (lanes with the same lg); every lane gets it.
__device__ __forceinline__ float sum_lr(float v) {
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o, 64);
  return v;
}
// Sum over the four lanes of a column (lanes with the same lr).
__device__ __forceinline__ float sum_lg(float v) {
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

// Eight waves over eight tiles of a triangle, w and 11 - w sharing a SIMD's pair of waves
// with tiles t and 7 - t: each pair carries the same number of tiles.
template <int NW> __device__ __forceinline__ int tri_tile(int w) { return NW == 8 && w >= 4 ? 11 - w : w; }

// Write strength of sample i (0 past the sequence).
template <int M>
__device__ __forceinline__ float strength(const ChunkArgs& f, int b, int h, int t0, int i) {
  const int t = t0 + samp_t<M>(i);
  if (t >= f.T) return 0.f;
  const long o = (long)(b * f.T + t) * f.H + h;
  return samp_r<M>(i) ? f.alpha[o] : f.beta[o];
}

// A's tile (I, J) of a chunk as the B operand of a product over its rows -- rows 4lg + e, the
// wave's column lr -- and over its columns (row lr, columns 4lg + e).
__device__ __forceinline__ f4 a_col(const float* Ac, int I, int J, int lr, int lg) {
  const float* p = Ac + tri(I, J) * 256 + 64 * lg + lr;
  return f4{p[0], p[16], p[32], p[48]};
}
__device__ __forceinline__ f4 a_row(const float* Ac, int I, int J, int lr, int lg) {
  return vload4(Ac + tri(I, J) * 256 + 16 * lr + 4 * lg);
}

// Whether the FULL form of ChunkRows takes these rows: D = DP, four-element alignment, and a
// chunk's span within a buffer resource's 32-bit offsets.
inline bool rows_full(int D, int DP, int H, int elem, std::initializer_list<const void*> ps) {
  bool ok = D == DP && (long)L * H * D * elem < 0x7fffffffL;
  for (const void* p : ps) ok = ok && (p == nullptr || (uintptr_t)p % (4 * elem) == 0);
  return ok;
}

}  // namespace

}  // namespace sgsa
