// Score-buffer form of K1's row lists, for up to BUF_MAXK keys (gfx950).
//
// The row kernel (topk.hip) sweeps a 64-row block's keys twice inside one
// workgroup, with its histograms, candidate collection and emission between the
// tiles: a call of a few thousand rows leaves most CUs idle, and every score is
// formed twice.  Where a row's scores fit a wave's registers it is cheaper to
// write them once:
//
//   buf_score_kernel   64 query rows x 256 keys per workgroup: the scores of the
//                      row kernel bit for bit (the same 32 or 4 dims per MFMA in
//                      the same order, score_of) into rows of a buffer;
//   buf_select_kernel  one wave per row, the row's scores in registers: a
//                      256-bin histogram between their extremes finds the bin of
//                      the cut, a bitwise search over that bin's keys the exact
//                      cut, and the kept keys leave in ascending index.
//
// The buffer is the row kernel's own workspace (TOPK_CAP 8-byte candidates per
// row, 4 KB); longer rows take several passes over slabs of row blocks.
//
// What bounds it, T = 4096 with 16 heads, k = 256: the scores the buffer's bytes (0.55 GB written, 215 us);
// the select VALU issue (92% busy by the counters; 260 us, its sort 78 more): 2620 instructions a row of 2048
// scores on average, some 600 of them the sort's, and one LDS atomic a score, whose bank conflicts take 10%
// of the CUs' cycles.
// B=1 H=16, score_topk before and after, us: bf16 D=128 T=1024 k=64 unsorted 128 -> 54, sorted
// 171 -> 58; T=2048 k=128 207 -> 129, 319 -> 145; T=4096 k=256 479 -> 432, 806 -> 524 (with 128
// heads 3013 -> 3132 unsorted, 3749 -> 3228 sorted); T=8192 1535 -> 2263, 2184 -> 2437.  D=64
// T=4096 1189 -> 385, T=8192 k=512 5172 -> 2113.  fp32 D=64 T=2048 707 -> 191, D=128 T=8192 3557 ->
// 3958.  So with D = 128, where the row kernel reads whole vectors, the line lies at 2048 keys, or
// 4096 where this form also sorts; elsewhere at 8192, the registers' limit.  Unsorted rows that keep
// most of their keys stay on the row kernel there (mostly_kept).
//
// Output contract as the row kernel: counts = min(slots, valid keys), slots past
// it index 0 and -FLT_MAX, top2 the two largest valid scores, ties at the cut to
// the lowest indices; the unsorted order is one ascending run (split = counts).
#include <float.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "wave_sort.h"

namespace sgsa {

namespace {

constexpr int QB = 64;     // query rows per workgroup of the score kernels
constexpr int KB = 256;    // keys per workgroup; buffer rows are a multiple of it
constexpr int DP = 128;
constexpr int CAP = BUF_SORT;   // keys of the cut's bin, and kept keys, that go through LDS

struct BufArgs {
  TopkArgs t;
  float* buf;      // [slab rows][pitch]
  int pitch;
  int g0, ng;      // row blocks of this pass: block g is head g % BH, rows 64 (nqb - 1 - g / BH)..
  int nqb;
};

__device__ __forceinline__ void block_of(const BufArgs& a, int x, int& bh, int& r0) {
  const int BH = a.t.B * a.t.H, g = a.g0 + x;
  bh = g % BH;   // with B*H a multiple of 8 a head's blocks share an XCD
  r0 = QB * (a.nqb - 1 - g / BH);
}
// Keys any row of the block may see.
__device__ __forceinline__ int block_keys(const TopkArgs& t, int r0) {
  return t.causal ? min(t.Tk, min(t.Tq, r0 + QB) + t.q_offset) : t.Tk;
}

// bf16, D = 32 NKS, 16-byte rows: wave w scores keys [64w, 64w + 64) of the workgroup's 256
// against its 64 rows; keys are the MFMA's A operand and rows its B operand, so a lane holds four
// consecutive keys of one row.
template <int NKS>
__global__ __launch_bounds__(256) void buf_score_kernel(BufArgs a, float mscale) {
  constexpr int TP = 68;   // pitch of a wave's 16 x 64 tile
  __shared__ __align__(16) float tile[4][16 * TP];
  int bh, r0;
  block_of(a, blockIdx.x, bh, r0);
  const TopkArgs& t = a.t;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int k0 = blockIdx.y * KB + 64 * w, kend = block_keys(t, r0);
  if (k0 >= kend) return;
  constexpr int D = 32 * NKS;
  const int b = bh / t.H, h = bh % t.H;
  const uint16_t* q = reinterpret_cast<const uint16_t*>(t.q) + ((long)b * t.Tq * t.H + h) * D + 8 * lg;
  const uint16_t* k = reinterpret_cast<const uint16_t*>(t.k) + ((long)b * t.Tk * t.H + h) * D + 8 * lg;
  const long rs = (long)t.H * D;
  bf16x8 qf[QB / 16][NKS], kf[4][NKS];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const uint16_t* p = k + min(k0 + 16 * g + lr, t.Tk - 1) * rs;
#pragma unroll
    for (int s = 0; s < NKS; ++s) kf[g][s] = *reinterpret_cast<const bf16x8*>(p + 32 * s);
  }
#pragma unroll
  for (int g = 0; g < QB / 16; ++g) {
    const uint16_t* p = q + min(r0 + 16 * g + lr, t.Tq - 1) * rs;
#pragma unroll
    for (int s = 0; s < NKS; ++s) qf[g][s] = *reinterpret_cast<const bf16x8*>(p + 32 * s);
  }
  // 16 rows x 64 keys at a time through the wave's LDS, so that a store covers four rows of 256
  // bytes and not sixteen of 64
  float* out = a.buf + ((long)blockIdx.x * QB + lg) * a.pitch + k0 + 4 * lr;
  float* ts = tile[w];
#pragma unroll
  for (int g = 0; g < QB / 16; ++g) {
    f4 c[4];
#pragma unroll
    for (int kg = 0; kg < 4; ++kg) {
      c[kg] = f4_zero();
#pragma unroll
      for (int s = 0; s < NKS; ++s) c[kg] = mma_bf16(kf[kg][s], qf[g][s], c[kg]);
    }
#pragma unroll
    for (int kg = 0; kg < 4; ++kg) *reinterpret_cast<f4*>(ts + lr * TP + 16 * kg + 4 * lg) = score_of(c[kg], mscale);
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<f4*>(out + (long)(16 * g + 4 * j) * a.pitch) = *reinterpret_cast<const f4*>(ts + (4 * j + lg) * TP + 4 * lr);
    wave_lds_sync();
  }
}

// Any type, dimension and alignment: 64 rows x 64 keys, the keys staged in LDS, wave w rows 16w...
template <typename X>
__global__ __launch_bounds__(256) void buf_score_any_kernel(BufArgs a, float mscale, int vec) {
  constexpr bool BF = sizeof(X) == 2;
  constexpr int P = DP + (BF ? 8 : 4), NS = BF ? DP / 32 : DP / 4, EPV = 16 / (int)sizeof(X);
  typedef typename elem_bits<X>::T U;
  __shared__ __align__(16) U ks[64 * P];
  int bh, r0;
  block_of(a, blockIdx.x, bh, r0);
  const TopkArgs& t = a.t;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int k0 = blockIdx.y * 64;
  if (k0 >= block_keys(t, r0)) return;   // block-uniform
  const int b = bh / t.H, h = bh % t.H, D = t.D;
  const U* kb = reinterpret_cast<const U*>(t.k) + ((long)b * t.Tk * t.H + h) * D;
  const long rs = (long)t.H * D;
  if (vec) {   // 16-byte rows, D a multiple of EPV; zero past D and past Tk
    for (int e = tid; e < 64 * (DP / EPV); e += 256) {
      const int r = e / (DP / EPV), d = EPV * (e % (DP / EPV));
      uint4 x = make_uint4(0, 0, 0, 0);
      if (k0 + r < t.Tk && d < D) x = *reinterpret_cast<const uint4*>(kb + (k0 + r) * rs + d);
      *reinterpret_cast<uint4*>(ks + r * P + d) = x;
    }
  } else {
    for (int e = tid; e < 64 * DP; e += 256) {
      const int r = e / DP, d = e % DP;
      U x = 0;
      if (k0 + r < t.Tk && d < D) x = kb[(k0 + r) * rs + d];
      ks[r * P + d] = x;
    }
  }
  const int qr = r0 + 16 * w + lr;
  const bool live = qr < t.Tq;
  const U* qp = reinterpret_cast<const U*>(t.q) + ((long)b * t.Tq * t.H + h) * D + (live ? qr : 0) * rs;
  f4 c[4] = {f4_zero(), f4_zero(), f4_zero(), f4_zero()};
  if constexpr (BF) {
    bf16x8 qf[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      u16x8 x;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int d = 32 * s + 8 * lg + j;
        x[j] = live && d < D ? qp[d] : (uint16_t)0;
      }
      qf[s] = __builtin_bit_cast(bf16x8, x);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
        c[g] = mma_bf16(*reinterpret_cast<const bf16x8*>(ks + (16 * g + lr) * P + 32 * s + 8 * lg), qf[s], c[g]);
    }
  } else {
    float qf[NS];
    const int ns = (D + 3) / 4;   // steps past D add zeros
#pragma unroll
    for (int s = 0; s < NS; ++s) qf[s] = live && 4 * s + lg < D ? qp[4 * s + lg] : 0.f;
    __syncthreads();
#pragma unroll
    for (int s0 = 0; s0 < NS; s0 += 8) {
      if (s0 >= ns) continue;
#pragma unroll
      for (int s = s0; s < s0 + 8; ++s) {
#pragma unroll
        for (int g = 0; g < 4; ++g) c[g] = mma_f32(ks[(16 * g + lr) * P + 4 * s + lg], qf[s], c[g]);
      }
    }
  }
  float* out = a.buf + ((long)blockIdx.x * QB + 16 * w + lr) * a.pitch + k0 + 4 * lg;
#pragma unroll
  for (int g = 0; g < 4; ++g) *reinterpret_cast<f4*>(out + 16 * g) = score_of(c[g], mscale);
}

// The kept keys of a row, `n` of them in ascending index as {order key, ~index} in LDS, to the
// row's slots: sorted by (score desc, index asc) in NS registers a lane, or as they are.
template <int NS>
__device__ __forceinline__ void put_row(const uint2* list, int n, bool sort, int32_t* oi, float* os, int lane) {
  uint32_t hi[NS], lo[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int i = 64 * s + lane;
    hi[s] = lo[s] = 0u;
    if (i < n) {
      const uint2 x = list[i];
      hi[s] = x.x;
      lo[s] = x.y;
    }
  }
  if (sort) wave_sort_desc<NS>(hi, lo, lane);
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int i = sort ? NS * lane + s : 64 * s + lane;
    if (i < n) {
      oi[i] = (int32_t)~lo[s];
      os[i] = key_to_f32(hi[s]);
    }
  }
}

// One wave per row; lane l holds keys 256 i + 4l + e of its row in v[i][e].
template <int NV>
__global__ __launch_bounds__(256) void buf_select_kernel(BufArgs a) {
  __shared__ __align__(16) uint32_t hist_s[4][256];
  __shared__ __align__(16) uint2 list_s[4][CAP];   // the cut bin's keys, then the kept ones
  int bh, r0;
  block_of(a, blockIdx.x / (QB / 4), bh, r0);
  const TopkArgs& t = a.t;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rb = 4 * (blockIdx.x % (QB / 4)) + w, qr = r0 + rb;
  if (qr >= t.Tq) return;   // wave-uniform; no block barrier below
  const int b = bh / t.H;
  const long row = (long)bh * t.Tq + qr;
  int nv = t.causal ? max(0, min(t.Tk, qr + t.q_offset + 1)) : t.Tk, slots = t.top_k;
  if (t.row_nv != nullptr) {
    nv = t.row_nv[(long)b * t.Tq + qr];
    slots = min(slots, t.row_kq[qr]);
  }
  nv = __builtin_amdgcn_readfirstlane(nv);
  const int kq = __builtin_amdgcn_readfirstlane(min(slots, nv));
  const float* sr = a.buf + ((long)(blockIdx.x / (QB / 4)) * QB + rb) * a.pitch + 4 * lane;
  uint32_t* hist = hist_s[w];
  uint2* list = list_s[w];

  // scores; -inf past the valid keys, below every finite score
  f4 v[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    v[i] = f4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if (256 * i < nv) v[i] = *reinterpret_cast<const f4*>(sr + 256 * i);   // wave-uniform
  }
  // the two largest, the smallest of the whole 256-key groups (any lower end serves the bins),
  // and whether one is an infinity or NaN (x * 0 is NaN then); med3 with an end of the finite
  // range is one instruction where fmaxf canonicalises its operands first
  float m1 = -FLT_MAX, m2 = -FLT_MAX, lo = FLT_MAX, zero = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (256 * i >= nv) continue;
    const bool whole = 256 * i + 256 <= nv;   // wave-uniform
    if (!whole) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool ok = 256 * i + 4 * lane + e < nv;
        zero = fmaf(ok ? v[i][e] : 0.f, 0.f, zero);
        if (i == 0) lo = ok ? fminf(lo, v[i][e]) : lo;
        v[i][e] = ok ? v[i][e] : -INFINITY;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = v[i][e];
      m2 = __builtin_amdgcn_fmed3f(m1, m2, x);
      m1 = __builtin_amdgcn_fmed3f(m1, x, FLT_MAX);
      if (whole) {
        lo = __builtin_amdgcn_fmed3f(lo, x, -FLT_MAX);
        zero = fmaf(x, 0.f, zero);
      }
    }
  }
  const bool odd = ballot64(!(zero == 0.f)) != 0;
  if (odd) {   // the largest two as comparisons order them, infinities among them
    m1 = m2 = -FLT_MAX;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if (256 * i >= nv) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float y = 256 * i + 4 * lane + e < nv ? v[i][e] : -FLT_MAX;
        m2 = fmaxf(m2, fminf(m1, y));
        m1 = fmaxf(m1, y);
      }
    }
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float b1 = __shfl_xor(m1, o, 64), b2 = __shfl_xor(m2, o, 64);
    m2 = fmaxf(fminf(m1, b1), fmaxf(m2, b2));
    m1 = fmaxf(m1, b1);
    lo = fminf(lo, __shfl_xor(lo, o, 64));
  }
  if (lane == 0) {
    if (t.top2 != nullptr) {
      t.top2[2 * row] = m1;
      t.top2[2 * row + 1] = m2;
    }
    if (t.counts != nullptr) t.counts[row] = kq;
    if (t.split != nullptr) t.split[row] = kq;
  }
  int32_t* oi = t.indices + row * t.top_k;
  float* os = t.scores + row * t.top_k;
  for (int i = kq + lane; i < t.top_k; i += 64) {
    oi[i] = 0;
    os[i] = -FLT_MAX;
  }
  if (kq <= 0) return;

  // the cut: the kq-th largest score, and how many scores equal to it to take
  uint32_t cut = 0u;
  int neq = 0;
  bool tie = false;    // more scores equal the cut than it takes
  bool keys = odd;     // v holds order keys (0 past the valid keys) instead of scores
  if (!odd && kq < nv) {
    // bin(x) = round((x - lo) 255 / (m1 - lo)) clamped to [0, 255], read from the mantissa of
    // 2^23 + bin: any map that does not decrease in x keeps the selection exact
    const float inv = 255.f / (m1 - lo), bc = 8388608.f - lo * inv;
    auto bin_of = [&](float x) __attribute__((always_inline)) {
      return __float_as_uint(__builtin_amdgcn_fmed3f(fmaf(x, inv, bc), 8388608.f, 8388863.f));
    };
    int cnt = CAP + 1, need = kq;
    uint32_t bin = 0;
    if (inv <= FLT_MAX && fabsf(lo * inv) <= 4194304.f) {
      *reinterpret_cast<uint4*>(hist + 4 * lane) = make_uint4(0, 0, 0, 0);
      wave_lds_sync();
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        if (256 * i >= nv) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) atomicAdd(&hist[bin_of(v[i][e]) & 255u], 1u);   // -inf: bin 0
      }
      wave_lds_sync();
      uint32_t c[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) c[q] = hist[255 - 4 * lane - q];
      const uint32_t tot = c[0] + c[1] + c[2] + c[3], inc = wave_incl_scan(tot), exc = inc - tot;
      const bool hit = exc < (uint32_t)kq && (uint32_t)kq <= inc;
      const int src = (int)__builtin_ctzll(ballot64(hit));   // the totals sum to nv or more: one lane hits
      uint32_t above = exc, cb = 0, bb = 0;
      bool found = false;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (!found && above + c[q] >= (uint32_t)kq) {
          found = true;
          cb = c[q];
          bb = 255 - 4 * lane - q;
        }
        if (!found) above += c[q];
      }
      bin = 0x4b000000u + (uint32_t)__builtin_amdgcn_readlane((int)bb, src);   // as bin_of returns it
      cnt = __builtin_amdgcn_readlane((int)cb, src);
      need = kq - __builtin_amdgcn_readlane((int)above, src);
    }
    if (cnt <= CAP) {
      // the bin's keys through LDS to at most eight registers a lane, then a bitwise search
      int n = 0;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        if (256 * i >= nv) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool in = bin_of(v[i][e]) == bin;
          const uint64_t m = ballot64(in);
          if (m != 0) {
            if (in) list[n + lane_rank(m)].x = f32_order_key(v[i][e]);
            n += popc64(m);
          }
        }
      }
      wave_lds_sync();
      auto search = [&](auto NC) __attribute__((always_inline)) {
        constexpr int N = decltype(NC)::value;
        uint32_t ck[N];
#pragma unroll
        for (int u = 0; u < N; ++u) ck[u] = 64 * u + lane < cnt ? list[64 * u + lane].x : 0u;
        auto count = [&](uint32_t x) __attribute__((always_inline)) {
          int s = 0;
#pragma unroll
          for (int u = 0; u < N; ++u) s += popc64(ballot64(ck[u] >= x));
          return s;
        };
        for (uint32_t bit = 0x80000000u; bit != 0; bit >>= 1)
          if (count(cut | bit) >= need) cut |= bit;
        neq = need - count(cut + 1u);   // the keys of finite scores end below 2^32 - 1
        tie = count(cut) > need;
      };
      if (cnt <= 64) search(std::integral_constant<int, 1>{});
      else search(std::integral_constant<int, CAP / 64>{});
      wave_lds_sync();
    } else {
      keys = true;
    }
  }
  if (keys) {
    // infinities, NaN, or a bin of more than CAP keys: the same search over every key
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if (256 * i >= nv) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[i][e] = __uint_as_float(256 * i + 4 * lane + e < nv ? f32_order_key(v[i][e]) : 0u);
    }
    auto count = [&](uint32_t x) __attribute__((always_inline)) {
      int s = 0;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        if (256 * i >= nv) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) s += popc64(ballot64(__float_as_uint(v[i][e]) >= x));
      }
      return s;
    };
    for (uint32_t bit = 0x80000000u; bit != 0; bit >>= 1)
      if (count(cut | bit) >= kq) cut |= bit;
    neq = kq - (cut == 0xffffffffu ? 0 : count(cut + 1u));
    tie = count(cut) > kq;
  }
  // the kept keys in ascending index, through LDS where they fit it
  const float fcut = kq < nv ? key_to_f32(cut) : -FLT_MAX;
  const bool lds = kq <= CAP;
  int pos = 0, eq = 0;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (256 * i >= nv) continue;
    bool s[4];
    if (!keys && !tie) {
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = v[i][e] >= fcut;
    } else {
      bool q[4];
      int eb = eq;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t key = keys ? __float_as_uint(v[i][e]) : f32_order_key(v[i][e]);
        s[e] = key > cut;
        q[e] = key == cut;   // a kept key's rank among its equals decides
        const uint64_t m = ballot64(q[e]);
        eb += (int)lane_rank(m);
        eq += popc64(m);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[e] = s[e] || (q[e] && eb < neq);
        eb += q[e];
      }
    }
    uint64_t m[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) m[e] = ballot64(s[e]);
    if ((m[0] | m[1] | m[2] | m[3]) == 0) continue;   // wave-uniform
    int at = pos + (int)(lane_rank(m[0]) + lane_rank(m[1]) + lane_rank(m[2]) + lane_rank(m[3]));
    pos += popc64(m[0]) + popc64(m[1]) + popc64(m[2]) + popc64(m[3]);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (s[e]) {
        const int j = 256 * i + 4 * lane + e;
        if (lds) {
          list[at] = make_uint2(keys ? __float_as_uint(v[i][e]) : f32_order_key(v[i][e]), ~(uint32_t)j);
        } else {
          oi[at] = j;
          os[at] = keys ? key_to_f32(__float_as_uint(v[i][e])) : v[i][e];
        }
        ++at;
      }
    }
  }
  if (!lds) return;
  wave_lds_sync();
  const bool sort = t.sort != 0;
  if (kq <= 64) put_row<1>(list, kq, sort, oi, os, lane);
  else if (kq <= 128) put_row<2>(list, kq, sort, oi, os, lane);
  else if (kq <= 256) put_row<4>(list, kq, sort, oi, os, lane);
  else put_row<8>(list, kq, sort, oi, os, lane);
}

}  // namespace

namespace {
// A row's keys rounded up to whole workgroups, and 256 bytes more: rows a power of two apart
// would meet in the same memory channels (T = 4096: 315 us for the scores without, 248 with).
int buf_pitch(const TopkArgs& t) { return (t.Tk + KB - 1) / KB * KB + 64; }
// Row blocks whose buffer rows fit the row kernel's candidate lists (TOPK_CAP entries of 8 bytes
// per query row).
long buf_room(const TopkArgs& t) { return (long)t.B * t.H * t.Tq * TOPK_CAP * 8 / ((long)QB * buf_pitch(t) * 4); }
// Keys of a head's first n rows (a padded sequence counted as a whole one).
long keys_of(const TopkArgs& t, long n) {
  if (!t.causal) return n * t.Tk;
  const long off = t.q_offset, a = std::min(n, std::max(0L, -off)), b = std::min(n, std::max(a, t.Tk - off - 1));
  return (b - a) * (a + b + 2 * off + 1) / 2 + (n - b) * t.Tk;
}
// D = 128, unsorted: whether the keys of rows that keep all of theirs decide.  The row kernel writes such a row
// from one sweep, at half of this form's time a key, and spends some 256 keys' time more on each other row;
// a workgroup's chain of tiles hides behind the others' work from 84 rows of full length to a CU on, 42 where no
// row selects.  Rows of all keys or nearly all, us, row kernel and this form: 32 heads T = 1024 k = 1024
// bf16 70 and 133, fp32 121 and 201; 64 heads T = 2048 k = 1024 651 and 695, k = 700 580 and 584;
// 64 heads T = 640 k = 520 109 and 84, 128 heads 150 and 182; T = 600 k = 300, 128 heads 190 and 140.
bool mostly_kept(const TopkArgs& t) {
  const long kept = t.top_k >= t.Tk ? t.Tq : t.causal ? std::min<long>(t.Tq, std::max<long>(0, (long)t.top_k - t.q_offset)) : 0;
  const long all = keys_of(t, kept), longest = t.causal ? std::min<long>(t.Tk, (long)t.Tq + t.q_offset) : t.Tk;
  return all > 0 && all >= 512 * (t.Tq - kept) && (long)t.B * t.H * keys_of(t, t.Tq) >= (kept < t.Tq ? 84 : 42) * 256 * longest;
}
}  // namespace

bool topk_buf_fits(const TopkArgs& a) {
  if (a.dump != nullptr || a.tl_list != nullptr || a.thr != nullptr) return false;
  const bool sorts = a.sort && a.top_k <= BUF_SORT;
  if (a.Tk > (a.D == DP ? (sorts ? 4096 : 2048) : BUF_MAXK)) return false;
  if (a.D == DP && !sorts && mostly_kept(a)) return false;
  // at most one pass more than whole row blocks take: a few rows of long heads stay on the row kernel
  const long blocks = (long)a.B * a.H * ((a.Tq + QB - 1) / QB);
  return buf_room(a) * ((buf_pitch(a) + 1023) / 1024 + 1) >= blocks;
}

hipError_t launch_score_topk_buf(const TopkArgs& t, float* buf, hipStream_t st) {
  BufArgs a{};
  a.t = t;
  a.buf = buf;
  a.pitch = buf_pitch(t);
  a.nqb = (t.Tq + QB - 1) / QB;
  const float ms = score_multiplier(t.scale, t.scale_mode);
  const int es = t.dtype == DT_F32 ? 4 : 2;
  const bool al = ((uintptr_t)t.q % 16) == 0 && ((uintptr_t)t.k % 16) == 0;
  const bool fast = t.dtype == DT_BF16 && t.D % 32 == 0 && al;
  const int vec = al && t.D % (16 / es) == 0;
  const long blocks = (long)t.B * t.H * a.nqb;
  const long room = buf_room(t);   // at least 1 (topk_buf_fits)
  const int nvec = a.pitch / 256;
  for (long g0 = 0; g0 < blocks; g0 += room) {
    a.g0 = (int)g0;
    a.ng = (int)std::min(room, blocks - g0);
    if (fast) {
      const dim3 g((unsigned)a.ng, (unsigned)(a.pitch / KB));
      switch (t.D / 32) {
        case 1: buf_score_kernel<1><<<g, 256, 0, st>>>(a, ms); break;
        case 2: buf_score_kernel<2><<<g, 256, 0, st>>>(a, ms); break;
        case 3: buf_score_kernel<3><<<g, 256, 0, st>>>(a, ms); break;
        default: buf_score_kernel<4><<<g, 256, 0, st>>>(a, ms); break;
      }
    } else {
      const dim3 g((unsigned)a.ng, (unsigned)((t.Tk + 63) / 64));
      if (t.dtype == DT_F32) buf_score_any_kernel<float><<<g, 256, 0, st>>>(a, ms, vec);
      else buf_score_any_kernel<bf16_t><<<g, 256, 0, st>>>(a, ms, vec);
    }
    const dim3 gs((unsigned)(a.ng * (QB / 4)));
    if (nvec <= 1) buf_select_kernel<1><<<gs, 256, 0, st>>>(a);
    else if (nvec <= 2) buf_select_kernel<2><<<gs, 256, 0, st>>>(a);
    else if (nvec <= 4) buf_select_kernel<4><<<gs, 256, 0, st>>>(a);
    else if (nvec <= 8) buf_select_kernel<8><<<gs, 256, 0, st>>>(a);
    else if (nvec <= 16) buf_select_kernel<16><<<gs, 256, 0, st>>>(a);
    else buf_select_kernel<32><<<gs, 256, 0, st>>>(a);
  }
  return hipGetLastError();
}

}  // namespace sgsa
