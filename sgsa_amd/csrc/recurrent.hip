// K6: recurrent SGSA, one token after another (decode step and the reference's
// "recurrent" backend).
//
// Replaces fused_recurrent_sgsa / recurrent_sgsa_fwd_triton
// (modelings/sgsa_ops/recurrent.py:138-175, recurrent_fwd_triton.py:25-145)
// with the semantics of naive_recurrent_sgsa (naive.py:34-57): per token
//   base = gamma_t S
//   S    = base + k_t (beta_t (v_t - base^T k_t))^T
//   S   += kh_t (alpha_t (vh_t - base^T kh_t))^T      (reads base, not the updated S)
//   o_t  = S^T q_t
// One block of 256 threads per (batch, head) and tile of RC = 128 / CS columns
// (the columns of the state, the value dim, evolve independently).  The D x D fp32
// state stays in registers for the whole sequence: thread t owns column j = t % RC
// of its tile and RR = RC / 2 rows ([RR (t / RC), +RR)).  Both predictions base^T k
// and base^T kh are formed from the same registers before either update; the row
// groups are combined through LDS in a fixed order.  The next token's vectors are
// prefetched into registers while the current token runs (recurrent_body.h); calls of four
// tokens or more take recurrent_seq_kernel below.  Decode (T = 1) is bound
// by reading and writing the state, 2 D^2 * 4 bytes per head: with few heads the
// columns are split over CS = 4 blocks so that the whole chip moves it.
#include "common.h"
#include "kernels.h"
#include "recurrent_body.h"

namespace sgsa {

template <typename X, bool SP, int CS>
__global__ __launch_bounds__(256) void recurrent_kernel(RecurrentArgs a) {
  recurrent_body<X, SP, CS>(a);
}

// ---------------------------------------------------------------------------
// Several tokens: the same recurrence without a block barrier per token.
//
// A wave owns 64 / NRG columns and every row: lane (c, rg), rg = lane % NRG, holds rows [16 rg,
// 16 rg + 16) of one column (NRG = 8 row groups, or 4 for D <= 64), so both predictions and the
// readout are sums over neighbouring lanes, a few DPP adds, and the token's only exchange; the
// order of every sum is recurrent_body's.  The vectors of TC tokens are staged in LDS as fp32 by the
// block's four waves, one chunk ahead in registers, with one barrier per chunk; they are stored
// so that the row groups read consecutive 16-byte pieces (no bank conflicts) and the lanes of one
// row group the same address.  Lane rg keeps the outputs of tokens rg (and rg + 4) of the chunk, so
// a chunk's outputs leave in one or two stores.
//
// Bound by the VALU at two waves per SIMD (16 rows x 6 operations a token and lane) and by the
// chain of a token at one.  T = 256, bf16 D = 128 with the sparse write, a call by events, before and after:
// 128 heads 338 -> 152 us, one head 300 -> 112, 512 heads 1060 -> 479; D = 64, 512 heads 1000 -> 164.
// Two columns a lane (half the LDS reads) were slower: 236 us at 128 heads, 192 at one.
// ---------------------------------------------------------------------------
namespace {

constexpr int TC = 8;   // tokens of a chunk

// Sum over the aligned group of N = 4 or 8 lanes, in every lane, in sum_chains' order: quad_perm ^1,
// ^2, then row_half_mirror.  With 4 groups the other four chains are zeros.
template <int N>
__device__ __forceinline__ float sum_row_groups(float x) {
  x += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0xb1, 0xf, 0xf, true));
  x += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0x4e, 0xf, 0xf, true));
  if constexpr (N == 8)
    x += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0x141, 0xf, 0xf, true));
  else
    x += 0.f;
  return x;
}

}  // namespace

template <typename X, bool SP, int NRG>
__global__ __launch_bounds__(256) void recurrent_seq_kernel(RecurrentArgs a, int vec4) {
  constexpr int ROWS = 16 * NRG, WC = 64 / NRG, BC = 4 * WC;   // rows; columns per wave, per block
  constexpr int NO = TC / NRG;   // outputs a lane keeps
  constexpr int NVEC = SP ? 3 : 2, NVAL = SP ? 2 : 1;
  __shared__ __align__(16) float vec[2][TC][NVEC][ROWS];   // k, q, k~
  __shared__ float val[2][TC][NVAL][BC];                   // v, v^ of the block's columns
  __shared__ float gate[2][TC][4];                         // beta, gamma, alpha

  const int bh = blockIdx.x, b = bh / a.H, h = bh % a.H;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = lane % NRG, cl = WC * w + lane / NRG;   // column within the block
  const int c0 = blockIdx.y * BC, col = c0 + cl;
  const int D = a.D, T = a.T, H = a.H;
  const long rs = (long)H * D;   // elements from one token to the next
  const long base = ((long)b * T * H + h) * D, gbase = (long)b * T * H + h;
  const X* src[3] = {reinterpret_cast<const X*>(a.k) + base, reinterpret_cast<const X*>(a.q) + base,
                     reinterpret_cast<const X*>(SP ? a.sparse_k : a.k) + base};
  const X* vsrc[2] = {reinterpret_cast<const X*>(a.v) + base, reinterpret_cast<const X*>(SP ? a.sparse_v : a.v) + base};

  float S[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = 16 * rg + r;
    S[r] = a.initial_state != nullptr && row < D && col < D ? a.initial_state[((long)bh * D + row) * D + col] : 0.f;
  }

  // one chunk's inputs in registers: thread (token, four rows) of each vector, a column of each
  // value row, thread < TC the gates; zero past T (no write, gamma 1) and past D
  const int vt = tid / (ROWS / 4), vd = 4 * (tid % (ROWS / 4));   // vt < TC holds a piece
  const int vp = 4 * NRG * ((vd >> 2) & 3) + (vd >> 4) * 4;       // where its four rows are stored
  constexpr int NX = NVAL * TC * BC / 256;
  f4 pv[NVEC];
  float px[NX], pg[3];
  auto fetch = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NVEC; ++n) {
      pv[n] = f4_zero();
      if (vt < TC && t0 + vt < T) {
        const X* p = src[n] + (t0 + vt) * rs;
        if (vec4) {
          if (vd < D) pv[n] = vload4(p + vd);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (vd + e < D) pv[n][e] = ld(p, vd + e);
        }
      }
    }
#pragma unroll
    for (int x = 0; x < NX; ++x) {
      const int i = tid + 256 * x, n = i / (TC * BC), t = t0 + (i / BC) % TC, vc = c0 + i % BC;
      px[x] = t < T && vc < D ? ld(vsrc[n], t * rs + vc) : 0.f;
    }
    if (tid < TC) {
      const int t = t0 + tid;
      const long o = gbase + (long)t * H;
      pg[0] = t < T ? a.beta[o] : 0.f;
      pg[1] = t < T ? a.gamma[o] : 1.f;
      pg[2] = SP && t < T ? a.alpha[o] : 0.f;
    }
  };
  auto publish = [&](int buf) __attribute__((always_inline)) {
    if (vt < TC) {
#pragma unroll
      for (int n = 0; n < NVEC; ++n) *reinterpret_cast<f4*>(&vec[buf][vt][n][vp]) = pv[n];
    }
#pragma unroll
    for (int x = 0; x < NX; ++x) {
      const int i = tid + 256 * x;
      val[buf][(i / BC) % TC][i / (TC * BC)][i % BC] = px[x];
    }
    if (tid < TC) {
#pragma unroll
      for (int n = 0; n < 3; ++n) gate[buf][tid][n] = pg[n];
    }
  };

  fetch(0);
  publish(0);
  __syncthreads();
  for (int t0 = 0, buf = 0; t0 < T; t0 += TC, buf ^= 1) {
    const bool more = t0 + TC < T;   // block-uniform
    if (more) fetch(t0 + TC);
    float out[NO];
    // a token's vectors are read while the one before it is worked on
    f4 kv[4], qv[4], hv[4];
    auto read = [&](int t) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        kv[j] = *reinterpret_cast<const f4*>(&vec[buf][t][0][4 * NRG * j + 4 * rg]);
        qv[j] = *reinterpret_cast<const f4*>(&vec[buf][t][1][4 * NRG * j + 4 * rg]);
        if constexpr (SP) hv[j] = *reinterpret_cast<const f4*>(&vec[buf][t][NVEC - 1][4 * NRG * j + 4 * rg]);
      }
    };
    read(0);
#pragma unroll
    for (int t = 0; t < TC; ++t) {
      const float bet = gate[buf][t][0], gam = gate[buf][t][1], alp = gate[buf][t][2];
      f4 k4[4], q4[4], h4[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        k4[j] = kv[j];
        q4[j] = qv[j];
        if constexpr (SP) h4[j] = hv[j];
      }
      if (t + 1 < TC) read(t + 1);
      // base = gamma S; predictions base^T k and base^T k~
      float pk = 0.f, ph = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        S[r] *= gam;
        pk = fmaf(S[r], k4[r / 4][r % 4], pk);
        if constexpr (SP) ph = fmaf(S[r], h4[r / 4][r % 4], ph);
      }
      // No writes past T, whatever the state holds: k, beta and alpha are 0 there, but 0 * inf is a NaN that
      // would enter every row of the column.  A mask (up to 2% of the time) and not a branch: a token's loads and
      // the next one's overlap (a loop that breaks at T: 8 to 15% slower with up to 128 heads).
      const uint32_t live = (uint32_t)((t0 + t - T) >> 31);   // all bits, or none
      auto kept = [&](float x) __attribute__((always_inline)) { return __uint_as_float(__float_as_uint(x) & live); };
      const float dl = kept(bet * (val[buf][t][0][cl] - sum_row_groups<NRG>(pk)));
      const float ds = SP ? kept(alp * (val[buf][t][NVAL - 1][cl] - sum_row_groups<NRG>(ph))) : 0.f;
      // rank-1 writes, then the readout o = S^T q
      float po = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        S[r] = fmaf(k4[r / 4][r % 4], dl, S[r]);
        if constexpr (SP) S[r] = fmaf(h4[r / 4][r % 4], ds, S[r]);
        po = fmaf(S[r], q4[r / 4][r % 4], po);
      }
      const float o = sum_row_groups<NRG>(po);
      out[t / NRG] = rg == t % NRG ? o : out[t / NRG];
    }
#pragma unroll
    for (int n = 0; n < NO; ++n) {
      const int t = t0 + rg + NRG * n;
      if (t < T && col < D) st(reinterpret_cast<X*>(a.out), base + t * rs + col, out[n]);
    }
    if (more) publish(buf ^ 1);
    __syncthreads();
  }
  if (a.final_state != nullptr) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = 16 * rg + r;
      if (row < D && col < D) a.final_state[((long)bh * D + row) * D + col] = S[r];
    }
  }
}

template <typename X, bool SP, int NRG>
static void launch_seq_t(const RecurrentArgs& a, hipStream_t st) {
  constexpr int BC = 4 * 64 / NRG;
  bool vec4 = a.D % 4 == 0;
  for (const void* p : {a.q, a.k, a.sparse_k}) vec4 = vec4 && (uintptr_t)p % (4 * sizeof(X)) == 0;
  const dim3 g((unsigned)(a.B * a.H), (unsigned)((a.D + BC - 1) / BC));
  recurrent_seq_kernel<X, SP, NRG><<<g, 256, 0, st>>>(a, vec4);
}

template <typename X, bool SP>
static void launch_rec_t(const RecurrentArgs& a, hipStream_t st) {
  // from 4 tokens on (512 heads of 128, bf16, one-token form and this one: T = 2 31.9 us and 36.3, T = 4 40.0 and 35.2)
  if (a.T >= 4) {
    if (a.D <= 64) launch_seq_t<X, SP, 4>(a, st);
    else launch_seq_t<X, SP, 8>(a, st);
    return;
  }
  if (a.B * a.H < 256) recurrent_kernel<X, SP, 4><<<dim3((unsigned)(a.B * a.H), 4), 256, 0, st>>>(a);
  else recurrent_kernel<X, SP, 1><<<dim3((unsigned)(a.B * a.H), 1), 256, 0, st>>>(a);
}

hipError_t launch_recurrent(const RecurrentArgs& a, hipStream_t st) {
  const bool sp = a.sparse_k != nullptr;
  if (a.dtype == DT_F32) {
    if (sp) launch_rec_t<float, true>(a, st);
    else launch_rec_t<float, false>(a, st);
  } else {
    if (sp) launch_rec_t<bf16_t, true>(a, st);
    else launch_rec_t<bf16_t, false>(a, st);
  }
  return hipGetLastError();
}

}  // namespace sgsa
