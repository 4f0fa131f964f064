// Backward of the chunked SGSA forward on gfx950 (chunk_sgsa's gradient).
//
// The reference differentiates chunk_sgsa by recomputing the forward in torch
// under autograd (modelings/sgsa_ops/chunk_bwd.py:12-77; the plan of a kernel
// backward is modelings/sgsa_bwd_derivation.md:699-832).  Here the gradient of
// the chunk form is written out and run on fp32 MFMA, for bf16 or fp32 inputs:
//
//   1. chunk_intra_kernel (chunk.hip): per chunk the WY inverse A = (I+T)^-1 and
//      the log-decay prefix l;
//   2. chunk_maps_kernel, parallel over chunks: the chunk's affine state map
//      S' = Phi S + Pm, Phi = e^l_L I - V^T diag(e^l_tau) kappa, Pm = V^T nu with
//      V = A^T diag(c) kappa; chunk_scan_kernel over the chunks: the chunk-start
//      states (the fp32 forward's own first stages, chunk.hip);
//   3. chunk_bwd_pre_kernel, parallel: X1 = P^T dO and the state-independent
//      part of the state gradient's step, Y2 = Q^T diag(e^l) dO -
//      kappa^T diag(e^l_tau) A^T X1; the scan from the last chunk: the state
//      gradient at every chunk end, G <- Phi^T G + Y2 (Phi^T is the adjoint of
//      the state map);
//   4. chunk_bwd_grad_kernel, parallel over chunks: every input gradient of a
//      chunk from its start state S, its end gradient G and its inputs.
//
// Per chunk (tokens t, samples i at token tau_i, M = 2L samples with the
// sparse write, lambda = beta / alpha per sample):
//
//   P_ti = 1[tau_i <= t] exp(l_t - l_tau_i) lambda_i (q_t . kappa_i)
//   c_i  = lambda_i exp(l_L - l_tau_i),   l_L the chunk's last prefix
//   R    = A (nu - diag(e^l_tau) kappa S),   o = diag(e^l) Q S + P R,   S' = e^l_L S + kappa^T diag(c) R
//
// and with dO the output gradient of the chunk and G = dS':
//
//   dR = P^T dO + diag(c) kappa G;   dnu = A^T dR;   Z = A^T dW = -dnu S^T  (W = A diag(e^l_tau) kappa)
//   dS = Q^T diag(e^l) dO + e^l_L G - W^T dR                 (the scan's step)
//   dP = dO R^T;  Y = dP * 1[tau<=t] exp(l_t - l_tau) lambda
//   dq = diag(e^l) dO S^T + Y kappa
//   dT = -A^T dA A^T = -(dnu U^T + Z W^T) = -dnu (U - W S)^T = -dnu R^T
//   X  = dT * 1[tau_j < tau_i] exp(l_tau_i - l_tau_j)
//   dkappa = Y^T Q + diag(c) R G^T + diag(e^l_tau) Z + X diag(lambda) kappa + diag(lambda) X^T kappa
//   dlambda_j = sum_t dP_tj exp(.) (q_t . kappa_j) + sum_i X_ij (kappa_i . kappa_j) + dc_j exp(l_L - l_tau_j)
//   dl: from P (dP_ti P_ti to l_t, minus to l_tau_i), from diag(e^l) Q S
//       (e^l_t q_t^T S dO_t), from c (dc_i c_i to l_L, minus to l_tau_i), from
//       e^l_L S (e^l_L <G, S>), from W (e^l_tau_i kappa_i . Z_i) and from T
//       (X_ij lambda_j (kappa_i . kappa_j) to l_tau_i, minus to l_tau_j);
//   dgamma_p = [gamma_p >= 1e-6] / gamma_p * sum_{t >= p in the chunk} dl_t
//
// with dc_i = (kappa G)_i . R_i, and d(initial_state) the scan's dS of chunk 0.
#include <float.h>

#include "chunk_f32.h"
#include "kernels.h"

namespace sgsa {

namespace {

// Stage 3a, parallel over chunks: X1 = P^T dO [M][DP] and the state-independent part of the
// state gradient's step, Y2 = Q^T diag(e^l) dO - kappa^T diag(e^l_tau) A^T X1 [DP][DP].
// grid (NT, B*H), one wave per 16 samples: wave w owns sample tile w of P, X1 and A^T X1, then a
// share of Y2's column tiles.
template <typename X, int M, int DP, bool FULL>
__global__ __launch_bounds__(4 * M) void chunk_bwd_pre_kernel(ChunkBwdArgs a, const float* __restrict__ Ag,
                                                                      const float* __restrict__ lgd,
                                                                      float* __restrict__ X1g,
                                                                      float* __restrict__ Y2g, int NT) {
  constexpr int NW = M / 16, RT = DP / 16, PD = DP + 4, IPT = M / L;
  constexpr int RA = (2 * L > M ? 2 * L : M) * PD;
  // Y2's tiles: NR row tiles of NC column tiles per wave
  constexpr int RS = NW > RT ? NW / RT : 1, NR = RT / RS, NC = RT > NW ? RT / NW : 1;
  __shared__ __align__(16) float ra[RA];       // q and dO rows, later X1, then -diag(e^l_tau) A^T X1
  __shared__ __align__(16) float ks_[M * PD];  // kappa
  __shared__ float logd[L], el[L];
  float* qs = ra;
  float* ds = ra + L * PD;

  const int c = blockIdx.x, bh = blockIdx.y;
  const int T = a.f.T, H = a.f.H, D = a.f.D;
  const int b = bh / H, h = bh % H;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int t0 = c * L;
  const long cb = (long)bh * NT + c;
  const ChunkRows<X, FULL> q((const X*)a.f.q, b, h, t0, T, H, D), dO((const X*)a.d_out, b, h, t0, T, H, D);
  const ChunkRows<X, FULL> kk((const X*)a.f.k, b, h, t0, T, H, D),
      ks((const X*)(M == 2 * L ? a.f.sparse_k : a.f.k), b, h, t0, T, H, D);
  const int it = tri_tile<NW>(w), i = 16 * it + lr, ti = samp_t<M>(i);
  f4 kown[RT];
#pragma unroll
  for (int n = 0; n < RT; ++n) {
    kown[n] = (samp_r<M>(i) ? ks : kk).row4(ti, 16 * n + 4 * lg);
    *reinterpret_cast<f4*>(&ks_[i * PD + 16 * n + 4 * lg]) = kown[n];
  }
  const float lam = strength<M>(a.f, b, h, t0, i);
  for (int e = tid; e < L * (DP / 4); e += 64 * NW) {
    const int t = e / (DP / 4), d = 4 * (e % (DP / 4));
    *reinterpret_cast<f4*>(&qs[t * PD + d]) = q.urow4(t, d);
    *reinterpret_cast<f4*>(&ds[t * PD + d]) = dO.urow4(t, d);
  }
  if (tid < L) {
    const float x = lgd[cb * L + tid];
    logd[tid] = x;
    el[tid] = expf(x);
  }
  __syncthreads();

  // P (columns of the wave's samples), then X1^T = dO^T P
  f4 x1[RT];
  zero_tiles(x1);
#pragma unroll
  for (int I = 0; I < L / 16; ++I) {
    if (it >= IPT * (I + 1)) continue;   // every sample of the wave after the tile's tokens
    f4 p0 = f4_zero(), p1 = f4_zero();
#pragma unroll
    for (int n = 0; n < RT; n += 2) {
      const f4 a0 = *reinterpret_cast<const f4*>(qs + (16 * I + lr) * PD + 16 * n + 4 * lg);
      const f4 a1 = *reinterpret_cast<const f4*>(qs + (16 * I + lr) * PD + 16 * (n + 1) + 4 * lg);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p0 = mma_f32(a0[e], kown[n][e], p0);
        p1 = mma_f32(a1[e], kown[n + 1][e], p1);
      }
    }
    f4 p;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 16 * I + 4 * lg + e;
      p[e] = ti <= t ? expf(logd[t] - logd[ti]) * lam * (p0[e] + p1[e]) : 0.f;
    }
    mm_col<RT, PD>(x1, ds + (16 * I + 4 * lg) * PD + lr, p);
  }
  float* X1 = X1g + cb * M * DP + (long)i * DP;
#pragma unroll
  for (int r = 0; r < RT; ++r) vstore4(X1 + 16 * r + 4 * lg, x1[r]);

  // Y2 = Q^T diag(e^l) dO ...
  const int r0 = NW > RT ? (w % RS) * NR : 0, n0 = NW > RT ? w / RS : w * NC;
  f4 y2[NC][NR];
#pragma unroll
  for (int cn = 0; cn < NC; ++cn) {
    zero_tiles(y2[cn]);
#pragma unroll
    for (int I = 0; I < L / 16; ++I) {
      f4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = 16 * I + 4 * lg + e;
        x[e] = el[t] * ds[t * PD + 16 * (n0 + cn) + lr];
      }
      mm_col<NR, PD>(y2[cn], qs + (16 * I + 4 * lg) * PD + 16 * r0 + lr, x);
    }
  }
  __syncthreads();   // q and dO are dead
#pragma unroll
  for (int r = 0; r < RT; ++r) *reinterpret_cast<f4*>(ra + i * PD + 16 * r + 4 * lg) = x1[r];
  __syncthreads();
  // ... - kappa^T diag(e^l_tau) A^T X1
  const float* Ac = Ag + cb * (NW * (NW + 1) / 2) * 256;
  zero_tiles(x1);
  f4 an = a_col(Ac, it, it, lr, lg);
  for (int kb = it; kb < NW; ++kb) {
    const f4 x = an;
    an = a_col(Ac, kb + 1 < NW ? kb + 1 : kb, it, lr, lg);
    mm_col<RT, PD>(x1, ra + (16 * kb + 4 * lg) * PD + lr, x);
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RT; ++r) *reinterpret_cast<f4*>(ra + i * PD + 16 * r + 4 * lg) = x1[r] * -el[ti];
  __syncthreads();
  float* Y2 = Y2g + cb * DP * DP;
#pragma unroll
  for (int cn = 0; cn < NC; ++cn) {
#pragma unroll 2
    for (int kb = 0; kb < NW; ++kb) {
      f4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = ra[(16 * kb + 4 * lg + e) * PD + 16 * (n0 + cn) + lr];
      mm_col<NR, PD>(y2[cn], ks_ + (16 * kb + 4 * lg) * PD + 16 * r0 + lr, x);
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        Y2[(16 * (r0 + r) + 4 * lg + e) * DP + 16 * (n0 + cn) + lr] = y2[cn][r][e];
    }
  }
}

// Stage 4.  grid (NT, B*H), one wave per 16 samples: every gradient of one chunk.  Wave w owns
// the samples of one tile: its columns of R^T, dR^T, dnu^T, X^T, Y and dkappa^T stay in
// registers from the product that makes them to the last that reads them.  LDS holds the two
// matrices the waves share at a time: S and B = nu - diag(e^l_tau) kappa S; S and G; S and dR; R and
// kappa; X, Y and kappa.
//
// fp32 MFMA work: 39 MFLOP per chunk at M = DP = 128 (triangular products cut at the tile, dT as one
// product) where the direct form of the gradient takes 69, and no intermediate leaves the CU.  bf16, B=4
// T=4096 H=8 D=128 (2048 chunks): 910 us, 87 TFLOP/s, against 3876 us with 16x16 tiles and R, dR, dW, Z,
// dA, X in a per-chunk workspace (968 us with the gate gradients in LDS atomics).  What remains over the 506 us
// of MFMA time is one workgroup per CU at two waves per SIMD: the barriers between phases and the LDS
// reads ahead of each product show.
template <typename X, int M, int DP, bool FULL>
__global__ __launch_bounds__(64 * (M / 16)) void chunk_bwd_grad_kernel(ChunkBwdArgs a,
                                                                       const float* __restrict__ X1g,
                                                                       const float* __restrict__ Hs,
                                                                       const float* __restrict__ lgd,
                                                                       const float* __restrict__ Ag,
                                                                       const float* __restrict__ Gend, int NT) {
  constexpr bool SP = M == 2 * L;
  constexpr int NW = M / 16, RT = DP / 16, PD = DP + 4, IPT = M / L;
  constexpr int NTL = NW * (NW + 1) / 2, NYT = IPT * 10;   // tiles of X, and of Y: sample tile J <= IPT I + IPT - 1
  constexpr int PS0 = (DP > M ? DP : M) * PD, PS1 = (NTL + NYT) * TLS;
  constexpr int NQ = 4 * RT / NW;                           // tiles of dq per wave: NDQ column tiles x NTQ token tiles
  constexpr int NTQ = NQ < 4 ? NQ : 4, NDQ = NQ / NTQ;
  __shared__ __align__(16) float P[PS0 > PS1 ? PS0 : PS1];   // S, then R, then the tiles of X and Y
  __shared__ __align__(16) float Q[(DP > M ? DP : M) * PD];  // B, then G, then dR, then kappa
  __shared__ float lam[M], logd[L], el[L];
  // each wave's own part of dlambda and dl, added up in wave order at the end: the gate gradients repeat bit for
  // bit, which atomics on one array shared by the waves did not
  __shared__ __align__(16) float dlam[NW][M], dl[NW][L];
  __shared__ float red[NW];
  auto yidx = [](int I, int J) { return NTL + IPT * (I * (I + 1) / 2) + J; };

  const int c = blockIdx.x, bh = blockIdx.y;
  const int T = a.f.T, H = a.f.H, D = a.f.D;
  const int b = bh / H, h = bh % H;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int t0 = c * L;
  const long cb = (long)bh * NT + c;
  const ChunkRows<X, FULL> q((const X*)a.f.q, b, h, t0, T, H, D), dO((const X*)a.d_out, b, h, t0, T, H, D);
  const ChunkRows<X, FULL> kk((const X*)a.f.k, b, h, t0, T, H, D),
      ks((const X*)(SP ? a.f.sparse_k : a.f.k), b, h, t0, T, H, D);
  const int it = tri_tile<NW>(w), i = 16 * it + lr, ti = samp_t<M>(i);
  const float* S = Hs + cb * DP * DP;      // [DP][DP] chunk-start state
  const float* G = Gend + cb * DP * DP;    // [DP][DP] state gradient at the chunk end

  const float* Ac = Ag + cb * NTL * 256;
  constexpr int NG = DP * (DP / 4) / (4 * M);   // four-element pieces of G per thread
  f4 kown[RT], gpre[NG];
#pragma unroll
  for (int n = 0; n < RT; ++n) kown[n] = (samp_r<M>(i) ? ks : kk).row4(ti, 16 * n + 4 * lg);
  for (int e = tid; e < DP * (DP / 4); e += 4 * M)
    *reinterpret_cast<f4*>(&P[(e / (DP / 4)) * PD + 4 * (e % (DP / 4))]) = vload4(S + 4 * e);
#pragma unroll
  for (int u = 0; u < NG; ++u) gpre[u] = vload4(G + 4 * (tid + 4 * M * u));
  if (tid < L) {
    const float x = lgd[cb * L + tid];
    logd[tid] = x;
    el[tid] = expf(x);
  }
  if (tid < M) lam[tid] = strength<M>(a.f, b, h, t0, tid);
  dl[w][lane] = 0.f;
#pragma unroll
  for (int u = 0; u < M / 64; ++u) dlam[w][64 * u + lane] = 0.f;
  __syncthreads();
  const float lami = lam[i], dec = expf(logd[L - 1] - logd[ti]), ci = lami * dec, ei = el[ti];
  float own_dlam = 0.f, own_dl = 0.f;   // this lane's part of sample i's dlambda and dl_tau

  // R = A B, B = nu - diag(e^l_tau) kappa S
  f4 rr[RT], dr[RT], dk[RT];
  zero_tiles(dr);
#pragma unroll
  for (int n = 0; n < RT; ++n) mm_col<RT, PD>(dr, P + (16 * n + 4 * lg) * PD + lr, kown[n]);
  {
    const ChunkRows<X, FULL> vv((const X*)a.f.v, b, h, t0, T, H, D),
        vs((const X*)(SP ? a.f.sparse_v : a.f.v), b, h, t0, T, H, D);
#pragma unroll
    for (int r = 0; r < RT; ++r)
      *reinterpret_cast<f4*>(Q + i * PD + 16 * r + 4 * lg) = (samp_r<M>(i) ? vs : vv).row4(ti, 16 * r + 4 * lg) - dr[r] * ei;
  }
  __syncthreads();
  zero_tiles(rr);
  for (int kb = 0; kb <= it; ++kb) mm_col<RT, PD>(rr, Q + (16 * kb + 4 * lg) * PD + lr, a_row(Ac, it, kb, lr, lg));
  __syncthreads();   // B is dead
#pragma unroll
  for (int u = 0; u < NG; ++u) {
    const int e = tid + 4 * M * u;
    *reinterpret_cast<f4*>(&Q[(e / (DP / 4)) * PD + 4 * (e % (DP / 4))]) = gpre[u];
  }
  __syncthreads();
  // kappa G gives dc and dR = X1 + diag(c) kappa G; dkappa starts as diag(c) R G^T
  zero_tiles(dr);
#pragma unroll
  for (int n = 0; n < RT; ++n) mm_col<RT, PD>(dr, Q + (16 * n + 4 * lg) * PD + lr, kown[n]);
  float dc = 0.f;
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const f4 x1 = vload4(X1g + (cb * M + i) * DP + 16 * r + 4 * lg);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      dc += dr[r][e] * rr[r][e];
      dr[r][e] = x1[e] + ci * dr[r][e];
    }
  }
  zero_tiles(dk);
#pragma unroll
  for (int n = 0; n < RT; ++n) mm_row<RT, PD>(dk, Q + lr * PD + 16 * n + 4 * lg, rr[n]);
#pragma unroll
  for (int r = 0; r < RT; ++r) dk[r] *= ci;
  dc = sum_lg(dc);
  own_dlam += lg == 0 ? dc * dec : 0.f;
  own_dl -= lg == 0 ? dc * ci : 0.f;

  // dq starts as diag(e^l) dO S^T (token tiles tq0.., column tiles dq0.. of the wave)
  const int tq0 = (w * NQ) % 4, dq0 = (w * NQ) / 4;
  f4 dq[NDQ][NTQ];
#pragma unroll
  for (int u = 0; u < NDQ; ++u) {
    zero_tiles(dq[u]);
#pragma unroll 2
    for (int n = 0; n < RT; ++n) {
      const f4 s = *reinterpret_cast<const f4*>(P + (16 * (dq0 + u) + lr) * PD + 16 * n + 4 * lg);
      f4 x[NTQ];
#pragma unroll
      for (int I = 0; I < NTQ; ++I) x[I] = dO.urow4(16 * (tq0 + I) + lr, 16 * n + 4 * lg);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int I = 0; I < NTQ; ++I) dq[u][I] = mma_f32(x[I][e], s[e], dq[u][I]);
      }
    }
#pragma unroll
    for (int I = 0; I < NTQ; ++I) {
      const int t = 16 * (tq0 + I) + 4 * lg;
      f4 p;
#pragma unroll
      for (int e = 0; e < 4; ++e) {   // dl_t += e^l_t q_t . (S dO_t)
        dq[u][I][e] *= el[t + e];
        p[e] = sum_lr(q.uat(t + e, 16 * (dq0 + u) + lr) * dq[u][I][e]);
      }
      if (lr == 0) *reinterpret_cast<f4*>(&dl[w][t]) += p;
    }
  }
  // <G, S>, for dl_L
  float gs = 0.f;
  for (int e = tid; e < DP * (DP / 4); e += 64 * NW) {
    const int o = (e / (DP / 4)) * PD + 4 * (e % (DP / 4));
    const f4 x = *reinterpret_cast<const f4*>(P + o), y = *reinterpret_cast<const f4*>(Q + o);
    gs += x[0] * y[0] + x[1] * y[1] + x[2] * y[2] + x[3] * y[3];
  }
  gs = wave_sum(gs) * el[L - 1] + wave_sum(lg == 0 ? dc * ci : 0.f);   // dc_i c_i goes to dl_L too
  if (lane == 0) red[w] = gs;
  __syncthreads();   // G is dead
#pragma unroll
  for (int r = 0; r < RT; ++r) *reinterpret_cast<f4*>(Q + i * PD + 16 * r + 4 * lg) = dr[r];
  __syncthreads();

  // dnu = A^T dR (the v / v-hat gradients), Z = -dnu S^T
  f4 dn[RT], z[RT];
  zero_tiles(dn);
  {
    for (int kb = it; kb < NW; ++kb) mm_col<RT, PD>(dn, Q + (16 * kb + 4 * lg) * PD + lr, a_col(Ac, kb, it, lr, lg));
    const ChunkRows<X, FULL> dv((const X*)a.dv, b, h, t0, T, H, D),
        dsv((const X*)(SP ? a.dsv : a.dv), b, h, t0, T, H, D);
#pragma unroll
    for (int r = 0; r < RT; ++r) (samp_r<M>(i) ? dsv : dv).put4(ti, 16 * r + 4 * lg, dn[r]);
  }
  zero_tiles(z);
#pragma unroll
  for (int n = 0; n < RT; ++n) mm_row<RT, PD>(z, P + lr * PD + 16 * n + 4 * lg, dn[n]);
#pragma unroll
  for (int r = 0; r < RT; ++r) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float y = ei * z[r][e];
      dk[r][e] -= y;
      own_dl -= y * kown[r][e];
    }
  }
  __syncthreads();   // S and dR are dead
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    *reinterpret_cast<f4*>(P + i * PD + 16 * r + 4 * lg) = rr[r];
    *reinterpret_cast<f4*>(Q + i * PD + 16 * r + 4 * lg) = kown[r];
  }
  __syncthreads();

  // X_ij = dT_ij e^(l_tau_i - l_tau_j), dT = -dnu R^T, on tau_j < tau_i, and the T-terms of
  // dlambda and dl (through kappa kappa^T); dkappa += X diag(lambda) kappa
  f4 xr[NW];
#pragma unroll
  for (int J0 = 0; J0 < NW; J0 += 2) {
    if (J0 > it) continue;   // wave-uniform
    f4 dt[2], gk[2];
    zero_tiles(dt);
    zero_tiles(gk);
#pragma unroll
    for (int n = 0; n < RT; ++n) {
      mm_row<2, PD>(dt, P + (16 * J0 + lr) * PD + 16 * n + 4 * lg, dn[n]);
      mm_row<2, PD>(gk, Q + (16 * J0 + lr) * PD + 16 * n + 4 * lg, kown[n]);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int j0 = 16 * (J0 + u) + 4 * lg;
      f4 xl, s, sl;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = j0 + e, tj = samp_t<M>(j);
        const float x = tj < ti ? -dt[u][e] * expf(logd[ti] - logd[tj]) : 0.f;
        const float xg = x * gk[u][e], lj = lam[j];
        xr[J0 + u][e] = x;
        xl[e] = x * lj;
        own_dl += xg * lj;
        s[e] = sum_lr(xg);
        sl[e] = s[e] * lj;
      }
      if (lr == 0) {
        *reinterpret_cast<f4*>(&dlam[w][j0]) = s;   // the wave's only term for these samples
        float* d = &dl[w][samp_t<M>(j0)];
        if constexpr (SP) {
          d[0] -= sl[0] + sl[1];
          d[1] -= sl[2] + sl[3];
        } else {
          *reinterpret_cast<f4*>(d) -= sl;
        }
      }
      if (J0 + u <= it) mm_col<RT, PD>(dk, Q + (16 * (J0 + u) + 4 * lg) * PD + lr, xl);
    }
  }
  wave_lds_sync();   // dl[w]: another lane's words from here on
  // Y and the P-terms of dlambda and dl; dkappa += Y^T Q
  f4 y[L / 16];
#pragma unroll
  for (int I = 0; I < L / 16; ++I) {
    if (it >= IPT * (I + 1)) continue;
    f4 qk = f4_zero(), dp = f4_zero();
#pragma unroll
    for (int n = 0; n < RT; ++n) {
      const f4 x = q.urow4(16 * I + lr, 16 * n + 4 * lg), x2 = dO.urow4(16 * I + lr, 16 * n + 4 * lg);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        qk = mma_f32(x[e], kown[n][e], qk);
        dp = mma_f32(x2[e], rr[n][e], dp);
      }
    }
    f4 s;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 16 * I + 4 * lg + e;
      const float E = ti <= t ? expf(logd[t] - logd[ti]) : 0.f;
      const float de = dp[e] * E;
      y[I][e] = de * lami;
      own_dlam += de * qk[e];
      const float v = y[I][e] * qk[e];
      own_dl -= v;
      s[e] = sum_lr(v);
    }
    if (lr == 0) *reinterpret_cast<f4*>(&dl[w][16 * I + 4 * lg]) += s;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float x[RT];
#pragma unroll
      for (int r = 0; r < RT; ++r) x[r] = q.uat(16 * I + 4 * lg + e, 16 * r + lr);
#pragma unroll
      for (int r = 0; r < RT; ++r) dk[r] = mma_f32(x[r], y[I][e], dk[r]);
    }
  }
  __syncthreads();   // R is dead
#pragma unroll
  for (int J = 0; J < NW; ++J) {
    if (J > it) continue;
    *reinterpret_cast<f4*>(P + tri(it, J) * TLS + lr * TLP + 4 * lg) = xr[J];
  }
#pragma unroll
  for (int I = 0; I < L / 16; ++I) {
    if (it >= IPT * (I + 1)) continue;
    tile_put(P + yidx(I, it) * TLS, y[I], lr, lg);
  }
  __syncthreads();

  // dkappa += diag(lambda) X^T kappa
  {
    f4 x2[RT];
    zero_tiles(x2);
    for (int kb = it; kb < NW; ++kb) {
      f4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = P[tri(kb, it) * TLS + (4 * lg + e) * TLP + lr];
      mm_col<RT, PD>(x2, Q + (16 * kb + 4 * lg) * PD + lr, x);
    }
    const ChunkRows<X, FULL> dko((const X*)a.dk, b, h, t0, T, H, D),
        dsk((const X*)(SP ? a.dsk : a.dk), b, h, t0, T, H, D);
#pragma unroll
    for (int r = 0; r < RT; ++r) (samp_r<M>(i) ? dsk : dko).put4(ti, 16 * r + 4 * lg, dk[r] + x2[r] * lami);
  }
  // dq += Y kappa
  {
    const ChunkRows<X, FULL> dqo((const X*)a.dq, b, h, t0, T, H, D);
#pragma unroll
    for (int u = 0; u < NDQ; ++u) {
      for (int J = 0; J < NW; ++J) {
        f4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = Q[(16 * J + 4 * lg + e) * PD + 16 * (dq0 + u) + lr];
#pragma unroll
        for (int I = 0; I < NTQ; ++I) {
          if (J >= IPT * (tq0 + I + 1)) continue;   // wave-uniform
          const f4 yv = *reinterpret_cast<const f4*>(P + yidx(tq0 + I, J) * TLS + lr * TLP + 4 * lg);
#pragma unroll
          for (int e = 0; e < 4; ++e) dq[u][I] = mma_f32(yv[e], x[e], dq[u][I]);
        }
      }
#pragma unroll
      for (int I = 0; I < NTQ; ++I) {
#pragma unroll
        for (int e = 0; e < 4; ++e) dqo.put(16 * (tq0 + I) + 4 * lg + e, 16 * (dq0 + u) + lr, dq[u][I][e]);
      }
    }
  }
  own_dlam = sum_lg(own_dlam);
  own_dl = sum_lg(own_dl);
  if constexpr (SP) own_dl = xor_add(own_dl, 1);   // a token's two samples are lanes 2n and 2n + 1
  if (lg == 0) {
    dlam[w][i] += own_dlam;
    if (!SP || (lr & 1) == 0) dl[w][ti] += own_dl;
  }
  __syncthreads();
  // dgamma from the suffix sums of dl (one token per lane); dbeta / dalpha from dlambda
  if (w == 0) {
    float x = 0.f;
#pragma unroll
    for (int u = 0; u < NW; ++u) x += dl[u][lane];
    if (lane == L - 1) {
#pragma unroll
      for (int u = 0; u < NW; ++u) x += red[u];
    }
#pragma unroll
    for (int o = 1; o < L; o <<= 1) {
      const float n = __shfl_down(x, o, 64);
      if (lane + o < L) x += n;
    }
    const int t = t0 + lane;
    if (t < T) {
      const long o = (long)(b * T + t) * H + h;
      const float g = a.f.gamma[o];
      a.dgamma[o] = g >= 1e-6f ? x / g : 0.f;
    }
  }
  if (tid < M) {
    const int t = t0 + samp_t<M>(tid);
    if (t < T) {
      const long o = (long)(b * T + t) * H + h;
      float x = 0.f;
#pragma unroll
      for (int u = 0; u < NW; ++u) x += dlam[u][tid];
      if (samp_r<M>(tid)) a.dalpha[o] = x;
      else a.dbeta[o] = x;
    }
  }
}

struct BwdWs {
  float *X1, *A, *lgd, *Phi, *PmY2, *Hs, *Gend;
  size_t bytes;
};

BwdWs bwd_ws(void* base, int B, int T, int H, int D, int sp) {
  const size_t NT = (T + L - 1) / L, M = sp ? 2 * L : L, BH = (size_t)B * H, DP = chunk_f32_dp(D);
  auto al = [](char* p) { return (char*)(((uintptr_t)p + 255) & ~(uintptr_t)255); };
  char* p0 = al((char*)base);
  char* p = p0;
  auto take = [&](size_t n) {
    float* r = (float*)p;
    p = al(p + 4 * n);
    return r;
  };
  BwdWs w;
  w.X1 = take(BH * NT * M * DP);
  w.A = take(BH * NT * (M / 16) * (M / 16 + 1) / 2 * 256);
  w.lgd = take(BH * NT * L);
  w.Phi = take(BH * NT * DP * DP);
  w.PmY2 = take(BH * NT * DP * DP);
  w.Hs = take(BH * NT * DP * DP);
  w.Gend = take(BH * NT * DP * DP);
  w.bytes = (size_t)(p - p0) + 256;
  return w;
}

template <typename X, int M, int DP, bool FULL>
hipError_t launch_bwd_t(const ChunkBwdArgs& a, const BwdWs& w, hipStream_t st) {
  const int NT = (a.f.T + L - 1) / L;
  const int BH = a.f.B * a.f.H;
  const dim3 chunks(NT, BH);
  chunk_bwd_pre_kernel<X, M, DP, FULL><<<chunks, 4 * M, 0, st>>>(a, w.A, w.lgd, w.X1, w.PmY2, NT);
  launch_chunk_scan(DP, true, w.Phi, w.PmY2, BH, NT, a.d_final_state, a.f.D, w.Gend, a.d_initial_state, st);
  chunk_bwd_grad_kernel<X, M, DP, FULL><<<chunks, 4 * M, 0, st>>>(a, w.X1, w.Hs, w.lgd, w.A, w.Gend, NT);
  return hipGetLastError();
}

template <typename X, int M, int DP>
hipError_t launch_bwd_d(const ChunkBwdArgs& a, const BwdWs& w, hipStream_t st) {
  const bool full = rows_full(a.f.D, DP, a.f.H, sizeof(X), {a.f.q, a.f.k, a.f.v, a.f.sparse_k, a.f.sparse_v, a.d_out,
                                                            a.dq, a.dk, a.dv, a.dsk, a.dsv});
  return full ? launch_bwd_t<X, M, DP, true>(a, w, st) : launch_bwd_t<X, M, DP, false>(a, w, st);
}

template <typename X>
hipError_t launch_bwd_x(const ChunkBwdArgs& a, const BwdWs& w, hipStream_t st) {
  const bool small = chunk_f32_dp(a.f.D) == 64;
  if (a.f.sparse_k != nullptr) return small ? launch_bwd_d<X, 2 * L, 64>(a, w, st) : launch_bwd_d<X, 2 * L, 128>(a, w, st);
  return small ? launch_bwd_d<X, L, 64>(a, w, st) : launch_bwd_d<X, L, 128>(a, w, st);
}

}  // namespace

size_t chunk_bwd_workspace_bytes(int B, int T, int H, int D, int has_sparse) {
  return bwd_ws(nullptr, B, T, H, D, has_sparse).bytes;
}

hipError_t launch_chunk_bwd(const ChunkBwdArgs& a, hipStream_t st) {
  const BwdWs w = bwd_ws(a.workspace, a.f.B, a.f.T, a.f.H, a.f.D, a.f.sparse_k != nullptr);
  launch_chunk_states(a.f, w.lgd, w.A, w.Phi, w.PmY2, w.Hs, nullptr, st);
  return a.f.dtype == DT_BF16 ? launch_bwd_x<bf16_t>(a, w, st) : launch_bwd_x<float>(a, w, st);
}

}  // namespace sgsa
