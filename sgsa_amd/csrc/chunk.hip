// Chunked SGSA forward on gfx950: the replacement for the per-chunk Python
// loop of modelings/sgsa_ops/chunk_fwd.py:39-129 and its Triton pieces
// (chunk_fwd_triton.py:19-260).
//
// Per (batch, head) the sequence is cut into chunks of L=64 tokens.  Each
// token carries two virtual write samples (local: k,v,beta; sparse: k~,v^,alpha)
// interleaved as sample i = 2t + r (chunk_fwd.py:53-56), so a chunk has M=128
// samples (M=64 without the sparse write).  With D_t the inclusive chunk-local
// product of gamma (kept as a log-cumsum), and S the state at the chunk start:
//
//   T_ij = 1[tau_j < tau_i] lam_j exp(logD_tau_i - logD_tau_j) (kappa_i . kappa_j)
//   A    = (I + T)^-1                       W = A diag(D_tau) kappa     U = A nu
//   R    = U - W S                          (residuals, all samples)
//   o_t  = D_t S^T q_t + sum_{tau_i <= t} lam_i (D_t / D_tau_i) (q_t . kappa_i) R_i
//   S'   = D_L S + sum_i kappa_i lam_i (D_L / D_tau_i) R_i^T
//
// Four kernels (the first three also open the backward, chunk_bwd.hip):
//   chunk_intra   parallel over all chunks: Gram, transition, blocked inverse A;
//   chunk_maps    parallel over all chunks: the chunk's affine state map
//                 S' = Phi S + Pm;
//   chunk_scan    the fp32 state recurrence over the chunks, per (b, h, 16-column
//                 slice of S); stores the chunk-start states;
//   chunk_out     parallel over all chunks: R and the readout.
// This file is the fp32-input path: all contractions use v_mfma_f32_16x16x4_f32
// with fp32 operands (chunk_f32.h).  bf16 inputs take chunk_bf16.hip.  The head
// dimension is padded to DP = 64 or 128 in LDS and in the workspace; padded
// rows and columns are zero and never stored.
#include "chunk_f32.h"
#include "kernels.h"

namespace sgsa {

// ---------------------------------------------------------------------------
// K3: intra-chunk transform.  grid (NT, B*H), one wave per 16 samples.
//
// Gram of kappa -> T (lower 16x16 tiles in LDS), each 16x16 diagonal block of
// A = (I + T)^-1 by forward substitution (a lane per column, the block's rows
// broadcast from LDS), the off-diagonal blocks by doubling, A_RC = -A_RR T_RC A_CC
// for 16-, 32- and 64-row halves.  A's lower tiles, [NTL][16][16] row-major, and the
// log-decay prefix are all that is written: the kernels that follow apply A where the
// reference's W = A diag(e^l) kappa and U = A nu stand, which saves writing and
// re-reading those two [M][DP] matrices.
//
// Bound by latency: the triangular solves are short dependent steps, so what counts is the two
// workgroups a CU holds (fp32 rows at DP = 128: one).  bf16, B=4 T=4096 H=8 D=128: 74 us; with W
// and U still written here 258 us, and 245 us for the bf16 kernel this one replaced.  fp32,
// B=4 T=1000 H=4 D=64: 17 us (106 us at DP = 128 with a scalar substitution loop).
// ---------------------------------------------------------------------------
// One step of the Gram's k sum for row tiles I0 and I0 + 1 against the wave's own columns,
// from the staged rows: bf16 products are exact in fp32 and take v_mfma_f32_16x16x32_bf16.
template <int DP>
__device__ __forceinline__ void gram2(f4 (&g)[2], const float* rows, int I0, int own, int lr, int lg) {
  constexpr int PK = DP + 4;
#pragma unroll
  for (int n = 0; n < DP / 16; ++n)
    mm_row<2, PK>(g, rows + (16 * I0 + lr) * PK + 16 * n + 4 * lg,
                  *reinterpret_cast<const f4*>(rows + own * PK + 16 * n + 4 * lg));
}
template <int DP>
__device__ __forceinline__ void gram2(f4 (&g)[2], const bf16_t* rows, int I0, int own, int lr, int lg) {
  constexpr int PK = DP + 8;
#pragma unroll
  for (int s = 0; s < DP / 32; ++s) {
    const bf16x8 b = *reinterpret_cast<const bf16x8*>(rows + own * PK + 32 * s + 8 * lg);
#pragma unroll
    for (int u = 0; u < 2; ++u)
      g[u] = mma_bf16(*reinterpret_cast<const bf16x8*>(rows + (16 * (I0 + u) + lr) * PK + 32 * s + 8 * lg), b, g[u]);
  }
}

template <typename X, int M, int DP, bool FULL>
__global__ __launch_bounds__(64 * (M / 16), sizeof(X) == 2 || DP == 64 ? 4 : 2) void chunk_intra_kernel(
    const X* __restrict__ k, const X* __restrict__ sk, const float* __restrict__ beta,
    const float* __restrict__ alpha, const float* __restrict__ gamma, int T, int H, int D, int NT,
    float* __restrict__ logd_out, float* __restrict__ Aout) {
  constexpr int NB = M / 16, PK = DP + 16 / (int)sizeof(X);
  constexpr int NTL = NB * (NB + 1) / 2;
  constexpr int ZT = NB * NB / 4;   // product tiles of one doubling step, at most
  constexpr int UB = M * PK * (int)sizeof(X) > ZT * TLS * 4 ? M * PK * (int)sizeof(X) : ZT * TLS * 4;
  __shared__ __align__(16) unsigned char ub[UB];     // kappa rows; later the doubling's products
  __shared__ __align__(16) float Tt[NTL * TLS];      // lower tiles of T, then of A
  __shared__ float lam[M];
  __shared__ float logd[L];

  const int c = blockIdx.x, bh = blockIdx.y;
  const int b = bh / H, h = bh % H;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform
  const int lr = lane & 15, lg = lane >> 4;
  const int t0 = c * L;
  const long cb = (long)bh * NT + c;
  const ChunkRows<X, FULL> kk(k, b, h, t0, T, H, D), ks(M == 2 * L ? sk : k, b, h, t0, T, H, D);

  if (tid < L) {
    const int t = t0 + tid;
    float x = 0.f;
    if (t < T) x = logf(fmaxf(gamma[(long)(b * T + t) * H + h], 1e-6f));
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float n = __shfl_up(x, o, 64);
      if (lane >= o) x += n;
    }
    logd[tid] = x;
    logd_out[cb * L + tid] = x;
  }
  if (tid < M) {
    const int t = t0 + samp_t<M>(tid);
    float lm = 0.f;
    if (t < T) lm = samp_r<M>(tid) ? alpha[(long)(b * T + t) * H + h] : beta[(long)(b * T + t) * H + h];
    lam[tid] = lm;
  }
  X* rows = reinterpret_cast<X*>(ub);
  float* un = reinterpret_cast<float*>(ub);
  for (int e = tid; e < M * (DP / 4); e += 4 * M) {
    const int i = e / (DP / 4), d = 4 * (e % (DP / 4));
    vstore4(rows + i * PK + d, (samp_r<M>(i) ? ks : kk).row4(samp_t<M>(i), d));   // bf16 rows round-trip exactly
  }
  __syncthreads();

  // Gram and T, columns of tile jt, row tiles I >= jt two at a time
  const int jt = tri_tile<NB>(w), own = 16 * jt + lr;
  for (int I0 = jt & ~1; I0 < NB; I0 += 2) {
    f4 g[2];
    zero_tiles(g);
    gram2<DP>(g, rows, I0, own, lr, lg);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (I0 + u < jt) continue;   // wave-uniform
      const int tj = samp_t<M>(own);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int ti = samp_t<M>(16 * (I0 + u) + 4 * lg + e);
        Tt[tri(I0 + u, jt) * TLS + (4 * lg + e) * TLP + lr] =
            tj < ti ? lam[own] * expf(logd[ti] - logd[tj]) * g[u][e] : 0.f;
      }
    }
  }
  __syncthreads();   // kappa's rows are dead from here on

  // diagonal blocks by forward substitution: lane c (of 16) solves (I + T) x = e_c, the rows of
  // T read ahead four at a time
  if (lane < 16) {
    float* Tb = Tt + tri(w, w) * TLS;
    float x[16];
#pragma unroll
    for (int hf = 0; hf < 4; ++hf) {
      f4 tr[4][4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int q = 0; q <= hf; ++q) tr[i][q] = *reinterpret_cast<const f4*>(Tb + (4 * hf + i) * TLP + 4 * q);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = 4 * hf + u;
        float s = i == lane ? 1.f : 0.f;
#pragma unroll
        for (int j = 0; j < i; ++j) s -= tr[u][j / 4][j % 4] * x[j];
        x[i] = s;
      }
    }
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < 16; ++i) Tb[i * TLP + lane] = x[i];
  }
  __syncthreads();

  // off-diagonal blocks by doubling: for halves of nb tiles, rows R = (2p+1)nb.., columns
  // C = 2p nb..: Z = T_RC A_CC, then A_RC = -A_RR Z
#pragma unroll
  for (int nb = 1; nb < NB; nb <<= 1) {
    const int items = NB / (2 * nb) * nb * nb;
    for (int it = w; it < items; it += NB) {
      const int p = it / (nb * nb), i = (it / nb) % nb, j = it % nb;
      const int Ri = (2 * p + 1) * nb + i, C0 = 2 * p * nb;
      f4 z = f4_zero();
      for (int x = j; x < nb; ++x) z = tile_mm(Tt + tri(Ri, C0 + x) * TLS, Tt + tri(C0 + x, C0 + j) * TLS, z, lr, lg);
      tile_put(un + it * TLS, z, lr, lg);
    }
    __syncthreads();
    for (int it = w; it < items; it += NB) {
      const int p = it / (nb * nb), i = (it / nb) % nb, j = it % nb;
      const int R0 = (2 * p + 1) * nb, C0 = 2 * p * nb;
      f4 a = f4_zero();
      for (int x = 0; x <= i; ++x)
        a = tile_mm(Tt + tri(R0 + i, R0 + x) * TLS, un + ((p * nb + x) * nb + j) * TLS, a, lr, lg);
      tile_put(Tt + tri(R0 + i, C0 + j) * TLS, -a, lr, lg);
    }
    __syncthreads();
  }

  float* Ac = Aout + cb * NTL * 256;
  for (int e = tid; e < NTL * 64; e += 4 * M)
    *reinterpret_cast<f4*>(Ac + 4 * e) = *reinterpret_cast<const f4*>(Tt + (e >> 2) * TLP + 4 * (e & 3));
}

// ---------------------------------------------------------------------------
// The chunk's affine state map S' = Phi S + Pm, parallel over chunks: Phi = e^l_L I - V^T diag(e^l) kappa and Pm = V^T nu for
// V = A^T diag(c) kappa, [DP][DP] each.  grid (NT, B*H), one wave per 16 samples: wave w makes
// V's columns of sample tile w, then a share of the column tiles of Phi and Pm, which use every
// read of the staged V twice.
//
// fp32 MFMA work, 656 products of 32 cycles per wave at M = DP = 128; the staged operand is read
// once for both maps.  bf16, B=4 T=4096 H=8 D=128: 235 us, 94 TFLOP/s, against 539 us for 16x16
// tiles that each read both operands from LDS.
// ---------------------------------------------------------------------------
template <typename X, int M, int DP, bool FULL>
__global__ __launch_bounds__(4 * M) void chunk_maps_kernel(ChunkArgs f, const float* __restrict__ lgd,
                                                               const float* __restrict__ Ag,
                                                               float* __restrict__ Phig, float* __restrict__ Pmg,
                                                               int NT) {
  constexpr int NW = M / 16, RT = DP / 16, PD = DP + 4, NTL = NW * (NW + 1) / 2;
  constexpr int RS = NW > RT ? NW / RT : 1, NR = RT / RS, NC = RT > NW ? RT / NW : 1;
  __shared__ __align__(16) float vs[M * PD];   // c_i kappa_i, then V
  __shared__ float el[L];
  const int c = blockIdx.x, bh = blockIdx.y;
  const int T = f.T, H = f.H;
  const int b = bh / H, h = bh % H;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int t0 = c * L;
  const long cb = (long)bh * NT + c;
  const ChunkRows<X, FULL> kk((const X*)f.k, b, h, t0, T, H, f.D),
      ks((const X*)(M == 2 * L ? f.sparse_k : f.k), b, h, t0, T, H, f.D);
  const ChunkRows<X, FULL> vv((const X*)f.v, b, h, t0, T, H, f.D),
      vsp((const X*)(M == 2 * L ? f.sparse_v : f.v), b, h, t0, T, H, f.D);
  const float* Ac = Ag + cb * NTL * 256;
  const float lL = lgd[cb * L + L - 1];
  if (tid < L) el[tid] = expf(lgd[cb * L + tid]);
  for (int e = tid; e < M * (DP / 4); e += 4 * M) {
    const int i = e / (DP / 4), d = 4 * (e % (DP / 4));
    const float ci = strength<M>(f, b, h, t0, i) * expf(lL - lgd[cb * L + samp_t<M>(i)]);
    *reinterpret_cast<f4*>(&vs[i * PD + d]) = (samp_r<M>(i) ? ks : kk).row4(samp_t<M>(i), d) * ci;
  }
  __syncthreads();
  const int it = tri_tile<NW>(w);
  f4 v[RT];
  zero_tiles(v);
  f4 an = a_col(Ac, it, it, lr, lg);
  for (int kb = it; kb < NW; ++kb) {
    const f4 x = an;
    an = a_col(Ac, kb + 1 < NW ? kb + 1 : kb, it, lr, lg);
    mm_col<RT, PD>(v, vs + (16 * kb + 4 * lg) * PD + lr, x);
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RT; ++r) *reinterpret_cast<f4*>(&vs[(16 * it + lr) * PD + 16 * r + 4 * lg]) = v[r];
  __syncthreads();
  const int r0 = NW > RT ? (w % RS) * NR : 0, n0 = NW > RT ? w / RS : w * NC;
  float* Phi = Phig + cb * DP * DP;
  float* Pm = Pmg + cb * DP * DP;
#pragma unroll 1
  for (int n = n0; n < n0 + NC; ++n) {
    const int col = 16 * n + lr;
    f4 ph[NR], pm[NR];
    zero_tiles(ph);
    zero_tiles(pm);
    auto load = [&](int kb, f4& bk, f4& bv) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int tl = samp_t<M>(16 * kb + 4 * lg + e);
        bk[e] = (samp_r<M>(e) ? ks : kk).uat(tl, col) * el[tl];
        bv[e] = (samp_r<M>(e) ? vsp : vv).uat(tl, col);
      }
    };
    f4 bk, bv;
    load(0, bk, bv);
    for (int kb = 0; kb < NW; ++kb) {
      f4 nk, nv;
      load(kb + 1 < NW ? kb + 1 : kb, nk, nv);
      const float* a = vs + (16 * kb + 4 * lg) * PD + 16 * r0 + lr;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const float x = a[e * PD + 16 * r];
          ph[r] = mma_f32(x, bk[e], ph[r]);
          pm[r] = mma_f32(x, bv[e], pm[r]);
        }
      }
      bk = nk;
      bv = nv;
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 16 * (r0 + r) + 4 * lg + e;
        Phi[row * DP + col] = (row == col ? el[L - 1] : 0.f) - ph[r][e];
        Pm[row * DP + col] = pm[r][e];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The chunk-to-chunk recurrence x <- Phi_c x + Y_c (TR: Phi_c^T, from the last
// chunk), writing x before each step.  Columns of x evolve independently:
// grid (B*H, DP/16), a block owns 16 columns, wave w the row tile w.  A step is
// one MFMA chain per wave over its own 16 rows of Phi, loaded straight into
// registers one step ahead, and one barrier to exchange x through LDS.
//
// A step takes 2.7 to 3.1 us at DP = 128, of which the two waves of a SIMD issue MFMAs (two chains of 16
// each) for 0.85; the rest is the wait for Phi, 64 KB per workgroup and step loaded one step ahead, and the
// barrier.  That is a quarter of a step with a head's whole state in one workgroup (12 us), which is why the
// chunks are not also split into segments: at B=4 T=4096 H=8 D=128 (64 chunks) 197 us against 340 us for
// a segmented scan in three passes.  Longest, 512 chunks of 16 heads: 1.40 ms forward and 1.23 back, against 1.38
// and 1.42 segmented; the whole backward of one head at T = 32768 2.72 against 3.84 ms.
// ---------------------------------------------------------------------------
template <int DP, bool TR>
__global__ __launch_bounds__(4 * DP) void chunk_scan_kernel(const float* __restrict__ phi, const float* __restrict__ y,
                                                            int NT, const float* __restrict__ init, int D,
                                                            float* __restrict__ out, float* __restrict__ last) {
  constexpr int RT = DP / 16, PX = DP + 4;
  __shared__ __align__(16) float xs[2][16 * PX];   // x transposed: [column][row]
  const int bh = blockIdx.x, ct = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int col = 16 * ct + lr, row = 16 * w + 4 * lg;
  const float* ph = phi + (long)bh * NT * DP * DP + (TR ? (long)(4 * lg) * DP + 16 * w + lr : (long)(16 * w + lr) * DP + 4 * lg);
  const float* yb = y + (long)bh * NT * DP * DP + (long)row * DP + col;
  auto load = [&](int c, f4 (&a)[RT], f4& yv) __attribute__((always_inline)) {
    const float* p = ph + (long)c * DP * DP;
    const float* q = yb + (long)c * DP * DP;
#pragma unroll
    for (int n = 0; n < RT; ++n) {
      if constexpr (TR) {
#pragma unroll
        for (int e = 0; e < 4; ++e) a[n][e] = p[(16 * n + e) * DP];
      } else {
        a[n] = vload4(p + 16 * n);
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) yv[e] = q[e * DP];
  };
  f4 x = f4_zero();
  if (init != nullptr) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (row + e < D && col < D) x[e] = init[((long)bh * D + row + e) * D + col];
  }
  f4 a[RT], yv;
  load(TR ? NT - 1 : 0, a, yv);
  *reinterpret_cast<f4*>(&xs[0][lr * PX + row]) = x;
  __syncthreads();
  for (int s = 0; s < NT; ++s) {
    const int c = TR ? NT - 1 - s : s;
    float* o = out + ((long)bh * NT + c) * DP * DP + (long)row * DP + col;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e * DP] = x[e];
    f4 na[RT], ny;
    load(s + 1 < NT ? (TR ? c - 1 : c + 1) : c, na, ny);
    f4 a0 = f4_zero(), a1 = f4_zero();
    const float* xb = &xs[s & 1][lr * PX + 4 * lg];
#pragma unroll
    for (int n = 0; n < RT; n += 2) {
      const f4 b0 = *reinterpret_cast<const f4*>(xb + 16 * n), b1 = *reinterpret_cast<const f4*>(xb + 16 * (n + 1));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a0 = mma_f32(a[n][e], b0[e], a0);
        a1 = mma_f32(a[n + 1][e], b1[e], a1);
      }
    }
    x = a0 + a1 + yv;
    *reinterpret_cast<f4*>(&xs[(s + 1) & 1][lr * PX + row]) = x;
    __syncthreads();   // the other buffer is rewritten only after the next step's barrier
#pragma unroll
    for (int n = 0; n < RT; ++n) a[n] = na[n];
    yv = ny;
  }
  if (last != nullptr) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (row + e < D && col < D) last[((long)bh * D + row + e) * D + col] = x[e];
  }
}

// ---------------------------------------------------------------------------
// K5: chunk readout.  grid (NT, B*H); wave w owns columns [16w, 16w + 16) of the value
// dimension: B = nu - diag(e^l) kappa S, R = A B and o = diag(e^l) q S + P R are one chain of
// its own columns; the waves share kappa and the tiles of P = mask(q kappa^T), made by tiles.
//
// fp32, B=4 T=1000 H=4 D=64: 23 us, against 69 us with S and R read per 16x16 tile from memory.
// ---------------------------------------------------------------------------
template <typename X, int M, int DP, bool FULL>
__global__ __launch_bounds__(4 * DP) void chunk_out_kernel(ChunkArgs f, const float* __restrict__ lgd,
                                                           const float* __restrict__ Ag, const float* __restrict__ Hs,
                                                           int NT) {
  constexpr int NB = M / 16, RT = DP / 16, PD = DP + 4, IPT = M / L, NTL = NB * (NB + 1) / 2;
  constexpr int NYT = IPT * 10;   // tiles of P: sample tile J <= IPT I + IPT - 1 of token tile I
  __shared__ __align__(16) float kap[M * PD];
  __shared__ __align__(16) float ps[NYT * TLS];
  __shared__ float lam[M], logd[L], el[L];
  auto pidx = [](int I, int J) { return IPT * (I * (I + 1) / 2) + J; };

  const int c = blockIdx.x, bh = blockIdx.y;
  const int T = f.T, H = f.H, D = f.D;
  const int b = bh / H, h = bh % H;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform
  const int lr = lane & 15, lg = lane >> 4;
  const int t0 = c * L, col = 16 * w + lr;
  const long cb = (long)bh * NT + c;
  const ChunkRows<X, FULL> q((const X*)f.q, b, h, t0, T, H, D);
  const ChunkRows<X, FULL> kk((const X*)f.k, b, h, t0, T, H, D),
      ks((const X*)(M == 2 * L ? f.sparse_k : f.k), b, h, t0, T, H, D);
  const ChunkRows<X, FULL> vv((const X*)f.v, b, h, t0, T, H, D),
      vs((const X*)(M == 2 * L ? f.sparse_v : f.v), b, h, t0, T, H, D);
  const float* S = Hs + cb * DP * DP + (long)(4 * lg) * DP + col;
  const float* Ac = Ag + cb * NTL * 256;

  f4 sown[RT];
#pragma unroll
  for (int n = 0; n < RT; ++n) {
#pragma unroll
    for (int e = 0; e < 4; ++e) sown[n][e] = S[(16 * n + e) * DP];
  }
  for (int e = tid; e < M * (DP / 4); e += 4 * DP) {
    const int i = e / (DP / 4), d = 4 * (e % (DP / 4));
    *reinterpret_cast<f4*>(&kap[i * PD + d]) = (samp_r<M>(i) ? ks : kk).row4(samp_t<M>(i), d);
  }
  if (tid < L) {
    const float x = lgd[cb * L + tid];
    logd[tid] = x;
    el[tid] = expf(x);
  }
  if (tid < M) lam[tid] = strength<M>(f, b, h, t0, tid);
  __syncthreads();

  for (int y = w; y < NYT; y += RT) {   // P's tiles
    int I = 0;
    while (pidx(I + 1, 0) <= y) ++I;
    const int J = y - pidx(I, 0);
    f4 p0 = f4_zero(), p1 = f4_zero();
#pragma unroll
    for (int n = 0; n < RT; n += 2) {
      const f4 a0 = q.urow4(16 * I + lr, 16 * n + 4 * lg), a1 = q.urow4(16 * I + lr, 16 * (n + 1) + 4 * lg);
      const f4 b0 = *reinterpret_cast<const f4*>(kap + (16 * J + lr) * PD + 16 * n + 4 * lg);
      const f4 b1 = *reinterpret_cast<const f4*>(kap + (16 * J + lr) * PD + 16 * (n + 1) + 4 * lg);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p0 = mma_f32(a0[e], b0[e], p0);
        p1 = mma_f32(a1[e], b1[e], p1);
      }
    }
    const int i = 16 * J + lr, ti = samp_t<M>(i);
    f4 p;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 16 * I + 4 * lg + e;
      p[e] = ti <= t ? lam[i] * expf(logd[t] - logd[ti]) * (p0[e] + p1[e]) : 0.f;
    }
    tile_put(ps + y * TLS, p, lr, lg);
  }
  // B, then R = A B
  f4 bb[NB], rr[NB];
  zero_tiles(bb);
  zero_tiles(rr);
#pragma unroll
  for (int n = 0; n < RT; ++n) mm_row<NB, PD>(bb, kap + lr * PD + 16 * n + 4 * lg, sown[n]);
#pragma unroll
  for (int J = 0; J < NB; ++J) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int tl = samp_t<M>(16 * J + 4 * lg + e);
      bb[J][e] = (samp_r<M>(e) ? vs : vv).uat(tl, col) - el[tl] * bb[J][e];
    }
  }
#pragma unroll
  for (int J = 0; J < NB; ++J) {
#pragma unroll
    for (int I = J; I < NB; ++I) {
      const f4 x = a_row(Ac, I, J, lr, lg);
#pragma unroll
      for (int e = 0; e < 4; ++e) rr[I] = mma_f32(x[e], bb[J][e], rr[I]);
    }
    __builtin_amdgcn_sched_barrier(0);   // else every tile of A is loaded ahead, and spills
  }
  // o = diag(e^l) q S + P R
  f4 o[L / 16];
  zero_tiles(o);
#pragma unroll
  for (int n = 0; n < RT; ++n) {
    f4 x[L / 16];
#pragma unroll
    for (int I = 0; I < L / 16; ++I) x[I] = q.urow4(16 * I + lr, 16 * n + 4 * lg);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
      for (int I = 0; I < L / 16; ++I) o[I] = mma_f32(x[I][e], sown[n][e], o[I]);
    }
  }
#pragma unroll
  for (int I = 0; I < L / 16; ++I) {
#pragma unroll
    for (int e = 0; e < 4; ++e) o[I][e] *= el[16 * I + 4 * lg + e];
  }
  __syncthreads();   // P's tiles
#pragma unroll
  for (int J = 0; J < NB; ++J) {
#pragma unroll
    for (int I = J / IPT; I < L / 16; ++I) {
      const f4 x = *reinterpret_cast<const f4*>(ps + pidx(I, J) * TLS + lr * TLP + 4 * lg);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[I] = mma_f32(x[e], rr[J][e], o[I]);
    }
  }
  const ChunkRows<X, FULL> out((const X*)f.out, b, h, t0, T, H, D);
#pragma unroll
  for (int I = 0; I < L / 16; ++I) {
#pragma unroll
    for (int e = 0; e < 4; ++e) out.put(16 * I + 4 * lg + e, col, o[I][e]);
  }
}

// ---------------------------------------------------------------------------
// Host launcher
// ---------------------------------------------------------------------------

namespace {

struct FwdWs {
  float *lgd, *A, *Phi, *Pm, *Hs;
  size_t bytes;
};

FwdWs fwd_ws(void* base, int B, int T, int H, int D, int sp) {
  const size_t NT = (T + L - 1) / L, NB = sp ? 8 : 4, BH = (size_t)B * H, DP = chunk_f32_dp(D);
  auto al = [](char* p) { return (char*)(((uintptr_t)p + 255) & ~(uintptr_t)255); };
  char* p0 = al((char*)base);
  char* p = p0;
  auto take = [&](size_t n) {
    float* r = (float*)p;
    p = al(p + 4 * n);
    return r;
  };
  FwdWs w;
  w.lgd = take(BH * NT * L);
  w.A = take(BH * NT * NB * (NB + 1) / 2 * 256);
  w.Phi = take(BH * NT * DP * DP);
  w.Pm = take(BH * NT * DP * DP);
  w.Hs = take(BH * NT * DP * DP);
  w.bytes = (size_t)(p - p0) + 256;
  return w;
}

template <typename X, int M, int DP, bool FULL>
void launch_states_t(const ChunkArgs& a, float* lgd, float* A, float* Phi, float* Pm, hipStream_t st) {
  const int NT = (a.T + L - 1) / L;
  const dim3 g(NT, a.B * a.H);
  chunk_intra_kernel<X, M, DP, FULL><<<g, 4 * M, 0, st>>>((const X*)a.k, (const X*)a.sparse_k, a.beta, a.alpha, a.gamma,
                                                          a.T, a.H, a.D, NT, lgd, A);
  chunk_maps_kernel<X, M, DP, FULL><<<g, 4 * M, 0, st>>>(a, lgd, A, Phi, Pm, NT);
}

template <typename X, int M, int DP>
void launch_states_d(const ChunkArgs& a, float* lgd, float* A, float* Phi, float* Pm, hipStream_t st) {
  if (rows_full(a.D, DP, a.H, sizeof(X), {a.k, a.sparse_k, a.v, a.sparse_v}))
    launch_states_t<X, M, DP, true>(a, lgd, A, Phi, Pm, st);
  else
    launch_states_t<X, M, DP, false>(a, lgd, A, Phi, Pm, st);
}

template <typename X>
void launch_states_x(const ChunkArgs& a, float* lgd, float* A, float* Phi, float* Pm, hipStream_t st) {
  const bool small = chunk_f32_dp(a.D) == 64;
  if (a.sparse_k != nullptr) {
    if (small) launch_states_d<X, 2 * L, 64>(a, lgd, A, Phi, Pm, st);
    else launch_states_d<X, 2 * L, 128>(a, lgd, A, Phi, Pm, st);
  } else {
    if (small) launch_states_d<X, L, 64>(a, lgd, A, Phi, Pm, st);
    else launch_states_d<X, L, 128>(a, lgd, A, Phi, Pm, st);
  }
}

template <int M, int DP>
void launch_out_d(const ChunkArgs& a, const FwdWs& w, hipStream_t st) {
  const int NT = (a.T + L - 1) / L;
  const dim3 g(NT, a.B * a.H);
  if (rows_full(a.D, DP, a.H, 4, {a.q, a.k, a.sparse_k, a.v, a.sparse_v, a.out}))
    chunk_out_kernel<float, M, DP, true><<<g, 4 * DP, 0, st>>>(a, w.lgd, w.A, w.Hs, NT);
  else
    chunk_out_kernel<float, M, DP, false><<<g, 4 * DP, 0, st>>>(a, w.lgd, w.A, w.Hs, NT);
}

}  // namespace

size_t chunk_workspace_bytes(int B, int T, int H, int D, int has_sparse) {
  const size_t f32 = fwd_ws(nullptr, B, T, H, D, has_sparse).bytes;
  const size_t b16 = chunk_bf16_workspace_bytes(B, T, H, has_sparse);
  return f32 > b16 ? f32 : b16;
}

void launch_chunk_scan(int dp, bool tr, const float* phi, const float* y, int BH, int NT, const float* init, int D,
                       float* out, float* last, hipStream_t st) {
  const dim3 g(BH, dp / 16);
  if (dp == 64) {
    if (tr) chunk_scan_kernel<64, true><<<g, 256, 0, st>>>(phi, y, NT, init, D, out, last);
    else chunk_scan_kernel<64, false><<<g, 256, 0, st>>>(phi, y, NT, init, D, out, last);
  } else {
    if (tr) chunk_scan_kernel<128, true><<<g, 512, 0, st>>>(phi, y, NT, init, D, out, last);
    else chunk_scan_kernel<128, false><<<g, 512, 0, st>>>(phi, y, NT, init, D, out, last);
  }
}

void launch_chunk_states(const ChunkArgs& a, float* lgd, float* A, float* Phi, float* Pm, float* Hs, float* ht,
                         hipStream_t st) {
  if (a.dtype == DT_BF16) launch_states_x<bf16_t>(a, lgd, A, Phi, Pm, st);
  else launch_states_x<float>(a, lgd, A, Phi, Pm, st);
  launch_chunk_scan(chunk_f32_dp(a.D), false, Phi, Pm, a.B * a.H, (a.T + L - 1) / L, a.initial_state, a.D, Hs, ht, st);
}

hipError_t launch_chunk_fwd(const ChunkArgs& a, hipStream_t st) {
  if (a.dtype == DT_BF16) return launch_chunk_bf16(a, st);
  const FwdWs w = fwd_ws(a.workspace, a.B, a.T, a.H, a.D, a.sparse_k != nullptr);
  launch_chunk_states(a, w.lgd, w.A, w.Phi, w.Pm, w.Hs, a.final_state, st);
  const bool small = chunk_f32_dp(a.D) == 64;
  if (a.sparse_k != nullptr) {
    if (small) launch_out_d<2 * L, 64>(a, w, st);
    else launch_out_d<2 * L, 128>(a, w, st);
  } else {
    if (small) launch_out_d<L, 64>(a, w, st);
    else launch_out_d<L, 128>(a, w, st);
  }
  return hipGetLastError();
}

}  // namespace sgsa
