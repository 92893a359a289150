// The gated delta rule over 64-token chunks (ops/seqmix.py::delta_rule_scan, portions of many tokens): per head, with
// decays g_t per key channel (or one for all of them),
//   S_t = g_t S_{t-1} + k_t w_t^T,  w_t = beta_t (v_t - (g_t S_{t-1})^T k_t),  o_t = S_t^T q_t.
// With D_t the product of the decays up to t inside the chunk, D_{s..t} that of those after s up to t, and S_in the state
// that enters it,
//   (I + A) W = beta V - (beta k D) S_in,   A[t, s] = beta_t sum_n k_t k_s D_{s..t}  (s < t)
//   S_out = D_end S_in + sum_s (k_s D_{s..end}) w_s^T
//   o_t = (q_t D_t)^T S_in + sum_{s<=t} C[t, s] w_s,   C[t, s] = sum_n q_t k_s D_{s..t}
// (1) delta_chunk_solve_kernel, parallel over chunks: A and C, then U and M with (I + A) [U | M] = [beta V | beta k D]
//     by forward substitution over 16-token blocks (the blocks' own 16 x 16 systems inverted); also q D, k D_{..end}, D_end.
// (2) delta_chunk_scan_kernel, chunk by chunk: W = U - M S_in and the next state, 4 to 16 value columns per workgroup.
// (3) delta_chunk_out_kernel, parallel over chunks: the outputs.
// Sums, products and decays are fp64 (v_mfma_f64_16x16x4_f64, 4x4x4_4b in (2), and plain FMAs); fp32 are the inputs, q D and k D_{..end}, the
// states that (3) reads and the one that leaves.  In fp32 the form loses to the recurrence: with keys alike (cosine 0.98,
// beta near 1) U and M S_in nearly cancel and the w_t of a chunk nearly add up to nothing, 1.1e-6 to 2e-6 against its 0.9e-7,
// with random keys 1.6e-7 to 2.6e-7 against 1.1e-7.  No decay ratio is a quotient: from a token s to a later 16-token block it
// is what s's block decays after s, times the blocks between, times t's block up to t; inside a block factor by factor.
// A product's register r holds row 4 r + g in lane group g, so its four registers are the second operand of four steps
// whose k runs over 4 r + g: results feed products without a shuffle.  What a first operand takes lies permuted (PERM), so
// that a lane's four numbers are neighbours.
//
// Bound: token by token, every token costs a chain of two row sums (about 530 clocks); here the chain is two products
// and two barriers per 64 tokens, in fp64 at half the rate of fp32.  16 heads, 4096 tokens, us, token by token / this: 64 x 64
// states 916 / 198 ((1) 90, (2) 74, (3) 37), 128 x 128 states 1512 / 421; 512 tokens 114 / 56 and 181 / 86.
#include "seqmix_common.h"

namespace {

typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));
__device__ __forceinline__ v4d mfma4d(double a, double b, v4d c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
// one 16-wide block of k, 4 r + g4 of it in element r of a and b
__device__ __forceinline__ v4d mma16(const v4d& a, const v4d& b, v4d c) {
#pragma unroll
  for (int r = 0; r < 4; ++r) c = mfma4d(a[r], b[r], c);
  return c;
}
__device__ __forceinline__ v4d widen(const float4& f) { return v4d{(double)f.x, (double)f.y, (double)f.z, (double)f.w}; }
__device__ __forceinline__ constexpr int PERM(int e) { return (e & 3) * 4 + (e >> 2); }   // where element e of 16 lies
__device__ __forceinline__ bool finite4(const v4d& x) {
  const v4d d = x - x;
  return d[0] == 0. && d[1] == 0. && d[2] == 0. && d[3] == 0.;
}

// What one launch covers: of every portion of `least` tokens or more (shorter ones run token by token) the chunks c0 .. c0 + most
// - 1, for at most `room` chunks of scratch in all
struct DeltaPart {
  int least, c0, most, room;
};
__device__ __forceinline__ int chunks_of(int len, const DeltaPart& dp) {
  return len < dp.least ? 0 : min(max((len + CL - 1) / CL - dp.c0, 0), dp.most);
}
// a portion's first chunk among those of the launch, and whether all of its chunks have room (the host counted them)
__device__ __forceinline__ bool first_chunk(const int* __restrict__ seq_len, int s, const DeltaPart& dp, size_t& b) {
  b = 0;
  for (int i = 0; i < s; ++i) b += chunks_of(seq_len[i], dp);
  return b + chunks_of(seq_len[s], dp) <= (size_t)dp.room;
}

// Scratch per (chunk, head), NP = 64, 128 or 256 channels (zero past N) and PP = P rounded up to 16:
//   fp64  M [4 token blocks][NP / 16][token][PERM channel]  U (later W) [64][PP]  Cs [4][4][token][PERM earlier token]
//         cdec [NP / 16][PERM channel]
//   fp32  Qe [4][NP / 16][token][PERM channel]  Kd [NP / 16][4][channel][PERM token]  states [NP / 16][PP][PERM channel]
struct DeltaScratch {
  double *M, *U, *Cs, *cdec;
  float *Qe, *Kd, *sin;
};
// VEC: 16-byte loads of the prepared rows.  ONE: one decay for all key channels of a head (the ratios are then taken out
// of the products).
template <typename T, bool VEC, bool ONE>
__global__ void __launch_bounds__(NT, 2) delta_chunk_solve_kernel(const float* __restrict__ prep, int prep_ld,
                                                                  const T* __restrict__ qkv, int Cq,
                                                                  const int* __restrict__ seq_len, const int* __restrict__ seq_off,
                                                                  DeltaScratch sc, DeltaPart dp, int H, int G, int N, int NP, int P, int PP) {
  constexpr int NK = 32, LQ = NK + 4, LA = CL + 4, LG = ONE ? 1 : CL;
  __shared__ __attribute__((aligned(16))) float Q_s[CL][LQ], K_s[CL][LQ], G_s[LG][LQ];
  // decays of a token's 16-token block up to and with it / after it; A takes their place
  __shared__ __attribute__((aligned(16))) double be_s[ONE ? CL * LA : 2 * CL * LQ];
  __shared__ double b_s[CL], g_s[CL], f_s[CL], r_s[CL], pc_s[CL], sc_s[CL];   // beta; ONE: decays, in the block, in the chunk
  static_assert(ONE || 2 * LQ >= LA, "A fits");
  auto B_s = reinterpret_cast<double(*)[LQ]>(be_s);
  auto E_s = reinterpret_cast<double(*)[LQ]>(be_s + CL * LQ);
  auto A_s = reinterpret_cast<double(*)[LA]>(be_s);
  const int c = blockIdx.x, s = blockIdx.y, h = blockIdx.z, len = seq_len[s];
  size_t cb;
  if (c >= chunks_of(len, dp) || !first_chunk(seq_len, s, dp, cb)) return;
  const int t0 = (dp.c0 + c) * CL, tc = min(CL, len - t0), GN = G * N, GD = ONE ? 1 : N;
  const size_t row0 = (size_t)seq_off[s] + t0;
  cb = (cb + c) * H + h;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g4 = lane >> 4;
  const float* pr = prep + row0 * prep_ld;
  const float *qb = pr + (h / (H / G)) * N, *kb = qb + GN, *gb = pr + 2 * GN + h * GD, *bb = pr + 2 * GN + H * GD + h;
  double *M = sc.M + cb * CL * NP, *U = sc.U + cb * CL * PP, *Cs = sc.Cs + cb * CL * CL, *cdec = sc.cdec + cb * NP;
  float *Qe = sc.Qe + cb * CL * NP, *Kd = sc.Kd + cb * CL * NP;
  if (tid < CL) {                                            // (one wave)
    const size_t at = (size_t)min(tid, tc - 1) * prep_ld;
    b_s[tid] = tid < tc ? (double)bb[at] : 0.;
    if constexpr (ONE) {
      const double g = tid < tc ? (double)gb[at] : 1.;
      double up = g, dn = g;
#pragma unroll
      for (int d = 1; d < 16; d <<= 1) {                     // inclusive products inside the 16-token block, both ways
        const double a = __shfl_up(up, d, 64), b = __shfl_down(dn, d, 64);
        if (l16 >= d) up *= a;
        if (l16 + d < 16) dn *= b;
      }
      const double after = __shfl_down(dn, 1, 64), ex = l16 < 15 ? after : 1.;
      double t[4], pre = 1., post = 1.;
#pragma unroll
      for (int j = 0; j < 4; ++j) t[j] = __shfl(up, 16 * j + 15, 64);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        pre *= j < g4 ? t[j] : 1.;
        post *= 3 - j > g4 ? t[3 - j] : 1.;
      }
      g_s[tid] = g;
      f_s[tid] = up;
      r_s[tid] = ex;
      pc_s[tid] = pre * up;
      sc_s[tid] = ex * post;
    }
  }
  const int t = 16 * wave + l16;
  v4d ao[4], co[4];                                          // A and C against block j <= this wave's
#pragma unroll
  for (int j = 0; j < 4; ++j) ao[j] = co[j] = v4d{0., 0., 0., 0.};
  double da[ONE ? 1 : 16], dc[ONE ? 1 : 16];                 // the block against itself: column l16, channels of this lane group
#pragma unroll
  for (int u = 0; u < (ONE ? 1 : 16); ++u) da[u] = dc[u] = 0.;
  for (int n0 = 0; n0 < NP; n0 += NK) {
    __syncthreads();                                         // the last channels' tiles are done with
    if constexpr (VEC) {
      auto pick = [](bool in, const float4& a, float o) {
        return make_float4(in ? a.x : o, in ? a.y : o, in ? a.z : o, in ? a.w : o);
      };
#pragma unroll
      for (int i = 0; i < CL * NK / 4 / NT; ++i) {
        const int e = tid + i * NT, tt = e / (NK / 4), n = (e % (NK / 4)) * 4;
        const bool in = tt < tc && n0 + n < N;
        const size_t at = (size_t)min(tt, tc - 1) * prep_ld + min(n0 + n, N - 4);
        const float4 q = *reinterpret_cast<const float4*>(qb + at), k = *reinterpret_cast<const float4*>(kb + at);
        *reinterpret_cast<float4*>(&Q_s[tt][n]) = pick(in, q, 0.f);
        *reinterpret_cast<float4*>(&K_s[tt][n]) = pick(in, k, 0.f);
        if constexpr (!ONE) {
          const float4 g = *reinterpret_cast<const float4*>(gb + at);
          *reinterpret_cast<float4*>(&G_s[tt][n]) = pick(in, g, 1.f);
        }
      }
    } else {
      for (int e = tid; e < CL * NK; e += NT) {
        const int tt = e / NK, n = e % NK;
        const bool in = tt < tc && n0 + n < N;
        const size_t at = (size_t)tt * prep_ld + n0 + n;
        Q_s[tt][n] = in ? qb[at] : 0.f;
        K_s[tt][n] = in ? kb[at] : 0.f;
        if constexpr (!ONE) G_s[tt][n] = in ? gb[at] : 1.f;
      }
    }
    __syncthreads();
    // thread: a channel and eight tokens; half a wave holds a block's first eight, the other half its last eight
    const int nn = tid % NK, seg = tid / NK, blk = seg >> 1, n = n0 + nn;
    double up[8], dn[8];                                     // decays up to and with / after each token, in the chunk at last
    if constexpr (ONE) {
#pragma unroll
      for (int i = 0; i < 8; ++i) { up[i] = pc_s[seg * 8 + i]; dn[i] = sc_s[seg * 8 + i]; }
    } else {
      double tot = 1.;
#pragma unroll
      for (int i = 0; i < 8; ++i) { up[i] = tot *= (double)G_s[seg * 8 + i][nn]; }
      const double other = __shfl_xor(tot, 32, 64), first = seg & 1 ? other : 1.;
      double after = seg & 1 ? 1. : other;
#pragma unroll
      for (int i = 7; i >= 0; --i) { dn[i] = after; after *= (double)G_s[seg * 8 + i][nn]; }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        up[i] *= first;
        B_s[seg * 8 + i][nn] = up[i];
        E_s[seg * 8 + i][nn] = dn[i];
      }
      __syncthreads();
      double pre = 1., post = 1.;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const double tj = B_s[16 * j + 15][nn];
        pre *= j < blk ? tj : 1.;
        post *= j > blk ? tj : 1.;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) { up[i] *= pre; dn[i] *= post; }
    }
    {
      const size_t tile = (size_t)(n >> 4) * 256;
      const int o0 = (seg & 1) * 8;                          // the first token's place in its block
      float* kd = Kd + ((size_t)(n >> 4) * 4 + blk) * 256 + (n & 15) * 16 + (o0 >> 2);
#pragma unroll
      for (int i = 0; i < 4; ++i)                            // tokens o0 + i and o0 + 4 + i are neighbours
        *reinterpret_cast<float2*>(kd + i * 4) = make_float2((float)((double)K_s[seg * 8 + i][nn] * dn[i]),
                                                             (float)((double)K_s[seg * 8 + 4 + i][nn] * dn[4 + i]));
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const size_t at = (size_t)blk * NP * 16 + tile + (o0 + i) * 16 + PERM(n & 15);
        Qe[at] = (float)((double)Q_s[seg * 8 + i][nn] * up[i]);
        M[at] = b_s[seg * 8 + i] * ((double)K_s[seg * 8 + i][nn] * up[i]);
      }
      if (seg == 7) cdec[(n & ~15) + PERM(n & 15)] = up[7];
    }
    if (n0 >= N) continue;                                   // (the whole workgroup)
#pragma unroll
    for (int kk = 0; kk < NK / 4; ++kk) {
      const int m = 4 * kk + g4;
      double kr = (double)K_s[t][m], qr = (double)Q_s[t][m];
      if constexpr (ONE) {
#pragma unroll
        for (int j = 3; j >= 0; --j)
          if (j <= wave) {
            const double ks = (double)K_s[16 * j + l16][m];
            ao[j] = mfma4d(kr, ks, ao[j]);
            co[j] = mfma4d(qr, ks, co[j]);
          }
      } else {
        const double eb = B_s[t][m];
        kr *= eb;
        qr *= eb;
        double mid = 1.;                                     // the blocks between j and this wave's
#pragma unroll
        for (int j = 2; j >= 0; --j)
          if (j < wave) {
            const double ks = (double)K_s[16 * j + l16][m] * (E_s[16 * j + l16][m] * mid);
            ao[j] = mfma4d(kr, ks, ao[j]);
            co[j] = mfma4d(qr, ks, co[j]);
            mid *= B_s[16 * j + 15][m];
          }
      }
    }
    if constexpr (!ONE) {                                    // the block against itself, row by row: a column's key times
      for (int m = 4 * g4; m < NK; m += 16) {                // the decays since
        const v4d ks = widen(*reinterpret_cast<const float4*>(&K_s[t][m]));
        v4d x = v4d{0., 0., 0., 0.};
        float4 g[2], k[2], q[2];
        auto rows = [&](int u) {
          g[u & 1] = *reinterpret_cast<const float4*>(&G_s[16 * wave + u][m]);
          k[u & 1] = *reinterpret_cast<const float4*>(&K_s[16 * wave + u][m]);
          q[u & 1] = *reinterpret_cast<const float4*>(&Q_s[16 * wave + u][m]);
        };
        rows(0);
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          if (u < 15) rows(u + 1);
          __builtin_amdgcn_sched_barrier(0);                 // (left alone, all rows are read at once and spill)
          const v4d gd = widen(g[u & 1]), kd = widen(k[u & 1]), qd = widen(q[u & 1]);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            x[i] = u == l16 ? ks[i] : u > l16 ? x[i] * gd[i] : 0.;
            da[u] = __builtin_fma(kd[i], x[i], da[u]);
            dc[u] = __builtin_fma(qd[i], x[i], dc[u]);
          }
        }
      }
    }
  }
  if constexpr (!ONE) {                                      // sums over the lane groups; group g4 keeps rows 4 r + g4
    const bool b1 = g4 & 2, b0 = g4 & 1;
    double a2[8], c2[8];                                     // rows 4 r + 2 b1 + e, e = 0, 1
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const double ga = b1 ? da[4 * r + e] : da[4 * r + 2 + e], gc = b1 ? dc[4 * r + e] : dc[4 * r + 2 + e];
        a2[2 * r + e] = (b1 ? da[4 * r + 2 + e] : da[4 * r + e]) + __shfl_xor(ga, 32, 64);
        c2[2 * r + e] = (b1 ? dc[4 * r + 2 + e] : dc[4 * r + e]) + __shfl_xor(gc, 32, 64);
      }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      ao[3][r] = (b0 ? a2[2 * r + 1] : a2[2 * r]) + __shfl_xor(b0 ? a2[2 * r] : a2[2 * r + 1], 16, 64);
      co[3][r] = (b0 ? c2[2 * r + 1] : c2[2 * r]) + __shfl_xor(b0 ? c2[2 * r] : c2[2 * r + 1], 16, 64);
    }
  }
  __syncthreads();                                           // B_s and E_s are done with; M's right-hand sides are written
  double mid = 1.;
#pragma unroll
  for (int j = 3; j >= 0; --j) {
    if (j > wave) continue;
    const v4d a = ONE || j < wave ? ao[j] : ao[3], cc = ONE || j < wave ? co[j] : co[3];   // where the block's own are
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * wave + 4 * i + g4, sc_ = 16 * j + l16;
      double e = 1.;
      if constexpr (ONE) {
        if (j == wave) {
#pragma unroll
          for (int u = 1; u < 16; ++u) e *= u > l16 && u <= 4 * i + g4 ? g_s[16 * wave + u] : 1.;
        } else e = f_s[r] * (mid * r_s[sc_]);
      }
      A_s[r][sc_] = sc_ < r ? b_s[r] * (e * a[i]) : 0.;
      Cs[(wave * 4 + j) * 256 + (4 * i + g4) * 16 + PERM(l16)] = sc_ <= r ? e * cc[i] : 0.;
    }
    if constexpr (ONE) mid *= j < wave ? f_s[16 * j + 15] : 1.;
  }
  __syncthreads();
  // the blocks' own systems: lane (block g4, column l16) of every wave solves (I + A_bb) x = e_l16
  {
    double x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      double v = i == l16 ? 1. : 0.;
#pragma unroll
      for (int j = 0; j < i; ++j) v -= A_s[16 * g4 + i][16 * g4 + j] * x[j];
      x[i] = v;
    }
    __syncthreads();
    if (wave == 0)
#pragma unroll
      for (int i = 0; i < 16; ++i) A_s[16 * g4 + i][16 * g4 + l16] = x[i];
  }
  __syncthreads();
  v4d ab[4][4];                                              // A_bj (j < b) and the inverses (j == b) as first operands
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int j = 0; j <= b; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) ab[b][j][r] = A_s[16 * b + l16][16 * j + 4 * r + g4];
  // 16 columns at a time (values, then key channels): X_b = T_b (R_b - sum_{j<b} A_bj X_j)
  const int vt = PP / 16;
  for (int ct = wave; ct < vt + NP / 16; ct += NT / 64) {
    const bool val = ct < vt;
    const int n = ct * 16 + l16;                             // this lane's value column
    double* m = M + (size_t)(ct - vt) * 256 + PERM(l16);     // or key channel
    v4d X[4];
    if (val) {
      const T* vb = qkv + row0 * Cq + 2 * GN + h * P + min(n, P - 1);
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) X[b][r] = (double)ldf<T>(vb + (size_t)min(16 * b + 4 * r + g4, tc - 1) * Cq);
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int tk = 16 * b + 4 * r + g4;
          X[b][r] = tk < tc ? b_s[tk] * X[b][r] : 0.;
        }
    } else {
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) X[b][r] = m[(size_t)b * NP * 16 + (4 * r + g4) * 16];
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      v4d z = v4d{0., 0., 0., 0.};
#pragma unroll
      for (int j = 0; j < b; ++j) z = mma16(ab[b][j], X[j], z);
      const v4d r = X[b] - z;
      if (__all(finite4(r))) {
        X[b] = mma16(ab[b][b], r, v4d{0., 0., 0., 0.});
      } else {                                               // 0 times an infinity or NaN would reach earlier tokens
        X[b] = v4d{0., 0., 0., 0.};
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const double v = __shfl(r[u >> 2], (u & 3) * 16 + l16, 64);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (u <= 4 * i + g4) X[b][i] += A_s[16 * b + 4 * i + g4][16 * b + u] * v;
        }
      }
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (val) U[(size_t)(16 * b + 4 * r + g4) * PP + n] = X[b][r];
        else m[(size_t)b * NP * 16 + (4 * r + g4) * 16] = X[b][r];
      }
  }
}

// 4 KS waves, NP = 64 KS, 4 CS value columns a workgroup: wave w keeps the state rows 16 w .., and computes the 16 tokens of block
// w % 4 of M S_in over the 64 channels of quarter w / 4 (the quarters' shares meet in LDS).  The next chunk's operands are requested in
// four parts between the steps of this one (48 KiB a workgroup: asked for at once they hold up the wave that asks, 233 -> 211 us with 8
// columns); nothing in the loop is conditional, so the waits for them are counted ones.
// v_mfma_f64_4x4x4 does 64 operations a clock and SIMD where 16x16x4 does 32, and takes four columns, so that more CUs share a
// head's columns.  Its four blocks take four fours of k of the same four rows: lane l, x = l >> 2, holds of row 4 g + (l & 3) the
// numbers 4 (x & 3) + s of tile x / 4 in steps s = 0..3 (neighbours: one 32-byte load), and of the other operand that k's number in
// column l & 3, read once for all four g.  four_sums adds up the blocks and leaves row 4 ((l >> 2) & 3) + l / 16, column l & 3.
// 16 heads, 4096 tokens of 64 x 64 states: 140 us on 64 workgroups with 16x16x4, now 74; of 128 x 128 158 -> 64.
__device__ __forceinline__ double mfma1d(double a, double b, double c) { return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0); }
__device__ __forceinline__ double lane_xor_d(double v, int o) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  return __builtin_bit_cast(double, (uint64_t)lane_xor((uint32_t)(u >> 32), o) << 32 | lane_xor((uint32_t)u, o));
}
__device__ __forceinline__ double four_sums(const double (&d)[4], int lane) {
  const bool b1 = lane & 8, b0 = lane & 4;
  const double e0 = (b1 ? d[2] : d[0]) + lane_xor_d(b1 ? d[0] : d[2], 8);
  const double e1 = (b1 ? d[3] : d[1]) + lane_xor_d(b1 ? d[1] : d[3], 8);
  return (b0 ? e1 : e0) + lane_xor_d(b0 ? e0 : e1, 4);
}
template <int KS, int CS>
__global__ void __launch_bounds__(256 * KS) delta_chunk_scan_kernel(DeltaScratch sc, float* __restrict__ state,
                                                                   const int* __restrict__ seq_slot,
                                                                   const int* __restrict__ seq_start,
                                                                   const int* __restrict__ seq_len, DeltaPart dp, int n, int H, int N, int P,
                                                                   int PP) {
  constexpr int NP = 64 * KS, PC = 4 * CS;
  __shared__ double S_s[NP][PC], W_s[CL][PC], P_s[KS > 1 ? KS : 1][KS > 1 ? CL : 1][PC];
  // the workgroups of a head share an L2: blocks are dealt to the eight dies in turn, every other eight heads half a round further (of four
  // heads, long and short sequences in turn fell on four dies each: 16 sequences of 35 to 863, 64 x 128 states, 140 / 125 us)
  const int nct = PP / PC, oct = ((int)blockIdx.x >> 3) / nct, ct = ((int)blockIdx.x >> 3) % nct;
  const int unit = (((int)blockIdx.x + 4 * oct) & 7) + 8 * oct;
  if (unit >= n * H) return;
  const int p0 = ct * PC, h = unit % H, s = unit / H, tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane & 3, x = lane >> 2;
  const int own = 4 * (x & 3) + (lane >> 4);                 // this lane's row of a wave's 16 (four_sums)
  const int tb = wave & 3, kq = wave >> 2, n0 = 16 * wave, nc = chunks_of(seq_len[s], dp);
  size_t cb0;
  if (nc == 0 || !first_chunk(seq_len, s, dp, cb0)) return;
  float* st = state + ((size_t)seq_slot[s] * H + h) * N * P;
  const bool cont = seq_start[s] > 0 || dp.c0 > 0;
  const int nr = n0 + own;
  double S[CS];
#pragma unroll
  for (int c = 0; c < CS; ++c) {
    const int p = p0 + 4 * c + j;
    S[c] = (cont && nr < N && p < P) ? (double)st[(size_t)nr * P + p] : 0.;
  }
  struct Chunk {
    v2d m[4][2];
    float4 kd[4];
    double dec, u[CS];
  };
  // KS > 1: a chunk's 64 x PC numbers of W are dealt to all threads
  static_assert(KS == 1 || KS == 2, "states of up to 128 rows");
  constexpr int UE = KS == 1 ? CS : (CL * PC + 256 * KS - 1) / (256 * KS);
  auto wrow = [&](int i) { return KS == 1 ? 16 * tb + own : (tid + 256 * KS * i) / PC; };
  auto wcol = [&](int i) { return KS == 1 ? 4 * i + j : (tid + 256 * KS * i) % PC; };
  static_assert(UE <= CS, "numbers of W a thread");
  auto load = [&](int c, Chunk& q, int part) {
    const size_t cb = (cb0 + c) * H + h;
    const double* mp = sc.M + cb * CL * NP + ((size_t)(tb * (NP / 16) + kq * 4 + (x >> 2)) * 16 + j) * 16 + 4 * (x & 3);
    const float* kp = sc.Kd + cb * CL * NP + ((size_t)(wave * 4 + (x >> 2)) * 16 + j) * 16 + 4 * (x & 3);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (part >= 0 && g != part) continue;
      q.m[g][0] = *reinterpret_cast<const v2d*>(mp + g * 64);
      q.m[g][1] = *reinterpret_cast<const v2d*>(mp + g * 64 + 2);
      q.kd[g] = *reinterpret_cast<const float4*>(kp + g * 64);
    }
    if (part > 0) return;
    q.dec = sc.cdec[cb * NP + n0 + PERM(own)];
#pragma unroll
    for (int i = 0; i < UE; ++i) {
      const int r = KS == 1 ? wrow(i) : min(wrow(i), CL - 1);
      q.u[i] = sc.U[(cb * CL + r) * PP + p0 + wcol(i)];
    }
  };
  auto step = [&](int c, const Chunk& q, int cn, Chunk& qn) {
    const size_t cb = (cb0 + c) * H + h;
    load(cn, qn, 0);
#pragma unroll
    for (int i = 0; i < CS; ++i) {
      sc.sin[cb * NP * PP + ((size_t)wave * PP + p0 + 4 * i + j) * 16 + PERM(own)] = (float)S[i];
      S_s[nr][4 * i + j] = S[i];
    }
    __syncthreads();
    double b[CS][4];
#pragma unroll
    for (int i = 0; i < CS; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) b[i][k] = S_s[64 * kq + 16 * (x >> 2) + 4 * k + (x & 3)][4 * i + j];
    __builtin_amdgcn_sched_barrier(0);                       // every read on its way before the first product waits
    load(cn, qn, 1);
    __builtin_amdgcn_sched_barrier(0);
    double v[CS];
#pragma unroll
    for (int i = 0; i < CS; ++i) {
      double d[4] = {0., 0., 0., 0.};
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int g = 0; g < 4; ++g) d[g] = mfma1d(q.m[g][k >> 1][k & 1], b[i][k], d[g]);
      v[i] = four_sums(d, lane);
    }
    __builtin_amdgcn_sched_barrier(0);
    load(cn, qn, 2);
    __builtin_amdgcn_sched_barrier(0);
    double z[UE];
    if constexpr (KS == 1) {
#pragma unroll
      for (int i = 0; i < UE; ++i) z[i] = q.u[i] - v[i];
    } else {
#pragma unroll
      for (int i = 0; i < CS; ++i) P_s[kq][16 * tb + own][4 * i + j] = v[i];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < UE; ++i) {
        double sum = 0.;
        const int r = min(wrow(i), CL - 1), cc = wcol(i);
#pragma unroll
        for (int k = 0; k < KS; ++k) sum += P_s[k][r][cc];
        z[i] = q.u[i] - sum;
      }
    }
#pragma unroll
    for (int i = 0; i < UE; ++i) {
      const int r = wrow(i), cc = wcol(i);
      if (KS == 1 || r < CL) {
        W_s[r][cc] = z[i];
        sc.U[(cb * CL + r) * PP + p0 + cc] = z[i];
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < CS; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) b[i][k] = W_s[16 * (x >> 2) + 4 * k + (x & 3)][4 * i + j];
    __builtin_amdgcn_sched_barrier(0);
    load(cn, qn, 3);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < CS; ++i) {
      double d[4] = {0., 0., 0., 0.};
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float4& f = q.kd[g];
          d[g] = mfma1d((double)(k == 0 ? f.x : k == 1 ? f.y : k == 2 ? f.z : f.w), b[i][k], d[g]);
        }
      S[i] = __builtin_fma(q.dec, S[i], four_sums(d, lane));
    }
  };
  Chunk even, odd;
  load(0, even, -1);
  int c = 0;
  for (; c + 1 < nc; c += 2) {
    step(c, even, c + 1, odd);
    step(c + 1, odd, min(c + 2, nc - 1), even);              // (past the end: the last chunk again, not used)
  }
  if (c < nc) step(c, even, c, odd);
#pragma unroll
  for (int i = 0; i < CS; ++i) {
    const int p = p0 + 4 * i + j;
    if (nr < N && p < P) st[(size_t)nr * P + p] = (float)S[i];
  }
}

// The same for states of 129 to 256 rows: 16 waves leave 128 registers a lane, too few for a chunk's operands on their way beside
// another's (8 heads of 256 x 256, us for all three kernels, this form / the one above: 4096 tokens 700 / 714, six sequences of 512 419 / 689).
// Wave w keeps the state rows 16 w .. of the workgroup's 16 value columns as a 16x16x4 accumulator.
__global__ void __launch_bounds__(1024) delta_chunk_scan_wide_kernel(DeltaScratch sc, float* __restrict__ state,
                                                                   const int* __restrict__ seq_slot,
                                                                   const int* __restrict__ seq_start,
                                                                   const int* __restrict__ seq_len, DeltaPart dp, int H, int N, int P,
                                                                   int PP) {
  constexpr int KS = 4, NP = 64 * KS;                        // rows of 16 numbers: four rows take each bank twice, the least
  __shared__ double S_s[NP][16], W_s[CL][16], P_s[KS][CL][16];
  const int p0 = blockIdx.x * 16, h = blockIdx.y, s = blockIdx.z, tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g4 = lane >> 4, p = p0 + l16;
  const int tb = wave & 3, kq = wave >> 2, n0 = 16 * wave, nc = chunks_of(seq_len[s], dp);
  size_t cb0;
  if (nc == 0 || !first_chunk(seq_len, s, dp, cb0)) return;
  float* st = state + ((size_t)seq_slot[s] * H + h) * N * P;
  const bool cont = seq_start[s] > 0 || dp.c0 > 0;
  v4d S;
#pragma unroll
  for (int r = 0; r < 4; ++r) S[r] = (cont && n0 + 4 * r + g4 < N && p < P) ? (double)st[(size_t)(n0 + 4 * r + g4) * P + p] : 0.;
  const int row = tid / 16;                                  // this thread's number of a W tile, column l16
  struct Chunk {
    v4d m[4], dec;
    float4 kd[4];
    double u;
  };
  auto load = [&](int c, Chunk& x) {
    const size_t cb = (cb0 + c) * H + h;
    const double* mp = sc.M + cb * CL * NP + ((size_t)(tb * (NP / 16) + kq * 4) * 16 + l16) * 16 + 4 * g4;
    const float* kp = sc.Kd + cb * CL * NP + ((size_t)wave * 64 + l16) * 16 + 4 * g4;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x.m[k] = *reinterpret_cast<const v4d*>(mp + k * 256);
      x.kd[k] = *reinterpret_cast<const float4*>(kp + k * 256);
    }
    x.dec = *reinterpret_cast<const v4d*>(sc.cdec + cb * NP + n0 + 4 * g4);
    x.u = sc.U[(cb * CL + row) * PP + p];
  };
  auto step = [&](int c, const Chunk& x) {
    const size_t cb = (cb0 + c) * H + h;
    *reinterpret_cast<float4*>(sc.sin + cb * NP * PP + ((size_t)wave * PP + p) * 16 + 4 * g4) =
        make_float4((float)S[0], (float)S[1], (float)S[2], (float)S[3]);
#pragma unroll
    for (int r = 0; r < 4; ++r) S_s[n0 + 4 * r + g4][l16] = S[r];
    __syncthreads();
    v4d b[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) b[k][r] = S_s[64 * kq + 16 * k + 4 * r + g4][l16];
    __builtin_amdgcn_sched_barrier(0);                       // every read on its way before the first product waits
    v4d v = v4d{0., 0., 0., 0.};
#pragma unroll
    for (int k = 0; k < 4; ++k) v = mma16(x.m[k], b[k], v);
#pragma unroll
    for (int r = 0; r < 4; ++r) P_s[kq][16 * tb + 4 * r + g4][l16] = v[r];
    __syncthreads();
    double sum = 0.;
#pragma unroll
    for (int k = 0; k < KS; ++k) sum += P_s[k][row][l16];
    const double z = x.u - sum;
    W_s[row][l16] = z;
    sc.U[(cb * CL + row) * PP + p] = z;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) b[k][r] = W_s[16 * k + 4 * r + g4][l16];
    __builtin_amdgcn_sched_barrier(0);
    v4d a = x.dec * S;
#pragma unroll
    for (int k = 0; k < 4; ++k) a = mma16(widen(x.kd[k]), b[k], a);
    S = a;
  };
  for (int c = 0; c < nc; ++c) {
    Chunk x;
    load(c, x);
    step(c, x);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = n0 + 4 * r + g4;
    if (n < N && p < P) st[(size_t)n * P + p] = (float)S[r];
  }
}

// y rows of one chunk, 16 PT value columns; wave i owns token block i.  Operands straight from L2: the waves of a
// workgroup share the state and W tiles, nothing else is read twice.
template <int PT>
__global__ void __launch_bounds__(NT) delta_chunk_out_kernel(DeltaScratch sc, const int* __restrict__ seq_len,
                                                             const int* __restrict__ seq_off, float* __restrict__ y, DeltaPart dp, int H,
                                                             int NP, int P, int PP, int ntp) {
  const int c = blockIdx.x / ntp, t0 = (blockIdx.x % ntp) * PT, s = blockIdx.y, h = blockIdx.z, len = seq_len[s];
  size_t cb;
  if (c >= chunks_of(len, dp) || !first_chunk(seq_len, s, dp, cb)) return;
  const int first = (dp.c0 + c) * CL, tc = min(CL, len - first), tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g4 = lane >> 4;
  if (16 * wave >= tc) return;
  const size_t row0 = (size_t)seq_off[s] + first;
  cb = (cb + c) * H + h;
  const int at = l16 * 16 + 4 * g4;
  const float *qp = sc.Qe + cb * CL * NP + (size_t)wave * NP * 16 + at, *sp = sc.sin + cb * NP * PP + at;
  const double *cp = sc.Cs + cb * CL * CL + wave * 4 * 256, *wp = sc.U + cb * CL * PP + l16;
  int tile[PT];                                              // column tiles; one past the last repeats it and is not stored
#pragma unroll
  for (int j = 0; j < PT; ++j) tile[j] = min(t0 + j, PP / 16 - 1);
  v4d o[PT];
#pragma unroll
  for (int j = 0; j < PT; ++j) o[j] = v4d{0., 0., 0., 0.};
#pragma unroll 2
  for (int n = 0; n < NP / 16; ++n) {
    const v4d a = widen(*reinterpret_cast<const float4*>(qp + n * 256));
#pragma unroll
    for (int j = 0; j < PT; ++j)
      o[j] = mma16(a, widen(*reinterpret_cast<const float4*>(sp + ((size_t)n * PP + tile[j] * 16) * 16)), o[j]);
  }
  for (int b0 = 0; b0 <= wave; ++b0) {
    const v4d a = *reinterpret_cast<const v4d*>(cp + b0 * 256 + at);
    v4d w[PT];
    bool finite = true;
#pragma unroll
    for (int j = 0; j < PT; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) w[j][r] = wp[(size_t)(16 * b0 + 4 * r + g4) * PP + tile[j] * 16];
      finite = finite && finite4(w[j]);
    }
    if (b0 < wave || __all(finite)) {
#pragma unroll
      for (int j = 0; j < PT; ++j) o[j] = mma16(a, w[j], o[j]);
    } else {                                                 // 0 times an infinity or NaN would reach earlier tokens
#pragma unroll
      for (int i = 0; i < 4; ++i)
        for (int t = 0; t <= 4 * i + g4; ++t) {
          const double x = cp[wave * 256 + (4 * i + g4) * 16 + PERM(t)];
#pragma unroll
          for (int j = 0; j < PT; ++j) o[j][i] += x * wp[(size_t)(16 * wave + t) * PP + tile[j] * 16];
        }
    }
  }
#pragma unroll
  for (int j = 0; j < PT; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * wave + 4 * i + g4, p = (t0 + j) * 16 + l16;
      if (t < tc && p < P) y[(row0 + t) * H * P + h * P + p] = (float)o[j][i];
    }
}

int channels(int N) { return N <= 64 ? 64 : N <= 128 ? 128 : 256; }
}  // namespace

extern "C" {

// fp32 words of scratch, per chunk and head: fp64 M [64 NP], U [64 PP], C [64 64], cdec [NP], fp32 Qe, Kd [64 NP], states [NP PP]
int64_t edge_sm_delta_chunk_floats(int64_t chunks, int64_t H, int64_t N, int64_t P) {
  const int64_t NP = channels((int)N), PP = (P + 15) & ~15LL;
  return chunks * H * (2 * (CL * NP + CL * PP + CL * CL + NP) + 2 * CL * NP + NP * PP);
}

// Portions of `least` tokens or more, `most` of their chunks at a time (what the scratch of `room` chunks holds), the state
// carried from one run of the kernels to the next; max_chunks: the longest portion's.
int edge_sm_delta_chunked(const float* prep, int prep_ld, const void* qkv, int Cq, float* state, const int* seq_slot,
                          const int* seq_start, const int* seq_len, const int* seq_off, float* scratch, float* y, int rows, int n,
                          int room, int most, int max_chunks, int least, int H, int G, int N, int P, int GD, int f32,
                          hipStream_t st) {
  if (n == 0 || rows == 0 || max_chunks <= 0) return 0;
  if (f32 || G <= 0 || H % G || N < 1 || N > 256 || P < 1 || (GD != N && GD != 1) || most < 1 || room < 1) return -2;
  const int NP = channels(N), PP = (P + 15) & ~15;
  const int64_t CH = (int64_t)room * H;
  if (((uintptr_t)scratch & 31) != 0) return -3;
  DeltaScratch sc;
  sc.M = reinterpret_cast<double*>(scratch);
  sc.U = sc.M + CH * CL * NP;
  sc.Cs = sc.U + CH * CL * PP;
  sc.cdec = sc.Cs + CH * CL * CL;
  sc.Qe = reinterpret_cast<float*>(sc.cdec + CH * NP);
  sc.Kd = sc.Qe + CH * CL * NP;
  sc.sin = sc.Kd + CH * CL * NP;
  const bool vec = N % 4 == 0 && prep_ld % 4 == 0 && ((uintptr_t)prep & 15) == 0;
  const int ntp = (PP + 63) / 64;
  for (int c0 = 0; c0 < max_chunks; c0 += most) {
    const DeltaPart dp{least, c0, most, room};
    const int mc = max_chunks - c0 < most ? max_chunks - c0 : most;
#define SM_DSOLVE(V, ONE)                                                                                           \
  hipLaunchKernelGGL((delta_chunk_solve_kernel<bf16_t, V, ONE>), dim3(mc, n, H), dim3(NT), 0, st, prep, prep_ld,    \
                     (const bf16_t*)qkv, Cq, seq_len, seq_off, sc, dp, H, G, N, NP, P, PP)
    if (GD == 1) {
      if (vec) SM_DSOLVE(true, true);
      else SM_DSOLVE(false, true);
    } else if (vec) SM_DSOLVE(true, false);
    else SM_DSOLVE(false, false);
#undef SM_DSOLVE
    // columns a workgroup: as few fours as 256 workgroups, one a CU, leave; more share the operands' reads.  States of up to 64 rows stop at
    // 8: their 16 columns (four waves) step no quicker than the 16x16x4 form did, and behind uneven portions, whose longest is the launch,
    // cost up to 12 % more than 8.  us for all three kernels, 4 / 8 / 16 columns: 16 heads of 64 x 64, 4096 tokens 198 / 211 / 283, 12 heads, eight
    // sequences of 24 to 1344 189 / 174 / 194, 32 heads, four of 2048 502 / 502 / 507; 16 of 128 x 128, 512 tokens 105 / 86 / 97, two sequences of 1386
    // 401 / 296 / 277, six of 512 230 / 231 / 231.  101 steps of up to 40 sequences: 0.953 of that form's time, at the worst 1.05
    // (eight sequences of 83 to 1325, 4 heads of 64 x 128, 151 / 159).
#define SM_DSCAN(KS, CS)                                                                                                        \
  hipLaunchKernelGGL((delta_chunk_scan_kernel<KS, CS>), dim3((H * n + 7) / 8 * 8 * (PP / (4 * CS))), dim3(256 * KS), 0, st, sc, \
                     state, seq_slot, seq_start, seq_len, dp, n, H, N, P, PP)
    const int fours = H * n * (PP / 4) <= 256 ? 1 : H * n * (PP / 8) <= 256 ? 2 : 4;
    if (NP == 64 && fours == 1) SM_DSCAN(1, 1);
    else if (NP == 64) SM_DSCAN(1, 2);
    else if (NP == 128 && fours == 1) SM_DSCAN(2, 1);
    else if (NP == 128 && fours == 2) SM_DSCAN(2, 2);
    else if (NP == 128) SM_DSCAN(2, 4);
    else
      hipLaunchKernelGGL(delta_chunk_scan_wide_kernel, dim3(PP / 16, H, n), dim3(1024), 0, st, sc, state, seq_slot, seq_start, seq_len, dp, H, N,
                         P, PP);
#undef SM_DSCAN
    hipLaunchKernelGGL((delta_chunk_out_kernel<4>), dim3(mc * ntp, n, H), dim3(NT), 0, st, sc, seq_len, seq_off, y, dp, H, NP, P,
                       PP, ntp);
  }
  return (int)hipGetLastError();
}

}  // extern "C"
