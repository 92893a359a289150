// The gated delta rule over 64-token chunks (ops/seqmix.py::delta_rule_scan, portions of many tokens): per head, with
// decays g_t per key channel (or one for all of them),
//   S_t = g_t S_{t-1} + k_t w_t^T,  w_t = beta_t (v_t - (g_t S_{t-1})^T k_t),  o_t = S_t^T q_t.
// With B_t the sum of log2 g inside the chunk and S_in the state that enters it,
//   (I + A) W = beta V - (beta k e^B) S_in,   A[t, s] = beta_t sum_n k_t k_s e^{B_t - B_s}  (s < t)
//   S_out = e^{B_end} S_in + sum_s (k_s e^{B_end - B_s}) w_s^T
//   o_t = (q_t e^{B_t})^T S_in + sum_{s<=t} C[t, s] w_s,   C[t, s] = sum_n q_t k_s e^{B_t - B_s}
// (1) delta_chunk_solve_kernel, parallel over chunks: A and C, then U and M with (I + A) [U | M] = [beta V | beta k e^B]
//     by forward substitution over 16-token blocks (the blocks' own 16 x 16 systems inverted); also q e^B,
//     k e^{B_end - B} and e^{B_end}.
// (2) delta_chunk_scan_kernel, chunk by chunk: W = U - M S_in and the next state, 16 value columns per workgroup.
// (3) delta_chunk_out_kernel, parallel over chunks: the outputs.
// No decay ratio is formed as a quotient and no exponent is positive: from a token s to a later 16-token block the
// ratio is e^{what s's block decays after s + the blocks between} e^{t's block up to t}, inside a block likewise over
// 4-token groups, inside a group the sum of the logs between: sums of terms of one sign, so that a weak decay behind a
// strong one loses nothing to cancellation.  Everything is fp32 (v_mfma_f32_16x16x4_f32 and plain FMAs).  A product's
// result holds rows 4 g .. 4 g + 3 in lane group g, so its four registers are the second operand of four steps whose
// k runs over rows 4 g + j: results feed products without a shuffle, and the first operands are 16-byte loads of rows.
//
// Bound: token by token, every token costs a chain of two row sums (about 530 clocks); here the chain is two products
// and two barriers per 64 tokens.  16 heads, 4096 tokens: 64 x 64 states 916 -> 172 us ((1) about 100, (2) 55, (3) 18),
// 128 x 128 states 1521 -> 378 us ((2) 154: 2.4 us a chunk).  (1) waits on memory and LDS latency at two workgroups per
// CU; (2) is the serial part.
#include "seqmix_common.h"

namespace {

// the first operand of one 16-wide block of k: row's elements 4 g4 .. 4 g4 + 3; the second: b[j] = element 4 g4 + j
__device__ __forceinline__ v4f mma16(const float4& a, float b0, float b1, float b2, float b3, v4f c) {
  c = mfma4(a.x, b0, c);
  c = mfma4(a.y, b1, c);
  c = mfma4(a.z, b2, c);
  return mfma4(a.w, b3, c);
}

// Scratch per (chunk, head), NP = 64, 128 or 256 channels (zero past N) and PP = P rounded up to 16, in 16 x 16 tiles whose
// rows are what a 16-byte operand load takes (every load and store of a wave is one contiguous KiB):
//   M, Qe [4 token blocks][NP / 16][token][channel]   Kd [NP / 16][4][channel][token]   Cs [4][4][token][earlier token]
//   U (later W) [4][PP][token]   states [NP / 16][PP][channel]
// VEC: 16-byte loads of the prepared rows.  ONE: one decay for
// all key channels of a head (the ratios are then taken out of the products).
template <typename T, bool VEC, bool ONE>
__global__ void __launch_bounds__(NT) delta_chunk_solve_kernel(const float* __restrict__ prep, int prep_ld,
                                                               const T* __restrict__ qkv, int Cq,
                                                               const int* __restrict__ seq_len, const int* __restrict__ seq_off,
                                                               float* la, float* __restrict__ U, float* __restrict__ M,
                                                               float* __restrict__ Qe, float* __restrict__ Kd,
                                                               float* __restrict__ Cs, float* __restrict__ cdec, int H, int G,
                                                               int N, int NP, int P, int PP) {
  constexpr int NK = 32, LQ = NK + 4, LA = CL + 4, LB = ONE ? 1 : CL;
  __shared__ __attribute__((aligned(16))) float Q_s[CL][LQ], K_s[CL][LQ], A_s[CL][LA];
  // logs; sums up to and with / after a token in its 16-token block; after it in its group of four; whole groups
  __shared__ __attribute__((aligned(16))) float L_s[LB][LQ], B_s[LB][LQ], E_s[LB][LQ], G_s[LB][LQ], T_s[ONE ? 1 : CL / 4][LQ];
  __shared__ float b_s[CL], l_s[CL], f_s[CL], r_s[CL];       // beta; ONE: logs, sums up to / after a token in its block
  const int c = blockIdx.x, s = blockIdx.y, h = blockIdx.z, len = seq_len[s];
  if (c * CL >= len) return;
  const int tc = min(CL, len - c * CL), GN = G * N, GD = ONE ? 1 : N;
  const size_t row0 = (size_t)seq_off[s] + (size_t)c * CL, cb = ((size_t)chunk_base(seq_len, s) + c) * H + h;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g4 = lane >> 4;
  const float* pr = prep + row0 * prep_ld;
  const float *qb = pr + (h / (H / G)) * N, *kb = qb + GN, *gb = pr + 2 * GN + h * GD, *bb = pr + 2 * GN + H * GD + h;
  auto lg = [](float g) { return g == 0.f ? -1e4f : log2f(g); };   // 0: a decay that has underflowed to nothing
  la += cb * CL * NP;                                        // the chunk's log2 decays [64, NP] (!ONE)
  if (tid < CL) {                                            // (one wave: it is in step with itself)
    const size_t at = (size_t)min(tid, tc - 1) * prep_ld;
    b_s[tid] = tid < tc ? bb[at] : 0.f;
    if constexpr (ONE) {
      const float l = tid < tc ? lg(gb[at]) : 0.f;
      float up = l, dn = l;
#pragma unroll
      for (int d = 1; d < 16; d <<= 1) {                     // inclusive sums inside the 16-token block, both ways
        const float a = __shfl_up(up, d, 64), b = __shfl_down(dn, d, 64);
        if (l16 >= d) up += a;
        if (l16 + d < 16) dn += b;
      }
      const float after = __shfl_down(dn, 1, 64);
      l_s[tid] = l;
      f_s[tid] = up;
      r_s[tid] = l16 < 15 ? after : 0.f;
    }
  }
  const int t = 16 * wave + l16;
  v4f ao[4], co[4];                                          // A and C against block j <= this wave's
#pragma unroll
  for (int j = 0; j < 4; ++j) ao[j] = co[j] = v4f{0.f, 0.f, 0.f, 0.f};
  for (int n0 = 0; n0 < N; n0 += NK) {
    __syncthreads();                                         // the last channels' tiles are done with
    if constexpr (VEC) {
#pragma unroll
      for (int i = 0; i < CL * NK / 4 / NT; ++i) {
        const int e = tid + i * NT, tt = e / (NK / 4), n = (e % (NK / 4)) * 4;
        const bool in = tt < tc && n0 + n < N;
        const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
        const size_t at = (size_t)min(tt, tc - 1) * prep_ld + min(n0 + n, N - 4);
        const float4 q = *reinterpret_cast<const float4*>(qb + at), k = *reinterpret_cast<const float4*>(kb + at);
        *reinterpret_cast<float4*>(&Q_s[tt][n]) = in ? q : z;
        *reinterpret_cast<float4*>(&K_s[tt][n]) = in ? k : z;
      }
    } else {
      for (int e = tid; e < CL * NK; e += NT) {
        const int tt = e / NK, n = e % NK;
        const bool in = tt < tc && n0 + n < N;
        Q_s[tt][n] = in ? qb[(size_t)tt * prep_ld + n0 + n] : 0.f;
        K_s[tt][n] = in ? kb[(size_t)tt * prep_ld + n0 + n] : 0.f;
      }
    }
    if constexpr (!ONE) {
      float g[CL * NK / NT];
#pragma unroll
      for (int i = 0; i < CL * NK / NT; ++i) {
        const int e = tid + i * NT;
        g[i] = gb[(size_t)min(e / NK, tc - 1) * prep_ld + min(n0 + e % NK, N - 1)];
      }
#pragma unroll
      for (int i = 0; i < CL * NK / NT; ++i) {
        const int e = tid + i * NT, tt = e / NK, n = e % NK;
        const float v = tt < tc && n0 + n < N ? lg(g[i]) : 0.f;
        L_s[tt][n] = v;
        if (n0 + n < NP) la[tt * NP + n0 + n] = v;
      }
      __syncthreads();
      // half a wave holds a block's first eight tokens, the other half its last eight
      const int nn = tid % NK, seg = tid / NK;
      float a[8], sum = 0.f, back = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) { a[i] = L_s[seg * 8 + i][nn]; sum += a[i]; }
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        float after = 0.f;
#pragma unroll
        for (int i = 3; i >= 0; --i) { G_s[seg * 8 + 4 * g + i][nn] = after; after += a[4 * g + i]; }
        T_s[seg * 2 + g][nn] = after;
      }
      const float other = __shfl_xor(sum, 32, 64);
      float fwd = seg & 1 ? other : 0.f;
      back = seg & 1 ? 0.f : other;
#pragma unroll
      for (int i = 0; i < 8; ++i) { fwd += a[i]; B_s[seg * 8 + i][nn] = fwd; }
#pragma unroll
      for (int i = 7; i >= 0; --i) { E_s[seg * 8 + i][nn] = back; back += a[i]; }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < NK / 4; ++kk) {
      const int n = 4 * kk + g4;
      float kr = K_s[t][n], qr = Q_s[t][n];
      if constexpr (ONE) {
#pragma unroll
        for (int j = 3; j >= 0; --j)
          if (j <= wave) {
            const float ks = K_s[16 * j + l16][n];
            ao[j] = mfma4(kr, ks, ao[j]);
            co[j] = mfma4(qr, ks, co[j]);
          }
      } else {
        float tot[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) tot[j] = j < wave ? B_s[16 * j + 15][n] : 0.f;
        const float eb = ex2(B_s[t][n]);
        kr *= eb;
        qr *= eb;
        float mid = 0.f;                                     // the blocks between j and this wave's
#pragma unroll
        for (int j = 2; j >= 0; --j)
          if (j < wave) {
            const float ks = K_s[16 * j + l16][n] * ex2(E_s[16 * j + l16][n] + mid);
            ao[j] = mfma4(kr, ks, ao[j]);
            co[j] = mfma4(qr, ks, co[j]);
            mid += tot[j];
          }
      }
    }
    if constexpr (!ONE) {                                    // the block against itself, results as the products' lie
      const int g0 = 4 * wave, gs = l16 >> 2;                // the lane's rows are group g4, its column is in group gs
      const int m1 = g0 + min(gs + 1, 3), m2 = g0 + min(gs + 2, 3);
      const float w0 = g4 > gs ? 1.f : 0.f, w1 = g4 > gs + 1 ? 1.f : 0.f, w2 = g4 > gs + 2 ? 1.f : 0.f;
#pragma unroll 2
      for (int n = 0; n < NK; n += 4) {
        const float4 ks = *reinterpret_cast<const float4*>(&K_s[t][n]), ga = *reinterpret_cast<const float4*>(&G_s[t][n]);
        const float4 t1 = *reinterpret_cast<const float4*>(&T_s[m1][n]), t2 = *reinterpret_cast<const float4*>(&T_s[m2][n]);
        // the decay from the column's token to the rows' group, then row by row
        float4 x = make_float4(w0 * ga.x + w1 * t1.x + w2 * t2.x, w0 * ga.y + w1 * t1.y + w2 * t2.y,
                               w0 * ga.z + w1 * t1.z + w2 * t2.z, w0 * ga.w + w1 * t1.w + w2 * t2.w);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * wave + 4 * g4 + i;
          const float4 kr = *reinterpret_cast<const float4*>(&K_s[r][n]), qr = *reinterpret_cast<const float4*>(&Q_s[r][n]);
          const float4 l = *reinterpret_cast<const float4*>(&L_s[r][n]);
          const float on = 4 * g4 + i > l16 ? 1.f : 0.f;
          x.x += on * l.x;
          x.y += on * l.y;
          x.z += on * l.z;
          x.w += on * l.w;
          const float e0 = ks.x * ex2(x.x), e1 = ks.y * ex2(x.y), e2 = ks.z * ex2(x.z), e3 = ks.w * ex2(x.w);
          ao[3][i] += kr.x * e0 + kr.y * e1 + kr.z * e2 + kr.w * e3;
          co[3][i] += qr.x * e0 + qr.y * e1 + qr.z * e2 + qr.w * e3;
        }
      }
    }
  }
  float* cr = Cs + cb * CL * CL + wave * 4 * 256 + l16;
  float mid = 0.f;
#pragma unroll
  for (int j = 3; j >= 0; --j) {
    if (j > wave) continue;
    const int a = ONE || j < wave ? j : 3;                   // where the block's own products are
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * wave + 4 * g4 + i, sc = 16 * j + l16;
      float e = 1.f;
      if constexpr (ONE) {
        float x = f_s[r] + (mid + r_s[sc]);
        if (j == wave) {
          x = 0.f;
#pragma unroll
          for (int u = 1; u < 16; ++u) x += u > l16 && u <= 4 * g4 + i ? l_s[16 * wave + u] : 0.f;
        }
        e = ex2(x);
      }
      A_s[r][sc] = sc < r ? b_s[r] * e * ao[a][i] : 0.f;
      cr[j * 256 + (4 * g4 + i) * 16] = sc <= r ? e * co[a][i] : 0.f;
    }
    if constexpr (ONE) mid += j < wave ? f_s[16 * j + 15] : 0.f;
  }
  __syncthreads();
  // the blocks' own systems: lane (block g4, column l16) of every wave solves (I + A_bb) x = e_l16
  float x[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    float v = i == l16 ? 1.f : 0.f;
#pragma unroll
    for (int j = 0; j < i; ++j) v -= A_s[16 * g4 + i][16 * g4 + j] * x[j];
    x[i] = v;
  }
  __syncthreads();
  if (wave == 0)
#pragma unroll
    for (int i = 0; i < 16; ++i) A_s[16 * g4 + i][16 * g4 + l16] = x[i];
  __syncthreads();
  float4 ab[4][4];                                           // A_bj (j < b) and the inverses (j == b) as first operands
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int j = 0; j <= b; ++j) ab[b][j] = *reinterpret_cast<const float4*>(&A_s[16 * b + l16][16 * j + 4 * g4]);
  // 16 columns at a time (values, then key channels): X_b = T_b (R_b - sum_{j<b} A_bj X_j)
  const int vt = PP / 16;
  for (int ct = wave; ct < vt + NP / 16; ct += NT / 64) {
    const bool val = ct < vt;
    const int n = (val ? ct : ct - vt) * 16 + l16;           // this lane's value column or key channel
    v4f X[4];
    if (val) {
      const T* vb = qkv + row0 * Cq + 2 * GN + h * P + min(n, P - 1);
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) X[b][i] = ldf<T>(vb + (size_t)min(16 * b + 4 * g4 + i, tc - 1) * Cq);
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * b + 4 * g4 + i;
          X[b][i] = r < tc ? b_s[r] * X[b][i] : 0.f;
        }
    } else {
      const int nn = min(n, N - 1);
      v4f q[4], l[4];
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * b + 4 * g4 + i;
          const size_t at = (size_t)min(r, tc - 1) * prep_ld + nn;
          X[b][i] = kb[at];
          q[b][i] = qb[at];
          l[b][i] = ONE ? l_s[r] : la[r * NP + nn];          // written above by this workgroup
        }
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) l[b][i] = n < N ? l[b][i] : 0.f;
      // sums of the logs up to and after each row: inside the lane's four, over the lane groups, over the blocks
      v4f f[4], e[4];
      float tot[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const float s1 = l[b][0] + l[b][1], s2 = l[b][2] + l[b][3], own = s1 + s2;
        const float o1 = __shfl_xor(own, 16, 64), two = own + o1, o2 = __shfl_xor(two, 32, 64);
        tot[b] = two + o2;
        const float pre = (g4 & 1 ? o1 : 0.f) + (g4 & 2 ? o2 : 0.f), post = (g4 & 1 ? 0.f : o1) + (g4 & 2 ? 0.f : o2);
        f[b][0] = pre + l[b][0];
        f[b][1] = f[b][0] + l[b][1];
        f[b][2] = f[b][1] + l[b][2];
        f[b][3] = f[b][2] + l[b][3];
        e[b][3] = post;
        e[b][2] = e[b][3] + l[b][3];
        e[b][1] = e[b][2] + l[b][2];
        e[b][0] = e[b][1] + l[b][1];
      }
      float back = 0.f, fwd = 0.f;
#pragma unroll
      for (int b = 3; b >= 0; --b) {
#pragma unroll
        for (int i = 0; i < 4; ++i) e[b][i] += back;
        back += tot[b];
      }
      float* kd = Kd + cb * CL * NP + ((size_t)(ct - vt) * 64 + l16) * 16 + 4 * g4;
      float* qe = Qe + cb * CL * NP + ((size_t)(ct - vt) * 16 + 4 * g4) * 16 + l16;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        float4 kv;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * b + 4 * g4 + i;
          const bool in = r < tc && n < N;
          const float k = in ? X[b][i] : 0.f, eb = ex2(f[b][i] + fwd);
          (&kv.x)[i] = k * ex2(e[b][i]);
          qe[(size_t)b * NP * 16 + i * 16] = in ? q[b][i] * eb : 0.f;
          X[b][i] = b_s[r] * k * eb;
        }
        *reinterpret_cast<float4*>(kd + b * 256) = kv;
        fwd += tot[b];
      }
      if (g4 == 0) cdec[cb * NP + n] = ex2(fwd);
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      v4f z = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < b; ++j) z = mma16(ab[b][j], X[j][0], X[j][1], X[j][2], X[j][3], z);
      const v4f r = X[b] - z, d = r - r;
      const bool finite = d[0] == 0.f && d[1] == 0.f && d[2] == 0.f && d[3] == 0.f;
      if (__all(finite)) {
        X[b] = mma16(ab[b][b], r[0], r[1], r[2], r[3], v4f{0.f, 0.f, 0.f, 0.f});
      } else {                                               // 0 times an infinity or NaN would reach earlier tokens
        X[b] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const float v = __shfl(r[u & 3], (u >> 2) * 16 + l16, 64);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (u <= 4 * g4 + i) X[b][i] += A_s[16 * b + 4 * g4 + i][16 * b + u] * v;
        }
      }
    }
    if (val) {
      float* u = U + cb * CL * PP + (size_t)n * 16 + 4 * g4;
#pragma unroll
      for (int b = 0; b < 4; ++b) *reinterpret_cast<v4f*>(u + (size_t)b * PP * 16) = X[b];
    } else {
      float* m = M + cb * CL * NP + ((size_t)(ct - vt) * 16 + 4 * g4) * 16 + l16;
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) m[(size_t)b * NP * 16 + i * 16] = X[b][i];
    }
  }
}

// 4 KS waves, NP = 64 KS: wave w keeps the state rows 16 w .. of the workgroup's 16 value columns as an MFMA
// accumulator, and computes the 16 tokens of block w % 4 of M S_in over the 64 channels of quarter w / 4 (the quarters'
// shares meet in LDS).  The operands of the next D - 1 chunks are in registers on their way; nothing in the loop is
// conditional, so the waits for them are counted ones.
template <int KS, int D>
__global__ void __launch_bounds__(256 * KS) delta_chunk_scan_kernel(float* __restrict__ U, const float* __restrict__ M,
                                                                   const float* __restrict__ Kd, const float* __restrict__ cdec,
                                                                   float* __restrict__ sin_, float* __restrict__ state,
                                                                   const int* __restrict__ seq_slot,
                                                                   const int* __restrict__ seq_start,
                                                                   const int* __restrict__ seq_len, int H, int N, int P, int PP) {
  constexpr int LS = 20, NP = 64 * KS, UE = 4 / KS;          // LS: four rows apart are a quarter of the banks apart
  __shared__ float S_s[NP][LS], W_s[CL][LS], P_s[KS > 1 ? KS : 1][CL][LS];
  const int s = blockIdx.x, h = blockIdx.y, p0 = blockIdx.z * 16, tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g4 = lane >> 4, p = p0 + l16;
  const int tb = wave & 3, kq = wave >> 2, n0 = 16 * wave, len = seq_len[s], nc = (len + CL - 1) / CL;
  if (nc == 0) return;
  const size_t cb0 = (size_t)chunk_base(seq_len, s);
  float* st = state + ((size_t)seq_slot[s] * H + h) * N * P;
  const bool cont = seq_start[s] > 0;
  v4f S;
#pragma unroll
  for (int i = 0; i < 4; ++i) S[i] = (cont && n0 + 4 * g4 + i < N && p < P) ? st[(size_t)(n0 + 4 * g4 + i) * P + p] : 0.f;
  // this thread's elements of a W tile: KS == 1: as the products' results lie; otherwise UE tokens in a row
  const int eb = KS == 1 ? wave : tid * UE / 256, ep = KS == 1 ? l16 : tid * UE / 16 % 16, et = KS == 1 ? 4 * g4 : tid * UE % 16;
  const size_t ue = ((size_t)eb * PP + p0 + ep) * 16 + et;
  struct Chunk {
    float4 m[4], kd[4], dec;
    float u[UE];
  };
  auto load = [&](int c, Chunk& x) {
    const size_t cb = (cb0 + c) * H + h;
    const float* mp = M + cb * CL * NP + ((size_t)(tb * (NP / 16) + kq * 4) * 16 + l16) * 16 + 4 * g4;
    const float* kp = Kd + cb * CL * NP + ((size_t)wave * 64 + l16) * 16 + 4 * g4;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x.m[k] = *reinterpret_cast<const float4*>(mp + k * 256);
      x.kd[k] = *reinterpret_cast<const float4*>(kp + k * 256);
    }
    x.dec = *reinterpret_cast<const float4*>(cdec + cb * NP + n0 + 4 * g4);
#pragma unroll
    for (int i = 0; i < UE; ++i) x.u[i] = U[cb * CL * PP + ue + i];
  };
  auto step = [&](int c, const Chunk& x) {
    const size_t cb = (cb0 + c) * H + h;
    *reinterpret_cast<v4f*>(sin_ + cb * NP * PP + ((size_t)wave * PP + p) * 16 + 4 * g4) = S;
#pragma unroll
    for (int i = 0; i < 4; ++i) S_s[n0 + 4 * g4 + i][l16] = S[i];
    __syncthreads();
    float b[16];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) b[4 * k + i] = S_s[64 * kq + 16 * k + 4 * g4 + i][l16];
    __builtin_amdgcn_sched_barrier(0);                       // every read on its way before the first product waits
    v4f w[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};   // two chains
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k & 1] = mma16(x.m[k], b[4 * k], b[4 * k + 1], b[4 * k + 2], b[4 * k + 3], w[k & 1]);
    const v4f v = w[0] + w[1];
    float z[UE];
    if constexpr (KS == 1) {
#pragma unroll
      for (int i = 0; i < UE; ++i) z[i] = x.u[i] - v[i];
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) P_s[kq][16 * tb + 4 * g4 + i][l16] = v[i];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < UE; ++i) {
        float sum = 0.f;
#pragma unroll
        for (int k = 0; k < KS; ++k) sum += P_s[k][16 * eb + et + i][ep];
        z[i] = x.u[i] - sum;
      }
    }
#pragma unroll
    for (int i = 0; i < UE; ++i) {
      W_s[16 * eb + et + i][ep] = z[i];
      U[cb * CL * PP + ue + i] = z[i];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) b[4 * k + i] = W_s[16 * k + 4 * g4 + i][l16];
    __builtin_amdgcn_sched_barrier(0);
    v4f a[2] = {v4f{x.dec.x * S[0], x.dec.y * S[1], x.dec.z * S[2], x.dec.w * S[3]}, v4f{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k & 1] = mma16(x.kd[k], b[4 * k], b[4 * k + 1], b[4 * k + 2], b[4 * k + 3], a[k & 1]);
    S = a[0] + a[1];
  };
  Chunk x[D];
#pragma unroll
  for (int d = 0; d < D - 1; ++d) load(min(d, nc - 1), x[d]);
  int c0 = 0;
  for (; c0 + D <= nc; c0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      load(min(c0 + d + D - 1, nc - 1), x[(d + D - 1) % D]); // (past the end: the last chunk again, not used)
      step(c0 + d, x[d]);
    }
  }
#pragma unroll
  for (int d = 0; d < D - 1; ++d)
    if (c0 + d < nc) step(c0 + d, x[d]);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = n0 + 4 * g4 + i;
    if (n < N && p < P) st[(size_t)n * P + p] = S[i];
  }
}

// y rows of one chunk, 16 PT value columns; wave i owns token block i.  Operands straight from L2: the waves of a
// workgroup share the state and W tiles, nothing else is read twice.
template <int PT>
__global__ void __launch_bounds__(NT) delta_chunk_out_kernel(const float* __restrict__ Qe, const float* __restrict__ sin_,
                                                             const float* __restrict__ Cs, const float* __restrict__ W,
                                                             const int* __restrict__ seq_len, const int* __restrict__ seq_off,
                                                             float* __restrict__ y, int H, int NP, int P, int PP, int ntp) {
  const int c = blockIdx.x / ntp, t0 = (blockIdx.x % ntp) * PT, s = blockIdx.y, h = blockIdx.z, len = seq_len[s];
  if (c * CL >= len) return;
  const int tc = min(CL, len - c * CL), tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g4 = lane >> 4;
  if (16 * wave >= tc) return;
  const size_t row0 = (size_t)seq_off[s] + (size_t)c * CL, cb = ((size_t)chunk_base(seq_len, s) + c) * H + h;
  const int at = l16 * 16 + 4 * g4;
  const float* qp = Qe + cb * CL * NP + (size_t)wave * NP * 16 + at;
  const float* cp = Cs + cb * CL * CL + wave * 4 * 256;
  int tile[PT];                                              // column tiles; one past the last repeats it and is not stored
#pragma unroll
  for (int j = 0; j < PT; ++j) tile[j] = min(t0 + j, PP / 16 - 1) * 256;
  const float *sp = sin_ + cb * NP * PP, *wp = W + cb * CL * PP;
  v4f o[PT];
#pragma unroll
  for (int j = 0; j < PT; ++j) o[j] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int n = 0; n < NP / 16; ++n) {
    const float4 a = *reinterpret_cast<const float4*>(qp + n * 256);
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const float4 b = *reinterpret_cast<const float4*>(sp + (size_t)n * PP * 16 + tile[j] + at);
      o[j] = mma16(a, b.x, b.y, b.z, b.w, o[j]);
    }
  }
  for (int b0 = 0; b0 <= wave; ++b0) {
    const float4 a = *reinterpret_cast<const float4*>(cp + b0 * 256 + at);
    float4 w[PT];
    bool finite = true;
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      w[j] = *reinterpret_cast<const float4*>(wp + (size_t)b0 * PP * 16 + tile[j] + at);
      const float4 d = make_float4(w[j].x - w[j].x, w[j].y - w[j].y, w[j].z - w[j].z, w[j].w - w[j].w);
      finite = finite && d.x == 0.f && d.y == 0.f && d.z == 0.f && d.w == 0.f;
    }
    if (b0 < wave || __all(finite)) {
#pragma unroll
      for (int j = 0; j < PT; ++j) o[j] = mma16(a, w[j].x, w[j].y, w[j].z, w[j].w, o[j]);
    } else {                                                 // 0 times an infinity or NaN would reach earlier tokens
#pragma unroll
      for (int i = 0; i < 4; ++i)
        for (int t = 0; t <= 4 * g4 + i; ++t) {
          const float x = cp[wave * 256 + (4 * g4 + i) * 16 + t];
#pragma unroll
          for (int j = 0; j < PT; ++j) o[j][i] += x * wp[(size_t)wave * PP * 16 + tile[j] + l16 * 16 + t];
        }
    }
  }
#pragma unroll
  for (int j = 0; j < PT; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * wave + 4 * g4 + i, p = (t0 + j) * 16 + l16;
      if (t < tc && p < P) y[(row0 + t) * H * P + h * P + p] = o[j][i];
    }
}

int channels(int N) { return N <= 64 ? 64 : N <= 128 ? 128 : 256; }
}  // namespace

extern "C" {

// fp32 words of scratch: log decays, M, Qe, Kd [chunks, H, 64 NP] | U [chunks, H, 64 PP] | C [chunks, H, 64 64] | states
// [chunks, H, NP PP] | cdec [chunks, H, NP]
int64_t edge_sm_delta_chunk_floats(int64_t chunks, int64_t H, int64_t N, int64_t P) {
  const int64_t NP = channels((int)N), PP = (P + 15) & ~15LL;
  return chunks * H * (4 * CL * NP + CL * PP + CL * CL + NP * PP + NP);
}

int edge_sm_delta_chunked(const float* prep, int prep_ld, const void* qkv, int Cq, float* state, const int* seq_slot,
                          const int* seq_start, const int* seq_len, const int* seq_off, float* scratch, float* y, int rows, int n,
                          int chunks, int max_chunks, int H, int G, int N, int P, int GD, int f32, hipStream_t st) {
  if (n == 0 || rows == 0 || max_chunks <= 0) return 0;
  if (G <= 0 || H % G || N < 1 || N > 256 || P < 1 || (GD != N && GD != 1)) return -2;
  const int NP = channels(N), PP = (P + 15) & ~15;
  const int64_t CH = (int64_t)chunks * H;
  float* la = scratch;
  float *M = la + CH * CL * NP, *Qe = M + CH * CL * NP, *Kd = Qe + CH * CL * NP, *U = Kd + CH * CL * NP;
  float *Cs = U + CH * CL * PP, *sin_ = Cs + CH * CL * CL, *cdec = sin_ + CH * NP * PP;
  const bool vec = N % 4 == 0 && prep_ld % 4 == 0 && ((uintptr_t)prep & 15) == 0;
  if (((uintptr_t)scratch & 15) != 0) return -3;
#define SM_DSOLVE(T, V, ONE)                                                                                              \
  hipLaunchKernelGGL((delta_chunk_solve_kernel<T, V, ONE>), dim3(max_chunks, n, H), dim3(NT), 0, st, prep, prep_ld,       \
                     (const T*)qkv, Cq, seq_len, seq_off, la, U, M, Qe, Kd, Cs, cdec, H, G, N, NP, P, PP)
#define SM_DSOLVE_T(T)                            \
  do {                                            \
    if (GD == 1) {                                \
      if (vec) SM_DSOLVE(T, true, true);          \
      else SM_DSOLVE(T, false, true);             \
    } else if (vec) SM_DSOLVE(T, true, false);    \
    else SM_DSOLVE(T, false, false);              \
  } while (0)
  if (f32) SM_DSOLVE_T(float);
  else SM_DSOLVE_T(bf16_t);
#undef SM_DSOLVE_T
#undef SM_DSOLVE
  const dim3 grid(n, H, PP / 16);
#define SM_DSCAN(KS, D)                                                                                                       \
  hipLaunchKernelGGL((delta_chunk_scan_kernel<KS, D>), grid, dim3(256 * KS), 0, st, U, M, Kd, cdec, sin_, state, seq_slot,    \
                     seq_start, seq_len, H, N, P, PP)
  if (NP == 64) SM_DSCAN(1, 3);
  else if (NP == 128) SM_DSCAN(2, 3);
  else SM_DSCAN(4, 2);
#undef SM_DSCAN
  const int ntp = (PP + 63) / 64;
  hipLaunchKernelGGL((delta_chunk_out_kernel<4>), dim3(max_chunks * ntp, n, H), dim3(NT), 0, st, Qe, sin_, Cs, U, seq_len, seq_off,
                     y, H, NP, P, PP, ntp);
  return (int)hipGetLastError();
}

}  // extern "C"
