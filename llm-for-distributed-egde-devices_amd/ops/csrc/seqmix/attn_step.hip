// Windowed attention with pooled blocks over a paged cache for steps of few queries (decode steps): attn_kernel's rule
// (seqmix.hip) of what a query sees and how its scores are formed, fp32 or bf16 rows.
//
// Bound by latency: a handful of queries, each over some hundred keys that lie in caches, so what counts is the length of the
// chain of dependent loads.  attn_kernel lets one thread walk a whole key row, 16 bytes a trip.  Here a wave owns 16 keys at a time:
// four lanes hold a key's row (all of it in flight at once, and the 16 value rows beside it), the scores of the SH heads come from
// the matrix cores (bf16 rows 16x16x32, fp32 rows 16x16x4; the heads are repeated over the 16 rows, so that every group of 16
// lanes holds all of them), and each wave keeps its own running maximum, sum and weighted values, fp32 and without a barrier;
// the waves meet once, in LDS, at the end.  A workgroup's time is its vector instructions then (some 1.5 us for 128 keys and four
// heads, 0.7 for one), so few queries run one head a workgroup; reading the next rows ahead took registers and gained nothing, and
// an unrolled end cost 30 KB of code that every launch has to fetch (6.0 -> 18 us).
// One head of fp32 rows takes its scores on the vector ALU: 16 products a lane and two exchanges instead of 16 matrix instructions of
// which 15 rows in 16 are idle, and half their error (4e-7 -> 2.7e-7 of the result, against 64 bits).  us, a launch in a graph, before /
// after: 16 heads of 64 in 4 groups, 2 tokens behind 777 (window 512, 16 blocks) 9.2 / 8.2, 8 behind 400 8.6 / 7.8; of 128, 1 behind 700 15.5 /
// 14.6.  What is left there is the bytes of one CU: four times the keys in flight, the next rows ahead and 64 keys a wave at a time gave
// nothing, other workgroups that fetch them into the L2 something where CUs are idle (attn_ssd_kernel).
// Rows of up to 64 numbers are held to 128 registers a lane, two workgroups to a CU: four fp32 heads with blocks need one more
// otherwise (us, 32 heads in 2 groups, 64 rows, window 512, 16 blocks, behind 800 27.4 / 22.8, 64 heads in 8, 32 rows behind 1600 30.3 / 24.6).
// us, attn_kernel with its sum over key splits / this (bf16 but for the first): fp32, 16 heads of 64 in 4 groups, 2 tokens behind
// 777 (window 512, 16 blocks) 15.3 / 9.9; latent rows of 160, 16 heads, 4 tokens behind 97 19.4 / 5.2; of 320, 6 behind 1100 (window 1024)
// 35.1 / 27.0, 1 behind 7600 56 / 21; 16 heads of 128 in 4 groups, 6 in chunks of 1000 20.7 / 13.3.
#include "common.h"
#include "seqmix/ssd_step.h"

extern "C" int edge_sm_attention_rmax(int rows, int H, int G, int D, int Dv);
extern "C" int edge_sm_attention_splits(int rows, int G, int chunks);

namespace {

__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false)));
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, false)));
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x124, 0xF, 0xF, false)));
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xF, 0xF, false)));
  return v;
}

struct StepArgs {
  const void *q, *gate, *kp, *vp;
  const float *kb, *vb;
  const int *tok_seq, *tok_pos, *seq_slot, *ptab;
  void* out;
  float* part;
  const float *slopes, *sink, *rel;
  const void* uv;                                            // [H, Dv, vdim]: each head's result times its matrix (null: as it is)
  int vdim, rows, gate_ld, ptab_ld, H, G, D, Dv, page, page_sh, PB, window, pool_sh, nsp, nsplit, kld, vld, chunked, gate_elem, keep_first, rel_n, out_ld;
  float scale, cap, out_scale;
};

// 16 keys' rows of one wave: lane (key = lane & 15, parts 4 c + (lane >> 4) of 8 numbers of its row) and values (LPK lanes a key, 8
// numbers each).  fp32 queries: the two halves of a part are 16 (of values 4 LPK) numbers apart, so that neighbouring lanes of every
// load read neighbouring 16 bytes (a workgroup's time is the bytes that its CU takes in, some 70 a ns)
template <typename KT, int NC, int DVL>
struct Tile {
  static constexpr int Q = sizeof(KT) / 2, VP = 2 * DVL;
  uint4 k[NC][Q], v[VP][Q];
};

template <typename KT, int NC, int DVL, bool F32>
__device__ __forceinline__ void tile_load(Tile<KT, NC, DVL>& t, const KT* kb, const KT* vb, int row, int kld, int vld, int D, int Dv) {
  constexpr int LPK = 8 * DVL, KPR = 64 / LPK;
  const int lane = threadIdx.x & 63, grp = lane >> 4, vl = lane % LPK;
  const KT* kr = kb + (size_t)row * kld;
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int q = 0; q < Tile<KT, NC, DVL>::Q; ++q)
      t.k[c][q] = *reinterpret_cast<const uint4*>(F32 ? kr + min(32 * c + 16 * q + 4 * grp, D - 4) : kr + min(32 * c + 8 * grp, D - 8) + 4 * q);
#pragma unroll
  for (int p = 0; p < Tile<KT, NC, DVL>::VP; ++p) {
    const KT* vr = vb + (size_t)__shfl(row, p * KPR + lane / LPK, 64) * vld;
#pragma unroll
    for (int q = 0; q < Tile<KT, NC, DVL>::Q; ++q)
      t.v[p][q] = *reinterpret_cast<const uint4*>(F32 ? vr + min(4 * (LPK * q + vl), Dv - 4) : vr + min(8 * vl, Dv - 8) + 4 * q);
  }
}

// halves the V numbers of a lane between partners S apart, down to partners S0 apart; off: the first number it is left with
template <int V, int S, int S0, int N>
__device__ __forceinline__ void halve(float (&v)[N], int& off, int lane) {
  if constexpr (S >= S0) {
    const bool hi = lane & S;
#pragma unroll
    for (int j = 0; j < V / 2; ++j) {
      const float give = hi ? v[j] : v[j + V / 2], keep = hi ? v[j + V / 2] : v[j];
      v[j] = keep + lane_xor(give, S);
    }
    off += hi ? V / 2 : 0;
    halve<V / 2, S / 2, S0>(v, off, lane);
  }
}

constexpr int MAX_VDIM = 128;                               // columns of a head's matrix
constexpr int STEP_NW = 8;                                  // waves of a workgroup

// e^x for x <= 0 (or NaN) to about one rounding: x log2(e) in two parts, the small one to first order
__device__ __forceinline__ float exp_neg(float x) {
  constexpr float L = 1.44269502e+00f, L2 = 1.92596299e-08f, LN2 = 6.93147182e-01f;     // log2(e) = L + L2
  x = x < -200.f ? -200.f : x;
  const float t = x * L, lo = fmaf(x, L2, fmaf(x, L, -t)), p = ex2(t);
  return fmaf(p * lo, LN2, p);
}

template <typename T, int NC, int DVL, int SH, bool POOL, bool EX>
__device__ __forceinline__ void attn_step_body(const StepArgs& a, int block) {
  constexpr int NW = STEP_NW, LPK = 8 * DVL, KPR = 64 / LPK, VP = 2 * DVL, RK = 16 * NW, DR = 64 * DVL;
  __shared__ __attribute__((aligned(16))) float p_s[NW][16][SH];
  __shared__ __attribute__((aligned(16))) float red[NW][SH][DR];
  __shared__ float m_s[NW][SH], l_s[NW][SH], tot_s[2][SH];
  __shared__ __attribute__((aligned(16))) float y_s[EX ? DR : 1], e_s[EX ? NW : 1][EX ? MAX_VDIM : 1];
  // consecutive workgroups go to the eight dies in turn: those of one (token, kv head, part of its keys) stay on one die, where they
  // read the same rows
  const int unit = block % 8 + 8 * (block / 8 / a.nsp), sub = block / 8 % a.nsp;
  if (unit >= a.rows * a.G * a.nsplit) return;
  const int z = unit % a.nsplit, g = unit / a.nsplit % a.G, t = unit / a.nsplit / a.G, r0 = sub * SH, D = a.D, Dv = a.Dv;
  const int R = min(SH, a.H / a.G - r0), hq0 = g * (a.H / a.G) + r0;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int key = lane & 15, grp = lane >> 4;
  const int i = a.tok_pos[t];
  const int* pt = a.ptab + (size_t)a.seq_slot[a.tok_seq[t]] * a.ptab_ld;
  // the queries as the matrix cores' rows: row = lane & 15 is head row % SH; numbers past D (or heads past R) are zero
  const T* qp = reinterpret_cast<const T*>(a.q) + ((size_t)t * a.H + hq0 + min(key % SH, R - 1)) * D;
  // (the widest rows of four fp32 heads have no registers for either: 128 bytes a lane spilled, 40 without)
  constexpr bool ROOM = SH == 1 || sizeof(T) == 2 || NC <= 4, F32 = sizeof(T) == 4 && ROOM, DOT = F32 && SH == 1;
  uint4 qr[NC][Tile<T, NC, DVL>::Q];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int e = 0; e < Tile<T, NC, DVL>::Q; ++e)
      qr[c][e] = *reinterpret_cast<const uint4*>(F32 ? qp + min(32 * c + 16 * e + 4 * grp, D - 4) : qp + min(32 * c + 8 * grp, D - 8) + 4 * e);
  if constexpr (ROOM) asm volatile("" ::: "memory");        // (all on their way before one is looked at)
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int e = 0; e < Tile<T, NC, DVL>::Q; ++e)
      if ((F32 ? 32 * c + 16 * e + 4 * grp : 32 * c + 8 * grp) >= D || (key % SH) >= R) qr[c][e] = uint4{0u, 0u, 0u, 0u};
  float m[SH], l[SH], acc[SH * 8];
#pragma unroll
  for (int r = 0; r < SH; ++r) { m[r] = -INFINITY; l[r] = 0.f; }
#pragma unroll
  for (int e = 0; e < SH * 8; ++e) acc[e] = 0.f;
  const int win = a.window;
  const int jlo = win > 0 ? (a.chunked ? i - i % win : max(0, i - win + 1)) : 0;
  const int kf = !a.chunked && win > 0 ? min(a.keep_first, jlo) : 0;
  const int nk = kf + i - jlo + 1;                           // tokens this query sees, the kept first ones in front
  const int nb = POOL && i - win + 1 > 0 ? (i - win + 1) >> a.pool_sh : 0;
  const int rounds_k = (nk + RK - 1) / RK, rounds = rounds_k + (nb + RK - 1) / RK;
  int first = 0, last = rounds;
  if (a.nsplit > 1) {
    const int per = (rounds + a.nsplit - 1) / a.nsplit;
    first = z * per;
    last = min(rounds, first + per);
  }

  // rounds [b, e) over n keys; row(x) the cached row of key x
  auto walk = [&](auto kt, const auto* kbase, const auto* vbase, int kld, int vld, int n, int b, int e, auto&& row, auto&& shape) {
    using KT = decltype(kt);
    using TL = Tile<KT, NC, DVL>;
    const int end = min(n, e * RK);
    int x0 = b * RK + wave * 16;
    if (x0 >= end) return;
    auto row_of = [&](int x) { return row(min(x + key, n - 1)); };
    int rw = row_of(x0);
#pragma unroll 1
    for (; x0 < end; x0 += RK) {
      TL tl;
      tile_load<KT, NC, DVL, F32>(tl, kbase, vbase, rw, kld, vld, D, Dv);
      rw = row_of(x0 + RK);                                  // (past the end: the last key's, not used)
      v4f s2[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};     // (two sums: half the chain)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        v4f& s = s2[c & 1];
        const bool in = 32 * c + 8 * grp < D;
        if constexpr (TL::Q == 1) {
          uint4 kv = tl.k[c][0];
          if (!in) kv = uint4{0u, 0u, 0u, 0u};
          s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8s, qr[c][0]), __builtin_bit_cast(v8s, kv), s, 0, 0, 0);
        } else {
          float qf[8], kf8[8];
          load8<T>(reinterpret_cast<const T*>(&qr[c][0]), qf);
          load8<float>(reinterpret_cast<const float*>(&tl.k[c][0]), kf8);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float kx = (F32 ? 32 * c + 16 * (j / 4) + 4 * grp < D : in) ? kf8[j] : 0.f;
            if constexpr (DOT) s[j & 3] = fmaf(qf[j], kx, s[j & 3]);
            else s = mfma4(qf[j], kx, s);
          }
        }
      }
      v4f s = s2[0] + s2[1];
      if constexpr (DOT) s[0] = xor_sum(xor_sum((s[0] + s[1]) + (s[2] + s[3]), 16), 32);
      s *= a.scale;
      shape(s, x0 + key);                                    // (s[r], r < SH: head r's score of this lane's key)
      const bool ok = x0 + key < n;
      float p[SH], mn[SH];
      bool grows = false;
#pragma unroll
      for (int r = 0; r < SH; ++r) {
        if (!ok) s[r] = -INFINITY;
        mn[r] = fmaxf(m[r], row16_max(s[r]));
        grows |= mn[r] != m[r];
      }
      if (__builtin_amdgcn_readfirstlane(grows)) {           // (every lane holds the same maxima)
#pragma unroll
        for (int r = 0; r < SH; ++r) {
          const float al = m[r] == -INFINITY ? 0.f : exp_neg(m[r] - mn[r]);
          l[r] *= al;
          m[r] = mn[r];
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[r * 8 + j] *= al;
        }
      }
#pragma unroll
      for (int r = 0; r < SH; ++r) {
        p[r] = exp_neg(s[r] - (mn[r] == -INFINITY ? 0.f : mn[r]));
        l[r] += row16_sum(p[r]);
      }
      if (grp == 0) {
        if constexpr (SH == 4) *reinterpret_cast<float4*>(&p_s[wave][key][0]) = make_float4(p[0], p[1], p[2], p[3]);
        else p_s[wave][key][0] = p[0];
      }
      __builtin_amdgcn_wave_barrier();                       // (a wave's own LDS accesses stay in order)
      const bool full = x0 + 16 <= n;
#pragma unroll
      for (int ps = 0; ps < VP; ++ps) {
        const int kx = ps * KPR + lane / LPK;
        float w[SH], vf[8];
        if constexpr (SH == 4) {
          const float4 w4 = *reinterpret_cast<const float4*>(&p_s[wave][kx][0]);
          w[0] = w4.x; w[1] = w4.y; w[2] = w4.z; w[3] = w4.w;
        } else w[0] = p_s[wave][kx][0];
        load8<KT>(reinterpret_cast<const KT*>(&tl.v[ps][0]), vf);
        if (!full && x0 + kx >= n) {                         // a key past the end: its weight is 0, its row some other key's
#pragma unroll
          for (int j = 0; j < 8; ++j) vf[j] = 0.f;
        }
#pragma unroll
        for (int r = 0; r < SH; ++r)
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[r * 8 + j] += w[r] * vf[j];
      }
      __builtin_amdgcn_wave_barrier();
    }
  };
  auto token = [&](int x) { return x < kf ? x : jlo + x - kf; };
  walk(T{}, reinterpret_cast<const T*>(a.kp) + g * D, reinterpret_cast<const T*>(a.vp) + g * Dv, a.kld, a.vld, nk, first,
       min(last, rounds_k), [&](int x) { const int j = token(x); return (pt[j >> a.page_sh] << a.page_sh) + (j & (a.page - 1)); },
       [&](v4f& s, int x) {
         if (a.cap > 0.f || a.slopes || a.rel) {             // uniform: nothing of this for plain scores
           const int dist = i - token(x);
#pragma unroll
           for (int r = 0; r < SH; ++r) {
             const int h = hq0 + min(r, R - 1);
             if (a.cap > 0.f) s[r] = a.cap * tanhf(s[r] / a.cap);
             if (a.slopes) s[r] -= a.slopes[h] * (float)dist;
             if (a.rel) s[r] += a.rel[(size_t)h * a.rel_n + min(max(dist, 0), a.rel_n - 1)];
           }
         }
       });
  if constexpr (POOL)
    walk(float{}, a.kb + g * D, a.vb + g * Dv, a.G * D, a.G * Dv, nb, max(first - rounds_k, 0), last - rounds_k,
         [&](int x) {
           const int p0 = x << a.pool_sh;
           return pt[p0 >> a.page_sh] * a.PB + ((p0 & (a.page - 1)) >> a.pool_sh);
         },
         [&](v4f&, int) {});

  // uv: eight columns a thread, rows rg, rg + EG, .. (a matrix of 64 DVL x 128: 8 DVL or 16 DVL registers, on its way from here)
  constexpr int UR = EX ? 2 * DVL : 1, TQ = sizeof(T) / 2;
  uint4 uvr[UR][TQ];
  const int vl = EX ? a.vdim / 8 : 64, uc = tid % vl * 8, rg = tid / vl, EG = NW * 64 / vl;
  if constexpr (EX) {
#pragma unroll
    for (int k = 0; k < UR; ++k)
#pragma unroll
      for (int q = 0; q < TQ; ++q)
        uvr[k][q] = reinterpret_cast<const uint4*>(reinterpret_cast<const T*>(a.uv) +
                                                   ((size_t)hq0 * Dv + min(rg + EG * k, Dv - 1)) * a.vdim + uc)[q];
  }
  // add up the lanes that walked different keys, then the waves
  int off = 0;
  halve<SH * 8, 32, LPK>(acc, off, lane);
  constexpr int VN = SH * 8 / KPR;                           // numbers a lane is left with, from off on
  const int d0 = lane % LPK * 8;
#pragma unroll
  for (int j = 0; j < VN; ++j) {
    const int e = (off + j) % 8;
    red[wave][(off + j) / 8][F32 ? 4 * (LPK * (e / 4) + lane % LPK) + e % 4 : d0 + e] = acc[j];
  }
  if (lane == 0) {
#pragma unroll
    for (int r = 0; r < SH; ++r) { m_s[wave][r] = m[r]; l_s[wave][r] = l[r]; }
  }
  __syncthreads();
  if (wave == 0) {                                           // lane = (wave, head): the waves' weights
    const int w = min(lane / SH, NW - 1), r = lane % SH;
    const bool sk = a.sink && z == 0;
    const float sv = sk ? a.sink[hq0 + min(r, R - 1)] : -INFINITY, mw = m_s[w][r];
    float M = fmaxf(mw, sv);
#pragma unroll
    for (int o = SH; o < 64; o <<= 1) M = xor_max(M, o);
    const float x = mw == -INFINITY ? 0.f : exp_neg(mw - M);
    float ls = lane < NW * SH ? x * l_s[w][r] : 0.f;
#pragma unroll
    for (int o = SH; o < 64; o <<= 1) ls = xor_sum(ls, o);
    if (sk) ls += exp_neg(sv - M);
    if (lane < NW * SH) m_s[w][r] = x;
    if (lane < SH) { tot_s[0][r] = M; tot_s[1][r] = ls; }
  }
  __syncthreads();
  const int d = tid % DR;
#pragma unroll 1
  for (int r = tid / DR; r < R; r += NW / DVL) {
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) o += m_s[w][r] * red[w][r][d];
    if (d >= Dv) continue;
    if (a.nsplit > 1) {                                      // unnormalised sums, maximum and sum per head (attn_merge_kernel's rows)
      float* dst = a.part + (((size_t)t * a.G * a.nsp + g * a.nsp + sub) * a.nsplit + z) * (SH * (Dv + 2));
      dst[r * Dv + d] = o;
      if (d == 0) { dst[SH * Dv + r] = tot_s[0][r]; dst[SH * Dv + SH + r] = tot_s[1][r]; }
    } else {
      const int h = hq0 + r;
      float y = o / tot_s[1][r];
      if constexpr (EX) {
        y_s[d] = y;
        continue;
      }
      if (a.gate) y *= sigmoidf_(ldf<T>(reinterpret_cast<const T*>(a.gate) + (size_t)t * a.gate_ld + (a.gate_elem ? h * Dv + d : h)));
      stf<T>(reinterpret_cast<T*>(a.out) + (size_t)t * a.out_ld + h * Dv + d, y * a.out_scale);
    }
  }
  if constexpr (EX) {
    __syncthreads();
    float e8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < UR; ++k) {
      const int r = rg + EG * k;
      float uf[8];
      load8<T>(reinterpret_cast<const T*>(&uvr[k][0]), uf);
      const float y = r < Dv ? y_s[min(r, DR - 1)] : 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) e8[e] += r < Dv ? y * uf[e] : 0.f;
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
      if (o >= vl) {
#pragma unroll
        for (int e = 0; e < 8; ++e) e8[e] = xor_sum(e8[e], o);
      }
    if (lane < vl)
#pragma unroll
      for (int e = 0; e < 8; ++e) e_s[wave][uc + e] = e8[e];
    __syncthreads();
    if (tid < a.vdim) {
      float y = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) y += e_s[w][tid];
      if (a.gate) y *= sigmoidf_(ldf<T>(reinterpret_cast<const T*>(a.gate) + (size_t)t * a.gate_ld + hq0 * a.vdim + tid));
      stf<T>(reinterpret_cast<T*>(a.out) + (size_t)t * a.out_ld + hq0 * a.vdim + tid, y);
    }
  }
}

template <typename T, int NC, int DVL, int SH, bool POOL, bool EX>
__global__ void __launch_bounds__(STEP_NW * 64, NC == 2 ? 4 : 2) attn_step_kernel(StepArgs a) {
  attn_step_body<T, NC, DVL, SH, POOL, EX>(a, blockIdx.x);
}

// One head a workgroup over whole keys, beside one token of the state-space recurrence, two heads a workgroup: a parallel layer's two
// mixers, which wait for nothing of each other and leave most of the chip idle each.  The workgroups behind those fetch: `fetch` of them
// bring a (query, kv head) pair's keys and values into the L2 of the die whose workgroups walk them, where one CU takes in what it waits for
// at the pace of its own misses.  us in a decode step whose weights have passed through the caches since (fp32, 16 heads of 64 in 4
// groups, 2 tokens behind 800, window 512, 16 state heads of 64 x 64): attention 11.2 and state 4.7 in two launches (attention with the
// fetching 9.9, with products on the vector ALU 10.8), this 9.1; a prompt of 777 and 15 such steps, four layers, 6.79 -> 6.47 ms.
// Fetched in the launch before instead (parallel_step.hip), attention is at 9.2 alone, but that launch at 6.8 instead of 4.6.
template <typename T, int NC, int DVL, bool POOL, int N, int P>
__global__ void __launch_bounds__(STEP_NW * 64) attn_ssd_kernel(StepArgs a, SsdStep s, int heads, int fetch) {
  __shared__ __attribute__((aligned(16))) float sum_s[STEP_NW * 64 / NT][NT / 64][P];
  const int units = a.rows * a.G, own = (units + 7) / 8 * 8 * a.nsp, tid = threadIdx.x;
  int b = blockIdx.x;
  if (b < own) return attn_step_body<T, NC, DVL, 1, POOL, false>(a, b);
  b -= own;
  if (b >= heads) {                                          // (heads: a multiple of 8, and so is own: b % 8 is the die)
    b -= heads;
    const int unit = b % 8 + 8 * (b / 8 / fetch), part = b / 8 % fetch;
    if (unit >= units) return;
    const int g = unit % a.G, t = unit / a.G, i = a.tok_pos[t], jlo = a.window > 0 ? max(0, i - a.window + 1) : 0;
    const int* pt = a.ptab + (size_t)a.seq_slot[a.tok_seq[t]] * a.ptab_ld;
    const int kparts = a.D * (int)sizeof(T) / 16, per = kparts + a.Dv * (int)sizeof(T) / 16, n = (i - jlo + 1) * per;
    uint32_t seen = 0;
#pragma unroll 4
    for (int e = part * (STEP_NW * 64) + tid; e < n; e += fetch * (STEP_NW * 64)) {
      const int j = jlo + e / per, c = e % per;
      const size_t row = (pt[j >> a.page_sh] << a.page_sh) + (j & (a.page - 1));
      const T* at = c < kparts ? reinterpret_cast<const T*>(a.kp) + row * a.kld + g * a.D + c * (16 / sizeof(T))
                               : reinterpret_cast<const T*>(a.vp) + row * a.vld + g * a.Dv + (c - kparts) * (16 / sizeof(T));
      seen |= *reinterpret_cast<const uint32_t*>(at);
    }
    asm volatile("" ::"v"(seen));
    return;
  }
  const int pairs = s.H / 2, q = b / pairs;
  if (q >= a.rows) return;
  ssd_step_body<T, N, P>(s, q, b % pairs * 2 + tid / NT, tid % NT, sum_s[tid / NT]);
}

template <typename T, int SH, bool EX>
int run_step(const StepArgs& a, hipStream_t st) {
  const dim3 grid((a.rows * a.G * a.nsplit + 7) / 8 * 8 * a.nsp), block(STEP_NW * 64);
  const bool pool = a.pool_sh >= 0;
#define STEP(NC, DL, P) hipLaunchKernelGGL((attn_step_kernel<T, NC, DL, SH, P, EX>), grid, block, 0, st, a)
  if constexpr (EX) {
    if (pool) return -2;
    if (a.D <= 128 && a.Dv <= 128) STEP(4, 2, false);
    else if (a.D <= 192 && a.Dv <= 128) STEP(6, 2, false);
    else STEP(10, 4, false);
    return (int)hipGetLastError();
  }
  if (a.D <= 64 && a.Dv <= 64) { if (pool) STEP(2, 1, true); else STEP(2, 1, false); }
  else if (a.D <= 128 && a.Dv <= 128) { if (pool) STEP(4, 2, true); else STEP(4, 2, false); }
  else if (pool) return -2;
  else if (a.D <= 192 && a.Dv <= 128) STEP(6, 2, false);
  else STEP(10, 4, false);
#undef STEP
  return (int)hipGetLastError();
}

template <typename T, int NC, int DVL, bool POOL>
int run_beside(const StepArgs& a, const SsdStep& s, int N, int P, hipStream_t st) {
  const int units8 = (a.rows * a.G + 7) / 8, own = units8 * 8 * a.nsp, heads = (a.rows * s.H / 2 + 7) / 8 * 8;
  const int fetch = max(0, min(12, (256 - own - heads) / (8 * units8)));    // as the chip has CUs left
#define BESIDE(NN, PP)                                                                                                          \
  if (N == NN && P == PP) {                                                                                                     \
    hipLaunchKernelGGL((attn_ssd_kernel<T, NC, DVL, POOL, NN, PP>), dim3(own + heads + units8 * 8 * fetch), dim3(STEP_NW * 64), 0, st, a, \
                       s, heads, fetch);                                                                                        \
    return (int)hipGetLastError();                                                                                              \
  }
  BESIDE(64, 64)
  BESIDE(128, 64)
  BESIDE(64, 128)
  BESIDE(128, 128)
#undef BESIDE
  return -2;
}

// Estimates in us, fitted to both kernels' times at 936 points (13 shapes of 8 to 64 heads of 32 to 320 numbers, both types, 1 to 400 rows
// behind 17 to 8000 keys; half of them were within 7 %; fp32 rows of one head a workgroup have since become 5 to 11 % quicker): a launch, then the longer of one workgroup's chain and the chip's work per CU,
// then the sum over key splits.
constexpr double LAUNCH_US = 4.5, MERGE_US = 4.5;

struct Cost {
  double chain, work;
  double us(int ns) const { return LAUNCH_US + (chain > work ? chain : work) + (ns > 1 ? MERGE_US : 0.); }
};
// groups workgroups of sh heads, each over its part of vis keys, 128 a round; a round's numbers count as the kernel pads them
Cost step_cost(int f32, int sh, int D, int Dv, long groups, long vis, int ns) {
  static const double fit[2][2][5] = {{{0.57, 0.0043, 0.0017, 0.21, 0.0037}, {1.8, 0.0063, 0.0071, 0.73, 0.0053}},
                                      {{0.28, 0.0096, 0.002, 0.13, 0.01}, {1.4, 0.014, 0.0068, 0.5, 0.016}}};
  const double* p = fit[f32 ? 1 : 0][sh == 4];
  const int w = D <= 64 && Dv <= 64 ? 128 : D <= 128 && Dv <= 128 ? 256 : D <= 192 && Dv <= 128 ? 320 : 576;
  const double rounds = (double)(((vis + 127) / 128 + ns - 1) / ns);
  return {p[0] + rounds * p[1] * w, groups / 256.0 * (p[2] * w + rounds * (p[3] + p[4] * w))};
}
double step_us(int f32, int sh, int D, int Dv, long groups, long vis, int ns) {
  return step_cost(f32, sh, D, Dv, groups, vis, ns).us(ns);
}

// attn_kernel on fp32 rows, with the heads that its own rule gives it
Cost attn_kernel_cost(int rows, int H, int G, int D, int Dv, long vis, int ns) {
  const int R = H / G, rm = edge_sm_attention_rmax(rows, H, G, D, Dv);
  if (rm == 0) return {1e30, 1e30};
  const double chunks = (double)(((vis + 255) / 256 + ns - 1) / ns), keys = (double)vis / ns;
  return {chunks * (2.6 + 0.0099 * D * rm) + keys * (0.0019 + 2.3e-5 * Dv * rm),
          rows * (double)G * ((R + rm - 1) / rm) * ns / 256.0 * (0.99 + keys * 1.5e-4 * (D + Dv) + chunks * 0.0068 * D * rm)};
}
double attn_kernel_us(int rows, int H, int G, int D, int Dv, long vis) {
  const int ns = edge_sm_attention_splits(rows, G, (int)((vis + 255) / 256));
  return attn_kernel_cost(rows, H, G, D, Dv, vis, ns).us(ns);
}

}  // namespace

extern "C" int edge_sm_attn_merge(const float* part, const void* gate, int gate_ld, void* out, int rows, int H, int G, int Dv, int nsp,
                                  int nsplit, int rmax, int gate_elem, int out_ld, float out_scale, int f32, hipStream_t st);

extern "C" {

// query heads of a workgroup in the low bits, workgroups that share one query's keys (vis: the most a query may see) above; 0: the
// step is not this kernel's.
int edge_sm_attention_step_plan(int rows, int H, int G, int D, int Dv, int kld, int vld, int page, int pool, long vis,
                                int f32, uintptr_t addresses) {
  if (rows < 1 || G < 1 || H % G || D < 8 || Dv < 8 || D > 320 || Dv > 256 || D % 8 || Dv % 8 || kld % 8 || vld % 8 || addresses % 16 ||
      page < 1 || (page & (page - 1)) || pool < 0 || (pool & (pool - 1)) || pool > page || (pool > 0 && (D > 128 || Dv > 128)))
    return 0;
  // One head a workgroup for few heads altogether; with more, four (one reading of the keys, one product for their scores), but not
  // for one or two heads a kv head, of which three or two places would stay empty.
  const int R = H / G, per4 = (R + 3) / 4;
  const bool few = (long)rows * H <= 256;
  const long groups4 = (long)rows * G * per4;
  if (!few) {
    if (R < 3) return 0;
    // fp32 rows: attn_kernel multiplies without the matrix cores' idle rows and is ahead once its workgroups fill the chip (us,
    // attn_kernel / four heads: 16 heads of 64 in 4 groups, 64 rows behind 400 19.8 / 15.6, a portion of 150 behind 1000 42 / 49; of 128, 64
    // behind 700 43 / 37, 400 behind 17 37 / 49; rows of 160, 256 behind 200 45 / 61) or splits long keys (64 heads of 128 in 8, 8
    // behind 8000 135 / 153)
    if (f32 && (D > 128 || groups4 * 4 * per4 * 64 > (D <= 64 ? 512L * D : 256L * 64) * R || (vis > 2500 && (long)rows * G <= 64)))
      return 0;
    // one chunk of attn_kernel's with all heads of a group in it (bf16, 64 heads of 128 in 8 groups, 256 rows behind 200 109 / 125)
    if (!f32 && per4 > 1 && groups4 >= 2048 && vis <= 256 && D >= 128) return 0;
  }
  // Of what is left the quickest by estimate: heads a workgroup, and workgroups for a query's keys.  For few heads of fp32 rows
  // attn_kernel is one of the choices; four heads a workgroup or long walks are not.  Keys are split from 1536 on (512 of fp32 rows): the
  // sum is a launch more, which a step whose sequences are far shorter than vis pays too.  us, attn_kernel / these forms' choice: fp32,
  // 16 heads of 64 in 4 groups, 1 row behind 700 14.8 / 11.5, 8 rows behind 8000 37 (attn_kernel's), of 128, 1 behind 2000 20.4 / 18.5; rows
  // of 160, 8 behind 200 14.8 / 11.8, 16 behind 4000 53 (attn_kernel's); bf16 rows of 320, 4 behind 700 34 / 21, 16 behind 8000 159 / 64
  double best = few && f32 ? attn_kernel_us(rows, H, G, D, Dv, vis) / 1.04 : 1e30;
  int plan = 0;
  for (int sh = 1; sh <= 4; sh += 3) {
    if (sh == 1 ? !few : R < 3 || (few && f32)) continue;
    const long groups = (long)rows * G * ((R + sh - 1) / sh);
    for (int ns = 1; ns <= 16; ns *= 2) {
      if ((ns > 1 && (vis <= (f32 ? 512 : 1536) || vis < 256 * ns || groups * ns > 1024)) || (few && f32 && vis > 1100L * ns)) continue;
      const double us = step_us(f32, sh, D, Dv, groups * ns, vis, ns);
      if (us < best) { best = us; plan = sh + 8 * ns; }
    }
  }
  return plan;
}

// us of an fp32 step of portions in attn_kernel or the kernels here, as edge_sm_attention_step_plan deals it: the chain of the row that sees
// the most keys, the work of rows that see `mean`.  Workgroups of several rounds overlap the two: attn_kernel's shares were fitted to 454
// steps of 1 to 9 portions (2 to 32 heads of 32 to 160 numbers; rms 12 %; the larger of the two, as above, is up to three times too much).
double edge_sm_attention_us(int rows, int H, int G, int D, int Dv, int kld, int vld, int page, int pool, long vis, long mean, uintptr_t addresses) {
  const int plan = edge_sm_attention_step_plan(rows, H, G, D, Dv, kld, vld, page, pool, vis, 1, addresses), sh = plan % 8, ns = plan / 8;
  if (plan) {
    const long groups = (long)rows * G * ((H / G + sh - 1) / sh) * ns;
    return Cost{step_cost(1, sh, D, Dv, groups, vis, ns).chain, step_cost(1, sh, D, Dv, groups, mean, ns).work}.us(ns);
  }
  const int parts = edge_sm_attention_splits(rows, G, (int)((vis + 255) / 256));
  return 4. + 0.7 * attn_kernel_cost(rows, H, G, D, Dv, vis, parts).chain + 0.4 * attn_kernel_cost(rows, H, G, D, Dv, mean, parts).work +
         (parts > 1 ? MERGE_US : 0.);
}

size_t edge_sm_attention_step_floats(int rows, int H, int G, int Dv, int plan) {
  const int sh = plan % 8, nsplit = plan / 8;
  return nsplit > 1 ? (size_t)rows * G * ((H / G + sh - 1) / sh) * nsplit * sh * (Dv + 2) : 0;
}

// The general form: with uv [H, Dv, vdim] every head's result is multiplied by its matrix (and gated behind it: gate [rows, H vdim]);
// for plans of one head a workgroup and whole keys (elsewhere a workgroup does not hold a finished head), vdim 64 or 128: 8 or 16
// lanes a row, up to 256 rows.  The matrix is on its way while the waves' shares are added up, the head stays fp32 in between, and a
// launch of latency is gone: 4 tokens a step, 63 steps, 16.67 -> 16.33 ms against the product in a launch of its own (runs of one
// side differ by 0.3%).
int edge_sm_attention_expand(const void* q, const void* gate, int gate_ld, const void* kp, const void* vp, const float* kb,
                             const float* vb, const int* tok_seq, const int* tok_pos, const int* seq_slot, const int* ptab,
                             int ptab_ld, void* out, int rows, int H, int G, int D, int Dv, int page, int PB, float scale,
                             int window, int pool, int f32, int plan, float* part, int kld, int vld, int chunked, float cap,
                             const float* slopes, const float* sink, int gate_elem, int keep_first, const float* rel, int rel_n,
                             int out_ld, float out_scale, const void* uv, int vdim, hipStream_t st) {
  if (rows == 0) return 0;
  const int sh = plan % 8, nsplit = plan / 8;
  if (uv && (sh != 1 || nsplit != 1 || (vdim != 64 && vdim != MAX_VDIM) || (uintptr_t)uv % 16 || out_scale != 1.f)) return -2;
  if (G <= 0 || H % G || (chunked && pool > 0) || keep_first < 0 || (rel && (rel_n < 1 || pool > 0)) || out_ld < H * (uv ? vdim : Dv) ||
      (sh != 1 && sh != 4) || nsplit < 1 || nsplit > 16 || (nsplit > 1 && !part) || D > 320 || Dv > 256 || page < 1 ||
      (page & (page - 1)) || (pool & (pool - 1)))
    return -2;
  const int nsp = (H / G + sh - 1) / sh, page_sh = __builtin_ctz(page), pool_sh = window > 0 && pool > 0 ? __builtin_ctz(pool) : -1;
  const StepArgs a{q, gate, kp, vp, kb, vb, tok_seq, tok_pos, seq_slot, ptab, out, part, slopes, sink, rel, uv, vdim, rows, gate_ld, ptab_ld, H, G, D,
                   Dv, page, page_sh, PB, window, pool_sh, nsp, nsplit, kld, vld, chunked, gate_elem, keep_first, rel_n, out_ld, scale,
                   cap, out_scale};
  if (uv) return f32 ? run_step<float, 1, true>(a, st) : run_step<bf16_t, 1, true>(a, st);
  const int r = sh == 1 ? (f32 ? run_step<float, 1, false>(a, st) : run_step<bf16_t, 1, false>(a, st))
                        : (f32 ? run_step<float, 4, false>(a, st) : run_step<bf16_t, 4, false>(a, st));
  if (r != 0 || nsplit == 1) return r;
  return edge_sm_attn_merge(part, gate, gate_ld, out, rows, H, G, Dv, nsp, nsplit, sh, gate_elem, out_ld, out_scale, f32, st);
}

// edge_sm_attention_step for plans of one head a workgroup over whole keys, rows of up to 128 numbers and plain scores, with
// edge_sm_ssd_step's token of every sequence in the same launch (rows: the sequences).  -2: nothing done
int edge_sm_attention_ssd(const void* q, const void* gate, int gate_ld, const void* kp, const void* vp, const float* kb, const float* vb,
                          const int* tok_seq, const int* tok_pos, const int* seq_slot, const int* ptab, int ptab_ld, void* out, int rows,
                          int H, int G, int D, int Dv, int page, int PB, float scale, int window, int pool, int f32, int plan, int kld,
                          int vld, const float* sink, int gate_elem, int out_ld, const void* xbc, int Cx, const void* u, int ld, int dt0,
                          const float* dt_bias, const float* A_log, const float* Dp, float* state, const int* seq_start,
                          const int* seq_off, float* y, int Hs, int P, int N, int groups, hipStream_t st) {
  if (plan != 9 || rows < 1 || G < 1 || H % G || D > 128 || Dv > 128 || page < 1 || (page & (page - 1)) || (pool & (pool - 1)) ||
      out_ld < H * Dv || ((uintptr_t)xbc | (uintptr_t)state) % 16 || Cx % 8 || groups < 1 || Hs < 2 || Hs % 2 || Hs % groups)
    return -2;
  const int pool_sh = window > 0 && pool > 0 ? __builtin_ctz(pool) : -1;
  const StepArgs a{q, gate, kp, vp, kb, vb, tok_seq, tok_pos, seq_slot, ptab, out, nullptr, nullptr, sink, nullptr, nullptr, 0, rows, gate_ld,
                   ptab_ld, H, G, D, Dv, page, __builtin_ctz(page), PB, window, pool_sh, H / G, 1, kld, vld, 0, gate_elem, 0, 0, out_ld,
                   scale, 0.f, 1.f};
  const SsdStep s{xbc, u, dt_bias, A_log, Dp, state, y, seq_slot, seq_start, seq_off, Cx, ld, dt0, Hs, groups};
#define BESIDE(TT)                                                                                                     \
  (D <= 64 && Dv <= 64 ? pool_sh >= 0 ? run_beside<TT, 2, 1, true>(a, s, N, P, st) : run_beside<TT, 2, 1, false>(a, s, N, P, st) \
                       : pool_sh >= 0 ? run_beside<TT, 4, 2, true>(a, s, N, P, st) : run_beside<TT, 4, 2, false>(a, s, N, P, st))
  return f32 ? BESIDE(float) : BESIDE(bf16_t);
#undef BESIDE
}

// plan as edge_sm_attention_step_plan says, part edge_sm_attention_step_floats numbers; the rest as edge_sm_attention's
int edge_sm_attention_step(const void* q, const void* gate, int gate_ld, const void* kp, const void* vp, const float* kb,
                           const float* vb, const int* tok_seq, const int* tok_pos, const int* seq_slot, const int* ptab,
                           int ptab_ld, void* out, int rows, int H, int G, int D, int Dv, int page, int PB, float scale,
                           int window, int pool, int f32, int plan, float* part, int kld, int vld, int chunked, float cap,
                           const float* slopes, const float* sink, int gate_elem, int keep_first, const float* rel, int rel_n,
                           int out_ld, float out_scale, hipStream_t st) {
  return edge_sm_attention_expand(q, gate, gate_ld, kp, vp, kb, vb, tok_seq, tok_pos, seq_slot, ptab, ptab_ld, out, rows, H, G, D, Dv, page,
                                  PB, scale, window, pool, f32, plan, part, kld, vld, chunked, cap, slopes, sink, gate_elem, keep_first,
                                  rel, rel_n, out_ld, out_scale, nullptr, 0, st);
}

}  // extern "C"
