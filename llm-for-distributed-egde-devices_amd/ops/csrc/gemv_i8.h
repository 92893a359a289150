// Bodies of the W8A8 / LLM.int8 decode GEMV (gemm_i8.hip says how the operands lie; decode_pair_i8.hip runs two in one
// launch).
#pragma once
#include "gemm_i8.h"
#include <type_traits>

namespace {
// int8 A fragment of k-tile k for this lane's row (ragged K: byte-wise, zero padded)
__device__ __forceinline__ v4i load_a_i8(const int8_t* __restrict__ arow_p, bool aval, int k, int kend, int akc,
                                         int K, bool k16) {
  const int kk = k * 64 + akc;
  if (aval && k < kend && kk + 16 <= K && k16) return *reinterpret_cast<const v4i*>(arow_p + kk);
  if (aval && k < kend && kk < K) {
    int8_t t[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) t[j] = (kk + j < K) ? arow_p[kk + j] : 0;
    return *reinterpret_cast<v4i*>(t);
  }
  return v4i{0, 0, 0, 0};
}

// ------------------------------------------------------------------------------------ gemv
// Weight-stationary over the rows: one workgroup owns NTW 16-column tiles for ALL M <= 16*MB
// rows, so every weight fragment is fetched once and feeds MB MFMAs.  NW = TG x KW waves: wave
// (tg, kw) holds tiles [tg*TPW, (tg+1)*TPW) and k-tiles kt = kw (mod KW); per step it keeps
// U x TPW nontemporal 1 KiB weight fragments in flight.  Sizing rule (tools/membw.hip on
// MI355X, cache-cold): 16 waves per CU-resident workgroup and >= 172 workgroups stream a
// 50-90 MB panel at 5.6-6.2 TB/s, while 4-wave workgroups or < 256 groups of few waves stall at
// 2-4 TB/s — so the launcher always runs 16 waves and sizes NTW for ~256 workgroups.
// Partial tiles are reduced across the KW k-waves through LDS (KW x NTW x MB KiB).  Everything
// the epilogue reads from global memory (weight scales, bias, per-token scales) is loaded at
// kernel start, so the tail of the kernel never waits on an HBM round trip.

#ifndef GEMV_UNROLL_FIXED
#define GEMV_UNROLL_FIXED 1
#endif

// Epilogue operands preloaded per owned fragment (EPI_OUT) or gate/up pair (GLU).
template <int OWN>
struct EpiPre {
  float s0[OWN], s1[OWN];    // sw[col] (EPI_OUT) | sw[gate col], sw[up col]
  float b0[OWN], b1[OWN];    // bias likewise (0 when absent)
};

template <int MB, int NTW, int NW, int EPI>
constexpr int epi_units() {
  return (EPI == EPI_OUT || EPI == EPI_PART || EPI == EPI_GELUQT || EPI == EPI_GELUQE) ? NTW * MB : NTW / 2 * MB;
}

template <int MB, int NTW, int NW, int EPI>
__device__ __forceinline__ EpiPre<(epi_units<MB, NTW, NW, EPI>() + NW - 1) / NW> epi_preload(
    const float* __restrict__ sw, const bf16_t* __restrict__ bias, int nt0, int NTt, int wave, int lane) {
  constexpr int UNITS = epi_units<MB, NTW, NW, EPI>(), OWN = (UNITS + NW - 1) / NW;
  EpiPre<OWN> p;
#pragma unroll
  for (int o = 0; o < OWN; ++o) {
    const int u = wave + o * NW;
    constexpr bool PAIR = EPI == EPI_GLU || EPI == EPI_GLUQ;
    const int t = PAIR ? 2 * (u / MB) : u / MB;                      // (gate) tile
    const bool ok = u < UNITS && nt0 + t + (PAIR ? 1 : 0) < NTt;
    (void)ok;                                   // out-of-range units are never stored: clamp, no branch
    const int N = NTt * 16;
    const int c0 = min((nt0 + t) * 16 + (lane & 15), N - 1), c1 = min(c0 + 16, N - 1);
    p.s0[o] = sw[c0];
    p.s1[o] = PAIR ? sw[c1] : 0.f;
    const bf16_t* bp = bias != nullptr ? bias : g_zero_bf16;   // absent bias: read a zero word
    p.b0[o] = bf2f(bp[bias != nullptr ? c0 : 0]);
    p.b1[o] = PAIR ? bf2f(bp[bias != nullptr ? c1 : 0]) : 0.f;
  }
  return p;
}

// Reduce the KW partial fragments in `red` ([KW][NTW*MB][64] v4i) and write the outputs.
// sa: per-token scales (A_TOKEN; may point to LDS), unused when SCALED.  EPI_GLUQ needs every
// wave to arrive (it holds a workgroup barrier).
template <int MB, int NTW, int NW, int KW, bool SCALED, int EPI, int OWN>
__device__ __forceinline__ void gemv_epilogue(const v4i* __restrict__ red, const float* sa, const EpiPre<OWN>& pre,
                                              void* __restrict__ outv, float* __restrict__ os, float (*gmax)[4][16],
                                              int M, int N, int NTt, int Mpad, int nt0, int wave, int lane, int ks = 0) {
  constexpr int F = NTW * MB;
  auto total = [&](int f) -> v4i {
    if constexpr (SCALED) {
      v4f s = __builtin_bit_cast(v4f, red[f * 64 + lane]);
#pragma unroll
      for (int w = 1; w < KW; ++w) s += __builtin_bit_cast(v4f, red[(w * F + f) * 64 + lane]);
      return __builtin_bit_cast(v4i, s);
    } else {
      v4i s = red[f * 64 + lane];
#pragma unroll
      for (int w = 1; w < KW; ++w) s += red[(w * F + f) * 64 + lane];
      return s;
    }
  };
  if constexpr (EPI == EPI_PART) {
    float* part = reinterpret_cast<float*>(outv) + (size_t)ks * M * N;
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const int f = wave + o * NW;
      const int t = f / MB, i = f % MB;
      if (f >= F || nt0 + t >= NTt) continue;
      const v4i tot = total(f);
      const int col = (nt0 + t) * 16 + (lane & 15);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = i * 16 + 4 * (lane >> 4) + q;
        if (row < M && col < N) {
          const float v = SCALED ? __builtin_bit_cast(v4f, tot)[q] : (float)tot[q] * sa[row];
          part[(size_t)row * N + col] = v * pre.s0[o] + (ks == 0 ? pre.b0[o] : 0.f);
        }
      }
    }
  } else if constexpr (EPI == EPI_OUT) {
    bf16_t* out = reinterpret_cast<bf16_t*>(outv);
    // os, unused by this epilogue, may carry a bf16 addend [M, N] (the other branch of a parallel-
    // residual block): out = bf16(bf16(y) + addend), the unfused bf16 add's value
    const bf16_t* add = reinterpret_cast<const bf16_t*>(os);
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const int f = wave + o * NW;
      const int t = f / MB, i = f % MB;
      if (f >= F || nt0 + t >= NTt) continue;
      const v4i tot = total(f);
      const int col = (nt0 + t) * 16 + (lane & 15);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = i * 16 + 4 * (lane >> 4) + q;
        if (row < M && col < N) {
          float v = SCALED ? __builtin_bit_cast(v4f, tot)[q] : (float)tot[q] * sa[row];
          v = v * pre.s0[o] + pre.b0[o];
          if (add != nullptr) v = bf2f(f2bf(v)) + bf2f(add[(size_t)row * N + col]);
          out[(size_t)row * N + col] = f2bf(v);
        }
      }
    }
  } else if constexpr (EPI == EPI_GELUQT || EPI == EPI_GELUQE) {
    // unit (tile t, row block i): gelu of the bf16-rounded output (the unfused GEMM's), row maxima
    // over the tile's 16 columns to LDS, one barrier, then each row's scale over the workgroup's
    // 4 tiles (= one 64-column group; N % 64 == 0) and the int8 store
    float h[OWN][4];
    bool owner[OWN];
    int tt[OWN], ii[OWN];
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const int f = wave + o * NW;
      const bool live = f < F;
      const int t = live ? f / MB : 0, i = live ? f % MB : 0;
      tt[o] = t;
      ii[o] = i;
      owner[o] = live && nt0 + t < NTt;
#pragma unroll
      for (int q = 0; q < 4; ++q) h[o][q] = 0.f;
      if (owner[o]) {
        const v4i tot = total(f);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int row = i * 16 + 4 * (lane >> 4) + q;
          const float v = (float)tot[q] * (row < M ? sa[row] : 0.f) * pre.s0[o] + pre.b0[o];
          const float a = bf2f(f2bf(v));
          float g;
          if constexpr (EPI == EPI_GELUQT) g = 0.5f * a * (1.f + tanhf(0.7978845608028654f * (a + 0.044715f * a * a * a)));
          else g = 0.5f * a * (1.f + erff(a * 0.7071067811865476f));
          h[o][q] = bf2f(f2bf(g));            // the unfused activation output is bf16
          float m = fabsf(h[o][q]);
#pragma unroll
          for (int d = 1; d < 16; d <<= 1) m = xor_max(m, d);
          if ((lane & 15) == 0) gmax[i][t][4 * (lane >> 4) + q] = m;
        }
      }
    }
    __syncthreads();
    int8_t* hq = reinterpret_cast<int8_t*>(outv);
    const int grp = nt0 / 4;
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      if (!owner[o]) continue;
      const int t = tt[o], i = ii[o];
      const int col = (nt0 + t) * 16 + (lane & 15);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int rr = 4 * (lane >> 4) + q, row = i * 16 + rr;
        const float amax = fmaxf(fmaxf(fmaxf(gmax[i][0][rr], gmax[i][1][rr]), fmaxf(gmax[i][2][rr], gmax[i][3][rr])), 1e-8f);
        if (row < M) hq[(size_t)row * N + col] = quant_i8(h[o][q], 127.f / amax);
        if (t == 0 && (lane & 15) == 0 && row < Mpad) os[(size_t)grp * Mpad + row] = row < M ? amax / 127.f : 0.f;
      }
    }
  } else {
    // pair p = (gate tile 2p, up tile 2p+1) -> feature (nt0/2 + p) * 16 + (lane & 15); a wave owns
    // pairs wave, wave + NW, ...  EPI_GLUQ: every owned pair's row maxima reach LDS before the
    // single barrier, then each 64-feature group (4 pairs) is quantised with one scale per row
    const int Fo = N / 2;
    constexpr int NP = NTW / 2 * MB;
    float h[OWN][4];
    bool owner[OWN];
    int pp[OWN], ii[OWN];
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const int pf = wave + o * NW;
      const bool live = pf < NP;
      const int p = live ? pf / MB : 0, i = live ? pf % MB : 0;
      pp[o] = p;
      ii[o] = i;
      owner[o] = live && nt0 + 2 * p + 1 < NTt;
      const int feat = (nt0 / 2 + p) * 16 + (lane & 15);
#pragma unroll
      for (int q = 0; q < 4; ++q) h[o][q] = 0.f;
      if (owner[o]) {
        const v4i g4 = total((2 * p) * MB + i), u4 = total((2 * p + 1) * MB + i);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int row = i * 16 + 4 * (lane >> 4) + q;
          const float s_a = row < M ? sa[row] : 0.f;
          float g = (float)g4[q] * s_a * pre.s0[o] + pre.b0[o];
          float u = (float)u4[q] * s_a * pre.s1[o] + pre.b1[o];
          g = bf2f(f2bf(g));                // the unfused GEMM output is bf16
          u = bf2f(f2bf(u));
          h[o][q] = g / (1.f + __expf(-g)) * u;
          if constexpr (EPI == EPI_GLU)
            if (row < M) reinterpret_cast<bf16_t*>(outv)[(size_t)row * Fo + feat] = f2bf(h[o][q]);
        }
        if constexpr (EPI == EPI_GLUQ) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float m = fabsf(h[o][q]);
#pragma unroll
            for (int d = 1; d < 16; d <<= 1) m = xor_max(m, d);
            if ((lane & 15) == 0) gmax[i][p][4 * (lane >> 4) + q] = m;
          }
        }
      }
    }
    if constexpr (EPI == EPI_GLUQ) {
      __syncthreads();
      int8_t* hq = reinterpret_cast<int8_t*>(outv);
      const int grp = nt0 / 8;
#pragma unroll
      for (int o = 0; o < OWN; ++o) {
        if (!owner[o]) continue;
        const int p = pp[o], i = ii[o];
        const int feat = (nt0 / 2 + p) * 16 + (lane & 15);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int rr = 4 * (lane >> 4) + q, row = i * 16 + rr;
          const float amax = fmaxf(fmaxf(fmaxf(gmax[i][0][rr], gmax[i][1][rr]), fmaxf(gmax[i][2][rr], gmax[i][3][rr])), 1e-8f);
          if (row < M) hq[(size_t)row * Fo + feat] = quant_i8(h[o][q], 127.f / amax);
          if (p == 0 && (lane & 15) == 0 && row < Mpad) os[(size_t)grp * Mpad + row] = row < M ? amax / 127.f : 0.f;
        }
      }
    }
  }
}

// Decode RMSNorm prologue (NRM > 0, M <= 4 rows): the activation rows are not an input but the
// RMSNorm of the previous split-K projection's fp32 partial slices plus the residual, quantised
// per token (rowwise.hip norm_kernel<PART, HAS_RES, QUANT> moved into the consumer: one launch
// fewer per norm, and the first weight steps are in flight while the rows are normalised).  The
// 1024 threads form four 256-thread groups, one row each; a group runs the norm kernel's
// exact element layout and reduction order (NCH chunks of 8 per thread), so the int8 rows and
// their scales are bit-identical.  Workgroup 0 writes the new residual rows.
struct NormIn {
  const float* part;      // [S][M][K] fp32 slices
  const bf16_t* res;      // [M][K] residual in
  const bf16_t* gamma;    // [K]
  bf16_t* res_out;        // [M][K] residual out (must not alias res: other workgroups still read it)
  float eps;
  int S;
  const bf16_t* x = nullptr;      // LN (NRM >= 64): [M][K] bf16 input rows, LayerNorm of x + res
  const bf16_t* beta = nullptr;   // LN: [K] (may be null)
  float thr = 0.f;                // LLM.int8 (NRM >= 128): outlier threshold on |x|
  const int8_t* wt = nullptr;     // LLM.int8: int8 W^T [K][N] (an outlier column is one row)
  const float* scb = nullptr;     // LLM.int8: per-row weight absmax SCB [N]
  const bf16_t* add = nullptr;    // LLM.int8: a row added to the (bf16) result (may be null)
  bf16_t* y_out = nullptr;        // LLM.int8 of a normed row: the normalised row too (may be null), ...
  const bf16_t* gamma2 = nullptr; // ... under these weights (a GPT-NeoX block's second norm of the same row)
  const bf16_t* beta2 = nullptr;
  const bf16_t* x2 = nullptr;     // LLM.int8 LN: the block's other branch, x + x2 rounded before the residual joins
  int act = 0;                    // LLM.int8, activation chosen per launch: 1 gelu tanh, 2 gelu erf
};
constexpr int NRM_ROWS = 4;
constexpr int L8_COUNT = 32;      // where l8_prologue leaves the outlier count (after every wave's total of every chunk)
constexpr int L8_CMAX = 256;      // LLM.int8 outlier columns per row held in LDS (llmint8.hip's cap)

// The prologue's global loads (slices, residual, gamma) are issued by norm_load BEFORE the
// weight stream and consumed by norm_prologue after it is issued: a wave's loads retire in issue
// order, so prologue loads queued behind the weights would wait for the whole stream and leave
// the norm, the MFMAs and the epilogue as a tail after the last weight byte.
template <int NCH, int SMAX>
struct NormRegs {
  uint4 rv[NCH];
  float4 pv[NCH][SMAX][2];                                // S <= SMAX slices (register budget)
  uint4 gv[NCH];
};

template <int NCH, int SMAX>
__device__ __forceinline__ void norm_load_now(const NormIn& na, int H, int M, NormRegs<NCH, SMAX>& r) {
  const int t = threadIdx.x & 255, row = threadIdx.x >> 8;
  if (row < M) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int e = min((c * 256 + t) * 8, H - 8);
      r.rv[c] = na.res != nullptr ? *reinterpret_cast<const uint4*>(na.res + (size_t)row * H + e)
                                  : uint4{0u, 0u, 0u, 0u};                 // no residual (a stage's first norm)
#pragma unroll
      for (int k = 0; k < SMAX; ++k)
        if (k < na.S) {
          const float4* p = reinterpret_cast<const float4*>(na.part + ((size_t)k * M + row) * H + e);
          r.pv[c][k][0] = p[0];
          r.pv[c][k][1] = p[1];
        }
      if constexpr (NCH * SMAX <= 4) r.gv[c] = *reinterpret_cast<const uint4*>(na.gamma + e);
    }
  }
}

// hoisted while NCH x SMAX <= 4 (K = 4096 with up to 2 slices, K = 2048 with up to 4); K = 4096
// with 3-4 slices would spill, so those load in the prologue
template <int NCH, int SMAX>
__device__ __forceinline__ void norm_load(const NormIn& na, int H, int M, NormRegs<NCH, SMAX>& r) {
  if constexpr (NCH * SMAX <= 4) {
    norm_load_now(na, H, M, r);
    asm volatile("" ::: "memory");                        // these loads issue before the weights
  }
}

template <int NCH, int SMAX>
__device__ __forceinline__ void norm_prologue(const NormIn& na, bool wg0, int H, int M, int8_t* aq, float* nsa, float* nred,
                                              const NormRegs<NCH, SMAX>& held) {
  const int t = threadIdx.x & 255, g = threadIdx.x >> 8, w = t >> 6;
  {                                                       // one pass: M <= NRM_ROWS = 4
    const int row = g;
    const bool act = row < M;
    float v[NCH][8];
    float ss = 0.f, amax = 0.f;
    if (act) {
      NormRegs<NCH, SMAX> late;                           // 3-4 slices: loaded here, as late as possible
      if constexpr (NCH * SMAX > 4) norm_load_now(na, H, M, late);
      const NormRegs<NCH, SMAX>& regs = NCH * SMAX > 4 ? late : held;
      const uint4* rv = regs.rv;
      const auto& pv = regs.pv;
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const int e = (c * 256 + t) * 8;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[c][j] = 0.f;
#pragma unroll
        for (int k = 0; k < SMAX; ++k)
          if (k < na.S) {
            const float4 p0 = pv[c][k][0], p1 = pv[c][k][1];
            v[c][0] += p0.x; v[c][1] += p0.y; v[c][2] += p0.z; v[c][3] += p0.w;
            v[c][4] += p1.x; v[c][5] += p1.y; v[c][6] += p1.z; v[c][7] += p1.w;
          }
        if (e < H) {
          unpack8(pack8(v[c]), v[c]);                       // the projection's bf16 output
          float r[8];
          unpack8(rv[c], r);
#pragma unroll
          for (int j = 0; j < 8; ++j) v[c][j] += r[j];
          const uint4 u = pack8(v[c]);                      // residual stream in bf16
          if (wg0) *reinterpret_cast<uint4*>(na.res_out + (size_t)row * H + e) = u;
          unpack8(u, v[c]);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[c][j] = 0.f;
        }
      }
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const int e = (c * 256 + t) * 8;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float d = (e < H) ? v[c][j] - 0.f : 0.f;
          ss += d * d;
        }
      }
      ss = wave_sum(ss);
      if ((t & 63) == 0) nred[4 * g + w] = ss;
    }
    __syncthreads();
    const float* gr = nred + 4 * g;
    const float rstd = rsqrtf((((0.f + gr[0]) + gr[1]) + gr[2] + gr[3]) / (float)H + na.eps);
    if (act) {
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const int e = (c * 256 + t) * 8;
        if (e < H) {
          float wf[8];
          unpack8(NCH * SMAX <= 4 ? held.gv[c] : *reinterpret_cast<const uint4*>(na.gamma + min(e, H - 8)), wf);
#pragma unroll
          for (int j = 0; j < 8; ++j) v[c][j] = (v[c][j] - 0.f) * rstd * wf[j];
        }
      }
#pragma unroll
      for (int c = 0; c < NCH; ++c)
#pragma unroll
        for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[c][j]));
      amax = wave_max(amax);
      if ((t & 63) == 0) nred[16 + 4 * g + w] = amax;     // (each reduction has words of its own: one barrier each)
    }
    __syncthreads();
    float gm = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) gm = fmaxf(gm, gr[16 + i]);
    gm = fmaxf(gm, 1e-8f);
    const float inv = 127.f / gm;
    if (act && t == 0) nsa[row] = gm / 127.f;
    if (act) {
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const int e = (c * 256 + t) * 8;
        if (e < H) {
          uint32_t lo = 0, hi = 0;
#pragma unroll
          for (int j = 0; j < 4; ++j) lo |= ((uint32_t)(uint8_t)quant_i8(v[c][j], inv)) << (8 * j);
#pragma unroll
          for (int j = 0; j < 4; ++j) hi |= ((uint32_t)(uint8_t)quant_i8(v[c][4 + j], inv)) << (8 * j);
          *reinterpret_cast<uint2*>(aq + (size_t)row * H + e) = make_uint2(lo, hi);
        }
      }
    }
    __syncthreads();                                      // aq complete
  }
}

// LayerNorm prologue (NRM >= 64: the parallel-residual decoders, GPT-NeoX / Phi): the LayerNorm of
// the bf16 rows x + residual, int8 per token, with norm_kernel<NCH, !RMS, HAS_RES, QUANT, !PART>'s
// element layout, reduction order and roundings (bit-identical rows and scales).  Its loads issue
// before the weight stream (ln_load), like the RMS form's.
template <int NCH>
struct LnRegs {
  uint4 xv[NCH], rv[NCH], gv[NCH], bv[NCH];
};

template <int NCH>
__device__ __forceinline__ void ln_load(const NormIn& na, int H, int M, LnRegs<NCH>& r) {
  const int t = threadIdx.x & 255, row = threadIdx.x >> 8;
  if (row < M) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int e = min((c * 256 + t) * 8, H - 8);
      r.xv[c] = *reinterpret_cast<const uint4*>(na.x + (size_t)row * H + e);
      r.rv[c] = na.res != nullptr ? *reinterpret_cast<const uint4*>(na.res + (size_t)row * H + e) : uint4{0u, 0u, 0u, 0u};
      r.gv[c] = *reinterpret_cast<const uint4*>(na.gamma + e);
      r.bv[c] = na.beta != nullptr ? *reinterpret_cast<const uint4*>(na.beta + e) : uint4{0u, 0u, 0u, 0u};
    }
  }
  asm volatile("" ::: "memory");                          // these loads issue before the weights
}

template <int NCH>
__device__ __forceinline__ void ln_prologue(const NormIn& na, bool wg0, int H, int M, int8_t* aq, float* nsa, float* nred,
                                            const LnRegs<NCH>& r) {
  const int t = threadIdx.x & 255, row = threadIdx.x >> 8, w = t >> 6;
  const bool act = row < M;
  float v[NCH][8];
  float sm = 0.f;
  if (act) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int e = (c * 256 + t) * 8;
      if (e < H) {
        unpack8(r.xv[c], v[c]);
        float rr[8];
        unpack8(r.rv[c], rr);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[c][j] += rr[j];
        const uint4 u = pack8(v[c]);                          // residual stream in bf16
        if (wg0) *reinterpret_cast<uint4*>(na.res_out + (size_t)row * H + e) = u;
        unpack8(u, v[c]);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[c][j] = 0.f;
      }
    }
#pragma unroll
    for (int c = 0; c < NCH; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) sm += v[c][j];
    sm = wave_sum(sm);
    if ((t & 63) == 0) nred[4 * row + w] = sm;
  }
  __syncthreads();
  const float* gr = nred + 4 * (row < NRM_ROWS ? row : 0);
  const float mean = ((((0.f + gr[0]) + gr[1]) + gr[2]) + gr[3]) / (float)H;
  float ss = 0.f;
  if (act) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int e = (c * 256 + t) * 8;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float d = (e < H) ? v[c][j] - mean : 0.f;
        ss += d * d;
      }
    }
    ss = wave_sum(ss);
    if ((t & 63) == 0) nred[16 + 4 * row + w] = ss;         // (each reduction has words of its own: one barrier each)
  }
  __syncthreads();
  const float rstd = rsqrtf(((((0.f + gr[16]) + gr[17]) + gr[18]) + gr[19]) / (float)H + na.eps);
  float amax = 0.f;
  if (act) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int e = (c * 256 + t) * 8;
      if (e < H) {
        float wf[8], bf[8];
        unpack8(r.gv[c], wf);
        unpack8(r.bv[c], bf);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[c][j] = (v[c][j] - mean) * rstd * wf[j] + bf[j];
      }
    }
#pragma unroll
    for (int c = 0; c < NCH; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[c][j]));
    amax = wave_max(amax);
    if ((t & 63) == 0) nred[32 + 4 * row + w] = amax;
  }
  __syncthreads();
  float gm = -INFINITY;
#pragma unroll
  for (int i = 0; i < 4; ++i) gm = fmaxf(gm, gr[32 + i]);
  gm = fmaxf(gm, 1e-8f);
  const float inv = 127.f / gm;
  if (act && t == 0) nsa[row] = gm / 127.f;
  if (act) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int e = (c * 256 + t) * 8;
      if (e < H) {
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) lo |= ((uint32_t)(uint8_t)quant_i8(v[c][j], inv)) << (8 * j);
#pragma unroll
        for (int j = 0; j < 4; ++j) hi |= ((uint32_t)(uint8_t)quant_i8(v[c][4 + j], inv)) << (8 * j);
        *reinterpret_cast<uint2*>(aq + (size_t)row * H + e) = make_uint2(lo, hi);
      }
    }
  }
  __syncthreads();                                        // aq complete
}

// LLM.int8 prologue (NRM >= 128, one row): llmint8.hip's decode preparation inside the GEMV, so a
// batch-1 LLM.int8 projection is one launch instead of three (prep, GEMV, outlier add).  Columns with |x| > thr
// are ranked in column order by a block prefix sum per chunk, the first L8_CMAX go to LDS (index,
// value); the per-token absmax over the other columns, then int8 x with the taken columns zeroed.
// The epilogue adds sum_j x[c_j] W^T[c_j][n] SCB[n] / 127 to the rounded output, in llmint8.hip's
// order and roundings: the output bits equal prep + GEMV + outlier kernel.
// SRC 1 / 2 (NRM = 192 + 8 NCH + SRC): the row is first the RMSNorm / LayerNorm of x + residual
// (norm_kernel's HAS_RES path, rounded to bf16 as its output), so an LLM.int8 layer's norm is no
// launch of its own either; workgroup 0 writes the new residual row and, when y_out is set, the
// normalised row (for a second consumer).
// Who holds the row: behind a norm threads 0-255 in norm_prologue's layout, column (c 256 + t) 8 + j (its sums' order); a row as
// it is (ranks and maxima have no order) all threads of the workgroup, 8 columns a chunk.  Every wave of the workgroup waits for
// this chain, so the counts and the maximum meet at one barrier: the maximum leaves out every outlier, and only a row of more than
// L8_CMAX of them takes it again over those past the cap.  us in a graph, one row, 256 threads and three barriers /
// now: 2560 x 10240 beside 2560 x 2560 10.5 / 8.1, 10240 x 2560 beside attention 9.5 / 8.3, 7680 x 2560 behind LayerNorm 8.3 / 7.6.
template <int NCH, int SRC, int NW>
constexpr int l8_chunks() { return SRC ? NCH : (NCH * 256 + NW * 64 - 1) / (NW * 64); }

template <int NC, int SRC>
struct L8Regs {
  uint4 xv[NC];
  uint4 rv[SRC ? NC : 1], gv[SRC ? NC : 1], bv[SRC == 2 ? NC : 1];
  uint4 x2v[SRC == 2 ? NC : 1], g2v[SRC == 2 ? NC : 1], b2v[SRC == 2 ? NC : 1];
};

template <int NC, int SRC, int NW>
__device__ __forceinline__ void l8_load(const NormIn& na, bool wg0, int H, L8Regs<NC, SRC>& r) {
  constexpr int NTH = SRC ? 256 : NW * 64;
  const int t = threadIdx.x;
  if (SRC == 0 || t < 256) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int e = min((c * NTH + t) * 8, H - 8);
      r.xv[c] = *reinterpret_cast<const uint4*>(na.x + e);
      if constexpr (SRC > 0) {
        r.rv[c] = na.res != nullptr ? *reinterpret_cast<const uint4*>(na.res + e) : uint4{0u, 0u, 0u, 0u};
        r.gv[c] = *reinterpret_cast<const uint4*>(na.gamma + e);
      }
      if constexpr (SRC == 2) {
        const bool two = wg0 && na.gamma2 != nullptr;
        r.bv[c] = na.beta != nullptr ? *reinterpret_cast<const uint4*>(na.beta + e) : uint4{0u, 0u, 0u, 0u};
        r.x2v[c] = na.x2 != nullptr ? *reinterpret_cast<const uint4*>(na.x2 + e) : uint4{0u, 0u, 0u, 0u};
        r.g2v[c] = two ? *reinterpret_cast<const uint4*>(na.gamma2 + e) : uint4{0u, 0u, 0u, 0u};
        r.b2v[c] = two && na.beta2 != nullptr ? *reinterpret_cast<const uint4*>(na.beta2 + e) : uint4{0u, 0u, 0u, 0u};
      }
    }
  }
  asm volatile("" ::: "memory");                          // these loads issue before the weights
}

template <int NC, int SRC, int NW>
__device__ __forceinline__ void l8_prologue(const NormIn& na, bool wg0, int H, int8_t* aq, float* nsa, float* nred, int* cols,
                                            float* xo, int* scr, const L8Regs<NC, SRC>& r, bf16_t* y_out) {
  constexpr int NTH = SRC ? 256 : NW * 64, WV = NTH / 64;   // threads and waves that hold the row
  static_assert(NC * WV <= L8_COUNT, "wave totals");
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const bool act = SRC == 0 || w < WV;
  float v[NC][8];
  if (act) {
#pragma unroll
    for (int c = 0; c < NC; ++c) unpack8(r.xv[c], v[c]);
  }
  if constexpr (SRC > 0) {
    float sm = 0.f;
    if (act) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int e = (c * 256 + t) * 8;
        if (e < H) {
          float rr[8];
          if constexpr (SRC == 2) {
            if (na.x2 != nullptr) {
              unpack8(r.x2v[c], rr);
#pragma unroll
              for (int j = 0; j < 8; ++j) v[c][j] += rr[j];
              unpack8(pack8(v[c]), v[c]);                   // the sum of the branches is a bf16 row
            }
          }
          unpack8(r.rv[c], rr);
#pragma unroll
          for (int j = 0; j < 8; ++j) v[c][j] += rr[j];
          const uint4 u = pack8(v[c]);                      // residual stream in bf16
          if (wg0) *reinterpret_cast<uint4*>(na.res_out + e) = u;
          unpack8(u, v[c]);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[c][j] = 0.f;
        }
      }
      if constexpr (SRC == 2) {
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int j = 0; j < 8; ++j) sm += v[c][j];
        sm = wave_sum(sm);
        if (lane == 0) nred[w] = sm;
      }
    }
    float mean = 0.f;
    if constexpr (SRC == 2) {
      __syncthreads();
      mean = ((((0.f + nred[0]) + nred[1]) + nred[2]) + nred[3]) / (float)H;
    }
    float ss = 0.f;
    if (act) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int e = (c * 256 + t) * 8;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float d = (e < H) ? v[c][j] - mean : 0.f;
          ss += d * d;
        }
      }
      ss = wave_sum(ss);
      if (lane == 0) nred[16 + w] = ss;                     // (each reduction has words of its own: one barrier each)
    }
    __syncthreads();
    const float rstd = rsqrtf(((((0.f + nred[16]) + nred[17]) + nred[18]) + nred[19]) / (float)H + na.eps);
    if (act) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int e = (c * 256 + t) * 8;
        if (e < H) {
          float wf[8], bf[8], n1[8];
          unpack8(r.gv[c], wf);
          if constexpr (SRC == 2) unpack8(r.bv[c], bf);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            float tv = (v[c][j] - mean) * rstd * wf[j];
            if constexpr (SRC == 2) tv += bf[j];
            n1[j] = tv;
          }
          const uint4 u = pack8(n1);                        // the norm's bf16 output row
          if (y_out != nullptr && wg0) {
            if (SRC == 2 && na.gamma2 != nullptr) {
              unpack8(r.g2v[SRC == 2 ? c : 0], wf);
              unpack8(r.b2v[SRC == 2 ? c : 0], bf);
#pragma unroll
              for (int j = 0; j < 8; ++j) n1[j] = (v[c][j] - mean) * rstd * wf[j] + bf[j];
              *reinterpret_cast<uint4*>(y_out + e) = pack8(n1);
            } else {
              *reinterpret_cast<uint4*>(y_out + e) = u;
            }
          }
          unpack8(u, v[c]);
        }
      }
    }
  }
  // outliers per thread and chunk, ranked in column order, and the largest other number
  uint32_t take[NC];
  int incl[NC];
  float am = 0.f;
  if (act) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      uint32_t bits = 0;
      if ((c * NTH + t) * 8 < H) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float a = fabsf(v[c][j]);
          const bool out = a > na.thr;
          bits |= (out ? 1u : 0u) << j;
          am = fmaxf(am, out ? 0.f : a);
        }
      }
      take[c] = bits;
      incl[c] = __popc(bits);
      if (__any(bits != 0)) {                               // outliers are few: most waves have none to rank
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int tt = __shfl_up(incl[c], o, 64);
          if (lane >= o) incl[c] += tt;
        }
      }
      if (lane == 63) scr[c * WV + w] = incl[c];
    }
    am = wave_max(am);
    if (lane == 0) nred[32 + w] = am;
  }
  __syncthreads();
  int count = 0;
#pragma unroll
  for (int i = 0; i < NC * WV; ++i) count += scr[i];
  if (t == 0) scr[L8_COUNT] = min(count, L8_CMAX);
  if (act && count > 0) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (take[c]) {
        int slot = incl[c] - __popc(take[c]);
        for (int i = 0; i < c * WV + w; ++i) slot += scr[i];
        uint32_t tk = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {                       // (static indices: v stays in registers)
          if ((take[c] >> j) & 1u) {
            if (slot < L8_CMAX) {
              cols[slot] = (c * NTH + t) * 8 + j;
              xo[slot] = v[c][j];
              tk |= 1u << j;
            }
            ++slot;
          }
        }
        take[c] = tk;
      }
  }
  float rm = 0.f;
#pragma unroll
  for (int i = 0; i < WV; ++i) rm = fmaxf(rm, nred[32 + i]);
  if (count > L8_CMAX) {                                    // workgroup-uniform: outliers past the cap are numbers like any
    __syncthreads();
    if (act) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if ((c * NTH + t) * 8 < H) {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (!((take[c] >> j) & 1u)) am = fmaxf(am, fabsf(v[c][j]));
        }
      am = wave_max(am);
      if (lane == 0) nred[32 + w] = am;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < WV; ++i) rm = fmaxf(rm, nred[32 + i]);
  }
  const float gm = fmaxf(rm, 1e-8f);
  if (t == 0) nsa[0] = gm / 127.f;
  const float inv = 127.f / gm;
  if (act) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int e = (c * NTH + t) * 8;
      if (e < H) {
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          lo |= ((uint32_t)(uint8_t)((take[c] >> j) & 1u ? 0 : quant_i8(v[c][j], inv))) << (8 * j);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          hi |= ((uint32_t)(uint8_t)((take[c] >> (4 + j)) & 1u ? 0 : quant_i8(v[c][4 + j], inv))) << (8 * j);
        *reinterpret_cast<uint2*>(aq + e) = make_uint2(lo, hi);
      }
    }
  }
  __syncthreads();                                        // aq, cols, xo, the count complete
}

// One workgroup (bid) of the GEMV.
template <int MB, int NTW, int TG, int KW, int U, int AMODE, int EPI, int NRM>
__device__ __forceinline__ void w8a8_gemv_body(int bid, const int8_t* __restrict__ A, const float* __restrict__ sa,
                                               const int8_t* __restrict__ Wp, const float* __restrict__ sw,
                                               const bf16_t* __restrict__ bias, void* __restrict__ outv,
                                               float* __restrict__ os, int M, int N, int K, int KT, int NTt, int Mpad, int S,
                                               const NormIn& na) {
  constexpr int NW = TG * KW, TPW = NTW / TG;
  static_assert(NTW % TG == 0, "tiles split evenly over tile groups");
  static_assert(NRM == 0 || (MB == 1 && AMODE == A_TOKEN && EPI != EPI_PART && (NW == 16 || (NRM >= 128 && NW >= 4))), "norm prologue: batch 1");
  // NRM: the int8 activation row lives in LDS (norm_prologue), its per-token scale in nsa[0]
  // NRM = 8 * NCH + SMAX (norm_prologue<NCH, SMAX>)
  constexpr bool L8_N = NRM >= 128;                          // LLM.int8 preparation (+ 128) ...
  constexpr int L8SRC_N = NRM >= 192 ? NRM % 8 : 0;          // ... of a normed row (+ 192 + 1 RMS / 2 LN
  constexpr int L8S_N = L8SRC_N & 3;                         //     (+ 4: SwiGLU of [gate | up] tiles)
  constexpr bool L8G_N = (L8SRC_N & 4) != 0;
  constexpr int L8ACT_N = NRM >= 256 ? (NRM - 256) / 64 + 1 : 0;   // + 256 (+ 64): gelu tanh (erf) epilogue; + 128: na.act
  constexpr bool LN_N = NRM >= 64 && !L8_N;                  // LayerNorm of bf16 rows (+ 64)
  constexpr int NCH_N = (NRM % 64) / 8, SMAX_N = LN_N || L8_N ? 1 : NRM % 8;
  static_assert(!L8_N || (EPI == EPI_OUT && MB == 1), "LLM.int8 prologue: one row, plain output");
  __shared__ int l8_cols[L8_N ? L8_CMAX : 1];
  __shared__ float l8_xo[L8_N ? L8_CMAX : 1];
  __shared__ int l8_scr[L8_COUNT + 1];
  __shared__ int8_t aq_l[NRM > 0 ? (L8_N ? 1 : NRM_ROWS) * NCH_N * 2048 : 16];
  __shared__ float nsa[16], nred[48];
  constexpr bool GELUQ = EPI == EPI_GELUQT || EPI == EPI_GELUQE;
  static_assert(EPI == EPI_OUT || EPI == EPI_PART || (AMODE == A_TOKEN && (GELUQ || TPW % 2 == 0)),
                "GLU: gate/up pairs per wave, per-token A");
  static_assert(EPI != EPI_GLUQ || NTW == 8, "quantising GLU: 64 features per workgroup");
  static_assert(!GELUQ || NTW == 4, "quantising GELU: 64 columns per workgroup");
  // LDS reduction buffer: one partial set per k-wave, or per pair of k-waves when that would
  // exceed 128 KiB (the upper half adds into the lower half first)
  constexpr int KR = KW * NTW * MB * 1024 <= 131072 ? KW : KW / 2;
  static_assert(KR * NTW * MB * 1024 <= 131072 && KW % KR == 0 && KW / KR <= 2, "LDS reduction budget");
  constexpr bool SCALED = AMODE == A_GROUP;
  __shared__ v4i red[KR][NTW * MB][64];
  __shared__ float gmax[MB][4][16];
  // EPI_PART (split-K): workgroup (group, s) reduces k-tiles [KT*s/S, KT*(s+1)/S) of its tiles and
  // writes fp32 partial sums part[s][M][N]; the consumer (norm kernel) adds the S slices in order
  const int grp = EPI == EPI_PART ? bid / S : bid;
  const int ks = EPI == EPI_PART ? bid % S : 0;
  const int kbeg = EPI == EPI_PART ? (int)((int64_t)KT * ks / S) : 0;
  const int kend = EPI == EPI_PART ? (int)((int64_t)KT * (ks + 1) / S) : KT;
  // L8G (SwiGLU, natural [gate | up] rows): the workgroup's 2 tiles are gate tile grp and up tile grp + NTt / 2
  const int nt0 = L8G_N ? grp : grp * NTW;
  static_assert(!L8G_N || (NTW == 2 && TG == 1), "LLM.int8 SwiGLU: one gate + one up tile per workgroup");
  // wave index in an SGPR: every k-loop guard below is then a scalar branch (an MFMA must never
  // sit under an EXEC-masked branch — it ignores EXEC and would add a clamped duplicate k-tile)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tg = wave / KW, kw = wave % KW, t0 = tg * TPW;
  const int akc = 16 * (lane >> 4);

  const v4i* wp[TPW];
#pragma unroll
  for (int j = 0; j < TPW; ++j) {
    const int nt = L8G_N ? (j == 0 ? nt0 : nt0 + NTt / 2) : min(nt0 + t0 + j, NTt - 1);
    // (the offset stays a scalar product: added to the lane's address in one go it is three vector multiplications in front of the first
    // weights; one row behind RMSNorm, us, so / scalar: 12288 x 4096 11.30 / 11.12, 22016 x 4096 18.99 / 18.68)
    size_t panel = (size_t)nt * KT * 1024;
    asm("" : "+s"(panel));
    wp[j] = reinterpret_cast<const v4i*>(Wp + panel) + lane;
  }
  const int8_t* ap[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
    ap[i] = (NRM > 0 ? aq_l : A) + (size_t)min(i * 16 + (lane & 15), M - 1) * K;
  const bool kfull = NRM > 0 || (K & 63) == 0;
  const auto pre = epi_preload<MB, NTW, NW, EPI>(sw, bias, nt0, NTt, wave, lane);
  v4i acc[TPW][MB];
  v4f accf[TPW][MB];
#pragma unroll
  for (int j = 0; j < TPW; ++j)
#pragma unroll
    for (int i = 0; i < MB; ++i) { acc[j][i] = v4i{0, 0, 0, 0}; accf[j][i] = v4f{0.f, 0.f, 0.f, 0.f}; }

  struct Step {
    v4i b[U][TPW];
    v4i a[U][MB];
    v4f sg[U][MB];
  };
  // one step = U k-tiles: weight fragments (nontemporal), activation fragments and (SCALED)
  // per-group scales; clamped addresses, no branches
  auto issue_w = [&](Step& st, int kbase) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < TPW; ++j)
        st.b[u][j] = __builtin_nontemporal_load(wp[j] + (size_t)min(kbase + u * KW, kend - 1) * 64);
  };
  auto issue_a = [&](Step& st, int kbase) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(kbase + u * KW, kend - 1);
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        if (kfull) st.a[u][i] = *reinterpret_cast<const v4i*>(ap[i] + k * 64 + akc);
        else st.a[u][i] = load_a_i8(ap[i], true, k, KT, akc, K, (K & 15) == 0);
        if constexpr (SCALED)
          st.sg[u][i] = *reinterpret_cast<const v4f*>(sa + (size_t)k * Mpad + min(i * 16, Mpad - 16) + 4 * (lane >> 4));
      }
    }
  };
  auto issue = [&](Step& st, int kbase) {
    issue_w(st, kbase);
    issue_a(st, kbase);
  };
  // NRM: the first step's weight loads go out before the norm prologue; its activations after
  NormRegs<(NRM > 0 && !LN_N && !L8_N ? NCH_N : 1), (NRM > 0 && !LN_N && !L8_N ? SMAX_N : 1)> nr;
  LnRegs<(LN_N ? NCH_N : 1)> lr;
  constexpr int L8C_N = L8_N ? l8_chunks<NCH_N, L8S_N, NW>() : 1;
  L8Regs<L8C_N, L8S_N> l8r;
  auto nload = [&]() {
    if constexpr (L8_N) l8_load<L8C_N, L8S_N, NW>(na, bid == 0, K, l8r);
    else if constexpr (LN_N) ln_load(na, K, M, lr);
    else norm_load(na, K, M, nr);
  };
  auto nprologue = [&]() {
    if constexpr (L8_N) l8_prologue<L8C_N, L8S_N, NW>(na, bid == 0, K, aq_l, nsa, nred, l8_cols, l8_xo, l8_scr, l8r, na.y_out);
    else if constexpr (LN_N) ln_prologue(na, bid == 0, K, M, aq_l, nsa, nred, lr);
    else norm_prologue(na, bid == 0, K, M, aq_l, nsa, nred, nr);
  };
  auto first = [&](Step& st, int kbase) {
    if constexpr (NRM > 0) {
      nload();
      issue_w(st, kbase);
      nprologue();
      issue_a(st, kbase);
    } else {
      issue(st, kbase);
    }
  };
  auto compute = [&](const Step& st, int kbase) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (kbase + u * KW < kend) {                       // wave-uniform tail guard
#pragma unroll
        for (int j = 0; j < TPW; ++j)
#pragma unroll
          for (int i = 0; i < MB; ++i) {
            if constexpr (SCALED) fold(accf[j][i], mfma_i8(st.a[u][i], st.b[u][j], v4i{0, 0, 0, 0}), st.sg[u][i]);
            else acc[j][i] = mfma_i8(st.a[u][i], st.b[u][j], acc[j][i]);
          }
      }
    }
  };
  // one step of U k-tiles per iteration: all its loads in flight, then its MFMAs.  The k range
  // lengths of the decode shapes (64, 32, 16 k-tiles) get a compile-time trip count, fully
  // unrolled, so the scheduler can hoist the next steps' loads above this step's MFMAs (a wave's
  // time is otherwise about one memory latency per step); other lengths take the runtime loop.
  auto fixed = [&](auto nk) {
    constexpr int NK = decltype(nk)::value, STEPS = (NK + KW * U - 1) / (KW * U);
    Step st[STEPS];
    if constexpr (NRM > 0 && STEPS <= 2 && NCH_N * SMAX_N <= 4 && (!L8_N || NCH_N <= (L8SRC_N ? 1 : 2))) {
      // batch-1 norm prologue: every step's weights (at most 2) in flight across it (K = 4096 with
      // 4 slices keeps one step: its prologue registers would spill)
      nload();
#pragma unroll
      for (int i = 0; i < STEPS; ++i) issue_w(st[i], kbeg + kw + i * KW * U);
      nprologue();
#pragma unroll
      for (int i = 0; i < STEPS; ++i) {
        issue_a(st[i], kbeg + kw + i * KW * U);
        compute(st[i], kbeg + kw + i * KW * U);
      }
      return;
    }
    first(st[0], kbeg + kw);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {                   // one step of lookahead, no register copies
      if (i + 1 < STEPS) issue(st[i + 1], kbeg + kw + (i + 1) * KW * U);
      compute(st[i], kbeg + kw + i * KW * U);
    }
  };
  // only where two steps plus the accumulators fit the register budget (measured: larger forms spill)
  constexpr int REG_EST = 2 * U * (TPW * 4 + MB * 4 * (SCALED ? 2 : 1)) + TPW * MB * 4;
  constexpr bool FIXED_OK = GEMV_UNROLL_FIXED && REG_EST <= (NW >= 16 ? 80 : 180) && (!SCALED || MB == 1);
  const int nk = kend - kbeg;
  if (FIXED_OK && nk == 64 && KW * U <= 64) fixed(std::integral_constant<int, 64>{});
  else if (FIXED_OK && nk == 32 && KW * U <= 32) fixed(std::integral_constant<int, 32>{});
  else if (FIXED_OK && nk == 16 && KW * U <= 16) fixed(std::integral_constant<int, 16>{});
  else if constexpr (NRM > 0) {
    // next step's weights in flight during this step's MFMAs (the loop below leaves that to the
    // scheduler; here the first step's weights are already loaded across the prologue)
    Step st;
    first(st, kbeg + kw);
    for (int kt = kbeg + kw; kt < kend; kt += KW * U) {
      Step nx;
      if (kt + KW * U < kend) issue_w(nx, kt + KW * U);
      compute(st, kt);
      if (kt + KW * U < kend) {
        issue_a(nx, kt + KW * U);
        st = nx;
      }
    }
  } else if constexpr (SCALED && MB <= 4 && 2 * REG_EST <= (NW >= 16 ? 160 : 360)) {
    // other k-range lengths (the down projection's 86 k-tiles per slice): one step of lookahead
    // in two named register sets, the loop run twice per iteration (no copies of a set with
    // loads outstanding).  Batch-1 down 11.6 us had three full memory round trips per wave here.
    // Grouped-scale inputs only (the model's o / down): cache-cold down at 64 rows 39.4 -> 34.3 us,
    // 1-32 rows unchanged; per-token inputs measured mixed (16 rows 14.5 -> 15.4 us), so they keep
    // the plain loop (profiles/gemv_lookahead_rows_r6.jsonl).
    Step s0, s1;
    int kt = kbeg + kw;
    if (kt < kend) issue(s0, kt);
    while (kt < kend) {
      const int k1 = kt + KW * U;
      if (k1 < kend) issue(s1, k1);
      compute(s0, kt);
      if (k1 >= kend) break;
      const int k2 = k1 + KW * U;
      if (k2 < kend) issue(s0, k2);
      compute(s1, k1);
      kt = k2;
    }
  } else {
    for (int kt = kbeg + kw; kt < kend; kt += KW * U) {
      Step st;
      issue(st, kt);
      compute(st, kt);
    }
  }
  if (KR == KW || kw >= KR) {
#pragma unroll
    for (int j = 0; j < TPW; ++j)
#pragma unroll
      for (int i = 0; i < MB; ++i)
        red[kw - (KW - KR)][(t0 + j) * MB + i][lane] = SCALED ? __builtin_bit_cast(v4i, accf[j][i]) : acc[j][i];
  }
  __syncthreads();
  if constexpr (KR != KW) {
    if (kw < KR) {
#pragma unroll
      for (int j = 0; j < TPW; ++j)
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          v4i& r = red[kw][(t0 + j) * MB + i][lane];
          if constexpr (SCALED) r = __builtin_bit_cast(v4i, __builtin_bit_cast(v4f, r) + accf[j][i]);
          else r += acc[j][i];
        }
    }
    __syncthreads();
  }
  if constexpr (L8G_N) {
    // wave 0, lanes 0-15: gate and up columns of feature nt0 * 16 + lane, each as the plain L8
    // epilogue below computes it (bf16), then silu(g) * u as rowwise.hip act_kernel MODE 0 does
    if (wave == 0 && lane < 16) {
      const v4i* rb = &red[0][0][0];
      float gu[2];
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        int tot = rb[jj * 64 + lane][0];
#pragma unroll
        for (int w = 1; w < KR; ++w) tot += rb[(w * NTW + jj) * 64 + lane][0];
        const int col = (jj == 0 ? nt0 : nt0 + NTt / 2) * 16 + lane;
        float y = (float)tot * nsa[0];
        y = y * sw[col] + (bias != nullptr ? bf2f(bias[col]) : 0.f);
        const int nt = l8_scr[L8_COUNT];
        if (nt > 0) {
          float a = 0.f;
          for (int j = 0; j < nt; ++j) a += l8_xo[j] * (float)na.wt[(size_t)l8_cols[j] * N + col];
          const float s = na.scb[col] / 127.f;
          y = bf2f(f2bf(y)) + a * s;
        }
        gu[jj] = bf2f(f2bf(y));
      }
      const float g = gu[0], u = gu[1];
      reinterpret_cast<bf16_t*>(outv)[nt0 * 16 + lane] = f2bf(g / (1.f + __expf(-g)) * u);
    }
  } else if constexpr (L8_N) {
    // row 0 of each tile (lanes 0-15, q = 0): the int8 part as the EPI_OUT epilogue rounds it, then
    // the outlier columns' 16-bit part (llmint8.hip llmint8_outlier_kernel's sum order and rounding)
    if (wave < NTW && lane < 16 && nt0 + wave < NTt) {
      const v4i* rb = &red[0][0][0];
      int tot = rb[wave * 64 + lane][0];
#pragma unroll
      for (int w = 1; w < KR; ++w) tot += rb[(w * NTW + wave) * 64 + lane][0];
      const int col = (nt0 + wave) * 16 + lane;
      if (col < N) {
        float y = (float)tot * nsa[0];
        y = y * pre.s0[0] + pre.b0[0];
        const int nt = l8_scr[L8_COUNT];
        if (nt > 0) {
          float a = 0.f;
          for (int j = 0; j < nt; ++j) a += l8_xo[j] * (float)na.wt[(size_t)l8_cols[j] * N + col];
          const float s = na.scb[col] / 127.f;
          y = bf2f(f2bf(y)) + a * s;
        }
        if constexpr (L8ACT_N > 0) {                    // rowwise.hip act_kernel MODE 1 / 2 of the bf16 output
          const float a = bf2f(f2bf(y));
          if (L8ACT_N == 1 || (L8ACT_N == 3 && na.act == 1)) y = 0.5f * a * (1.f + tanhf(0.7978845608028654f * (a + 0.044715f * a * a * a)));
          else y = 0.5f * a * (1.f + erff(a * 0.7071067811865476f));
        }
        if (na.add != nullptr) y = bf2f(f2bf(y)) + bf2f(na.add[col]);   // the other branch's row
        reinterpret_cast<bf16_t*>(outv)[col] = f2bf(y);
      }
    }
  } else {
    gemv_epilogue<MB, NTW, NW, KR, SCALED, EPI>(&red[0][0][0], NRM > 0 ? nsa : sa, pre, outv, os, gmax, M, N, NTt,
                                                Mpad, nt0, wave, lane, ks);
  }
}
}  // namespace
