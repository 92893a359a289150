// Bodies of the 16-bit decode GEMV (gemv_bf16.hip says how it works; decode_pair.hip runs two in one launch).
#pragma once
#include "common.h"

namespace {
constexpr int EPI_OUT = 0, EPI_GLU = 1, EPI_GELU_TANH = 2, EPI_GELU = 3, EPI_PART = 4,
              EPI_GELU_ANY = 5,               // gelu, tanh where F is 1, else erf
              EPI_ADD = 6,                    // EPI_OUT and an addend
              EPI_F32 = 7;                    // EPI_OUT's 16-bit numbers, stored as fp32
constexpr int GEMV_NW = 16;

typedef _Float16 v8h __attribute__((ext_vector_type(8)));

template <bool HF>
__device__ __forceinline__ v4f mfma_16(const v8s& a, const v8s& b, const v4f& c) {
  if constexpr (HF)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ v8s ld_nt(const bf16_t* p) {
  return __builtin_bit_cast(v8s, __builtin_nontemporal_load(reinterpret_cast<const v4i*>(p)));
}

// Decode RMSNorm prologue for the 16-bit GEMV (NRM > 0, M <= 4 rows, K 2048 / 4096): the activation
// rows are RMSNorm(sum of S fp32 split-K slices + residual), computed in the consumer instead of a
// norm launch of its own (rowwise.hip norm_kernel<NCH, RMS, HAS_RES, !QUANT, PART>: the same
// element layout, reduction order and roundings, so the rows are bit-identical).  Four 256-thread
// groups, one row each; the normalised 16-bit rows go to LDS, where the k-loop reads its A
// fragments.  The slices, residual and gamma loads all issue before any use.  Workgroup 0 writes
// the new residual rows.  NRM = 8 * NCH + SMAX (S <= SMAX slices).
// LN (NRM >= 64): LayerNorm of x + residual with 16-bit input rows x (the parallel-residual
// decoders, Phi-2 / GPT-NeoX: norm_kernel<NCH, !RMS, HAS_RES, !QUANT, !PART>), K up to 4096.
struct NormIn16 {
  const float* part;      // [S][M][K] fp32 slices (RMS)
  const bf16_t* res;      // [M][K] residual in (null: none, a stage's first norm over the embedding)
  const bf16_t* gamma;    // [K]
  bf16_t* res_out;        // [M][K] residual out (must not alias res)
  float eps;
  int S;
  const bf16_t* x;        // [M][K] 16-bit input rows (LN)
  const bf16_t* x2;       // [M][K] (LN; may be null): the block's other branch, x + x2 rounded before the residual joins
  const bf16_t* beta;     // [K] (LN; may be null)
  bf16_t* y_out;          // [M][K] (LN; may be null): workgroup 0 also writes the normalised rows here, ...
  const bf16_t* gamma2;   // [K] ... under these weights (a GPT-NeoX block's second norm of the same rows)
  const bf16_t* beta2;
};
constexpr int NRM16_ROWS = 4;

template <int NCH, int SMAX, bool LN = false>
struct NormRegs16 {
  uint4 rv[NCH], gv[NCH];
  float4 pv[NCH][LN ? 1 : SMAX][2];
  uint4 xv[NCH], bv[NCH], x2v[NCH], g2v[NCH], b2v[NCH];
};

template <int NCH, int SMAX, bool LN>
__device__ __forceinline__ void norm16_load(const NormIn16& na, bool wg0, int H, int M, NormRegs16<NCH, SMAX, LN>& nr) {
  const int t = threadIdx.x & 255, row = threadIdx.x >> 8;
  uint4 (&rv)[NCH] = nr.rv;
  uint4 (&gv)[NCH] = nr.gv;
  auto& pv = nr.pv;
  if constexpr (LN) {
    if (row < M) {
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const int e = min((c * 256 + t) * 8, H - 8);
        nr.xv[c] = *reinterpret_cast<const uint4*>(na.x + (size_t)row * H + e);
        nr.x2v[c] = na.x2 != nullptr ? *reinterpret_cast<const uint4*>(na.x2 + (size_t)row * H + e) : uint4{0u, 0u, 0u, 0u};
        rv[c] = na.res != nullptr ? *reinterpret_cast<const uint4*>(na.res + (size_t)row * H + e) : uint4{0u, 0u, 0u, 0u};
        gv[c] = *reinterpret_cast<const uint4*>(na.gamma + e);
        nr.bv[c] = na.beta != nullptr ? *reinterpret_cast<const uint4*>(na.beta + e) : uint4{0u, 0u, 0u, 0u};
        const bool two = wg0 && na.gamma2 != nullptr;
        nr.g2v[c] = two ? *reinterpret_cast<const uint4*>(na.gamma2 + e) : uint4{0u, 0u, 0u, 0u};
        nr.b2v[c] = two && na.beta2 != nullptr ? *reinterpret_cast<const uint4*>(na.beta2 + e) : uint4{0u, 0u, 0u, 0u};
      }
    }
    asm volatile("" ::: "memory");
    return;
  }
  if (row < M) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int e = min((c * 256 + t) * 8, H - 8);
      rv[c] = na.res != nullptr ? *reinterpret_cast<const uint4*>(na.res + (size_t)row * H + e) : uint4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int k = 0; k < SMAX; ++k)
        if (k < na.S) {
          const float4* p = reinterpret_cast<const float4*>(na.part + ((size_t)k * M + row) * H + e);
          pv[c][k][0] = p[0];
          pv[c][k][1] = p[1];
        }
      gv[c] = *reinterpret_cast<const uint4*>(na.gamma + e);
    }
  }
  asm volatile("" ::: "memory");                          // these loads issue before the weights
}

// LayerNorm form (norm_kernel's !RMS, HAS_RES, !PART path: x + residual rounded to 16 bits, the
// mean, then the variance of the rounded row, gamma and beta)
template <int NCH, bool HF>
__device__ __forceinline__ void ln16_prologue(const NormIn16& na, bool wg0, int H, int M, bf16_t* xs, float* nred,
                                              const NormRegs16<NCH, 1, true>& nr) {
  const int t = threadIdx.x & 255, row = threadIdx.x >> 8, w = t >> 6;
  const bool act = row < M;
  float v[NCH][8];
  float sm = 0.f;
  if (act) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int e = (c * 256 + t) * 8;
      if (e < H) {
        unpack8e<HF>(nr.xv[c], v[c]);
        float r[8];
        if (na.x2 != nullptr) {
          unpack8e<HF>(nr.x2v[c], r);
#pragma unroll
          for (int j = 0; j < 8; ++j) v[c][j] += r[j];
          unpack8e<HF>(pack8e<HF>(v[c]), v[c]);              // the sum of the branches is a 16-bit row
        }
        unpack8e<HF>(nr.rv[c], r);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[c][j] += r[j];
        const uint4 u = pack8e<HF>(v[c]);                    // the residual stream in 16 bits
        if (wg0) *reinterpret_cast<uint4*>(na.res_out + (size_t)row * H + e) = u;
        unpack8e<HF>(u, v[c]);
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
  float mean = 0.f, ss = 0.f;
  if (act) {
    const float* gr = nred + 4 * row;
    mean = ((((0.f + gr[0]) + gr[1]) + gr[2]) + gr[3]) / (float)H;
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
  if (act) {
    const float* gr = nred + 16 + 4 * row;
    const float rstd = rsqrtf(((((0.f + gr[0]) + gr[1]) + gr[2]) + gr[3]) / (float)H + na.eps);
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int e = (c * 256 + t) * 8;
      if (e < H) {
        float wf[8], bf[8], d0[8];
        unpack8e<HF>(nr.gv[c], wf);
        unpack8e<HF>(nr.bv[c], bf);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          d0[j] = v[c][j] - mean;
          v[c][j] = d0[j] * rstd * wf[j] + bf[j];
        }
        const uint4 u = pack8e<HF>(v[c]);
        *reinterpret_cast<uint4*>(xs + (size_t)row * H + e) = u;
        if (na.y_out != nullptr && wg0) {
          if (na.gamma2 != nullptr) {
            unpack8e<HF>(nr.g2v[c], wf);
            unpack8e<HF>(nr.b2v[c], bf);
            float v2[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v2[j] = d0[j] * rstd * wf[j] + bf[j];
            *reinterpret_cast<uint4*>(na.y_out + (size_t)row * H + e) = pack8e<HF>(v2);
          } else {
            *reinterpret_cast<uint4*>(na.y_out + (size_t)row * H + e) = u;
          }
        }
      }
    }
  }
  __syncthreads();                                        // the rows are complete in LDS
}

template <int NCH, int SMAX, bool HF>
__device__ __forceinline__ void norm16_prologue(const NormIn16& na, bool wg0, int H, int M, bf16_t* xs, float* nred,
                                                const NormRegs16<NCH, SMAX>& nr) {
  const int t = threadIdx.x & 255, row = threadIdx.x >> 8, w = t >> 6;
  const bool act = row < M;
  const uint4* rv = nr.rv;
  const uint4* gv = nr.gv;
  const auto& pv = nr.pv;
  float v[NCH][8];
  float ss = 0.f;
  if (act) {
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
        unpack8e<HF>(pack8e<HF>(v[c]), v[c]);                 // the projection's 16-bit output
        float r[8];
        unpack8e<HF>(rv[c], r);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[c][j] += r[j];
        const uint4 u = pack8e<HF>(v[c]);                    // the residual stream in 16 bits
        if (wg0) *reinterpret_cast<uint4*>(na.res_out + (size_t)row * H + e) = u;
        unpack8e<HF>(u, v[c]);
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
    if ((t & 63) == 0) nred[4 * row + w] = ss;
  }
  __syncthreads();
  if (act) {
    const float* gr = nred + 4 * row;
    const float rstd = rsqrtf((((0.f + gr[0]) + gr[1]) + gr[2] + gr[3]) / (float)H + na.eps);
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int e = (c * 256 + t) * 8;
      if (e < H) {
        float wf[8];
        unpack8e<HF>(gv[c], wf);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[c][j] = (v[c][j] - 0.f) * rstd * wf[j];
        *reinterpret_cast<uint4*>(xs + (size_t)row * H + e) = pack8e<HF>(v[c]);
      }
    }
  }
  __syncthreads();                                        // the rows are complete in LDS
}

// Workgroup bid of nwg of the GEMV of one row block (M <= 16): 16-column tiles bid, bid + nwg, ... one after the other,
// NWV waves that split K, U k-pairs of a wave requested before the first is used.
// What bounds it is the chain of memory round trips, so every load of a step is issued before any use (the fence: left
// alone, the compiler moves loads behind the products and under the guards of ragged ends, two to four round trips a wave
// instead of one), the next tile's first PRE k-pairs are requested before this one's sums meet, a wave holds one tile's
// numbers only, so that two workgroups fit a CU (gemv_bf16.hip: without a norm), and the instructions behind the last load are few.
// RB: groups of four rows (M <= 4 RB): a tile's rows are one number quadruple of 16 RB lanes, and the 64 lanes of one wave
// each add up NWV RB / 4 waves' sums.
// GLU: a tile is 8 gate columns and their 8 up columns (halves of two weight tiles, whole 128-byte lines of both).
// NRM: the first tile's k-pairs are in flight while the norm runs; the norm runs once for all tiles.
template <int NWV, int U, int PRE, int EPI, bool HF, int NRM, int RB>
__device__ __forceinline__ void gemv_tiles_body(int bid, int nwg, const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                const bf16_t* __restrict__ bias, bf16_t* __restrict__ out, int M, int N,
                                                int K, int F, int S, const bf16_t* __restrict__ add, const NormIn16& na) {
  static_assert(NRM == 0 || (NWV == GEMV_NW && RB == 1 && EPI != EPI_PART), "norm prologue: 16 waves, up to 4 rows");
  constexpr bool LN_N = NRM >= 64;
  constexpr int NCH_N = (NRM % 64) / 8, SMAX_N = LN_N ? 1 : NRM % 8;
  constexpr int RL = 16 * RB, WG = 4 / RB;                  // lanes of a wave's rows, waves that a wave adds up side by side
  __shared__ v4f red[2][NWV][RL];
  __shared__ __attribute__((aligned(16))) bf16_t xs[NRM > 0 ? NRM16_ROWS * NCH_N * 2048 : 8];
  __shared__ float nred[32];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15;
  const int KP = K / 64, tiles = N / 16 * (EPI == EPI_PART ? S : 1);
  // tile tt: this lane's fragments, the wave's first k-pair and the end of the tile's k-pairs
  const bf16_t* wp;
  int kp, kend;
  auto enter = [&](int tt) {
    if constexpr (EPI == EPI_GLU) {
      const int row = 8 * tt + (r < 8 ? r : F + r - 8);
      wp = W + ((size_t)(row >> 4) * (2 * KP) * 64 + (lane & 48) + (row & 15)) * 8;
    } else {
      wp = W + ((size_t)(EPI == EPI_PART ? tt / S : tt) * (2 * KP) * 64 + lane) * 8;
    }
    const int ks = EPI == EPI_PART ? tt % S : 0;
    kp = (EPI == EPI_PART ? KP * ks / S : 0) + wave;
    kend = EPI == EPI_PART ? KP * (ks + 1) / S : KP;
  };
  v8s p0[PRE > 0 ? PRE : 1][2];
  auto ahead = [&]() {
#pragma unroll
    for (int u = 0; u < PRE; ++u) {                          // clamped: loads never branch
      const int k = min(kp + NWV * u, kend - 1);
      p0[u][0] = ld_nt(wp + (size_t)k * 1024);               // tiles 2 kp, 2 kp + 1: 2 KiB contiguous
      p0[u][1] = ld_nt(wp + (size_t)k * 1024 + 512);
    }
  };
  const bf16_t* ar = (NRM > 0 ? xs : A) + (size_t)min(r, M - 1) * K + 8 * (lane >> 4);
  int t = bid;
  enter(t);
  if constexpr (NRM > 0) {
    NormRegs16<(NRM > 0 ? NCH_N : 1), (NRM > 0 ? SMAX_N : 1), LN_N> nr;
    norm16_load(na, bid == 0, K, M, nr);
    ahead();
    if constexpr (LN_N) ln16_prologue<NCH_N, HF>(na, bid == 0, K, M, xs, nred, nr);
    else norm16_prologue<NCH_N, SMAX_N, HF>(na, bid == 0, K, M, xs, nred, nr);
  } else ahead();
  for (int buf = 0; t < tiles; buf ^= 1) {
    const int ks = EPI == EPI_PART ? t % S : 0, tile = EPI == EPI_PART ? t / S : t;
    const int row0 = RB == 1 ? 0 : 4 * (lane >> 4), c = EPI == EPI_GLU ? 8 * tile + (r & 7) : 16 * tile + r;
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    // what the writing wave adds to its sums is requested with its first weights
    float bv = 0.f;
    bf16_t addv[4] = {0, 0, 0, 0};                          // (as they are: a conversion here would wait for them here)
    if (wave == 0) {
      if (bias != nullptr && (EPI != EPI_PART || ks == 0)) bv = e2f<HF>(bias[EPI == EPI_GLU && r >= 8 ? F + c : c]);
      if constexpr (EPI == EPI_ADD) {
#pragma unroll
        for (int q = 0; q < 4; ++q) addv[q] = add[(size_t)min(row0 + q, M - 1) * N + c];
      }
    }
    if constexpr (PRE > 0) {
      v8s a[PRE][2];
#pragma unroll
      for (int u = 0; u < PRE; ++u) {
        const int k = min(kp + NWV * u, kend - 1);
        a[u][0] = *reinterpret_cast<const v8s*>(ar + k * 64);
        a[u][1] = *reinterpret_cast<const v8s*>(ar + k * 64 + 32);
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int u = 0; u < PRE; ++u)
        if (kp + NWV * u < kend) {                           // wave-uniform (scalar) guard
          acc = mfma_16<HF>(a[u][0], p0[u][0], acc);
          acc = mfma_16<HF>(a[u][1], p0[u][1], acc);
        }
    }
    for (kp += NWV * PRE; kp < kend; kp += NWV * U) {
      v8s a[U][2], b[U][2];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = U == 1 ? kp : min(kp + u * NWV, kend - 1);
        b[u][0] = ld_nt(wp + (size_t)k * 1024);
        b[u][1] = ld_nt(wp + (size_t)k * 1024 + 512);
        a[u][0] = *reinterpret_cast<const v8s*>(ar + k * 64);
        a[u][1] = *reinterpret_cast<const v8s*>(ar + k * 64 + 32);
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (U == 1 || kp + u * NWV < kend) {
          acc = mfma_16<HF>(a[u][0], b[u][0], acc);
          acc = mfma_16<HF>(a[u][1], b[u][1], acc);
        }
    }
    t += nwg;
    if (t < tiles) {
      enter(t);
      ahead();
    }
    if (RB == 4 || lane < RL) red[buf][wave][lane & (RL - 1)] = acc;
    // two buffers: the wave that reads this one has passed the next barrier before anybody writes it again
    __syncthreads();
    if (wave == 0) {
      v4f s = red[buf][lane / RL][lane & (RL - 1)];
      // (16 rows: five reads at a time; all 15 at once are 60 registers, the second workgroup's)
#pragma unroll(RB == 4 ? 5 : NWV / WG)
      for (int w = 1; w < NWV / WG; ++w) s += red[buf][WG * w + lane / RL][lane & (RL - 1)];
      if constexpr (RB == 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] = xor_sum(s[q], 16);
      }
      if constexpr (RB <= 2) {
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] = xor_sum(s[q], 32);
      }
      if constexpr (EPI == EPI_GLU) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float g = e2f<HF>(f2e<HF>(s[q] + bv)), u = lane_xor(g, 8);
          if (r < 8 && (RB == 4 || lane < RL) && row0 + q < M)
            out[(size_t)(row0 + q) * F + c] = f2e<HF>(g / (1.f + __expf(-g)) * u);
        }
      } else if (RB == 4 || lane < RL) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int row = row0 + q;
          float v = s[q] + bv;
          if constexpr (EPI == EPI_PART) {
            if (row < M) reinterpret_cast<float*>(out)[((size_t)ks * M + row) * N + c] = v;
          } else {
            if constexpr (EPI == EPI_GELU_TANH || EPI == EPI_GELU || EPI == EPI_GELU_ANY) {
              const float x = e2f<HF>(f2e<HF>(v)), k0 = 0.7978845608028654f, k1 = 0.044715f;
              if (EPI == EPI_GELU_TANH || (EPI == EPI_GELU_ANY && F == 1))
                v = 0.5f * x * (1.f + tanhf(k0 * (x + k1 * x * x * x)));
              else v = 0.5f * x * (1.f + erff(x * 0.7071067811865476f));
            } else if constexpr (EPI == EPI_ADD) {
              // (parallel-residual block): rnd(rnd(y) + add), the unfused add
              v = e2f<HF>(f2e<HF>(v)) + e2f<HF>(addv[q]);
            }
            if constexpr (EPI == EPI_F32) {
              if (row < M) reinterpret_cast<float*>(out)[(size_t)row * N + c] = e2f<HF>(f2e<HF>(v));
            } else {
              if (row < M) out[(size_t)row * N + c] = f2e<HF>(v);
            }
          }
        }
      }
    }
  }
}

// One workgroup (bid) of the GEMV of more rows: NTW tiles, MB row blocks of 16.
template <int MB, int NTW, int U, int EPI, bool HF>
__device__ __forceinline__ void gemv_bf16_body(int bid, const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                               const bf16_t* __restrict__ bias, bf16_t* __restrict__ out, int M, int N,
                                               int K, int F, int S, const bf16_t* __restrict__ add) {
  constexpr int NWV = GEMV_NW;
  static_assert(EPI != EPI_GLU || NTW % 2 == 0, "GLU: gate/up tile pairs");
  static_assert(MB * NTW <= 8 && MB * (EPI == EPI_GLU ? NTW / 2 : NTW) <= NWV, "LDS reduction / output waves");
  __shared__ v4f red[NWV][MB * NTW][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, kq = 8 * (lane >> 4);
  // output column of tile j for this lane (EPI_GLU: gate tiles then the matching up tiles)
  const int grp = EPI == EPI_PART ? bid / S : bid;
  const int ks = EPI == EPI_PART ? bid % S : 0;
  auto col_of = [&](int j) -> int {
    if constexpr (EPI == EPI_GLU) {
      const int f0 = grp * (NTW / 2) * 16;
      return j < NTW / 2 ? f0 + j * 16 + r : F + f0 + (j - NTW / 2) * 16 + r;
    } else {
      return (grp * NTW + j) * 16 + r;
    }
  };
  const int KP = K / 64;
  const int kbeg = EPI == EPI_PART ? KP * ks / S : 0, kend = EPI == EPI_PART ? KP * (ks + 1) / S : KP;
  const bf16_t* wrow[NTW];                                  // tile row of this lane's fragments
#pragma unroll
  for (int j = 0; j < NTW; ++j) wrow[j] = W + ((size_t)(min(col_of(j), N - 1) >> 4) * (2 * KP) * 64 + lane) * 8;
  const bf16_t* arow[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) arow[mb] = A + (size_t)min(16 * mb + r, M - 1) * K + kq;
  v4f acc[MB][NTW];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int j = 0; j < NTW; ++j) acc[mb][j] = v4f{0.f, 0.f, 0.f, 0.f};
  for (int kp = kbeg + wave; kp < kend; kp += NWV * U) {
    v8s a[U][MB][2], b[U][NTW][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(kp + u * NWV, kend - 1) * 64;        // clamped: loads never branch
#pragma unroll
      for (int j = 0; j < NTW; ++j) {                        // tiles 2 kp, 2 kp + 1: 2 KiB contiguous
        b[u][j][0] = ld_nt(wrow[j] + (size_t)k * 16);
        b[u][j][1] = ld_nt(wrow[j] + (size_t)k * 16 + 512);
      }
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        a[u][mb][0] = *reinterpret_cast<const v8s*>(arow[mb] + k);
        a[u][mb][1] = *reinterpret_cast<const v8s*>(arow[mb] + k + 32);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (kp + u * NWV < kend) {                             // wave-uniform (scalar) guard
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int j = 0; j < NTW; ++j) {
            acc[mb][j] = mfma_16<HF>(a[u][mb][0], b[u][j][0], acc[mb][j]);
            acc[mb][j] = mfma_16<HF>(a[u][mb][1], b[u][j][1], acc[mb][j]);
          }
      }
    }
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int j = 0; j < NTW; ++j) red[wave][mb * NTW + j][lane] = acc[mb][j];
  __syncthreads();
  // output units (row block, tile): wave w < MB * OUTS writes tile w % OUTS of row block w / OUTS
  constexpr int OUTS = EPI == EPI_GLU ? NTW / 2 : NTW;
  if (wave < MB * OUTS) {
    const int mb = wave / OUTS, tw = wave - mb * OUTS;
    auto total = [&](int j) {                               // 4 LDS reads in flight (bounded registers)
      v4f s = red[0][mb * NTW + j][lane];
#pragma unroll 4
      for (int w = 1; w < NWV; ++w) s += red[w][mb * NTW + j][lane];
      return s;
    };
    const int c0 = col_of(tw);
    if constexpr (EPI == EPI_GLU) {
      const int c1 = col_of(tw + NTW / 2);
      const v4f g4 = total(tw), u4 = total(tw + NTW / 2);
      const float bg = bias != nullptr ? e2f<HF>(bias[c0]) : 0.f, bu = bias != nullptr ? e2f<HF>(bias[min(c1, N - 1)]) : 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = 16 * mb + 4 * (lane >> 4) + q;
        const float g = e2f<HF>(f2e<HF>(g4[q] + bg)), u = e2f<HF>(f2e<HF>(u4[q] + bu));
        if (row < M && c0 < F) out[(size_t)row * F + c0] = f2e<HF>(g / (1.f + __expf(-g)) * u);
      }
    } else if constexpr (EPI == EPI_PART) {
      const v4f s4 = total(tw);
      const float bv = bias != nullptr && c0 < N && ks == 0 ? e2f<HF>(bias[c0]) : 0.f;
      float* part = reinterpret_cast<float*>(out) + (size_t)ks * M * N;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = 16 * mb + 4 * (lane >> 4) + q;
        if (row < M && c0 < N) part[(size_t)row * N + c0] = s4[q] + bv;
      }
    } else {
      const v4f s4 = total(tw);
      const float bv = bias != nullptr && c0 < N ? e2f<HF>(bias[c0]) : 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = 16 * mb + 4 * (lane >> 4) + q;
        float v = s4[q] + bv;
        if constexpr (EPI == EPI_GELU_TANH || EPI == EPI_GELU) {
          const float a = e2f<HF>(f2e<HF>(v)), k0 = 0.7978845608028654f, k1 = 0.044715f;
          if (EPI == EPI_GELU_TANH)
            v = 0.5f * a * (1.f + tanhf(k0 * (a + k1 * a * a * a)));
          else v = 0.5f * a * (1.f + erff(a * 0.7071067811865476f));
        } else {
          // EPI_OUT with an addend (parallel-residual block): rnd(rnd(y) + add), the unfused add
          if (add != nullptr && row < M && c0 < N) v = e2f<HF>(f2e<HF>(v)) + e2f<HF>(add[(size_t)row * N + c0]);
        }
        if constexpr (EPI == EPI_F32) {
          if (row < M && c0 < N) reinterpret_cast<float*>(out)[(size_t)row * N + c0] = e2f<HF>(f2e<HF>(v));
        } else {
          if (row < M && c0 < N) out[(size_t)row * N + c0] = f2e<HF>(v);
        }
      }
    }
  }
}
}  // namespace
