// Four-tap causal convolutions over ragged rows, shared by the kernel files that instantiate it.
#pragma once
#include "common.h"
#include "seqmix/seqmix_common.h"

namespace {

// One 16-byte run of channels (CV numbers) of TB consecutive tokens per thread.  SILU: out = silu(bias + sum_k w[:, k] x_k);
// else out = x_3 + sum_k w[:, k] x_k, with x_k the input at position pos - 3 + k: a row of the step (row t of the step is
// position start + t - off of its sequence), before the portion one of the slot's tail [3][C], before position 0 zero.
// Bound by latency on decode-sized steps, by the rows' bytes on prompts: so every load is issued before any is used (the
// TB + 3 rows, then the tail's where the portion begins, from clamped addresses; chosen afterwards), a channel's four
// weights are one load, and TB tokens share rows and weights.
// Other tap counts and unaligned columns run the general kernels (taps in a loop, loads under conditions).  us, general /
// this: silu 3072 of bf16 over 4096 tokens 51 / 22.5, over 4 9.3 / 4.3; plain 1024 of fp32 over 4096 tokens 32.9 / 7.9,
// over 4 5.2 / 3.4; silu 1152 of fp32 over 2 tokens 7.8 / 4.0.  Four tokens per thread from 512 rows on, one below: there
// are enough workgroups then.
// Every sequence brings one token (not ENDS): a thread is the only reader of its channels' tail, and moves it up.
// ENDS (portions): the first `ends` rows of the grid are a sequence each.  They alone touch the tails: a thread forms its sequence's
// first three tokens, which read the old tail, and leaves the portion's last three rows there, so that no launch for that stands behind
// this one (us in a graph, with that launch / now: plain 1024 over 4096 tokens 12.1 / 6.8, over 512 8.5 / 4.0; silu 3072 of bf16 26.4 / 23.1, 9.4 / 7.2).
template <typename TI, typename TO, int TB, bool SILU, bool ENDS>
__global__ void __launch_bounds__(NT) tap4_kernel(const TI* __restrict__ u, int ld, int c0, int C, const float* __restrict__ w,
                                                  const float* __restrict__ bias, TI* state,
                                                  const int* __restrict__ tok_seq, const int* __restrict__ tok_pos,
                                                  const int* __restrict__ seq_slot, const int* __restrict__ seq_start,
                                                  TO* __restrict__ out, int rows, int ends, const int* __restrict__ seq_len,
                                                  const int* __restrict__ seq_off) {
  constexpr int CV = 16 / sizeof(TI);
  const int c = (blockIdx.y * NT + threadIdx.x) * CV, t0 = ((int)blockIdx.x - (ENDS ? ends : 0)) * TB;
  if (c >= C) return;
  auto load = [](const TI* p, float (&f)[CV]) {
    if constexpr (CV == 8) load8<TI>(p, f);
    else {
      const float4 v = *reinterpret_cast<const float4*>(p);
      f[0] = v.x; f[1] = v.y; f[2] = v.z; f[3] = v.w;
    }
  };
  float br[CV];
  float4 wr[CV];
  auto weights = [&]() {
#pragma unroll
    for (int e = 0; e < CV; ++e) {
      wr[e] = *reinterpret_cast<const float4*>(w + (size_t)(c + e) * 4);
      br[e] = SILU ? bias[c + e] : 0.f;
    }
  };
  auto token = [&](const float (&v)[4][CV], int t) {
    float y[CV];
#pragma unroll
    for (int e = 0; e < CV; ++e) {
      float acc = br[e];
      acc += wr[e].x * v[0][e];
      acc += wr[e].y * v[1][e];
      acc += wr[e].z * v[2][e];
      acc += wr[e].w * v[3][e];
      y[e] = SILU ? siluf_(acc) : v[3][e] + acc;
    }
    TO* o = out + (size_t)t * C + c;
    if constexpr (CV == 8) store8<TO>(o, y);
    else if constexpr (sizeof(TO) == 4) *reinterpret_cast<float4*>(o) = make_float4(y[0], y[1], y[2], y[3]);
    else *reinterpret_cast<uint2*>(o) = make_uint2(pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3]));
  };
  auto keep = [&](TI* d, const float (&v)[CV]) {
    if constexpr (CV == 8) store8<TI>(d, v);
    else *reinterpret_cast<float4*>(d) = make_float4(v[0], v[1], v[2], v[3]);
  };
  if (ENDS && t0 < 0) {
    const int s = blockIdx.x, start = seq_start[s], len = seq_len[s], off = seq_off[s];
    TI* const tail = state + (size_t)seq_slot[s] * 3 * C + c;
    if (len < 1) {                                           // (no rows: of the tail, what lies in front of the sequence is cleared)
      const float none[CV] = {};
#pragma unroll
      for (int k = 0; k < 3; ++k)
        if (start - 3 + k < 0) keep(tail + (size_t)k * C, none);
      return;
    }
    float v[9][CV];                                          // the old tail, the first three rows, the last three
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      load(tail + (size_t)k * C, v[k]);
      load(u + (size_t)(off + min(k, len - 1)) * ld + c0 + c, v[3 + k]);
      load(u + (size_t)(off + max(len - 3 + k, 0)) * ld + c0 + c, v[6 + k]);
    }
    weights();
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int e = 0; e < CV; ++e) v[k][e] = start - 3 + k >= 0 ? v[k][e] : 0.f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      if (i >= len) break;
      float x[4][CV];
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int e = 0; e < CV; ++e) x[k][e] = v[i + k][e];
      token(x, off + i);
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {                            // position len - 3 + k of the portion, or the old tail's len + k
      float x[CV];
#pragma unroll
      for (int e = 0; e < CV; ++e) {
        const float old = len == 1 ? v[min(1 + k, 2)][e] : v[min(2 + k, 2)][e];
        x[e] = len - 3 + k >= 0 ? v[6 + k][e] : old;
      }
      keep(tail + (size_t)k * C, x);
    }
    return;
  }
  float x[TB + 3][CV];
  int sq[TB], ps[TB], st0[TB], slot[TB];
#pragma unroll
  for (int i = 0; i < TB; ++i) { sq[i] = tok_seq[min(t0 + i, rows - 1)]; ps[i] = tok_pos[min(t0 + i, rows - 1)]; }
#pragma unroll
  for (int r = 0; r < TB + 3; ++r) load(u + (size_t)min(max(t0 - 3 + r, 0), rows - 1) * ld + c0 + c, x[r]);
  weights();
#pragma unroll
  for (int i = 0; i < TB; ++i) { st0[i] = seq_start[sq[i]]; slot[i] = seq_slot[sq[i]]; }
#pragma unroll
  for (int i = 0; i < TB; ++i) {
    const int t = t0 + i, have = ps[i] - st0[i];             // rows of this portion before the token
    if (t >= rows) return;
    float v[4][CV];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int e = 0; e < CV; ++e) v[k][e] = x[i + k][e];
    if (ENDS && have < 3) continue;                          // the sequence's own row has it
    if (!ENDS && have < 3) {
      float tail[3][CV];
#pragma unroll
      for (int k = 0; k < 3; ++k) load(state + ((size_t)slot[i] * 3 + min(have + k, 2)) * C + c, tail[k]);
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int e = 0; e < CV; ++e) v[k][e] = k >= 3 - have ? v[k][e] : (ps[i] - 3 + k >= 0 ? tail[k][e] : 0.f);
    }
    token(v, t);
    if constexpr (!ENDS) {
#pragma unroll
      for (int k = 0; k < 3; ++k) keep(state + ((size_t)slot[i] * 3 + k) * C + c, v[k + 1]);
    }
  }
}

// whether every 16-byte access of tap4_kernel is aligned (the [rows, C] output: 16 bytes, or 8 behind fp32 inputs in bf16)
template <typename TI>
inline bool tap4_ok(int taps, int ld, int c0, int C, const void* u, const void* w, const void* state, const void* out) {
  constexpr int CV = 16 / sizeof(TI);
  return taps == 4 && ld % CV == 0 && c0 % CV == 0 && C % CV == 0 &&
         (((uintptr_t)u | (uintptr_t)w | (uintptr_t)state | (uintptr_t)out) & 15) == 0;
}

// one: every sequence brings one token.  The tails move up either way.
template <typename TI, typename TO, bool SILU>
void launch_tap4(const TI* u, int ld, int c0, int C, const float* w, const float* bias, TI* state, const int* tok_seq,
                 const int* tok_pos, const int* seq_slot, const int* seq_start, const int* seq_len, const int* seq_off, TO* out, int rows,
                 int n, bool one, hipStream_t st) {
  const int gy = (C / (16 / (int)sizeof(TI)) + NT - 1) / NT;
#define TAP4(TB, E)                                                                                                              \
  hipLaunchKernelGGL((tap4_kernel<TI, TO, TB, SILU, E>), dim3((E ? n : 0) + (rows + TB - 1) / TB, gy), dim3(NT), 0, st, u, ld, c0, C, w, \
                     bias, state, tok_seq, tok_pos, seq_slot, seq_start, out, rows, n, seq_len, seq_off)
  if (rows >= 512) {
    if (one) TAP4(4, false);
    else TAP4(4, true);
  } else if (one) TAP4(1, false);
  else TAP4(1, true);
#undef TAP4
}

}  // namespace
