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
// state_w (every sequence brings one token: this thread is the only reader of its channels' tail): the tail moves up here.
template <typename TI, typename TO, int TB, bool SILU>
__global__ void __launch_bounds__(NT) tap4_kernel(const TI* __restrict__ u, int ld, int c0, int C, const float* __restrict__ w,
                                                  const float* __restrict__ bias, const TI* state,
                                                  const int* __restrict__ tok_seq, const int* __restrict__ tok_pos,
                                                  const int* __restrict__ seq_slot, const int* __restrict__ seq_start,
                                                  TO* __restrict__ out, TI* state_w, int rows) {
  constexpr int CV = 16 / sizeof(TI);
  const int c = (blockIdx.y * NT + threadIdx.x) * CV, t0 = blockIdx.x * TB;
  if (c >= C) return;
  auto load = [](const TI* p, float (&f)[CV]) {
    if constexpr (CV == 8) load8<TI>(p, f);
    else {
      const float4 v = *reinterpret_cast<const float4*>(p);
      f[0] = v.x; f[1] = v.y; f[2] = v.z; f[3] = v.w;
    }
  };
  float x[TB + 3][CV], br[CV];
  float4 wr[CV];
  int sq[TB], ps[TB], st0[TB], slot[TB];
#pragma unroll
  for (int i = 0; i < TB; ++i) { sq[i] = tok_seq[min(t0 + i, rows - 1)]; ps[i] = tok_pos[min(t0 + i, rows - 1)]; }
#pragma unroll
  for (int r = 0; r < TB + 3; ++r) load(u + (size_t)min(max(t0 - 3 + r, 0), rows - 1) * ld + c0 + c, x[r]);
#pragma unroll
  for (int e = 0; e < CV; ++e) {
    wr[e] = *reinterpret_cast<const float4*>(w + (size_t)(c + e) * 4);
    br[e] = SILU ? bias[c + e] : 0.f;
  }
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
    if (have < 3) {
      float tail[3][CV];
#pragma unroll
      for (int k = 0; k < 3; ++k) load(state + ((size_t)slot[i] * 3 + min(have + k, 2)) * C + c, tail[k]);
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int e = 0; e < CV; ++e) v[k][e] = k >= 3 - have ? v[k][e] : (ps[i] - 3 + k >= 0 ? tail[k][e] : 0.f);
    }
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
    if (state_w) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        TI* d = state_w + ((size_t)slot[i] * 3 + k) * C + c;
        if constexpr (CV == 8) store8<TI>(d, v[k + 1]);
        else *reinterpret_cast<float4*>(d) = make_float4(v[k + 1][0], v[k + 1][1], v[k + 1][2], v[k + 1][3]);
      }
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

template <typename TI, typename TO, bool SILU>
void launch_tap4(const TI* u, int ld, int c0, int C, const float* w, const float* bias, TI* state, const int* tok_seq,
                 const int* tok_pos, const int* seq_slot, const int* seq_start, TO* out, int rows, bool one, hipStream_t st) {
  const int gy = (C / (16 / (int)sizeof(TI)) + NT - 1) / NT;
  if (rows >= 512)
    hipLaunchKernelGGL((tap4_kernel<TI, TO, 4, SILU>), dim3((rows + 3) / 4, gy), dim3(NT), 0, st, u, ld, c0, C, w, bias, state,
                       tok_seq, tok_pos, seq_slot, seq_start, out, one ? state : (TI*)nullptr, rows);
  else
    hipLaunchKernelGGL((tap4_kernel<TI, TO, 1, SILU>), dim3(rows, gy), dim3(NT), 0, st, u, ld, c0, C, w, bias, state, tok_seq,
                       tok_pos, seq_slot, seq_start, out, one ? state : (TI*)nullptr, rows);
}

}  // namespace
