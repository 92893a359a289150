// One token of one head of the state-space recurrence by 256 threads (ssd_step.hip says how and why), for a kernel of its own and for one
// in which attention's workgroups run beside it.
#pragma once
#include "seqmix/seqmix_common.h"

namespace {

struct SsdStep {
  const void *xbc, *u;
  const float *dt_bias, *A_log, *D;
  float *state, *y;                                          // state [slots, H, N, P]; y [rows, H P]
  const int *seq_slot, *seq_start, *seq_off;
  int Cx, ld, dt0, H, groups;
};

// the workgroup's threads tid 0 .. 255 take head h of sequence s; sum_s: P numbers a wave.  Every thread of the workgroup comes to its barrier
template <typename T, int N, int P>
__device__ __forceinline__ void ssd_step_body(const SsdStep& a, int s, int h, int tid, float (*sum_s)[P]) {
  constexpr int PG = P / 4, RGS = NT / PG, NR = N / RGS, NW = NT / 64;
  static_assert(P % 4 == 0 && PG <= 64 && 64 % PG == 0 && N % RGS == 0, "shape");
  // the wave's number as a scalar: conditions and addresses that depend on it alone take the scalar unit (a prompt of 777 and 15 steps
  // of four parallel layers 6.85 -> 6.79 ms with the kernels beside it)
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slot = a.seq_slot[s], start = a.seq_start[s];
  const size_t t = a.seq_off[s];
  const int p0 = (tid % PG) * 4, n0 = tid / PG * NR, g = h / (a.H / a.groups), inner = a.H * P;
  float* st = a.state + (((size_t)slot * a.H + h) * N + n0) * P + p0;
  float4 S[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) S[i] = start > 0 ? *reinterpret_cast<const float4*>(st + (size_t)i * P) : make_float4(0.f, 0.f, 0.f, 0.f);
  const T* row = reinterpret_cast<const T*>(a.xbc) + t * a.Cx;
  float x[4], B[NR], C[NR];
  load4<T>(row + h * P + p0, x);
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    B[i] = ldf<T>(row + inner + g * N + n0 + i);
    C[i] = ldf<T>(row + inner + (a.groups + g) * N + n0 + i);
  }
  const float raw = ldf<T>(reinterpret_cast<const T*>(a.u) + t * a.ld + a.dt0 + h) + a.dt_bias[h];
  const float dt = raw > 20.f ? raw : log1pf(expf(raw)), dec = expf(-expf(a.A_log[h]) * dt);
  float y[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    float v[4] = {S[i].x, S[i].y, S[i].z, S[i].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = dec * v[e] + B[i] * (dt * x[e]);
      y[e] += v[e] * C[i];
    }
    *reinterpret_cast<float4*>(st + (size_t)i * P) = make_float4(v[0], v[1], v[2], v[3]);
  }
#pragma unroll
  for (int o = PG; o < 64; o <<= 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = xor_sum(y[e], o);
  if (lane < PG) *reinterpret_cast<float4*>(&sum_s[wave][p0]) = make_float4(y[0], y[1], y[2], y[3]);
  __syncthreads();
  if (tid < P) {
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) o += sum_s[w][tid];
    a.y[t * inner + h * P + tid] = o + a.D[h] * ldf<T>(row + h * P + tid);
  }
}

}  // namespace
