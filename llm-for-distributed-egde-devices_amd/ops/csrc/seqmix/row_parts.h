// A row of a mixture's results in registers: four consecutive numbers per access and thread, CH accesses.
#pragma once
#include "common.h"
#include "seqmix/seqmix_common.h"

namespace {

// v[i] += sum_k pw[t, k] parts[t, k] (pw null: ones) at columns (threadIdx.x + i NT) 4, four parts' loads at a time; columns past W
// read the last ones again
template <typename T, int CH>
__device__ __forceinline__ void add_parts(float (&v)[CH][4], const T* __restrict__ parts, const float* __restrict__ pw, int K, size_t t,
                                          int W) {
  for (int k0 = 0; k0 < K; k0 += 4) {
    float p[4][CH][4], pk[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      pk[k] = pw ? pw[t * K + min(k0 + k, K - 1)] : 1.f;
#pragma unroll
      for (int i = 0; i < CH; ++i)
        load4<T>(parts + (t * K + min(k0 + k, K - 1)) * W + min(((int)threadIdx.x + i * NT) * 4, W - 4), p[k][i]);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < CH; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i][e] = k0 + k < K ? v[i][e] + pk[k] * p[k][i][e] : v[i][e];
  }
}

// sum of s over the workgroup of NW waves (r: NW numbers of LDS, used once)
template <int NW = NT / 64>
__device__ __forceinline__ float row_total(float s, float* r) {
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) r[threadIdx.x >> 6] = s;
  __syncthreads();
  float o = 0.f;
#pragma unroll
  for (int i = 0; i < NW; ++i) o += r[i];
  return o;
}

}  // namespace
