// Preparation of the gated delta rule's rows, shared by the kernel files that instantiate it.
#pragma once
#include "common.h"
#include "seqmix/seqmix_common.h"

namespace {

// prep row = q [G, N] | k [G, N] | decay [H, N] (HEAD: [H]) | beta [H], all fp32: q and k of unit length (q / sqrt(N)),
// decay = exp(-exp(A_log) softplus(raw + dt_bias)) with raw = a [rows, H N] (HEAD: columns a0.. of u), beta = sigmoid(u[b0..]).
// A unit (q or k of one head) belongs to 16 lanes, four numbers per access; a workgroup of a token takes 16 units or 1024
// decays, so one token's chain is one load, one sum over 16 lanes, one store.  (One workgroup per token walked 2 G units, a
// wave each, and then the decays.)  us, G = H = 16, N = 64, one workgroup per token / this: 4096 tokens 38 / 24.9, 4 tokens
// 10.5 / 3.6; HEAD, N = 128, 6 tokens 12.3 / 5.2.  N % 4 == 0, N <= 256, H % 4 == 0, Cq % 4 == 0 and 16-byte rows (launch_delta_prep16
// asks).
template <typename T, bool HEAD>
__global__ void __launch_bounds__(NT) delta_prep16_kernel(const T* __restrict__ qkv, int Cq, const T* __restrict__ u, int ld,
                                                          int b0, int a0, const float* __restrict__ a,
                                                          const float* __restrict__ dt_bias, const float* __restrict__ A_log,
                                                          float* __restrict__ prep, int H, int G, int N) {
  const size_t t = blockIdx.x;
  const int tid = threadIdx.x, l16 = tid & 15, GN = G * N, DN = HEAD ? H : H * N, UB = (2 * G + 15) / 16;
  float* pr = prep + t * (2 * GN + DN + H);
  if ((int)blockIdx.y < UB) {
    const int unit = blockIdx.y * 16 + (tid >> 4);
    const bool on = unit < 2 * G;
    const T* src = qkv + t * Cq + (size_t)(on ? unit : 0) * N;
    float v[4][4], ss = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = l16 * 4 + 64 * i;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i][e] = 0.f;
      if (64 * i < N) load4<T>(src + min(n, N - 4), v[i]);
#pragma unroll
      for (int e = 0; e < 4; ++e) ss += n < N ? v[i][e] * v[i][e] : 0.f;
    }
    const float r = 1.f / sqrtf(row16_sum(ss) + 1e-6f) * (unit < G ? 1.f / sqrtf((float)N) : 1.f);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = l16 * 4 + 64 * i;
      if (on && n < N)
        *reinterpret_cast<float4*>(pr + (size_t)unit * N + n) = make_float4(v[i][0] * r, v[i][1] * r, v[i][2] * r, v[i][3] * r);
    }
    return;
  }
  auto decay = [](float raw, float al) {
    const float sp = raw > 20.f ? raw : log1pf(expf(raw));
    return expf(-expf(al) * sp);
  };
  const int blk = blockIdx.y - UB;
  if constexpr (!HEAD) {
    const int e = (blk * NT + tid) * 4;
    if (e < DN) {
      const float4 av = *reinterpret_cast<const float4*>(a + t * DN + e), dv = *reinterpret_cast<const float4*>(dt_bias + e);
      const float al = A_log[e / N];
      *reinterpret_cast<float4*>(pr + 2 * GN + e) =
          make_float4(decay(av.x + dv.x, al), decay(av.y + dv.y, al), decay(av.z + dv.z, al), decay(av.w + dv.w, al));
    }
  }
  if (blk == 0)
    for (int e = tid; e < H; e += NT) {
      if constexpr (HEAD) pr[2 * GN + e] = decay(ldf<T>(u + t * ld + a0 + e) + dt_bias[e], A_log[e]);
      pr[2 * GN + DN + e] = sigmoidf_(ldf<T>(u + t * ld + b0 + e));
    }
}

// true when it took the call
template <typename T, bool HEAD>
bool launch_delta_prep16(const T* qkv, int Cq, const T* u, int ld, int b0, int a0, const float* a, const float* dt_bias,
                         const float* A_log, float* prep, int rows, int H, int G, int N, hipStream_t st) {
  if (N % 4 || N < 4 || N > 256 || H % 4 || Cq % 4 ||
      (((uintptr_t)qkv | (uintptr_t)a | (uintptr_t)dt_bias | (uintptr_t)prep) & 15))
    return false;
  const int gy = (2 * G + 15) / 16 + (HEAD ? 1 : (H * N / 4 + NT - 1) / NT);
  hipLaunchKernelGGL((delta_prep16_kernel<T, HEAD>), dim3(rows, gy), dim3(NT), 0, st, qkv, Cq, u, ld, b0, a0, a, dt_bias, A_log,
                     prep, H, G, N);
  return true;
}

}  // namespace
