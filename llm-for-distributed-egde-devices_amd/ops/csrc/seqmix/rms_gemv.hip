// Up to 16 bf16 rows, RMS-normed and projected in one launch: the query latents of a decode step.  W lies as gemv_bf16.hip says.
// Bound by latency: the norm was a launch of some KB in front of a launch of some hundred KB.  A wave takes a tile of 16 features over all of
// K (up to 512) and asks for its weights, the rows and the norm's weights at once; the rows lie in the matrix cores' order, so
// a row's sum of squares is two exchanges away and nothing passes through the LDS.  The normed row is rounded as rms_cols_kernel rounds it.
// us, two launches / one, bf16: 384 x 1536, 1 row 5.2 / 4.0, 4 rows 5.3 / 4.2, 16 rows 5.8 / 4.2; 512 x 8192, 4 rows 6.7 / 5.3, 16 rows 7.9 / 5.4; 128 x
// 512, 4 rows 5.1 / 3.0; a decode of 4 sequences, 63 steps of two such layers, 14.77 -> 14.51 ms.
#include "common.h"
#include "seqmix/seqmix_common.h"

namespace {

template <int KS>
__global__ void __launch_bounds__(64) rms_gemv_kernel(const bf16_t* __restrict__ u, int ld, const float* __restrict__ g,
                                                      const bf16_t* __restrict__ W, bf16_t* __restrict__ out, int M, int N, int ks,
                                                      float eps) {
  const int tile = blockIdx.x, lane = threadIdx.x, r = lane & 15, grp = lane >> 4, K = 32 * ks;
  const bf16_t* ur = u + (size_t)min(r, M - 1) * ld + 8 * grp;
  const bf16_t* wp = W + ((size_t)tile * ks * 64 + lane) * 8;
  uint4 x[KS], w[KS];
  float gv[KS][8];
#pragma unroll
  for (int k = 0; k < KS; ++k) {                             // clamped: loads never branch
    const int c = min(k, ks - 1);
    x[k] = *reinterpret_cast<const uint4*>(ur + 32 * c);
    load8<float>(g + 32 * c + 8 * grp, gv[k]);
    w[k] = *reinterpret_cast<const uint4*>(wp + (size_t)c * 512);
  }
  asm volatile("" ::: "memory");
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < KS; ++k)
    if (k < ks) {
      float f[8];
      unpack8(x[k], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
    }
  ss = xor_sum(xor_sum(ss, 16), 32);
  const float rr = 1.f / sqrtf(ss / (float)K + eps);
  v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < KS; ++k)
    if (k < ks) {
      float f[8];
      unpack8(x[k], f);
      uint4 a;
      a.x = pack_bf2(f[0] * rr * gv[k][0], f[1] * rr * gv[k][1]);
      a.y = pack_bf2(f[2] * rr * gv[k][2], f[3] * rr * gv[k][3]);
      a.z = pack_bf2(f[4] * rr * gv[k][4], f[5] * rr * gv[k][5]);
      a.w = pack_bf2(f[6] * rr * gv[k][6], f[7] * rr * gv[k][7]);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8s, a), __builtin_bit_cast(v8s, w[k]), acc, 0, 0, 0);
    }
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (4 * grp + q < M) out[(size_t)(4 * grp + q) * N + 16 * tile + r] = f2bf(acc[q]);
}

}  // namespace

// -2: not taken
extern "C" int edge_sm_rms_gemv(const void* u, int ld, const float* g, const void* W, void* out, int M, int N, int K, float eps,
                                hipStream_t st) {
  if (M < 1 || M > 16 || N < 16 || N % 16 || K < 32 || K > 512 || K % 32 || ld % 8 || ((uintptr_t)u | (uintptr_t)g | (uintptr_t)W) % 16)
    return -2;
  const int ks = K / 32;
#define RG(KS)                                                                                                              \
  hipLaunchKernelGGL(rms_gemv_kernel<KS>, dim3(N / 16), dim3(64), 0, st, (const bf16_t*)u, ld, g, (const bf16_t*)W, (bf16_t*)out, M, N, \
                     ks, eps)
  if (ks <= 4) RG(4);
  else if (ks <= 8) RG(8);
  else if (ks <= 12) RG(12);
  else RG(16);
#undef RG
  return (int)hipGetLastError();
}
