// One token per sequence through the state-space recurrence (ssd_kernel's and its rounding, seqmix.hip):
//   S <- e^{-e^{A_log} dt} S + B (dt x)^T,  y = S^T C + D x,  dt = softplus(u + dt_bias), S [N, P] fp32.
//
// Bound by latency and, with many sequences, by the states' bytes.  ssd_kernel gives a head to one wave, a column a lane: N loads of 256
// bytes each in a row and 64 to 128 registers of state.  Here a workgroup of four waves takes a head, a thread four columns of N P
// / 1024 rows through 16-byte accesses, all in flight at once, and the sums over rows meet by shuffles and once in LDS.
// us, one wave / this: 16 heads of 64 x 64, bf16, 2 tokens 12.8 / 4.0, 64 17.7 / 8.6 (3.9 TB/s, read and written), fp32, 2 tokens 7.8 / 4.0; 32
// heads of 128 x 64, bf16, 2 tokens 25.9 / 4.3, 64 80 / 30.
#include "common.h"
#include "seqmix/seqmix_common.h"

namespace {

struct SsdStep {
  const void *xbc, *u;
  const float *dt_bias, *A_log, *D;
  float *state, *y;                                          // state [slots, H, N, P]; y [rows, H P]
  const int *seq_slot, *seq_start, *seq_off;
  int Cx, ld, dt0, H, groups;
};

template <typename T, int N, int P>
__global__ void __launch_bounds__(NT) ssd_step_kernel(SsdStep a) {
  constexpr int PG = P / 4, RGS = NT / PG, NR = N / RGS, NW = NT / 64;
  static_assert(P % 4 == 0 && PG <= 64 && 64 % PG == 0 && N % RGS == 0, "shape");
  __shared__ __attribute__((aligned(16))) float sum_s[NW][P];
  // the wave's number as a scalar: conditions and addresses that depend on it alone take the scalar unit (13-layer
  // step 6.85 -> 6.79 ms with the kernels beside it)
  const int s = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
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

template <typename T>
int run(const SsdStep& a, int n, int N, int P, hipStream_t st) {
#define SS(NN, PP)                                                                          \
  if (N == NN && P == PP) {                                                                 \
    hipLaunchKernelGGL((ssd_step_kernel<T, NN, PP>), dim3(n, a.H), dim3(NT), 0, st, a);     \
    return (int)hipGetLastError();                                                          \
  }
  SS(64, 64)
  SS(128, 64)
  SS(64, 128)
  SS(128, 128)
#undef SS
  return -2;
}

}  // namespace

// -2: not this kernel's (states of other sizes, rows that do not lie on 16 bytes)
extern "C" int edge_sm_ssd_step(const void* xbc, int Cx, const void* u, int ld, int dt0, const float* dt_bias, const float* A_log,
                                const float* D, float* state, const int* seq_slot, const int* seq_start, const int* seq_off, float* y,
                                int n, int H, int P, int N, int groups, int f32, hipStream_t st) {
  if (((uintptr_t)xbc | (uintptr_t)state) % 16 || Cx % 8 || groups < 1 || H < 1 || H % groups) return -2;
  const SsdStep a{xbc, u, dt_bias, A_log, D, state, y, seq_slot, seq_start, seq_off, Cx, ld, dt0, H, groups};
  return f32 ? run<float>(a, n, N, P, st) : run<bf16_t>(a, n, N, P, st);
}
