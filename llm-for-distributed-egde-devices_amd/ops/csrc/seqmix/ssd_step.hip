// One token per sequence through the state-space recurrence (ssd_kernel's and its rounding, seqmix.hip):
//   S <- e^{-e^{A_log} dt} S + B (dt x)^T,  y = S^T C + D x,  dt = softplus(u + dt_bias), S [N, P] fp32.
//
// Bound by latency and, with many sequences, by the states' bytes.  ssd_kernel gives a head to one wave, a column a lane: N loads of 256
// bytes each in a row and 64 to 128 registers of state.  Here a workgroup of four waves takes a head, a thread four columns of N P
// / 1024 rows through 16-byte accesses, all in flight at once, and the sums over rows meet by shuffles and once in LDS.
// us, one wave / this: 16 heads of 64 x 64, bf16, 2 tokens 12.8 / 4.0, 64 17.7 / 8.6 (3.9 TB/s, read and written), fp32, 2 tokens 7.8 / 4.0; 32
// heads of 128 x 64, bf16, 2 tokens 25.9 / 4.3, 64 80 / 30.
#include "common.h"
#include "seqmix/ssd_step.h"

namespace {

template <typename T, int N, int P>
__global__ void __launch_bounds__(NT) ssd_step_kernel(SsdStep a) {
  __shared__ __attribute__((aligned(16))) float sum_s[NT / 64][P];
  ssd_step_body<T, N, P>(a, blockIdx.x, blockIdx.y, threadIdx.x, sum_s);
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
