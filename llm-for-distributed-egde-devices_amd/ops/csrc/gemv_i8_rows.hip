// Split-K W8A8 decode GEMV of up to 16 rows with one scale per (row, 64 numbers): the o and down projections before an RMSNorm
// that adds their fp32 slices.  One 16-column tile and one part of K a workgroup; operands lie as gemm_i8.h says.
// What bounds it is the chain around the weights: a memory round trip, the sums over the waves, the launch.  So 16 waves split
// the part, a wave's k-tiles are requested in pairs ahead of their products (behind a fence: the compiler sinks loads under the
// guards of ragged ends otherwise), a wave holds one tile's numbers, so that two workgroups fit a CU, and only the lanes of the
// rows that exist meet in the LDS: RB groups of four rows are number quadruples of 16 RB lanes, and the 64 lanes of one wave
// each add up 4 RB waves' sums.  us in a graph, weights from memory, against two tiles a workgroup: one row 4096 x 4096
// 5.5 -> 5.1, 4096 x 11008 10.9 -> 9.7, 4096 x 14336 12.9 -> 11.5, 2048 x 8192 5.5 -> 5.1.
#include <algorithm>

#include "gemm_i8.h"

namespace {
constexpr int RW = 16, PRE = 2;            // waves, k-tiles of a wave's in flight

template <int RB>
__global__ void __launch_bounds__(RW * 64) w8a8_rows_kernel(const int8_t* __restrict__ A, const float* __restrict__ sa,
                                                           const int8_t* __restrict__ Wp, const float* __restrict__ sw,
                                                           const bf16_t* __restrict__ bias, float* __restrict__ part, int M,
                                                           int N, int K, int Mpad, int S) {
  constexpr int RL = 16 * RB, WG = 4 / RB;                  // lanes of a wave's rows, waves that a wave adds up side by side
  __shared__ v4f red[RW][RL];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15;
  const int KT = K / 64, tile = blockIdx.x / S, ks = blockIdx.x % S, kend = (int)((int64_t)KT * (ks + 1) / S);
  const v4i* wp = reinterpret_cast<const v4i*>(Wp + (size_t)tile * KT * 1024) + lane;
  const int8_t* ar = A + (size_t)min(r, M - 1) * K + 16 * (lane >> 4);
  const float* sr = sa + (RB == 1 ? 0 : 4 * (lane >> 4));   // (RB 1: only lanes 0 .. 15 hold rows that exist)
  const int c = 16 * tile + r;
  float wsc = 0.f, bv = 0.f;                                // what the writing wave needs is requested with its first weights
  if (wave == 0) {
    wsc = sw[c];
    if (bias != nullptr && ks == 0) bv = bf2f(bias[c]);
  }
  v4f acc = {0.f, 0.f, 0.f, 0.f};
  for (int kt = (int)((int64_t)KT * ks / S) + wave; kt < kend; kt += RW * PRE) {
    v4i b[PRE], a[PRE];
    v4f s[PRE];
#pragma unroll
    for (int u = 0; u < PRE; ++u) {                         // clamped: loads never branch
      const int k = min(kt + RW * u, kend - 1);
      b[u] = __builtin_nontemporal_load(wp + (size_t)k * 64);
      a[u] = *reinterpret_cast<const v4i*>(ar + (size_t)k * 64);
      s[u] = *reinterpret_cast<const v4f*>(sr + (size_t)k * Mpad);
    }
    asm volatile("" ::: "memory");
#pragma unroll
    for (int u = 0; u < PRE; ++u)
      if (kt + RW * u < kend) fold(acc, mfma_i8(a[u], b[u], v4i{0, 0, 0, 0}), s[u]);   // wave-uniform (scalar) guard
  }
  if (RB == 4 || lane < RL) red[wave][lane & (RL - 1)] = acc;
  __syncthreads();
  if (wave == 0) {
    v4f s = red[lane / RL][lane & (RL - 1)];
#pragma unroll
    for (int w = 1; w < RW / WG; ++w) s += red[WG * w + lane / RL][lane & (RL - 1)];
    const int row0 = RB == 1 ? 0 : 4 * (lane >> 4);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float v = s[q];
      if constexpr (RB == 1) v = xor_sum(v, 16);
      if constexpr (RB <= 2) v = xor_sum(v, 32);
      if ((RB == 4 || lane < RL) && row0 + q < M) part[((size_t)ks * M + row0 + q) * N + c] = v * wsc + bv;
    }
  }
}
}  // namespace

// Slices of K for M rows (S > 0: that many are asked for): two workgroups a CU, each wave a k-tile or more; us at S = 1 / 2 / 4, one
// row: 4096 x 4096 5.4 / 5.2 / 6.3, 4096 x 11008 11.1 / 9.9 / 10.7, 2048 x 2048 3.7 / 3.2 / 3.4, 2048 x 8192 7.9 / 5.4 / 5.1.  0 where gemm_i8.hip's two tiles a workgroup are quicker: every tile reads all the rows and their scales, beside up to 4 rows no matter
// and below 16 MB of weights less than the shorter chain gives, else some 8 to 30 % unless two tiles leave CUs idle in a last round.
// us, two tiles / one: 5 rows 4096 x 4096 5.9 / 5.8, 4096 x 11008 11.5 / 12.0, 8192 x 8192 13.9 / 15.2, 8192 x 28672 37 / 46, 5120 x 13824 19.4 / 16.8; 16
// rows 6.4 / 6.4, 12.1 / 13.0, 15.1 / 17.5, 43 / 56, 22.8 / 20.1.
extern "C" int edge_w8a8_rows_splits(int M, int N, int K, int S) {
  const int64_t tiles = N / 16, KT = K / 64;
  if (M < 1 || M > 16 || N < 16 || N % 16 != 0 || K < 64 || K % 64 != 0 || S > KT) return 0;
  const int64_t one = S > 0 ? S : std::max<int64_t>(1, std::min<int64_t>({4, (512 + tiles / 2) / tiles, KT / 16}));
  if (M <= 4 || (int64_t)N * K <= 1 << 24) return (int)one;
  const int64_t groups = (tiles + 1) / 2, two = S > 0 ? S : std::max<int64_t>(1, std::min<int64_t>({8, (256 + groups / 2) / groups, KT}));
  // tiles' passes over all of K that the busiest CU has to do
  const double t1 = (double)((tiles * one + 255) / 256) / one, t2 = 2. * ((groups * two + 255) / 256) / two;
  return 1.25 * t1 < t2 ? (int)one : 0;
}

// part [S, M, N] (bias in slice 0): M <= 16 int8 rows A [M, K] with scales sa [K / 64][Mpad].  -2: not taken.
extern "C" int edge_w8a8_rows_splitk(const void* A, const float* sa, const void* Wp, const float* sw, const void* bias, float* part,
                                     int M, int N, int K, int Mpad, int S, hipStream_t st) {
  if (S < 1 || Mpad < 16 || edge_w8a8_rows_splits(M, N, K, S) != S) return -2;
  const dim3 grid(N / 16 * S), block(RW * 64);
#define ROWS(RB)                                                                                                       \
  hipLaunchKernelGGL(w8a8_rows_kernel<RB>, grid, block, 0, st, (const int8_t*)A, sa, (const int8_t*)Wp, sw, (const bf16_t*)bias, \
                     part, M, N, K, Mpad, S)
  if (M <= 4) ROWS(1);
  else if (M <= 8) ROWS(2);
  else ROWS(4);
#undef ROWS
  return (int)hipGetLastError();
}
