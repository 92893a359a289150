// fp32 projection of a few rows: y[M, N] = x[M, K] . W[N, K]^T (+ bias), M <= 8, K % 4 == 0, in fp32 throughout.
// Bound by reading W once, and below some 16 MB by the launch itself.  W stays in its [N, K] layout (no copy is made): a
// wave takes R rows by 256 k at a time, each load one contiguous KiB of a row (with 16 rows by 16 k per load, the matrix
// instruction's layout, the loads themselves were the bound: 1024 x 4096, launched one by one, 12.8 us against 5.9 here), the next 256 k on
// their way meanwhile: the loop's loads stand under no guard (one that may not run is moved behind the products before it), and
// nothing past the end is loaded, so the last two 256 k are taken behind it.  Few rows: KW waves of a workgroup share a row's k (until about 2048 waves are at work: us at 1 row, 1024 / 2048 / 4096 waves,
// 4096 x 1024 5.8 / 4.9 / 5.0, 7840 x 1024 8.4 / 7.7 / 7.2, 8192 x 2048 13.3 / 13.3 / 14.0, 2048 x 8192 14.9 / 12.5 / 12.5) and add up
// through LDS.  All sums in a fixed order.
// N x K at 2 rows in a graph, weights from memory, us, loads past the end / guarded behind a fence / now: 384 x 1024 3.3 / 2.8 / 2.7, 1024 x
// 4096 5.9 / 5.5 / 5.3, 4096 x 1024 6.2 / 5.6 / 5.4, 7840 x 1024 9.3 / 8.6 / 8.0, 8192 x 2048 14.9 / 15.1 / 14.6, 2048 x 8192 14.6 / 13.7 / 13.1, 32000 x
// 1024 25.6 / 26.9 / 25.7 (5.1 TB/s); relative error against 64-bit sums 1e-7 here, 2 to 8e-7 in the library's product.
#include "common.h"

namespace {

// A gated norm in front of a projection: its input is x silu(z) / rms(x silu(z)) * w over the whole row.
struct Gate {
  const float* z;       // [M, K], rows ld apart
  const float* w;       // [K]
  int ld;
  float eps;
};

// GATED: the waves that share a row's k read all of it between them, so the row's sum of squares costs no load: they sum x silu(z) w
// times the weights, and the sums are divided by the root mean square at the end (a launch of its own for the norm was 4.7 us of the
// 37.7 that a layer's step of 2 rows, 1024 wide, took; this launch 7.4 us without and 7.5 with it).
template <int MV, int R, bool GATED = false>
__device__ __forceinline__ void gemv_f32_body(int bid, const float* __restrict__ x, const float* __restrict__ W,
                                              const float* __restrict__ bias, float* __restrict__ y, int M, int N, int K, int KW,
                                              const Gate& g = Gate{}) {
  constexpr int V = MV * R;
  __shared__ float part[16 * V];
  __shared__ float sqs[GATED ? 16 * MV : 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  const int rg = wave / KW, kw = wave - rg * KW, n0 = (bid * (waves / KW) + rg) * R;
  const int C = (K + 255) / 256;
  float acc[V];
#pragma unroll
  for (int i = 0; i < V; ++i) acc[i] = 0.f;
  v4f wv[2][R], xv[2][MV], zv[GATED ? 2 : 1][MV], gv[GATED ? 2 : 1];
  float sq[MV];
#pragma unroll
  for (int m = 0; m < MV; ++m) sq[m] = 0.f;
  auto load = [&](int b, int c) {                            // rows past the last and k past the end: a clamped one
    const int k = min(min(c, C - 1) * 256 + lane * 4, K - 4);
#pragma unroll
    for (int r = 0; r < R; ++r) wv[b][r] = *reinterpret_cast<const v4f*>(W + (size_t)min(n0 + r, N - 1) * K + k);
#pragma unroll
    for (int m = 0; m < MV; ++m) xv[b][m] = *reinterpret_cast<const v4f*>(x + (size_t)min(m, M - 1) * K + k);
    if constexpr (GATED) {
#pragma unroll
      for (int m = 0; m < MV; ++m) zv[b][m] = *reinterpret_cast<const v4f*>(g.z + (size_t)min(m, M - 1) * g.ld + k);
      gv[b] = *reinterpret_cast<const v4f*>(g.w + k);
    }
  };
  auto use = [&](int b, int c) {
    if (c * 256 + lane * 4 >= K) return;
    if constexpr (GATED) {
#pragma unroll
      for (int m = 0; m < MV; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float v = xv[b][m][j] * (zv[b][m][j] * (1.f / (1.f + expf(-zv[b][m][j]))));
          sq[m] = __builtin_fmaf(v, v, sq[m]);
          xv[b][m][j] = v * gv[b][j];
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int m = 0; m < MV; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[r * MV + m] = __builtin_fmaf(wv[b][r][j], xv[b][m][j], acc[r * MV + m]);
  };
  int c = kw;
  if (c < C) load(0, c);
  for (; c + 2 * KW < C; c += 2 * KW) {
    load(1, c + KW);
    use(0, c);
    load(0, c + 2 * KW);
    use(1, c + KW);
  }
  if (c + KW < C) load(1, c + KW);
  if (c < C) use(0, c);
  if (c + KW < C) use(1, c + KW);
  int idx = 0;
  lane_sums<V, 32>(acc, idx, lane);
  // the first bits of the lane number chose; lanes that differ only in the others hold the same sum
  static_assert(V <= 64, "one sum per lane");
  if (lane % (64 / V) == 0) part[wave * V + idx] = acc[0];
  if constexpr (GATED) {
#pragma unroll
    for (int m = 0; m < MV; ++m) {
      sq[m] = wave_sum(sq[m]);
      if (lane == 0) sqs[wave * MV + m] = sq[m];
    }
  }
  __syncthreads();
  for (int e = tid; e < waves / KW * V; e += blockDim.x) {
    const int gq = e / V, v = e - gq * V, m = v % MV, n = (bid * (waves / KW) + gq) * R + v / MV;
    float sum = 0.f;
    for (int w = 0; w < KW; ++w) sum += part[(gq * KW + w) * V + v];
    if constexpr (GATED) {
      float s2 = 0.f;
      for (int w = 0; w < KW; ++w) s2 += sqs[(gq * KW + w) * MV + m];
      sum *= 1.f / sqrtf(s2 / (float)K + g.eps);
    }
    if (m < M && n < N) y[(size_t)m * N + n] = sum + (bias ? bias[n] : 0.f);
  }
}

template <int MV, int R>
__global__ void __launch_bounds__(1024) gemv_f32_kernel(const float* __restrict__ x, const float* __restrict__ W,
                                                        const float* __restrict__ bias, float* __restrict__ y, int M, int N,
                                                        int K, int KW) {
  gemv_f32_body<MV, R>(blockIdx.x, x, W, bias, y, M, N, K, KW);
}

// three projections of M rows each, workgroups [0, n[0]), [n[0], n[1]), [n[1], ..) of the grid
struct Jobs3 {
  const float *x[3], *W[3];
  float* y[3];
  int N[3], K[3], KW[3], n[2];
};
// RG > 0: the last one's input is gated and normed, RG weight rows a wave (four at 4 rows spilled: 36 bytes a lane)
template <int MV, int R, int RG>
__global__ void __launch_bounds__(1024) gemv_f32x3_kernel(Jobs3 a, int M, Gate g) {
  const int bid = blockIdx.x, j = bid < a.n[0] ? 0 : bid < a.n[1] ? 1 : 2;
  if constexpr (RG > 0)
    if (j == 2) return gemv_f32_body<MV, RG, true>(bid - a.n[1], a.x[2], a.W[2], nullptr, a.y[2], M, a.N[2], a.K[2], a.KW[2], g);
  gemv_f32_body<MV, R>(bid - (j == 0 ? 0 : a.n[j - 1]), a.x[j], a.W[j], nullptr, a.y[j], M, a.N[j], a.K[j], a.KW[j]);
}

// waves of a workgroup that share a row's k
int share_k(int groups, int K) {
  const int C = (K + 255) / 256;
  int KW = 1;
  while (KW < 16 && KW * 2 <= C && groups * KW < 2048) KW *= 2;
  return KW;
}

template <int MV, int R>
void launch_f32(const float* x, const float* W, const float* bias, float* y, int M, int N, int K, hipStream_t st) {
  const int groups = (N + R - 1) / R, KW = share_k(groups, K);
  const int waves = KW < 4 ? 4 : KW, per = waves / KW;
  hipLaunchKernelGGL((gemv_f32_kernel<MV, R>), dim3((groups + per - 1) / per), dim3(waves * 64), 0, st, x, W, bias, y, M, N, K, KW);
}

template <int MV, int R, int RG>
void launch_f32x3(Jobs3 a, int M, const Gate& g, hipStream_t st) {
  int waves = 4, blocks = 0;
  auto rows = [](int j) { return j == 2 && RG > 0 ? RG : R; };
  for (int j = 0; j < 3; ++j) {
    a.KW[j] = share_k((a.N[j] + rows(j) - 1) / rows(j), a.K[j]);
    waves = a.KW[j] > waves ? a.KW[j] : waves;
  }
  for (int j = 0; j < 3; ++j) {
    const int per = waves / a.KW[j];
    blocks += ((a.N[j] + rows(j) - 1) / rows(j) + per - 1) / per;
    if (j < 2) a.n[j] = blocks;
  }
  hipLaunchKernelGGL((gemv_f32x3_kernel<MV, R, RG>), dim3(blocks), dim3(waves * 64), 0, st, a, M, g);
}
}  // namespace

// y_j = x_j W_j^T for three projections of the same M rows' inputs, each as edge_gemv_f32 forms it: a parallel layer's three output
// projections, whose launches' ramps and ends then overlap.  us in a graph, weights from memory, three launches / one, 1024 x 4096 and
// twice 1024 x 1024: 1 row 11.1 / 6.8, 2 11.5 / 7.0, 8 15.1 / 11.4; 2048 x 8192 and twice 2048 x 2048, 2 rows 24.0 / 18.8
// gate_z (null: none; up to 4 rows): x_2 is gated by its rows, z_ld apart, and normed under gate_w first; 16-byte aligned, z_ld % 4 == 0
extern "C" int edge_gemv_f32x3(const float* const* x, const float* const* W, float* const* y, int M, const int* N, const int* K,
                               const float* gate_z, int z_ld, const float* gate_w, float eps, hipStream_t st) {
  const Gate g{gate_z, gate_w, z_ld, eps};
  if (gate_z != nullptr && (gate_w == nullptr || z_ld % 4)) return -2;
  Jobs3 a{};
  for (int j = 0; j < 3; ++j) {
    if (N[j] < 1 || K[j] < 4 || K[j] % 4) return -2;
    a.x[j] = x[j]; a.W[j] = W[j]; a.y[j] = y[j]; a.N[j] = N[j]; a.K[j] = K[j];
  }
  if (M < 1 || M > (gate_z ? 4 : 8)) return -2;
  if (gate_z != nullptr) {
    if (M == 1) launch_f32x3<1, 4, 4>(a, M, g, st);
    else if (M == 2) launch_f32x3<2, 4, 4>(a, M, g, st);
    else launch_f32x3<4, 4, 2>(a, M, g, st);
  } else if (M == 1) launch_f32x3<1, 4, 0>(a, M, g, st);
  else if (M == 2) launch_f32x3<2, 4, 0>(a, M, g, st);
  else if (M <= 4) launch_f32x3<4, 4, 0>(a, M, g, st);
  else launch_f32x3<8, 2, 0>(a, M, g, st);
  return (int)hipGetLastError();
}

// x, W: 16-byte aligned.  5 - 8 rows: two weight rows per wave (four leave no registers for the next loads: 4096 x 1024 at
// 8 rows, launched one by one, 13.7 us, two 7.9, library 11.6)
extern "C" int edge_gemv_f32(const float* x, const float* W, const float* bias, float* y, int M, int N, int K,
                             hipStream_t st) {
  if (M < 1 || M > 8 || N < 1 || K < 4 || K % 4) return -2;
  if (M == 1) launch_f32<1, 4>(x, W, bias, y, M, N, K, st);
  else if (M == 2) launch_f32<2, 4>(x, W, bias, y, M, N, K, st);
  else if (M <= 4) launch_f32<4, 4>(x, W, bias, y, M, N, K, st);
  else launch_f32<8, 2>(x, W, bias, y, M, N, K, st);
  return (int)hipGetLastError();
}
