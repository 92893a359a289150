// Experts of decode-sized steps: every (token, choice) pair's product with its expert's rows.
#pragma once
#include "common.h"
#include "seqmix/seqmix_common.h"

namespace {

constexpr int MR_GLU = 0, MR_PLAIN = 1, MR_RELU2 = 2;
constexpr int MR_MAX_PAIRS = 65535;                          // a grid's second dimension

// Pairs p < routed are (token, choice) of the routed experts, pairs after them one per token of the shared expert (own
// weights w_sh, widths K_sh -> R_sh).  MR_GLU: out = act(gate . x, up . x), weights [E, 2 R, K], rows of x per token; act =
// silu(rw g) (rw u) (silu, rw = in_w[pair] or 1) or the clamped form (limit; limit_sh for the shared expert).  MR_RELU2:
// out = max(W x, 0)^2, rows of x per token.  MR_PLAIN: out = W x, rows of x per pair.
// Bound by the chosen experts' weights.  A workgroup is (pair, 4 waves of 4 weight rows).  `share` (launch_moe_rows): pairs
// of one expert belong to the first of them (at most 64 routed pairs, so one ballot names them), which runs them together,
// up to four per reading of the rows; the others leave at once.  A wave has its four rows' next 1024 numbers (2048 for one
// pair) in flight as contiguous KiBs and the inputs beside them in registers; the sums over lanes end with one sum per lane.
// us for both launches, one wave per row and pair / this, bf16: 3 of 16 experts of 1024 x 1024, 1 token 11.1 / 7.4, 4 tokens
// 18.8 / 17.2, 9 29.4 / 24.1; 4 of 32 of 2048 x 2048 26.5 / 20.9, 74 / 62, 159 / 107 (5.4 TB/s).  fp32 only for one
// token (15.1 / 9.6): rows shared by several pairs need more registers than they save there (4 of 16 of 1024 x 1024,
// 6 tokens 48.6 / 54.7, 16 tokens 102 / 141).
// A grid's x dimension is the features: consecutive workgroups go to the eight dies in turn, and with the pairs there a count of 8,
// 16 or 24 pairs gave every expert to one die's 32 CUs (us, pairs first / features first: 4 of 32 experts of 2048 x 2048, 4 tokens
// 65.7 / 61.9, 6 88.0 / 74.9, 8 114 / 92.5 (5.4 TB/s); 4 of 16 of 1024 x 1024, 8 tokens 44.6 / 25.9; 2 of 8 of 512 x 520, 8 11.8 / 11.1).
template <typename T, int MODE, int MT, int CH>
__device__ __forceinline__ void moe_rows_run(const T* const (&wr)[4], const T* const (&xr)[MT], int K, float (&acc)[4 * MT]) {
  constexpr int Q = sizeof(T) / 2;                           // 16-byte loads per 8 numbers
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < 4 * MT; ++i) acc[i] = 0.f;
  for (int c0 = lane * 8; c0 < K + lane * 8; c0 += 512 * CH) {
    uint4 w[CH][4][Q], x[CH][MT][Q];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = min(c0 + 512 * i, K - 8);
#pragma unroll
      for (int q = 0; q < Q; ++q) {
#pragma unroll
        for (int r = 0; r < 4; ++r) w[i][r][q] = reinterpret_cast<const uint4*>(wr[r] + c)[q];
#pragma unroll
        for (int m = 0; m < MT; ++m) x[i][m][q] = reinterpret_cast<const uint4*>(xr[m] + c)[q];
      }
    }
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      if (c0 + 512 * i >= K) continue;
      float xf[MT][8];
#pragma unroll
      for (int m = 0; m < MT; ++m) load8<T>(reinterpret_cast<const T*>(&x[i][m][0]), xf[m]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float wf[8];
        load8<T>(reinterpret_cast<const T*>(&w[i][r][0]), wf);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[r * MT + m] += wf[e] * xf[m][e];
      }
    }
  }
}

template <typename T, int MODE>
__global__ void __launch_bounds__(NT) moe_rows_kernel(const T* __restrict__ in, const T* __restrict__ in_sh,
                                                      const int* __restrict__ idx, int routed, int pairs, int top,
                                                      const T* __restrict__ w, const T* __restrict__ w_sh, int K, int R, int K_sh,
                                                      int R_sh, int E, float limit, float limit_sh, int silu,
                                                      const float* __restrict__ in_w, T* __restrict__ out, T* __restrict__ out_sh,
                                                      int share) {
  constexpr int NF = MODE == MR_GLU ? 2 : 4;                 // output features of a wave
  const int pair = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool sh = pair >= routed;
  const int k = sh ? K_sh : K, n = sh ? R_sh : R, f0 = (blockIdx.x * (NT / 64) + wave) * NF;
  uint64_t mine = 1;                                         // pairs of this expert, from `first` on
  int first = pair;
  const T* we = w_sh;
  if (!sh) {
    const int e = min(max(idx[pair], 0), E - 1);
    we = w + (size_t)e * (MODE == MR_GLU ? 2 : 1) * R * K;
    if (share) {
      mine = __ballot(lane < routed && min(max(idx[min(lane, routed - 1)], 0), E - 1) == e);
      first = 0;
      if (__ffsll((unsigned long long)mine) - 1 != pair) return;
    }
  } else if (share) {
    if (pair != routed) return;
    const int rows = pairs - routed;
    mine = rows >= 64 ? ~0ull : (1ull << rows) - 1;
  }
  if (f0 >= n) return;
  const T* wr[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    wr[r] = we + (MODE == MR_GLU ? (size_t)(r >= 2 ? n : 0) + min(f0 + (r & 1), n - 1) : (size_t)min(f0 + r, n - 1)) * k;
  auto group = [&](auto mtc, auto chc) {
    constexpr int MT = decltype(mtc)::value, V = 4 * MT;
    int p[MT];
    const T* xr[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {                           // the next MT of them (the last one again past the end)
      p[m] = mine ? first + __ffsll((unsigned long long)mine) - 1 : p[m > 0 ? m - 1 : 0];
      mine &= mine - 1;
      xr[m] = sh ? in_sh + (size_t)(p[m] - routed) * k : in + (size_t)(MODE == MR_PLAIN ? p[m] : p[m] / top) * k;
    }
    float acc[V];
    moe_rows_run<T, MODE, MT, decltype(chc)::value>(wr, xr, k, acc);
    int id = 0;
    lane_sums<V, 32>(acc, id, lane);                         // lane (64 / V) v holds sum v = row MT + pair
    const float up = lane_xor(acc[0], 32);             // (GLU: the up row of a gate row, two rows on)
    const int m = id % MT, f = f0 + id / MT;
    int pm = p[0];
#pragma unroll
    for (int i = 1; i < MT; ++i) pm = m == i ? p[i] : pm;
    if (lane % (64 / V) == 0 && id / MT < NF && f < n) {
      float y = acc[0];
      if constexpr (MODE == MR_GLU) {
        const float rw = in_w && !sh ? in_w[pm] : 1.f;
        y = silu ? siluf_(rw * y) * (rw * up) : glu_clamp_f(y, up, sh ? limit_sh : limit);
      }
      if constexpr (MODE == MR_RELU2) { y = fmaxf(y, 0.f); y *= y; }
      stf<T>((sh ? out_sh + (size_t)(pm - routed) * n : out + (size_t)pm * n) + f, y);
    }
  };
  using std::integral_constant;
  while (mine) {
    const int left = __popcll(mine);
    if constexpr (sizeof(T) == 4) group(integral_constant<int, 1>{}, integral_constant<int, 2>{});
    else if (left == 1 && k > 1024) group(integral_constant<int, 1>{}, integral_constant<int, 4>{});
    else if (left == 1) group(integral_constant<int, 1>{}, integral_constant<int, 2>{});
    else if (left == 2) group(integral_constant<int, 2>{}, integral_constant<int, 2>{});
    else group(integral_constant<int, 4>{}, integral_constant<int, 2>{});
  }
}

// whether the kernel takes rows of these widths at these addresses
inline bool moe_rows_ok(int K, int K_sh, std::initializer_list<const void*> ps) {
  uintptr_t u = 0;
  for (const void* p : ps) u |= (uintptr_t)p;
  return K % 8 == 0 && K >= 8 && K_sh % 8 == 0 && u % 16 == 0;
}

template <typename T, int MODE>
void launch_moe_rows(const T* in, const T* in_sh, const int* idx, int routed, int pairs, int top, const T* w, const T* w_sh, int K,
                     int R, int K_sh, int R_sh, int E, float limit, float limit_sh, int silu, const float* in_w, T* out, T* out_sh,
                     hipStream_t st) {
  constexpr int FW = (MODE == MR_GLU ? 2 : 4) * (NT / 64);
  const int big = pairs > routed && R_sh > R ? R_sh : R;
  // Sharing pays where rows come from memory: an expert of a million numbers or more, and few tokens, for the expert's
  // pairs then run one group after another.  us for both launches, each pair for itself / shared: 2 of 8 experts of 512 x
  // 520, 16 tokens 9.9 / 17.8; 2 of 4 of 64 x 64, 9 tokens 6.5 / 12.8; 3 of 16 of 1024 x 1536, 9 tokens 27.8 / 20.8;
  // with a shared expert of 1024 x 1536 beside them, 9 tokens 42 / 36, 10 40.0 / 39.5, 16 49 / 92
  const int share = sizeof(T) == 2 && routed <= 64 && routed <= 12 * top && pairs - routed <= 12 &&
                    (int64_t)K * R * (MODE == MR_GLU ? 2 : 1) >= 1 << 20;
  hipLaunchKernelGGL((moe_rows_kernel<T, MODE>), dim3((big + FW - 1) / FW, pairs), dim3(NT), 0, st, in, in_sh, idx, routed, pairs,
                     top, w, w_sh, K, R, K_sh, R_sh, E, limit, limit_sh, silu, in_w, out, out_sh, share);
}

}  // namespace
