// Two independent parts of a parallel-residual block (GPT-NeoX, Phi) in one launch of a 16-bit decode step, up to 4 rows:
//   * attention beside the MLP's up projection (both need only the qkv launch's results);
//   * the o projection beside the down projection, each into rows of its own (the next layer's norm adds them up).
// What bounds a step of such a layer is not its bytes but the launches: each costs some 3.3 us of ramp, first loads and
// reduction beside the time of its weights, and the attention's 5 us leave the memory idle.  Five launches a layer are
// three this way.  The workgroups are the parts' own (attn_decode.h, gemv_bf16.h), one tile of 16 columns each, beside the
// attention with 8 waves instead of 16: two to a CU under 128 VGPRs, so that the attention's workgroups take no CU away from
// the projection (with 16 waves 9.1 -> 10.7 us).  The attention's come first in the grid: they are the longest chains.  us a
// layer, fp16, one row, before the projections requested all of a step's weights at once and now: Pythia-1B attention with up
// 10.3 -> 9.1, o with down 10.9 -> 9.3; Phi-2 o with down 14.7 (8 waves) -> 13.5.
// Whole answers against five launches, one row: Pythia-1B 48 tokens 33.9 -> 26.9 ms.
#include "decode_pair.h"
#include "gemv_bf16.h"

namespace {
struct Proj {
  const bf16_t *x, *w, *bias;              // rows [M, K], packed weights, bias [N] or null
  bf16_t* out;
  int N, K;
};

constexpr int OW = GEMV_NW;                // waves of an o or down workgroup

// One workgroup of a projection, a round's loads ahead of its products.  8 waves: 5 or 4 k-pairs of a wave a round where they divide its
// rounds evenly (a round that runs over the end loads its last k-pair again), else 2.  Eight pairs of weights and rows are 128
// registers by themselves: under the bound of two workgroups a CU they spill, us with 8 / 4: attention beside 16384 x 4096, 1 row
// 32.4 / 25.5, 4 rows 36.9 / 26.2; rows3 1024 x 4096 and twice 1024 x 1024, 1 row 6.3 / 5.5, 2048 x 8192 and twice 2048 x 2048 12.5 / 11.6.
// 16 waves: 5 where that divides the rounds, else 1 (2048 x 8192 beside 2048 x 2048 9.3 us, with 8 in flight 11.4).
template <int NWV, int EPI, bool HF>
__device__ __forceinline__ void proj_body(int bid, const Proj& p, int M, int act) {
  const int KP = p.K / 64;
  const NormIn16 none{};
#define RUN(UU, PP) gemv_tiles_body<NWV, UU, PP, EPI, HF, 0, 1>(bid, 1 << 30, p.x, p.w, p.bias, p.out, M, p.N, p.K, act, 1, nullptr, none)
  if constexpr (NWV == GEMV_NW) {
    if (KP % (5 * NWV) == 0) RUN(5, 0);
    else RUN(1, 1);
  } else {
    if (KP % (5 * NWV) == 0) RUN(5, 0);
    else if (KP % (4 * NWV) == 0) RUN(4, 0);
    else RUN(2, 0);
  }
#undef RUN
}

// Three projections of the same rows (a parallel layer of attention, recurrence and feed-forward); d first, its chains are the
// longest.  us in a graph, bf16, three launches / one, 1024 x 4096 and twice 1024 x 1024: 1 row 13.1 / 6.5, 4 rows 14.1 / 7.1; 2048 x
// 8192 and twice 2048 x 2048 19.8 / 12.3, 22.7 / 14.7.
template <bool HF>
__global__ void __launch_bounds__(PW * 64, 4) rows3_kernel(Proj d, Proj o, Proj r, int M) {
  const int nd = d.N / 16, no = nd + o.N / 16, bid = blockIdx.x;
  proj_body<PW, EPI_OUT, HF>(bid < nd ? bid : bid < no ? bid - nd : bid - no, bid < nd ? d : bid < no ? o : r, M, 0);
}

template <int D, bool DIRECT, bool HF>
__global__ void __launch_bounds__(PW * 64, 4) attn_up_kernel(AttnArgs a, Proj p, int M, int act, int na) {
  __shared__ __attribute__((aligned(16))) float smem[attn_part_lds<D>()];
  const int bid = blockIdx.x;
  if (bid < na) {
    attn_part<D, DIRECT, HF>(smem, bid, a);
  } else {
    proj_body<PW, EPI_GELU_ANY, HF>(bid - na, p, M, act);
  }
}

// The down projection's workgroups first: their chains are the longer ones.
template <bool HF>
__global__ void __launch_bounds__(OW * 64) o_down_kernel(Proj o, Proj d, int M) {
  const int nd = d.N / 16, bid = blockIdx.x;
  const bool down = bid < nd;
  proj_body<OW, EPI_OUT, HF>(down ? bid : bid - nd, down ? d : o, M, 0);
}

template <bool HF>
int run_attn_up(const AttnArgs& a, const Proj& p, int B, int D, int act, hipStream_t st) {
  const int na = a.nsplit * a.ny * B;
  const dim3 grid(na + p.N / 16), block(PW * 64);
#define AU(DD)                                                                                                   \
  if (a.nsplit == 1) hipLaunchKernelGGL((attn_up_kernel<DD, true, HF>), grid, block, 0, st, a, p, B, act, na);    \
  else hipLaunchKernelGGL((attn_up_kernel<DD, false, HF>), grid, block, 0, st, a, p, B, act, na);                 \
  break
  switch (D) {
    case 64: AU(64);
    case 80: AU(80);
    case 128: AU(128);
    case 256: AU(256);
    default: return -2;
  }
#undef AU
  return (int)hipGetLastError();
}
}  // namespace

// edge_decode_attn's FUSED form (B <= 4 rows, 16-bit output, every query head a workgroup of its own) beside
// h = gelu(y . Wup^T + bias) of the B rows y [B, K]: act 1 tanh, 0 erf.  -2: not taken.
extern "C" int edge_attn_up(const void* qkv, int64_t q_sb, void* kc, void* vc, int64_t c_sb, int64_t c_sh, const int* seq_lens,
                            int B, int Hq, int Hkv, int D, float scale, int ch, int nsplit, void* out, int64_t o_sb,
                            float* part_acc, float* part_ml, const int* pos, const float* cs, int rot, const void* y,
                            const void* w, const void* bias, void* h, int N, int K, int act, int h16, hipStream_t st) {
  if (B < 1 || B > 4 || Hkv < 1 || Hq % Hkv != 0 || N <= 0 || N % 16 != 0 || K <= 0 || K % 64 != 0 || nsplit < 1) return -2;
  if (pos == nullptr || (rot > 0 && (cs == nullptr || rot % 16 != 0 || rot > D))) return -2;
  const AttnArgs a{(const bf16_t*)qkv, q_sb, (bf16_t*)kc, (bf16_t*)vc, c_sb, c_sh, seq_lens, scale * 1.4426950408889634f,
                   ch, nsplit, Hq, (bf16_t*)out, o_sb, part_acc, part_ml,
                   Fuse{pos, cs, rot, q_sb, nullptr, nullptr, 0, Hq / Hkv, 1}};
  const Proj p{(const bf16_t*)y, (const bf16_t*)w, (const bf16_t*)bias, (bf16_t*)h, N, K};
  const int r = h16 ? run_attn_up<true>(a, p, B, D, act, st) : run_attn_up<false>(a, p, B, D, act, st);
  if (r != 0 || nsplit == 1) return r;
  return edge_decode_attn_combine(part_acc, part_ml, nsplit, B, Hq, D, out, o_sb, h16, st);
}

// a = x . Wo^T + bo (x [M, Ko]) beside y = h . Wd^T + bd (h [M, Kd]), M <= 4 rows of N numbers each.  -2: not taken.
extern "C" int edge_o_down(const void* x, const void* wo, const void* bo, void* a, int Ko, const void* h, const void* wd,
                           const void* bd, void* y, int Kd, int M, int N, int h16, hipStream_t st) {
  if (M < 1 || M > 4 || N <= 0 || N % 16 != 0 || Ko <= 0 || Ko % 64 != 0 || Kd <= 0 || Kd % 64 != 0) return -2;
  const Proj o{(const bf16_t*)x, (const bf16_t*)wo, (const bf16_t*)bo, (bf16_t*)a, N, Ko};
  const Proj d{(const bf16_t*)h, (const bf16_t*)wd, (const bf16_t*)bd, (bf16_t*)y, N, Kd};
  const dim3 grid(2 * (N / 16)), block(OW * 64);
  if (h16) hipLaunchKernelGGL(o_down_kernel<true>, grid, block, 0, st, o, d, M);
  else hipLaunchKernelGGL(o_down_kernel<false>, grid, block, 0, st, o, d, M);
  return (int)hipGetLastError();
}

// y_j = x_j . W_j^T (x_j [M, K_j], packed weights), M <= 4 rows of N_j numbers, j = 0 .. 2.  -2: not taken.
extern "C" int edge_rows3(const void* const* x, const void* const* w, void* const* y, const int* N, const int* K, int M, int h16,
                          hipStream_t st) {
  Proj p[3];
  int blocks = 0;
  for (int j = 0; j < 3; ++j) {
    if (N[j] <= 0 || N[j] % 16 != 0 || K[j] <= 0 || K[j] % 64 != 0) return -2;
    p[j] = Proj{(const bf16_t*)x[j], (const bf16_t*)w[j], nullptr, (bf16_t*)y[j], N[j], K[j]};
    blocks += N[j] / 16;
  }
  if (M < 1 || M > 4) return -2;
  if (h16) hipLaunchKernelGGL(rows3_kernel<true>, dim3(blocks), dim3(PW * 64), 0, st, p[0], p[1], p[2], M);
  else hipLaunchKernelGGL(rows3_kernel<false>, dim3(blocks), dim3(PW * 64), 0, st, p[0], p[1], p[2], M);
  return (int)hipGetLastError();
}
