// decode_pair.hip's launches for LLM.int8 at batch 1: attention beside up, o beside down.  Each projection keeps its own
// preparation (outlier ranking and quantisation of its row) in front of its weights; side by side the
// preparations of two overlap, and the attention's reads hide behind up's.  8 waves a workgroup, two workgroups to a CU.
// us a layer of Phi-2: attention 5.7 and up 9.1 are 8.3 together, o 6.0 and down 10.2 are 8.1 (9.7 and 11.1 while 256 threads
// prepared the row); whole answers against separate launches: Phi-2 32 tokens 47.8 -> 33.6 ms.
#include "decode_pair.h"
#include "gemv_i8.h"

namespace {
struct Proj8 {
  const int8_t* w;
  const float* sw;
  const bf16_t* bias;
  bf16_t* out;
  int N, K;
  NormIn in;                               // row, threshold, W^T, SCB, activation
};

template <int NTW, int U, int NRM>
__device__ __forceinline__ void proj8_body(int bid, const Proj8& p) {
  w8a8_gemv_body<1, NTW, 1, PW, U, A_TOKEN, EPI_OUT, NRM>(bid, nullptr, nullptr, p.w, p.sw, p.bias, p.out, nullptr, 1, p.N, p.K,
                                                         p.K / 64, p.N / 16, 16, 1, p.in);
}

// NCH: up's row in chunks of 2048; two tiles a workgroup (640 tiles of Phi-2 beside 32 heads are one round of the chip).
// 5 k-tiles in flight per wave: all of Phi-2's 2560.
template <int D, bool DIRECT, int NCH>
__global__ void __launch_bounds__(PW * 64, 4) l8_attn_up_kernel(AttnArgs a, Proj8 p, int na) {
  __shared__ __attribute__((aligned(16))) float smem[attn_part_lds<D>()];
  const int bid = blockIdx.x;
  if (bid < na) {
    attn_part<D, DIRECT, false>(smem, bid, a);
  } else {
    proj8_body<2, NCH == 1 ? 4 : 5, 384 + 8 * NCH>(bid - na, p);
  }
}

// The down projection's workgroups first: their chains are the longer ones.
template <int NCO, int NCD>
__global__ void __launch_bounds__(PW * 64, 4) l8_o_down_kernel(Proj8 o, Proj8 d) {
  const int nd = d.N / 16, bid = blockIdx.x;
  if (bid < nd) proj8_body<1, 5, 128 + 8 * NCD>(bid, d);
  else proj8_body<1, NCO == 1 ? 4 : 5, 128 + 8 * NCO>(bid - nd, o);
}

Proj8 proj8(const void* x, float thr, const void* w, const float* sw, const void* bias, const void* wt, const float* scb, void* out,
            int N, int K, int act) {
  Proj8 p{(const int8_t*)w, sw, (const bf16_t*)bias, (bf16_t*)out, N, K, NormIn{}};
  p.in.x = (const bf16_t*)x;
  p.in.thr = thr;
  p.in.wt = (const int8_t*)wt;
  p.in.scb = scb;
  p.in.act = act;
  return p;
}
}  // namespace

// edge_decode_attn's FUSED form (one bf16 row, every query head a workgroup of its own) beside h = gelu(up) of the row y [K]
// as edge_llmint8_gemv computes it: act 1 tanh, 2 erf.  K <= 4096.  -2: not taken.
extern "C" int edge_llmint8_attn_up(const void* qkv, int64_t q_sb, void* kc, void* vc, int64_t c_sb, int64_t c_sh,
                                    const int* seq_lens, int Hq, int Hkv, int D, float scale, int ch, int nsplit, void* out,
                                    float* part_acc, float* part_ml, const int* pos, const float* cs, int rot, const void* y,
                                    float thr, const void* w, const float* sw, const void* bias, const void* wt, const float* scb,
                                    void* h, int N, int K, int act, hipStream_t st) {
  if (Hkv < 1 || Hq % Hkv != 0 || N <= 0 || N % 16 != 0 || K < 64 || K > 4096 || K % 64 != 0 || nsplit < 1) return -2;
  if (pos == nullptr || (rot > 0 && (cs == nullptr || rot % 16 != 0 || rot > D)) || (act != 1 && act != 2)) return -2;
  const AttnArgs a{(const bf16_t*)qkv, q_sb, (bf16_t*)kc, (bf16_t*)vc, c_sb, c_sh, seq_lens, scale * 1.4426950408889634f,
                   ch, nsplit, Hq, (bf16_t*)out, Hq * D, part_acc, part_ml,
                   Fuse{pos, cs, rot, q_sb, nullptr, nullptr, 0, Hq / Hkv, 1}};
  const Proj8 p = proj8(y, thr, w, sw, bias, wt, scb, h, N, K, act);
  const int na = nsplit * Hq;
  const dim3 grid(na + (N / 16 + 1) / 2), block(PW * 64);
#define AU(DD, DI)                                                                                       \
  if (K <= 2048) hipLaunchKernelGGL((l8_attn_up_kernel<DD, DI, 1>), grid, block, 0, st, a, p, na);        \
  else hipLaunchKernelGGL((l8_attn_up_kernel<DD, DI, 2>), grid, block, 0, st, a, p, na);
#define AUD(DD)                       \
  if (nsplit == 1) { AU(DD, true) }   \
  else { AU(DD, false) }              \
  break
  switch (D) {
    case 64: AUD(64);
    case 80: AUD(80);
    case 128: AUD(128);
    case 256: AUD(256);
    default: return -2;
  }
#undef AUD
#undef AU
  const int r = (int)hipGetLastError();
  if (r != 0 || nsplit == 1) return r;
  return edge_decode_attn_combine(part_acc, part_ml, nsplit, 1, Hq, D, out, Hq * D, 0, st);
}

// a = o(x) beside y = down(h), both as edge_llmint8_gemv computes them, one row of N numbers each: Ko <= 4096 < Kd <= 12288.
// -2: not taken.
extern "C" int edge_llmint8_o_down(const void* x, float thr_o, const void* wo, const float* swo, const void* bo, const void* wto,
                                   const float* scbo, void* a, int Ko, const void* h, float thr_d, const void* wd,
                                   const float* swd, const void* bd, const void* wtd, const float* scbd, void* y, int Kd, int N,
                                   hipStream_t st) {
  if (N <= 0 || N % 16 != 0 || Ko < 64 || Ko > 4096 || Ko % 64 != 0 || Kd <= 4096 || Kd > 12288 || Kd % 64 != 0) return -2;
  const Proj8 o = proj8(x, thr_o, wo, swo, bo, wto, scbo, a, N, Ko, 0), d = proj8(h, thr_d, wd, swd, bd, wtd, scbd, y, N, Kd, 0);
  const dim3 grid(2 * (N / 16)), block(PW * 64);
#define OD(NCD)                                                                                     \
  if (Ko <= 2048) hipLaunchKernelGGL((l8_o_down_kernel<1, NCD>), grid, block, 0, st, o, d);          \
  else hipLaunchKernelGGL((l8_o_down_kernel<2, NCD>), grid, block, 0, st, o, d);                     \
  break
  switch ((Kd + 2047) / 2048) {
    case 3: OD(3);
    case 4: OD(4);
    case 5: OD(5);
    default: OD(6);
  }
#undef OD
  return (int)hipGetLastError();
}
