// The attention half of a two-part launch (decode_pair.hip, decode_pair_i8.hip): its operands and its workgroups.
#pragma once
#include "attn_decode.h"

namespace {
constexpr int PW = 8;                      // waves a workgroup

struct AttnArgs {
  const bf16_t* q;
  int64_t q_sb;
  bf16_t *kc, *vc;
  int64_t c_sb, c_sh;
  const int* seq_lens;
  float scale_log2;
  int ch, nsplit, ny;                      // ny: query heads (each a workgroup of its own)
  bf16_t* out;
  int64_t o_sb;
  float *part_acc, *part_ml;
  Fuse fz;
};

// Workgroup bid of nsplit x ny x rows.
template <int D, bool DIRECT, bool HF>
__device__ __forceinline__ void attn_part(float* smem, int bid, const AttnArgs& a) {
  const int s = bid % a.nsplit, r = bid / a.nsplit;
  decode_attn_body<D, 1, DIRECT, true, false, 4, HF, PW, UNROLL_DEF>(smem, s, r % a.ny, a.ny, r / a.ny, a.q, a.q_sb, a.kc, a.vc,
                                                                    a.c_sb, a.c_sh, a.seq_lens, a.scale_log2, a.ch, a.nsplit,
                                                                    a.out, a.o_sb, a.part_acc, a.part_ml, a.fz);
}
template <int D>
constexpr int attn_part_lds() { return PW * D + 2 * PW; }      // floats
}  // namespace

extern "C" int edge_decode_attn_combine(const float* part_acc, const float* part_ml, int nsplit, int B, int Hq, int D, void* out,
                                        int64_t o_sb, int h16, hipStream_t st);
