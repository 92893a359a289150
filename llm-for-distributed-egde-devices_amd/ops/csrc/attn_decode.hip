// Split-K flash-decoding over a head-major KV cache.
//
// q [B, Hq, D] (one new token per sequence), caches [B, Hkv, S, D] with row stride D, valid
// positions [0, seq_lens[b]).  Decode attention is HBM-bound on the K/V read, so the kernel is
// shaped for streaming rather than MFMA: one workgroup = (split, kv-head, batch); its G = Hq/Hkv
// query heads share every K/V row it loads (GQA reuse), and LPK lanes cooperate on one key row
// (LPK*16 B contiguous per key, 1 KiB per wave-instruction at D=128 -> fully coalesced).
// One pass over the split: every wave runs an online softmax (running max m, sum l, acc) over
// its key slice with K and V rows of a chunk loaded together and the next chunk prefetched, then
// the 4 waves are merged in LDS.  At decode contexts of a few hundred keys the kernel is bound by
// the serial load-latency chain, so fusing the old scores / softmax / P.V phases (each a round
// of dependent loads) is what matters.
// With nsplit > 1 each split writes (acc, m, l) and a combine kernel merges them; with one
// split the normalised output is written directly.
//
// FUSED variant (decode step of the model): q comes straight from the QKV projection row and is
// rotated in-kernel (HF rotate_half on the first `rot` dims, cos/sin from the host table, rounded
// to bf16 exactly like ops.rope_kv_write), and the split that owns the new position appends the
// rotated k and the v row to the head-major cache before reading it — the separate RoPE/KV-write
// launch disappears.  QOUT additionally emits the output as int8 with one scale per (token, 64
// columns) (layout [cols/64][Mpad]) for the W8A8 o-projection, replacing the per-token quant launch.
#include "attn_decode.h"

namespace {
template <int D, int G, bool DIRECT, bool FUSED, bool QOUT, int OCC, bool HF, int NWV = ATTN_NW, int UNROLL = UNROLL_DEF>
__global__ void __launch_bounds__(NWV * 64, OCC > 0 ? OCC : 1) decode_attn_kernel(
    const bf16_t* __restrict__ q, int64_t q_sb, bf16_t* __restrict__ kc, bf16_t* __restrict__ vc,
    int64_t c_sb, int64_t c_sh, const int* __restrict__ seq_lens, float scale_log2, int CH, int nsplit,
    bf16_t* __restrict__ out, int64_t o_sb, float* __restrict__ part_acc, float* __restrict__ part_ml, Fuse fz) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  decode_attn_body<D, G, DIRECT, FUSED, QOUT, OCC, HF, NWV, UNROLL>(smem, blockIdx.x, blockIdx.y, gridDim.y, blockIdx.z, q, q_sb,
                                                                   kc, vc, c_sb, c_sh, seq_lens, scale_log2, CH, nsplit, out,
                                                                   o_sb, part_acc, part_ml, fz);
}

// Sums of the key splits of one (row, head), in split order (blockDim.x >= D).  Up to UN <= 8 splits: every maximum, sum and
// partial sum is requested at once and each thread forms the weights itself, with no barrier between (through LDS, as below,
// 2 splits took 1.0 us longer than this and 4 0.3).
template <bool QOUT, bool HF, int UN>
__global__ void __launch_bounds__(256) decode_combine_few_kernel(const float* __restrict__ part_acc,
                                                                 const float* __restrict__ part_ml, int nsplit, int D,
                                                                 bf16_t* __restrict__ out, int64_t o_sb, Fuse fz) {
  const int hq = blockIdx.x, b = blockIdx.y, Hq = gridDim.x, tid = threadIdx.x;
  const float* ml = part_ml + ((size_t)b * Hq + hq) * nsplit * 2;
  const float* pa = part_acc + ((size_t)b * Hq + hq) * nsplit * D + min(tid, D - 1);
  float m[UN], l[UN], p[UN], M = -INFINITY, L = 0.f, a = 0.f;
#pragma unroll
  for (int j = 0; j < UN; ++j) {                             // (past the last: the last again, not used)
    const int s = min(j, nsplit - 1);
    m[j] = ml[2 * s];
    l[j] = ml[2 * s + 1];
    p[j] = pa[(size_t)s * D];
  }
#pragma unroll
  for (int j = 0; j < UN; ++j) M = fmaxf(M, m[j]);
#pragma unroll
  for (int j = 0; j < UN; ++j)
    if (j < nsplit && m[j] != -INFINITY) {
      const float w = exp2f(m[j] - M);
      L += w * l[j];
      a += w * p[j];
    }
  if (tid >= D) return;
  const float invL = 1.f / L;
  if constexpr (QOUT) {
    const int col = hq * D + tid;
    quant_group_store(e2f<HF>(f2e<HF>(a * invL)), fz.out_q + (size_t)b * Hq * D + col,
                      fz.out_s + (size_t)(col >> 6) * fz.Mpad + b, tid & 63);
  } else {
    out[b * o_sb + (size_t)hq * D + tid] = f2e<HF>(a * invL);
  }
}

// More splits: their weights meet in LDS first, then a coordinate's
// partial sums are requested 32 at a time; walked one by one, each behind its maximum's load and test, the
// 32 splits of a 7967-key step took 15.5 us, now 5.7.
template <bool QOUT, bool HF>
__global__ void __launch_bounds__(256) decode_combine_kernel(const float* __restrict__ part_acc,
                                                             const float* __restrict__ part_ml, int nsplit, int D,
                                                             bf16_t* __restrict__ out, int64_t o_sb, Fuse fz) {
  constexpr int UN = 32;
  __shared__ float w_s[256], l_s[256], red[4];               // a split's weight (-1: it had no keys) and sum
  const int hq = blockIdx.x, b = blockIdx.y, Hq = gridDim.x, tid = threadIdx.x, nt = blockDim.x;
  const float* ml = part_ml + ((size_t)b * Hq + hq) * nsplit * 2;
  float M = -INFINITY;
  for (int s = tid; s < nsplit; s += nt) M = fmaxf(M, ml[2 * s]);
  M = wave_max(M);
  if ((tid & 63) == 0) red[tid >> 6] = M;
  __syncthreads();
  for (int w = 0; w < nt / 64; ++w) M = fmaxf(M, red[w]);
  const float* pa = part_acc + ((size_t)b * Hq + hq) * nsplit * D + min(tid, D - 1);
  float a = 0.f, L = 0.f;
  for (int s0 = 0; s0 < nsplit; s0 += nt) {
    const int n = min(nt, nsplit - s0);
    if (tid < n) {
      const float m = ml[2 * (s0 + tid)];
      w_s[tid] = m == -INFINITY ? -1.f : exp2f(m - M);
      l_s[tid] = ml[2 * (s0 + tid) + 1];
    }
    __syncthreads();
    for (int j0 = 0; j0 < n; j0 += UN) {
      float p[UN];
#pragma unroll
      for (int j = 0; j < UN; ++j) p[j] = pa[(size_t)(s0 + min(j0 + j, n - 1)) * D];
#pragma unroll
      for (int j = 0; j < UN; ++j) {
        const float w = j0 + j < n ? w_s[j0 + j] : -1.f;
        if (w >= 0.f) {
          L += w * l_s[j0 + j];
          a += w * p[j];
        }
      }
    }
    __syncthreads();
  }
  if (tid >= D) return;
  const float invL = 1.f / L;
  if constexpr (QOUT) {
    const int col = hq * D + tid;
    quant_group_store(e2f<HF>(f2e<HF>(a * invL)), fz.out_q + (size_t)b * Hq * D + col,
                      fz.out_s + (size_t)(col >> 6) * fz.Mpad + b, tid & 63);
  } else {
    out[b * o_sb + (size_t)hq * D + tid] = f2e<HF>(a * invL);
  }
}
}  // namespace

// Workspace sizes (floats) for a given launch; the binding allocates them.
static int g_target_wg = 512;   // >= 2 workgroups per CU before splitting K
// fused kernels: 4 (default) / 5 = single-buffered, barrier-free, >= 4 / 5 waves per SIMD; 0 = the
// double-buffered form with the append barrier (168 VGPRs, 3 waves per SIMD).  Measured at 128
// sequences x 32 heads, context 160 (tools/bench_ops.py attn_fused): 57.7 / 60.4 / 66.6 us.
static int g_attn_occ = 4;
// query-head split for small grids (tune "decode_attn_gsplit"): 0 automatic, 1 off, 2 always (GQA)
static int g_attn_gsplit = 0, g_attn_early = 1;
// key groups per wave per chunk of the barrier-free MHA D = 128 form (4 / 8; tune "decode_attn_unroll")
static int g_attn_unroll = 4;
extern "C" void edge_decode_attn_unroll(int v) { g_attn_unroll = v == 8 ? 8 : 4; }
// MHA grids below this many workgroups (batch 1: 32 on Llama-2-7B) take the double-buffered form:
// each workgroup walks its keys in several chunks, and there the next chunk in flight beats the
// single-buffered form's extra occupancy.  us, single / double buffered, 32 heads of 128, 41 / 141 / 251 keys: 64
// workgroups 4.75 6.8 7.9 / 4.15 5.9 6.75, 128 5.0 7.2 8.3 / 4.7 6.3 7.8, 256 5.4 8.0 9.5 / 5.1 8.1 10.8.  Tune "decode_attn_small".
static int g_attn_small_wg = 192;
extern "C" void edge_decode_attn_small(int v) { g_attn_small_wg = v; }
extern "C" void edge_decode_attn_gsplit(int v) { g_attn_gsplit = v; }
extern "C" void edge_decode_attn_early(int v) { g_attn_early = v; }
extern "C" void edge_decode_attn_config(int target_wg) { g_target_wg = target_wg > 0 ? target_wg : 512; }
extern "C" void edge_decode_attn_occ(int occ) { g_attn_occ = occ == 0 || occ == 5 ? occ : 4; }

namespace {
template <int D, int G, bool DI, bool FU, bool QO, bool HF>
void launch_attn(dim3 grid, size_t lds, hipStream_t st, const void* q, int64_t q_sb, void* k_cache, void* v_cache,
                 int64_t c_sb, int64_t c_sh, const int* seq_lens, float sl2, int ch, int nsplit, void* out,
                 int64_t o_sb, float* part_acc, float* part_ml, const Fuse& fz, bool small_grid) {
#define ATTN_ARGS grid, dim3(ATTN_NT), lds, st, (const bf16_t*)q, q_sb, (bf16_t*)k_cache, (bf16_t*)v_cache, c_sb, c_sh, \
                  seq_lens, sl2, ch, nsplit, (bf16_t*)out, o_sb, part_acc, part_ml, fz
  if constexpr (FU) {                           // the model's decode step: barrier-free form selectable
    // occupancy target per GQA group size: the per-head q / accumulator registers grow with G, and
    // a 4-waves-per-SIMD bound spills 250-900 B/lane at G >= 4 (ISA resource report)
    constexpr int OCC4 = G <= 2 ? 4 : (G == 4 ? 2 : 1), OCC5 = G <= 2 ? 5 : OCC4;
    // (8- and 16-wave workgroups for batch-1 grids measured slower: Llama-3.2-1B decode step
    // 1.08 -> 1.19 ms with 8 waves)
    if constexpr (D == 128 && G == 1) {
      if (g_attn_occ == 4 && !small_grid && g_attn_unroll == 8) {
        hipLaunchKernelGGL((decode_attn_kernel<D, G, DI, FU, QO, OCC4, HF, ATTN_NW, 8>), ATTN_ARGS);
        return;
      }
    }
    if (g_attn_occ == 4 && !small_grid) { hipLaunchKernelGGL((decode_attn_kernel<D, G, DI, FU, QO, OCC4, HF>), ATTN_ARGS); return; }
    if (g_attn_occ == 5) { hipLaunchKernelGGL((decode_attn_kernel<D, G, DI, FU, QO, OCC5, HF>), ATTN_ARGS); return; }
  }
  hipLaunchKernelGGL((decode_attn_kernel<D, G, DI, FU, QO, 0, HF>), ATTN_ARGS);
#undef ATTN_ARGS
}
}  // namespace

extern "C" int edge_decode_attn_plan(int B, int Hkv, int max_len, int D, int* ch_out, int* nsplit_out) {
  const int target_wg = g_target_wg;
  int per = B * Hkv;
  int nsplit = (target_wg + per - 1) / per;
  int ch = (max_len + nsplit - 1) / nsplit;
  ch = ((ch + 63) / 64) * 64;
  // at least 256 keys per split: below that the combine launch and the partial round trip cost
  // more than the split saves (batch 1, Llama-3.2-1B, context <= 256: 15.7 + 4.8 us per layer with
  // 4 splits of 64 keys; Llama-2-7B W8A8 batch 1 at context ~200: 2.16 ms/token direct against
  // 2.33-2.42 ms with 2 splits of 128 keys + combine)
  const int ch_min = 256;
  if (ch < ch_min) ch = ch_min;
  if (ch > 1024) ch = 1024;
  nsplit = (max_len + ch - 1) / ch;
  if (nsplit < 1) nsplit = 1;
  *ch_out = ch;
  *nsplit_out = nsplit;
  return 0;
}

namespace {
template <bool HF>
void launch_combine(const float* part_acc, const float* part_ml, int nsplit, int B, int Hq, int D, void* out, int64_t o_sb,
                    bool qout, const Fuse& fz, hipStream_t st) {
  const dim3 cg(Hq, B), cb(D <= 128 ? 128 : 256);
#define DCOMBINE(Q, H)                                                                                                       \
  do {                                                                                                                       \
    if (nsplit <= 4)                                                                                                         \
      hipLaunchKernelGGL((decode_combine_few_kernel<Q, H, 4>), cg, cb, 0, st, part_acc, part_ml, nsplit, D, (bf16_t*)out, o_sb, fz); \
    else if (nsplit <= 8)                                                                                                    \
      hipLaunchKernelGGL((decode_combine_few_kernel<Q, H, 8>), cg, cb, 0, st, part_acc, part_ml, nsplit, D, (bf16_t*)out, o_sb, fz); \
    else                                                                                                                     \
      hipLaunchKernelGGL((decode_combine_kernel<Q, H>), cg, cb, 0, st, part_acc, part_ml, nsplit, D, (bf16_t*)out, o_sb, fz);  \
  } while (0)
  if constexpr (!HF) {
    if (qout) {
      DCOMBINE(true, false);
      return;
    }
  }
  DCOMBINE(false, HF);
#undef DCOMBINE
}

template <bool HF>
int run_attn(const void* q, int64_t q_sb, void* k_cache, void* v_cache, int64_t c_sb, int64_t c_sh,
             const int* seq_lens, int B, int Hq, int Hkv, int D, float scale, int ch, int nsplit, void* out,
             int64_t o_sb, float* part_acc, float* part_ml, const int* pos, const float* cs, int rot, void* out_q,
             float* out_s, int Mpad, hipStream_t st) {
  const int G0 = Hq / Hkv;
  const bool fused = pos != nullptr, qout = out_q != nullptr;
  // grids of a few dozen workgroups (batch 1-4 on a GQA model: 8 KV heads) are bound by each
  // workgroup's serial chain over its keys x G query heads: give every query head its own
  // workgroup instead (K/V rows re-read G times, from L2).  Needs the barrier-free fused form
  // (the new key in registers) or the plain kernel: no workgroup reads a row another one appends.
  const bool gs_ok = G0 > 1 && (!fused || g_attn_occ != 0);
  const int gs = gs_ok && (g_attn_gsplit == 2 || (g_attn_gsplit == 0 && B * Hkv * nsplit < 128)) ? G0 : 1;
  const int G = G0 / gs;
  const Fuse fz{pos, cs, fused ? rot : 0, q_sb, (int8_t*)out_q, out_s, Mpad, gs, g_attn_early};
  const float sl2 = scale * 1.4426950408889634f;
  const size_t lds = (size_t)(ATTN_NW * G * D + 2 * ATTN_NW * G) * sizeof(float);
  const dim3 grid(nsplit, Hkv * gs, B);
  const bool direct = nsplit == 1;
  const bool small_grid = G0 == 1 && direct && fused && B * Hkv < g_attn_small_wg;
  // fp16 rows (HF) have no int8-output form: the fp16 agents' o-projection is fp16
#define DK(DD, GG, DI, FU, QO)                                                                                     \
  launch_attn<DD, GG, DI, FU, QO, HF>(grid, lds, st, q, q_sb, k_cache, v_cache, c_sb, c_sh, seq_lens, sl2, ch, nsplit, \
                                      out, o_sb, part_acc, part_ml, fz, small_grid)
#define DLAUNCH(DD, GG)                                                     \
  do {                                                                      \
    if (direct) {                                                           \
      if constexpr (!HF) {                                                  \
        if (qout) { if (fused) DK(DD, GG, true, true, true); else DK(DD, GG, true, false, true); break; } \
      }                                                                     \
      if (fused) DK(DD, GG, true, true, false); else DK(DD, GG, true, false, false);             \
    } else {                                                                \
      if (fused) DK(DD, GG, false, true, false); else DK(DD, GG, false, false, false);           \
    }                                                                       \
  } while (0)
#define GSW(DD)                                   \
  switch (G) {                                    \
    case 1: DLAUNCH(DD, 1); break;                \
    case 2: DLAUNCH(DD, 2); break;                \
    case 4: DLAUNCH(DD, 4); break;                \
    case 8: DLAUNCH(DD, 8); break;                \
    default: return -3;                           \
  }
  switch (D) {
    case 64: GSW(64); break;
    case 80: GSW(80); break;
    case 128: GSW(128); break;
    case 256: GSW(256); break;
    default: return -4;
  }
#undef GSW
#undef DLAUNCH
#undef DK
  if (!direct) launch_combine<HF>(part_acc, part_ml, nsplit, B, Hq, D, out, o_sb, qout, fz, st);
  return (int)hipGetLastError();
}
}  // namespace

// q: [B, *] rows with the Hq query heads at offset 0 (q_sb elements apart).  FUSED (pos != null):
// q points at the QKV projection output, rows hold [q heads | k heads | v heads], the new token's
// k/v are appended to the caches at pos[b] and q is rotated in-kernel.  QOUT (out_q != null,
// D % 64 == 0, bf16 only): int8 output + [Hq*D/64][Mpad] scales instead of `out`.  h16: q, caches
// and out are fp16.
extern "C" int edge_decode_attn(const void* q, int64_t q_sb, void* k_cache, void* v_cache, int64_t c_sb,
                                int64_t c_sh, const int* seq_lens, int B, int Hq, int Hkv, int D, float scale,
                                int ch, int nsplit, void* out, int64_t o_sb, float* part_acc, float* part_ml,
                                const int* pos, const float* cs, int rot, void* out_q, float* out_s, int Mpad,
                                int h16, hipStream_t st) {
  if (B == 0) return 0;
  const int G0 = Hq / Hkv;
  if (G0 * Hkv != Hq) return -2;
  const bool fused = pos != nullptr, qout = out_q != nullptr;
  if (qout && (D % 64 != 0 || Mpad < B || h16)) return -2;
  if (fused && rot > 0 && (cs == nullptr || rot % 16 != 0 || rot > D)) return -2;
  return h16 ? run_attn<true>(q, q_sb, k_cache, v_cache, c_sb, c_sh, seq_lens, B, Hq, Hkv, D, scale, ch, nsplit, out,
                              o_sb, part_acc, part_ml, pos, cs, rot, out_q, out_s, Mpad, st)
             : run_attn<false>(q, q_sb, k_cache, v_cache, c_sb, c_sh, seq_lens, B, Hq, Hkv, D, scale, ch, nsplit, out,
                               o_sb, part_acc, part_ml, pos, cs, rot, out_q, out_s, Mpad, st);
}

// The sums over the key splits alone, for partial results that decode_pair.hip's launch has written (16-bit output).
extern "C" int edge_decode_attn_combine(const float* part_acc, const float* part_ml, int nsplit, int B, int Hq, int D, void* out,
                                        int64_t o_sb, int h16, hipStream_t st) {
  if (h16) launch_combine<true>(part_acc, part_ml, nsplit, B, Hq, D, out, o_sb, false, Fuse{}, st);
  else launch_combine<false>(part_acc, part_ml, nsplit, B, Hq, D, out, o_sb, false, Fuse{}, st);
  return (int)hipGetLastError();
}
