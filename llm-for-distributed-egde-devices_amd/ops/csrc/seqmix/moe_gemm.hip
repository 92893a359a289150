// Mixture of experts at prompt sizes (bf16, MFMA): the (token, choice) pairs are grouped by expert and every expert's
// rows run through its gate | up weights (activation in the epilogue) and then its down weights, one launch for all
// experts each.
//
//   moe_sort_kernel   one workgroup: counts per expert, rows[p] = the pair (t * top + k) at sorted position p, and
//                     the list of row tiles (expert, first position, rows), a tile never spanning two experts
//   moe_gemm_kernel   tile lists x column tiles; the activations' rows are gathered (first product: h[t]) or taken in
//                     sorted order (second), and the second product's rows go straight back to their pair's row
//
// Nothing crosses to the host: the grid covers the largest possible tile count and workgroups past the real one leave.
//
// Measured (both products, sorting and activation; MI355X) against one library product per expert with the sort, the
// gather, the activation and the scatter as launches of their own: 4096 tokens x 3 of 16 experts 1024 -> 1024,
// 758 -> 127 us (610 TFLOP/s); 7680 x 3 of 32, 2048 -> 3072, 1679 -> 664 us (874); 512 x 4 of 32, 2048 -> 2048,
// 1369 -> 169 us, where the experts' 805 MB (4.8 TB/s) are the bound.  At 128-row tiles the bound is the LDS: 64 B per clock and
// CU come in and 128 are read at the full MFMA rate (tile_rows says what 256-row tiles change); 128 x 256 tiles gained 3-6 %
// from 2048 columns on and lost below, deeper rings with one workgroup of 128 x 128 per CU lose 40 %; a third stage for the
// weights alone still leaves two workgroups a CU (deep_ring).
#include "seqmix_common.h"

namespace {
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr int SORT_NT = 1024, SORT_E = 512;
enum { ACT_NONE = 0, ACT_GLU_CLAMP = 1, ACT_GLU_SILU = 2, ACT_RELU2 = 3 };

// tiles: [0] = their number, tile i at [4 + 4 i] = (expert, first sorted position, rows, 0).
// Counting by LDS atomics, one table per wave (16 waves share a CU: the lanes of one wave meet on at most E
// counters).  The order of an expert's rows follows the atomics; no result depends on it.
__global__ void __launch_bounds__(SORT_NT) moe_sort_kernel(const int* __restrict__ idx, int R, int E, int BM,
                                                           int* __restrict__ rows, int* __restrict__ tiles) {
  constexpr int NW = SORT_NT / 64;
  __shared__ int cnt[NW][SORT_E];
  __shared__ int scan_r[SORT_E], scan_t[SORT_E];
  const int tid = threadIdx.x, wave = tid >> 6;
  for (int i = tid; i < NW * SORT_E; i += SORT_NT) (&cnt[0][0])[i] = 0;
  __syncthreads();
  for (int i = tid; i < R; i += SORT_NT) atomicAdd(&cnt[wave][min(max(idx[i], 0), E - 1)], 1);
  __syncthreads();
  int total = 0, nt = 0;
  if (tid < E) {
    for (int w = 0; w < NW; ++w) {                           // the wave tables become offsets inside the expert
      const int c = cnt[w][tid];
      cnt[w][tid] = total;
      total += c;
    }
    nt = (total + BM - 1) / BM;
  }
  if (tid < SORT_E) {
    scan_r[tid] = total;
    scan_t[tid] = nt;
  }
  __syncthreads();
  for (int d = 1; d < E; d <<= 1) {                          // inclusive sums over the experts
    int a = 0, b = 0;
    if (tid < E && tid >= d) { a = scan_r[tid - d]; b = scan_t[tid - d]; }
    __syncthreads();
    if (tid < E) { scan_r[tid] += a; scan_t[tid] += b; }
    __syncthreads();
  }
  if (tid < E) {
    const int r0 = scan_r[tid] - total, t0 = scan_t[tid] - nt;
    for (int w = 0; w < NW; ++w) cnt[w][tid] += r0;
    for (int i = 0; i < nt; ++i)
      *reinterpret_cast<int4*>(tiles + 4 + 4 * (t0 + i)) = make_int4(tid, r0 + i * BM, min(BM, total - i * BM), 0);
    if (tid == E - 1) tiles[0] = scan_t[tid];
  }
  __syncthreads();
  for (int i = tid; i < R; i += SORT_NT) rows[atomicAdd(&cnt[wave][min(max(idx[i], 0), E - 1)], 1)] = i;
}

__device__ __forceinline__ void glds16(const void* g, void* lds_base) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)lds_base, 16, 0, 0);
}
__device__ __forceinline__ uint32_t lds_off(const void* p) {
  return (uint32_t)(uintptr_t)((__attribute__((address_space(3))) const void*)p);
}
// N ds_read_b128 at addr + 2048 i, which the compiler does not track: callers wait and pin before use
template <int I, int N>
__device__ __forceinline__ void lds_frags(uint32_t addr, v4i (&f)[N]) {
  if constexpr (I < N) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f[I]) : "v"(addr), "n"(I * 2048));
    lds_frags<I + 1, N>(addr, f);
  }
}
template <int N>
__device__ __forceinline__ void pin(v4i (&f)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(f[i]));
}

// out[r] = act(A[row(r)] W_e^T) for the rows r of each tile's expert e.  A: K-contiguous rows, W [E, NW, K].
//  * BM x BN block tile (BN weight rows), WM x WN waves, 64-k stages.  Both operands go global -> LDS by LDS-DMA in
//    1 KiB pieces of 8 rows x 128 B (whole cache lines); the 16-byte chunk c of row r sits at slot c ^ (r & 7), so
//    the 16 rows of a fragment read spread over the banks.  R stages ride ahead of the arithmetic (counted vmcnt, one
//    bare barrier per stage, fragments double-buffered in registers and read by asm so that no read drains the ring).
//  * The weights are the MFMA's first operand: a lane's accumulator holds four consecutive output columns of one row,
//    stored as 8 bytes.  Gated units (NW = 2 ff): a wave's 64 (or 32) weight rows are half gate rows and half the
//    up rows of the same features, so one lane holds both halves and the activation never leaves the registers
//    (fp32; the unfused form rounds both halves to bf16 first).
//  * blockIdx -> tile: each XCD takes a contiguous range of the (real) tiles, walked in groups of four row tiles
//    column by column, so neighbours in an L2 share an expert's weights.
template <int BM, int BN, int WM, int WN, int RA, int RW, int ACT, bool GATHER>
__global__ void __launch_bounds__(64 * WM * WN, 2) moe_gemm_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                                  const int* __restrict__ rows, const int* __restrict__ tiles,
                                                                  bf16_t* __restrict__ out, int top, int N, int NW, int K,
                                                                  int grid_n, const float* __restrict__ row_w, float limit, int spread) {
  constexpr bool GLU = ACT == ACT_GLU_CLAMP || ACT == ACT_GLU_SILU;
  constexpr int NWV = WM * WN, AP = BM / 8, BP = BN / 8, PA = AP / NWV, PB = BP / NWV;   // pieces of a stage, of a wave
  constexpr int MI = BM / WM / 16, NJ = BN / WN / 16;
  constexpr int RS = RA < RW ? RA : RW, DEEP = RA > RW ? PA : RW > RA ? PB : 0;           // pieces of the operand one stage further ahead
  static_assert(AP % NWV == 0 && BP % NWV == 0 && (!GLU || NJ % 2 == 0) && (RA - RW) * (RA - RW) <= 1, "tile shape");
  static_assert((RA * AP + RW * BP) * 1024 <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024))) int8_t ring[(RA * AP + RW * BP) * 1024];
  // equal rings: a stage's rows and weights side by side (apart, 64-row tiles of small steps took 0.3 to 0.5 us of 21 more); else two rings
  constexpr bool EVEN = RA == RW;
  constexpr int W0 = (EVEN ? 1 : RA) * AP * 1024, SA = (AP + (EVEN ? BP : 0)) * 1024, SW = (BP + (EVEN ? AP : 0)) * 1024;

  const int nwg = tiles[0] * grid_n, orig = blockIdx.x;
  if (orig >= nwg) return;
  const int xcd = orig & 7, q8 = nwg >> 3, r8 = nwg & 7;
  const int wgid = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (orig >> 3);
  constexpr int GM = 4;
  const int per_group = GM * grid_n, grp = wgid / per_group, gsz = min(GM, tiles[0] - grp * GM);
  const int inr = wgid - grp * per_group, bm = grp * GM + inr % gsz, bn = inr / gsz;
  const int4 tile = *reinterpret_cast<const int4*>(tiles + 4 + 4 * bm);   // (expert, first position, rows)
  const bf16_t* We = W + (size_t)tile.x * NW * K;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN, KT = K / 64;
  constexpr int FN = GLU ? BN / 2 : BN;                      // output columns of a block tile
  // this wave's DMA pieces p = wave + NWV i: activation rows 8 p .. (p < AP), or weight rows
  const char* src[PA + PB];
#pragma unroll
  for (int i = 0; i < PA + PB; ++i) {
    const int p = wave + NWV * i, r = (p < AP ? p : p - AP) * 8 + (lane >> 3);
    const int ck = ((lane & 7) ^ (r & 7)) * 16;
    size_t row;
    const bf16_t* base;
    if (p < AP) {
      const int pos = tile.y + min(r, tile.z - 1);
      row = GATHER ? rows[pos] / top : pos;
      base = A;
    } else {
      int f;
      if constexpr (GLU) {
        const int w = r / (16 * NJ), j = (r / 16) % NJ;
        f = min(bn * FN + w * (8 * NJ) + (j % (NJ / 2)) * 16 + (r & 15), N - 1) + (j >= NJ / 2 ? N : 0);
      } else {
        f = min(bn * FN + r, N - 1);
      }
      row = f;
      base = We;
    }
    src[i] = reinterpret_cast<const char*>(base + row * (size_t)K) + ck;
  }
  // stages past the last re-load the last one into a slot that is not read again: the counts stay constant
  // spread: column blocks and experts start at different k and go round.  In step, every workgroup reads the same 128 bytes
  // of rows 2 K bytes apart, which lie in few memory channels
  const int k0 = spread ? (tile.x * 7 + bn * 5) % KT : 0;
  auto issue = [&](int st, bool weights) {
    const int kt = min(st, KT - 1) + k0;
    const size_t ko = (size_t)(kt < KT ? kt : kt - KT) * 128;
    int8_t* slot = ring + (weights ? W0 + (st % RW) * SW : (st % RA) * SA) + wave * 1024;
#pragma unroll
    for (int i = 0; i < (weights ? PB : PA); ++i) glds16(src[weights ? PA + i : i] + ko, slot + NWV * i * 1024);
  };
  // the operand that is further ahead last: its pieces may still be on their way when the other's have landed
  auto issue_both = [&](int st) {
    issue(RA > RW ? st + RW : st + RA, RA > RW);
    issue(RA > RW ? st + RA : st + RW, RA <= RW);
  };
  // fragment (16 rows x 32 k of step ks): row lane & 15, chunk 4 ks + (lane >> 4)
  const uint32_t fo = lds_off(ring) + (lane & 15) * 128 + (((lane >> 4) ^ (lane & 7)) << 4);
  auto read = [&](int st, int ks, v4i (&fa)[MI], v4i (&fw)[NJ]) {
    const uint32_t b = fo ^ (ks << 6);
    lds_frags<0, MI>(b + (st % RA) * SA + wm * (MI * 2048), fa);
    lds_frags<0, NJ>(b + W0 + (st % RW) * SW + wn * (NJ * 2048), fw);
  };
  v4f acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  auto mma = [&](v4i (&fa)[MI], v4i (&fw)[NJ]) {
    pin(fa);
    pin(fw);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, fw[j]), __builtin_bit_cast(v8bf, fa[i]),
                                                            acc[i][j], 0, 0, 0);
  };
  auto pin_acc = [&]() {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) asm volatile("" : "+v"(acc[i][j]));
  };

#pragma unroll
  for (int st = 0; st < RS; ++st) {
    issue(st, RA > RW);
    issue(st, RA <= RW);
  }
  if constexpr (DEEP != 0) issue(RS, RW > RA);
  v4i a0[MI], w0[NJ], a1[MI], w1[NJ];
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RS - 1) * (PA + PB) + DEEP) : "memory");
  __builtin_amdgcn_s_barrier();
  read(0, 0, a0, w0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  for (int s = 0; s < KT; ++s) {
    read(s, 1, a1, w1);
    mma(a0, w0);
    pin_acc();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (s + 1 < KT) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RS - 2) * (PA + PB) + DEEP) : "memory");   // own pieces of stage s + 1
      __builtin_amdgcn_s_barrier();                          // stage s + 1 is there, stage s has been read by all
      issue_both(s);
      read(s + 1, 0, a0, w0);
    }
    mma(a1, w1);
    pin_acc();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // the re-loads past the end

  // lane: row i * 16 + (lane & 15), columns 4 (lane >> 4) + 0..3 of column tile j
  const int c4 = 4 * (lane >> 4);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int r = (wm * MI + i) * 16 + (lane & 15);
    if (r >= tile.z) continue;
    const int pos = tile.y + r;
    const size_t orow = GATHER ? (size_t)pos : (size_t)rows[pos];
    const float rw = (ACT == ACT_GLU_SILU && row_w != nullptr) ? row_w[rows[pos]] : 1.f;
    constexpr int NO = GLU ? NJ / 2 : NJ;
#pragma unroll
    for (int j = 0; j < NO; ++j) {
      const int col = bn * FN + (wn * NO + j) * 16 + c4;
      if (col >= N) continue;                                // N % 16 == 0: a column tile is whole or absent
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float x = acc[i][j][q];
        if constexpr (ACT == ACT_GLU_CLAMP) v[q] = glu_clamp_f(x, acc[i][j + NO][q], limit);
        else if constexpr (ACT == ACT_GLU_SILU) v[q] = siluf_(rw * x) * (rw * acc[i][j + NO][q]);
        else if constexpr (ACT == ACT_RELU2) { const float m = fmaxf(x, 0.f); v[q] = m * m; }
        else v[q] = x;
      }
      *reinterpret_cast<uint2*>(out + orow * (size_t)N + col) = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
    }
  }
}

// Row tiles of E experts that R pairs fall on at random: a normal count an expert, sum over k of P(count > k BM), the first always
// (an expert without rows costs its launch slot too)
double expected_tiles(double R, int E, int BM) {
  const double m = R / E, s = sqrt(m > 1. ? m : 1.);
  const int sure = m > 5. * s + BM ? (int)((m - 5. * s) / BM) : 0;       // (tiles that every such count fills)
  double n = 1. + sure;
  for (int k = sure + 1; k * BM < m + 5. * s; ++k) n += 0.5 * (1. + erf((m - k * BM) / (s * 1.4142135623730951)));
  return E * n;
}
// The weights of a stage come from HBM, the rows from an L2: a 128-row tile's ring of three stages for the weights and two for the rows
// (80 KB, still two workgroups a CU) asks for the weights a stage earlier and does not pay for the rows' half of the LDS.  A launch of
// one round in which CUs hold a second workgroup to wait beside (1.1 to 2.05 workgroups a CU) keeps two stages: there the third cost 1 to
// 2 % of the launch (43 launches; at the most 8), with fewer workgroups it gained 14 to 21 % where k has more than 16 stages and 4 % below
// (97), with more 3 to 4 % (164).  Both products, us, two stages / this: 8 experts of 3072 -> 1024 (relu2), 64 rows an expert 68 / 54; 8 of
// 2048 -> 3072 (gated), 668 278 / 257; 24 of 1536 -> 1536 (gated), 510 290 / 278.  256-row tiles (160 KB) keep two stages: a third gained 2 to 3 %
// at 510 rows an expert, but lost 1 to 6 % at 384 and up to 5 % above 800.
bool deep_ring(double tiles, int columns) { return tiles * columns <= 1.1 * 256 || tiles * columns > 2.05 * 256; }

template <int BM, int BN, int WM, int WN, int R, bool DEEP = false>
int launch_pair(const void* h, const void* w_gu, const void* w_down, const int* rows, const int* tiles, void* y, void* out,
                int max_tiles, int pairs, int E, int top, int W, int ff, int act, const float* row_w, float limit, int spread,
                hipStream_t st) {
  const dim3 blk(64 * WM * WN);
  const int up = act == ACT_RELU2 ? 1 : 2, fn = act == ACT_RELU2 ? BN : BN / 2;
  const int g1 = (ff + fn - 1) / fn, g2 = (W + BN - 1) / BN;
  const double likely = expected_tiles(pairs, E, BM);
#define MOE_FIRST(ACT, RW)                                                                                                 \
  hipLaunchKernelGGL((moe_gemm_kernel<BM, BN, WM, WN, R, RW, ACT, true>), dim3(max_tiles * g1), blk, 0, st, (const bf16_t*)h,   \
                     (const bf16_t*)w_gu, rows, tiles, (bf16_t*)y, top, ff, up * ff, W, g1, row_w, limit, spread)
#define MOE_ACT(RW)                                           \
  do {                                                        \
    if (act == ACT_GLU_CLAMP) MOE_FIRST(ACT_GLU_CLAMP, RW);   \
    else if (act == ACT_GLU_SILU) MOE_FIRST(ACT_GLU_SILU, RW); \
    else MOE_FIRST(ACT_RELU2, RW);                            \
  } while (0)
#define MOE_SECOND(RW)                                                                                                          \
  hipLaunchKernelGGL((moe_gemm_kernel<BM, BN, WM, WN, R, RW, ACT_NONE, false>), dim3(max_tiles * g2), blk, 0, st, (const bf16_t*)y, \
                     (const bf16_t*)w_down, rows, tiles, (bf16_t*)out, top, W, W, ff, g2, nullptr, 0.f, spread)
  if (DEEP && deep_ring(likely, g1)) MOE_ACT(R + DEEP);
  else MOE_ACT(R);
  if (DEEP && deep_ring(likely, g2)) MOE_SECOND(R + DEEP);
  else MOE_SECOND(R);
#undef MOE_FIRST
#undef MOE_ACT
#undef MOE_SECOND
  return (int)hipGetLastError();
}

// us of both products with tiles of BM rows, fitted to 525 points (15 sets of 8 to 64 experts of 512 to 4096 x 512 to 4096, 26 to 1300 rows
// an expert, all with equal rings; half of the estimates are within 5 %): workgroups come in rounds of 512 (two to a CU; 256 of the 256-row tiles), a round
// costs its 64-k stages and its start and end, and a partly filled last round more than its share; the experts' bytes are partly
// hidden behind that, or (256 rows) bound it from below.
double tile_us(int BM, double R, int E, int W, int ff, int up) {
  //                              us a stage, a start, both launches, TB/s, whole rounds' part
  static const double fit[3][5] = {{0.621, 4.35, 5.4, 9.36, 0.266}, {0.991, 7.2, 3.53, 13.3, 0.429}, {1.64, 16.1, 5.69, 4.04, 0.585}};
  const double* p = fit[BM == 64 ? 0 : BM == 128 ? 1 : 2];
  const int BN = BM == 256 ? 256 : 128, slots = BM == 256 ? 256 : 512;
  const double tiles = expected_tiles(R, E, BM);
  double us = p[2];
  for (int j = 0; j < 2; ++j) {
    const int N = j ? W : ff * up, K = j ? ff : W;
    const double x = tiles * ((N + BN - 1) / BN) / slots, rounds = p[4] * ceil(x - 0.02) + (1. - p[4]) * x;
    const double work = rounds * (p[0] * K / 64 + p[1]), bytes = 2e-6 * E * N * K / p[3];
    us += BM == 256 ? (work > bytes ? work : bytes) : work + bytes;
  }
  return us;
}
// Rows of a tile: up to 24 an expert the weights' bytes are all that counts (32 rows: two fragments, the smallest ring); above, the
// quickest by estimate.  A tile much taller than an expert's rows multiplies padding, a lower one reads the weights once more for an
// expert's second tile, and 256 x 256 tiles (one workgroup of 8 waves a CU, 128 x 64 a wave) halve what 128 x 128 ones read from and
// bring into the LDS per product, which is their bound, but fill the chip in whole rounds of 256 workgroups.  us for both products, 64 /
// 128 / 256 rows: 32 experts of 2048 -> 3072 (relu2), 48 rows an expert 162 / 172, 60 195 / 178 / 218, 135 323 / 299 / 232, 720 760 (128) / 664
// (874 TFLOP/s); 32 of 1024 -> 1024 (gated), 48 53 / 58, 94 72 / 62 / 77, 410 160 (128) / 133, 510 188 (128) / 201; 8 of 2048 -> 4096
// (gated), 54 102 / 120, 150 159 / 147 / 167, 600 358 (128) / 299; 24 of 1536 -> 1536 (relu2), 250 141 / 139 / 116, 330 168 / 141 / 193.
int tile_rows(int64_t R, int E, int W, int ff, int up) {
  if (R <= (int64_t)E * 24) return 32;
  const int widest = ff * up > W ? ff * up : W;              // up to half a tile a CU: the lowest (4 of 256 -> 512, 72 rows an expert 16 / 19)
  if (expected_tiles((double)R, E, 64) * ((widest + 127) / 128) <= 128.) return 64;
  const double low = tile_us(64, (double)R, E, W, ff, up), mid = tile_us(128, (double)R, E, W, ff, up);
  return tile_us(256, (double)R, E, W, ff, up) < 0.97 * (low < mid ? low : mid) ? 256 : low < mid ? 64 : 128;
}
int max_tiles(int64_t R, int E, int BM) { return (int)((R + BM - 1) / BM + (R < E ? R : E)); }
}  // namespace

extern "C" {

// int32 words of scratch: the sorted pairs and the tile list (its longest: taller tiles are fewer)
int64_t edge_sm_moe_gemm_ints(int64_t R, int E) { return ((R + 3) & ~3LL) + 4 + 4LL * max_tiles(R, E, R > (int64_t)E * 24 ? 64 : 32); }

// 0 when the kernels take these sizes
int edge_sm_moe_gemm_ok(int64_t T, int top, int E, int W, int ff) {
  const int64_t R = T * top;
  return W % 64 == 0 && ff % 64 == 0 && W > 0 && ff > 0 && E >= 1 && E <= SORT_E && R >= 1 && R < (1LL << 24) ? 0 : -2;
}

// h [T, W] bf16, idx [T, top], w_gu [E, 2 ff | ff, W], w_down [E, W, ff]; y: scratch [T top, ff]; out [T, top, W].
int edge_sm_moe_gemm(const void* h, const int* idx, const void* w_gu, const void* w_down, int* ints, void* y, void* out, int T,
                     int top, int E, int W, int ff, int act, const float* row_w, float limit, hipStream_t st) {
  if (edge_sm_moe_gemm_ok(T, top, E, W, ff) != 0 || act < ACT_GLU_CLAMP || act > ACT_RELU2) return -2;
  const int R = T * top, BM = tile_rows(R, E, W, ff, act == ACT_RELU2 ? 1 : 2), mt = max_tiles(R, E, BM);
  int *rows = ints, *tiles = ints + ((R + 3) & ~3);
  // while the weights' bytes are the bound (up to some 500 rows an expert) the workgroups' k starts are spread: us for both
  // products, 32 experts of 2048 x 2048, 4 each: 24 tokens 194 / 139, 128 209 / 147 (5.5 TB/s), 384 210 / 158, 800 224 / 179,
  // 3000 476 / 474; with more rows it costs 2 % (7680 tokens of 3, ff 3072: 779 / 798)
  const int spread = R <= E * 512;
  hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(SORT_NT), 0, st, idx, R, E, BM, rows, tiles);
#define MOE_PAIR(...) launch_pair<__VA_ARGS__>(h, w_gu, w_down, rows, tiles, y, out, mt, R, E, top, W, ff, act, row_w, limit, spread, st)
  if (BM == 256) return MOE_PAIR(256, 256, 2, 4, 2);
  if (BM == 128) return MOE_PAIR(128, 128, 2, 2, 2, true);
  if (BM == 64) return MOE_PAIR(64, 128, 1, 4, 3);
  return MOE_PAIR(32, 128, 1, 4, 3);
#undef MOE_PAIR
}

}  // extern "C"
