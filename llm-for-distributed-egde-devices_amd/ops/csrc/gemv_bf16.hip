// Decode GEMV for bf16 weights: y[M, N] = x[M, K] . W[N, K]^T (+ bias) -> bf16, M <= 64
// (MB = 1..4 row blocks of 16: every weight fragment feeds MB MFMAs, so 17-64 decode rows read the
// weights once instead of hipBLASLt's small-M kernels).
// The fp16/bf16 evaluators (Phi-2, Pythia-1B, Llama-3.2-1B at batch 1) spend
// most of a decode step here; hipBLASLt's small-M kernels stream the weights at about 2 TB/s.
//
// Weights are read in MFMA fragment order (ops.pack_bf16_weight, a decode-only copy of the HF
// [N, K] tensor that prefill keeps using): 1 KiB tiles of 16 rows x 32 k, tile (nt, kt) at
// ((nt * K/32) + kt) * 512 elements, lane l's 8 elements = W[16 nt + (l & 15)][32 kt + 8 (l >> 4) ..]
// — the B fragment of v_mfma_f32_16x16x32_bf16.  A wave walks K in pairs of k-steps, i.e. 2 KiB
// of contiguous weights per tile per pair (the [N, K] layout gave each load instruction 16 rows x
// 64 B: 36 % more bytes fetched and 2.3 TB/s on Llama-3.2-1B's gate_up).  Few rows run gemv_tiles_body (gemv_bf16.h):
// one tile of a workgroup's at a time.  More rows, where a tile's reads of the rows weigh: a workgroup = 16 waves
// on NTW 16-column tiles; wave w takes k-pairs w, w + 16, ..., keeping U pairs of weight loads in
// flight (nontemporal: each weight byte is read once per step).  The 16 partial tiles are
// reduced through LDS.  Rows >= M load a clamped row and are never stored.
//   EPI_OUT: + bias, bf16 [M, N].
//   EPI_GLU: W = [gate (F rows) | up (F rows)] (the natural gate_up concatenation); a workgroup's
//            tiles are NTW/2 gate tiles and the matching up tiles, and it writes
//            h = silu(gate) * up as bf16 [M, F] (gate and up rounded to bf16 first, as the
//            unfused GEMM output is) — the separate SwiGLU launch disappears.
//   EPI_GELU_TANH / EPI_GELU: gelu(bf16(y + bias)) -> bf16 [M, N] (Phi-2 / Pythia MLP up
//            projection; the same math as rowwise.hip::act_kernel modes 1 / 2).
//   EPI_PART: split-K, workgroup (group, ks) reduces k-pairs [KP ks / S, KP (ks + 1) / S) and
//            writes fp32 partials part[ks][M][N] (bias in slice 0) for a norm kernel that sums
//            them (the o / down projections of RMSNorm decoders; N = 2048 has only 128 tiles).
// HF: fp16 activations / weights / outputs on v_mfma_f32_16x16x32_f16 (the reference's fp16 agents,
// Phi-2 / Pythia); the same fragment layout and epilogues with fp16 roundings.
#include "gemv_bf16.h"

namespace {
template <int MB, int NTW, int U, int EPI, bool HF>
__global__ void __launch_bounds__(GEMV_NW * 64) gemv_bf16_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                            const bf16_t* __restrict__ bias, bf16_t* __restrict__ out,
                                                            int M, int N, int K, int F, int S,
                                                            const bf16_t* __restrict__ add) {
  gemv_bf16_body<MB, NTW, U, EPI, HF>((int)blockIdx.x, A, W, bias, out, M, N, K, F, S, add);
}

template <int MB, int NTW, int U, int EPI, bool HF>
int launch_mb(const void* A, const void* W, const void* bias, void* out, int M, int N, int K, int F, int tiles,
              hipStream_t st, int S, const void* add = nullptr) {
  constexpr int per = EPI == EPI_GLU ? NTW / 2 : NTW;       // output tiles a workgroup
  const int groups = (tiles + per - 1) / per;
  hipLaunchKernelGGL((gemv_bf16_kernel<MB, NTW, U, EPI, HF>), dim3(groups * S), dim3(GEMV_NW * 64), 0, st,
                     (const bf16_t*)A, (const bf16_t*)W, (const bf16_t*)bias, (bf16_t*)out, M, N, K, F, S,
                     (const bf16_t*)add);
  return (int)hipGetLastError();
}

template <int PRE, int EPI, bool HF, int NRM, int RB, int TWICE>
__global__ void __launch_bounds__(GEMV_NW * 64, TWICE ? 8 : 4) gemv_tiles_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                                 const bf16_t* __restrict__ bias, bf16_t* __restrict__ out,
                                                                 int M, int N, int K, int F, int S,
                                                                 const bf16_t* __restrict__ add, NormIn16 na) {
  gemv_tiles_body<GEMV_NW, 1, PRE, EPI, HF, NRM, RB>((int)blockIdx.x, (int)gridDim.x, A, W, bias, out, M, N, K, F, S, add, na);
}

// Workgroups of the tiles form.  Without a norm up to 1024, two to a CU and two rounds of them: 128256 x 2048 takes 82 us on
// 256, 77 on 512, 75.8 on 1024, 75.6 on 2048.  With a norm one to a CU (the norm's loads and sums are each workgroup's own):
// 22016 x 4096 29.4 us on 256, 29.6 on 512, 30.9 on 1024; 6144 x 4096 (384 tiles) 10.1 on 256, 11.5 on 384.
// Two to a CU are 64 registers a lane, which the forms without a norm are held to (at 66 to 106, one to a CU: 8192 x 2048, 16 rows,
// GELU 10.9 us, now 9.6; 6144 x 4096 16.6, 15.3).  Not with an addend of up to 256 tiles: its loads then wait for each other, and one
// workgroup a CU is all there is (2560 x 10240 at 8 rows 13.5 us, held to 64 15.8; 8192 x 2048, 512 tiles, at 8 rows 9.5 / 8.3).
template <int EPI, bool HF, int NRM, int RB>
int launch_tiles(const void* A, const void* W, const void* bias, void* out, int M, int N, int K, hipStream_t st, int S = 1,
                 const void* add = nullptr, const NormIn16& na = NormIn16{}) {
  const int tiles = N / 16 * S, cap = NRM > 0 ? 256 : 1024;
  const dim3 grid(EPI == EPI_PART || tiles < cap ? tiles : cap);
#define TILES(TW)                                                                                                              \
  hipLaunchKernelGGL((gemv_tiles_kernel<(NRM > 0 ? 2 : 1), EPI, HF, NRM, RB, TW>), grid, dim3(GEMV_NW * 64), 0, st, (const bf16_t*)A, \
                     (const bf16_t*)W, (const bf16_t*)bias, (bf16_t*)out, M, N, K, EPI == EPI_GLU ? N / 2 : 0, S, (const bf16_t*)add, na)
  if constexpr (EPI == EPI_ADD && RB > 1) {
    if (tiles <= 256) TILES(0);
    else TILES(1);
  } else TILES(NRM == 0);
#undef TILES
  return (int)hipGetLastError();
}

template <int EPI, bool HF>
int launch_tiles_rows(const void* A, const void* W, const void* bias, void* out, int M, int N, int K, hipStream_t st, int S = 1,
                      const void* add = nullptr) {
  if (M <= 4) return launch_tiles<EPI, HF, 0, 1>(A, W, bias, out, M, N, K, st, S, add);
  if (M <= 8) return launch_tiles<EPI, HF, 0, 2>(A, W, bias, out, M, N, K, st, S, add);
  return launch_tiles<EPI, HF, 0, 4>(A, W, bias, out, M, N, K, st, S, add);
}

// Whether the tiles form takes M rows: up to 4 always, 5 to 16 where its tiles' reads of the rows (each tile reads all of
// them) stay small beside the weights.  us, several tiles a workgroup / tiles form: 1 row 1024 x 1024 3.4 / 2.7, 4096 x 2048 (4 rows)
// 5.4 / 4.7, 32000 x 1024 12.7 / 11.8; 12 rows 4096 x 2048 6.1 / 5.4, 12288 x 4096 22.4 / 19.5, 16 rows 8192 x 2048 9.2 / 9.2, 32000 x 2048
// 23.5 / 27; SwiGLU 16384 x 2048 1 row 13.0 / 11.7, 8 rows 13.3 / 13.8.  Where two tiles a workgroup (N from 8192 on) take as many rounds of
// the CUs and all their k-pairs in whole fours, their halved reads win from some 10 rows on: 8192 x 4096, 9 / 12 / 16 rows, 14.3 / 13.6 /
// 14.1 against 13.7 / 13.9 / 15.5, 14336 x 8192 43.0 / 43.6 / 44.0 against 43.0 / 46 / 51.
bool tiles_form(int M, int N, int K, int epi) {
  if (M <= 4) return true;
  if (M > 16 || epi == EPI_GLU || N >= 16384) return false;
  const int nt = N / 16;
  return M <= 10 || nt < 512 || K % 4096 != 0 || (nt + 255) / 256 < 2 * ((nt + 511) / 512);
}

// NTW / U chosen for one row block (NTW = 1 has none: the tiles form takes those); more row blocks keep U = 2 (registers) and at
// most 8 / MB tiles (the LDS reduction holds MB x NTW tiles of 16 waves)
template <int NTW, int U, int EPI, bool HF>
int launch(const void* A, const void* W, const void* bias, void* out, int M, int N, int K, int F, int tiles,
           hipStream_t st, int S = 1, const void* add = nullptr) {
  constexpr int G = EPI == EPI_GLU ? 2 : 1;                 // GLU keeps gate / up pairs
  constexpr int N2 = NTW > 4 ? 4 : (NTW < G ? G : NTW), N34 = NTW > 2 ? 2 : (NTW < G ? G : NTW);
  const int mb = (M + 15) / 16;
  if constexpr (NTW > 1) {
    if (mb <= 1) return launch_mb<1, NTW, U, EPI, HF>(A, W, bias, out, M, N, K, F, tiles, st, S, add);
  }
  if (mb <= 2) return launch_mb<2, N2, 2, EPI, HF>(A, W, bias, out, M, N, K, F, tiles, st, S, add);
  if (mb == 3) return launch_mb<3, N34, 2, EPI, HF>(A, W, bias, out, M, N, K, F, tiles, st, S, add);
  return launch_mb<4, N34, 2, EPI, HF>(A, W, bias, out, M, N, K, F, tiles, st, S, add);
}

// W: fragment-packed bf16 (ops.pack_bf16_weight).  epi 0: out bf16 [M, N] (+ the bf16 addend `add`
// [M, N] when not null: a parallel-residual block's other branch); epi 1 (GLU):
// W = [gate | up] with N = 2F, out = silu(gate) * up bf16 [M, F] (F % 16 == 0); epi 2 / 3: gelu (tanh / erf) of the bf16 output; epi 7: epi 0's
// numbers as fp32 (bf16, M <= 16, no addend).  M <= 64, K % 64 == 0,
// N % 16 == 0.  Returns -2 for shapes it does not take.
template <bool HF>
int gemv_run(const void* A, const void* W, const void* bias, void* out, int M, int N, int K, int epi, hipStream_t st,
             const void* add) {
  if (M <= 0 || M > 64 || K % 64 != 0 || N % 16 != 0 || N <= 0 || K <= 0) return -2;
  if (epi == EPI_F32) {                                      // scores that a program reads in fp32: up to 16 bf16 rows, no copy behind them
    if (HF || M > 16 || add != nullptr) return -2;
    const int nt = N / 16;
    if (tiles_form(M, N, K, epi)) return launch_tiles_rows<EPI_F32, false>(A, W, bias, out, M, N, K, st);
    return nt >= 1024 ? launch_mb<1, 4, 2, EPI_F32, false>(A, W, bias, out, M, N, K, 0, nt, st, 1)
                      : launch_mb<1, 2, 4, EPI_F32, false>(A, W, bias, out, M, N, K, 0, nt, st, 1);
  }
  if (tiles_form(M, N, K, epi)) {
    switch (epi) {
      case EPI_OUT: return add == nullptr ? launch_tiles_rows<EPI_OUT, HF>(A, W, bias, out, M, N, K, st)
                                          : launch_tiles_rows<EPI_ADD, HF>(A, W, bias, out, M, N, K, st, 1, add);
      case EPI_GLU: return N % 32 != 0 ? -2 : launch_tiles<EPI_GLU, HF, 0, 1>(A, W, bias, out, M, N, K, st);
      case EPI_GELU_TANH: return launch_tiles_rows<EPI_GELU_TANH, HF>(A, W, bias, out, M, N, K, st);
      case EPI_GELU: return launch_tiles_rows<EPI_GELU, HF>(A, W, bias, out, M, N, K, st);
      default: return -2;
    }
  }
  if (epi == EPI_GLU) {
    if (N % 32 != 0) return -2;
    const int F = N / 2, ft = F / 16;
    if (ft >= 512) return launch<4, 2, EPI_GLU, HF>(A, W, bias, out, M, N, K, F, ft, st);
    return K >= 4096 ? launch<2, 4, EPI_GLU, HF>(A, W, bias, out, M, N, K, F, ft, st)
                     : launch<2, 2, EPI_GLU, HF>(A, W, bias, out, M, N, K, F, ft, st);
  }
  if (epi != EPI_OUT && epi != EPI_GELU_TANH && epi != EPI_GELU) return -2;
  const int nt = N / 16;
  // ~256 workgroups: one tile each below 512 tiles, then 2 or 4
#define PICK(EP, ADD)                                                                                       \
  if (nt >= 1024) return launch<4, 2, EP, HF>(A, W, bias, out, M, N, K, 0, nt, st, 1, ADD);                   \
  if (nt >= 512) return launch<2, 4, EP, HF>(A, W, bias, out, M, N, K, 0, nt, st, 1, ADD);                    \
  return launch<1, 2, EP, HF>(A, W, bias, out, M, N, K, 0, nt, st, 1, ADD);
  if (epi == EPI_GELU_TANH) { PICK(EPI_GELU_TANH, nullptr) }
  if (epi == EPI_GELU) { PICK(EPI_GELU, nullptr) }
  PICK(EPI_OUT, add)                                         // optionally + a bf16 addend [M, N]
#undef PICK
}

// The 16-bit GEMV over RMSNorm(sum(parts) + residual) (norm16_prologue): M <= 4, K 2048 / 4096,
// S <= 4 slices; epi 0 (EPI_OUT) or 1 (EPI_GLU).  Not taken: 3 or 4 slices of K = 4096 before 16384 outputs or more (no
// model's projections leave that many slices; the norm is a launch of its own there).
template <bool HF, int NRM>
int gemv_norm_geo(const NormIn16& na, const void* W, const void* bias, void* out, int M, int N, int K, int epi,
                  hipStream_t st) {
  if (NRM == 20 && N / 16 >= 1024) return -2;
  if constexpr (NRM < 64) {
    if (epi == EPI_GLU) return launch_tiles<EPI_GLU, HF, NRM, 1>(nullptr, W, bias, out, M, N, K, st, 1, nullptr, na);
  } else {
    if (epi == EPI_GELU_TANH) return launch_tiles<EPI_GELU_TANH, HF, NRM, 1>(nullptr, W, bias, out, M, N, K, st, 1, nullptr, na);
    if (epi == EPI_GELU) return launch_tiles<EPI_GELU, HF, NRM, 1>(nullptr, W, bias, out, M, N, K, st, 1, nullptr, na);
  }
  return launch_tiles<EPI_OUT, HF, NRM, 1>(nullptr, W, bias, out, M, N, K, st, 1, nullptr, na);
}

// LayerNorm prologue over 16-bit rows x (+ residual): K <= 4096 (K % 64 == 0), epi 0 / 2 / 3.
template <bool HF>
int gemv_ln_run(const NormIn16& na, const void* W, const void* bias, void* out, int M, int N, int K, int epi,
                hipStream_t st) {
  if (M < 1 || M > NRM16_ROWS || K > 4096 || K % 64 != 0 || N % 16 != 0 || na.x == nullptr ||
      (epi != EPI_OUT && epi != EPI_GELU_TANH && epi != EPI_GELU) || na.res_out == nullptr || na.res == na.res_out ||
      na.x == na.res_out || na.x2 == na.res_out || (na.x2 != nullptr && na.y_out == na.x2) || na.y_out == na.x || na.y_out == na.res_out)
    return -2;
  return K <= 2048 ? gemv_norm_geo<HF, 64 + 8>(na, W, bias, out, M, N, K, epi, st)
                   : gemv_norm_geo<HF, 64 + 16>(na, W, bias, out, M, N, K, epi, st);
}

template <bool HF>
int gemv_norm_run(const NormIn16& na, const void* W, const void* bias, void* out, int M, int N, int K, int epi,
                  hipStream_t st) {
  if (M < 1 || M > NRM16_ROWS || na.S < 1 || na.S > 4 || (K != 2048 && K != 4096) || N % 16 != 0 ||
      (epi != EPI_OUT && epi != EPI_GLU) || (epi == EPI_GLU && N % 32 != 0) || na.res_out == nullptr ||
      na.res == na.res_out)
    return -2;
  if (K == 4096) return na.S <= 2 ? gemv_norm_geo<HF, 18>(na, W, bias, out, M, N, K, epi, st)
                                  : gemv_norm_geo<HF, 20>(na, W, bias, out, M, N, K, epi, st);
  return na.S <= 2 ? gemv_norm_geo<HF, 10>(na, W, bias, out, M, N, K, epi, st)
                   : gemv_norm_geo<HF, 12>(na, W, bias, out, M, N, K, epi, st);
}

// Split-K form: fp32 partial slices part [S, M, N] (bias in slice 0), one 16-column tile per group.
template <bool HF>
int gemv_splitk_run(const void* A, const void* W, const void* bias, float* part, int M, int N, int K, int S,
                    hipStream_t st) {
  if (M <= 0 || M > 64 || K % 64 != 0 || N % 16 != 0 || N <= 0 || S < 1 || S > K / 64) return -2;
  if (M <= 16) return launch_tiles_rows<EPI_PART, HF>(A, W, bias, part, M, N, K, st, S);
  return launch<1, 2, EPI_PART, HF>(A, W, bias, part, M, N, K, 0, N / 16, st, S);
}
}  // namespace

// h16: fp16 operands / outputs (fragment-packed fp16 weights), else bf16
extern "C" int edge_gemv_bf16(const void* A, const void* W, const void* bias, void* out, int M, int N, int K, int epi,
                              hipStream_t st, const void* add, int h16) {
  return h16 ? gemv_run<true>(A, W, bias, out, M, N, K, epi, st, add)
             : gemv_run<false>(A, W, bias, out, M, N, K, epi, st, add);
}

extern "C" int edge_gemv_bf16_splitk(const void* A, const void* W, const void* bias, float* part, int M, int N, int K,
                                     int S, hipStream_t st, int h16) {
  return h16 ? gemv_splitk_run<true>(A, W, bias, part, M, N, K, S, st)
             : gemv_splitk_run<false>(A, W, bias, part, M, N, K, S, st);
}

// 16-bit decode GEMV (M <= 4) over RMSNorm(sum of S fp32 slices part [S, M, K] + res) in its
// prologue; res may be null (a stage's first norm); res_out [M, K] gets the new residual rows
// (workgroup 0).  epi 0: out [M, N]; 1: SwiGLU of W = [gate | up], out [M, N / 2].  -2: not taken.
extern "C" int edge_gemv_bf16_norm(const float* part, int S, const void* res, const void* gamma, float eps,
                                   void* res_out, const void* W, const void* bias, void* out, int M, int N, int K,
                                   int epi, hipStream_t st, int h16) {
  const NormIn16 na{part, (const bf16_t*)res, (const bf16_t*)gamma, (bf16_t*)res_out, eps, S, nullptr, nullptr, nullptr,
                    nullptr, nullptr, nullptr};
  return h16 ? gemv_norm_run<true>(na, W, bias, out, M, N, K, epi, st)
             : gemv_norm_run<false>(na, W, bias, out, M, N, K, epi, st);
}

// 16-bit decode GEMV (M <= 4) over LayerNorm(x (+ x2, rounded) + res) (x2, res may be null) in its prologue; res_out
// [M, K] gets the sum (workgroup 0), y_out (when not null) the normalised rows, for a second consumer: under gamma2 /
// beta2 where those are given, else the same ones.  epi 0: out [M, N]; 2 / 3: gelu (tanh / erf).  -2: not taken.
extern "C" int edge_gemv_bf16_ln(const void* x, const void* x2, const void* res, const void* gamma, const void* beta,
                                 float eps, void* res_out, const void* W, const void* bias, void* out, int M, int N, int K,
                                 int epi, hipStream_t st, int h16, void* y_out, const void* gamma2, const void* beta2) {
  const NormIn16 na{nullptr, (const bf16_t*)res, (const bf16_t*)gamma, (bf16_t*)res_out, eps, 0, (const bf16_t*)x,
                    (const bf16_t*)x2, (const bf16_t*)beta, (bf16_t*)y_out, (const bf16_t*)gamma2, (const bf16_t*)beta2};
  return h16 ? gemv_ln_run<true>(na, W, bias, out, M, N, K, epi, st)
             : gemv_ln_run<false>(na, W, bias, out, M, N, K, epi, st);
}
