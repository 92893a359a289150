// Projections of 17 to 64 rows: y[M, N] = x[M, K] . W[N, K]^T (+ bias), bf16, fp16 or int8, over the fragment-packed weight of the
// decode GEMVs (gemv_bf16.hip, gemm_i8.h: byte for byte the same tiles of 16 rows x 64 bytes, so int8 operands are read as half as
// many 16-bit numbers).
//
// Bound by the weights' bytes, then by what reading the rows costs beside them.  A workgroup is 8 waves on NT tiles of 16 outputs;
// wave w takes the k-pairs (2 KiB of a tile) w, w + 8, ... and holds one pair of each tile in flight while another is multiplied.
// The rows of a k-pair come as whole 128-byte lines into the wave's own LDS (LDS-DMA, 8 rows a KiB, 16-byte chunk c of row r at
// c ^ (r & 7)); read in fragment order from memory, 16 rows x 64 B, a KiB takes twice as many lines through the L1 (4096 x 11008, 64 rows,
// 25.7 -> 22.4 us; 2048 x 8192, 32 rows, 20.8 -> 15.8).  No barrier until the waves' sums meet.  NT spreads the tiles over one
// round of the CUs: each further tile of a workgroup saves one reading of the rows.
//
// us, 18 / 32 / 64 rows, in a graph over 800 MB of weights, here | before (the 128-row ring kernel, or the library where it was ahead):
//   12288 x 4096           19.7 / 20.9 / 24.8 | 23.9 / 24.4 / 26.4       2048 x 2048   5.4 / 6.0 / 7.9 | 8.7 / 8.9 / 9.2
//   8192 x 2048             9.0 /  9.5 / 10.7 | 11.8 / 12.0 / 12.0       2048 x 8192  13.9 / 15.8 / 22.1 | 14.1 / 16.4 / 23.0
//   SwiGLU 22016 x 4096    33.4 / 34.1 (40: 36.1) | 39.0 / 39.5 (39.9)   16384 x 2048 14.8 / 15.5 / 17.3 | 21.7 / 21.9 / 24.0
//   4 slices, 4096 x 4096   9.5 /  9.8 / 11.5 | 11.7 / 12.1 / 12.4       4096 x 11008 18.3 / 18.9 / 22.4 | 22.1 / 21.9 / 23.8
// int8 (plain outputs; 30 shapes of 256 to 128256 outputs, K up to 32 N: 0.71 of the time before, at the worst 1.02): us, 17 / 45 / 64 rows, here |
// before (the decode GEMV with four row blocks):
//   7680 x 2560   6.5 / 8.0 / 8.8 | 10.7 / 17.0 / 18.8     2560 x 10240  11.1 / 14.2 / 16.6 | 13.8 / 22.2 / 24.8     12288 x 4096  12.1 / 14.3 / 15.4 | 13.4 / 18.3 / 19.1
#include "gemv_bf16.h"

namespace {
constexpr int GR_NW = 8;
constexpr int ROWS_OUT = 0, ROWS_GLU = 1, ROWS_PART = 2;
constexpr int DT_BF16 = 0, DT_FP16 = 1, DT_I8 = 2;
constexpr int OUTLIERS = 32;                                // outlier columns in LDS at a time

struct RowsArgs {
  const bf16_t *x, *w, *bias, *add;                         // bias [N], add [M, N]: may be null
  void* out;
  int M, N, K, S, act;                                      // act (ROWS_OUT): 0, or gelu of the 16-bit output (2 tanh, 3 erf)
  // int8: scales of the rows and of the outputs; LLM.int8's columns (count null: none): x before quantisation [M, 2 K], W^T [2 K, N]
  const float *sa, *sw;
  const bf16_t* xo;
  const int *cols, *count;
  const int8_t* wt;
  const float* scb;
};
template <int DT>
struct Sum {
  using type = v4f;
};
template <>
struct Sum<DT_I8> {
  using type = v4i;
};
template <int DT>
__device__ __forceinline__ typename Sum<DT>::type rows_mma(const v8s& w, const v4i& x, const typename Sum<DT>::type& c) {
  if constexpr (DT == DT_I8) return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, w), x, c, 0, 0, 0);
  else return mfma_16<DT == DT_FP16>(w, __builtin_bit_cast(v8s, x), c);
}

__device__ __forceinline__ void glds16(const void* g, void* lds_base) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)lds_base, 16, 0, 0);
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)((__attribute__((address_space(3))) const void*)p);
}
// A k-pair's rows from the LDS, MB 16-row blocks and two halves, and the wait for them in one block: between a read and its wait the
// compiler would take the registers as written.  (Plain loads would wait for the LDS-DMA in flight.)
template <int MB>
__device__ __forceinline__ void read_rows(uint32_t b0, uint32_t b1, v4i (&a)[2][MB]) {
  static_assert(MB >= 2 && MB <= 4, "17 to 64 rows");
  if constexpr (MB == 2)
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\t"
                 "ds_read_b128 %2, %4 offset:2048\n\tds_read_b128 %3, %5 offset:2048\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(a[0][0]), "=&v"(a[1][0]), "=&v"(a[0][1]), "=&v"(a[1][1]) : "v"(b0), "v"(b1) : "memory");
  else if constexpr (MB == 3)
    asm volatile("ds_read_b128 %0, %6\n\tds_read_b128 %1, %7\n\t"
                 "ds_read_b128 %2, %6 offset:2048\n\tds_read_b128 %3, %7 offset:2048\n\t"
                 "ds_read_b128 %4, %6 offset:4096\n\tds_read_b128 %5, %7 offset:4096\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(a[0][0]), "=&v"(a[1][0]), "=&v"(a[0][1]), "=&v"(a[1][1]), "=&v"(a[0][2]), "=&v"(a[1][2])
                 : "v"(b0), "v"(b1) : "memory");
  else
    asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\t"
                 "ds_read_b128 %2, %8 offset:2048\n\tds_read_b128 %3, %9 offset:2048\n\t"
                 "ds_read_b128 %4, %8 offset:4096\n\tds_read_b128 %5, %9 offset:4096\n\t"
                 "ds_read_b128 %6, %8 offset:6144\n\tds_read_b128 %7, %9 offset:6144\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(a[0][0]), "=&v"(a[1][0]), "=&v"(a[0][1]), "=&v"(a[1][1]), "=&v"(a[0][2]), "=&v"(a[1][2]), "=&v"(a[0][3]),
                   "=&v"(a[1][3])
                 : "v"(b0), "v"(b1) : "memory");
}
// tiles whose sums meet at a time: at most 128 KiB of them, gate and up tiles together
constexpr int sums_together(int MB, int NT, bool glu) {
  int c = NT;
  while (c * MB > 16 || NT % c != 0 || (glu && c % 2 != 0)) --c;
  return c;
}

template <int MB, int NT, int EPI, int DT>
__global__ void __launch_bounds__(GR_NW * 64, 2) gemm_rows16_kernel(RowsArgs p) {
  using Acc = typename Sum<DT>::type;
  constexpr bool GLU = EPI == ROWS_GLU, HF = DT == DT_FP16, I8 = DT == DT_I8;
  static_assert(!I8 || EPI == ROWS_OUT, "int8: plain outputs");
  constexpr int CT = sums_together(MB, NT, GLU), LOADS = 2 * MB + 2 * NT;   // of a wave and k-pair
  constexpr int XW = 2 * MB * 2048, RB = GR_NW * MB * CT * 1024, LB = GR_NW * XW > RB ? GR_NW * XW : RB;
  __shared__ __attribute__((aligned(1024))) char lds[LB];    // the waves' rows (two k-pairs each), then their sums
  __shared__ float xs[I8 ? OUTLIERS : 1][I8 ? 16 * MB : 1];  // outlier columns of the rows
  Acc (*red)[MB * CT][64] = reinterpret_cast<Acc (*)[MB * CT][64]>(lds);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15;
  const int M = p.M, N = p.N, K = p.K, KP = K / 64, nt = N / 16;
  const int grp = EPI == ROWS_PART ? (int)blockIdx.x / p.S : (int)blockIdx.x, ks = EPI == ROWS_PART ? (int)blockIdx.x % p.S : 0;
  const int kbeg = EPI == ROWS_PART ? KP * ks / p.S : 0, kend = EPI == ROWS_PART ? KP * (ks + 1) / p.S : KP;
  const bf16_t* wr[NT];                                     // GLU: gate tiles, then the up tiles of the same features
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    int t = min(grp * NT + j, nt - 1);
    if constexpr (GLU) t = min(grp * (NT / 2) + j % (NT / 2), nt / 2 - 1) + (j < NT / 2 ? 0 : nt / 2);
    wr[j] = p.w + ((size_t)t * (2 * KP) * 64 + lane) * 8;
  }
  const bf16_t* xr[2 * MB];                                 // 8 rows of 64 k each (rows past M: the last one again)
#pragma unroll
  for (int m = 0; m < 2 * MB; ++m) xr[m] = p.x + (size_t)min(8 * m + (lane >> 3), M - 1) * K + 8 * ((lane & 7) ^ (lane >> 3));
  char* const xw = lds + wave * XW;
  const uint32_t fr = lds_addr(xw) + (r >> 3) * 1024 + (r & 7) * 128 + (((lane >> 4) ^ (r & 7)) << 4);
  const int n = kend - kbeg > wave ? (kend - kbeg - wave + GR_NW - 1) / GR_NW : 0;   // this wave's k-pairs

  Acc acc[MB][NT];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[m][j] = Acc{};
  v8s A[NT][2], B[NT][2];
  auto load = [&](int u, v8s (&f)[NT][2]) {                  // k-pair u of this wave
    const size_t kp = kbeg + wave + GR_NW * u;
#pragma unroll
    for (int m = 0; m < 2 * MB; ++m) glds16(xr[m] + kp * 64, xw + (u & 1) * (XW / 2) + m * 1024);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      f[j][0] = ld_nt(wr[j] + kp * 1024);
      f[j][1] = ld_nt(wr[j] + kp * 1024 + 512);
    }
    asm volatile("" ::: "memory");
  };
  // `more`: the next k-pair's loads, and no others, are behind this one's
  auto mma = [&](int u, v8s (&f)[NT][2], bool more) {
    if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    v4i a[2][MB];
    const uint32_t b0 = fr + (u & 1) * (XW / 2), b1 = b0 ^ 64;
    read_rows<MB>(b0, b1, a);                                // (all there: the next load may overwrite them)
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int m = 0; m < MB; ++m) acc[m][j] = rows_mma<DT>(f[j][s], a[s][m], acc[m][j]);
  };
  if (n > 0) load(0, A);
  if (n > 1) load(1, B);
  int u = 0;
  for (; u + 3 < n; u += 2) {                                // no guard inside: the counts above are constants
    mma(u, A, true);
    load(u + 2, A);
    mma(u + 1, B, true);
    load(u + 3, B);
  }
  const int left = n - u;
  if (left > 0) mma(u, A, left > 1);
  if (left > 2) load(u + 2, A);
  if (left > 1) mma(u + 1, B, left > 2);
  if (left > 2) mma(u + 2, A, false);

  // the weights are the products' first operand: a lane holds outputs 4 (lane >> 4) + 0..3 of row r of each 16 x 16 block
  const int c4 = 4 * (lane >> 4);
#pragma unroll
  for (int c0 = 0; c0 < NT; c0 += CT) {
    __syncthreads();                                         // the rows, or the sums before, have been read
#pragma unroll
    for (int c = 0; c < CT; ++c)                             // GLU: a gate tile and its up tile side by side
#pragma unroll
      for (int m = 0; m < MB; ++m) red[wave][c * MB + m][lane] = acc[m][GLU ? (c & 1) * (NT / 2) + (c0 + c) / 2 : c0 + c];
    __syncthreads();
    constexpr int BLOCKS = MB * CT / (GLU ? 2 : 1), OWN = (BLOCKS + GR_NW - 1) / GR_NW;   // 16 x 16 outputs, of a wave
    float extra[I8 ? OWN : 1][4];
    bool outliers = false;
    if constexpr (I8) {
      const int nt_out = p.count != nullptr ? *p.count : 0;
      outliers = nt_out > 0;
#pragma unroll
      for (int o = 0; o < OWN; ++o)
#pragma unroll
        for (int q = 0; q < 4; ++q) extra[o][q] = 0.f;
      for (int j0 = 0; j0 < nt_out; j0 += OUTLIERS) {        // (no such column: one load)
        __syncthreads();
        for (int i = threadIdx.x; i < OUTLIERS * 16 * MB; i += GR_NW * 64) {
          const int jj = i / (16 * MB), row = i % (16 * MB);
          xs[jj][row] = j0 + jj < nt_out && row < M ? bf2f(p.xo[(size_t)row * (2 * K) + p.cols[j0 + jj]]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
          const int b = wave + o * GR_NW, col = min(16 * (grp * NT + c0 + b / MB) + c4, N - 4);
          if (b >= BLOCKS) continue;
          for (int jj = 0; jj < min(OUTLIERS, nt_out - j0); ++jj) {
            const char4 w4 = *reinterpret_cast<const char4*>(p.wt + (size_t)p.cols[j0 + jj] * N + col);
            const float xv = xs[jj][16 * (b % MB) + r];
            extra[o][0] += xv * (float)w4.x;
            extra[o][1] += xv * (float)w4.y;
            extra[o][2] += xv * (float)w4.z;
            extra[o][3] += xv * (float)w4.w;
          }
        }
      }
    }
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const int b = wave + o * GR_NW;
      if (b >= BLOCKS) continue;
      const int m = b % MB, c = (b / MB) * (GLU ? 2 : 1), row = 16 * m + r;
      auto total = [&](int s) {
        Acc t = red[0][s][lane];
#pragma unroll
        for (int w = 1; w < GR_NW; ++w) t += red[w][s][lane];
        return t;
      };
      const Acc s0 = total(c * MB + m);
      const int t = GLU ? grp * (NT / 2) + (c0 + c) / 2 : grp * NT + c0 + c, F = GLU ? N / 2 : N, col = 16 * t + c4;
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = (float)s0[q];
      if constexpr (GLU) {
        const v4f s1 = total((c + 1) * MB + m);
        if (row >= M || t >= nt / 2) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float g = e2f<HF>(f2e<HF>(v[q] + (p.bias != nullptr ? e2f<HF>(p.bias[col + q]) : 0.f)));
          const float h = e2f<HF>(f2e<HF>(s1[q] + (p.bias != nullptr ? e2f<HF>(p.bias[F + col + q]) : 0.f)));
          v[q] = g / (1.f + __expf(-g)) * h;
        }
      } else {
        if (row >= M || t >= nt) continue;
        if constexpr (I8) {
          const float sr = p.sa[row];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            v[q] = v[q] * sr;
            v[q] = v[q] * p.sw[col + q] + (p.bias != nullptr ? bf2f(p.bias[col + q]) : 0.f);
            if (outliers) v[q] = bf2f(f2bf(v[q])) + extra[o][q] * (p.scb[col + q] / 127.f);
          }
        } else if (p.bias != nullptr && ks == 0) {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] += e2f<HF>(p.bias[col + q]);
        }
        if constexpr (EPI == ROWS_PART) {
          *reinterpret_cast<float4*>((float*)p.out + ((size_t)ks * M + row) * N + col) = float4{v[0], v[1], v[2], v[3]};
          continue;
        }
        if (p.act != 0)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float y = e2f<HF>(f2e<HF>(v[q])), k0 = 0.7978845608028654f, k1 = 0.044715f;
            v[q] = p.act == 2 ? 0.5f * y * (1.f + tanhf(k0 * (y + k1 * y * y * y))) : 0.5f * y * (1.f + erff(y * 0.7071067811865476f));
          }
        if (p.add != nullptr)                                // rnd(rnd(y) + add): the unfused sum
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = e2f<HF>(f2e<HF>(v[q])) + e2f<HF>(p.add[(size_t)row * N + col + q]);
      }
      *reinterpret_cast<uint2*>((bf16_t*)p.out + (size_t)row * F + col) = uint2{pack_e2<HF>(v[0], v[1]), pack_e2<HF>(v[2], v[3])};
    }
  }
}

template <int MB, int NT, int EPI, int DT>
int launch_rows(const RowsArgs& p, hipStream_t st) {
  const int tiles = EPI == ROWS_GLU ? p.N / 32 : p.N / 16, per = EPI == ROWS_GLU ? NT / 2 : NT;
  hipLaunchKernelGGL((gemm_rows16_kernel<MB, NT, EPI, DT>), dim3((tiles + per - 1) / per * p.S), dim3(GR_NW * 64), 0, st, p);
  return (int)hipGetLastError();
}

// Tiles of a workgroup: what one round of 256 of them needs, up to 4 (SwiGLU: 3 pairs; 64 rows of three pairs spill).  Outputs
// that need more take several rounds of small workgroups, two to a CU (32000 x 4096, 18 rows, 2 / 3 / 4 / 6 tiles: 46.0 / 48.3 / 49.5 / 57.4).
template <int MB, int EPI, int DT>
int rows_dispatch(const RowsArgs& p, hipStream_t st) {
  if constexpr (EPI == ROWS_GLU) {
    const int pairs = p.N / 32;
    if (pairs <= 256) return launch_rows<MB, 2, EPI, DT>(p, st);
    if constexpr (MB < 4)
      if (pairs > 512 && pairs <= 768) return launch_rows<MB, 6, EPI, DT>(p, st);
    return launch_rows<MB, 4, EPI, DT>(p, st);
  } else {
    const int tiles = p.N / 16 * p.S;
    if (tiles <= 256) return launch_rows<MB, 1, EPI, DT>(p, st);
    if (tiles <= 512 || (EPI == ROWS_OUT && tiles > 1024)) return launch_rows<MB, 2, EPI, DT>(p, st);
    if (tiles <= 768) return launch_rows<MB, 3, EPI, DT>(p, st);
    return launch_rows<MB, 4, EPI, DT>(p, st);
  }
}

template <int EPI, int DT>
int rows_run(const RowsArgs& p, hipStream_t st) {
  if (p.M <= 32) return rows_dispatch<2, EPI, DT>(p, st);
  return p.M <= 48 ? rows_dispatch<3, EPI, DT>(p, st) : rows_dispatch<4, EPI, DT>(p, st);
}
}  // namespace

// Whether the kernel is the one for these sizes (epi 0: plain, 1: SwiGLU, 3: split-K).  Above 32 rows the rows' reads outweigh what
// several rounds of workgroups save on 128-row tiles: us, here / ring kernel, 50304 x 2048, 40 rows 49.2 / 41.6, 32000 x 4096, 64 rows 57.6 /
// 49.8; SwiGLU 28672 x 4096, 40 rows 49.0 / 47.0, 22016 x 4096, 64 rows 48.8 / 44.2.
extern "C" int edge_gemm_rows16_ok(int M, int N, int K, int epi) {
  if (M < 17 || M > 64 || K <= 0 || K % 64 != 0 || N <= 0 || N % (epi == 1 ? 32 : 16) != 0) return 0;
  if (epi == 1) return M <= 32 || N <= 32 * 512 || (M <= 48 && N <= 32 * 768);
  return epi == 3 || M <= 32 || N <= 16 * 1024;
}

// x [M, K], w packed [N, K], 16-byte aligned.  epi 0: out [M, N] (+ add [M, N]); 1: w = [gate | up], out = silu(gate) * up [M, N / 2];
// 2 / 3: gelu (tanh / erf) of the 16-bit output.  S > 1: fp32 slices out [S, M, N] (epi 0, bias in slice 0).  -2: not taken.
extern "C" int edge_gemm_rows16(const void* x, const void* w, const void* bias, const void* add, void* out, int M, int N, int K,
                                int epi, int S, int h16, hipStream_t st) {
  if (edge_gemm_rows16_ok(M, N, K, S > 1 ? 3 : epi == 1 ? 1 : 0) == 0 || epi < 0 || epi > 3 || S < 1 || S > K / 64) return -2;
  if ((epi != 0 || h16) && S > 1) return -2;
  if (add != nullptr && (epi != 0 || S > 1)) return -2;
  const RowsArgs p{(const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)bias, (const bf16_t*)add, out, M, N, K, S, epi >= 2 ? epi : 0,
                   nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  if (S > 1) return rows_run<ROWS_PART, DT_BF16>(p, st);
  if (epi == 1) return h16 ? rows_run<ROWS_GLU, DT_FP16>(p, st) : rows_run<ROWS_GLU, DT_BF16>(p, st);
  return h16 ? rows_run<ROWS_OUT, DT_FP16>(p, st) : rows_run<ROWS_OUT, DT_BF16>(p, st);
}

// int8: A [M, K] row-major with scales sa [M], w packed (K / 64 tiles a row block), scales sw [N], out bf16 [M, N] = gelu (act 2 / 3, 0:
// none) of the rounded output, + add [M, N].  count not null: LLM.int8's outlier columns cols [*count] of x [M, K] bf16 against wt = W^T
// [K, N], scaled by scb / 127, join the rounded product.  -2: not taken.
extern "C" int edge_gemm_rows_i8(const void* A, const float* sa, const void* w, const float* sw, const void* bias, const void* add, void* out,
                                 int M, int N, int K, int act, const void* x, const int* cols, const int* count, const void* wt,
                                 const float* scb, hipStream_t st) {
  if (K % 128 != 0 || edge_gemm_rows16_ok(M, N, K / 2, 0) == 0 || (act != 0 && act != 2 && act != 3) ||
      ((uintptr_t)A | (uintptr_t)w) % 16 != 0 || (count != nullptr && (uintptr_t)wt % 4 != 0))
    return -2;
  const RowsArgs p{(const bf16_t*)A, (const bf16_t*)w, (const bf16_t*)bias, (const bf16_t*)add, out, M, N, K / 2, 1, act, sa, sw,
                   (const bf16_t*)x, cols, count, (const int8_t*)wt, scb};
  return rows_run<ROWS_OUT, DT_I8>(p, st);
}
