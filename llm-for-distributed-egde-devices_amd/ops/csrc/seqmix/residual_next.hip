// A sublayer's result joins the fp32 residual stream and the row that the next sublayer (or the output projection) reads is formed in
// the same launch, for the three kinds of layers that do the two in a row: LayerNorm of the result, then the stream's four-tap
// convolution (steps in which every sequence brings one token) or, behind the last layer, its LayerNorm; group RMS norm of the
// result, then the next group RMS norm; the two branches of a parallel mixer, then the next RMS norm.  (ops/seqmix.py has the rules;
// widths, types and addresses that do not fit run the separate kernels.)
//
// Bound by latency on decode-sized steps: each of the two launches was one chain of loads, a reduction over the row and a store, and
// the second began by reading back what the first had written.  A workgroup holds a row in registers, four numbers per access, and
// issues every load (weights and the convolution's tail too) before the first reduction.
// us, two launches / one, bf16 results: LayerNorm of a result and three parts, then taps, rows of 1024, 4 tokens 6.2 / 4.0, of 2048 6.7 /
// 5.0, 64 tokens 8.2 / 5.5; two group norms, 1024, 4 tokens 7.2 / 3.8, 4096 21.9 / 11.1, 2048 7.7 / 5.4, 34.2 / 23.6; branches, then
// a norm, 1024, 4 tokens 7.0 / 3.7, 2048 9.5 / 4.2, 4096 tokens 52.9 / 24.8.
#include "common.h"
#include "seqmix/row_parts.h"
#include "seqmix/route_few.h"

namespace {

__device__ __forceinline__ bool in_row(int i, int W) { return ((int)threadIdx.x + i * NT) * 4 < W; }
__device__ __forceinline__ int col(int i, int W) { return min(((int)threadIdx.x + i * NT) * 4, W - 4); }

// x += LayerNorm(y + sum_k pw[k] parts[k]) w + b;  out = x + sum_k cw[:, k] x_(pos - 3 + k), x_pos this row and the three before it
// the slot's tail [3][W] (zero before position 0), which moves up.  The sums are ln_residual4_kernel's and tap4_kernel's.
constexpr int RT_MOST = 1024, RT_ROWS = 256;                // widest row and most rows with the choice of experts in the launch
struct Taps {
  const float* w;                                            // [W, 4]
  float* state;                                              // [slots, 3, W]
  const int *tok_seq, *tok_pos, *seq_slot;
};
// by NW waves; done(c, o): the four numbers of out from column c on
template <typename T, int CH, int NW, typename E, typename F>
__device__ __forceinline__ void ln_residual_taps_row(size_t t, float* __restrict__ x, const T* __restrict__ y, const T* __restrict__ parts,
                                                     const float* __restrict__ pw, int K, const float* __restrict__ w,
                                                     const float* __restrict__ b, int W, float eps, const Taps& a, T* __restrict__ out,
                                                     float (*red)[NW], E&& early, F&& done) {
  const int pos = a.tok_pos[t], seq = a.tok_seq[t];
  float v[CH][4], xv[CH][4], wv[CH][4], bv[CH][4], sum = 0.f;
  float4 cw[CH][4];
  float tail[CH][3][4];
  const bool holds = NW == NT / 64 || __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * 256 < W;   // (a wave with part of the row)
  float* st = a.state + (size_t)a.seq_slot[seq] * 3 * W;
  if (holds) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = col(i, W);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i][e] = 0.f;
      if (y) load4<T>(y + t * W + c, v[i]);
      load4<float>(x + t * W + c, xv[i]);
      load4<float>(w + c, wv[i]);
      load4<float>(b + c, bv[i]);
#pragma unroll
      for (int e = 0; e < 4; ++e) cw[i][e] = *reinterpret_cast<const float4*>(a.w + (size_t)(c + e) * 4);
    }
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
      for (int k = 0; k < 3; ++k) load4<float>(st + (size_t)k * W + col(i, W), tail[i][k]);
  }
  early();
  if (holds) add_parts<T, CH>(v, parts, pw, K, t, W);
#pragma unroll
  for (int i = 0; i < CH; ++i)
    if (in_row(i, W)) sum += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
  const float mean = row_total<NW>(sum, red[0]) / (float)W;
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < CH; ++i)
    if (in_row(i, W))
#pragma unroll
      for (int e = 0; e < 4; ++e) { const float d = v[i][e] - mean; ss += d * d; }
  const float r = 1.f / sqrtf(row_total<NW>(ss, red[1]) / (float)W + eps);
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    if (!in_row(i, W)) continue;
    const int c = col(i, W);
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      xv[i][e] += (v[i][e] - mean) * r * wv[i][e] + bv[i][e];
#pragma unroll
      for (int k = 0; k < 3; ++k) tail[i][k][e] = pos - 3 + k >= 0 ? tail[i][k][e] : 0.f;
      float acc = 0.f;
      acc += cw[i][e].x * tail[i][0][e];
      acc += cw[i][e].y * tail[i][1][e];
      acc += cw[i][e].z * tail[i][2][e];
      acc += cw[i][e].w * xv[i][e];
      o[e] = xv[i][e] + acc;
    }
    store4<float>(x + t * W + c, xv[i]);
    store4<T>(out + t * W + c, o);
    store4<float>(st + c, tail[i][1]);
    store4<float>(st + W + c, tail[i][2]);
    store4<float>(st + 2 * (size_t)W + c, xv[i]);
    done(c, o);
  }
}

template <typename T, int CH>
__global__ void __launch_bounds__(NT) ln_residual_taps_kernel(float* __restrict__ x, const T* __restrict__ y,
                                                              const T* __restrict__ parts, const float* __restrict__ pw, int K,
                                                              const float* __restrict__ w, const float* __restrict__ b, int W,
                                                              float eps, Taps a, T* __restrict__ out) {
  __shared__ float red[2][NT / 64];
  ln_residual_taps_row<T, CH, NT / 64>(blockIdx.x, x, y, parts, pw, K, w, b, W, eps, a, out, red, [] {}, [](int, const float*) {});
}

// The same with the choice of the row's experts: the row stays in LDS and 16 waves form the scores of an expert each, whose router rows
// are on their way behind the row's own (route_few_kernel's sums and choice).  us, two launches / this, rows of 1024, 16 experts, bf16: 4
// rows 6.3 / 5.4, 64 6.6 / 5.7, 256 8.1 / 6.7; of 512, 4 rows 5.8 / 5.0; a decode of 4 sequences, 63 steps of four such layers, 14.98 -> 14.78 ms.  Two
// scores a wave over rows of 2048 leave one CU with a router of 256 KB: 4 rows 8.6 / 10.6, 256 12.1 / 13.5, so those stay two launches.
template <typename T>
__global__ void __launch_bounds__(RF_WAVES * 64) ln_residual_taps_route_kernel(
    float* __restrict__ x, const T* __restrict__ y, const T* __restrict__ parts, const float* __restrict__ pw, int K,
    const float* __restrict__ w, const float* __restrict__ b, int W, float eps, Taps a, T* __restrict__ out, RouteFew r) {
  constexpr int MOST = RT_MOST / 512;
  __shared__ float red[2][RF_WAVES], z_s[RF_WAVES];
  __shared__ __attribute__((aligned(16))) float h_s[RT_MOST];
  const size_t t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float rv[MOST][8];
  auto early = [&] {                                         // (behind the row's loads, which are waited for first)
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < MOST; ++i)
      load8<float>(r.router + (size_t)min(wave, r.E - 1) * W + min(i * 512 + lane * 8, W - 8), rv[i]);
    asm volatile("" ::: "memory");
  };
  ln_residual_taps_row<T, 1, RF_WAVES>(t, x, y, parts, pw, K, w, b, W, eps, a, out, red, early, [&](int c, const float* o) {
    float h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      T v;
      stf<T>(&v, o[e]);
      h[e] = ldf<T>(&v);
    }
    store4<float>(h_s + c, h);
  });
  __syncthreads();
  float acc = 0.f;
#pragma unroll
  for (int i = 0; i < MOST; ++i) {
    const int c = i * 512 + lane * 8;
    if (c >= W) break;
    float h[8];
    load8<float>(h_s + c, h);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc += h[j] * rv[i][j];
  }
  const float s = wave_sum(acc);
  if (lane == 0 && wave < r.E) z_s[wave] = s + (r.bias ? r.bias[wave] : 0.f);
  __syncthreads();
  if (wave == 0) route_choose<false>(r, z_s, nullptr, nullptr, t);
}

// x += LayerNorm(y + sum_k pw[k] parts[k]) w + b;  out = LayerNorm(x) w2 + b2
// The final norm behind the last layer's residual sum.  At a decode step's few rows either launch is latency, not bytes (4 rows of 1024
// in bf16: 4.7 us for the sum, 5.1 us for the norm), so the row stays in registers for both.  Against two launches, timed in turn: a
// decode of such rows 16.96 -> 16.78 ms for 63 steps (runs of one side differ by 0.5%).
template <typename T, int CH>
__global__ void __launch_bounds__(NT) ln_residual_ln_kernel(float* __restrict__ x, const T* __restrict__ y,
                                                            const T* __restrict__ parts, const float* __restrict__ pw, int K,
                                                            const float* __restrict__ w, const float* __restrict__ b, int W, float eps,
                                                            const float* __restrict__ w2, const float* __restrict__ b2, float eps2,
                                                            T* __restrict__ out) {
  __shared__ float red[4][NT / 64];
  const size_t t = blockIdx.x;
  float v[CH][4], xv[CH][4], wv[CH][4], bv[CH][4], w2v[CH][4], b2v[CH][4];
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = col(i, W);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[i][e] = 0.f;
    if (y) load4<T>(y + t * W + c, v[i]);
    load4<float>(x + t * W + c, xv[i]);
    load4<float>(w + c, wv[i]);
    load4<float>(b + c, bv[i]);
    load4<float>(w2 + c, w2v[i]);
    load4<float>(b2 + c, b2v[i]);
  }
  add_parts<T, CH>(v, parts, pw, K, t, W);
  auto norm = [&](float (&z)[CH][4], float* r0, float* r1, float e0, float& mean) {   // 1 / deviation
    float sum = 0.f, ss = 0.f;
#pragma unroll
    for (int i = 0; i < CH; ++i)
      if (in_row(i, W)) sum += (z[i][0] + z[i][1]) + (z[i][2] + z[i][3]);
    mean = row_total(sum, r0) / (float)W;
#pragma unroll
    for (int i = 0; i < CH; ++i)
      if (in_row(i, W))
#pragma unroll
        for (int e = 0; e < 4; ++e) { const float d = z[i][e] - mean; ss += d * d; }
    return 1.f / sqrtf(row_total(ss, r1) / (float)W + e0);
  };
  float mean;
  const float r = norm(v, red[0], red[1], eps, mean);
#pragma unroll
  for (int i = 0; i < CH; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) xv[i][e] += (v[i][e] - mean) * r * wv[i][e] + bv[i][e];
    if (in_row(i, W)) store4<float>(x + t * W + col(i, W), xv[i]);
  }
  const float r2 = norm(xv, red[2], red[3], eps2, mean);
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    if (!in_row(i, W)) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) xv[i][e] = (xv[i][e] - mean) * r2 * w2v[i][e] + b2v[i][e];
    store4<T>(out + t * W + col(i, W), xv[i]);
  }
}

// 1 / rms over the part of gs numbers that this thread's run i lies in (gs a multiple of a wave's 256: sq[i] its four squares' sum)
template <int CH>
__device__ __forceinline__ void part_inv(const float (&sq)[CH], float (&inv)[CH], float* red, int gs, float eps, int W) {
  const int wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const float s = wave_sum(in_row(i, W) ? sq[i] : 0.f);
    if ((threadIdx.x & 63) == 0) red[i * (NT / 64) + wave] = s;
  }
  __syncthreads();
  const int nb = gs / 256;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int b0 = (i * (NT / 64) + wave) / nb * nb;
    float s = 0.f;
    for (int k = 0; k < nb; ++k) s += red[min(b0 + k, CH * (NT / 64) - 1)];
    inv[i] = 1.f / sqrtf(s / (float)gs + eps);
  }
}

// x += mult group-norm(y + sum_k pw[k] parts[k]) w;  out = group-norm(x) w2
template <typename T, int CH>
__global__ void __launch_bounds__(NT) group_residual_norm_kernel(float* __restrict__ x, const T* __restrict__ y,
                                                                 const T* __restrict__ parts, const float* __restrict__ pw, int K,
                                                                 const float* __restrict__ w, int W, int gs, float eps, float mult,
                                                                 const float* __restrict__ w2, int gs2, float eps2,
                                                                 T* __restrict__ out) {
  __shared__ float red[2][CH * (NT / 64)];
  const size_t t = blockIdx.x;
  float v[CH][4], xv[CH][4], wv[CH][4], w2v[CH][4], sq[CH], inv[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = col(i, W);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[i][e] = 0.f;
    if (y) load4<T>(y + t * W + c, v[i]);
    load4<float>(x + t * W + c, xv[i]);
    load4<float>(w + c, wv[i]);
    load4<float>(w2 + c, w2v[i]);
  }
  add_parts<T, CH>(v, parts, pw, K, t, W);
#pragma unroll
  for (int i = 0; i < CH; ++i) sq[i] = (v[i][0] * v[i][0] + v[i][1] * v[i][1]) + (v[i][2] * v[i][2] + v[i][3] * v[i][3]);
  part_inv<CH>(sq, inv, red[0], gs, eps, W);
#pragma unroll
  for (int i = 0; i < CH; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) xv[i][e] += mult * (v[i][e] * inv[i] * wv[i][e]);
    if (in_row(i, W)) store4<float>(x + t * W + col(i, W), xv[i]);
    sq[i] = (xv[i][0] * xv[i][0] + xv[i][1] * xv[i][1]) + (xv[i][2] * xv[i][2] + xv[i][3] * xv[i][3]);
  }
  part_inv<CH>(sq, inv, red[1], gs2, eps2, W);
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    if (!in_row(i, W)) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) xv[i][e] = xv[i][e] * (inv[i] * w2v[i][e]);
    store4<T>(out + t * W + col(i, W), xv[i]);
  }
}

// x += 0.5 (l / rms(l) wl + r / rms(r) wr) + extra;  out = x / rms(x) gain
template <typename T, int CH>
__global__ void __launch_bounds__(NT) combine_norm_kernel(float* __restrict__ x, const T* __restrict__ l, const T* __restrict__ r,
                                                          const float* __restrict__ wl, const float* __restrict__ wr,
                                                          const T* __restrict__ extra, int W, float eps,
                                                          const float* __restrict__ gain, float eps2, T* __restrict__ out) {
  __shared__ float red[3][NT / 64];
  const size_t t = blockIdx.x;
  float lv[CH][4], rv[CH][4], ev[CH][4], xv[CH][4], wlv[CH][4], wrv[CH][4], sl = 0.f, sr = 0.f, sx = 0.f;
  const float gn = gain[0];
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = col(i, W);
    load4<T>(l + t * W + c, lv[i]);
    load4<T>(r + t * W + c, rv[i]);
#pragma unroll
    for (int e = 0; e < 4; ++e) ev[i][e] = 0.f;
    if (extra) load4<T>(extra + t * W + c, ev[i]);
    load4<float>(x + t * W + c, xv[i]);
    load4<float>(wl + c, wlv[i]);
    load4<float>(wr + c, wrv[i]);
  }
#pragma unroll
  for (int i = 0; i < CH; ++i)
    if (in_row(i, W)) {
      sl += (lv[i][0] * lv[i][0] + lv[i][1] * lv[i][1]) + (lv[i][2] * lv[i][2] + lv[i][3] * lv[i][3]);
      sr += (rv[i][0] * rv[i][0] + rv[i][1] * rv[i][1]) + (rv[i][2] * rv[i][2] + rv[i][3] * rv[i][3]);
    }
  sr = wave_sum(sr);
  if ((threadIdx.x & 63) == 0) red[1][threadIdx.x >> 6] = sr;
  sl = row_total(sl, red[0]);                                // (its barrier serves both)
  sr = ((red[1][0] + red[1][1]) + red[1][2]) + red[1][3];
  const float il = 1.f / sqrtf(sl / (float)W + eps), ir = 1.f / sqrtf(sr / (float)W + eps);
#pragma unroll
  for (int i = 0; i < CH; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) xv[i][e] += 0.5f * (lv[i][e] * il * wlv[i][e] + rv[i][e] * ir * wrv[i][e]) + ev[i][e];
    if (in_row(i, W)) {
      store4<float>(x + t * W + col(i, W), xv[i]);
      sx += (xv[i][0] * xv[i][0] + xv[i][1] * xv[i][1]) + (xv[i][2] * xv[i][2] + xv[i][3] * xv[i][3]);
    }
  }
  const float s = 1.f / sqrtf(row_total(sx, red[2]) / (float)W + eps2) * gn;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    if (!in_row(i, W)) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) xv[i][e] *= s;
    store4<T>(out + t * W + col(i, W), xv[i]);
  }
}

// rows of whole runs of four in the registers of NT threads, all addresses on 16 bytes
bool row_ok(int W, std::initializer_list<const void*> ps) {
  uintptr_t u = 0;
  for (const void* p : ps) u |= (uintptr_t)p;
  return W % 4 == 0 && W >= 256 && W <= 16 * NT && u % 16 == 0;
}

}  // namespace

// f32: the type of the results and of the next sublayer's row
#define RN_CH(KERNEL, TT, ...)                                                                                         \
  do {                                                                                                                 \
    if (W <= 4 * NT) hipLaunchKernelGGL((KERNEL<TT, 1>), dim3(rows), dim3(NT), 0, st, __VA_ARGS__);                \
    else if (W <= 8 * NT) hipLaunchKernelGGL((KERNEL<TT, 2>), dim3(rows), dim3(NT), 0, st, __VA_ARGS__);           \
    else hipLaunchKernelGGL((KERNEL<TT, 4>), dim3(rows), dim3(NT), 0, st, __VA_ARGS__);                            \
  } while (0)

extern "C" {

// all of them: -2 where the row does not fit

int edge_sm_ln_residual_ln(float* x, const void* y, const void* parts, const float* pw, int K, const float* w, const float* b, float eps,
                           const float* w2, const float* b2, float eps2, void* out, int rows, int W, int f32, hipStream_t st) {
  if (!row_ok(W, {x, y, parts, w, b, w2, b2, out})) return -2;
  if (rows == 0) return 0;
  if (f32) RN_CH(ln_residual_ln_kernel, float, x, (const float*)y, (const float*)parts, pw, K, w, b, W, eps, w2, b2, eps2, (float*)out);
  else RN_CH(ln_residual_ln_kernel, bf16_t, x, (const bf16_t*)y, (const bf16_t*)parts, pw, K, w, b, W, eps, w2, b2, eps2, (bf16_t*)out);
  return (int)hipGetLastError();
}

int edge_sm_ln_residual_taps(float* x, const void* y, const void* parts, const float* pw, int K, const float* w, const float* b,
                             const float* cw, float* state, const int* tok_seq, const int* tok_pos, const int* seq_slot, void* out,
                             int rows, int W, float eps, int f32, hipStream_t st) {
  if (!row_ok(W, {x, y, parts, w, b, cw, state, out})) return -2;
  if (rows == 0) return 0;
  const Taps a{cw, state, tok_seq, tok_pos, seq_slot};
  if (f32) RN_CH(ln_residual_taps_kernel, float, x, (const float*)y, (const float*)parts, pw, K, w, b, W, eps, a, (float*)out);
  else RN_CH(ln_residual_taps_kernel, bf16_t, x, (const bf16_t*)y, (const bf16_t*)parts, pw, K, w, b, W, eps, a, (bf16_t*)out);
  return (int)hipGetLastError();
}

// edge_sm_ln_residual_taps and edge_sm_moe_route (postnorm.hip) of its rows, up to 16 experts
int edge_sm_ln_residual_taps_route(float* x, const void* y, const void* parts, const float* pw, int K, const float* w, const float* b,
                                   const float* cw, float* state, const int* tok_seq, const int* tok_pos, const int* seq_slot, void* out,
                                   int rows, int W, float eps, const float* router, const float* bias, int E, int top, float scale,
                                   int sigm, int* idx, float* wts, int f32, hipStream_t st) {
  if (!row_ok(W, {x, y, parts, w, b, cw, state, out, router}) || W > RT_MOST || W % 8 || rows > RT_ROWS || E < 1 || E > RF_WAVES ||
      top < 1 || top > E)
    return -2;
  if (rows == 0) return 0;
  const Taps a{cw, state, tok_seq, tok_pos, seq_slot};
  const RouteFew r{router, bias, W, E, 0, 1, 1, top, sigm, scale, idx, wts, nullptr};
#define RT(TT)                                                                                                               \
  hipLaunchKernelGGL(ln_residual_taps_route_kernel<TT>, dim3(rows), dim3(RF_WAVES * 64), 0, st, x, (const TT*)y, (const TT*)parts, pw, K, w, \
                     b, W, eps, a, (TT*)out, r)
  if (f32) RT(float);
  else RT(bf16_t);
#undef RT
  return (int)hipGetLastError();
}

int edge_sm_group_residual_norm(float* x, const void* y, const void* parts, const float* pw, int K, const float* w, int groups,
                                float eps, float mult, const float* w2, int groups2, float eps2, void* out, int rows, int W, int f32,
                                hipStream_t st) {
  if (groups < 1 || groups2 < 1 || W % groups || W % groups2 || W / groups % 256 || W / groups2 % 256 ||
      !row_ok(W, {x, y, parts, w, w2, out}))
    return -2;
  // long rows and many: a thread's four runs with both norms' weights leave too few wavefronts in flight (us, two launches / one, bf16 rows
  // of 3072: 256 rows 10.9 / 10.5, 1024 17.5 / 21.9, 8192 81 / 110)
  if (W > 8 * NT && rows > 512) return -2;
  if (rows == 0) return 0;
  const int gs = W / groups, gs2 = W / groups2;
  if (f32) RN_CH(group_residual_norm_kernel, float, x, (const float*)y, (const float*)parts, pw, K, w, W, gs, eps, mult, w2, gs2,
                 eps2, (float*)out);
  else RN_CH(group_residual_norm_kernel, bf16_t, x, (const bf16_t*)y, (const bf16_t*)parts, pw, K, w, W, gs, eps, mult, w2, gs2,
             eps2, (bf16_t*)out);
  return (int)hipGetLastError();
}

int edge_sm_combine_norm(float* x, const void* l, const void* r, const float* wl, const float* wr, const void* extra, float eps,
                         const float* gain, float eps2, void* out, int rows, int W, int f32, hipStream_t st) {
  if (!row_ok(W, {x, l, r, wl, wr, extra, out})) return -2;
  if (rows == 0) return 0;
  if (f32) RN_CH(combine_norm_kernel, float, x, (const float*)l, (const float*)r, wl, wr, (const float*)extra, W, eps, gain, eps2,
                 (float*)out);
  else RN_CH(combine_norm_kernel, bf16_t, x, (const bf16_t*)l, (const bf16_t*)r, wl, wr, (const bf16_t*)extra, W, eps, gain,
             eps2, (bf16_t*)out);
  return (int)hipGetLastError();
}

}  // extern "C"
