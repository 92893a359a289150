// A gated delta rule's whole decode step between its two projections, one workgroup per (sequence, head) with one token each: the
// four-tap convolution and silu of the head's q | k | v, unit-length q and k, beta, the decays (a low-rank product per key channel,
// or one number), the recurrence on the head's [N, P] fp32 state, the head's RMS norm and its gate (a low-rank product with a
// sigmoid, or columns of the projection with silu).  What each part is and where it rounds is as in the kernels that longer
// portions run: tap4_kernel, delta_prep16_kernel, delta_scan_kernel, head_norm_gate16_kernel.
//
// Bound by latency: by themselves the parts are six launches (two of them products over a rank of 32 or 64), each a chain of a
// load, a sum and a store of a few KB.  Every load here (state, tail, weights) hangs on the slot alone and is issued first; then
// two barriers.  With s = S^T k and o = S^T q over the decayed state, w = beta (v - s), the new state's product with q is
// o + w (k . q), so one sum over the rows serves both.  A head's convolution channels are its own (q and k not shared between
// heads): no other workgroup reads the tail that this one moves up.
// us of a whole mixer with its two projections, six launches (four with per-head decays) / one between them, bf16, 16 heads: 64 x 64
// states of width 1024, a decay per channel, 4 tokens 31.2 / 13.7, 64 57.6 / 29.0; 128 x 128 of 2048 40.2 / 22.5, 126 / 67; a decay per head
// 21.3 / 13.9, 50 / 29; 32.8 / 23.7, 118 / 66; fp32, 64 x 64, a decay per channel, 4 tokens 32.0 / 15.7.
#include "common.h"
#include "seqmix/seqmix_common.h"

namespace {

struct DeltaStep {
  const void *u, *a2, *g2;                                   // a2 [H N, ra], g2 [H P, rg] (HEAD: none)
  const float *conv_w, *conv_b, *dt_bias, *A_log, *norm_w;   // conv_w [C, 4]; dt_bias [H N] (HEAD: [H])
  void *tail, *out;                                          // tail [slots, 3, C]; out [rows, H P]
  float* state;                                              // [slots, H, N, P]
  const int *seq_slot, *seq_start, *seq_off;
  int ld, H, b0, a0, ra, z0, rg;                             // columns of u: beta, decay (inner rows), gate (inner rows)
  float eps;
};

template <typename T, int N, int P, bool HEAD>
__global__ void __launch_bounds__(N * P / 32 < 256 ? 256 : 512) delta_step_kernel(DeltaStep a) {
  constexpr int NTH = N * P / 32 < 256 ? 256 : 512, NW = NTH / 64;
  constexpr int PG = P / 4, RGS = NTH / PG, NR = N / RGS;    // threads across a state row, row groups, rows of a thread
  static_assert(2 * N + P <= NTH && N % 64 == 0 && P % 64 == 0 && N % RGS == 0 && PG <= 64, "shape");
  __shared__ __attribute__((aligned(16))) float q_s[N], k_s[N], g_s[N], v_s[P], z_s[P], sk_s[NW][P], sq_s[NW][P];
  __shared__ float ss_s[NW], kq_s;
  const int s = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), H = a.H;
  const int slot = a.seq_slot[s], start = a.seq_start[s];
  const size_t t = a.seq_off[s];
  const int C = 2 * H * N + H * P;
  const T* ur = reinterpret_cast<const T*>(a.u) + t * a.ld;
  // the state: rows rg NR .., four columns a thread
  const int p0 = (tid % PG) * 4, rg = tid / PG;
  float* st = a.state + (((size_t)slot * H + h) * N + rg * NR) * P + p0;
  float4 S[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) S[i] = start > 0 ? *reinterpret_cast<const float4*>(st + (size_t)i * P) : make_float4(0.f, 0.f, 0.f, 0.f);
  // one convolution channel a thread
  const bool conv = tid < 2 * N + P;
  const int ci = min(tid, 2 * N + P - 1);
  const int c = ci < N ? h * N + ci : ci < 2 * N ? H * N + h * N + ci - N : 2 * H * N + h * P + ci - 2 * N;
  T* tl = reinterpret_cast<T*>(a.tail) + (size_t)slot * 3 * C + c;
  const float x0 = start >= 3 ? ldf<T>(tl) : 0.f, x1 = start >= 2 ? ldf<T>(tl + C) : 0.f, x2 = start >= 1 ? ldf<T>(tl + 2 * (size_t)C) : 0.f;
  const T x3 = ur[c];
  const float4 w = *reinterpret_cast<const float4*>(a.conv_w + (size_t)c * 4);
  const float cb = a.conv_b[c];
  const float beta = sigmoidf_(ldf<T>(ur + a.b0 + h)), al = expf(a.A_log[h]);
  // the low-rank products: threads below N a decay each, the next P a gate each
  float low = 0.f;
  if constexpr (!HEAD) {
    const bool dec = tid < N;
    if (tid < N + P) {
      const int rank = dec ? a.ra : a.rg;
      const T* x = ur + (dec ? a.a0 : a.z0);
      const T* m = dec ? reinterpret_cast<const T*>(a.a2) + (size_t)(h * N + tid) * rank
                       : reinterpret_cast<const T*>(a.g2) + (size_t)(h * P + tid - N) * rank;
#pragma unroll 4
      for (int r = 0; r < rank; r += 8) {
        float xf[8], mf[8];
        load8<T>(x + r, xf);
        load8<T>(m + r, mf);
#pragma unroll
        for (int e = 0; e < 8; ++e) low += xf[e] * mf[e];
      }
    }
  } else if (tid < P) {
    low = ldf<T>(ur + a.z0 + h * P + tid);
  }
  auto decay = [&](float raw) { return expf(-al * (raw > 20.f ? raw : log1pf(expf(raw)))); };
  {
    float acc = cb;
    acc += w.x * x0;
    acc += w.y * x1;
    acc += w.z * x2;
    acc += w.w * ldf<T>(&x3);
    T y;
    stf<T>(&y, siluf_(acc));                                 // (rows of q | k | v are T)
    const float v = ldf<T>(&y);
    if (conv) {
      (ci < N ? q_s[ci] : ci < 2 * N ? k_s[ci - N] : v_s[ci - 2 * N]) = v;
      stf<T>(tl, x1);
      stf<T>(tl + C, x2);
      tl[2 * (size_t)C] = x3;
    }
    const float ss = wave_sum(conv ? v * v : 0.f);
    if (lane == 0) ss_s[wave] = ss;
  }
  if constexpr (HEAD) {
    if (tid < N) g_s[tid] = decay(ldf<T>(ur + a.a0 + h) + a.dt_bias[h]);
    if (tid < P) z_s[tid] = siluf_(low);
  } else {
    if (tid < N) g_s[tid] = decay(low + a.dt_bias[h * N + tid]);
    else if (tid < N + P) {
      T z;
      stf<T>(&z, low);                                       // (the gate's rows are T)
      z_s[tid - N] = sigmoidf_(ldf<T>(&z));
    }
  }
  __syncthreads();
  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int i = 0; i < N / 64; ++i) { sq += ss_s[i]; sk += ss_s[N / 64 + i]; }
  const float rq = 1.f / sqrtf(sq + 1e-6f) * (1.f / sqrtf((float)N)), rk = 1.f / sqrtf(sk + 1e-6f);
  float4 dk = make_float4(0.f, 0.f, 0.f, 0.f), dq = dk;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int n = rg * NR + i;
    const float g = g_s[n], k = k_s[n], q = q_s[n];
    S[i].x *= g; S[i].y *= g; S[i].z *= g; S[i].w *= g;
    dk.x += S[i].x * k; dk.y += S[i].y * k; dk.z += S[i].z * k; dk.w += S[i].w * k;
    dq.x += S[i].x * q; dq.y += S[i].y * q; dq.z += S[i].z * q; dq.w += S[i].w * q;
  }
#pragma unroll
  for (int o = PG; o < 64; o <<= 1) {
    dk.x = xor_sum(dk.x, o); dk.y = xor_sum(dk.y, o); dk.z = xor_sum(dk.z, o); dk.w = xor_sum(dk.w, o);
    dq.x = xor_sum(dq.x, o); dq.y = xor_sum(dq.y, o); dq.z = xor_sum(dq.z, o); dq.w = xor_sum(dq.w, o);
  }
  if (lane < PG) {
    *reinterpret_cast<float4*>(&sk_s[wave][p0]) = dk;
    *reinterpret_cast<float4*>(&sq_s[wave][p0]) = dq;
  }
  if (wave == NW - 1) {
    float d = 0.f;
#pragma unroll
    for (int i = 0; i < N / 64; ++i) d += k_s[lane + 64 * i] * q_s[lane + 64 * i];
    d = wave_sum(d);
    if (lane == 0) kq_s = d;
  }
  __syncthreads();
  float4 tk = make_float4(0.f, 0.f, 0.f, 0.f), tq = tk;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const float4 x = *reinterpret_cast<const float4*>(&sk_s[i][p0]);
    tk.x += x.x; tk.y += x.y; tk.z += x.z; tk.w += x.w;
  }
  const float4 v = *reinterpret_cast<const float4*>(&v_s[p0]);
  const float4 wv = make_float4(beta * (v.x - rk * tk.x), beta * (v.y - rk * tk.y), beta * (v.z - rk * tk.z), beta * (v.w - rk * tk.w));
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const float k = k_s[rg * NR + i] * rk;
    *reinterpret_cast<float4*>(st + (size_t)i * P) =
        make_float4(S[i].x + k * wv.x, S[i].y + k * wv.y, S[i].z + k * wv.z, S[i].w + k * wv.w);
  }
  if (wave != 0) return;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const float4 x = *reinterpret_cast<const float4*>(&sq_s[i][p0]);
    tq.x += x.x; tq.y += x.y; tq.z += x.z; tq.w += x.w;
  }
  const float kq = kq_s * rk * rq;
  const float y[4] = {rq * tq.x + wv.x * kq, rq * tq.y + wv.y * kq, rq * tq.z + wv.z * kq, rq * tq.w + wv.w * kq};
  const float ss = wave_sum(lane < PG ? (y[0] * y[0] + y[1] * y[1]) + (y[2] * y[2] + y[3] * y[3]) : 0.f);
  const float r = 1.f / sqrtf(ss / (float)P + a.eps);
  if (lane < PG) {
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = y[e] * r * a.norm_w[p0 + e] * z_s[p0 + e];
    store4<T>(reinterpret_cast<T*>(a.out) + (t * H + h) * P + p0, o);
  }
}

template <typename T, bool HEAD>
int run(const DeltaStep& a, int n, int N, int P, hipStream_t st) {
#define DS(NN, PP) hipLaunchKernelGGL((delta_step_kernel<T, NN, PP, HEAD>), dim3(n, a.H), dim3(NN * PP / 32 < 256 ? 256 : 512), 0, st, a)
  if (N == 64 && P == 64) DS(64, 64);
  else if (N == 128 && P == 128) DS(128, 128);
  else return -2;
#undef DS
  return (int)hipGetLastError();
}

}  // namespace

// ra, rg 0: one decay per head and a gate that is columns of u; -2: not this kernel's
extern "C" int edge_sm_delta_step(const void* u, int ld, int b0, int a0, int z0, const void* a2, int ra, const void* g2, int rg,
                                  const float* conv_w, const float* conv_b, void* tail, float* state, const float* dt_bias,
                                  const float* A_log, const float* norm_w, const int* seq_slot, const int* seq_start,
                                  const int* seq_off, void* out, int n, int H, int N, int P, float eps, int f32, hipStream_t st) {
  const uintptr_t all = (uintptr_t)u | (uintptr_t)a2 | (uintptr_t)g2 | (uintptr_t)conv_w | (uintptr_t)state | (uintptr_t)out;
  const bool head = ra == 0 && rg == 0;
  if (all % 16 || H < 1 || (!head && (ra < 8 || rg < 8 || ra % 8 || rg % 8 || ra > 256 || rg > 256 || ld % 8 || a0 % 8 || z0 % 8))) return -2;
  if (!((N == 64 && P == 64) || (N == 128 && P == 128))) return -2;
  if (n == 0) return 0;
  const DeltaStep a{u, a2, g2, conv_w, conv_b, dt_bias, A_log, norm_w, tail, out, state, seq_slot, seq_start, seq_off, ld, H, b0, a0,
                    ra, z0, rg, eps};
  if (head) return f32 ? run<float, true>(a, n, N, P, st) : run<bf16_t, true>(a, n, N, P, st);
  return f32 ? run<float, false>(a, n, N, P, st) : run<bf16_t, false>(a, n, N, P, st);
}
