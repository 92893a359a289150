// What a parallel layer (attention beside a state-space mixer and a feed-forward) does with its one input projection's row in a
// decode step, in one launch: the rotated queries and the new key and value rows in their pages, the block means that this token
// completes, the convolved and activated x | B | C rows with their tail, and the feed-forward's squared ReLU.  Each part reads
// other columns of the row and none reads another's result, but for the means, which the workgroup that wrote the key and value forms
// behind a barrier.  Their arithmetic is rope_write_kernel's, pool_kernel's, tap4_kernel's and relu2_kernel's.
//
// Bound by latency: by themselves the parts are four launches for a few KB each.  us in a decode step of two sequences, fp32, 16 heads
// of 64, 1152 channels, 4096 columns: rotation 4.8, means 4.0, convolution 4.6, squared ReLU 4.7; together 5.2.
#include "common.h"
#include "seqmix/seqmix_common.h"

namespace {

struct ParallelIn {
  const void* u;
  const int *tok_seq, *tok_pos, *seq_slot, *ptab;
  const float *cs, *conv_w, *conv_b;                         // cs [positions, rot / 2, 2]; conv_w [C, 4]
  void *q, *kp, *vp, *tail, *xbc, *act;                      // tail [slots, 3, C]
  float *kb, *vb;
  int ld, ptab_ld, H, G, D, Dv, rot, page, PB, pool, c0, C, cblocks, f0, F;
};

template <typename T>
__global__ void __launch_bounds__(NT) parallel_in_kernel(ParallelIn a) {
  const int t = blockIdx.x, tid = threadIdx.x, role = blockIdx.y;
  const T* row = reinterpret_cast<const T*>(a.u) + (size_t)t * a.ld;
  if (role > a.cblocks) {                                    // squared ReLU, eight columns a thread
    const int c = ((role - 1 - a.cblocks) * NT + tid) * 8;
    if (c >= a.F) return;
    float f[8];
    load8<T>(row + a.f0 + c, f);
#pragma unroll
    for (int e = 0; e < 8; ++e) { const float v = fmaxf(f[e], 0.f); f[e] = v * v; }
    store8<T>(reinterpret_cast<T*>(a.act) + (size_t)t * a.F + c, f);
    return;
  }
  const int pos = a.tok_pos[t], slot = a.seq_slot[a.tok_seq[t]];
  if (role > 0) {                                            // convolution, eight channels a thread
    const int c = ((role - 1) * NT + tid) * 8;
    if (c >= a.C) return;
    T* tl = reinterpret_cast<T*>(a.tail) + (size_t)slot * 3 * a.C + c;
    float x[4][8], b[8], y[8];
    float4 w[8];
#pragma unroll
    for (int k = 0; k < 3; ++k) load8<T>(tl + (size_t)k * a.C, x[k]);
    load8<T>(row + a.c0 + c, x[3]);
    load8<float>(a.conv_b + c, b);
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = *reinterpret_cast<const float4*>(a.conv_w + (size_t)(c + e) * 4);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[k][e] = pos - 3 + k >= 0 ? x[k][e] : 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float acc = b[e];
      acc += w[e].x * x[0][e];
      acc += w[e].y * x[1][e];
      acc += w[e].z * x[2][e];
      acc += w[e].w * x[3][e];
      y[e] = siluf_(acc);
    }
    store8<T>(reinterpret_cast<T*>(a.xbc) + (size_t)t * a.C + c, y);
#pragma unroll
    for (int k = 0; k < 3; ++k) store8<T>(tl + (size_t)k * a.C, x[k + 1]);
    return;
  }
  // rotation and the page rows, eight coordinates a thread
  const int *pt = a.ptab + (size_t)slot * a.ptab_ld, half = a.rot >> 1, nq = a.H * a.D, nqk = nq + a.G * a.D, nk = a.G * a.D, nv = a.G * a.Dv;
  const size_t prow = (size_t)pt[pos / a.page] * a.page + pos % a.page;
  const float* cs = a.cs ? a.cs + (size_t)pos * a.rot : nullptr;
  T *kp = reinterpret_cast<T*>(a.kp), *vp = reinterpret_cast<T*>(a.vp);
  for (int e = tid * 8; e < nqk + nv; e += NT * 8) {
    float v[8];
    load8<T>(row + e, v);
    if (e >= nqk) {
      store8<T>(vp + prow * nv + e - nqk, v);
      continue;
    }
    const int d = e % a.D;
    if (d < a.rot) {
      const int i = d < half ? d : d - half;
      float o[8], tab[16];
      load8<T>(row + (d < half ? e + half : e - half), o);
      load8<float>(cs + 2 * i, tab);
      load8<float>(cs + 2 * i + 8, tab + 8);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        v[k] = d < half ? v[k] * tab[2 * k] - o[k] * tab[2 * k + 1] : v[k] * tab[2 * k] + o[k] * tab[2 * k + 1];
    }
    if (e < nq) store8<T>(reinterpret_cast<T*>(a.q) + (size_t)t * nq + e, v);
    else store8<T>(kp + prow * nk + e - nq, v);
  }
  if (a.pool == 0 || (pos + 1) % a.pool != 0) return;        // (the whole workgroup)
  __syncthreads();                                           // the block's last row is in its page
  const int p0 = pos + 1 - a.pool;
  const size_t dst = (size_t)pt[p0 / a.page] * a.PB + (p0 % a.page) / a.pool;
  const float inv = 1.f / (float)a.pool;
  for (int e = tid; e < nk + nv; e += NT) {
    float acc = 0.f;
#pragma unroll 4
    for (int j = 0; j < a.pool; ++j) {
      const int p = p0 + j;
      const size_t r = (size_t)pt[p / a.page] * a.page + p % a.page;
      acc += e < nk ? ldf<T>(kp + r * nk + e) : ldf<T>(vp + r * nv + (e - nk));
    }
    if (e < nk) a.kb[dst * nk + e] = acc * inv;
    else a.vb[dst * nv + (e - nk)] = acc * inv;
  }
}

}  // namespace

// columns of u [rows, ld]: q | k | v from 0 on, x | B | C (C of them) from c0, the feed-forward's F from f0.  -2: not taken
extern "C" int edge_sm_parallel_in(const void* u, int ld, const int* tok_seq, const int* tok_pos, const int* seq_slot, const int* ptab,
                                   int ptab_ld, const float* cs, void* q, void* kp, void* vp, float* kb, float* vb, int H, int G, int D,
                                   int Dv, int rot, int page, int PB, int pool, int c0, int C, const float* conv_w, const float* conv_b,
                                   void* tail, void* xbc, int f0, int F, void* act, int rows, int f32, hipStream_t st) {
  const uintptr_t all = (uintptr_t)u | (uintptr_t)q | (uintptr_t)kp | (uintptr_t)vp | (uintptr_t)tail | (uintptr_t)xbc | (uintptr_t)act |
                        (uintptr_t)conv_w | (uintptr_t)conv_b | (uintptr_t)cs;
  if (all % 16 || ld % 8 || D % 8 || Dv % 8 || rot % 16 || rot > D || (rot > 0 && !cs) || c0 % 8 || C % 8 || f0 % 8 || F % 8 ||
      page < 1 || pool < 0 || (pool > 0 && (!kb || !vb)))
    return -2;
  if (rows == 0) return 0;
  const int cblocks = (C / 8 + NT - 1) / NT, fblocks = (F / 8 + NT - 1) / NT;
  const ParallelIn a{u, tok_seq, tok_pos, seq_slot, ptab, cs, conv_w, conv_b, q, kp, vp, tail, xbc, act, kb, vb, ld, ptab_ld, H, G, D, Dv,
                     rot, page, PB, pool, c0, C, cblocks, f0, F};
  const dim3 grid(rows, 1 + cblocks + fblocks);
  if (f32) hipLaunchKernelGGL(parallel_in_kernel<float>, grid, dim3(NT), 0, st, a);
  else hipLaunchKernelGGL(parallel_in_kernel<bf16_t>, grid, dim3(NT), 0, st, a);
  return (int)hipGetLastError();
}
