// Prompt attention over latent rows (one cached row is the key, its first DV numbers the value), bf16 on the matrix cores.
#include "common.h"
#include "seqmix/seqmix_common.h"

namespace {

// Eight waves of one workgroup take eight heads of a kv group over the same 32 queries (fewer heads in a group: the other
// waves take later queries), so one staged tile of 64 keys serves 256 query rows, and it is the value tile too.  Bound by
// LDS reads and the matrix cores alike (72 KB and 72 32x32x16 products per wave and tile of 320-wide rows), hence
//  * S^T = K Q^T and O^T += V^T P^T: a lane keeps one query, its maximum and sum are in registers, and P^T leaves the
//    score accumulators in the layout the value product reads, with no trip through LDS.
//  * 32 queries per wave, all of Q and O^T in registers (208 of 256 at 320 / 256): two waves per SIMD, one's softmax under
//    the other's products.  At 320 the scores go by 32 keys, and key / value fragments are read two products ahead by hand:
//    left to itself the compiler reads each right before its product (or spills).
//  * tiles by LDS-DMA, two slots, the next tile's issued at the barrier that opens this one.  Tiles lie as panels of 64 or
//    32 numbers so that a lane's DMA source is one offset; the chunk permutation spreads both the 16-byte key reads and the
//    transposed value reads over all banks.
//  * query rows come and result rows go through LDS as whole lines: stored from the accumulators' layout, 8 bytes a row,
//    a 16-token call at 320 / 256 took 24 us, now 12.
// 16 heads, one causal prompt (us, the 64-row kernel with separate query and head tiles / this one):
//   320 / 256  256 tokens 28 / 24, 1024 92 / 61, 2048 342 / 118, 4096 1157 / 231, 7680 3044 / 514 (1057 TFLOP/s)
//   160 / 128  256 tokens 21 / 15, 1024 67 / 37, 7680 1270 / 278;  192 / 128  7680 1337 / 298;  128 / 96  7680 938 / 240
// Nearer the peak than this the 32-key softmax steps and the last, partly filled wave of workgroups stand in the way.
constexpr int LW = 8, LNT = LW * 64, LKT = 64;              // waves, threads, keys per tile (one page)

template <int D>
struct LatGeo {
  static constexpr int WC = D % 64 == 0 ? 8 : 4;             // 16-byte chunks of a panel row
  static constexpr int PANEL = LKT * WC * 16;                // bytes of one panel: 64 keys x WC chunks
  static constexpr int NP = D / (8 * WC);                    // panels of a tile
  static constexpr int TILE = LKT * D * 2;
  static constexpr int RPI = 64 / WC;                        // key rows of one DMA instruction
  static constexpr int PIECES = TILE / 1024, RB = LKT / RPI; // DMA instructions of a tile, row blocks of a panel
  static constexpr int RING = 2;
  static constexpr int STAGE = LW * 32 * 144;                // query / output rows on their way
  static constexpr int LDS = RING * TILE > STAGE ? RING * TILE : STAGE;
  static constexpr int NB = D <= 192 ? 2 : 1;                // 32-key blocks per softmax step
  static constexpr int RK = D <= 192 ? 4 : 3, RV = D <= 192 ? 4 : 3;   // key / value fragments in registers
  __device__ static __forceinline__ int swz(int r) {         // a row's chunk permutation
    if constexpr (WC == 8) return (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
    else return (r >> 2) & 3;
  }
};

__device__ __forceinline__ float half_max_l(float x) {       // over lanes i, i ^ 32
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum_l(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ void glds16_l(const void* g, void* lds_base) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)lds_base, 16, 0, 0);
}
// (through the builtin the compiler waits for the tile DMA in flight before every transposed read)
template <int OFF>
__device__ __forceinline__ v4s tr16_l(uint32_t addr) {       // four keys of this lane's value column
  v4s r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "i"(OFF));
  return r;
}

// O^T += V^T P^T over 32 keys.  Step I takes value block I % DB of the 16 keys I / DB; its columns are read RV - 1 steps
// ahead.  The reads are not tracked by the compiler: the wait counts them and names their registers.
template <int D, int DB, int RV>
struct LatPv {
  using L = LatGeo<D>;
  static constexpr int A = L::WC / 4, N = 2 * DB;
  template <int I>
  __device__ static __forceinline__ void read(uint32_t vr, v4s (&lo)[RV], v4s (&hi)[RV]) {
    if constexpr (I < N) {
      constexpr int OFF = I / DB * 16 * L::WC * 16 + I % DB / A * L::PANEL;
      lo[I % RV] = tr16_l<OFF>(vr ^ (I % DB % A * 64));
      hi[I % RV] = tr16_l<OFF>((vr ^ (I % DB % A * 64 + 32)) + 8 * L::WC * 16);
    }
  }
  template <int I>
  __device__ static __forceinline__ void step(uint32_t vr, const v8s (&pb)[2], v16f (&o)[DB],
                                              v4s (&lo)[RV], v4s (&hi)[RV]) {
    read<I + RV - 1>(vr, lo, hi);
    constexpr int AHEAD = 2 * (N - 1 - I < RV - 1 ? N - 1 - I : RV - 1);
    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(lo[I % RV]), "+v"(hi[I % RV]) : "n"(AHEAD));
    __builtin_amdgcn_sched_barrier(0);
    const v4s a = lo[I % RV], b = hi[I % RV];
    const v8s vf = v8s{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    o[I % DB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pb[I / DB], o[I % DB], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (I + 1 < N) step<I + 1>(vr, pb, o, lo, hi);
  }
  __device__ static __forceinline__ void run(uint32_t vr, const v8s (&pb)[2], v16f (&o)[DB]) {
    v4s lo[RV], hi[RV];
    read<0>(vr, lo, hi);
    if constexpr (RV > 2) read<1>(vr, lo, hi);
    if constexpr (RV > 3) read<2>(vr, lo, hi);
    step<0>(vr, pb, o, lo, hi);
  }
};

template <int D, int DV>
__global__ void __launch_bounds__(LNT) latent_attn_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ gate, int gate_ld, const bf16_t* __restrict__ kp,
    const int* __restrict__ seq_slot, const int* __restrict__ seq_start, const int* __restrict__ seq_len,
    const int* __restrict__ seq_off, const int* __restrict__ ptab, int ptab_ld, bf16_t* __restrict__ out, int n, int H,
    int G, int hw, float scale_log2, int window, int kld, int out_ld, float out_scale, int vec_out) {
  using L = LatGeo<D>;
  constexpr int KK = D / 16, DB = DV / 32, NB = L::NB, WC = L::WC;
  static_assert(D % 32 == 0 && DV % 32 == 0 && DV <= D && L::PIECES % 4 == 0, "panels");
  __shared__ __attribute__((aligned(1024))) char smem[L::LDS];
  // (hw is a power of two: a step of 100 short sequences walks up to 100 lengths here, and a division each cost 5 us)
  const int lhw = __ffs(hw) - 1, ltm = 8 - lhw, TM = 1 << ltm;
  static_assert(LW == 8, "32 queries by 8 waves");
  // neighbours share a query tile and differ in heads; late query tiles see the most keys: they go first
  const int hgs = H / hw, hg = blockIdx.x % hgs;
  int qt = (int)((gridDim.x - 1 - blockIdx.x) / hgs), s = 0;
  for (; s < n; ++s) {
    const int nq = (seq_len[s] + TM - 1) >> ltm;
    if (qt < nq) break;
    qt -= nq;
  }
  if (s == n) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 31, g2 = lane >> 5;
  const int h = hg * hw + (wave & (hw - 1)), g = hg * hw / (H / G);
  const int start = seq_start[s], len = seq_len[s], off = seq_off[s];
  const int* pt = ptab + (size_t)seq_slot[s] * ptab_ld;
  const int wq0 = qt * TM + (wave >> lhw) * 32, tq = wq0 + c, qpos = start + tq;
  const int imin = start + qt * TM, imax = start + min(len, qt * TM + TM) - 1;
  const int t0 = window > 0 ? max(0, imin - window + 1) / LKT : 0, ntiles = imax / LKT - t0 + 1;

  // query rows come in runs of 32 QB numbers and turn into fragments in LDS (the tiles' memory, before the first tile)
  constexpr int QB = D % 64 == 0 ? 2 : 1, QS = QB * 64 + 16, QPR = QB * 4, QR = 64 / QPR, QI = 32 / QR;
  static_assert(LW * 32 * QS <= L::STAGE, "query rows");
  v8s qf[KK];
  {
    v8s in[KK];                                              // [run][row block]
#pragma unroll
    for (int i = 0; i < KK; ++i)
      in[i] = *reinterpret_cast<const v8s*>(q + ((size_t)(off + min(wq0 + i % QI * QR + lane / QPR, len - 1)) * H + h) * D +
                                            i / QI * QB * 32 + lane % QPR * 8);
    char* const qw = smem + wave * 32 * QS;
#pragma unroll
    for (int i0 = 0; i0 < KK; i0 += QI) {
#pragma unroll
      for (int i = 0; i < QI; ++i) *reinterpret_cast<v8s*>(qw + (i * QR + lane / QPR) * QS + lane % QPR * 16) = in[i0 + i];
      __builtin_amdgcn_s_waitcnt(0xC07F);                    // lgkmcnt(0)
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < QI; ++i) qf[i0 + i] = *reinterpret_cast<const v8s*>(qw + c * QS + (i * 2 + g2) * 16);
      __builtin_amdgcn_wave_barrier();
    }
  }
  __syncthreads();

  // tile DMA: instruction p brings 64 / WC rows of one panel; row and permuted chunk of a lane are the same for all of
  // a wave's instructions where the row blocks divide the waves
  static_assert(LW % L::RB == 0, "a wave keeps its row block");
  const int drow = (wave % L::RB) * L::RPI + lane / WC, dchunk = (lane % WC) ^ L::swz(drow);
  const uint32_t dsrc = (uint32_t)(drow * kld + g * D + dchunk * 8) * 2 + (wave / L::RB) * WC * 16;
  auto issue = [&](int t, int page) {
    char* slot = smem + (t % L::RING) * L::TILE;
    const char* base = reinterpret_cast<const char*>(kp) + (size_t)page * LKT * kld * 2;
#pragma unroll
    for (int i = 0; i < (L::PIECES + LW - 1) / LW; ++i) {
      const int p = wave + i * LW;
      if (L::PIECES % LW == 0 || p < L::PIECES)
        glds16_l(base + dsrc + i * (LW / L::RB) * WC * 16, slot + p * 1024);
    }
  };

  v16f o[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  float m_i = -INFINITY, l_i = 0.f;

  // per-lane LDS offsets inside a tile, key row c and the value columns of keys 4 g2 + qq (+ 8); the other chunks of a
  // panel differ in the bits that the permutation leaves to an exclusive or
  const uint32_t ka = c * WC * 16 + ((g2 ^ L::swz(c)) << 4);
  const int u = lane & 15, vrow = 4 * g2 + (u >> 2);
  const uint32_t va = vrow * WC * 16 + ((((lane >> 4) & 1) * 2 + ((u & 3) >> 1) ^ L::swz(vrow)) << 4) + 8 * (u & 1);
  const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) const char*)smem);

  issue(0, pt[t0]);
  int page1 = pt[t0 + min(1, ntiles - 1)];
  for (int t = 0; t < ntiles; ++t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                            // tile t has landed, tile t - 1's slot is free
    if (t + 1 < ntiles) issue(t + 1, page1);
    page1 = pt[t0 + min(t + 2, ntiles - 1)];
    const int k0 = (t0 + t) * LKT;
    if (wq0 >= len || k0 > start + wq0 + 31 || (window > 0 && k0 + LKT - 1 <= start + wq0 - window)) continue;
    const uint32_t vb = lds0 + (t % L::RING) * L::TILE + va;
    const bool full = k0 + LKT - 1 <= start + wq0 && (window <= 0 || start + wq0 + 31 - k0 < window);
#pragma unroll 1
    for (int b0 = 0; b0 < 2; b0 += NB) {
      v16f sc[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[nb][r] = 0.f;
        const uint32_t kr = (t % L::RING) * L::TILE + (b0 + nb) * 32 * WC * 16 + ka;
        auto key_frag = [&](int kk) {
          return *reinterpret_cast<const v8s*>(smem + (kr ^ (kk % (WC / 2) << 5)) + (kk / (WC / 2)) * L::PANEL);
        };
        v8s kf[L::RK];
#pragma unroll
        for (int kk = 0; kk < L::RK - 1; ++kk) kf[kk] = key_frag(kk);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          if (kk + L::RK - 1 < KK) kf[(kk + L::RK - 1) % L::RK] = key_frag(kk + L::RK - 1);
          __builtin_amdgcn_sched_barrier(0);
          sc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[kk % L::RK], qf[kk], sc[nb], 0, 0, 0);
        }
      }
      // lane holds S[key = 8 (r >> 2) + 4 g2 + (r & 3)][query c]
      if (!full) {                                           // keys counted from this block's first one of the lane
        const int last = qpos - k0 - b0 * 32 - 4 * g2, first = window > 0 ? last - window : INT_MIN;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = nb * 32 + 8 * (r >> 2) + (r & 3);
            sc[nb][r] = key <= last && key > first ? sc[nb][r] : -INFINITY;
          }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[nb][r]);
      mx = half_max_l(mx);
      const float mnew = fmaxf(m_i, mx * scale_log2);
      const float msafe = mnew == -INFINITY ? 0.f : mnew;
      const float alpha = __builtin_amdgcn_exp2f(m_i - msafe);
      m_i = mnew;
      v8s pb[NB][2];
      float rs = 0.f;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[nb][r], scale_log2, -msafe));
          rs += p;
          pb[nb][r >> 3][r & 7] = (short)f2bf(p);
        }
      l_i = l_i * alpha + rs;
      if (__any(alpha != 1.f)) {                             // a factor of exactly 1 changes nothing
#pragma unroll
        for (int i = 0; i < DB; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        LatPv<D, DB, L::RV>::run(vb + (b0 + nb) * 32 * WC * 16, pb[nb], o);
      }
    }
  }
  const float l = half_sum_l(l_i);
  float inv = l > 0.f ? 1.f / l : 0.f;
  if (gate) inv *= sigmoidf_(bf2f(gate[(size_t)(off + min(tq, len - 1)) * gate_ld + h]));
  if (!vec_out) {
    if (tq >= len) return;
    bf16_t* orow = out + (size_t)(off + tq) * out_ld + h * DV + 4 * g2;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) orow[db * 32 + 8 * (r >> 2) + (r & 3)] = f2bf(o[db][r] * inv * out_scale);
    return;
  }
  // rows leave through LDS as runs of 32 OB numbers: a lane holds 4 of a row, and as 8-byte stores they cost more than a
  // short prompt's tiles (the tiles' memory is free once every wave is past its last one)
  constexpr int OB = DB % 2 == 0 ? 2 : 1, OS = OB * 64 + 16, LPR = OB * 4, RPS = 64 / LPR;
  static_assert(LW * 32 * OS <= L::STAGE, "output rows");
  __syncthreads();
  char* const ow = smem + wave * 32 * OS;
#pragma unroll
  for (int d0 = 0; d0 < DB; d0 += OB) {
#pragma unroll
    for (int db = 0; db < OB; ++db)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const v16f& v = o[d0 + db];
        *reinterpret_cast<uint2*>(ow + c * OS + (db * 32 + 8 * j + 4 * g2) * 2) =
            make_uint2(pack_bf2(v[4 * j] * inv * out_scale, v[4 * j + 1] * inv * out_scale),
                       pack_bf2(v[4 * j + 2] * inv * out_scale, v[4 * j + 3] * inv * out_scale));
      }
    __builtin_amdgcn_s_waitcnt(0xC07F);                      // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < LPR / 2; ++i) {
      const int row = i * RPS + lane / LPR, e = lane % LPR;
      const uint4 v = *reinterpret_cast<const uint4*>(ow + row * OS + e * 16);
      if (wq0 + row < len) *reinterpret_cast<uint4*>(out + (size_t)(off + wq0 + row) * out_ld + h * DV + d0 * 32 + e * 8) = v;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

template <int D, int DV>
int launch_latent(const void* q, const void* gate, int gate_ld, const void* kp, const int* seq_slot, const int* seq_start,
                  const int* seq_len, const int* seq_off, const int* ptab, int ptab_ld, void* out, int n, int qtiles, int H,
                  int G, int hw, float sl2, int window, int kld, int out_ld, float out_scale, hipStream_t st) {
  const int vec_out = out_ld % 8 == 0 && (uintptr_t)out % 16 == 0;
  hipLaunchKernelGGL((latent_attn_kernel<D, DV>), dim3((H / hw) * (hw == 8 ? 2 * qtiles : qtiles)), dim3(LNT), 0, st,
                     (const bf16_t*)q, (const bf16_t*)gate, gate_ld, (const bf16_t*)kp, seq_slot, seq_start, seq_len, seq_off,
                     ptab, ptab_ld, (bf16_t*)out, n, H, G, hw, sl2, window, kld, out_ld, out_scale, vec_out);
  return (int)hipGetLastError();
}

}  // namespace

extern "C" {

// Full and sliding-window causal attention of prompt portions over latent pages of 64 rows; H % G == 0, kld % 8 == 0, rows
// and queries 16-byte aligned.  Returns 1 when it does not take the call (the caller then runs the general kernel).
int edge_sm_attention_latent(const void* q, const void* gate, int gate_ld, const void* kp, const int* seq_slot,
                             const int* seq_start, const int* seq_len, const int* seq_off, const int* ptab, int ptab_ld,
                             void* out, int n, int qtiles, int H, int G, int D, int Dv, float scale_log2, int window, int kld,
                             int out_ld, float out_scale, hipStream_t st) {
  // eight heads a workgroup once that gives one for every CU: on short steps eight waves of 320-wide rows only wait longer
  const int R = H / G, hw = R % 8 == 0 && 2 * qtiles * (H / 8) >= 256 ? 8 : R % 4 == 0 ? 4 : R % 2 == 0 ? 2 : 1;
  if (!(scale_log2 > 0.f) || (int64_t)LKT * kld * 2 > INT_MAX) return 1;   // the maximum is taken before the scale
#define LAT(DD, DDV)                                                                                                       \
  return launch_latent<DD, DDV>(q, gate, gate_ld, kp, seq_slot, seq_start, seq_len, seq_off, ptab, ptab_ld, out, n, qtiles, \
                                H, G, hw, scale_log2, window, kld, out_ld, out_scale, st)
  if (D == 128 && Dv == 96) LAT(128, 96);
  if (D == 160 && Dv == 128) LAT(160, 128);
  if (D == 192 && Dv == 128) LAT(192, 128);
  if (D == 320 && Dv == 256) LAT(320, 256);
#undef LAT
  return 1;
}

}  // extern "C"
