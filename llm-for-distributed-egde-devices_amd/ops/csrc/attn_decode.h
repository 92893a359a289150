// Body of the split-K decode attention (attn_decode.hip says how it works; decode_pair.hip runs it beside a projection).
#pragma once
#include "common.h"

namespace {
constexpr int ATTN_NT = 256;
constexpr int ATTN_NW = ATTN_NT / 64;
constexpr int UNROLL_DEF = 4;   // key groups per wave per chunk (tune "decode_attn_unroll": 8 at MHA D = 128)

struct Fuse {
  const int* pos;       // [B] cache position of the new token (seq_lens - 1)
  const float* cs;      // rope table [max_pos, rot/2] float2 (cos, sin) or null
  int rot;              // rotary dims (0: no rotation)
  int64_t qkv_sb;       // row stride of the QKV input (elements)
  int8_t* out_q;        // QOUT: [B, Hq*D] int8
  float* out_s;         // QOUT: [(Hq*D)/64][Mpad] scales
  int Mpad;
  int gs;               // query heads of one KV head split over gs workgroups (G = 1 in the kernel)
  int early;            // OCC > 0: issue the first K/V chunk at kernel entry (A/B knob decode_attn_early)
};

// Rotate the 8 values at head offset e0 (HF rotate_half convention), x/partner read from `head`.
template <bool HF>
__device__ __forceinline__ void rope8(const bf16_t* __restrict__ head, int e0, int rot, const float2* csp,
                                      float (&v)[8]) {
  const int half = rot / 2;
  const bool lo = e0 < half;
  const int pe = lo ? e0 + half : e0 - half;
  const int fi = lo ? e0 : e0 - half;
  float p[8];
  unpack8e<HF>(*reinterpret_cast<const uint4*>(head + pe), p);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float2 r = csp[fi + j];
    v[j] = lo ? (v[j] * r.x - p[j] * r.y) : (v[j] * r.x + p[j] * r.y);
  }
}

// Quantise one 64-column group held one value per lane (a full wave) and store it.
__device__ __forceinline__ void quant_group_store(float v, int8_t* q, float* s_slot, int lane) {
  const float amax = fmaxf(wave_max(fabsf(v)), 1e-8f);
  *q = quant_i8(v, 127.f / amax);
  if (lane == 0) *s_slot = amax / 127.f;
}

template <int D> struct Lanes { static constexpr int v = (D / 8 <= 8) ? 8 : ((D / 8 <= 16) ? 16 : 32); };

// OCC > 0: single-buffered key loop, nontemporal K/V loads and at least OCC waves per SIMD
// (occupancy instead of a second register buffer), and FUSED keeps the new key in registers (no
// append barrier); OCC = 0: two register buffers, no occupancy target.  NWV: waves per workgroup.
// HF: q / K / V / out are IEEE fp16 instead of bf16 (the reference's fp16 agents); fp32 softmax.
// One workgroup (bx: key split, by of ny: KV head x head split, b: row) of NWV waves.
template <int D, int G, bool DIRECT, bool FUSED, bool QOUT, int OCC, bool HF, int NWV, int UNROLL>
__device__ __forceinline__ void decode_attn_body(
    float* smem, int bx, int by, int ny, int b, const bf16_t* __restrict__ q, int64_t q_sb, bf16_t* __restrict__ kc,
    bf16_t* __restrict__ vc, int64_t c_sb, int64_t c_sh, const int* __restrict__ seq_lens, float scale_log2, int CH,
    int nsplit, bf16_t* __restrict__ out, int64_t o_sb, float* __restrict__ part_acc, float* __restrict__ part_ml,
    const Fuse& fz) {
  constexpr int LPK = Lanes<D>::v;        // lanes per key row
  constexpr int KPW = 64 / LPK;           // keys per wave-instruction
  constexpr int KPB = KPW * NWV;           // keys per workgroup step
  float* red = smem;                      // [NWV][G][D] per-wave accumulators
  float* wm = red + NWV * G * D;           // [NWV][G] per-wave running max
  float* wl = wm + NWV * G;                // [NWV][G] per-wave sums

  // head split (fz.gs > 1, G = 1): workgroup y serves query head y of KV head y / gs; every
  // such workgroup rebuilds the new key / value in registers, only the first one stores it
  const int split = bx, kvh = by / fz.gs, qh0 = by * G;
  const int Hq = ny * G;
  const int len = seq_lens[b];
  const int start = split * CH;
  const int end = min(start + CH, len);
  const int n = end - start;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int dl = lane % LPK, kl = lane / LPK;
  const int d0 = dl * 8;
  const bool dvalid = d0 < D;

  if (n <= 0) {  // empty split (seq shorter than the grid's hint): publish an empty partial
    if (!DIRECT) {
      for (int i = threadIdx.x; i < G * D; i += (NWV * 64)) {
        const int h = i / D, d = i - h * D;
        part_acc[(((size_t)b * Hq + qh0 + h) * nsplit + split) * D + d] = 0.f;
      }
      if (threadIdx.x < G) {
        float* ml = part_ml + (((size_t)b * Hq + qh0 + threadIdx.x) * nsplit + split) * 2;
        ml[0] = -INFINITY; ml[1] = 0.f;
      }
    }
    return;
  }

  const bf16_t* kb = kc + b * c_sb + kvh * c_sh + (size_t)start * D;
  const bf16_t* vb = vc + b * c_sb + kvh * c_sh + (size_t)start * D;

  // K / V loads of UNROLL key groups from `base`: rows at or past `bound` load row 0 (unconditional
  // 16-byte loads; consume() masks every key past nl)
  constexpr int STEP = KPB * UNROLL;      // keys per workgroup per chunk
  const int dc = dvalid ? d0 : 0;
  auto load_b = [&](int base, int bound, uint4 (&kr)[UNROLL], uint4 (&vr)[UNROLL]) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int k = base + kl + u * KPB;
      const size_t off = (size_t)(k < bound ? k : 0) * D + dc;
      if (UNROLL > UNROLL_DEF && base + u * KPB >= bound) {   // wave-uniform: a whole group past the end
        kr[u] = uint4{0, 0, 0, 0};                              // (masked in consume; zero, never NaN)
        vr[u] = uint4{0, 0, 0, 0};
        continue;
      }
      if constexpr (OCC > 0) {                   // read once per step: nontemporal
        kr[u] = __builtin_bit_cast(uint4, __builtin_nontemporal_load(reinterpret_cast<const v4i*>(kb + off)));
        vr[u] = __builtin_bit_cast(uint4, __builtin_nontemporal_load(reinterpret_cast<const v4i*>(vb + off)));
      } else {
        kr[u] = *reinterpret_cast<const uint4*>(kb + off);
        vr[u] = *reinterpret_cast<const uint4*>(vb + off);
      }
    }
  };
  // OCC > 0: the wave's first chunk goes out now, before the q / RoPE / append work below (it
  // needs only the split's start and length), so one memory round trip of each workgroup's
  // critical path overlaps the q loads.  Bound n, not nl: in the split that owns the new position
  // that row may load stale, and consume() masks it (key nl) like every key past nl.
  const int base0 = wave * KPW;
  uint4 ka[UNROLL], va[UNROLL];
  if constexpr (OCC > 0) {
    if (fz.early && base0 < n) load_b(base0, n, ka, va);
  }

  // q first: its loads (and the RoPE partner loads) overlap the KV append below
  float qf[G][8];
#pragma unroll
  for (int h = 0; h < G; ++h) {
    if (dvalid) {
      const bf16_t* qh = q + b * q_sb + (size_t)(qh0 + h) * D;
      unpack8e<HF>(*reinterpret_cast<const uint4*>(qh + d0), qf[h]);
      if constexpr (FUSED) {
        if (d0 < fz.rot) {
          rope8<HF>(qh, d0, fz.rot, reinterpret_cast<const float2*>(fz.cs) + (size_t)fz.pos[b] * (fz.rot / 2), qf[h]);
#pragma unroll
          for (int j = 0; j < 8; ++j) qf[h][j] = e2f<HF>(f2e<HF>(qf[h][j]));   // q is 16-bit in the unfused path
        }
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[h][j] *= scale_log2;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[h][j] = 0.f;
    }
  }

  // OCC > 0 keeps the new token's rotated k and v in wave 0's registers (lanes kl = 0 / 1 hold
  // dims d0..d0+7) and adds that key to the softmax directly, so no barrier orders the append
  // before the cache reads and the K/V loads start at once; the cache loop skips the new key.
  float knew[8], vnew[8];
  bool own = false;
  if constexpr (FUSED) {
    // append the new token's rotated k and its v (only the split that owns the position)
    const int pos = fz.pos[b];
    own = pos >= start && pos < end;
    const int Hkv = ny / fz.gs;
    const bf16_t* row = q + b * fz.qkv_sb;
    const float2* csp = reinterpret_cast<const float2*>(fz.cs) + (size_t)pos * (fz.rot / 2);
    if constexpr (OCC > 0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) { knew[j] = 0.f; vnew[j] = 0.f; }
      if (own && wave == 0 && kl < 2 && dvalid) {
        const bool is_v = kl == 1;
        const bf16_t* head = row + (size_t)((is_v ? Hq + Hkv : Hq) + kvh) * D;
        float v[8];
        unpack8e<HF>(*reinterpret_cast<const uint4*>(head + d0), v);
        if (!is_v && d0 < fz.rot) rope8<HF>(head, d0, fz.rot, csp, v);
        if (by % fz.gs == 0)
          *reinterpret_cast<uint4*>((is_v ? vc : kc) + b * c_sb + kvh * c_sh + (size_t)pos * D + d0) = pack8e<HF>(v);
#pragma unroll
        for (int j = 0; j < 8; ++j) {                // the cached 16-bit value
          const float r = e2f<HF>(f2e<HF>(v[j]));
          knew[j] = is_v ? 0.f : r;
          vnew[j] = is_v ? r : 0.f;
        }
      }
    } else {
      if (own) {
        for (int c = threadIdx.x; c < 2 * (D / 8); c += (NWV * 64)) {
          const bool is_v = c >= D / 8;
          const int e0 = (is_v ? c - D / 8 : c) * 8;
          const bf16_t* head = row + (size_t)((is_v ? Hq + Hkv : Hq) + kvh) * D;
          float v[8];
          unpack8e<HF>(*reinterpret_cast<const uint4*>(head + e0), v);
          if (!is_v && e0 < fz.rot) rope8<HF>(head, e0, fz.rot, csp, v);
          *reinterpret_cast<uint4*>((is_v ? vc : kc) + b * c_sb + kvh * c_sh + (size_t)pos * D + e0) = pack8e<HF>(v);
        }
      }
      // Only this workgroup reads the new row, so the barrier's workgroup-scope release/acquire is
      // enough (an agent-scope __threadfence would write back L2 in every workgroup: 3x slower).
      __syncthreads();
    }
  }
  const int nl = (OCC > 0 && FUSED && own) ? n - 1 : n;   // keys read from the cache

  // ---- one pass: each wave keeps an online softmax (m, l, acc) over its key slice; K and V rows
  // are loaded together and the next chunk is in flight while the current one is consumed
  // (two register buffers, alternated by a 2x unrolled loop: copying a buffer that still has
  // loads outstanding would force a full wait).  Out-of-range keys load a clamped row and are
  // masked in the score (unconditional 16-byte loads; a conditional one compiles to branches).
  float m[G], l[G], acc[G][8];
#pragma unroll
  for (int h = 0; h < G; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[h][j] = 0.f;
  }
  auto load = [&](int base, uint4 (&kr)[UNROLL], uint4 (&vr)[UNROLL]) { load_b(base, nl, kr, vr); };
  auto consume = [&](int base, const uint4 (&kr)[UNROLL], const uint4 (&vr)[UNROLL]) {
    float s[UNROLL][G];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      float kf[8];
      unpack8e<HF>(kr[u], kf);
#pragma unroll
      for (int h = 0; h < G; ++h) {
        float a = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) a += qf[h][j] * kf[j];
        s[u][h] = a;
      }
    }
#pragma unroll
    for (int o = LPK / 2; o > 0; o >>= 1)
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
#pragma unroll
        for (int h = 0; h < G; ++h) s[u][h] = xor_sum(s[u][h], o);
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
      if (base + kl + u * KPB >= nl) {
#pragma unroll
        for (int h = 0; h < G; ++h) s[u][h] = -INFINITY;
      }
#pragma unroll
    for (int h = 0; h < G; ++h) {
      float cm = s[0][h];
#pragma unroll
      for (int u = 1; u < UNROLL; ++u) cm = fmaxf(cm, s[u][h]);
#pragma unroll
      for (int o = LPK; o < 64; o <<= 1) cm = xor_max(cm, o);
      // cm is finite: key `base` (kl = 0, u = 0) is in range whenever a chunk is consumed
      const float mn = fmaxf(m[h], cm);
      const float alpha = __builtin_amdgcn_exp2f(m[h] - mn);        // 0 on the first chunk (m = -inf)
      m[h] = mn;
      l[h] *= alpha;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[h][j] *= alpha;
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      float vf[8];
      unpack8e<HF>(vr[u], vf);
#pragma unroll
      for (int h = 0; h < G; ++h) {
        const float p = __builtin_amdgcn_exp2f(s[u][h] - m[h]);    // masked keys: exp2(-inf) = 0
        l[h] += p;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[h][j] += p * vf[j];
      }
    }
  };
  if constexpr (OCC > 0 && FUSED) {
    if (own && wave == 0) {                          // the new key first: m = its score, l = 1
#pragma unroll
      for (int h = 0; h < G; ++h) {
        float sp = 0.f;
        if (kl == 0) {
#pragma unroll
          for (int j = 0; j < 8; ++j) sp += qf[h][j] * knew[j];
        }
#pragma unroll
        for (int o = LPK / 2; o > 0; o >>= 1) sp = xor_sum(sp, o);
        m[h] = __shfl(sp, dl, 64);                   // lane dl holds the kl = 0 group's sum
        if (kl == 1) {
          l[h] = 1.f;
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[h][j] = vnew[j];
        }
      }
    }
  }
  if constexpr (OCC > 0) {
    for (int base = base0; base < nl; base += STEP) {  // wave-uniform trip count (shuffles inside)
      if (base != base0 || !fz.early) load(base, ka, va);   // (early: the first chunk went out at entry)
      consume(base, ka, va);
    }
  } else {
    uint4 kb2[UNROLL], vb2[UNROLL];
    int base = wave * KPW;                           // wave-uniform trip count (shuffles inside)
    if (base < nl) load(base, ka, va);
    while (base < nl) {
      const int nb = base + STEP;
      if (nb < nl) load(nb, kb2, vb2);
      consume(base, ka, va);
      if (nb >= nl) break;
      const int nb2 = nb + STEP;
      if (nb2 < nl) load(nb2, ka, va);
      consume(nb, kb2, vb2);
      base = nb2;
    }
  }
  // reduce over the KPW key groups of this wave (lanes sharing dl)
#pragma unroll
  for (int o = LPK; o < 64; o <<= 1)
#pragma unroll
    for (int h = 0; h < G; ++h) {
      l[h] = xor_sum(l[h], o);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[h][j] = xor_sum(acc[h][j], o);
    }
  // merge the waves: every wave's sums and maximum meet at one barrier, and each output thread weighs the waves itself
  // (maxima, scaled sums and denominators in a step each were three barriers of all waves; one sequence of 41 / 141 / 251 keys, us:
  // 32 heads of 64 in 8 groups 5.35 / 5.5 / 5.95 -> 4.65 / 4.7 / 5.3, 32 heads of 128 in 8 groups 5.6 / 8.0 / 9.4 -> 4.9 / 6.9 / 8.2)
#pragma unroll
  for (int h = 0; h < G; ++h) {
    if (kl == 0 && dvalid) {
      float4* dst = reinterpret_cast<float4*>(&red[(wave * G + h) * D + d0]);
      dst[0] = make_float4(acc[h][0], acc[h][1], acc[h][2], acc[h][3]);
      dst[1] = make_float4(acc[h][4], acc[h][5], acc[h][6], acc[h][7]);
    }
    if (lane == 0) { wm[wave * G + h] = m[h]; wl[wave * G + h] = l[h]; }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < G * D; i += (NWV * 64)) {
    const int h = i / D, d = i - h * D;
    float M = wm[h];
#pragma unroll
    for (int w = 1; w < NWV; ++w) M = fmaxf(M, wm[w * G + h]);
    float a = 0.f, L = 0.f;
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      const float x = __builtin_amdgcn_exp2f(wm[w * G + h] - M);    // wave without keys: exp2(-inf) = 0
      L += wl[w * G + h] * x;
      a += red[(w * G + h) * D + d] * x;
    }
    const int hq = qh0 + h;
    if (DIRECT) {
      if constexpr (QOUT) {     // D % 64 == 0: each 64-column group is one wave of this loop
        const float vq = e2f<HF>(f2e<HF>(a / L));
        const int col = hq * D + d;
        quant_group_store(vq, fz.out_q + (size_t)b * Hq * D + col, fz.out_s + (size_t)(col >> 6) * fz.Mpad + b,
                          threadIdx.x & 63);
      } else {
        out[b * o_sb + (size_t)hq * D + d] = f2e<HF>(a / L);
      }
    } else {
      part_acc[(((size_t)b * Hq + hq) * nsplit + split) * D + d] = a;
      if (d == 0) {
        float* ml = part_ml + (((size_t)b * Hq + hq) * nsplit + split) * 2;
        ml[0] = M;
        ml[1] = L;
      }
    }
  }
}
}  // namespace
