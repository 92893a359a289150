// Prompt attention over a paged cache in fp32 (pages of 64 tokens) on the fp32 matrix instruction: every number stays 32 bits wide.
// Bound by that instruction's rate (a quarter of attn_kernel's fused multiply-adds a clock would be as much, but those wait for LDS
// reads of both factors).  Scores are formed transposed, keys x queries, so that a lane holds four keys of its own query: the softmax
// is the lane's own but for two exchanges, and the weights are the value product's operand as they stand, without a way through the LDS.
// A workgroup has KS groups of RW waves.  A group's waves are 16 positions of HW query heads of one kv head each (HW = 4, 2 or 1: a
// staged tile serves 16 RW rows), the groups take the key tiles in turn and add up through the LDS, for few workgroups leave a SIMD with one
// wave, whose softmax nothing covers.  The next tile's rows travel to registers beside the products.
// Values of keys that a query does not see never meet it, not even as 0 x infinity: rows past the workgroup's last position are staged
// as zeros, and a tile that holds numbers that are not finite is multiplied key by key where its mask cuts.
#include <type_traits>

#include "common.h"
#include "seqmix/seqmix_common.h"

namespace {

struct F32Attn {
  const float *q, *gate, *kp, *vp, *kb, *vb, *slopes, *sink, *rel;
  const int *seq_slot, *seq_start, *seq_len, *seq_off, *ptab;
  float* out;
  int n, H, G, PB, gate_ld, gate_elem, ptab_ld, window, pool_sh, kld, vld, chunked, keep_first, rel_n, out_ld, hw;
  float scale, cap, out_scale;
};

constexpr int FK = 64;                                       // keys of a tile: one page

// LDS of a group of RW waves, in floats: the key and the value tile, or at the end its sums
template <int D, int Dv, bool KVS, int RW>
constexpr int group_floats() {
  constexpr int tile = FK * (D + 4) + (KVS ? 0 : FK * Dv), sums = (Dv / 4 + 2) * 64 * RW;
  return tile > sums ? tile : sums;
}

template <int D, int Dv, bool KVS, int RW, int KS>
__global__ void __launch_bounds__(64 * RW * KS, 2) attn_f32_kernel(F32Attn a) {
  constexpr float LOG2E = 1.4426950408889634f;
  constexpr int KLD = D + 4, VLD = KVS ? KLD : Dv, NB = Dv / 64, HB = Dv % 64 / 32, GF = group_floats<D, Dv, KVS, RW>(), GT = 64 * RW;
  static_assert(D % 16 == 0 && Dv % 32 == 0 && (!KVS || Dv <= D), "rows of whole matrix operands");
  __shared__ __attribute__((aligned(16))) float smem[KS * GF];
  __shared__ int odd_s[KS];                                  // the last tile of a group with a value that is not finite
  const int lane = threadIdx.x & 63, g4 = lane >> 4, c16 = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kg = wv / RW, wave = wv % RW, tid = threadIdx.x % GT;
  float* const k_lds = smem + kg * GF;
  float* const v_lds = KVS ? k_lds : k_lds + FK * KLD;
  const int QT = 16 * RW / a.hw;                                 // positions of a workgroup
  int qt = gridDim.y - 1 - blockIdx.y, s = 0;                // the last positions, which see the most keys, first
  for (; s < a.n; ++s) {
    const int nq = (a.seq_len[s] + QT - 1) / QT;
    if (qt < nq) break;
    qt -= nq;
  }
  if (s == a.n) return;
  const int h0 = blockIdx.x * a.hw, g = h0 / (a.H / a.G), h = h0 + wave % a.hw;
  const int start = a.seq_start[s], len = a.seq_len[s], off = a.seq_off[s];
  const int* pt = a.ptab + (size_t)a.seq_slot[s] * a.ptab_ld;
  const int w0 = qt * QT + wave / a.hw * 16, t = w0 + c16, qpos = start + t;   // this wave's first and this lane's row
  float qf[D / 4];
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    const v4f x = *reinterpret_cast<const v4f*>(a.q + ((size_t)(off + min(t, len - 1)) * a.H + h) * D + kk * 16 + 4 * g4);
#pragma unroll
    for (int j = 0; j < 4; ++j) qf[kk * 4 + j] = x[j] * a.scale;
  }
  v4f o[Dv / 16];
#pragma unroll
  for (int i = 0; i < Dv / 16; ++i) o[i] = v4f{0.f, 0.f, 0.f, 0.f};
  const bool sk = a.sink && kg == 0;                         // the sink: a starting maximum with sum 1 and no value
  float m = sk ? a.sink[h] * LOG2E : -INFINITY, l = sk && g4 == 0 ? 1.f : 0.f;   // l: this lane's keys' share of the sum
  const float slope = a.slopes ? a.slopes[h] : 0.f;
  const float* relh = a.rel ? a.rel + (size_t)h * a.rel_n : nullptr;
  const int window = a.window, imin = start + qt * QT, imax = start + min(len, qt * QT + QT) - 1;
  const int lo = window > 0 ? (a.chunked ? qpos / window * window : max(0, qpos - window + 1)) : 0;   // this row's first key
  const int wlast = start + w0 + 15, lolast = window > 0 ? (a.chunked ? wlast / window * window : max(0, wlast - window + 1)) : 0;
  const bool pooled = !KVS && window > 0 && a.pool_sh >= 0;
  const int seen = pooled && qpos - window + 1 > 0 ? (qpos - window + 1) >> a.pool_sh : 0;
  const int seen0 = pooled && start + w0 - window + 1 > 0 ? (start + w0 - window + 1) >> a.pool_sh : 0;
  const int jlo = window > 0 ? (a.chunked ? imin / window * window : max(0, imin - window + 1)) : 0;
  const int nbmax = pooled && imax - window + 1 > 0 ? (imax - window + 1) >> a.pool_sh : 0;
  // the tiles that hold kept first tokens and lie wholly before the window's first tile come first
  const int nfirst = min((a.keep_first + FK - 1) / FK, jlo / FK);
  const int tok_tiles = nfirst + imax / FK - jlo / FK + 1, ntiles = tok_tiles + (nbmax + FK - 1) / FK;
  auto tile_base = [&](int tile) {                           // first position (token tiles) / block (pooled tiles) of a tile
    return tile < nfirst ? tile * FK : tile < tok_tiles ? (jlo / FK + tile - nfirst) * FK : (tile - tok_tiles) * FK;
  };
  // A tile's rows on their way: of the keys while the values' product runs, of the values while the keys' does (both at once would take
  // the registers of two more waves a SIMD); one tile for both travels beside the two products.
  constexpr int KL = D / (4 * RW), VL = Dv / (4 * RW);                 // 16-byte pieces per thread and tile
  v4f stage[KL > VL || KVS ? KL : VL];
  auto load_tile = [&](int tile, auto keys) {
    constexpr bool K = decltype(keys)::value;
    constexpr int W = K ? D : Dv, cpr = W / 4;
    const bool tok = tile < tok_tiles;
    const int base = tile_base(tile), ld = K ? a.kld : a.vld, last = (tok ? imax : nbmax - 1) - base;
    if (KVS || tok) {                                        // (rows past the last: that one, zeroed on their way to the LDS)
      const float* const rows = (K ? a.kp : a.vp) + (size_t)pt[base / FK] * FK * ld + g * W;
#pragma unroll
      for (int i = 0; i < W / (4 * RW); ++i) {
        const int e = tid + i * GT;
        stage[i] = *reinterpret_cast<const v4f*>(rows + (unsigned)(min(e / cpr, last) * ld + e % cpr * 4));
      }
    } else {
#pragma unroll
      for (int i = 0; i < W / (4 * RW); ++i) {
        const int e = tid + i * GT, p0 = (base + min(e / cpr, last)) << a.pool_sh;
        const size_t row = ((size_t)pt[p0 / FK] * a.PB + (p0 % FK >> a.pool_sh)) * a.G + g;
        stage[i] = *reinterpret_cast<const v4f*>((K ? a.kb : a.vb) + row * W + e % cpr * 4);
      }
    }
  };
  auto store_tile = [&](int tile, auto keys) {
    constexpr bool K = decltype(keys)::value;
    constexpr int W = K ? D : Dv, LD = K ? KLD : VLD;
    const int last = (tile < tok_tiles ? imax : nbmax - 1) - tile_base(tile);
    bool odd = false;
#pragma unroll
    for (int i = 0; i < W / (4 * RW); ++i) {
      const int e = tid + i * GT;
      const v4f x = e / (W / 4) <= last ? stage[i] : v4f{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<v4f*>((K ? k_lds : v_lds) + e / (W / 4) * LD + e % (W / 4) * 4) = x;
      if (!K || KVS) odd |= !(x[0] * 0.f + x[1] * 0.f + x[2] * 0.f + x[3] * 0.f == 0.f);   // infinities and NaN
    }
    if ((!K || KVS) && odd) odd_s[kg] = tile;
  };
  constexpr std::integral_constant<bool, true> KEYS{};
  constexpr std::integral_constant<bool, false> VALUES{};
  if (tid == 0) odd_s[kg] = -1;
  if (kg < ntiles) {
    load_tile(kg, KEYS);
    if (!KVS) store_tile(kg, KEYS);
  }
  for (int t0 = 0; t0 < ntiles; t0 += KS) {
    const int tile = t0 + kg;
    const bool mine = tile < ntiles;
    __syncthreads();                                         // every wave is done with the tile before
    if constexpr (KVS) {
      if (mine) store_tile(tile, KEYS);
      __syncthreads();
      if (tile + KS < ntiles) load_tile(tile + KS, KEYS);
    } else if (mine) load_tile(tile, VALUES);
    const bool tok = tile < tok_tiles;
    const int base = tile_base(tile);
    // whether every row of the wave sees every key of the tile
    const bool whole = tok ? base + FK - 1 <= start + w0 && base >= lolast : base + FK <= seen0;
    auto visible = [&](int key) { return tok ? key <= qpos && (key >= lo || key < a.keep_first) : key < seen; };
    float al = 1.f;
    v4f sc[4];                                               // [i]: the key 16 nt + 4 g4 + i of the tile, the lane's own query
    if (mine) {
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {                         // four sums a score: a quarter of the terms, half the error, and no chain
      constexpr v4f zero{0.f, 0.f, 0.f, 0.f};
      v4f part[4] = {zero, zero, zero, zero};
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) {
        const v4f kf = *reinterpret_cast<const v4f*>(k_lds + (nt * 16 + c16) * KLD + kk * 16 + 4 * g4);
#pragma unroll
        for (int j = 0; j < 4; ++j) part[j] = mfma4(kf[j], qf[kk * 4 + j], part[j]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) sc[nt][i] = (part[0][i] + part[1][i]) + (part[2][i] + part[3][i]);
    }
    if (tok) {
      if (KVS && a.cap > 0.f) {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int i = 0; i < 4; ++i) sc[nt][i] = a.cap * tanhf(sc[nt][i] / a.cap);
      }
      if (KVS && a.slopes) {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int i = 0; i < 4; ++i) sc[nt][i] -= slope * (float)(qpos - (base + nt * 16 + 4 * g4 + i));
      }
      if (!KVS && relh) {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int i = 0; i < 4; ++i) sc[nt][i] += relh[min(max(qpos - (base + nt * 16 + 4 * g4 + i), 0), a.rel_n - 1)];
      }
    }
    if (!whole) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) sc[nt][i] = visible(base + nt * 16 + 4 * g4 + i) ? sc[nt][i] : -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sc[nt][i]);
    mx = xor_max(xor_max(mx, 16), 32);
    const float mn = fmaxf(m, mx * LOG2E), ms = mn == -INFINITY ? 0.f : mn;   // (no key seen so far: every weight is 0)
    al = ex2(m - ms);
    float ls = 0.f;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sc[nt][i] = ex2(fmaf(sc[nt][i], LOG2E, -ms));
        ls += sc[nt][i];
      }
    l = l * al + ls;
    m = mn;
    }
    if constexpr (!KVS) {
      if (mine) store_tile(tile, VALUES);
      __syncthreads();
      if (tile + KS < ntiles) load_tile(tile + KS, KEYS);
    }
    if (mine && !whole && odd_s[kg] == tile) {               // rare: as the mask says, key by key
#pragma unroll
      for (int i = 0; i < Dv / 16; ++i) o[i] *= al;
      for (int key = 0; key < FK; ++key) {
        float p = 0.f;
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (key / 16 == nt && key % 4 == i) p = __shfl(sc[nt][i], (key % 16 / 4) * 16 + c16);
        if (!visible(base + key)) continue;
        const float* vr = v_lds + key * VLD;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
          for (int e = 0; e < 4 * NB; ++e) o[e][i] += p * vr[e / 4 * 64 + 16 * g4 + 4 * i + e % 4];
#pragma unroll
          for (int e = 0; e < 2 * HB; ++e) o[4 * NB + e][i] += p * vr[NB * 64 + 8 * g4 + 2 * i + e];
        }
      }
    } else if (mine) {
      // a tile's products in sums of their own (one sum over all keys was two to three times further from 64 bits behind 1000 keys)
#pragma unroll
      for (int b = 0; b < NB + HB; ++b) {
        constexpr v4f zero{0.f, 0.f, 0.f, 0.f};
        v4f part[4] = {zero, zero, zero, zero};
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float* vr = v_lds + (nt * 16 + 4 * g4 + j) * VLD + b * 64;
            if (b < NB) {
              const v4f vf = *reinterpret_cast<const v4f*>(vr + 4 * c16);
#pragma unroll
              for (int e = 0; e < 4; ++e) part[e] = mfma4(vf[e], sc[nt][j], part[e]);
            } else {
              const float2 vf = *reinterpret_cast<const float2*>(vr + 2 * c16);
              part[0] = mfma4(vf.x, sc[nt][j], part[0]);
              part[1] = mfma4(vf.y, sc[nt][j], part[1]);
            }
          }
#pragma unroll
        for (int e = 0; e < (b < NB ? 4 : 2); ++e)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[4 * b + e][i] = fmaf(o[4 * b + e][i], al, part[e][i]);
      }
    }
    if constexpr (!KVS) {
      if (tile + KS < ntiles) store_tile(tile + KS, KEYS);
    }
  }
  l = xor_sum(xor_sum(l, 16), 32);
  if constexpr (KS > 1) {                                    // the groups' sums, each number in its lane's place
    __syncthreads();
    if (kg > 0) {
      float* dst = smem + kg * GF + tid;
#pragma unroll
      for (int i = 0; i < Dv / 16; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[(i * 4 + e) * GT] = o[i][e];
      dst[Dv / 4 * GT] = m;
      dst[(Dv / 4 + 1) * GT] = l;
    }
    __syncthreads();
    if (kg > 0) return;
    float mg[KS], M = m;
#pragma unroll
    for (int k = 1; k < KS; ++k) { mg[k] = smem[k * GF + Dv / 4 * GT + tid]; M = fmaxf(M, mg[k]); }
    const float ms = M == -INFINITY ? 0.f : M;
    const float f0 = ex2(m - ms);
    l *= f0;
#pragma unroll
    for (int i = 0; i < Dv / 16; ++i) o[i] *= f0;
#pragma unroll
    for (int k = 1; k < KS; ++k) {
      const float f = ex2(mg[k] - ms);
      const float* src = smem + k * GF + tid;
      l += src[(Dv / 4 + 1) * GT] * f;
#pragma unroll
      for (int i = 0; i < Dv / 16; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[i][e] += src[(i * 4 + e) * GT] * f;
    }
  }
  if (t >= len) return;
  const float* gr = a.gate ? a.gate + (size_t)(off + t) * a.gate_ld : nullptr;
  const float gh = gr && !a.gate_elem ? sigmoidf_(gr[h]) : 1.f;
  float* orow = a.out + (size_t)(off + t) * a.out_ld + h * Dv;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int b = 0; b < NB + HB; ++b) {
      const int w = b < NB ? 4 : 2, c = b < NB ? b * 64 + 16 * g4 + 4 * i : NB * 64 + 8 * g4 + 2 * i;
      float y[4];
#pragma unroll
      for (int e = 0; e < w; ++e) {
        y[e] = o[4 * b + e][i] / l;
        if (gr) y[e] *= a.gate_elem ? sigmoidf_(gr[h * Dv + c + e]) : gh;
        y[e] *= a.out_scale;
      }
      if (b < NB) *reinterpret_cast<v4f*>(orow + c) = v4f{y[0], y[1], y[2], y[3]};
      else { orow[c] = y[0]; orow[c + 1] = y[1]; }
    }
  }
}

}  // namespace

extern "C" {

double edge_sm_attention_us(int rows, int H, int G, int D, int Dv, int kld, int vld, int page, int pool, long vis, long mean, uintptr_t addresses);

// Waves of query rows of a group in the low bits, groups above; 0: the step is not this kernel's.  vis: the most keys that a row sees,
// mean: as many as a row sees on average.  By estimates: an iteration is one tile of every group, its us were fitted to steps of up to six
// portions of 16 to 600 tokens behind 0 to 1500 (112 of them, eight head shapes of 32 to 160 numbers); the kernels before are taken at
// 0.85 of theirs (edge_sm_attention_us); or the form that the caller wants.  Chosen so, 600 other steps (16 head shapes of 2 to 32 heads, 16 to 6000
// rows, windows, pooled blocks) took 0.586 of the time before, at the worst 1.03 (two steps of 11.5 us), and 0.576 by the best form of each; at
// 1.0 of the estimate up to 1.24.  us before / four waves and two groups / two and two / two and four: 16 heads of 64 in 4 groups, 2000
// tokens 342 / 102 / 118 / 123, 500 behind 2000 215 / 112 / 85 / 68, 100 8.8 / 10.9 / 9.2 / 9.6, 20 behind 1000 16.7 / 48 / 37 / 30; of 128, 1000 tokens
// 205 / 87 / 78, 191 17.1 / 23.5 / 21.2; 16 of 160 over one latent, 300 tokens 65 / 33 / 26; a group per head of 64, 2000 tokens 1115 / 102 / 117 / 122.
// Error against 64 bits, relative: 1000 tokens 2.3e-7 before, 1.4e-7 here; 500 behind 2000 3.4e-7, 2.0e-7.
int edge_sm_attention_f32_plan(int rows, int n, int H, int G, int D, int Dv, int kld, int vld, int page, int pool, int out_ld, bool same, bool rel,
                               bool chunked, bool windowed, long vis, long mean, int want, uintptr_t addresses) {
  if ((same ? pool > 0 || rel : chunked) || (pool & (pool - 1)) || page != FK || G < 1 || H % G || rows < 1 || kld % 4 || vld % 4 ||
      out_ld % 4 || addresses % 16 || rows / 16 + n > 65535)   // (the grid's second number)
    return 0;
  const bool square = D == Dv && (D == 32 || D == 64 || D == 96 || D == 128);
  if (!square && !(same ? D == 160 && Dv == 128 : (D == 64 && Dv == 128) || (D == 128 && Dv == 64))) return 0;
  if (want) return want == 4 + 16 || want == 2 + 16 || (want == 2 + 32 && D <= 64 && Dv <= 64) ? want : 0;
  double best = 0.85 * edge_sm_attention_us(rows, H, G, D, Dv, kld, vld, page, pool, vis, mean, addresses);
  int plan = 0;
  const double w = (D + Dv) / 2, tiles = mean / (double)FK + 0.8, waves = rows * (double)H / 16;
  const long longest = (vis + FK - 1) / FK + (windowed ? 1 : 0);   // (a window begins inside a tile)
  // us: an iteration; crowd: what workgroups that share a CU lose over one that has it.  Behind a window all workgroups are as long, and
  // come in rounds of 256 (530 rows of 16 heads, window 512: 272 workgroups of two and four 44 us, 136 of four and two 34)
  const bool even = windowed && mean * 10 >= vis * 8;
  const int R = H / G;
  auto form = [&](int rw, int ks, double us, double crowd) {
    const int hw = rw == 4 && R % 4 == 0 ? 4 : R % 2 == 0 ? 2 : 1;
    const double chain = (longest + ks - 1) / ks * us, wgs = (rows * hw / (16. * rw) + n / 2.) * (H / hw);
    const double work = even ? ceil(wgs / 256 - 0.02) * chain : crowd * waves / rw / 256 * tiles / ks * us;
    const double t = 5.5 + (chain > work ? chain : work);
    if (t < best) { best = t; plan = rw + 8 * ks; }
  };
  form(4, 2, 0.7 + 0.064 * w, 1.);
  form(2, 2, 0.4 + 0.054 * w, 1.2);
  if (D <= 64 && Dv <= 64) form(2, 4, 0.8 + 0.068 * w, 1.5);
  return plan;
}

int edge_sm_attention_f32(const void* q, const void* gate, int gate_ld, const void* kp, const void* vp, const float* kb, const float* vb,
                          const int* seq_slot, const int* seq_start, const int* seq_len, const int* seq_off, const int* ptab, int ptab_ld,
                          void* out, int rows, int n, int H, int G, int D, int Dv, int PB, float scale, int window, int pool, int kld,
                          int vld, int chunked, float cap, const float* slopes, const float* sink, int gate_elem, int keep_first,
                          const float* rel, int rel_n, int out_ld, float out_scale, int plan, hipStream_t st) {
  if (n < 1 || rows < 1) return 0;
  if (G < 1 || H % G || (chunked && (pool > 0 || window < 0)) || keep_first < 0 || (rel && (rel_n < 1 || pool > 0)) || out_ld < H * Dv || (pool > 0 && window > 0 && (!kb || !vb)))
    return -2;
  const int R = H / G, rw = plan % 8, ks = plan / 8, hw = rw == 4 && R % 4 == 0 ? 4 : R % 2 == 0 ? 2 : 1;
  const F32Attn a{(const float*)q, (const float*)gate, (const float*)kp, (const float*)vp, kb, vb, slopes, sink, rel, seq_slot, seq_start,
                  seq_len, seq_off, ptab, (float*)out, n, H, G, PB, gate_ld, gate_elem, ptab_ld, window, pool > 0 ? __builtin_ctz(pool) : -1, kld, vld, chunked,
                  chunked || window <= 0 ? 0 : keep_first, rel_n, out_ld, hw, scale, cap, out_scale};
  const dim3 grid(H / hw, rows * hw / (16 * rw) + n);        // heads, then ceil(len / QT) of every sequence, or a few more
  const bool same = kp == vp && kld == vld;
#define F32_LAUNCH(DD, DDV, S, RW, KS) \
  hipLaunchKernelGGL((attn_f32_kernel<DD, DDV, S, RW, KS>), grid, dim3(64 * RW * KS), 0, st, a)
#define F32_KS(DD, DDV, S)                                              \
  do {                                                                  \
    if (rw == 2 && ks == 2) F32_LAUNCH(DD, DDV, S, 2, 2);               \
    else if (rw == 2 && ks == 4) {                                      \
      if constexpr (DD <= 64 && DDV <= 64) F32_LAUNCH(DD, DDV, S, 2, 4); \
      else return -2;                                                   \
    } else if (rw == 4 && ks == 2) F32_LAUNCH(DD, DDV, S, 4, 2);        \
    else return -2;                                                     \
    return (int)hipGetLastError();                                      \
  } while (0)
#define F32_BOTH(DD)                  \
  if (D == DD && Dv == DD) {          \
    if (same) F32_KS(DD, DD, true);   \
    else F32_KS(DD, DD, false);       \
  }
  F32_BOTH(32)
  F32_BOTH(64)
  F32_BOTH(96)
  F32_BOTH(128)
  if (same && D == 160 && Dv == 128) F32_KS(160, 128, true);
  if (!same && D == 64 && Dv == 128) F32_KS(64, 128, false);
  if (!same && D == 128 && Dv == 64) F32_KS(128, 64, false);
#undef F32_BOTH
#undef F32_KS
#undef F32_LAUNCH
  return -2;
}

}  // extern "C"
