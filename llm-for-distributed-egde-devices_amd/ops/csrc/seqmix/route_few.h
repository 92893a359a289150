// The choice of one token's experts by one wave, from scores that its workgroup has left in LDS (route_few_kernel in postnorm.hip,
// ln_residual_taps_route_kernel in residual_next.hip).
#pragma once
#include "seqmix/seqmix_common.h"

namespace {

constexpr int RF_WAVES = 16, RF_SCORES = 48;
struct RouteFew {
  const float *router, *bias;                                // bias: GROUPED the correction of the choice
  int W, E, gate, groups, keep, top, sigm;
  float scale;
  int* idx;
  float *wts, *gate_w;
};

// what the whole wave holds most of among lanes with v > floor: its lowest lane, -1 for none
__device__ __forceinline__ int best_lane(float v, float floor, float& best) {
  const bool in = v > floor;
  float m = in ? v : -INFINITY;
  m = fmaxf(m, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, m), 0xB1, 0xF, 0xF, false)));
  m = fmaxf(m, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, m), 0x4E, 0xF, 0xF, false)));
  m = fmaxf(m, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, m), 0x124, 0xF, 0xF, false)));
  m = fmaxf(m, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, m), 0x128, 0xF, 0xF, false)));
  auto row = [&](int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), l)); };
  best = fmaxf(fmaxf(row(0), row(16)), fmaxf(row(32), row(48)));
  return __ffsll((unsigned long long)__ballot(in && v == best)) - 1;
}

// z_s: E scores (and the gate's); c_s, g_s: 64 numbers of LDS each where GROUPED.  One expert a lane
template <bool GROUPED>
__device__ __forceinline__ void route_choose(const RouteFew& a, const float* z_s, float* c_s, float* g_s, size_t t) {
  const int lane = threadIdx.x & 63;
  const int E = a.E, top = a.top;
  const bool live = lane < E;
  const float z = live ? z_s[lane] : -INFINITY;
  auto softmax = [&]() {
    const float mx = wave_max(z), ex = live ? expf(z - mx) : 0.f;
    return ex / wave_sum(ex);
  };
  float tot = 0.f, my_w = 0.f;
  int my_i = 0;                                              // lane k keeps the k-th choice
  if constexpr (GROUPED) {
    const float s = softmax();
    float c = live ? s + (a.bias ? a.bias[lane] : 0.f) : -INFINITY;
    if (a.groups > 1) {
      const int size = E / a.groups, g = min(lane / size, a.groups - 1);
      c_s[lane] = c;
      __builtin_amdgcn_wave_barrier();                       // (one wave: its LDS accesses keep their order)
      float b = -INFINITY;
      for (int e = g * size; e < (g + 1) * size; ++e) b = fmaxf(b, c_s[e]);
      g_s[g] = b;
      __builtin_amdgcn_wave_barrier();
      int better = 0;
      for (int o = 0; o < a.groups; ++o) better += g_s[o] > b || (g_s[o] == b && o < g);
      if (better >= a.keep) c = -INFINITY;
    }
    for (int k = 0; k < top; ++k) {
      float best;
      int bi = best_lane(c, -INFINITY, best);
      if (bi < 0) bi = k;                                    // scores that compare with nothing (NaN): keep the ids in range
      const float w = __shfl(s, bi, 64);
      if (lane == k) { my_w = w; my_i = bi; }
      tot += w;
      if (lane == bi) c = -INFINITY;
    }
    if (a.gate && lane == 0) a.gate_w[t] = sigmoidf_(z_s[E]);
  } else {
    float v = z;
    if (!a.sigm) {                                           // (every lane takes part in its sums)
      v = softmax();
      if (!live) v = -2.f;
    }
    const float floor = a.sigm ? -INFINITY : -1.f, gone = a.sigm ? -INFINITY : -2.f;
    for (int k = 0; k < top; ++k) {
      float best;
      int bi = best_lane(v, floor, best);
      if (bi < 0) {
        bi = k;
        best = 0.f;
      }
      if (lane == k) { my_w = best; my_i = bi; }
      if (lane == bi) v = gone;
      tot += best;
    }
  }
  float soft = 0.f;
  if (!GROUPED && a.sigm == 2) {
    const float ex = lane < top ? expf(my_w - __shfl(my_w, 0, 64)) : 0.f;
    soft = ex / wave_sum(ex);
  }
  if (lane < top) {
    a.idx[t * top + lane] = my_i;
    a.wts[t * top + lane] = (!GROUPED && a.sigm == 2) ? soft * a.scale : (!GROUPED && a.sigm) ? sigmoidf_(my_w) * a.scale
                                                                                             : my_w / (tot + 1e-20f) * a.scale;
  }
}

}  // namespace
