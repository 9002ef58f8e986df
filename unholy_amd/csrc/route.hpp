// Routing of one token by one wave (the routers' kernels and those that route in their own launch).
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "numerics.hpp"

namespace unholy::kernels {

using namespace uh;

// ---- routers: a wave per token ---------------------------------------------------------------------------------------
__device__ __forceinline__ float ds_score(float x) { return sqrtf(x > 20.0f ? x : log1pf(expf(x))); }
__device__ __forceinline__ float sigmoid(float x) {
#pragma clang fp contract(off)
  return 1.0f / (1.0f + uh::exp_f32(-x));
}
__device__ __forceinline__ float lane_f32(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// One token's routing by one wave (MODE 0: DSV4 sqrt-softplus + bias or the hash row, 1: GLM sigmoid + bias, 2:
// softmax top-K; E <= 64 * NV). Lane l holds the keys of experts l + 64 i. Top-K with ties to the lower index, in
// selection order: per round the largest key (a DPP max of the order-preserving bits), then the lowest expert holding
// it (a DPP min); the pick's logit comes from the lane that holds it (readlane, no memory access). The picks are kept
// spread over lanes (lane k holds pick k) and every loop over them is a rolled loop over K: this code runs once per
// launch from a cold instruction cache, so its size sets its time more than its instruction count does.
// Weights (lane 0's order of operations in the reference's routers): GLM reports its picks in ascending id, the
// weights follow that order; mode 0 score / sum * scale, 1 sigmoid / (sum + 1e-20) * scale, 2 exp(l - l_first) / sum,
// the sum taken pick by pick from zero. Lanes k < K write pick k to sel_t / wt_t and to ssel / swt,
// where set.
// pre (may be null): the lane's logits already loaded (pre[i] = lr[lane + 64 i], 0 past E).
template <int MODE, int NV>
__device__ __forceinline__ void route_wave(const float* lr, const float* bias, const int32_t* hash_row, int E, int K,
                                           float route_scale, int32_t* sel_t, float* wt_t, int* ssel, float* swt,
                                           const float* pre = nullptr) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  int pick = 0;
  float lgt = 0.0f;
  if (MODE == 0 && hash_row) {
    if (lane < K) {
      pick = hash_row[lane];
      lgt = lr[pick];
    }
  } else {
    float key[NV], raw[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int e = lane + 64 * i;
      raw[i] = pre ? pre[i] : e < E ? lr[e] : 0.0f;
      float v = -INFINITY;
      if (e < E) {
        if constexpr (MODE == 2) v = raw[i];
        else if constexpr (MODE == 1) v = sigmoid(raw[i]) + bias[e];
        else v = ds_score(raw[i]) + bias[e];
      }
      key[i] = v;
    }
    for (int k = 0; k < K; ++k) {
      float bv = -INFINITY;
      uint32_t bi = 0xffffffffu;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int e = lane + 64 * i;
        if (e < E && (key[i] > bv || bi == 0xffffffffu)) bv = key[i], bi = uint32_t(e);
      }
      const uint32_t ob = bi == 0xffffffffu ? 0u : orderable(bv);
      const uint32_t m = wave_reduce_u32<true>(ob);
      // The lowest expert holding the largest key: when one lane holds it (the usual case) that lane's candidate,
      // else the DPP min over the lanes that do.
      const uint64_t holders = __ballot(ob == m);
      const uint32_t idx = __popcll(holders) == 1
                               ? uint32_t(__builtin_amdgcn_readlane(int(bi), int(__builtin_ctzll(holders))))
                               : wave_reduce_u32<false>(ob == m ? bi : 0xffffffffu);
      const int slot = int(idx >> 6), owner = int(idx & 63);
      float v = 0.0f;
#pragma unroll
      for (int i = 0; i < NV; ++i)
        if (slot == i) {
          v = raw[i];
          if (lane == owner) key[i] = -INFINITY;
        }
      const float l = lane_f32(v, owner);
      if (lane == k) pick = int(idx), lgt = l;
    }
  }
  if constexpr (MODE == 1) {  // ascending id: lane k's pick moves to lane (number of smaller picks)
    int r = lane;
    if (lane < K) {
      r = 0;
      for (int q = 0; q < K; ++q) r += __builtin_amdgcn_readlane(pick, q) < pick;
    }
    pick = __builtin_amdgcn_ds_permute(r * 4, pick);
    lgt = __int_as_float(__builtin_amdgcn_ds_permute(r * 4, __float_as_int(lgt)));
  }
  const float w = MODE == 2 ? uh::exp_f32(lgt - lane_f32(lgt, 0)) : MODE == 1 ? sigmoid(lgt) : ds_score(lgt);
  float sum = 0.0f;
  for (int k = 0; k < K; ++k) sum += lane_f32(w, k);
  if (lane < K) {
    const float wk = MODE == 2 ? w / sum : MODE == 1 ? w / (sum + 1e-20f) * route_scale : (w / sum) * route_scale;
    if (sel_t) {
      sel_t[lane] = pick;
      wt_t[lane] = wk;
    }
    if (ssel) {
      ssel[lane] = pick;
      swt[lane] = wk;
    }
  }
}

}  // namespace unholy::kernels
