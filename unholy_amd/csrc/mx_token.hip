// The routed-expert FFN of a step of very few tokens (uh_mx_moe_forward) in two launches. At one token the weights of
// its picks are 80 MB, 10 us of HBM, and the general path (dispatch, w1 / w3 GEMV, w2 GEMV, combine) took 29.5 us: 5 +
// 4.5 us of launches with next to nothing in them, and GEMVs whose workgroups (64 or 128 columns of one expert) do not
// divide over 256 CUs. Here
// - moe_token_up_kernel routes each token in every workgroup (a wave per token, ~1 us, instead of a launch), quantizes the
//   token rows, and streams w1 / w3: a unit is a 16-column tile of one pick, a workgroup three units with K split over
//   four waves each. One token with 6 picks of I = 2048: 768 units, 256 workgroups of 12 waves, one per CU;
// - moe_token_down_kernel streams w2 and combines: a workgroup is 16 output columns of one token, two waves per pick;
//   the picks' bf16 sums are added in LDS in ascending expert order, as moe_combine does. 256 workgroups at D = 4096.
// Whole forward, us, general path / this: E = 256, D = 4096, I = 2048: T = 1 29.8 / 23.8, 2 41.9 / 41.0, 3 58.4 /
// 58.7, 4 66.9 / 74.3; E = 32: T = 1 29.8 / 23.4, 2 40.9 / 39.7, 3 46.4 / 55.3; E = 64, D = 2048, I = 1024: T = 1 21.4
// / 14.0, 2 22.5 / 15.8, 3 23.9 / 24.7. So up to two tokens, and only while the first launch is one round of
// workgroups: in a second one most of the chip waits for a few, and full or not it is the general path's measure at
// best (T, picks K, us, general / this; E = 256, D = 4096, I = 2048: T = 1 K = 6 (256 workgroups) 30.7 / 25.0, 7 (299)
// 32.3 / 35.6, 8 34.5 / 37.3; T = 2 K = 3 30.1 / 24.4, 4 33.4 / 34.6, 6 (512) 41.9 / 41.4, 7 45.6 / 56.1; E = 16, D =
// 7168: T = 2 K = 3 42.2 / 32.7, 6 55.1 / 61.2; E = 8, I = 6144: T = 1 K = 2 35.8 / 24.6, 5 48.0 / 54.1; E = 64, D =
// 2048, I = 1024: T = 2 K = 6 22.7 / 17.7, 7 23.7 / 25.4).
// The arithmetic is the GEMV's (exact dequantization, one bf16 MFMA per 32-input block), a K part's blocks in input
// order, the parts added in order. A pick streams its expert's weights whether or not another token picked it too.
#include <algorithm>
#include <stdexcept>

#include "common.hpp"
#include "numerics.hpp"
#include "mx_internal.hpp"
#include "route.hpp"

namespace unholy::kernels {

using namespace uh;

namespace {

// 128-input steps in flight per wave; a dword of scales covers 4 (8 measured slower: w1 / w3 15.6 -> 15.8 us, w2 8.6
// -> 10.1, the unrolled steps run once from a cold instruction cache).
constexpr int TK_PF = 4, TK_SW = TK_PF / 4;

// Steps [sb, se) of one 16-column tile nt of NP matrices against the bf16 row at ap (lane (nl, g): inputs 8 g .. + 7 of
// block 0; lanes nl > 0 are given a zero row): acc[p] += the block sums in input order. Weights and scales are read as in
// mx_gemv_kernel (a half-wave reads a contiguous 512-byte chunk, a lane one dword of scales per 4 steps).
// between() runs after the first loads are issued.
template <int NP, class Between>
__device__ __forceinline__ void token_stream(const uint8_t* const (&wp)[NP], const uint8_t* const (&sp)[NP], int ntn,
                                             int nt, int sb, int se, int KS, const uint16_t* ap, v4f (&acc)[NP],
                                             const Between& between) {
  const int lane = threadIdx.x & 63, nl = lane & 15, g = lane >> 4;
  const uint32_t cofs = uint32_t(((g >> 1) * ntn + nt) * 512 + nl * 32 + (g & 1) * 16), cstep = uint32_t(2 * ntn * 512);
  v4i bq[TK_PF][NP];
  uint32_t sq[TK_SW][NP], sn[TK_SW][NP];
  const auto load_step = [&](int s, int slot) {
#pragma unroll
    for (int p = 0; p < NP; ++p)
      bq[slot][p] =
          __builtin_nontemporal_load(reinterpret_cast<gptr<v4i>>(as_global(wp[p]) + (cofs + uint32_t(s) * cstep)));
  };
  const auto load_scales = [&](int s0, uint32_t (&dst)[TK_SW][NP]) {
#pragma unroll
    for (int j = 0; j < TK_SW; ++j) {
      const uint32_t slab = uint32_t(min(2 * (s0 + 4 * j) + (lane >> 3), 2 * KS - 1));
      const uint32_t so = (slab * uint32_t(ntn) + uint32_t(nt)) * 32u + uint32_t(lane & 7) * 4u;
#pragma unroll
      for (int p = 0; p < NP; ++p) dst[j][p] = *reinterpret_cast<gptr<uint32_t>>(as_global(sp[p]) + so);
    }
  };
  const auto step = [&](int s, int i) {
    bf16x8 af[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) af[t] = *reinterpret_cast<const bf16x8*>(ap + s * 128 + 32 * t);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      uint32_t sw[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        sw[j] = uint32_t(__builtin_amdgcn_ds_bpermute(((2 * (i % 4) + j) * 8 + (nl >> 1)) * 4, int(sq[i / 4][p]))) >>
                (16 * (nl & 1));
      const auto r02 = __builtin_amdgcn_permlane32_swap(uint32_t(bq[i][p][0]), uint32_t(bq[i][p][2]), false, false);
      const auto r13 = __builtin_amdgcn_permlane32_swap(uint32_t(bq[i][p][1]), uint32_t(bq[i][p][3]), false, false);
      const auto r01 = __builtin_amdgcn_permlane16_swap(r02[0], r13[0], false, false);
      const auto r23 = __builtin_amdgcn_permlane16_swap(r02[1], r13[1], false, false);
      const uint32_t wd[4] = {r01[0], r01[1], r23[0], r23[1]};
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float sc = __uint_as_float(((sw[t >> 1] >> (8 * (t & 1))) & 0xffu) << 23);
        acc[p] = mfma_bf16(af[t], fp4x8_to_bf16(wd[t], sc), acc[p]);
      }
    }
  };
  const bool any = sb < se;  // uniform
  if (any) {
    load_scales(sb, sq);
#pragma unroll
    for (int i = 0; i < TK_PF; ++i) load_step(min(sb + i, se - 1), i);
  }
  between();
  if (!any) return;
  int s0 = sb;
  for (; s0 + TK_PF < se; s0 += TK_PF) {
#pragma unroll
    for (int i = 0; i < TK_PF; ++i) {
      step(s0 + i, i);
      load_step(min(s0 + i + TK_PF, se - 1), i);
      if (i == 0) load_scales(s0 + TK_PF, sn);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < TK_SW; ++j)
#pragma unroll
      for (int p = 0; p < NP; ++p) sq[j][p] = sn[j][p];
  }
#pragma unroll
  for (int i = 0; i < TK_PF; ++i) {
    if (s0 + i < se) step(s0 + i, i);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// 8 bf16 values (16 consecutive lanes one 128-block) through act_quant_fp8 and back, exact.
__device__ __forceinline__ bf16x8 fake_quant8(const uint4 raw) {
  const uint32_t rw[4] = {raw.x, raw.y, raw.z, raw.w};
  float v[8], am = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __uint_as_float(rw[i] << 16);
    v[2 * i + 1] = __uint_as_float(rw[i] & 0xffff0000u);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) am = fmaxf(am, fabsf(v[i]));
  const Fp8Block b = fp8_block_scale(row16_max(am));
  uint32_t lo, hi;
  fp8_codes8(v, b, lo, hi);
  return fp8x8_to_bf16(lo, hi, b.sc);
}

constexpr int TU_UNITS = 3, TU_PARTS = 4, TU_WAVES = TU_UNITS * TU_PARTS;

template <int NV>
__global__ __launch_bounds__(64 * TU_WAVES) void moe_token_up_kernel(MoeTokenArgs a) {
  extern __shared__ __align__(16) uint8_t smem[];  // bf16 rows [T + 1][D + 8], the last one zero
  __shared__ int spick[kTokenMaxT * 8];
  __shared__ float swt[kTokenMaxT * 8];
  __shared__ float red[TU_UNITS][TU_PARTS][2][16];
  const int T = a.T, K = a.K, D = a.D, I = a.I, ldx = D + 8, ntn = I / 16, KS = D / 128;
  const int tid = threadIdx.x, lane = tid & 63, nl = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint16_t* const rows = reinterpret_cast<uint16_t*>(smem);
  if (wave < T) {  // route token `wave`; its picks and weights in ascending expert order into LDS
    const bool first = blockIdx.x == 0;
    route_wave<2, NV>(a.logits + size_t(wave) * a.E, nullptr, nullptr, a.E, K, 1.0f,
                      first && a.sel ? a.sel + wave * K : nullptr, a.wt + wave * K, spick + wave * 8, swt + wave * 8);
    const int pick = lane < K ? spick[wave * 8 + lane] : 0;
    const float wk = lane < K ? swt[wave * 8 + lane] : 0.0f;
    int r = 0;
    for (int q = 0; q < K; ++q) {
      const int o = __builtin_amdgcn_readlane(pick, q);
      r += o < pick || (o == pick && q < lane);
    }
    if (lane < K) {
      spick[wave * 8 + r] = pick;
      swt[wave * 8 + r] = wk;
      if (first) a.row_expert[wave * K + r] = pick;
    }
  } else {
    const int t0 = tid - 64 * T, nt = 64 * (TU_WAVES - T), per = D / 8;
    for (int base = 0; base < T * per; base += nt) {  // uniform bound, per % 16 == 0: 16-lane groups stay whole
      const int i = min(base + t0, T * per - 1), m = i / per, c = (i % per) * 8;
      const bf16x8 v = fake_quant8(*reinterpret_cast<const uint4*>(a.x + size_t(m) * D + c));
      if (base + t0 < T * per) *reinterpret_cast<bf16x8*>(rows + m * ldx + c) = v;
    }
    for (int i = t0 * 8; i < ldx; i += nt * 8) *reinterpret_cast<uint4*>(rows + T * ldx + i) = uint4{0u, 0u, 0u, 0u};
  }
  __syncthreads();
  const int u = wave / TU_PARTS, part = wave % TU_PARTS, unit = blockIdx.x * TU_UNITS + u;
  const bool live = unit < T * K * ntn;  // uniform per wave
  const int p = live ? unit / ntn : 0, nt = unit % ntn, t = p / K, j = p % K, e = spick[t * 8 + j];
  v4f acc[2] = {v4f{0.0f, 0.0f, 0.0f, 0.0f}, v4f{0.0f, 0.0f, 0.0f, 0.0f}};
  const int per = (KS + TU_PARTS - 1) / TU_PARTS, sb = min(KS, part * per), se = min(KS, sb + per);
  if (live) {
    const uint8_t* const wp[2] = {a.tab[e], a.tab[2 * a.E + e]};
    const uint8_t* const sp[2] = {a.tab[a.E + e], a.tab[3 * a.E + e]};
    if (wp[0] && wp[1] && sp[0] && sp[1])
      token_stream<2>(wp, sp, ntn, nt, sb, se, KS, rows + (nl == 0 ? t : T) * ldx + g * 8, acc, [] {});
  }
  if (g == 0) {  // row 0 of the tile: lanes 0..15
    red[u][part][0][nl] = acc[0][0];
    red[u][part][1][nl] = acc[1][0];
  }
  __syncthreads();
  if (part == 0 && lane < 16 && live) {
    float gs = red[u][0][0][nl], us = red[u][0][1][nl];
#pragma unroll
    for (int q = 1; q < TU_PARTS; ++q) gs += red[u][q][0][nl], us += red[u][q][1][nl];
    a.h[size_t(p) * I + nt * 16 + nl] =
        f32_to_bf16(swiglu_value(round_bf16(gs), round_bf16(us), swt[t * 8 + j], true, a.limit));
  }
}

constexpr int TD_PARTS = 2;

// TD_PARTS K waves (K picks): wave = pick * TD_PARTS + part; blockIdx.x = 16 output columns, blockIdx.y = token.
__global__ __launch_bounds__(1024) void moe_token_down_kernel(MoeTokenArgs a) {
  extern __shared__ __align__(16) uint8_t smem[];  // bf16 rows [K + 1][I + 8], the last one zero
  __shared__ float red[8][TD_PARTS][16];
  const int K = a.K, D = a.D, I = a.I, ldh = I + 8, ntn = D / 16, KS = I / 128, tk = blockIdx.y, nt = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, nl = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), j = wave / TD_PARTS, part = wave % TD_PARTS;
  uint16_t* const rows = reinterpret_cast<uint16_t*>(smem);
  const int e = a.row_expert[tk * K + j];
  const uint8_t* const wp[1] = {a.tab[4 * a.E + e]};
  const uint8_t* const sp[1] = {a.tab[5 * a.E + e]};
  const int per_part = (KS + TD_PARTS - 1) / TD_PARTS, sb = min(KS, part * per_part);
  // (an expert that is not here: nothing, its rows are undefined)
  const int se = wp[0] && sp[0] ? min(KS, sb + per_part) : sb;
  v4f acc[1] = {v4f{0.0f, 0.0f, 0.0f, 0.0f}};
  token_stream<1>(wp, sp, ntn, nt, sb, se, KS, rows + (nl == 0 ? j : K) * ldh + g * 8, acc, [&] {
    const int nthr = blockDim.x, per = I / 8;
    for (int base = 0; base < K * per; base += nthr) {
      const int i = min(base + tid, K * per - 1), m = i / per, c = (i % per) * 8;
      const bf16x8 v = fake_quant8(*reinterpret_cast<const uint4*>(a.h + (size_t(tk) * K + m) * I + c));
      if (base + tid < K * per) *reinterpret_cast<bf16x8*>(rows + m * ldh + c) = v;
    }
    for (int i = tid * 8; i < ldh; i += nthr * 8) *reinterpret_cast<uint4*>(rows + K * ldh + i) = uint4{0u, 0u, 0u, 0u};
    __syncthreads();
  });
  if (g == 0) red[j][part][nl] = acc[0][0];
  __syncthreads();
  if (tid < 16) {
    float s = 0.0f;
    for (int q = 0; q < K; ++q) {
      float v = red[q][0][tid];
#pragma unroll
      for (int w = 1; w < TD_PARTS; ++w) v += red[q][w][tid];
      s += round_bf16(v);
    }
    a.out[size_t(tk) * D + nt * 16 + tid] = f32_to_bf16(s + 0.0f);
  }
}

size_t up_lds(const MoeTokenArgs& a) { return size_t(a.T + 1) * (a.D + 8) * 2; }
size_t down_lds(const MoeTokenArgs& a) { return size_t(a.K + 1) * (a.I + 8) * 2; }
}  // namespace

bool moe_token_fits(const MoeTokenArgs& a) {
  return a.T >= 1 && a.T <= kTokenMaxT && a.K >= 1 && a.K <= 8 && a.K <= a.E && a.E <= 1024 && a.D % 128 == 0 &&
         a.I % 128 == 0 && size_t(a.T) * a.K * (a.I / 16) <= size_t(256) * TU_UNITS &&  // one round of workgroups
         up_lds(a) <= 96 * 1024 && down_lds(a) <= 96 * 1024;
}
void launch_moe_token_up(const MoeTokenArgs& a, hipStream_t st) {
  if (!moe_token_fits(a)) throw std::runtime_error("moe token: shape");
  auto* kern = a.E <= 256 ? &moe_token_up_kernel<4> : &moe_token_up_kernel<16>;
  const size_t lds = up_lds(a);
  if (lds > 48 * 1024)
    UH_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 int(lds)));
  kern<<<cdiv(size_t(a.T) * a.K * (a.I / 16), TU_UNITS), 64 * TU_WAVES, lds, st>>>(a);
  UH_CHECK_LAUNCH();
}
void launch_moe_token_down(const MoeTokenArgs& a, hipStream_t st) {
  auto* kern = &moe_token_down_kernel;
  const size_t lds = down_lds(a);
  if (lds > 48 * 1024)
    UH_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 int(lds)));
  kern<<<dim3(unsigned(a.D / 16), unsigned(a.T)), unsigned(64 * TD_PARTS * a.K), lds, st>>>(a);
  UH_CHECK_LAUNCH();
}

}  // namespace unholy::kernels
