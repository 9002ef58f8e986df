// Launch descriptors shared between the MXFP4 kernel files (not part of the public interface).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "unholy/kernels/exl3_moe.hpp"

namespace unholy::kernels {

// One grouped GEMV / GEMM launch: activations as e4m3 codes + e8m0 scales per 128 (aq, as) or fake-quantized
// bf16 (xa); one or two projections (index 1 null: one); optional SwiGLU epilogue (hh and/or hq + hs).
struct MxGemvArgs {
  const uint8_t* aq;
  const uint8_t* as;
  const uint16_t* xa;
  const int32_t* x_rows;  // activation mode 2: pair row r reads token row x_rows[r] of x (xa, row stride ldx)
  int ldx;
  int K, N, ldo;
  const Exl3Tile* tiles;
  int ntiles;  // tiles the grid covers (set by the launcher; the grid may be padded past it)
  const int* ntiles_dev;
  const uint8_t* const* w_tab[2];
  const uint8_t* const* s_tab[2];
  uint16_t* out[2];
  float* out32;  // non-null: projection 0 written as fp32 (before bf16 rounding) instead
  int rows_cap;
  const float* gw;
  const int32_t* grow_expert;
  const uint8_t* const* gs_tab;
  uint16_t* hh;
  uint8_t* hq;
  uint8_t* hs;
  uint16_t* hraw;  // SwiGLU rows as bf16, not requantized (MxGlu::h)
  float limit;
  // > 0: one matrix, two column streams per wave: projection 1 is projection 0's matrix from 16-column tile `split`
  // on (codes, scales and outputs offset by split tiles); the grid covers split tiles.
  int split;
  int tiles_hint = 0;     // GEMV: the tiles expected to be live, of ntiles (0: all; a choice of kernel, not a bound)
  bool few_rows = false;  // GEMM on bf16 rows: most tiles hold at most 64 rows (a choice of kernel, not a bound)
};

// amode: 0 e4m3 codes + scales, 1 fake-quantized bf16 rows, 2 raw bf16 token rows (act_quant in the kernel).
void launch_mx_gemv(const MxGemvArgs& a, int ntiles, int amode, hipStream_t st);
// Exhaustive check of the hardware e4m3 encode against the software one on [-448, 448]; returns the mismatches
// (*total: values compared).
unsigned long long fp8_check_encode(unsigned long long* total);
// Exhaustive check of the hardware bf16 rounding against f32_to_bf16 over all fp32 bit patterns; returns the
// mismatches at non-NaN inputs (*nan_bad: at NaN inputs).
unsigned long long bf16_check_encode(unsigned long long* nan_bad);
struct MoePlan;
// moe_count + moe_plan + moe_scatter of a step whose experts are all resident, in one launch; the tiles longest first.
void launch_moe_dispatch_all(const int32_t* sel, const float* wt, int T, int K, int E, MoePlan* plan, Exl3Tile* tiles,
                             int max_tiles, int tile_rows, int32_t* eidx, float* ewt, int32_t* row_expert,
                             int32_t* pidx, hipStream_t st);
// route_softmax and mx_xform_in of the token rows x [T, D] (fake-quantized into xa) in one launch.
void launch_route_xform(const float* logits, int32_t* sel, float* weights, int T, int E, int K, const uint16_t* x,
                        uint16_t* xa, int D, hipStream_t st);
// remote_combine over rows of stride ld (the grid strides over the device-side token count; max_tokens only sizes it).
void launch_remote_combine(const uint16_t* pair_out, int ld, const int32_t* u2p, const MoePlan* plan, uint16_t* dst,
                           int K, int dim, int max_tokens, hipStream_t st);
void launch_mx_gemm(const MxGemvArgs& a, int ntiles, int amode, hipStream_t st);
// mx_grouped_gemm_rows with MxGemvArgs::few_rows; the pipelined GEMMs (UH_GEMM_PIPE) are on.
struct MxGlu;
void launch_mx_gemm_rows(const uint16_t* xa, const int32_t* x_rows, int K, const Exl3Tile* tiles, int ntiles,
                         const uint8_t* const* w_tab, const uint8_t* const* s_tab, uint16_t* out, int ldo, int N,
                         hipStream_t st, const int* ntiles_dev, const uint8_t* const* w_tab2,
                         const uint8_t* const* s_tab2, uint16_t* out2, const MxGlu& glu, bool few_rows);
bool mx_gemm_pipe_on();
// mx_grouped_gemv_x with MxGemvArgs::tiles_hint.
void launch_mx_gemv_x(const uint16_t* x, int ldx, const int32_t* x_rows, int K, const Exl3Tile* tiles, int ntiles,
                      const uint8_t* const* w_tab, const uint8_t* const* s_tab, uint16_t* out, int ldo, int N,
                      hipStream_t st, const int* ntiles_dev, const uint8_t* const* w_tab2,
                      const uint8_t* const* s_tab2, uint16_t* out2, int max_rows, const MxGlu& glu, int tiles_hint);
void launch_mx_transform(int mode, const uint16_t* x, int ldx, const int32_t* x_rows, const uint16_t* u,
                         const float* w, float limit, const int32_t* row_expert, const uint8_t* const* s_tab,
                         uint16_t* out, uint8_t* q, uint8_t* qs, int K, int P, hipStream_t st);

// h = bf16(SwiGLU(g, u)) (no routing weight) of M rows x I, act_quant per 128 into q / qs (and / or fake-quantized
// bf16 into hh): the second half of gemv_w8a8_glu.
void launch_swiglu_quant(const uint16_t* g, int ldg, const uint16_t* u, int ldu, int M, int I, float limit,
                         uint16_t* hh, uint8_t* q, uint8_t* qs, hipStream_t st);

// The forward of a step of at most kTokenMaxT tokens in two launches (mx_token.hip): routing + w1 / w3 + SwiGLU into h
// [T K, I] (each token's picks in ascending expert order, also written to row_expert [T K]), then w2 + combine. sel
// (may be null, then wt is not written) / wt: the routing. tab: the forward's 6 E pointers.
constexpr int kTokenMaxT = 2;
struct MoeTokenArgs {
  const uint16_t* x;
  const float* logits;
  int T, K, E, D, I;
  const uint8_t* const* tab;
  float limit;
  int32_t* sel;
  float* wt;
  int32_t* row_expert;
  uint16_t* h;
  uint16_t* out;
};
bool moe_token_fits(const MoeTokenArgs& a);
// About the live tiles of a step: the distinct experts that T K uniform picks hit, each with its rows in tiles of tile_rows.
inline double moe_experts_hit(int T, int K, int E) { return E * (1.0 - std::pow(1.0 - double(K) / E, T)); }
inline int moe_live_tiles(int T, int K, int E, int tile_rows) {
  const double hit = moe_experts_hit(T, K, E), rows = double(T) * K / hit;
  const double per = std::min(std::max(1.0, rows / tile_rows + 0.5), double((T + tile_rows - 1) / tile_rows));
  return std::max(1, int(std::lround(hit * per)));
}
// Up to 64 tokens: whether the GEMM on bf16 rows beats the GEMV. Its workgroups (a tile x 128 columns of w1 / w3)
// stream the weights no faster than their chain of stages, so it needs more than one a CU, or weights that take the
// GEMV longer: the GEMV reads an expert once per 16 rows. us per forward, GEMV / GEMM: E = 256, D = 4096, I = 2048, 6
// picks (workgroups past 280): T = 8 111 / 114, 9 119 / 113, 16 173 / 162, 64 353 / 337; E = 64, D = 2048, I = 1024, 4
// picks: T = 9 (226) 32.0 / 35.0, 12 (277) 34.7 / 35.5, 16 (330) 40.9 / 38.1; E = 8, D = 4096, I = 2048 (128), 4
// picks: T = 9 (107 MB) 42.6 / 51.1, 32 (161) 56.0 / 65.5, 64 (268) 87.3 / 78.2; 8 picks, T = 48 (375) 97.3 / 75.2; E
// = 16, D = 7168, 4 picks, T = 12 (364) 100 / 77. Over 517 calls timed with both the choice is 0.1% slower than the
// best on average, 8% at worst.
inline bool moe_gemm_pays(int T, int K, int E, int D, int I) {
  const double mb = 3.0 * D * I * (17.0 / 32.0) * 1e-6;  // an expert's weights
  return T > 8 && (moe_experts_hit(T, K, E) * (I / 128) >= 280.0 || moe_live_tiles(T, K, E, 16) * mb >= 260.0);
}
// Whether a single-projection GEMV of ntiles x column_tiles tiles splits K over a workgroup's waves.
bool gemv_splits_k(size_t ntiles, size_t column_tiles, int K);
// The workgroup shape of the forward's w1 / w3 GEMV: 4 waves, or 8 (launch_gemv_t).
bool gemv_four_waves(size_t workgroups8, int rows, int K);
void launch_moe_token_up(const MoeTokenArgs& a, hipStream_t st);
void launch_moe_token_down(const MoeTokenArgs& a, hipStream_t st);

}  // namespace unholy::kernels
