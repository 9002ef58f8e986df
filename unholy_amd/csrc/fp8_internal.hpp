// Launch descriptor of the dense fp8 GEMM kernels (not part of the public interface).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>

namespace unholy::kernels {

// C[M, N] (bf16, ldc) = A[M, K] (e4m3) x W[N, K]^T (e4m3), per-128 scales: e8m0 (sa8 [M, K/128], sw8
// [ceil(N/128), K/128]) or fp32 (sa32, sw32, same shapes).
struct Fp8GemmArgs {
  const uint8_t* a;
  const uint8_t* sa8;
  const float* sa32;
  const uint8_t* w;
  const uint8_t* sw8;
  const float* sw32;
  uint16_t* c;
  int ldc, M, N, K;
  int rows_cap;
  const uint16_t* xa = nullptr;  // raw bf16 activations [M, ldx] quantized in the GEMV (fp32 scales, M <= 16)
  int ldx = 0;
};

// Up to three column ranges on one input (gemv_w8a8_parts): range i has its own weights, e8m0 scales, output, ldc
// and width; t0[i] is its first 16-column tile in the grid (t0[n] = total tiles).
struct Fp8Parts {
  int n;
  const uint8_t* w[3];
  const uint8_t* sw[3];
  uint16_t* c[3];
  int ldc[3], N[3], t0[4];
};

void launch_fp8_skinny(const Fp8GemmArgs& a, hipStream_t st);
// M <= 64: one workgroup per 16-column tile, K split over its 8 waves (bandwidth-shaped).
void launch_fp8_gemv(const Fp8GemmArgs& a, hipStream_t st, const Fp8Parts* parts = nullptr);
// The LDS-ring MFMA GEMM (N % 128, K % 128, ldc % 8; fp8_tiled_fits says whether a shape qualifies).
bool fp8_tiled_fits(const Fp8GemmArgs& a);
void launch_fp8_tiled(const Fp8GemmArgs& a, hipStream_t st);
// A workgroup per output tile of up to 96 x 64, K split over its waves (K <= 8192), and its estimated time; the column
// ranges of gemv_w8a8_parts (M <= 32), and bf16 rows quantized in the kernel (fp32 scales, M <= 16).
bool fp8_kpart_fits(const Fp8GemmArgs& a);
double fp8_kpart_us(const Fp8GemmArgs& a);
std::pair<int, int> fp8_kpart_form(const Fp8GemmArgs& a);  // the tile it would use, in 16-row and 16-column blocks
void launch_fp8_kpart(const Fp8GemmArgs& a, hipStream_t st);
bool fp8_kpart_parts_fits(const Fp8GemmArgs& a, const Fp8Parts& pp);
void launch_fp8_kpart_parts(const Fp8GemmArgs& a, const Fp8Parts& pp, hipStream_t st);
void launch_fp8_kpart_xq(const Fp8GemmArgs& a, hipStream_t st);
double fp8_tiled_us(const Fp8GemmArgs& a);
// The same for the grouped projection (R % 16, K <= 65536).
bool grouped_kpart_fits(int M, int G, int R, int K);
double grouped_kpart_us(int M, int G, int R, int K);
std::pair<int, int> grouped_kpart_form(int M, int G, int R, int K);
void launch_grouped_kpart(const uint16_t* a, const uint8_t* w, const uint8_t* sw, uint16_t* c, int M, int G, int R, int K,
                          hipStream_t st);
// The kernel of a dense product: the K-part kernel or the tiled GEMM, by their estimated times; where neither fits (K
// > 8192, unaligned operands) the GEMV (M <= 64) or the row-group kernel. The first two load operands straight into LDS, 16 bytes
// a lane, and are kept to 16-byte aligned operands; the GEMV and the row groups take any.
enum class Fp8Route { kpart, tiled, gemv, skinny };
Fp8Route fp8_route(const Fp8GemmArgs& a);
inline bool fp8_aligned(const void* a, const void* w) {
  return (reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w)) % 16 == 0;
}
void launch_fp8_gemm(const Fp8GemmArgs& a, hipStream_t st);
// The kernel of a grouped projection (grouped_fp8w.hip).
enum class GroupedRoute { rows, kpart, gemv, tiled, ref };
GroupedRoute grouped_route(const void* a, const void* w, int M, int G, int R, int K);

}  // namespace unholy::kernels
