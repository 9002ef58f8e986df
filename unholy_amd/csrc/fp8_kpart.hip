// Dense fp8 GEMM for up to ~700 rows at 4096 x 4096: C[M, N] (bf16) = A[M, K] (e4m3) x W[N, K]^T (e4m3), per-128 scales
// (e8m0 or fp32, as fp8_tiled.hip).
//
// What bounds these sizes is getting each CU's share of W and A to it: 4096 x 4096 weights are 64 KB per CU, and a
// tile of R x C outputs reads (R + C) K bytes, mostly from L2. A grid of about one workgroup per CU therefore wants the
// largest tile that still makes 256 workgroups, with many bytes in flight and no barrier to wait at.
// - A workgroup = 8 waves over one tile of 16 RB rows x 16 CB columns; wave w takes the w-th eighth of K's 128-blocks
//   and computes the whole tile over it. The waves share nothing (each has its own LDS slot and no barrier) until their
//   partial tiles are added through LDS in wave order.
// - Operands go through LDS by direct loads of 8 rows x 128 bytes with consecutive lanes along a row. Loads straight
//   into MFMA operand order (lane l: row l % 16) read at most 9.5 TB/s from L2, whatever is in flight: four
//   consecutive lanes lie in four rows; with consecutive lanes along a row L2 delivers 25-33 TB/s (a read-only probe,
//   all CUs). 64 x 4096 x 4096 step 14.2 us with the register loads, 12.1 with these; 300 rows 29 / 21.8.
// - A lane's 16 bytes of an operand row feed two 16x16x32 bf16 MFMAs as they stand (the same input permutation on
//   both sides), converted exactly. e8m0 scales are folded into the conversions (exact); with fp32 scales each
//   block's MFMA chain starts from zero and is folded as acc += raw * (sa * sw).
// Steps (act_quant + GEMM, us, 4096 x 4096) against the kernels that ran before it: e8m0 M = 32 15.5 -> 11.1, 64 20.0 ->
// 12.1, 128 38.5 -> 15.2, 256 41.6 -> 19.9, 300 41.3 -> 21.8, 512 42.3 -> 32.0; fp32 M = 64 13.6 -> 11.9, 256 34.6 ->
// 20.2, 300 43.5 -> 23.3. 32768 x 1024, e8m0, M = 64: 97 -> 19. Decode rows (before: every lane 32 bytes of its own row):
// e8m0 M = 1 10.5 -> 8.7, 16 12.2 -> 9.6, 16 x 32768 x 1024 36 -> 14; the fused form M = 1 7.2 -> 6.3, 4 10.5 -> 8.7.
#include <algorithm>
#include <stdexcept>
#include <utility>

#include "common.hpp"
#include "numerics.hpp"
#include "fp8_internal.hpp"
#include "pipe.hpp"

namespace unholy::kernels {

using namespace uh;
using namespace pipe;

namespace {

constexpr int KP_WAVES = 8;
constexpr int NSET = 2;  // scale registers per row block: NSET sets of 4 128-input blocks

// The waves' partial tiles added in wave order through LDS (every wave is past its own LDS use after the first barrier),
// PB column blocks at a time, so that a pass's partials fit 128 KB; store(row, column, sum) of each output.
template <int RB, int CB>
constexpr int kp_pass() { return RB * CB <= 16 ? CB : CB / 2; }
template <int RB, int CB>
constexpr size_t kp_reduce_lds() { return size_t(KP_WAVES) * RB * kp_pass<RB, CB>() * 64 * 16; }
template <int RB, int CB, class Store>
__device__ __forceinline__ void kp_reduce(const v4f (&acc)[RB][CB], uint8_t* smem, const Store& store) {
  constexpr int PB = kp_pass<RB, CB>(), NV = RB * PB;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  v4f* const red = reinterpret_cast<v4f*>(smem);
#pragma unroll
  for (int p = 0; p < CB; p += PB) {
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int cb = 0; cb < PB; ++cb) red[(wave * NV + rb * PB + cb) * 64 + lane] = acc[rb][p + cb];
    __syncthreads();
    for (int v = wave; v < NV; v += KP_WAVES) {
      v4f s = red[v * 64 + lane];
#pragma unroll
      for (int w = 1; w < KP_WAVES; ++w) s += red[(w * NV + v) * 64 + lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) store((v / PB) * 16 + 4 * g + i, (p + v % PB) * 16 + l16, s[i]);
    }
  }
}

// One operand of a tile for N direct loads of RPL rows each: `rows` rows of `stride` bytes from row row0 of b on, `width`
// bytes of each at byte k, lane l taking the 16 bytes at piece(i) of row l / (64 / RPL) of load i. Rows past the tile repeat
// its last, or that row's end: in bounds, and their results are not stored.
// HOLD: an offset register per load. Without it load i's rows go into the scalar base, a few scalar instructions a load, and
// two lane offsets serve them all (piece(i) is then piece(i % 2)): the largest tiles have no registers for 20 offsets. (With
// them 6 x 4 and the grouped 8 x 4 spilled some, and every reload waited for the direct loads in flight: 384 x 4096 x
// 4096 21.9 us, 19.6 so; fp32 scales, 5 x 4, 300 rows 18.7, 18.0; grouped 512 x 8192 x 4096 49.3, 47.7. The smaller
// tiles are up to 3% faster with them.)
template <int RPL, int N, bool HOLD>
struct KpRows {
  const uint8_t* base;
  uint32_t stride, last, end, lane_off[2];
  uint32_t off[HOLD && N ? N : 1];
  template <class Piece>
  __device__ __forceinline__ KpRows(const void* b, size_t row0, uint32_t stride_, int rows, int width, const Piece& piece)
      : base(static_cast<const uint8_t*>(b) + row0 * stride_), stride(stride_) {
    const int q = int(threadIdx.x & 63) / (64 / RPL);
    if constexpr (HOLD) {
#pragma unroll
      for (int i = 0; i < N; ++i) off[i] = uint32_t(min(i * RPL + q, rows - 1)) * stride + piece(i);
    } else {
      for (int i = 0; i < 2; ++i) lane_off[i] = uint32_t(q) * stride + piece(i);
      last = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t((rows - 1) / RPL * RPL) * stride)));
      end = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(rows - 1) * stride + uint32_t(width - 16))));
    }
  }
  __device__ __forceinline__ void load(size_t k, uint32_t lds) const {
    if constexpr (HOLD) {
#pragma unroll
      for (int i = 0; i < N; ++i) dma16(base + k, off[i], lds + uint32_t(i * 1024));
    } else {
      uint32_t lst = last, e = end;  // opaque: the addresses are formed in this step, not ahead of the loop (in registers)
      asm volatile("" : "+s"(lst), "+s"(e));
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const uint32_t at = min(uint32_t(i * RPL) * stride, lst);
        dma16(base + k + at, min(lane_off[i % 2], e - at), lds + uint32_t(i * 1024));
      }
    }
  }
};

// XQ (fp32 scales, one row block): A arrives as bf16 rows (a.xa), quantized here as act_quant_fp8_f32s does (s = max(amax,
// 1e-4) * fp32(1/448), codes e4m3(x / s); 8 values per lane, a block's amax a DPP row max over 16 lanes). Each wave
// quantizes the rows of its own K part into its own LDS, behind its first weight loads: no wave waits for another.
// pp.n > 0 (gemv_w8a8_parts: e8m0 scales, one row tile, CB = 1): column ranges, each with its weights and output.
template <bool F32S, int RB, int CB, bool XQ = false>
__global__ __launch_bounds__(64 * KP_WAVES) __attribute__((amdgpu_waves_per_eu(2))) void fp8_kpart_kernel(
    Fp8GemmArgs a, Fp8Parts pp, int row_tiles, int tile_rows) {
  static_assert(!XQ || (F32S && RB == 1));
  extern __shared__ __align__(16) uint8_t smem[];
  const int M = a.M, K = a.K, KS = K / 128;
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Work item = column block x row tiles + row tile; XCD x takes the x-th eighth of the items, so that the row tiles of
  // a column block share one L2.
  const int nw = gridDim.x, lin = blockIdx.x;
  int wi = nw % 8 ? lin : (lin & 7) * (nw >> 3) + (lin >> 3);
  if constexpr (!F32S && CB == 1)
    if (pp.n) {
      int p = 0;
      while (p + 1 < pp.n && wi >= pp.t0[p + 1]) ++p;
      wi -= pp.t0[p];
      a.w = pp.w[p];
      a.sw8 = pp.sw[p];
      a.c = pp.c[p];
      a.ldc = pp.ldc[p];
      a.N = pp.N[p];
    }
  const int N = a.N, row0 = (wi % row_tiles) * tile_rows, col0 = (wi / row_tiles) * (16 * CB);
  const int Mt = min(tile_rows, M - row0);
  const int per = (KS + KP_WAVES - 1) / KP_WAVES, b0 = min(KS, wave * per), n = min(KS, b0 + per) - b0;  // blocks

  // Scales of the wave's blocks in registers. Lane group g holds block g (NSET sets of 4): the rows' of row block rb
  // in lane l16 = row; the weights' (16 CB columns lie in one 128-row weight block) of block l in lane l.
  float sav[NSET][RB], swv = 0.0f;
  const auto sa_at = [&](int r, int kb) {
    const size_t i = size_t(row0 + min(r, Mt - 1)) * KS + min(kb, KS - 1);
    return F32S ? a.sa32[i] : e8m0_to_f32(a.sa8[i]);
  };
#pragma unroll
  for (int q = 0; q < NSET; ++q)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) sav[q][rb] = !XQ && q * 4 < per ? sa_at(rb * 16 + l16, b0 + 4 * q + g) : 0.0f;
  {
    const size_t i = size_t(col0 / 128) * KS + min(b0 + (lane & 7), KS - 1);
    swv = F32S ? a.sw32[i] : e8m0_to_f32(a.sw8[i]);
  }

  // The wave's slot in LDS: one 128-input block, RB row blocks then CB column blocks of 16 rows x 128 bytes. A direct
  // load covers 8 rows x 128 bytes; the 16-byte piece p of row r sits at p ^ ((r >> 1) & 7).
  // XQ: the weights' blocks only; the quantized rows of all the wave's blocks lie behind the slots, [per][16][128] codes
  // (pieces as above) and [per][16] fp32 scales.
  constexpr int AB = XQ ? 0 : RB, SLOT = (AB + CB) * 2048, NL = 2 * (AB + CB);
  uint8_t* const slot = smem + wave * SLOT;
  uint8_t* const xcodes = smem + KP_WAVES * SLOT + wave * (per * (2048 + 64));
  float* const xscale = reinterpret_cast<float*>(xcodes + per * 2048);
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(slot));
  const auto piece = [&](int i) { return uint32_t(((lane & 7) ^ (lane >> 4) ^ (i & 1 ? 4 : 0)) * 16); };
  constexpr bool HOLD = RB * CB <= (F32S ? 16 : 20);
  const KpRows<8, 2 * AB, HOLD> arows(a.a, row0, K, Mt, 128, piece);
  const KpRows<8, 2 * CB, HOLD> wrows(a.w, col0, K, min(16 * CB, N - col0), 128, piece);
  const auto issue = [&](int c) {
    const size_t k = size_t(b0 + c) * 128;
    arows.load(k, lds0);
    wrows.load(k, lds0 + uint32_t(AB * 2048));
  };
  // Item it = (row, block, piece of 8 values), 16 lanes a block.
  const int xitems = M * n * 16;
  const auto x_src = [&](int it) {
    const int c = min(it, xitems - 1), r = c / (16 * n), rem = c % (16 * n);
    return a.xa + size_t(r) * a.ldx + size_t(b0) * 128 + rem * 8;
  };
  const auto quant_item = [&](int it, const v4i raw) {
    const int r = it / (16 * n), rem = it % (16 * n), blk = rem >> 4, l = rem & 15;
    float v[8], am = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(uint32_t(raw[i]) << 16);
      v[2 * i + 1] = __uint_as_float(uint32_t(raw[i]) & 0xffff0000u);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) am = fmaxf(am, fabsf(v[i]));
    am = row16_max(am);
    if (it >= xitems) return;
    const float sc = fmaxf(am, 1e-4f) * (1.0f / 448.0f);
    uint32_t c0, c1;
    fp8_codes8(v, sc, c0, c1);
    *reinterpret_cast<uint2*>(xcodes + blk * 2048 + r * 128 + ((l >> 1) ^ ((r >> 1) & 7)) * 16 + (l & 1) * 8) =
        make_uint2(c0, c1);
    if (l == 0) xscale[blk * 16 + r] = sc;
  };
  if (n > 0) {
    if constexpr (XQ) {  // one block of code from the untracked load to its wait: its register is never merged or moved
      v4i x0 = vload16(x_src(lane));
      issue(0);
      wait_vm<NL>();  // the rows' first pass; the weights stay in flight
      asm volatile("" : "+v"(x0));
      quant_item(lane, x0);
      for (int base = 64; base < xitems; base += 256) {  // uniform bound: 16-lane groups stay whole; 4 passes' loads at once
        v4i x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = *reinterpret_cast<const v4i*>(x_src(base + 64 * i + lane));
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (base + 64 * i < xitems) quant_item(base + 64 * i + lane, x[i]);
      }
    } else {
      issue(0);
    }
  }
  v4f acc[RB][CB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  // The scales are waited for here, once (with the first block's loads behind them), not in the loop.
  asm volatile("" : "+v"(swv));
#pragma unroll
  for (int q = 0; q < NSET; ++q)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) asm volatile("" : "+v"(sav[q][rb]));

  const uint8_t* const rd = slot + l16 * 128;
  const int p0 = (g ^ ((l16 >> 1) & 7)) * 16, p1 = ((4 + g) ^ ((l16 >> 1) & 7)) * 16;
#pragma unroll 1  // run from a cold instruction cache: small beats unrolled
  for (int c = 0; c < n; ++c) {
    wait_vm<0>();
    asm volatile("" ::: "memory");
    v4i aq[RB][2], bq[CB][2];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      bq[cb][0] = *reinterpret_cast<const v4i*>(rd + (AB + cb) * 2048 + p0);
      bq[cb][1] = *reinterpret_cast<const v4i*>(rd + (AB + cb) * 2048 + p1);
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const uint8_t* const ra = XQ ? xcodes + c * 2048 + l16 * 128 : rd + rb * 2048;
      aq[rb][0] = *reinterpret_cast<const v4i*>(ra + p0);
      aq[rb][1] = *reinterpret_cast<const v4i*>(ra + p1);
    }
    if (c + 1 < n) {  // the next block into the slot as soon as it has been read: in flight under this block's MFMAs
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      asm volatile("" ::: "memory");
      issue(c + 1);
    }
    const float sw = __uint_as_float(uint32_t(__builtin_amdgcn_readlane(int(__float_as_uint(swv)), c & 7)));
    const auto sa_of = [&](int rb, int row) {  // the scale of row `row` of the row block in block c
      if constexpr (XQ) return xscale[c * 16 + row];
      const float v = c >= 4 ? sav[1][rb] : sav[0][rb];
      return __uint_as_float(uint32_t(__builtin_amdgcn_ds_bpermute(((c & 3) * 16 + row) * 4, int(__float_as_uint(v)))));
    };
    bf16x8 bf[CB][4];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        bf[cb][t] = fp8x8_to_bf16(uint32_t(bq[cb][t >> 1][2 * (t & 1)]), uint32_t(bq[cb][t >> 1][2 * (t & 1) + 1]),
                                  F32S ? 1.0f : sw);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const float asc = F32S ? 1.0f : sa_of(rb, l16);
      v4f raw[CB];
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) raw[cb] = F32S ? v4f{0.0f, 0.0f, 0.0f, 0.0f} : acc[rb][cb];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const bf16x8 af = fp8x8_to_bf16(uint32_t(aq[rb][t >> 1][2 * (t & 1)]),
                                        uint32_t(aq[rb][t >> 1][2 * (t & 1) + 1]), asc);
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) raw[cb] = mfma_bf16(af, bf[cb][t], raw[cb]);
      }
      if constexpr (F32S) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float f = sa_of(rb, 4 * g + i) * sw;
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) acc[rb][cb][i] += raw[cb][i] * f;
        }
      } else {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = raw[cb];
      }
    }
  }

  kp_reduce(acc, smem, [&](int r, int col, float v) {
    if (r < Mt && col0 + col < N) a.c[size_t(row0 + r) * a.ldc + col0 + col] = f32_to_bf16(v);
  });
}

template <bool F32S, int RB, int CB, bool XQ = false>
void launch_t(const Fp8GemmArgs& a, hipStream_t st, const Fp8Parts& pp = Fp8Parts{}) {
  constexpr size_t red = kp_reduce_lds<RB, CB>(), slots = size_t(KP_WAVES) * ((XQ ? 0 : RB) + CB) * 2048;
  static_assert(std::max(red, slots) <= 160 * 1024);
  const size_t rows = XQ ? size_t(KP_WAVES) * ((a.K / 128 + KP_WAVES - 1) / KP_WAVES) * (2048 + 64) : 0;
  const size_t lds = std::max(red, slots + rows);
  const int rt = (a.M + 16 * RB - 1) / (16 * RB), tile_rows = ((a.M + rt - 1) / rt + 15) / 16 * 16;
  auto* kern = &fp8_kpart_kernel<F32S, RB, CB, XQ>;
  if (lds > 65536)
    UH_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 int(lds)));
  const unsigned cols = pp.n ? unsigned(pp.t0[pp.n]) : cdiv(size_t(a.N), 16 * CB);
  kern<<<dim3(cols * unsigned(rt)), 64 * KP_WAVES, lds, st>>>(a, pp, rt, tile_rows);
  UH_CHECK_LAUNCH();
}

// The same for the grouped projection c[m][g][r] = sum_k a[m][g][k] w[g R + r][k]: bf16 rows as they are (twice the
// bytes of the weights' rows), e8m0 weight scales per 128 x 128 folded into the conversions. KB inputs per step and
// slot: 128 (A 16 rows x 256 bytes, W 16 rows x 128 bytes per block), or 64 for the forms whose 128-input slots do not
// fit (A 16 x 128, W 16 x 64).
template <int RB, int CB, int KB>
struct GKp {
  static constexpr int AB = 16 * KB * 2, WB = 16 * KB, SLOT = RB * AB + CB * WB, NA = RB * AB / 1024, NW = CB * WB / 1024;
  static constexpr int AR = 1024 / (2 * KB), WR = 1024 / KB;  // rows per direct load
  // Piece (16 bytes) p of row r of a block: the 16 rows that an operand read covers touch each LDS bank once.
  static __device__ __forceinline__ int aswz(int r) { return KB == 128 ? r : (r >> 1) & 7; }
  static __device__ __forceinline__ int wswz(int r) { return KB == 128 ? (r >> 1) & 7 : (r >> 2) & 3; }
  static constexpr size_t lds() { return std::max<size_t>(kp_reduce_lds<RB, CB>(), size_t(KP_WAVES) * SLOT); }
};
template <int RB, int CB, int KB>
__global__ __launch_bounds__(64 * KP_WAVES) __attribute__((amdgpu_waves_per_eu(2))) void grouped_kpart_kernel(
    const uint16_t* a, const uint8_t* w, const uint8_t* sw, uint16_t* c, int M, int G, int R, int K, int row_tiles,
    int tile_rows) {
  using T = GKp<RB, CB, KB>;
  extern __shared__ __align__(16) uint8_t smem[];
  const int KS = K / 128, N = G * R;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int nw = gridDim.x, lin = blockIdx.x;
  const int wi = nw % 8 ? lin : (lin & 7) * (nw >> 3) + (lin >> 3);
  const int row0 = (wi % row_tiles) * tile_rows, col0 = (wi / row_tiles) * (16 * CB), grp = col0 / R;  // R % (16 CB) == 0
  const int Mt = min(tile_rows, M - row0);
  const int per = (KS + KP_WAVES - 1) / KP_WAVES, b0 = min(KS, wave * per), n = (min(KS, b0 + per) - b0) * (128 / KB);
  // The scale of the wave's block l in lane l (the host: at most 64 blocks a wave).
  float swv = e8m0_to_f32(sw[size_t(col0 / 128) * KS + min(b0 + lane, KS - 1)]);
  uint8_t* const slot = smem + wave * T::SLOT;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(slot));
  constexpr int AP = 64 / T::AR, WP = 64 / T::WR;  // pieces per row
  const auto apiece = [&](int i) {
    return uint32_t(((lane % AP) ^ T::aswz(lane / AP) ^ T::aswz(i * T::AR & 15)) * 16);
  };
  const auto wpiece = [&](int i) {
    return uint32_t(((lane % WP) ^ T::wswz(lane / WP) ^ T::wswz(i * T::WR & 15)) * 16);
  };
  constexpr bool HOLD = RB < 8;
  const KpRows<T::AR, T::NA, HOLD> arows(a + size_t(grp) * K, row0, uint32_t(G) * uint32_t(K) * 2u, Mt, 2 * KB, apiece);
  const KpRows<T::WR, T::NW, HOLD> wrows(w, col0, K, 16 * CB, KB, wpiece);
  const auto issue = [&](int s) {
    const size_t k = size_t(b0) * 128 + size_t(s) * KB;
    wrows.load(k, lds0 + uint32_t(RB * T::AB));
    arows.load(2 * k, lds0);
  };
  if (n > 0) issue(0);
  v4f acc[RB][CB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  asm volatile("" : "+v"(swv));  // waited for here, once, not in the loop
  constexpr int H = KB / 64;     // 64-input halves: one 16-byte piece of W and two of A per lane
#pragma unroll 1
  for (int s = 0; s < n; ++s) {
    wait_vm<0>();
    asm volatile("" ::: "memory");
    v4i wq[CB][H];
    bf16x8 aq[RB][2 * H];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int x = 0; x < H; ++x)
        wq[cb][x] = *reinterpret_cast<const v4i*>(slot + RB * T::AB + cb * T::WB + l16 * KB +
                                                  ((4 * x + g) ^ T::wswz(l16)) * 16);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int t = 0; t < 2 * H; ++t)  // inputs 64 (t / 2) + 16 g + 8 (t % 2) .. + 7, as W's conversion t
        aq[rb][t] = *reinterpret_cast<const bf16x8*>(slot + rb * T::AB + l16 * KB * 2 +
                                                     ((8 * (t >> 1) + 2 * g + (t & 1)) ^ T::aswz(l16)) * 16);
    if (s + 1 < n) {  // the next step into the slot as soon as it has been read
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      asm volatile("" ::: "memory");
      issue(s + 1);
    }
    const float sc = __uint_as_float(uint32_t(__builtin_amdgcn_readlane(int(__float_as_uint(swv)), s * KB / 128)));
#pragma unroll
    for (int t = 0; t < 2 * H; ++t) {
      bf16x8 wf[CB];
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
        wf[cb] = fp8x8_to_bf16(uint32_t(wq[cb][t >> 1][2 * (t & 1)]), uint32_t(wq[cb][t >> 1][2 * (t & 1) + 1]), sc);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = mfma_bf16(aq[rb][t], wf[cb], acc[rb][cb]);
    }
  }
  kp_reduce(acc, smem, [&](int r, int col, float v) {
    if (r < Mt) c[size_t(row0 + r) * N + col0 + col] = f32_to_bf16(v);
  });
}
template <int RB, int CB, int KB>
void launch_g(const uint16_t* a, const uint8_t* w, const uint8_t* sw, uint16_t* c, int M, int G, int R, int K,
              hipStream_t st) {
  constexpr size_t lds = GKp<RB, CB, KB>::lds();
  static_assert(lds <= 160 * 1024);
  const int rt = (M + 16 * RB - 1) / (16 * RB), tile_rows = ((M + rt - 1) / rt + 15) / 16 * 16;
  auto* kern = &grouped_kpart_kernel<RB, CB, KB>;
  UH_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                               int(lds)));
  kern<<<dim3(unsigned(G * R / (16 * CB)) * unsigned(rt)), 64 * KP_WAVES, lds, st>>>(a, w, sw, c, M, G, R, K, rt,
                                                                                     tile_rows);
  UH_CHECK_LAUNCH();
}

}  // namespace

namespace {
// The forms (16-row blocks x 16-column blocks), and what a launch of each takes, us: `start` (the launch, the first
// loads and the reduction) and `read` per 1,000 inputs (each workgroup's rows and columns of K) for a round of 256
// workgroups, `next` more for a round past the first, and `miss` per MB that an XCD's 32 workgroups in flight read
// from beyond its L2: their row tiles (`abytes` a value) and column blocks. Fitted to 2,900 launches of the dense
// forms (K = 640 to 8192, N = 640 to 32768, M = 17 to 4096, up to 6 rounds; fp32 scales take 1.035 times as long) and
// 830 of the grouped ones: rms 6% and 9%. With the tiled GEMM's estimate (fp8_tiled_us) it picks a form that is 0.1%
// slower than the best on average over 1,200 dense calls measured with each, 8% at worst; grouped (tiled_us) 0.2%,
// 12%.
struct KpForm {
  int rb, cb;
  double start, next, read;
};
double launch_us(const KpForm& f, int M, size_t N, int K, int abytes, double miss) {
  const size_t rt = (size_t(M) + 16 * f.rb - 1) / (16 * f.rb), wg = rt * cdiv(N, 16 * f.cb), rounds = (wg + 255) / 256;
  const size_t xcd = std::min<size_t>(32, (wg + 7) / 8);
  const double rows = 16.0 * (double(abytes * f.rb) * double(std::min(rt, xcd)) + f.cb * double((xcd + rt - 1) / rt));
  return f.start + double(rounds - 1) * f.next + double(rounds) * K * (f.read * 1e-3 + miss * rows * 1e-6);
}
constexpr KpForm kForms[] = {{1, 1, 2.97, 0.05, 0.46}, {2, 1, 3.20, 0.2, 0.70}, {2, 2, 3.34, 0.46, 0.87},
                             {4, 2, 3.63, 2.20, 1.48}, {4, 4, 4.76, 3.20, 2.03}, {5, 4, 5.64, 3.99, 2.43},
                             {6, 4, 6.07, 4.40, 2.93}};
// (Workgroups of one 16 x 16 tile take longer with e8m0 scales than with fp32 ones: 1 x 8192 x 1024 5.0 / 4.3 us, 2 x
// 2 4.7.)
double form_us(const Fp8GemmArgs& a, const KpForm& f) {
  const double us = launch_us(f, a.M, size_t(a.N), a.K, 1, 0.23);
  return a.sa32 ? 1.035 * us : f.rb * f.cb == 1 ? us + 0.35 : us;
}
int best_form(const Fp8GemmArgs& a) {
  int best = 0;
  for (int i = 1; i < 7; ++i)
    if (form_us(a, kForms[i]) < form_us(a, kForms[best])) best = i;
  return best;
}
}  // namespace

bool fp8_kpart_fits(const Fp8GemmArgs& a) {
  return a.M > 0 && a.N > 0 && a.K > 0 && a.K % 128 == 0 && a.K <= 128 * KP_WAVES * 4 * NSET && fp8_aligned(a.a, a.w) &&
         (a.sa32 || a.xa ? a.sw32 != nullptr : a.sa8 && a.sw8);
}
bool fp8_kpart_parts_fits(const Fp8GemmArgs& a, const Fp8Parts& pp) {
  for (int i = 0; i < pp.n; ++i)
    if (!fp8_aligned(a.a, pp.w[i])) return false;
  return a.M > 0 && a.M <= 32 && a.K <= 128 * KP_WAVES * 4 * NSET;
}
void launch_fp8_kpart_parts(const Fp8GemmArgs& a, const Fp8Parts& pp, hipStream_t st) {
  if (a.M <= 16) launch_t<false, 1, 1>(a, st, pp);
  else launch_t<false, 2, 1>(a, st, pp);
}
void launch_fp8_kpart_xq(const Fp8GemmArgs& a, hipStream_t st) { launch_t<true, 1, 1, true>(a, st); }
double fp8_kpart_us(const Fp8GemmArgs& a) { return form_us(a, kForms[best_form(a)]); }
std::pair<int, int> fp8_kpart_form(const Fp8GemmArgs& a) { return {kForms[best_form(a)].rb, kForms[best_form(a)].cb}; }

void launch_fp8_kpart(const Fp8GemmArgs& a, hipStream_t st) {
  if (!fp8_kpart_fits(a)) throw std::runtime_error("fp8 kpart: shape");
  if (!a.a || !a.w || !a.c) throw std::runtime_error("fp8 gemm: null operand");
  if (a.sa32) {
    switch (best_form(a)) {
      case 0: return launch_t<true, 1, 1>(a, st);
      case 1: return launch_t<true, 2, 1>(a, st);
      case 2: return launch_t<true, 2, 2>(a, st);
      case 3: return launch_t<true, 4, 2>(a, st);
      case 4: return launch_t<true, 4, 4>(a, st);
      case 5: return launch_t<true, 5, 4>(a, st);
      default: return launch_t<true, 6, 4>(a, st);
    }
  }
  switch (best_form(a)) {
    case 0: return launch_t<false, 1, 1>(a, st);
    case 1: return launch_t<false, 2, 1>(a, st);
    case 2: return launch_t<false, 2, 2>(a, st);
    case 3: return launch_t<false, 4, 2>(a, st);
    case 4: return launch_t<false, 4, 4>(a, st);
    case 5: return launch_t<false, 5, 4>(a, st);
    default: return launch_t<false, 6, 4>(a, st);
  }
}

// ---- grouped ---------------------------------------------------------------------------------------------------------
namespace {
// As above; the rows are bf16.
constexpr KpForm kGForms[] = {{1, 1, 3.19, 0.06, 0.57}, {1, 2, 2.93, 0.32, 0.83}, {2, 2, 3.16, 1.46, 1.15},
                              {2, 4, 3.73, 1.26, 1.66}, {4, 4, 4.89, 1.75, 2.34}, {6, 4, 6.21, 3.10, 2.78},
                              {8, 4, 6.75, 3.81, 3.76}};
double gform_us(int M, int N, int K, const KpForm& f) { return launch_us(f, M, size_t(N), K, 2, 0.41); }
int best_gform(int M, int G, int R, int K) {
  int best = 0;
  for (int i = 1; i < 7; ++i)
    if (R % (16 * kGForms[i].cb) == 0 && gform_us(M, G * R, K, kGForms[i]) < gform_us(M, G * R, K, kGForms[best])) best = i;
  return best;
}
}  // namespace

// (a tile's rows span up to 128 G K bf16 from its base, in 32-bit offsets)
bool grouped_kpart_fits(int M, int G, int R, int K) {
  return M > 0 && R > 0 && R % 16 == 0 && K > 0 && K % 128 == 0 && K <= 128 * KP_WAVES * 64 &&
         size_t(128) * G * K * 2 < (size_t(1) << 32);
}
double grouped_kpart_us(int M, int G, int R, int K) { return gform_us(M, G * R, K, kGForms[best_gform(M, G, R, K)]); }
std::pair<int, int> grouped_kpart_form(int M, int G, int R, int K) {
  const KpForm& f = kGForms[best_gform(M, G, R, K)];
  return {f.rb, f.cb};
}
void launch_grouped_kpart(const uint16_t* a, const uint8_t* w, const uint8_t* sw, uint16_t* c, int M, int G, int R, int K,
                          hipStream_t st) {
  if (!grouped_kpart_fits(M, G, R, K)) throw std::runtime_error("grouped kpart: shape");
  switch (best_gform(M, G, R, K)) {
    case 0: return launch_g<1, 1, 128>(a, w, sw, c, M, G, R, K, st);
    case 1: return launch_g<1, 2, 128>(a, w, sw, c, M, G, R, K, st);
    case 2: return launch_g<2, 2, 128>(a, w, sw, c, M, G, R, K, st);
    case 3: return launch_g<2, 4, 128>(a, w, sw, c, M, G, R, K, st);
    case 4: return launch_g<4, 4, 64>(a, w, sw, c, M, G, R, K, st);
    case 5: return launch_g<6, 4, 64>(a, w, sw, c, M, G, R, K, st);
    default: return launch_g<8, 4, 64>(a, w, sw, c, M, G, R, K, st);
  }
}

}  // namespace unholy::kernels
