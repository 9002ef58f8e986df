// Prints the kernel that the library's dispatch chooses for each call described on stdin, one per line. Nothing is
// launched and no pointer is read, so it runs without a GPU (tests/test_routes.py).
//   dense M N K ldc f32 a_offset w_offset       -> kpart | tiled | gemv | skinny
//   form  M N K ldc f32 a_offset w_offset       -> the K-part kernel's tile, row x column blocks of 16
//   gform M G R K                               -> the grouped K-part kernel's tile
//   token T K E D I                             -> token (two launches) | general
//   shape T K E D I                             -> w4 | w8, the forward's w1 / w3 GEMV
//   moe T K E D I                               -> gemm | gemv, the forward up to 64 tokens
//   split tiles N K                             -> split | whole, a single-projection GEMV
//   grouped M G R K a_offset w_offset           -> rows | kpart | gemv | tiled | ref
#include <algorithm>
#include <cstdint>
#include <iostream>
#include <sstream>
#include <string>

#include "fp8_internal.hpp"
#include "mx_internal.hpp"

using namespace unholy::kernels;

static const uint8_t* at(uintptr_t offset) { return reinterpret_cast<const uint8_t*>(0x100000 + offset); }

int main() {
  static const char* const kDense[] = {"kpart", "tiled", "gemv", "skinny"};
  static const char* const kGrouped[] = {"rows", "kpart", "gemv", "tiled", "ref"};
  for (std::string line; std::getline(std::cin, line);) {
    std::istringstream in(line);
    std::string kind;
    in >> kind;
    if (kind == "dense" || kind == "form") {
      Fp8GemmArgs a{};
      int f32 = 0;
      uintptr_t ao = 0, wo = 0;
      in >> a.M >> a.N >> a.K >> a.ldc >> f32 >> ao >> wo;
      a.a = at(ao);
      a.w = at(wo);
      a.c = reinterpret_cast<uint16_t*>(0x100000);
      if (f32) a.sa32 = a.sw32 = reinterpret_cast<const float*>(0x100000);
      else a.sa8 = a.sw8 = at(0);
      if (kind == "form") {
        const auto [rb, cb] = fp8_kpart_form(a);
        std::cout << rb << "x" << cb << "\n";
      } else {
        std::cout << kDense[int(fp8_route(a))] << "\n";
      }
    } else if (kind == "grouped") {
      int M, G, R, K;
      uintptr_t ao = 0, wo = 0;
      in >> M >> G >> R >> K >> ao >> wo;
      std::cout << kGrouped[int(grouped_route(at(ao), at(wo), M, G, R, K))] << "\n";
    } else if (kind == "gform") {
      int M, G, R, K;
      in >> M >> G >> R >> K;
      const auto [rb, cb] = grouped_kpart_form(M, G, R, K);
      std::cout << rb << "x" << cb << "\n";
    } else if (kind == "token") {
      MoeTokenArgs a{};
      in >> a.T >> a.K >> a.E >> a.D >> a.I;
      std::cout << (moe_token_fits(a) ? "token" : "general") << "\n";
    } else if (kind == "shape") {
      int T, K, E, D, I;
      in >> T >> K >> E >> D >> I;
      const size_t n = size_t(moe_live_tiles(T, K, E, 16)) * size_t(I / 128);
      std::cout << (gemv_four_waves(n, std::min(16, T), D) ? "w4" : "w8") << "\n";
    } else if (kind == "moe") {
      int T, K, E, D, I;
      in >> T >> K >> E >> D >> I;
      std::cout << (moe_gemm_pays(T, K, E, D, I) ? "gemm" : "gemv") << "\n";
    } else if (kind == "split") {
      int tiles, N, K;
      in >> tiles >> N >> K;
      std::cout << (gemv_splits_k(size_t(tiles), size_t(N / 16), K) ? "split" : "whole") << "\n";
    } else {
      return 1;
    }
  }
}
