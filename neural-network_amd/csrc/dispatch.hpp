// Rules on sizes that choose between kernels, apart from the launch code: plain
// host arithmetic, so that a test can ask them without a GPU.
#pragma once

#include <algorithm>
#include <cstdint>

namespace nnhip {

// Tile of the tall digit-plane GEMM (gemm_tall_kernel).
constexpr int kTallM = 128, kTallN = 256;

// Where the 128 x 256-tile GEMM takes a digit-plane product over from the
// LDS-resident GEMM (vs_lds) or the digit-plane one.  A tile takes 8 (K = 512)
// to 60 us (K = 4096) however few there are and however few of its rows are
// filled, and 256 run at once; the other two GEMMs' time grows with rows x N.
// So there have to be 96 tiles, a row tile must not be mostly empty, and the
// outputs must be worth a round of tiles: those of 96 full tiles, or, against
// the digit-plane GEMM, whose outputs cost more at a small K, fewer there.
// Measured, the other GEMM / this one, in us:
//   LDS GEMM, K = 1024, N = 32000: 16 rows 10.9 / 22.0, 64 18.1 / 25.2, 96 22.9
//     / 25.6, 128 27.6 / 24.3, 192 37.4 / 29.7; N = 24576: 96 rows 20.5 / 24.7,
//     128 25.1 / 23.5; N = 8192: 512 rows 25.7 / 24.2, 1024 45.9 / 28.8
//   digit-plane GEMM, K = 4096: 64 x 32000 61 / 74, 192 x 12288 56 / 72, 288 x
//     8192 59 / 71, 384 x 8192 75 / 71, 4096 x 1024 130 / 75; K = 2048: 64 x
//     32768 39.8 / 43.6, 192 x 12288 39.0 / 40.7, 256 x 12288 47.8 / 39.4; K =
//     1024, N = 32000: 32 rows 16.0 / 23.6, 64 26.2 / 25.3; K = 512, N = 32768:
//     32 rows 12.6 / 15.1, 64 23.3 / 16.8
inline bool gemm_tall_shape(int rows, int K, int N, bool vs_lds) {
  constexpr int64_t kMinTiles = 96, kFull = kMinTiles * kTallM * kTallN;
  const int64_t tiles = (int64_t)((rows + kTallM - 1) / kTallM) * ((N + kTallN - 1) / kTallN);
  const int64_t least = vs_lds ? kFull : std::min(kFull, ((int64_t)1 << 20) + 1024 * (int64_t)K);
  return K % 128 == 0 && N % 32 == 0 && tiles >= kMinTiles &&
         rows >= (vs_lds ? kTallM : kTallM / 2) && (int64_t)rows * N >= least;
}

}  // namespace nnhip
