// Rules on sizes that choose between kernels, apart from the launch code: plain
// host arithmetic, so that a test can ask them without a GPU.
#pragma once

#include <algorithm>
#include <cmath>
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

// Launches of the prompt attention kernel, tiles of 32 queries of one
// (sequence, head), against the split-K kernel, 8 queries a workgroup, for
// caches of up to max_keys keys.  16 positions a sequence take as long either
// way and 20 are faster in tiles (16 x 16 heads after 300 keys: 19.8 / 19.7 us,
// 27.1 -> 20.3); below 160 tiles the MFMAs of a few CUs would carry the launch
// that the split-K kernel spreads over the chip (4 heads x 22 tiles: 23.2 us
// there, 26.6 here; 8 x 22: 22.3 -> 17.2).
// Over long caches both are bound by their products, the tiles' including
// those of the empty rows of a tile and of the CUs without a tile in the last
// round of 256: `waste` is the tiles' products over the split-K kernel's.  With
// `share` the time of a tile's product in the split-K kernel's, the tiles are
// the faster while waste x share is below 1 (1.05: ties).  Measured shares of
// waste 1.6 to 2.6 at 1024 / 2048 / 4096 / 8192 keys: 8 dims 0.45 / 0.56 / 0.60 /
// 0.68, 16 dims 0.43 / 0.51 / 0.54 / 0.57, 32 dims 0.40 / 0.39 / 0.40 / 0.46,
// 40 dims 0.39 / 0.46 / 0.49 / 0.51, 64 dims 0.39 / 0.37 / 0.36 / 0.39, over int8
// rows up to 0.43.  160 pairs x 40 positions over 16000 keys (waste 2.6),
// split-K / tiles: 16 dims 200 / 298 us, 40 dims 477 / 590, 64 dims of int8 rows
// 612 / 703; over 4000 keys 64 dims 203 / 177.
constexpr int kPromptTile = 32;
inline bool attention_prompt_shape(int B, int S, int H, int D, bool q8, int max_keys) {
  const int64_t pairs = (int64_t)B * H;
  const int64_t tiles = pairs * ((S + kPromptTile - 1) / kPromptTile);
  if (S < 20 || tiles < 160) return false;
  const double waste = (double)((tiles + 255) / 256 * 256 * kPromptTile) /
                       (double)(pairs * ((S + 7) / 8) * 8);
  const double doublings = std::max(-1.0, std::log2(max_keys / 1024.0));
  const double share = D <= 16               ? 0.45 + 0.08 * doublings
                       : D == 64 && !q8      ? 0.40
                       : D == 64 || D == 32  ? 0.40 + 0.02 * doublings
                                             : 0.40 + 0.04 * doublings;
  return waste * share <= 1.05;
}

// fp32 products (and int8 ones of shapes the digit GEMMs do not take).  The
// fp32 MFMA GEMM takes the GEMV over from 16 rows and 90000 outputs on: the
// GEMV runs at about 20 TFLOP/s, the GEMM costs 7 ns per entry of K and wave
// whatever the size, so the line does not depend on K.  Measured (GEMV /
// GEMM): 64 x 2048 at K = 512 11.1 / 7.9 us, 64 x 512 at K = 2048 8.5 / 18.4,
// 128 x 512 at K = 512 6.7 / 7.8, 128 x 3072 at K = 1024 54 / 18.5.
inline bool gemm_f32_shape(int rows, int N) {
  return rows >= 16 && (int64_t)rows * N >= 90000;
}

// Its tile, 64 x 64 (0) or 32 x 32 with K over 4 or 8 waves (returned).  64 x 64
// when there are enough of them and more than half of their rows are filled
// (2048 x 4096 at K = 1024, 2048 tiles: 175 us with 64 x 64, 254 with 32 x 32;
// 512 x 1024, 128 tiles: 32 / 19; 16 x 62501 at K = 1024, int8 codes: 96 / 63,
// GEMV 77).  8 waves when their workgroups run at once (64 x 1024 at K = 4096:
// 41 us over 4 waves, 34 over 8; 16 x 5626, 176 tiles, at K = 4096, int8 codes:
// 39 / 30, GEMV 32; 16 x 12501, 391 tiles: 55 / 58).  K below 64 is too short to
// split (256 x 352, 64 x 64 / 4 waves: K = 64 5.2 / 4.6 us, K = 252 10.1 / 5.6,
// GEMV 5.8).
inline int gemm_f32_waves(int rows, int K, int N) {
  const int64_t t64 = (int64_t)((rows + 63) / 64) * ((N + 63) / 64);
  const int64_t t32 = (int64_t)((rows + 31) / 32) * ((N + 31) / 32);
  if (K < 64 || (t64 >= 448 && rows > 32)) return 0;
  return t32 > 256 || K < 512 ? 4 : 8;
}

// Backend products that run on matmul_short_kernel and not on matmul_kernel:
// those with too little K to fill the latter's steps of 32, over many tiles
// (of 64 x 64): the fewer the shorter the K and the emptier the tiles.
// Measured, matmul_kernel / short, in us:
//   up to 32 rows or columns: 1 x 4 x 65536 6.4 / 6.0, 1 x 16 x 100000 12.5 / 9.3, 8 x
//     4 x 131072 10.1 / 6.3, 8 x 24 x 131072 17.2 / 14.4, 8 x 32 x 131072 17.2 / 17.4,
//     32 x 12 x 1 M 86 / 61, 8 x 40 x 1 M 151 / 127, 8 x 64 x 1 M 193 / 215
//   up to 64: 64 x 12 x 262144 28.1 / 31.4, 64 x 12 x 1 M 145 / 123
//   more: 4096 x 4 x 16384 73 / 89, 32768 x 4 x 4096 193 / 176, 100 x 12 x 1 M 189 /
//     168, 131072 x 4 x 1000 267 / 189, 131072 x 32 x 1000 352 / 393
inline bool matmul_short_shape(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64), side = std::min(M, N);
  if (K >= 32) return K < 64 && side <= 32 && tiles >= 8192;
  return tiles >= (side <= 32 ? 64 * std::max<int64_t>(K, 16) : side <= 64 ? 16384 : 32768);
}

// Sums of the backend that run with a thread an output (sum_short_kernel) and
// not in tiles through LDS (sum_kernel): short ones, longer where neighbouring
// outputs are neighbours in memory (along_r false), and there of any length from
// 65536 outputs on, whose threads fill the chip; along the sums also those that
// leave much of a 32-entry tile empty.  Measured, tiles / threads, in us (a
// thread an output with one load at a time, before both):
//   along the outputs: 2 x 1 M 25.2 / 7.5 (8.5), 32 x 8192 6.2 / 5.8 (12.9), 64 x
//     8192 5.5 / 6.1 (22), 40 x 131072 17.8 / 5.8 (16.5), 64 x 262144 30.6 / 12.1
//     (41), 300 x 131072 169 / 31 (148), 1000 x 16384 47 / 74 (439)
//   along the sums: 8 x 1 M 28.2 / 17.1 (19.5), 12 x 1 M 29.7 / 19.6 (27.4), 16 x
//     1 M 31.6 / 32.6 (40), 17 x 262144 14.7 / 8.3 (12.5), 24 x 1 M 59 / 51 (201),
//     32 x 1 M 67 / 89 (531), 64 x 262144 27.6 / 44.8 (71)
inline bool sum_short_shape(int64_t n_out, int64_t n_red, bool along_r) {
  if (!along_r) return n_red <= 32 || n_out >= 65536;
  return n_red <= 12 || (n_red > 16 && n_red <= 24 && n_out >= 131072);
}

}  // namespace nnhip
