// Which kernel a dense GEMM runs on and its tile: host arithmetic alone, no
// HIP, so that a CPU build can walk the rules over their ranges.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace pih_amd {

constexpr uint32_t kCus = 256;
constexpr uint32_t kWalkStep = 128;  // bytes of a row per K step of the tile-walking kernel

// ---- the kernels beside gemm_tile.hip
// Small-M GEMM (gemm_small_m.hip): m <= 64 rows, and up to kSmallMRows in
// 64-row chunks while the 128 x 128 kernel would have fewer than 128 tiles
// (too few blocks to stream the weights).
constexpr uint32_t kSmallMChunkRows = 64, kSmallMRows = 256;
inline bool SmallMTakes(uint32_t m, uint32_t n, uint32_t problems) {
  if (m <= kSmallMChunkRows) return m > 0;
  return m <= kSmallMRows && (uint64_t)((m + 127) / 128) * ((n + 127) / 128) * problems < 128;
}
// the 128 x 256 tiles pay from 64 tiles on (measured at M = 2048: N = 1024,
// 64 tiles on 64 CUs, 40.7 us against 64 us for the 128 x 128 kernel's 128
// tiles)
inline bool BigTileWorthIt(uint32_t m, uint32_t n) {
  return m >= 256 && (uint64_t)((m + 127) / 128) * ((n + 255) / 256) >= 64;
}
// BF16 GEMMs above 64 rows against the 128 x 128 kernel: the 128 x 256 tiles
// (K split into the queried workspace when they are few) from 512-deep K and
// 256 columns on: Qwen3-8B projections at M 65-384 ran 1.3-3.8x faster
// (4096 -> 4096 M 192 64 -> 25 us, 12288 -> 4096 M 192 181 -> 47 us, 4096 ->
// 1024 M 1024 58 -> 28 us) and nowhere slower.
inline bool Bf16BigTiles(uint32_t m, uint32_t n, uint32_t k) {
  return BigTileWorthIt(m, n) || (m > 64 && k >= 512 && n >= 256);
}
// K splits of the 128 x 256 tiles for k_steps 128-byte K steps (1: none):
// below a round of tiles the smallest count that reaches one, with at least 8
// K steps a split, else the largest such count up to 8
inline uint32_t DenseKSplits(uint32_t m, uint32_t n, uint32_t k_steps) {
  const uint64_t tiles = (uint64_t)((m + 127) / 128) * ((n + 255) / 256);
  if (tiles == 0 || tiles >= 192) return 1;
  uint32_t best = 1;
  for (uint32_t s = 2; s <= 8; ++s) {
    if (k_steps % s || k_steps / s < 8) continue;
    if (tiles * s >= 192) return s;
    best = s;
  }
  return best;
}
// rows of their M tiles: with fewer 128-row tiles than about a round (and no
// K split) 64 or 32, up to four times the tiles at the same K depth (same
// arithmetic per element; the tiles stream their W tile from L2)
inline uint32_t DenseTileRows(uint32_t m, uint32_t n, uint32_t problems, uint32_t k_splits) {
  uint32_t rows = 128;
  const uint64_t nt = (n + 255) / 256;
  while (k_splits <= 1 && rows > 32 && (uint64_t)((m + rows - 1) / rows) * nt * problems < 192) rows /= 2;
  return rows;
}

// ---- the tile: 16 mb x 16 nb output elements, one per block or (grid) one
// block per CU walking them
struct TilePick {
  uint32_t mb = 0, nb = 0;
  bool grid = false;
};

// The tile for a shape, by an estimate of its time: the rounds of tiles on the
// CUs times what a CU loads for one (at ~64 GB/s), no less than the weights at
// the 6.2 TB/s they stream at, and 1.5 us for each round after the first (the
// start-up that the tile-walking kernel hides).  16 x 16 tiles share a CU two
// at a time: their weights were measured to stream at 7 TB/s (12288 x 4096
// bf16 at m 8: 16.5 us, 18.4 with 16 x 48 tiles) and a round is 512 of them,
// 1.1 us apart.
inline TilePick PickTile(bool bf16, uint32_t m, uint32_t n, uint32_t row_bytes, uint32_t problems) {
  TilePick best;
  double best_ns = 0.0;
  const double w_bytes = (double)n * problems * row_bytes;
  auto consider = [&](uint32_t mb, uint32_t nb, bool grid) {
    if (n % (16 * nb) || (mb > 1 && 16 * (mb - 1) >= m && mb < 8)) return;
    const uint64_t tiles = (uint64_t)((m + 16 * mb - 1) / (16 * mb)) * (n / (16 * nb)) * problems;
    const bool paired = mb == 1 && nb == 1;
    const double rounds = (double)((tiles + kCus - 1) / kCus);
    const double load = rounds * 16.0 * (mb + nb) * row_bytes / 64.0;
    const double hbm = w_bytes / (paired ? 7000.0 : 6200.0);
    const double start = grid     ? 0.0
                         : paired ? (double)((tiles + 2 * kCus - 1) / (2 * kCus) - 1) * 1100.0
                                  : (rounds - 1.0) * 1500.0;
    const double ns = std::max(load, hbm) + start + 0.02 * load;
    // as good: the more nearly square tile, then the taller one
    const bool tie = ns < best_ns + 1e-6 && (std::min(mb, nb) > std::min(best.mb, best.nb) ||
                                             (std::min(mb, nb) == std::min(best.mb, best.nb) && mb > best.mb));
    if (!best.mb || ns < best_ns - 1e-6 || tie) {
      best = TilePick{mb, nb, grid};
      best_ns = ns;
    }
  };
  for (uint32_t mb : {1u, 2u, 3u, 4u, 5u, 6u, 8u})
    for (uint32_t nb : {1u, 2u, 3u, 4u, 8u})
      if ((bf16 || nb != 3) && (nb != 8 || mb <= 4)) consider(mb, nb, false);
  // (a tile's scale panel is reused two tiles later: the ring must not run
  // further ahead than one tile)
  if (row_bytes / kWalkStep >= 8) {
    consider(8, 8, true);
    consider(12, 8, true);
    if (bf16) consider(16, 8, true);
  }
  return best;
}

// Estimates for the choice between the two kernels, us.  A round is a tile on
// every CU.  128 x 256 tiles: a 128-byte K step and a tile's epilogue take
// what was measured for full, 64- and 32-row tiles, and split parts cost a
// second launch that reads them.  These tiles: a CU's intake (64 KB/us; less
// where the walking kernel is MFMA-bound), or what the eight XCDs' L2s must
// take in where each walks many A rows of few W rows (7 MB/us), the stores
// (15 KB/us a CU) and a start for each round that is not walked.  The rates
// are fits to calls within a factor of 2 of each other on both.  Over 1995
// measured calls (M 1-4096, 41 BF16 shapes with the K split's workspace and
// without, 30 FP8 shapes, K 128-28672) the choice was 0.2 % slower than the
// better kernel on average, more than 12 % in 5.
// Where these tiles were taken always, they lost up to a factor of 2, us 128
// x 256 tiles -> here: BF16 16384 -> 1024 at M 4096 119 -> 257, 12288 -> 4096
// at M 1024 103 -> 118, 7680 -> 2560 at M 1024 52 -> 72; FP8 512 -> 32768 at
// M 4096 170 -> 313, 7168 -> 2048 at M 4096 67 -> 81, 8192 -> 4096 at M 2048
// 76 -> 80.
inline bool BigTilesFaster(bool bf16, uint32_t m, uint32_t n, uint32_t k, uint32_t problems, bool f32_out,
                           const TilePick& t, uint32_t k_splits) {
  const double rb = bf16 ? 2.0 * k : k, osz = f32_out ? 4.0 : 2.0;
  const double w_us = (double)n * problems * rb / 6.2e6;
  auto rounds = [](uint64_t tiles) { return (double)((tiles + kCus - 1) / kCus); };

  const uint32_t rows = DenseTileRows(m, n, problems, k_splits);
  const uint64_t big = (uint64_t)((m + rows - 1) / rows) * ((n + 255) / 256) * problems * k_splits;
  const double step = bf16 ? (rows == 128 ? 0.84 : rows == 64 ? 0.65 : 0.58) : (rows == 128 ? 1.04 : rows == 64 ? 0.79 : 0.62);
  const double end = (bf16 ? 6.3 : 7.0) * (osz == 2.0 || k_splits > 1 ? 1.0 : 1.4);
  double big_us = std::max(3.0 + rounds(big) * (rb / 128.0 / k_splits * step + end), w_us + 2.0);
  if (k_splits > 1) big_us += 1.7 + (double)k_splits * m * n * 4.0 / 3.3e6;

  const uint64_t m_tiles = (m + 16 * t.mb - 1) / (16 * t.mb);
  const uint64_t tiles = m_tiles * (n / (16 * t.nb)) * problems;
  const uint64_t per_xcd = std::min<uint64_t>(32, (tiles + 7) / 8);
  const double load = 16.0 * (t.mb + t.nb) * rb / (t.grid ? (bf16 ? 61e3 : 55e3) : (bf16 ? 65e3 : 63e3));
  const double l2 = 8.0 * 16.0 *
                    (std::min(m_tiles, per_xcd) * t.mb + (per_xcd + m_tiles - 1) / m_tiles * t.nb) * rb / 7e6;
  const double r = rounds(tiles);
  const double us = r * (std::max(load, l2) + 256.0 * t.mb * t.nb * osz / 15e3) + (t.grid ? 0.0 : (r - 1.0) * 2.0);
  return big_us < 2.5 + std::max(us, w_us);
}

// ---- the rules
// e4m3 with UE8M0 scales, shapes that TileGemmTakes: true when they run on
// the tile `t`.  The other kernels keep: up to 8 rows where the work is less
// than the tiles' start-up (K <= 1024, N <= 4096; up to 16 rows of K 512), us
// small-M kernel -> tiles: 512 -> 256 at M 2 2.75 -> 3.15, 512 -> 2048 at M 8
// 3.07 -> 3.31, 1024 -> 4096 at M 1 3.45 -> 3.72 (from N 8192 the tiles win, 512
// -> 7168 at M 8 3.9 -> 3.5), or where the tile would be a walked one (1024 ->
// 129280 at M 1 27 -> 34); and what the 128 x 256 tiles are faster for.  The
// latter only under the code check: without it (the grouped GEMM) they read a
// block under a 0xFF weight scale, and a NaN code in it would show.
inline bool Fp8OnTiles(uint32_t m, uint32_t n, uint32_t k, uint32_t problems, bool f32_out, bool check_codes, bool big,
                       const TilePick& t) {
  const uint64_t cols = (uint64_t)n * problems;
  if (m <= 8 && ((k <= 1024 && cols <= 4096) || t.grid)) return false;
  if (m <= 16 && k <= 512 && cols <= 4096) return false;
  return !(big && check_codes && BigTilesFaster(false, m, n, k, problems, f32_out, t, 1));
}
// whether the 128 x 256 tiles take an FP8 call that the tiles above do not.
// Above 64 rows they also take what the 128 x 128 kernel took before (more
// than 256 rows, or too many 128 x 128 tiles for the small-M kernel) and the
// small-M kernel's 64-row chunks once together they would stream more than 20
// MB of weights (each chunk streams all of W).  At 33..64 rows they also win
// where the small-M kernel's one pass over W (~1.15 TB/s at 64 rows) takes
// longer than a round of big tiles (~0.8 us per 128-deep K step + ~5 us).
// fp32 scales, K -> N at M rows, us before -> after: 4096 -> 1024 M 384 63 ->
// 26; 8192 -> 4096 M 128 56 -> 50, M 256 111 -> 50; 4096 -> 2048 M 512 63 ->
// 28; 1024 -> 32768 M 64 25 -> 16; below those sizes the small-M kernel stays
// faster (4096 -> 1024 at M 256: 16 against 26 us).
inline bool Fp8BigTiles(uint32_t m, uint32_t n, uint32_t k, uint32_t problems) {
  if (BigTileWorthIt(m, n * problems)) return true;
  const uint64_t w_bytes = (uint64_t)n * k * problems;
  if (m > kSmallMChunkRows) {
    const uint64_t chunks = (m + kSmallMChunkRows - 1) / kSmallMChunkRows;
    return m > kSmallMRows || !SmallMTakes(m, n, problems) || chunks * w_bytes > (20ull << 20);
  }
  return m > 32 && w_bytes / 1150 > (uint64_t)(k / 128) * 800 + 5000;  // ns
}

// BF16: very wide weights against 2..255 rows (the LM heads: a round of
// 256-column tiles without a K split) take the 128 x 256 tiles, which stream
// the weights once (twice through L2 above 128 rows) with the batch in one M
// tile, where the GEMV re-reads the batch's rows from L2 for every 16 weight
// rows and the 128 x 128 kernel is MFMA-bound on its small tiles (DeepSeek LM
// head, 4096 -> 129280: m = 2 186 -> 165 us, m = 16 194 -> 170 us, m = 64 177
// us, m = 128 233 -> 186 us; m = 1 stays on the GEMV, 159 us).
inline bool Bf16Wide(uint32_t m, uint32_t n, uint32_t k) {
  return m >= 2 && m < 256 && n % 128 == 0 && k % 64 == 0 && n / 256 >= 192;
}
// Shapes that TileGemmTakes: from two rows up (above 64 only whole 128-column
// groups, as the other kernels take them there).  Left out: very wide weights
// up to 128 rows (HBM-bound on the 128 x 256 tiles: 6.1 TB/s; 129 rows 270 ->
// 242 us here); what the GEMV's blocks have done before these have started, 5
// to 16 rows of N <= 256 and K <= 768 or of N <= 1024 and K <= 256, and up to 32
// of K 128 (us GEMV -> here: 512 -> 256 at M 8 2.5 -> 3.0, 256 -> 1024 at M 8
// 2.45 -> 2.9, 128 -> 1024 at M 8 2.1 -> 2.8; but 768 -> 1024 at M 8 3.7 -> 3.1,
// 1152 -> 256 at M 8 4.0 -> 3.6); and what the 128 x 256 tiles are faster for.
// (K 1024, which the GEMV's waves split evenly: alone and with cold weights 1024
// -> 3072 at M 16 3.85 -> 4.05, but the MLP block of two such calls, SiLU and
// 3072 -> 1024 18.5 -> 17.6.)
inline bool Bf16OnTiles(uint32_t m, uint32_t n, uint32_t k, bool f32_out, bool big, uint32_t k_splits,
                        const TilePick& t) {
  if (m < 2 || (m > 64 && n % 128) || (m <= 128 && Bf16Wide(m, n, k))) return false;
  const bool short_k = (k <= 768 && n <= 256) || (k <= 256 && n <= 1024);
  if ((m >= 5 && m <= 16 && short_k) || (m <= 32 && k == 128)) return false;
  return m <= 64 || !big || !BigTilesFaster(true, m, n, k, 1, f32_out, t, k_splits);
}

// W4A16 (w4a16_tile.hip), count problems of n[i] rows, shapes that it runs (k %
// 512 == 0): the 16-row weight blocks of a tile, or 0 for the GEMV kernels.  By
// measurement (one MI355X, asymmetric, us GEMV -> here; blocks: 16-row weight
// blocks of the launch):
//   K 4096, 384 blocks      m 2   6.1 -> 7.5    m 8   9.2 -> 7.2    m 16  10.1 -> 7.3   m 32  17.2 -> 9.3
//   K 4096, 256 blocks      m 2   4.8 -> 5.9    m 9   5.30 -> 5.55  m 16  5.9 -> 5.6    m 32  9.5 -> 8.0
//   K 4096, 1536 blocks     m 2   15.5 -> 13.1  m 8   16.9 -> 13.7  m 16  18.0 -> 13.8  m 32  49 -> 17.7
//   K 12288, 256 blocks     m 2   8.8 -> 11.9   m 9   11.0 -> 10.5  m 16  12.9 -> 10.9  m 32  21.8 -> 17.0
//   K 2048, 768 blocks      m 2   5.54 -> 6.10  m 4   6.3 -> 6.1    m 16  7.3 -> 6.4    m 32  16.2 -> 8.0
//   K 4096, 16 blocks       m 9   4.96 -> 5.10  m 12  5.08 -> 5.15  m 16  5.32 -> 5.20  m 32  8.7 -> 7.4
//   K 2048, 128 blocks      m 9   4.03 -> 4.08  m 12  3.96 -> 4.37  m 16  4.3 -> 4.3    m 32  6.2 -> 5.7
//   K 3072, 64 blocks       m 9   5.8 -> 4.6    m 16  6.9 -> 4.7    (the GEMV's waves do not split it evenly)
//   K 1024, 192 blocks      m 16  3.95 -> 3.65  m 17  4.09 -> 4.21  m 24  4.33 -> 4.33  m 32  4.1 -> 4.7
//   K 1024, 256 blocks      m 16  11.2 -> 3.7   m 17  4.29 -> 4.38  m 24  4.18 -> 4.64  m 32  4.4 -> 4.8
//   K 512, 256 blocks       m 9   3.13 -> 3.26  m 16  3.30 -> 3.27  m 20  3.56 -> 3.76  m 32  3.81 -> 3.81
// so: never one row; two rows from 1024 blocks on, 3-4 from 512, 5-8 above
// 256; 9-14 above 256, or where K is more than 4096 or the GEMV splits it
// unevenly; 15-16 always; 17-32 above 256 or from K 1536 on.
inline uint32_t W4a16TileBlocks(uint32_t m, uint32_t k, const uint32_t* n, uint32_t count) {
  uint64_t blocks16 = 0;
  for (uint32_t i = 0; i < count; ++i) blocks16 += n[i] / 16;
  if (m < 2 || m > 32) return 0;
  if (m <= 4 ? blocks16 < (m == 2 ? 1024 : 512) : m <= 8 && blocks16 <= 256) return 0;
  if (m >= 9 && m <= 14 && blocks16 <= 256 && (k == 512 || k == 2048 || k == 4096)) return 0;
  if (m >= 17 && blocks16 <= 256 && k <= 1024) return 0;
  // the tile: as PickTile, x rows whole
  const double x_bytes = (m <= 16 ? 16.0 : 32.0) * 2.0 * k, w_bytes = 16.0 * (k / 2);
  uint32_t nb = 0;
  double best = 0.0;
  for (uint32_t c : {1u, 2u, 3u, 4u, 6u}) {
    uint64_t tiles = 0;
    bool fits = true;
    for (uint32_t i = 0; i < count; ++i) {
      fits = fits && n[i] % (16 * c) == 0;
      tiles += n[i] / (16 * c);
    }
    if (!fits) continue;
    const double rounds = (double)((tiles + kCus - 1) / kCus);
    const double load = rounds * (x_bytes + c * w_bytes) / 64.0;
    const double ns = std::max(load, blocks16 * w_bytes / 6200.0) + (rounds - 1.0) * 1500.0 + 0.02 * load;
    if (!nb || ns < best) {
      nb = c;
      best = ns;
    }
  }
  return nb;
}

}  // namespace pih_amd
