// dense_route.hpp behind a C interface, for test_dense_route.py
#include "dense_route.hpp"

using namespace pih_amd;

extern "C" {
// mb | nb << 8 | grid << 16
uint32_t pick_tile(uint32_t bf16, uint32_t m, uint32_t n, uint32_t k, uint32_t problems) {
  const TilePick t = PickTile(bf16 != 0, m, n, bf16 ? 2 * k : k, problems);
  return t.mb | t.nb << 8 | (uint32_t)t.grid << 16;
}
uint32_t fp8_on_tiles(uint32_t m, uint32_t n, uint32_t k, uint32_t problems, uint32_t f32_out, uint32_t check_codes) {
  return Fp8OnTiles(m, n, k, problems, f32_out != 0, check_codes != 0, Fp8BigTiles(m, n, k, problems),
                    PickTile(false, m, n, k, problems));
}
// with the queried workspace, or without one
uint32_t bf16_on_tiles(uint32_t m, uint32_t n, uint32_t k, uint32_t f32_out, uint32_t workspace) {
  return Bf16OnTiles(m, n, k, f32_out != 0, Bf16BigTiles(m, n, k) || Bf16Wide(m, n, k),
                     workspace ? DenseKSplits(m, n, k / 64) : 1, PickTile(true, m, n, 2 * k, 1));
}
uint32_t w4a16_blocks(uint32_t m, uint32_t k, const uint32_t* n, uint32_t count) { return W4a16TileBlocks(m, k, n, count); }
}
