// How a CC pair's grid is cut into blocks, and the grids that fw_cc_pair_noalloc takes. Plain integers, so
// that the rules are checked on the host.
#pragma once

#include <algorithm>

namespace fw::hip {

constexpr int kCcTileX = 32, kCcTileY = 8;        // a CC block's columns and rows
constexpr int kCcTileZ = 16, kCcMinBlocks = 512;  // where the tuning table sets only the other knob
constexpr long long kCcCus = 256, kCcMostBlocks = 8192;

inline long long cc_columns(int nx, int ny) {
  return (long long)((nx + kCcTileX - 1) / kCcTileX) * ((ny + kCcTileY - 1) / kCcTileY);
}

// The longest run of max_tile, max_tile / 2, ..., 1 planes that cuts `columns` columns of nz planes into
// at least min_blocks blocks.
inline int halved_run(long long columns, int nz, int max_tile, int min_blocks) {
  int t = std::max(1, max_tile);
  while (t > 1 && columns * ((nz + t - 1) / t) < std::max(1, min_blocks)) t /= 2;
  return t;
}

// The z run of a CC block. With a choice of the tuning table: halved_run of max_tile. By default (max_tile
// 0) the run that takes the least time: a block walks tile_z + 2R planes one after another, a CU holds two
// blocks (187 registers at radius 4), and a plane takes a pair of blocks kCcPairTime times a block alone
// (both are bound by f64 arithmetic for most of it).
constexpr double kCcPairTime = 1.5;
inline int cc_run(int nx, int ny, int nz, int radius, int max_tile, int min_blocks) {
  const long long tiles = cc_columns(nx, ny);
  if (max_tile > 0) return halved_run(tiles, nz, max_tile, min_blocks);
  int best = nz;
  double least = 1e300;
  // at most kCcMostBlocks blocks, beyond one a tile
  for (long long chunks = 1; chunks <= nz && (chunks == 1 || chunks * tiles <= kCcMostBlocks); ++chunks) {
    const int t = (int)((nz + chunks - 1) / chunks);
    const long long per_cu = (tiles * ((nz + t - 1) / t) + kCcCus - 1) / kCcCus;
    const double time = double(t + 2 * radius) * (double(per_cu / 2) * kCcPairTime + double(per_cu % 2));
    if (time < least) {
      least = time;
      best = t;
    }
  }
  return best;
}

// What fw_cc_pair_noalloc takes, whatever the blocks of the kernel behind it: at most kNoAllocMaxUnits
// units of 64 x 8 columns over a z run, cut as halved_run cuts it with the tuning table's knobs cc.tile_z
// and cc.min_blocks (0 where it sets none: 16 planes, 512 units). On grids of 2^22 to 2^23 - 1 voxels a
// table without these knobs counts as 64 planes, 256 units, which the shipped table held when callers first met
// the limit: what was taken is still taken. 182 x 218 x 182 has 504 units, 1024 x 1024 x 128 has 16,384.
constexpr long long kNoAllocMaxUnits = 16384;
inline long long noalloc_units(int nx, int ny, int nz, int tile_knob, int blocks_knob) {
  const long long n = (long long)nx * ny * nz;
  const bool neither = tile_knob == 0 && blocks_knob == 0;
  const bool mid = neither && n >= (1ll << 22) && n < (1ll << 23);
  const long long columns = (long long)((nx + 63) / 64) * ((ny + 7) / 8);
  const int t = halved_run(columns, nz, mid ? 64 : tile_knob ? tile_knob : kCcTileZ,
                           mid ? 256 : blocks_knob ? blocks_knob : kCcMinBlocks);
  return columns * ((nz + t - 1) / t);
}

// The CC blocks of any grid within that limit: two a unit (one for each half of its columns) where the
// table sets the run, and by the default rule at most kCcMostBlocks, or one a column of tiles.
constexpr int kNoAllocMaxBlocks = 2 * int(kNoAllocMaxUnits);
static_assert(kCcMostBlocks <= kNoAllocMaxBlocks, "the scratch holds every default z split");

}  // namespace fw::hip
