// How a CC pair's grid is cut into blocks, and the grids that fw_cc_pair_noalloc takes. Plain integers, so
// that the rules are checked on the host.
#pragma once

#include <algorithm>
#include <cstddef>

namespace fw::hip {

constexpr int kCcTileX = 32, kCcTileY = 8;        // a CC block's columns and rows
constexpr int kCcTileZ = 16, kCcMinBlocks = 512;  // where the tuning table sets only the other knob
constexpr long long kCcCus = 256, kCcMostBlocks = 8192;
// runs of a column, so that a batch's columns stay below the 65,536 blocks that a launch may have along z
constexpr long long kCcMostRuns = 2048;

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

// The time of `blocks` blocks of k_cc2 of one run on a CU, in units of a block alone. Its registers let two
// run beside each other, three up to radius 3, four at radius 1; a second block adds 0.3, each further one
// 0.25 (256 x 64 x 64 n grids in runs of 16 planes, launch taken off: 1 to 4 blocks a CU take 24, 31, 37, 43 us
// at radius 1, 28, 36, 43, 64 at radius 2, 37, 49, 81, 94 at radius 4).
inline double cc_cu_time(long long blocks, int radius) {
  constexpr double beside[5] = {0.0, 1.0, 1.3, 1.55, 1.8};
  const int fit = radius == 1 ? 4 : radius <= 3 ? 3 : 2;
  return double(blocks / fit) * beside[fit] + beside[blocks % fit];
}

// The z run of a block of k_cc2 (which walks its planes one after another). With a choice of the tuning
// table: halved_run of max_tile. By default (max_tile 0) the run that takes the least time: a block walks
// tile_z + 2R planes, and the fullest CU takes cc_cu_time.
inline int cc_run(int nx, int ny, int nz, int radius, int max_tile, int min_blocks) {
  const long long tiles = cc_columns(nx, ny);
  if (max_tile > 0) return halved_run(tiles, nz, max_tile, min_blocks);
  int best = nz;
  double least = 1e300;
  // at most kCcMostBlocks blocks, beyond one a tile
  const long long most = std::min({(long long)nz, kCcMostRuns, std::max<long long>(1, kCcMostBlocks / tiles)});
  for (long long chunks = 1; chunks <= most; ++chunks) {
    const int t = (int)((nz + chunks - 1) / chunks);
    const long long per_cu = (tiles * ((nz + t - 1) / t) + kCcCus - 1) / kCcCus;
    const double time = double(t + 2 * radius) * cc_cu_time(per_cu, radius);
    if (time < least) {
      least = time;
      best = t;
    }
  }
  return best;
}

// A CC pair's launch: k_cc2 over runs of planes, or k_cc2_plane, which computes every plane of its run by
// itself.
struct CcPlan {
  int run;
  bool plane;
};

// On oblique grids k_cc2 is there from these radii on, without and with a mask. Below them k_cc2_plane is
// the faster one on every grid (k_cc2's gathers spill beside the windows' registers): 182 x 218 x 182 at
// radius 4 takes 398 us for 510, radius 6 536 for 600, radius 3 with a mask 420 for 647. From them on
// k_cc2 is faster on large grids: radius 7 640 us for 655, radius 5 with a mask 607 for 692.
constexpr int kCcObliquePlain = 7, kCcObliqueMasked = 4;

// The planes of 32 x 8 tiles up to which k_cc2_plane is taken. A block of k_cc2 walks 2R planes beyond its
// run, one after another, which pays where the run is long; k_cc2_plane reads every plane of the window
// for each plane it computes, all loads at once. Plain, radius 4: 24 x 28 x 24 (96 planes) 7.9 us for
// 15.8, 45 x 54 x 45 (630) 11.6 for 19, 96 x 112 x 96 (4,032) 37 for 42, 112^3 (6,272) 49 for 48, 256 x 256 x 24
// (6,144) 50 for 43. Up to radius 3 three blocks of k_cc2 fit a CU, and the line lies lower: radius 3 at
// 2,400 planes 21 for 28, at 4,032 32 for 31, at 6,144 42 for 38. With a mask k_cc2_plane's lanes carry a third
// load and a count: radius 6 at 1,024 planes 33 for 44, at 2,000 51 for 52, at 2,400 62 for 57.
constexpr long long kCcPlanes = 4096, kCcPlanesSmallRadius = 3072, kCcPlanesMasked = 2048;

inline CcPlan cc_plan(int nx, int ny, int nz, int radius, bool masked, bool diagonal, int tile_knob, int blocks_knob) {
  const bool walks = diagonal || radius >= (masked ? kCcObliqueMasked : kCcObliquePlain);
  if (tile_knob != 0 || blocks_knob != 0)
    return {cc_run(nx, ny, nz, radius, tile_knob ? tile_knob : kCcTileZ, blocks_knob ? blocks_knob : kCcMinBlocks), !walks};
  const long long tiles = cc_columns(nx, ny);
  const long long line = !diagonal ? kCcPlanes : masked ? kCcPlanesMasked : radius <= 3 ? kCcPlanesSmallRadius : kCcPlanes;
  if (walks && tiles * nz > line) return {cc_run(nx, ny, nz, radius, 0, 0), false};
  const long long chunks = std::min({(long long)nz, kCcMostRuns, std::max<long long>(1, kCcMostBlocks / tiles)});
  return {int((nz + chunks - 1) / chunks), true};
}

// The sum of a pair's block partials, in an order that a block of kCcLanes threads adds as well: lane t takes
// blocks t, t + kCcLanes, ..., then halves of the lanes are added to each other. (On one thread in block
// order a pair of 630 blocks took 22 us in all on the device; this way it takes 13.)
constexpr int kCcLanes = 256;
struct CcTotal {
  double cc;
  long long count;
};
inline CcTotal cc_total(const float* cc, const int* count, size_t blocks) {
  double lane[kCcLanes] = {};
  long long counted = 0;
  for (size_t b = 0; b < blocks; ++b) {
    lane[b % kCcLanes] += double(cc[b]);
    counted += count[b];
  }
  for (int half = kCcLanes / 2; half > 0; half /= 2)
    for (int t = 0; t < half; ++t) lane[t] += lane[t + half];
  return {lane[0], counted};
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
// table sets the run, and by the default rules at most kCcMostBlocks, or one a column of tiles.
constexpr int kNoAllocMaxBlocks = 2 * int(kNoAllocMaxUnits);
static_assert(kCcMostBlocks <= kNoAllocMaxBlocks, "the scratch holds every default z split");

}  // namespace fw::hip
