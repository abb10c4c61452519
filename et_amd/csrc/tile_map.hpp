// The order in which a product's workgroups take the tiles of its output, for the
// kernels with 256-row tiles (gemm_residue.hip, gemm_bf16.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "common.hpp"

namespace etg {

constexpr int kTileM = 256;                   // output rows of a tile
constexpr int kXcds = 8;
constexpr int kGroupM = 8;                    // row tiles of a group

// The tiles of one launch.  A slot is a tile's place in the order of work (groups of
// row tiles, in each column tile by column tile) and in the array of residues.  Of a
// lower block triangle (Gemm::lower) a group holds the column tiles that its last row
// needs; the few above the diagonal among them do nothing.  Cut into sixteen column
// pieces instead, each from its first row on, a triangle of 5776 rows (k = 1270) took
// 16 launches of 1035 workgroups and fewer, two or three rounds of the chip each: 0.60
// ms against 0.35.  At 23104 rows both run at the kernel's rate (9.5 ms).
constexpr int kMaxGroups = 64;
struct TileMap {
  int tiles_m, tiles_n, tile_n;
  int64_t lower, row0, col0;       // of the product's output, for the triangle
  int group, groups, count;        // row tiles of a group; slots
  uint32_t first[kMaxGroups];      // first slot of each group
};

// Tile of a slot; false: nothing to do.  Called by whole wavefronts.
__device__ inline bool tile_of(const TileMap& t, int slot, int& tm, int& tn) {
  if (t.lower == 0) {
    const int group = kGroupM * t.tiles_n;
    const int first_m = (slot / group) * kGroupM;
    const int gsize = min(t.tiles_m - first_m, kGroupM);
    tm = first_m + (slot % group) % gsize;
    tn = (slot % group) / gsize;
    return true;
  }
  const int lane = threadIdx.x & 63;
  const uint32_t f = lane < t.groups ? t.first[lane] : ~0u;
  const int g = __popcll(__ballot(uint32_t(slot) >= f)) - 1;
  const int first_m = g * t.group;
  const int gsize = min(t.tiles_m - first_m, t.group);
  const int l = slot - __builtin_amdgcn_readlane(int(f), g);
  tm = first_m + l % gsize;
  tn = l / gsize;
  return t.row0 + (tm + 1) * int64_t(kTileM) > (t.col0 + tn * int64_t(t.tile_n)) / t.lower * t.lower;
}

// Slot of a workgroup: contiguous ranges of slots per XCD (their tiles share an L2).
__device__ inline int slot_of(int bid, int nb) {
  const int per = nb / kXcds, rem = nb % kXcds;
  const int xcd = bid % kXcds, idx = bid / kXcds;
  return (xcd < rem) ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
}

inline TileMap map_tiles(int64_t m, int64_t n, int tile_n, int64_t lower, int64_t row0, int64_t col0) {
  TileMap t{};
  t.tiles_m = int(ceil_div(m, kTileM));
  t.tiles_n = int(ceil_div(n, tile_n));
  t.tile_n = tile_n;
  t.lower = lower;
  t.row0 = row0;
  t.col0 = col0;
  if (lower == 0) {
    t.count = t.tiles_m * t.tiles_n;
    return t;
  }
  t.group = std::max(kGroupM, int(ceil_div(t.tiles_m, kMaxGroups)));
  t.groups = int(ceil_div(t.tiles_m, t.group));
  for (int g = 0; g < t.groups; ++g) {
    const int64_t end = std::min(t.tiles_m, (g + 1) * t.group);          // first row tile after the group
    // its last row needs the columns before the end of that row's block
    const int64_t columns = ceil_div(row0 + end * kTileM, lower) * lower - col0;
    t.first[g] = uint32_t(t.count);
    t.count += int(end - g * t.group) * int(std::clamp<int64_t>(ceil_div(columns, tile_n), 0, t.tiles_n));
  }
  return t;
}

}  // namespace etg
