// How the keys of a build are sorted with the automatic configuration (host code, no HIP).
#pragma once

#include <algorithm>
#include <cstdint>

namespace gprt {

// Workgroups per tile of the sort by ranks (one for each 64 keys of the largest mesh in a tile), or 0 for
// the digit passes.
//
// Ranks cost comparisons, of which they do up to 2^27, one mesh of 11,585 primitives. A build, us, by the
// digit passes and by ranks: 500 triangles 62 / 43, 2,000 74 / 59, 5,000 85 / 67, 10,000 88 / 79, 16,384
// 93 / 92, 20,000 92 / 130; 16 meshes of up to 4,096 92 / 77, 300 of them 191 / 275.
//
// Every tile gets the same number of workgroups, so small meshes beside a large one launch idle ones: 2.6 us
// per thousand, where the passes cost 12 us and 50 per thousand tiles. Hence at most 16 idle ones a tile and
// 8,192. Passes / ranks: 1,000 meshes of 8 primitives 193 / 133, 4,096 of 8 to 150 716 / 544, 65,500 of 8
// 9,434 / 6,939, 600 and 2,000 of 64 378 / 295, 2,000 and 500 of 8 135 / 128; not taken: 2,000 and 1,000 of 8
// 216 / 222, 8,000 and 4,000 of 8 635 / 741. A launch holds fewer than 2^32 threads, 2^22 workgroups of 1,024.
constexpr uint64_t kRankPairs = 1ull << 27;
constexpr uint64_t kRankIdlePerTile = 16, kRankIdle = 8192;
constexpr uint64_t kRankGroups = 1ull << 21;

template <class Size>
inline uint32_t rank_groups(uint32_t meshes, uint32_t tileKeys, Size size) {
  uint64_t pairs = 0, tiles = 0, largest = 0, busy = 0;
  for (uint32_t m = 0; m < meshes; ++m) {
    const uint64_t n = size(m);
    pairs += n * n;
    tiles += (n + tileKeys - 1) / tileKeys;
    busy += (n + 63) / 64;
    largest = std::max(largest, n);
  }
  const uint64_t perTile = (std::min<uint64_t>(largest, tileKeys) + 63) / 64, groups = tiles * perTile;
  const bool few = groups <= kRankGroups && groups - busy <= kRankIdlePerTile * tiles + kRankIdle;
  return pairs <= kRankPairs && few ? (uint32_t)perTile : 0u;
}

}  // namespace gprt
