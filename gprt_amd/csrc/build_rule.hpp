// How the primitives of a build are cut into tiles and their keys sorted with the automatic configuration
// (host code, no HIP).
#pragma once

#include <algorithm>
#include <cstdint>

namespace gprt {

// The automatic tile size. Bounds, keys and sort passes run one workgroup per tile, so few primitives
// want small tiles, that every CU gets one, and batches of small meshes, that their tiles are not mostly
// empty; large meshes want large ones, for fewer look-back steps. One mesh of n triangles, us, with tiles of
// 2,048 / 4,096 / 8,192 / 16,384: 16,384: 92 / 104 / 118 / 138, 200,000: 126 / 135 / 148 / 185, 500,000:
// 159 / 157 / 168 / 198, 1 million: 236 / 212 / 205 / 237, 2 million: 367 / 317 / 288 / 314, 3 million: 501 /
// 429 / 399 / 388. A thousand meshes of 970 on average: 421 / 468 / 607 / 914, of 9,400: 1372 / 1285 / 1387 /
// 1687; 64 of 65,536 with their top level: 2594 / 2433 / 2323 / 2281. Three hundred alike, with tiles of 4,096 /
// 8,192: of 12,000 435 / 488, of 13,000 537 / 496 (four tiles of 4,096 or two of 8,192), of 15,000 538 / 511.
template <class Size>
inline int auto_tile_keys(uint32_t meshes, Size size) {
  uint64_t prims = 0;
  for (uint32_t m = 0; m < meshes; ++m) prims += size(m);
  const uint64_t mean = prims / meshes;
  if (prims <= 384u << 10 || mean < 2048) return 2048;
  if (prims <= 768u << 10 || mean <= 12288) return 4096;
  return mean < 5u << 19 ? 8192 : 16384;
}

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
