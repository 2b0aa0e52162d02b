// How a tree level's samples are cut into work items of the histogram kernel
// and dealt to the XCDs (host side; no HIP).
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace pd {
namespace engine {

// Samples per work item of a level of level_samples samples with nF candidates
// (ftiles tiles) and nT thresholds, nC classes, on cus CUs.
//  * blocks_per_cu items a CU, or
//  * at least 1024 samples an item (shorter ones pay for the candidate set-up and
//    the histogram flush), down to 64 where the level would otherwise leave CUs
//    without two items: a wave walks its samples one after the other, so a level
//    of few items lasts as long as one of them (8192 samples x 100 candidates, 10
//    thresholds, 4 classes: 92 us a level in 16 items of 1024, 17 us in 256 of 64),
//    unless the flush eats that up: every item of a node cut in several adds its
//    counts into the node's histogram, nF nT nC atomics for all tiles of a chunk at
//    about 18 ps, a sample of an item lasts 78 ns, and level_samples / c chunks of c
//    samples are the shortest at c = sqrt(level_samples nF nT nC 18 ps / 78 ns).
//    4000 samples x 4000 candidates, 32 thresholds, 16 classes: the first two levels
//    0.61 ms in items of 1024, 1.01 in items of 492; 2000 samples x 2000, 20, 8: a
//    tree's histograms 0.41 ms in items of 395, 0.60 in items of 125.
// A level launched node by node (launches of them) waits for every node's items in
// turn: c is the shortest for the mean node.
inline uint32_t item_chunk(uint64_t level_samples, uint32_t nF, uint32_t ftiles, uint32_t nT, uint32_t nC,
                           uint32_t cus, uint32_t blocks_per_cu, uint32_t launches = 1)
{
  const uint64_t target_blocks = (uint64_t)cus * blocks_per_cu;
  uint64_t c = (level_samples * ftiles + target_blocks - 1) / target_blocks;
  const uint64_t two_per_cu = level_samples * ftiles / (2u * (uint64_t)cus);
  const uint64_t flush = (uint64_t)(std::sqrt((double)level_samples / launches * nF * nT * nC) / 64.0);
  c = std::max<uint64_t>(c, std::min<uint64_t>(std::max<uint64_t>({two_per_cu, flush, 64u}), 1024u));
  return (uint32_t)std::min<uint64_t>(c, 32768u);
}

}  // namespace engine
}  // namespace pd
