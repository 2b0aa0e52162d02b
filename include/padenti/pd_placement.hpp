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

// First record of chunk k of a node whose n records begin at `begin` and are cut
// into `chunks` (k = chunks: the node's end).  Shares are equal, their boundaries
// moved down to a 64-byte line of the record list (4 records of 16 bytes; a share
// is at most 3 records longer for it): the waves of a block walk neighbouring
// records through the scalar cache, and a chunk that begins inside a line makes
// every step of its block touch one line more.  5000 images, 10 M samples, 4000 x 32
// candidates: the histograms of a 20-level tree 2.42 s cut at any record, 2.30 on
// lines; node by node the first seven levels 1.10 and 0.95 s (boundaries at multiples
// of 16 or 32 records: the same).
inline uint32_t chunk_begin(uint32_t begin, uint32_t n, uint32_t chunks, uint32_t k)
{
  if (k == 0u || k == chunks) return k ? begin + n : begin;
  return (uint32_t)((begin + (uint64_t)n * k / chunks) & ~(uint64_t)3);
}

// Launch order of a level's groups (a chunk of a node's samples with all its
// tiles) and the XCD of each.
//
// Groups run in node order, except that the smallest ones (a tenth of the samples
// together) come last, largest first, so that a level does not end on a long
// block; each goes to the XCD with the fewest samples so far.  Dealt round robin,
// one of 47 random-sized groups an XCD is some 8% above the mean; sorted by size
// throughout, the blocks resident on a CU run their gather-bound and their split
// phases at the same time.  351 nodes of 500..6000 samples, 2000 x 20 candidates:
// 5.7 -> 5.2 ms a level, 968 nodes 7.6 -> 6.8 ms (round robin -> this); sorted by
// size throughout, the histograms of a 16-level tree took 77.7 ms instead of 73.2
// (round robin 75.0).
//
// The launch interleaves the XCDs' lists and pads the shorter ones, so its items
// are the longest list's times the XCDs.  By samples alone, 7 groups of 30000 and
// 350 of 20 would put all of the latter on the eighth XCD, 2800 rows of items for
// 357 groups: an XCD takes at most a quarter more groups than its share.
struct GroupOrder {
  std::vector<uint32_t> order;   // groups in launch order
  std::vector<uint32_t> xcd;     // of each group
  size_t rows = 0;               // groups of the XCD that has most
};

inline GroupOrder deal_groups(const std::vector<uint32_t> &samples, uint32_t n_xcc)
{
  const size_t X = n_xcc, ng = samples.size(), share = (ng + X - 1) / X, most = share + share / 4 + 1;
  GroupOrder r;
  r.order.resize(ng);
  r.xcd.resize(ng);
  for (size_t g = 0; g < ng; g++) r.order[g] = (uint32_t)g;
  uint64_t all = 0;
  for (uint32_t n : samples) all += n;
  std::vector<uint32_t> by_size(r.order);
  std::stable_sort(by_size.begin(), by_size.end(), [&](uint32_t x, uint32_t y) { return samples[x] > samples[y]; });
  uint64_t rest = 0;
  size_t cut = ng;   // by_size[cut..) come last
  while (cut > 0 && rest + samples[by_size[cut - 1]] <= all / 10) rest += samples[by_size[--cut]];
  std::vector<uint8_t> last(ng, 0);
  for (size_t i = cut; i < ng; i++) last[by_size[i]] = 1;
  size_t w = 0;
  for (size_t g = 0; g < ng; g++)
    if (!last[g]) r.order[w++] = (uint32_t)g;
  std::copy(by_size.begin() + cut, by_size.end(), r.order.begin() + w);
  std::vector<uint64_t> load(X, 0);
  std::vector<size_t> len(X, 0);
  for (uint32_t g : r.order) {
    size_t x = X;
    for (size_t i = 0; i < X; i++)
      if (len[i] < most && (x == X || load[i] < load[x])) x = i;
    r.xcd[g] = (uint32_t)x;
    load[x] += samples[g] + 64u;   // (a block costs something without samples too)
    r.rows = std::max(r.rows, ++len[x]);
  }
  return r;
}

}  // namespace engine
}  // namespace pd
