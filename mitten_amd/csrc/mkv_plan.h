// Piece boundaries of a decode plan (host only, no HIP).
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace mkv {

constexpr int kPieceBlocks = 64;        // most blocks of a piece (one per lane)
constexpr int kBlockWeight = 8;         // weight of one block in a piece ...
constexpr int kSwitchWeight = 12;       // ... and of a sequence start inside it (about 1.5 blocks)
constexpr int kFirstRoundWeight = 116;  // cap of the first-dispatched pieces, percent
constexpr int kOddXcdWeight = 96;       // cap of pieces dealt to odd-numbered XCDs, percent

// A greedy fill of the flattened blocks of B sequences (sequence b: blocks
// blk0[b] .. blk0[b + 1], at least one) under a weight cap per piece. A block
// weighs kBlockWeight; a sequence that starts inside a piece (not at its first
// block) adds kSwitchWeight. A piece takes at least one block and at most
// kPieceBlocks. Pieces below `first` have kFirstRoundWeight percent of the
// cap; with odd_light, odd ones kOddXcdWeight percent of theirs. f0s receives
// each piece's first block, then the total. Whole runs of a sequence's blocks
// are taken at once: the cost is the number of sequences and pieces, not of
// blocks (a plan tries about a dozen caps; block by block that was 0.4 ms of
// host time per step at 64 sequences of 1-8k tokens).
inline void cut_pieces(const int32_t *blk0, int32_t B, int64_t cap, int64_t first, bool odd_light,
                       std::vector<int32_t> &f0s) {
  f0s.clear();
  const int64_t total = blk0[B];
  int32_t b = 0;
  for (int64_t f = 0; f < total;) {
    const int64_t idx = (int64_t)f0s.size();
    f0s.push_back((int32_t)f);
    const int64_t cq0 = idx < first ? cap * kFirstRoundWeight / 100 : cap;
    const int64_t cq = odd_light && (idx & 1) ? cq0 * kOddXcdWeight / 100 : cq0;
    while (blk0[b + 1] <= f) b++;
    int64_t w = kBlockWeight, cnt = 1;
    f++;
    for (;;) {
      const int64_t room = cq > w ? (cq - w) / kBlockWeight : 0;
      const int64_t take = std::min({(int64_t)blk0[b + 1] - f, kPieceBlocks - cnt, room});
      f += take;
      cnt += take;
      w += take * kBlockWeight;
      // The piece ends inside the sequence, at the last block, or where the
      // next sequence's first block does not fit.
      if (f < blk0[b + 1] || f == total || cnt == kPieceBlocks || w + kBlockWeight + kSwitchWeight > cq) break;
      b++;
      f++;
      cnt++;
      w += kBlockWeight + kSwitchWeight;
    }
  }
  f0s.push_back((int32_t)total);
}

}  // namespace mkv
