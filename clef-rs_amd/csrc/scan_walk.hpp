// Launch rule of a ragged scan's carry (plain C++: also compiled on its own by
// the tests).
#pragma once
#include <cstdint>

namespace clef {

// Whether one work-group per (v-head, 16 value columns) walks all sequences'
// chunks in a row (scan_carry MODE 3), instead of one per sequence (MODE 2).
// `groups` = heads x column tiles; a work-group fills a CU.
//
// In a row a batch takes whole rounds of all its chunks, and a sequence
// boundary 0.7 us; by sequence the work-groups fill the CUs as they end, but
// each starts with an empty ring, 4 to 6 us.  In chunks of the walk (f16 1.0
// us, f32 5) that is 0.7 and 4.3 (f16), 0.1 and 1.3 (f32).  So with whole rounds
// (32 heads x 128: 256 work-groups) the walk always wins; where the last round
// is partly empty only over short sequences.  us in a row -> side by side, whole
// scans, 128-wide heads: 40 heads, 16 sequences of 2550 tokens f16 2227 -> 1629,
// f32 6591 -> 4482, of 600 557 -> 457, 1667 -> 1247; 48 heads, 2550 tokens 2211
// -> 1877, 6539 -> 5157; but 40 heads, 64 sequences of 64 tokens f32 747 -> 968.
// With fewer groups than CUs sequences side by side use the idle ones.  The
// lengths are on the device: the sequences are taken as equal, with half-full
// last chunks, a batch of unequal ones as balanced by its longest-first order;
// a predicted gain below 7% is not taken.
inline bool scan_walks_in_a_row(int groups, int cus, int tokens, int nseq, bool f16) {
  if (groups < cus) return false;
  const double chunks = tokens / 64.0 + 0.5 * nseq;
  const double boundary = f16 ? 0.7 : 0.1, start = f16 ? 4.3 : 1.3;
  const auto rounds = [&](int64_t n) { return (double)((n + cus - 1) / cus); };
  return rounds(groups) * (chunks + boundary * nseq) <= 1.07 * rounds((int64_t)groups * nseq) * (chunks / nseq + start);
}

}  // namespace clef
