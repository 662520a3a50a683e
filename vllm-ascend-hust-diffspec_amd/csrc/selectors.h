// Row selectors of the single-launch retrieval step (host arithmetic only).
#pragma once

#include <algorithm>
#include <cstdint>

namespace ds355 {

// Row selectors (fewer when the batch has fewer rows).  8 against 16, events
// around each launch, two rounds: 16 rows of 4k-40k tokens 82.5-82.7 against
// 82.8-83.4 us (other seeds 0.3-1.4 us faster), 16 x 40k 156.2-156.4
// against 157.1-157.6 us, 64 rows equal or faster.  A selector's rows
// complete tens of microseconds apart, and the freed slots score.  4
// selectors: 0.5-0.9 us slower on the first draw, up to 1 us faster on
// others; 2: 25-45% slower on ragged rows (selections queue).
constexpr int kSelectors = 8;
// Short rows complete together, and then the selections queue: a selector
// takes about 5 us a row, in which 256 CUs stream about 27 MB of keys, 108 KB
// each.  So a batch whose score buffer holds few keys gets enough selectors
// for its selections to take no longer than its scoring, at most one per 4
// CUs (a workgroup that selects does not score: a twelfth of the resident
// ones; a device of 32 CUs keeps to kSelectors).  us with 8 / as many as rows /
// this rule: 36 rows of 1.7k tokens (16/2 heads x 64) 48.6 / 27.6 / 27.7,
// 11 rows of 469-1591 23.9 / 18.5 / 18.5, 16 rows of 1-2k (32/4 x 128) 32.8 /
// 32.1 / 32.9; but 64 rows of 1-4k 122.3 / 126.6, 16 x 40k 147.5 / 150.5:
// workgroups that only wait lengthen the scoring there.  (Counted from the
// rows' own lengths on the device instead, every launch was 1-3 us slower.)
// The rule sees the score buffer's width, not the rows' lengths: short rows in
// a buffer made for long ones get kSelectors.
constexpr int kCusPerSelector = 4;
constexpr int64_t kBytesPerSelectionCu = int64_t{108} << 10;

// Selectors for `rows` rows whose score buffer holds `key_bytes` of keys on a
// device of `cus` compute units.
inline int row_selectors(int rows, int64_t key_bytes, int cus) {
  const int64_t want = rows * (kBytesPerSelectionCu * cus) / std::max<int64_t>(1, key_bytes);
  const int most = std::max(kSelectors, cus / kCusPerSelector);
  return std::min(rows, static_cast<int>(std::max<int64_t>(kSelectors, std::min<int64_t>(want, most))));
}

}  // namespace ds355
