// m2l_chunk.h — the unit of M2L work: one target's sources [begin, end) in
// the target-sorted directed list; and the sizes of the source rows, which the
// kernels (m2l_kernel.h) and the buffers that hold them (m2l.hip) share.
#pragma once
#include <stdint.h>

#include "common.h"

namespace fmmh {

struct M2lChunk {
  uint32_t target;
  uint32_t begin;
  uint32_t end;
};

// FP64 rows, orders up to 10: the first m2l_row_direct(p) doubles of the real
// layout and the centre are read by each lane, the rest goes through LDS in
// m2l_row_segs(p) segments of 64 bytes (m2l_kernel.h: why the line lies there).
constexpr int m2l_row_direct(int p) { return p == 8 ? 9 : 1; }
constexpr int m2l_row_segs(int p) { return (hdim(p) - m2l_row_direct(p) + 7) / 8; }
constexpr int m2l_row_tail(int p) { return (3 + m2l_row_direct(p) + 7) / 8 * 8; }
constexpr int m2l_row_words(int p) { return 8 * m2l_row_segs(p) + m2l_row_tail(p); }

// Rows of the mixed form, orders 3 to 8 (0 words: none): segments of scaled
// moments, then centre, scale and the first m2l32_row_direct(p) moments.
constexpr bool m2l32_staged(int p) { return p >= 3 && p <= 8; }
constexpr int m2l32_row_segs(int p) { return (hnpos(p) - 2) / 8; }
constexpr int m2l32_row_direct(int p) { return hnpos(p) - 8 * m2l32_row_segs(p); }
constexpr int m2l32_row_words(int p) {
  return m2l32_staged(p) ? (m2l32_row_segs(p) * 8 + 4 + m2l32_row_direct(p) + 7) / 8 * 8 : 0;
}

}  // namespace fmmh
