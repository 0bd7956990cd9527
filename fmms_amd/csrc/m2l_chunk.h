// m2l_chunk.h — the unit of M2L work: one target's sources [begin, end) in
// the target-sorted directed list.
#pragma once
#include <stdint.h>

namespace fmmh {

struct M2lChunk {
  uint32_t target;
  uint32_t begin;
  uint32_t end;
};

}  // namespace fmmh
