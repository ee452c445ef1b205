// The counter that deals out the chunks of one-read scans: (tag << 32) | chunks drawn. A scan's workgroups draw its chunks from
// it in order; whoever draws the last one sets the counter up for the next scan of the stream, under the next tag.
// No tag is 0, which the words that scans publish hold at first, and no two scans in a row have the same: tags go from 1 to
// 2^32 - 1 and start again. A word that nobody has written since the scan 2^32 - 1 before would be taken for a new one.
#pragma once
#include <cstdint>

namespace thc {

constexpr uint64_t scan_counter(uint32_t tag) { return (uint64_t)tag << 32; }
constexpr uint32_t scan_tag(uint64_t counter) { return (uint32_t)(counter >> 32); }
constexpr uint32_t scan_chunk(uint64_t counter) { return (uint32_t)counter; }
constexpr uint64_t next_scan(uint64_t counter) {
  return scan_counter(scan_tag(counter) == 0xffffffffu ? 1u : scan_tag(counter) + 1u);
}

}  // namespace thc
