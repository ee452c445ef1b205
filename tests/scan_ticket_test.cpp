// The counter of one-read scans (cutorch_amd/csrc/scan_ticket.hpp) where its tags start again: scans of several chunks, drawn as the
// kernels draw them, from a few tags before the last one on. Every chunk is dealt out once, no tag is 0 (what unwritten words hold),
// and no scan meets a word of the one before it that it would take for its own.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "scan_ticket.hpp"

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)

int main() {
  constexpr uint32_t kMost = 5;
  for (uint32_t first : {1u, 7u, 0xfffffff0u, 0xffffffffu}) {
    uint64_t counter = thc::scan_counter(first);
    uint32_t words[kMost] = {};
    for (int scan = 0; scan < 40; ++scan) {
      const uint32_t chunks = 1 + scan % kMost;
      uint32_t tag = 0;
      for (uint32_t c = 0; c < chunks; ++c) {
        const uint64_t t = counter++;
        CHECK(thc::scan_chunk(t) == c);
        if (c == 0) tag = thc::scan_tag(t);
        CHECK(tag != 0 && thc::scan_tag(t) == tag);
        if (thc::scan_chunk(t) == chunks - 1) counter = thc::next_scan(t);
        for (uint32_t later = c; later < chunks; ++later) CHECK(words[later] != tag);  // nothing there before it is published
        words[c] = tag;
      }
    }
  }
  CHECK(thc::next_scan(thc::scan_counter(0xffffffffu)) == thc::scan_counter(1));
  std::puts("ok");
}
