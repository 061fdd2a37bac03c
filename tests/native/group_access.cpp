// Runs the kernels' group accesses (csrc/sr_group_access.h) on the host, at
// every start of a group that a view can have: groups of four elements of 4,
// 2 and 1 bytes from any element of a buffer, with the bytes around the group
// kept.  The functions are out of line, so that the addresses are unknown
// where the accesses are compiled: an access that promises more alignment
// than the address has then faults where the CPU checks it (16 bytes), and
// test_group_access.py reads the promised alignments of all widths.
#include <cstdint>
#include <cstdio>
#include <cstring>

#include "sr_group_access.h"

namespace {

template <int BYTES, bool kCached>
__attribute__((noinline)) void load(const char* from, uint32_t* words) {
  sr::load_words<BYTES, kCached>(from, words);
}

template <int BYTES>
__attribute__((noinline)) void store(char* to, const uint32_t* words) {
  sr::store_words<BYTES>(to, words);
}

template <int BYTES, bool kCached>
int moves() {
  constexpr int kElement = BYTES / 4;
  alignas(64) char from[128], to[128];
  int failures = 0;
  for (int start = 0; start < 64; start += kElement) {
    for (int i = 0; i < 128; ++i) from[i] = static_cast<char>(3 * i + 1), to[i] = static_cast<char>(i);
    uint32_t words[4] = {};
    load<BYTES, kCached>(from + start, words);
    store<BYTES>(to + start, words);
    if (std::memcmp(words, from + start, BYTES)) ++failures;
    for (int i = 0; i < 128; ++i) {
      const bool written = i >= start && i < start + BYTES;
      if (to[i] != static_cast<char>(written ? 3 * i + 1 : i)) ++failures;
    }
  }
  return failures;
}

}  // namespace

int main() {
  const int failures = moves<16, false>() + moves<16, true>() + moves<8, false>() + moves<4, false>();
  std::printf("%d failures\n", failures);
  return failures != 0;
}
