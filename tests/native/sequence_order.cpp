// Checks the grid of launches in sequence (csrc/sr_tile_order.h) on the host:
// sequence_shape covers every tile exactly once, each dimension within its
// work-item limit and fewer than one row of padding, and workgroup numbers
// stay within 32 bits; use_sequence starts at its element count for every
// workgroup size; workgroups_in keeps within its largest cap.
#include <cstdint>
#include <cstdio>
#include <initializer_list>

#include "sr_tile_order.h"

int main() {
  int failures = 0, shapes = 0;
  for (uint32_t tiles : {1u, 63u, 20480u, 33554431u, 33554432u, 33556480u, 0x7FFFF000u}) {
    for (uint32_t block : {64u, 128u, 256u, 512u, 1024u}) {
      for (uint64_t limit : {1ull << 16, 1ull << 24, 0xFFFFFFFFull}) {
        const sr::LaunchShape shape = sr::sequence_shape(tiles, block, limit);
        const uint64_t total = static_cast<uint64_t>(shape.x) * shape.y;
        ++shapes;
        // Workgroup b takes tile b, so covering [0, tiles) is total >= tiles.
        if (total < tiles || total - tiles >= shape.x || static_cast<uint64_t>(shape.x) * block > limit ||
            total >= (1ull << 32)) {
          std::printf("tiles %u block %u limit %llu: %u x %u\n", tiles, block, (unsigned long long)limit, shape.x,
                      shape.y);
          ++failures;
        }
      }
    }
  }
  // The least elements, each side of the edge: moments that round
  // stochastically to FP16 or FP8, bytes per element, edge.
  const uint32_t edges[][3] = {{0, 10, 5u << 21}, {0, 12, 5u << 21}, {0, 14, 13u << 21}, {0, 22, 13u << 21},
                               {1, 12, 5u << 21}, {1, 14, 5u << 21}, {1, 16, 13u << 21}, {2, 14, 5u << 21},
                               {2, 16, 13u << 21}};
  for (uint32_t block : {128u, 256u, 512u, 1024u}) {
    for (const auto& e : edges) {
      const uint32_t edge = e[2] / (block * 4);
      if (!sr::use_sequence(edge, block, 4, true, e[0], e[1]) ||
          sr::use_sequence(edge - 1, block, 4, true, e[0], e[1]) ||
          sr::use_sequence(0x7FFFF000u, block, 4, false, e[0], e[1])) {
        std::printf("block %u, %u moments, %u bytes: the rule's edge moved\n", block, e[0], e[1]);
        ++failures;
      }
    }
  }
  // Momentum SGD: both ends, and the operands.
  for (uint32_t block : {128u, 256u, 512u, 1024u}) {
    const uint32_t first = (1u << 24) / (block * 4), last = (1u << 28) / (block * 4);
    if (!sr::use_sequence_sgdm(first, block, 4, true, true, true) ||
        sr::use_sequence_sgdm(first - 1, block, 4, true, true, true) ||
        !sr::use_sequence_sgdm(last, block, 4, true, true, true) ||
        sr::use_sequence_sgdm(last + 1, block, 4, true, true, true) ||
        sr::use_sequence_sgdm(first, block, 4, false, true, true) ||
        sr::use_sequence_sgdm(first, block, 4, true, false, true) ||
        sr::use_sequence_sgdm(first, block, 4, true, true, false)) {
      std::printf("block %u: momentum SGD's range moved\n", block);
      ++failures;
    }
  }
  for (uint32_t bytes = 6; bytes <= 28; ++bytes) {
    for (uint32_t block : {64u, 128u, 1024u}) {
      for (uint32_t moments : {0u, 1u, 2u}) {
        const uint32_t budget = sr::sequence_in_flight(moments), cap = sr::workgroups_in(budget, block, 4, bytes);
        const uint32_t tile = block * 4 * bytes;
        if (cap > sr::kResidentCapMax || (cap && (2 * cap * tile > 2 * budget + tile || 2 * (cap + 1) * tile < 2 * budget))) {
          std::printf("cap %u for %u bytes, block %u, budget %u\n", cap, bytes, block, budget);
          ++failures;
        }
      }
    }
  }
  // The caps of 128-lane launches (none: 0), by moments that round
  // stochastically to FP16 or FP8 and bytes per element; larger workgroups
  // hold the same bytes, and none where 128 lanes would hold too many.
  const uint32_t caps[][3] = {{0, 14, 13}, {0, 22, 8}, {0, 12, 0}, {0, 10, 0}, {1, 12, 0},
                              {1, 14, 0},  {1, 16, 12}, {1, 18, 11}, {2, 14, 0}, {2, 16, 13}};
  for (const auto& c : caps) {
    const uint32_t wide = sr::sequence_cap(c[0], 512, 4, c[1]);
    if (sr::sequence_cap(c[0], 128, 4, c[1]) != c[2] || (c[2] == 0) != (wide == 0) || 4 * wide > c[2] + 2) {
      std::printf("%u moments, %u bytes: cap %u, %u at 512 lanes\n", c[0], c[1],
                  sr::sequence_cap(c[0], 128, 4, c[1]), wide);
      ++failures;
    }
  }
  std::printf("%d shapes, %d failures\n", shapes, failures);
  return failures != 0;
}
