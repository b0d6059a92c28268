// How the waves of a persistent pass share its items 0..n-1 (trav_persist.h).
// Slice s of `slice` consecutive items belongs to counter s % counters, and
// block b takes the slices of counter b % counters, in order.  Every counter
// needs a block to serve it, so a grid smaller than kWorkCounters has as many
// counters as blocks.
#pragma once

namespace bgpu {

constexpr unsigned int kWorkCounters = 16;
constexpr unsigned int work_counters(unsigned int blocks) { return blocks < kWorkCounters ? blocks : kWorkCounters; }

// The counter of a block, and the first item of the k-th slice it hands out.
constexpr unsigned int counter_of(unsigned int block, unsigned int blocks) { return block % work_counters(blocks); }
constexpr unsigned long long slice_begin(unsigned int k, unsigned int block, unsigned int blocks, unsigned int slice) {
  return ((unsigned long long)k * work_counters(blocks) + counter_of(block, blocks)) * slice;
}

// Items per slice: `wide` where every wave gets two such slices or more, else
// 64, one group of lanes.  Closest-hit scattered rays, always 64 against always
// 128, in us: 100,000 rays 118 and 139 (1 M-triangle grid), 88 and 119
// (100 k-triangle stack); 1,000,003 rays 251 and 255, 263 and 285; from 1.6 M
// rays on alike, and any-hit faster by 128 (16.8 M rays: 1127 and 1027, 1327
// and 1235).  With 6144 waves the line lies at 1.57 M rays.
constexpr unsigned int slice_items(unsigned int n, unsigned int waves, unsigned int wide) {
  return n / wide >= 2u * waves ? wide : 64u;
}

}  // namespace bgpu
