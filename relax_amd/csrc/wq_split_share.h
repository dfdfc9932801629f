// Which parts of a tile a workgroup finishes, where the windows of a split share that (wq_gemm_stream.hip): the steps at the tile's counter and what
// is written to memory between them, apart from how either is done, so that a host program can take them in any order.
#pragma once
#include <stdint.h>

namespace wq {

// The counter of a tile in `windows` windows, at most eight: arrivals (bits 0 - 7), a bit for each window that has resigned (8 - 15), parts
// accounted for (from 16 on).  `add` adds to it and returns what was there before.
struct SplitCounter {
  static constexpr uint32_t kArrived = 1, kAccounted = 1u << 16;
  static constexpr uint32_t resigned(int w) { return 0x100u << w; }
  static constexpr bool all_in(uint32_t v, int windows) { return (v & 0xFFu) == (uint32_t)windows; }
  static constexpr uint32_t all_resigned(uint32_t v) { return v >> 8 & 0xFFu; }
};

// The parts (a bit each) that window w's workgroup finishes, 0 for none.  In order: it writes the other windows' parts of its own sums; counts
// itself in and looks for the others, `looks` times; if they are not all in it resigns, that is, writes its own part too and says so.  Every part
// has one workgroup: the last to arrive takes those of the windows that had resigned by then, and who resigns after that, which its add to
// the counter shows, keeps its own.  With all parts accounted for nobody touches the counter any more and it returns to zero.
// `one(f)`: f's value, asked for once, in the whole workgroup.
template <class Write, class One, class Add, class Zero>
constexpr uint32_t split_parts(int windows, int w, int looks, Write&& write, One&& one, Add&& add, Zero&& zero) {
  using C = SplitCounter;
  const uint32_t own = 1u << w;
  write(~own);
  uint32_t parts = one([&]() __attribute__((always_inline)) -> uint32_t {
    uint32_t v = add(C::kArrived) + C::kArrived;
    const uint32_t left = C::all_in(v, windows) ? C::all_resigned(v) : 0u;
    for (int i = 0; i < looks && !C::all_in(v, windows); ++i) v = add(0u);
    return C::all_in(v, windows) ? own | left : 0u;
  });
  if (parts == 0) {
    write(own);
    parts = one([&]() __attribute__((always_inline)) -> uint32_t { return C::all_in(add(C::resigned(w)), windows) ? own : 0u; });
  }
  if (parts != 0) zero([&]() __attribute__((always_inline)) -> bool {
    const uint32_t mine = C::kAccounted * (uint32_t)__builtin_popcount(parts);
    return add(mine) + mine >= C::kAccounted * (uint32_t)windows;
  });
  return parts;
}

}  // namespace wq
