// list_capacity.h -- room for the traversal's interaction lists (traverse.hip).
// Plain arithmetic, for the device and for host code.  Totals are counted in 64
// bits; a list entry's place is an int, so a list holds at most kListMax entries.
#pragma once
#include <cstdint>

#ifndef __HIPCC__
#define XF_HD
#else
#define XF_HD __host__ __device__
#endif

namespace xf {

constexpr int64_t kListMax = (int64_t(1) << 31) - 1;

// Place of a run of n entries that begins at `first` (an int also where the
// pass overflows: it is repeated or fails, and reads nothing past `cap`).
XF_HD inline int list_place(uint64_t first, int64_t cap) {
  return int(first < uint64_t(cap) ? int64_t(first) : cap);
}
XF_HD inline bool list_overflows(uint64_t first, int64_t n, int64_t cap) { return first + uint64_t(n) > uint64_t(cap); }

// Capacity of a first pass for `per` entries per cell.
inline int64_t list_capacity(int64_t cells, int64_t per) {
  return cells > kListMax / per ? kListMax : cells * per;
}
// Capacity for the pass after one that counted `total` entries: the same where
// they fit, else at least twice (a pass whose hand-down list overflowed is cut
// short, its totals are lower bounds).  0: more entries than a list can hold.
inline int64_t list_grow(int64_t cap, uint64_t total) {
  if (total <= uint64_t(cap)) return cap;
  if (total > uint64_t(kListMax)) return 0;
  const int64_t twice = cap > kListMax / 2 ? kListMax : 2 * cap;
  return twice > int64_t(total) ? twice : int64_t(total);
}

}  // namespace xf
