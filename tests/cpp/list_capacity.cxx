// The interaction lists' room (minimal_amd/csrc/list_capacity.h) near 2^31
// entries: the arithmetic of a pass's reservations and of the capacities that
// follow, run by run.  A run is written only where its places lie in [0, cap);
// a pass that reserves more than its capacity says so, whatever the totals; and
// repeated passes end with room for everything or with an error.
#include <cstdint>
#include <cstdio>
#include <initializer_list>

#include "../../minimal_amd/csrc/list_capacity.h"

using namespace xf;

// One pass over `total` entries in runs of n: its flag, by the device's rules.
static bool pass(uint64_t total, int64_t n, int64_t cap, bool &ok, uint64_t &counted) {
  bool flag = false;
  counted = 0;
  // the runs around every point where something could change, not all 2^31
  for (uint64_t at : {uint64_t(0), uint64_t(cap) - uint64_t(cap) % uint64_t(n), uint64_t(1) << 31, uint64_t(1) << 32,
                      (uint64_t(1) << 32) + (uint64_t(1) << 31), total})
    for (int64_t d = -3; d <= 3; d++) {
      const int64_t first = int64_t(at / uint64_t(n) * uint64_t(n)) + d * n;
      if (first < 0 || uint64_t(first) >= total) continue;
      const int64_t m = uint64_t(first) + uint64_t(n) <= total ? n : int64_t(total - uint64_t(first));
      const bool over = list_overflows(uint64_t(first), m, cap);
      flag = flag || over;
      const int64_t place = list_place(uint64_t(first), cap);
      if (place < 0 || place > cap) ok = false;
      if (!over && place != first) ok = false;
      for (int64_t pos : {int64_t(0), m - 1}) {
        const bool write = place + pos < cap;  // the kernel's guard, in 64 bits
        if (!over && !write) ok = false;
      }
    }
  if ((total > uint64_t(cap)) != flag) ok = false;
  counted = total;
  return flag;
}

int main() {
  for (uint64_t total : {uint64_t(1), uint64_t(1000), uint64_t(kListMax) - 1, uint64_t(kListMax), uint64_t(kListMax) + 1,
                         (uint64_t(1) << 31) + 77, (uint64_t(1) << 32) + 5, uint64_t(3) << 31})
    for (int64_t cells : {int64_t(1), int64_t(5000), int64_t(11000000), int64_t(60000000)})
      for (int64_t per : {96, 200})
        for (int64_t n : {1, 7, 1500}) {
          int64_t cap = list_capacity(cells, per);
          if (cap < 1 || cap > kListMax) return 1;
          bool ok = true, ended = false;
          for (int attempt = 0; attempt < 64 && !ended; attempt++) {
            uint64_t counted;
            const bool flag = pass(total, n, cap, ok, counted);
            if (!flag) {
              ended = uint64_t(cap) >= total;
              break;
            }
            const int64_t next = list_grow(cap, counted);
            if (next == 0) {
              ended = total > uint64_t(kListMax);
              break;
            }
            if (next <= cap || next > kListMax) ok = false;
            cap = next;
          }
          if (!ok || !ended) {
            std::printf("total %llu cells %lld n %lld\n", (unsigned long long)total, (long long)cells, (long long)n);
            return 2;
          }
        }
  // a list that fits keeps its capacity
  if (list_grow(100, 100) != 100 || list_grow(100, 101) != 200 || list_grow(100, 1000) != 1000) return 3;
  return 0;
}
