// ensure_all (minimal_amd/csrc/grow.h) over arrays whose allocator fails on
// demand and may return the old address: after a failure anywhere in a group,
// the next call leaves every array large enough, and a call that allocated any
// array says so.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "../../minimal_amd/csrc/grow.h"

static int left = -1;  // allocations until one fails (-1: none)

struct Array {
  int *p = nullptr;
  size_t cap = 0;
  int made = 0;
  int storage[1];  // every allocation at the same address
  void ensure(size_t n) {
    if (n <= cap && p) return;
    p = nullptr;
    cap = 0;
    if (left == 0) throw 1;
    if (left > 0) left--;
    p = storage;
    cap = n;
    made++;
  }
};

int main() {
  for (int fail = 0; fail < 4; fail++)
    for (size_t next : {size_t(1), size_t(10), size_t(100), size_t(200)}) {
      Array a, b, c, d;
      left = -1;
      if (!xf::ensure_all(10, a, b, c, d) || xf::ensure_all(10, a, b, c, d) || xf::ensure_all(5, a, b, c, d)) return 1;
      left = fail;
      try {
        xf::ensure_all(100, a, b, c, d);
        return 2;
      } catch (int) {
      }
      left = -1;
      const int before = a.made + b.made + c.made + d.made;
      const bool moved = xf::ensure_all(next, a, b, c, d);
      const bool made = a.made + b.made + c.made + d.made > before;
      if (moved != made) return 3;
      for (const Array *x : {&a, &b, &c, &d})
        if (!x->p || x->cap < next) {
          std::printf("failure %d, next size %d\n", fail, int(next));
          return 4;
        }
    }
  return 0;
}
