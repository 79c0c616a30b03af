// grow.h -- growing a group of device arrays together.
#pragma once
#include <cstddef>

namespace xf {

// Grows every array to n elements, each by its own capacity: an earlier call
// may have failed (out of memory) between two of them.  True if any of them was
// allocated again -- its contents are lost, whether or not the new memory lies
// at the old address.
template <class... Bufs>
bool ensure_all(size_t n, Bufs &...bufs) {
  bool moved = false;
  auto one = [&](auto &b) {
    if (b.p && b.cap >= n) return;
    b.ensure(n);
    moved = true;
  };
  (one(bufs), ...);
  return moved;
}

}  // namespace xf
