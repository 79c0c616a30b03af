// The stream-K schedule (minimal_amd/csrc/sk_schedule.h): over every slot count
// from 1 to twice the workgroups, the segments that the sum of a tile reads are
// those that the launch wrote, and every slot is taken once.
#include <algorithm>
#include <cstdio>
#include <set>
#include <utility>
#include <vector>

#include "../../minimal_amd/csrc/sk_schedule.h"

using namespace xf;

static bool check(int64_t grid, const std::vector<int> &tiles) {
  int64_t S = 0;
  std::vector<int64_t> base;
  for (int n : tiles) {
    base.push_back(S);
    S += n;
  }
  // the launch: workgroup w, tile t -> segment w + t
  const int64_t W = sk_active(grid, S);
  std::set<std::pair<int, int>> written;
  std::set<int64_t> segments;
  int64_t taken = 0;
  for (int64_t w = 0; w < grid; w++) {
    if (w >= W) continue;
    const int64_t s0 = sk_slot(w, S, W), s1 = sk_slot(w + 1, S, W);
    if (s0 >= s1) return false;
    taken += s1 - s0;
    for (size_t t = 0; t < tiles.size(); t++)
      if (std::min(s1, base[t] + tiles[t]) > std::max(s0, base[t])) {
        written.insert({int(w), int(t)});
        if (!segments.insert(w + int64_t(t)).second) return false;
      }
  }
  if (taken != S) return false;
  // the sum
  std::set<std::pair<int, int>> read;
  for (size_t t = 0; t < tiles.size(); t++)
    if (tiles[t])
      for (int w = sk_owner(base[t], S, W); w <= sk_owner(base[t] + tiles[t] - 1, S, W); w++) read.insert({w, int(t)});
  return read == written;
}

int main() {
  unsigned seed = 1;
  for (int64_t grid : {1, 3, 64, 256}) {
    for (int64_t S = 1; S <= 2 * grid + 3; S++)
      for (int pieces : {1, 2, 5, 17}) {
        std::vector<int> tiles(pieces, 0);  // some stay empty
        for (int64_t s = 0; s < S; s++) {
          seed = seed * 1664525u + 1013904223u;
          tiles[(seed >> 16) % pieces]++;
        }
        if (!check(grid, tiles)) {
          std::printf("grid %d slots %d tiles %d\n", int(grid), int(S), pieces);
          return 1;
        }
      }
  }
  const std::vector<int> large{1 << 30, 5, (1 << 30) - 7};  // products beyond 32 bits
  if (!check(256, large)) return 2;
  return 0;
}
