// tree.hip -- octree construction on the GPU, bit-exact with the reference.
//
// Reference: 3d/build_tree.h:7-96.  The reference builds the tree top-down
// by recursive stable octant partitions against FP64 cell centres
// (child centre = parent centre +/- R0/2^(l+1), strict '>'), stopping at
// NBODY <= ncrit.  Here each body's full octant path is computed once from
// the same FP64 centre sequence (63-bit key, 21 levels), the keys are
// radix-sorted (stable, so bodies with equal prefixes keep input order),
// levels are split by binary search on the sorted keys, and each leaf's
// bodies are put back into input order -- which is the order the
// reference's stable partitions leave inside a leaf.  Cells are stored
// level by level (BFS); the reference's numbering (children blocks in DFS
// preorder of their parents) is computed on export.
#include <algorithm>

#include "fmm_internal.h"
#include "grow.h"

namespace xf {

constexpr int kHistLevels = 7;
__host__ __device__ constexpr int hist_off(int l) {  // offset of level l (1..7) in the histogram array
  return l <= 1 ? 0 : hist_off(l - 1) + (1 << (3 * (l - 1)));
}
constexpr int kHistTotal = hist_off(kHistLevels + 1);
constexpr int kMiscInts = 64;

// ---------------------------------------------------------------- bounds
// It also clears the level-7 histogram of the launch after the next.  part:
// per workgroup [lo, hi, 1 if a coordinate or charge is not finite].
constexpr int kBoundsBlocks = 256, kBoundsInts = 7;
__global__ void __launch_bounds__(256) k_bounds_part(const exafmm_body *__restrict__ b, int64_t n,
                                                     double *__restrict__ part, int4 *__restrict__ hist7) {
  __shared__ double s[6][256];
  for (int i = blockIdx.x * 256 + threadIdx.x; i < (1 << (3 * kHistLevels)) / 4; i += gridDim.x * 256)
    hist7[i] = make_int4(0, 0, 0, 0);
  double lo[3] = {b[0].X[0], b[0].X[1], b[0].X[2]};
  double hi[3] = {lo[0], lo[1], lo[2]};
  int bad = 0;
  for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) {
    for (int d = 0; d < 3; d++) {
      const double x = b[i].X[d];
      if (!isfinite(x)) bad = 1;
      lo[d] = fmin(x, lo[d]);
      hi[d] = fmax(x, hi[d]);
    }
    if (!isfinite(b[i].q)) bad = 1;
  }
  bad = __syncthreads_or(bad);
  for (int d = 0; d < 3; d++) {
    s[d][threadIdx.x] = lo[d];
    s[3 + d][threadIdx.x] = hi[d];
  }
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o)
      for (int d = 0; d < 3; d++) {
        s[d][threadIdx.x] = fmin(s[d][threadIdx.x], s[d][threadIdx.x + o]);
        s[3 + d][threadIdx.x] = fmax(s[3 + d][threadIdx.x], s[3 + d][threadIdx.x + o]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 6) part[blockIdx.x * kBoundsInts + threadIdx.x] = s[threadIdx.x][0];
  if (threadIdx.x == 6) part[blockIdx.x * kBoundsInts + 6] = bad ? 1.0 : 0.0;
}

// The root cell and the build's counters.
struct RootOut {
  double *root;   // X0, R0
  int *misc;      // flags and counters (see tree_build)
  int *lcount, *lstart;
  double4 *cx;
  int *cbeg, *ccnt, *cparent, *clevel;
  int64_t n;
};
__device__ inline void write_root(const RootOut &o, double x, double y, double z, double r) {
  o.root[0] = x;
  o.root[1] = y;
  o.root[2] = z;
  o.root[3] = r;
  o.cx[0] = make_double4(x, y, z, r);
  o.cbeg[0] = 0;
  o.ccnt[0] = int(o.n);
  o.cparent[0] = -1;
  o.clevel[0] = 0;
  o.lcount[0] = 1;
  o.lstart[0] = 0;
}
// (threads 0 .. 255; thread 0 has written misc[0] already)
__device__ inline void clear_counters(const RootOut &o) {
  const int t = threadIdx.x;
  if (t > 0 && t < kMiscInts) o.misc[t] = 0;
  if (t > 0 && t < kMaxLevel + 2) o.lcount[t] = 0;
}

// X0 = (max+min)/2, R0 = max half-extent * 1.00001 (3d/build_tree.h:7-21).
__global__ void __launch_bounds__(kBoundsBlocks) k_bounds_final(const double *__restrict__ part, RootOut out) {
  __shared__ double s[6][256];
  const int t = threadIdx.x;
  double v[6];
  for (int d = 0; d < 6; d++) v[d] = part[t * kBoundsInts + d];
  const int bad = __syncthreads_or(part[t * kBoundsInts + 6] != 0.0);
  if (t == 0) out.misc[0] = bad ? 1 : 0;
  clear_counters(out);
  for (int d = 0; d < 6; d++) s[d][t] = v[d];
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (t < o)
      for (int d = 0; d < 3; d++) {
        s[d][t] = fmin(s[d][t], s[d][t + o]);
        s[3 + d][t] = fmax(s[3 + d][t], s[3 + d][t + o]);
      }
    __syncthreads();
  }
  if (t != 0) return;
  double lo[3], hi[3], X0[3];
  for (int d = 0; d < 3; d++) {
    lo[d] = s[d][0];
    hi[d] = s[3 + d][0];
    X0[d] = (hi[d] + lo[d]) / 2;
  }
  double R0 = 0;
  for (int d = 0; d < 3; d++) {
    R0 = fmax(X0[d] - lo[d], R0);
    R0 = fmax(hi[d] - X0[d], R0);
  }
  R0 *= 1.00001;
  write_root(out, X0[0], X0[1], X0[2], R0);
}

// Forest: counters, the histogram and the unit root cube of levels 0 ..
// kForestLevel - 1 (problem-index cells, never paired by the traversal).
__global__ void __launch_bounds__(256) k_forest_init(RootOut out, int4 *__restrict__ hist7) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < (1 << (3 * kHistLevels)) / 4; i += gridDim.x * 256)
    hist7[i] = make_int4(0, 0, 0, 0);
  if (blockIdx.x > 0) return;
  if (threadIdx.x == 0) {
    out.misc[0] = 0;
    write_root(out, 0.0, 0.0, 0.0, 1.0);
  }
  clear_counters(out);
}

// Forest: the root of k_bounds_final per problem (min / max are exact, so any
// reduction order gives the same root).  Empty problems get a unit root.  A
// problem's bodies are shared by kForestShares workgroups (one alone took 30 -
// 68 us for 100,000 bodies); part: [problem][share][lo, hi].
constexpr int kForestShares = 16;
__global__ void __launch_bounds__(256) k_forest_bounds(const exafmm_body *__restrict__ b,
                                                       const int64_t *__restrict__ off, double *__restrict__ part,
                                                       int *__restrict__ flags) {
  __shared__ double s[256 / kWave][6];
  const int p = blockIdx.y, t = threadIdx.x, lane = t % kWave, w = t / kWave;
  const int64_t o0 = off[p], n = off[p + 1] - o0;
  if (n <= 0) return;
  const int64_t i0 = o0 + n * blockIdx.x / kForestShares, i1 = o0 + n * (blockIdx.x + 1) / kForestShares;
  double lo[3] = {b[o0].X[0], b[o0].X[1], b[o0].X[2]};
  double hi[3] = {lo[0], lo[1], lo[2]};
  int bad = 0;
  for (int64_t i = i0 + t; i < i1; i += 256) {
    for (int d = 0; d < 3; d++) {
      const double x = b[i].X[d];
      if (!isfinite(x)) bad = 1;
      lo[d] = fmin(x, lo[d]);
      hi[d] = fmax(x, hi[d]);
    }
    if (!isfinite(b[i].q)) bad = 1;
  }
  if (bad) atomicOr(flags, 1);
  for (int d = 0; d < 3; d++)
    for (int o = 1; o < kWave; o <<= 1) {
      lo[d] = fmin(lo[d], __shfl_xor(lo[d], o));
      hi[d] = fmax(hi[d], __shfl_xor(hi[d], o));
    }
  if (lane == 0)
    for (int d = 0; d < 3; d++) {
      s[w][d] = lo[d];
      s[w][3 + d] = hi[d];
    }
  __syncthreads();
  if (t < 6) {
    double v = s[0][t];
    for (int k = 1; k < 256 / kWave; k++) v = t < 3 ? fmin(v, s[k][t]) : fmax(v, s[k][t]);
    part[(int64_t(p) * kForestShares + blockIdx.x) * 6 + t] = v;
  }
}

__global__ void __launch_bounds__(64) k_forest_roots(const int64_t *__restrict__ off, const double *__restrict__ part,
                                                     int nprob, double4 *__restrict__ roots) {
  const int p = blockIdx.x * 64 + threadIdx.x;
  if (p >= nprob) return;
  if (off[p + 1] <= off[p]) {
    roots[p] = make_double4(0.0, 0.0, 0.0, 1.0);
    return;
  }
  const double *q = part + int64_t(p) * kForestShares * 6;
  double lo[3], hi[3], X0[3], R0 = 0;
  for (int d = 0; d < 3; d++) {
    lo[d] = q[d];
    hi[d] = q[3 + d];
    for (int k = 1; k < kForestShares; k++) {
      lo[d] = fmin(lo[d], q[k * 6 + d]);
      hi[d] = fmax(hi[d], q[k * 6 + 3 + d]);
    }
    X0[d] = (hi[d] + lo[d]) / 2;
  }
  for (int d = 0; d < 3; d++) {
    R0 = fmax(X0[d] - lo[d], R0);
    R0 = fmax(hi[d] - X0[d], R0);
  }
  R0 *= 1.00001;
  roots[p] = make_double4(X0[0], X0[1], X0[2], R0);
}

// ---------------------------------------------------------------- keys
// Octant path of each body through the reference's centre sequence and, with
// HIST, the population of its level-7 prefix (dense, 8^7 bins) by atomics.
// Without it the histogram is taken from the sorted keys (k_hist_sorted):
// deep trees are sorted by radix anyway, and their crowded prefixes (a Plummer
// core) make the XCDs' atomics pass the same counters around (1.5M clustered
// bodies: 243 us, even with each workgroup's bodies counted in LDS first; 32 us
// without, and 12 for k_hist_sorted).  One wave in kOrderSample adds the number of
// runs of equal level-4 prefixes among its lanes to order[0], its lanes to order[1]
// (above the leaves of the sets it is looked at for: below them the order is the
// caller's).
constexpr int kOrderSample = 64;
constexpr int kKeysThreads = 256;
template <bool HIST>
__global__ void __launch_bounds__(kKeysThreads) k_keys(const exafmm_body *__restrict__ b, int64_t n,
                                                       const double *__restrict__ root,
                                                       unsigned long long *__restrict__ key, int *__restrict__ val,
                                                       int *__restrict__ hist7, const double4 *__restrict__ froots,
                                                       const int64_t *__restrict__ off, int nprob,
                                                       int *__restrict__ order) {
  const int64_t i = int64_t(blockIdx.x) * kKeysThreads + threadIdx.x;
  if (i >= n) return;
  const double x = b[i].X[0], y = b[i].X[1], z = b[i].X[2];
  double R0 = root[3], cx = root[0], cy = root[1], cz = root[2];
  unsigned long long k = 0;
  int l0 = 0;
  if (froots) {
    // forest: the problem's index fills the digits of levels 0 .. kForestLevel - 1,
    // its own root's octant path the rest
    int lo = 0, hi = nprob - 1;  // last problem with off[p] <= i
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (off[mid] <= i)
        lo = mid;
      else
        hi = mid - 1;
    }
    const double4 Rt = froots[lo];
    cx = Rt.x;
    cy = Rt.y;
    cz = Rt.z;
    R0 = Rt.w;
    k = (unsigned long long)lo;
    l0 = kForestLevel;
  }
  for (int l = l0; l < kMaxLevel; l++) {
    const int bx = x > cx, by = y > cy, bz = z > cz;
    const int oct = bx + (by << 1) + (bz << 2);
    k = (k << 3) | unsigned(oct);
    const double rr = R0 / (1 << (l - l0 + 1));
    cx += bx ? rr : -rr;
    cy += by ? rr : -rr;
    cz += bz ? rr : -rr;
  }
  key[i] = k;
  val[i] = int(i);
  if (i / kWave % kOrderSample == 0) {  // uniform
    const unsigned p4 = unsigned(k >> (3 * (kMaxLevel - 4)));
    const unsigned prev = __shfl_up(p4, 1);
    const int lane = threadIdx.x & (kWave - 1);
    const int runs = __popcll(__ballot(lane == 0 || prev != p4)), lanes = __popcll(__ballot(true));
    if (lane == 0) {
      atomicAdd(order, runs);
      atomicAdd(order + 1, lanes);
    }
  }
  if (HIST) atomicAdd(&hist7[unsigned(k >> (3 * (kMaxLevel - kHistLevels)))], 1);
}

// Level-7 populations from the sorted keys: the ends of a prefix's run add up
// to its length (two atomics per prefix that occurs).
__global__ void __launch_bounds__(256) k_hist_sorted(const unsigned long long *__restrict__ key, int64_t n,
                                                     int *__restrict__ hist7) {
  constexpr int sh = 3 * (kMaxLevel - kHistLevels);
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const unsigned bin = unsigned(key[i] >> sh);
  if (i == 0 || unsigned(key[i - 1] >> sh) != bin) atomicAdd(&hist7[bin], -int(i));
  if (i == n - 1 || unsigned(key[i + 1] >> sh) != bin) atomicAdd(&hist7[bin], int(i) + 1);
}

// Levels 6..3 of the prefix histogram from level 7 (prefixes are in Morton
// order, so prefix p of level l has children 8p..8p+7 at level l+1).  Block
// b sums the 4096 level-7 bins under level-3 prefix b: thread t loads bins
// 4t..4t+3 in one 16-byte load, lane shuffles give levels 6 and 5, LDS
// levels 4 and 3.  The block's largest population per level goes to
// bmax[8b + l] (l = 3..7).
static_assert(kHistLevels == 7, "k_hist_pyramid is shaped for 8^7 level-7 bins");
__global__ void __launch_bounds__(1024) k_hist_pyramid(int *__restrict__ hist, int *__restrict__ bmax) {
  __shared__ int w4[16], wm[16][3], s4[8];
  const int t = threadIdx.x, b = blockIdx.x, lane = t & (kWave - 1), w = t / kWave;
  const int4 v = reinterpret_cast<const int4 *>(hist + hist_off(7))[b * 1024 + t];
  int m7 = max(max(v.x, v.y), max(v.z, v.w));
  int s6 = v.x + v.y + v.z + v.w;
  s6 += __shfl_xor(s6, 1);  // 8 level-7 bins: 2 threads
  int s5 = s6 + __shfl_xor(s6, 2);
  s5 += __shfl_xor(s5, 4);
  s5 += __shfl_xor(s5, 8);  // 64 bins: 16 threads
  int h = s5 + __shfl_xor(s5, 16);
  h += __shfl_xor(h, 32);  // the wave's half of a level-4 prefix
  if ((t & 1) == 0) hist[hist_off(6) + b * 512 + (t >> 1)] = s6;
  if ((t & 15) == 0) hist[hist_off(5) + b * 64 + (t >> 4)] = s5;
  int m6 = s6, m5 = s5;
  for (int o = 1; o < kWave; o <<= 1) {
    m7 = max(m7, __shfl_xor(m7, o));
    m6 = max(m6, __shfl_xor(m6, o));
    m5 = max(m5, __shfl_xor(m5, o));
  }
  if (lane == 0) {
    w4[w] = h;
    wm[w][0] = m7;
    wm[w][1] = m6;
    wm[w][2] = m5;
  }
  __syncthreads();
  if (t < 8) {
    s4[t] = w4[2 * t] + w4[2 * t + 1];
    hist[hist_off(4) + b * 8 + t] = s4[t];
  }
  __syncthreads();
  if (t == 0) {
    int a7 = 0, a6 = 0, a5 = 0, a4 = 0, s3 = 0;
    for (int i = 0; i < 16; i++) {
      a7 = max(a7, wm[i][0]);
      a6 = max(a6, wm[i][1]);
      a5 = max(a5, wm[i][2]);
    }
    for (int i = 0; i < 8; i++) {
      a4 = max(a4, s4[i]);
      s3 += s4[i];
    }
    hist[hist_off(3) + b] = s3;
    bmax[8 * b + 3] = s3;
    bmax[8 * b + 4] = a4;
    bmax[8 * b + 5] = a5;
    bmax[8 * b + 6] = a6;
    bmax[8 * b + 7] = a7;
  }
}

// Levels 2 and 1 from level 3, and the largest population of every level
// (lmax[l], l = 1..7) from the blocks' maxima: the first 512 threads of one
// workgroup (every thread calls it).
__device__ inline void hist_top(int *hist, const int *__restrict__ bmax, int *lmax) {
  __shared__ int wmax[5][8], s2[64];
  const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
  if (t < 512) {
    for (int l = 3; l <= 7; l++) {
      int m = bmax[8 * t + l];
      for (int o = 1; o < kWave; o <<= 1) m = max(m, __shfl_xor(m, o));
      if (lane == 0) wmax[l - 3][w] = m;
    }
  }
  if (t < 64) {
    int s = 0;
    for (int c = 0; c < 8; c++) s += hist[hist_off(3) + t * 8 + c];
    s2[t] = s;
    hist[hist_off(2) + t] = s;
  }
  __syncthreads();
  if (t >= 3 && t <= 7) {
    int m = 0;
    for (int i = 0; i < 8; i++) m = max(m, wmax[t - 3][i]);
    lmax[t] = m;
  }
  if (t == 0) {
    int a2 = 0, a1 = 0;
    for (int i = 0; i < 64; i++) a2 = max(a2, s2[i]);
    for (int o = 0; o < 8; o++) {
      int s = 0;
      for (int c = 0; c < 8; c++) s += s2[o * 8 + c];
      hist[hist_off(1) + o] = s;
      a1 = max(a1, s);
    }
    lmax[2] = a2;
    lmax[1] = a1;
  }
  __syncthreads();
}
__global__ void __launch_bounds__(512) k_hist_top(int *hist, const int *__restrict__ bmax, int *lmax) {
  hist_top(hist, bmax, lmax);
}

// Bodies by their level-l prefix (counting sort: cursor holds the prefixes'
// first places): the order within a prefix is left to k_leaf_gather, which
// puts every leaf's bodies back into input order.
__global__ void __launch_bounds__(256) k_place(const unsigned long long *__restrict__ key, int64_t n, int shift,
                                               int *__restrict__ cursor, unsigned long long *__restrict__ key_out,
                                               int *__restrict__ val_out) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const unsigned long long k = key[i];
  const int bin = int(k >> shift), lane = threadIdx.x & (kWave - 1);
  // A run of equal prefixes among neighbouring lanes takes its places with one
  // atomic: bodies that come in tree order (those of the step before) have
  // nothing but such runs, and one atomic each made the lanes of a wave wait for
  // one counter (10^6 uniform bodies in tree order, a build: ncrit 64 277 -> 191 us,
  // ncrit 300 502 -> 209; 4 x 10^6 and ncrit 300 1,086 -> 515; bodies in random order
  // the same).
  const int prev = __shfl_up(bin, 1);
  const unsigned long long here = __ballot(true), starts = __ballot(lane == 0 || prev != bin);
  int pos;
  if (starts == here) {  // uniform
    pos = atomicAdd(&cursor[bin], 1);
  } else {
    const int first = 63 - __clzll((long long)(starts & (~0ull >> (63 - lane))));
    const unsigned long long later = starts & ~(~0ull >> (63 - first));
    const int end = later ? __ffsll((long long)later) - 1 : __popcll(here);
    int at = 0;
    if (lane == first) at = atomicAdd(&cursor[bin], end - first);
    pos = __shfl(at, first) + lane - first;
  }
  key_out[pos] = k;
  val_out[pos] = int(i);
}

// Bodies up to which a counting sort is taken whatever their order (tree_build):
// two radix passes instead (up to five levels), three (six and seven).
constexpr int64_t kPlaceMax5 = 750000, kPlaceMax7 = 1500000;

// ---------------------------------------------------------------- levels
// Node t of level l: if it holds more than ncrit bodies, find the body
// sub-ranges of its 8 octants (keys are sorted by the level-(l+1) digit
// inside the node's range) by binary search.
// Child boundaries of a level-l cell holding bodies [beg, beg + cnt) of the
// sorted keys: b[o] .. b[o + 1] are octant o's bodies.  Returns the number of
// non-empty children (0: the cell is a leaf, b untouched).
__device__ inline int split_bounds(int l, int ncrit, int beg, int cnt, const unsigned long long *__restrict__ key,
                                   const int *__restrict__ hist, int b[9], int lforce) {
  // levels above lforce (a forest's problem-index levels) always split
  if ((cnt <= ncrit && l >= lforce) || cnt == 0 || l >= kMaxLevel) return 0;
  const int sh = 3 * (kMaxLevel - 1 - l);
  b[0] = beg;
  b[8] = beg + cnt;
  if (l + 1 <= kHistLevels) {
    // the children's populations are the level-(l+1) prefix histogram
    // entries of this node's prefix (all its bodies share it)
    const unsigned long long pre = key[beg] >> (sh + 3);
    const int *h = hist + hist_off(l + 1) + int(pre) * 8;
    for (int o = 1; o < 8; o++) b[o] = b[o - 1] + h[o - 1];
  } else {
    // first index with digit >= o: the seven searches side by side, so that a
    // step waits once for seven loads (one after the other they made the deep
    // levels of 1.5M clustered bodies wait up to 38 us each)
    int lo[8], hi[8];
    for (int o = 1; o < 8; o++) {
      lo[o] = beg;
      hi[o] = beg + cnt;
    }
    for (bool more = true; more;) {
      int d[8];
#pragma unroll
      for (int o = 1; o < 8; o++) d[o] = int((key[min((lo[o] + hi[o]) >> 1, beg + cnt - 1)] >> sh) & 7ull);
      more = false;
#pragma unroll
      for (int o = 1; o < 8; o++) {
        if (lo[o] >= hi[o]) continue;
        const int mid = (lo[o] + hi[o]) >> 1;
        if (d[o] < o)
          lo[o] = mid + 1;
        else
          hi[o] = mid;
        more |= lo[o] < hi[o];
      }
    }
    for (int o = 1; o < 8; o++) b[o] = lo[o];
  }
  int k = 0;
  for (int o = 0; o < 8; o++) k += b[o + 1] > b[o];
  return k;
}

// Writes the non-empty children of level-l cell c (boundaries b) to cells
// first, first + 1, ... in octant order.
// r = R_parent / 2 is R0 / 2^(l+1) exactly.  Forest: the cells of level
// kForestLevel are the problems' roots (froots, by the problem index in the
// top key digits).
__device__ inline void emit_children(int l, int c, int first, const int b[9], const double4 *__restrict__ froots,
                                     const unsigned long long *__restrict__ key, double4 *__restrict__ cx,
                                     int *__restrict__ cbeg, int *__restrict__ ccnt, int *__restrict__ cchild,
                                     int *__restrict__ cparent, int *__restrict__ clevel,
                                     unsigned char *__restrict__ coct) {
  cchild[c] = first;
  const double4 P = cx[c];
  const double r = P.w * 0.5;
  int j = 0;
  for (int o = 0; o < 8; o++) {
    const int b0 = b[o], b1 = b[o + 1];
    if (b1 <= b0) continue;
    const int ch = first + j++;
    double4 X;
    X.x = P.x + ((o & 1) ? r : -r);
    X.y = P.y + ((o & 2) ? r : -r);
    X.z = P.z + ((o & 4) ? r : -r);
    X.w = r;
    if (froots && l + 1 == kForestLevel) X = froots[int(key[b0] >> (3 * (kMaxLevel - kForestLevel)))];
    cx[ch] = X;
    cbeg[ch] = b0;
    ccnt[ch] = b1 - b0;
    cparent[ch] = c;
    clevel[ch] = l + 1;
    coct[ch] = (unsigned char)o;
  }
}

// Exclusive prefix, over the workgroups of a launch, of one count each
// (decoupled look-back).  A workgroup's number comes from *ticket (zero at
// the launch), so those before it have started and never wait for it: every
// wait ends.  A workgroup publishes one word, [tag | state | value] -- state 1
// its own count, 2 the sum up to and with it -- and no other data is passed, so
// relaxed atomics are enough.  `tag` differs from that of every earlier launch
// on the array.  Call with the whole workgroup (at least 64 threads).
//
// The workgroups that have something to count, 1,024 items each (one at
// least), of a grid that is sized for a bound: the others leave without a
// number.  (27,000 of them for the 21 levels of 4 x 10^6 clustered bodies, ncrit
// 16, queued for numbers at one counter: a build of them in tree order 1,590 -> 1,391 us.)
__device__ inline int lookback_groups(int items) { return max(1, min(int(gridDim.x), (items + 1023) / 1024)); }
__device__ inline int lookback_ticket(int *ticket) {
  __shared__ int id;
  if (threadIdx.x == 0) id = atomicAdd(ticket, 1);
  __syncthreads();
  return id;
}
__device__ inline int lookback_prefix(int id, int count, unsigned tag, unsigned long long *words) {
  __shared__ int prefix;
  if (threadIdx.x < kWave) {
    const int lane = threadIdx.x;
    auto word = [&](int state, int v) {
      return (unsigned long long)tag << 40 | (unsigned long long)state << 32 | unsigned(v);
    };
    auto put = [&](int i, unsigned long long v) {
      __hip_atomic_store(words + i, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    if (lane == 0) put(id, word(id == 0 ? 2 : 1, count));
    int sum = 0;
    for (int top = id - 1; top >= 0; top -= kWave) {  // windows of 64 predecessors, nearest first
      const int i = top - lane;
      unsigned long long v = 0;
      int state = 2;  // before the first: an empty prefix
      if (i >= 0) {
        do {
          v = __hip_atomic_load(words + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } while (unsigned(v >> 40) != tag);
        state = int(v >> 32) & 3;
      }
      const unsigned long long done = __ballot(state == 2);
      const int last = done ? __ffsll((long long)done) - 1 : kWave - 1;
      int x = i >= 0 && lane <= last ? int(unsigned(v)) : 0;
      for (int o = 1; o < kWave; o <<= 1) x += __shfl_xor(x, o);
      sum += x;
      if (done) break;
    }
    if (lane == 0) {
      if (id > 0) put(id, word(2, sum + count));
      prefix = sum;
    }
  }
  __syncthreads();
  return prefix;
}

// Exclusive scan of one count per thread over a workgroup of 1024.
__device__ inline int block_scan(int v, int &total) {
  __shared__ int wsum[1024 / kWave];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  int incl = v;
  for (int d = 1; d < kWave; d <<= 1) {
    const int x = __shfl_up(incl, d);
    if (lane >= d) incl += x;
  }
  __syncthreads();  // the last use of wsum
  if (lane == kWave - 1) wsum[w] = incl;
  __syncthreads();
  int before = 0;
  total = 0;
  for (int i = 0; i < 1024 / kWave; i++) {
    before += i < w ? wsum[i] : 0;
    total += wsum[i];
  }
  return before + incl - v;
}

// Splits level l (one cell per thread): child boundaries, the children's
// places in level l + 1 by a look-back over the workgroups, and the children,
// in octant order (3d/build_tree.h:115-132): centre = parent centre +
// r*(+/-1), r = R0/2^(l+1); R = R0/2^(l+1).  One launch per level where split,
// scan, level sizes and emission took four.
__global__ void __launch_bounds__(1024) k_split_level(int l, int ncrit, int lforce, int *lcount, int *lstart,
                                                      const unsigned long long *__restrict__ key,
                                                      const int *__restrict__ hist, const double4 *__restrict__ froots,
                                                      double4 *__restrict__ cx, int *cbeg, int *ccnt,
                                                      int *__restrict__ cchild, int *__restrict__ cnch,
                                                      int *__restrict__ cparent, int *__restrict__ clevel,
                                                      unsigned char *__restrict__ coct, int *__restrict__ nsplit, int *__restrict__ ticket, unsigned tag,
                                                      unsigned long long *__restrict__ words) {
  const int count = lcount[l], start = lstart[l], next = start + count;
  const int groups = lookback_groups(count);
  if (int(blockIdx.x) >= groups) return;
  const int id = lookback_ticket(ticket);
  const int t = id * 1024 + threadIdx.x, c = start + t;
  const bool in = t < count;
  int b[9];
  const int k = in ? split_bounds(l, ncrit, cbeg[c], ccnt[c], key, hist, b, lforce) : 0;
  // cells that split, counted per wave (leaves = cells - split cells)
  const unsigned long long sp = __ballot(k > 0);
  if ((threadIdx.x & (kWave - 1)) == 0 && sp) atomicAdd(nsplit, int(__popcll(sp)));
  int total;
  const int off = block_scan(k, total);
  const int before = lookback_prefix(id, total, tag, words);
  if (in) {
    cnch[c] = k;
    if (k == 0)
      cchild[c] = -1;
    else
      emit_children(l, c, next + before + off, b, froots, key, cx, cbeg, ccnt, cchild, cparent, clevel, coct);
  }
  if (id == groups - 1 && threadIdx.x == 0) {
    lcount[l + 1] = before + total;
    lstart[l + 1] = next;
  }
}

// The leaves, in breadth-first order, and the cells of the deepest sorted
// level l, which are leaves: more than ncrit bodies there means the tree needs
// more levels.
__global__ void __launch_bounds__(1024) k_leaves(int l, int ncrit, const int *__restrict__ lcount,
                                                 const int *__restrict__ lstart, const int *__restrict__ ccnt,
                                                 int *cchild, int *cnch, int *__restrict__ leaves, int *__restrict__ misc,
                                                 int *__restrict__ ticket, unsigned tag,
                                                 unsigned long long *__restrict__ words) {
  const int last = lstart[l], nc = last + lcount[l];
  const int groups = lookback_groups(nc);
  if (int(blockIdx.x) >= groups) return;
  const int id = lookback_ticket(ticket);
  const int c = id * 1024 + threadIdx.x;
  bool leaf = false;
  if (c < nc) {
    leaf = c >= last || cnch[c] == 0;
    if (c >= last) {
      cnch[c] = 0;
      cchild[c] = -1;
      if (ccnt[c] > ncrit) atomicOr(misc, 2);
    }
  }
  int total;
  const int off = block_scan(leaf, total);
  const int before = lookback_prefix(id, total, tag, words);
  if (leaf) leaves[before + off] = c;
  if (id == groups - 1 && threadIdx.x == 0) misc[17] = before + total;
}

// The top levels, 0 .. lend - 1, split by one workgroup (which also finishes
// the histogram, hist_top): per level what k_split_level does, with a
// workgroup scan and barriers.  Level l holds at most
// 8^l cells, so levels up to kTopLevels - 1 fit kTopPer cells per thread;
// thread t owns cells kTopPer t .. kTopPer t + kTopPer - 1 of its level.
// Level 4 (4096 cells) stays on the multi-workgroup kernels: one workgroup
// walking four cells per thread through their dependent loads (counts, key,
// histogram, centre) took longer than the four launches it saves.
constexpr int kTopThreads = 1024, kTopPer = 1, kTopLevels = 4;
static_assert(1 << (3 * (kTopLevels - 1)) <= kTopThreads * kTopPer, "top levels exceed the workgroup");
__global__ void __launch_bounds__(kTopThreads)
    k_top_levels(int lend, int ncrit, int lforce, int *__restrict__ lcount, int *__restrict__ lstart,
                 const unsigned long long *__restrict__ key, int *hist, const int *__restrict__ bmax,
                 int *__restrict__ lmax, const double4 *__restrict__ froots, double4 *__restrict__ cx, int *__restrict__ cbeg,
                 int *__restrict__ ccnt, int *__restrict__ cchild, int *__restrict__ cnch,
                 int *__restrict__ cparent, int *__restrict__ clevel, unsigned char *__restrict__ coct,
                 int *__restrict__ nsplit) {
  __shared__ int wsum[kTopThreads / kWave];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
  if (bmax) hist_top(hist, bmax, lmax);
  int cnt = lcount[0], start = lstart[0];
  for (int l = 0; l < lend; l++) {
    int b[kTopPer][9], k[kTopPer];
    int mine = 0, nspl = 0;
#pragma unroll
    for (int j = 0; j < kTopPer; j++) {
      const int t = tid * kTopPer + j;
      k[j] = 0;
      if (t < cnt) {
        const int c = start + t;
        k[j] = split_bounds(l, ncrit, cbeg[c], ccnt[c], key, hist, b[j], lforce);
      }
      mine += k[j];
      nspl += k[j] > 0;
    }
    // exclusive scan of the children counts over the workgroup
    int incl = mine;
    for (int d = 1; d < kWave; d <<= 1) {
      const int v = __shfl_up(incl, d);
      if (lane >= d) incl += v;
    }
    for (int d = kWave / 2; d > 0; d >>= 1) nspl += __shfl_xor(nspl, d);
    if (lane == 0 && nspl) atomicAdd(nsplit, nspl);  // cells that split
    if (lane == kWave - 1) wsum[w] = incl;
    __syncthreads();
    int off = incl - mine, total = 0;
    for (int i = 0; i < kTopThreads / kWave; i++) {
      off += i < w ? wsum[i] : 0;
      total += wsum[i];
    }
    const int next = start + cnt;
#pragma unroll
    for (int j = 0; j < kTopPer; j++) {
      const int t = tid * kTopPer + j;
      if (t < cnt) {
        const int c = start + t;
        cnch[c] = k[j];
        if (k[j] == 0)
          cchild[c] = -1;
        else
          emit_children(l, c, next + off, b[j], froots, key, cx, cbeg, ccnt, cchild, cparent, clevel, coct);
        off += k[j];
      }
    }
    if (tid == 0) {
      lcount[l + 1] = total;
      lstart[l + 1] = next;
    }
    __syncthreads();  // children written before the next level reads them
    start = next;
    cnt = total;
  }
}

__global__ void k_root(RootOut out) {
  out.cx[0] = make_double4(out.root[0], out.root[1], out.root[2], out.root[3]);
  out.cbeg[0] = 0;
  out.ccnt[0] = int(out.n);
  out.cparent[0] = -1;
  out.clevel[0] = 0;
}

// One workgroup per leaf: restore input order inside the leaf (rank of
// each original index among the leaf's), then gather X, q (FP64) and the
// leaf-relative FP32 copy used by P2P.  The first workgroup also hands the
// level sizes, the counters and the root to the host (pinned memory).
struct TreeReport {
  const int *lcount, *misc;
  const double *root;
  int *host_levels, *host_misc;
  double *host_root;
};
__global__ void __launch_bounds__(64) k_leaf_gather(const int *__restrict__ leaves, const int *__restrict__ nleaves,
                                                    const int *__restrict__ cbeg, const int *__restrict__ ccnt,
                                                    const double4 *__restrict__ cx, const int *__restrict__ val,
                                                    const exafmm_body *__restrict__ b, int *__restrict__ perm,
                                                    double4 *__restrict__ xs, float4 *__restrict__ xq,
                                                    int *__restrict__ body_leaf, int ncrit, TreeReport rep) {
  extern __shared__ int sidx[];  // ncrit ints
  if (blockIdx.x == 0) {
    auto put = [](auto *p, auto v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); };
    const int t = threadIdx.x;
    if (t < kMaxLevel + 2) put(rep.host_levels + t, rep.lcount[t]);
    if (t < 21) put(rep.host_misc + t, rep.misc[t]);
    if (t < 4) put(rep.host_root + t, rep.root[t]);
  }
  const int nl = *nleaves;
  for (int li = blockIdx.x; li < nl; li += gridDim.x) {
    const int c = leaves[li];
    const int beg = cbeg[c], cnt = ccnt[c];
    // a leaf above ncrit: a tree the host rejects or builds again (flag 2)
    if (cnt > ncrit) continue;
    for (int i = threadIdx.x; i < cnt; i += 64) sidx[i] = val[beg + i];
    __syncthreads();
    const double4 C = cx[c];
    for (int i = threadIdx.x; i < cnt; i += 64) {
      const int me = sidx[i];
      int r = 0;
      for (int j = 0; j < cnt; j++) r += sidx[j] < me;
      const int pos = beg + r;
      perm[pos] = me;
      const double x = b[me].X[0], y = b[me].X[1], z = b[me].X[2], q = b[me].q;
      xs[pos] = make_double4(x, y, z, q);
      xq[pos] = make_float4(float(x - C.x), float(y - C.y), float(z - C.z), float(q));
      body_leaf[pos] = c;
    }
    __syncthreads();
  }
}

// Reference permutes X and q of the caller's array in place (p, F stay).
// Bodies back to the caller in tree order -- unless the build flagged a
// non-finite input (bit 1) or a leaf above ncrit (bit 2): the caller's
// array is then left as it was.
__global__ void __launch_bounds__(256) k_writeback(int64_t n, const double4 *__restrict__ xs,
                                                   exafmm_body *__restrict__ b, const int *__restrict__ flags) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n || (*flags & 3)) return;
  const double4 v = xs[i];
  b[i].X[0] = v.x;
  b[i].X[1] = v.y;
  b[i].X[2] = v.z;
  b[i].q = v.w;
}

// Sort depth from the largest prefix population of levels 1..7 (lmax[l]).
static int sort_depth(const int *lmax, int64_t n, int ncrit, bool forest, int lforce) {
  if (n <= ncrit && !forest) return 0;
  for (int l = std::max(1, lforce); l <= kHistLevels; l++)
    if (lmax[l] <= ncrit) return l;
  return kMaxLevel;
}

void writeback_bodies(Ctx &c, hipStream_t s) {
  const int64_t n = c.t.n;
  hipLaunchKernelGGL(k_writeback, dim3(ceil_div(n, 256)), dim3(256), 0, s, n, c.t.xs.p, c.bodies, c.t.misc.p);
  XF_LAUNCH();
  c.writeback_pending = false;
}

void tree_build(Ctx &c) {
  Tree &t = c.t;
  const int64_t n = t.n;
  hipStream_t s = c.s0;
  const int ncrit = c.cfg.ncrit;
  if (n > (int64_t(1) << 30)) fail(EXAFMM_ERR_ARG, "N above 2^30 is not supported");

  // misc layout (ints): [0] flags, [1..8] level max, [17] leaves, [18] cells
  // that split, [19, 20] runs and lanes sampled by k_keys, [24 + l] look-back tickets of level l's split, [46] of k_leaves
  t.misc.ensure(kMiscInts);
  t.bounds_part.ensure(kBoundsBlocks * kBoundsInts + 8);
  double *root = t.bounds_part.p + kBoundsBlocks * kBoundsInts;
  t.lcount.ensure(kMaxLevel + 2);
  t.lstart_d.ensure(kMaxLevel + 2);
  t.hist.ensure(kHistTotal);
  static_assert(hist_off(kHistLevels) % 4 == 0, "level 7 is cleared 16 bytes at a time");
  int4 *hist7 = reinterpret_cast<int4 *>(t.hist.p + hist_off(kHistLevels));

  // forest: per-problem roots under the problem-index cells
  const bool forest = c.forest_n > 0;
  const double4 *froots = forest ? c.forest_roots.p : nullptr;
  const int lforce = forest ? kForestLevel : 0;
  t.lroot = lforce;
  // bounds on the cells of each level (a depth of kMaxLevel until Ds is known)
  const int64_t ub_split = 8 * (n / (ncrit + 1)) + 8;
  auto level_bound = [&](int l) {
    int64_t u = std::min<int64_t>(l >= 10 ? n : (int64_t(1) << (3 * l)), n);
    // nodes of level l are children of level-(l-1) nodes holding > ncrit bodies
    return l > lforce ? std::min(u, ub_split) : u;  // (a forest's top levels split unconditionally)
  };
  auto cells_bound = [&](int Ds) {
    int64_t tot = 0;
    for (int l = 0; l <= Ds; l++) tot += level_bound(l);
    return tot;
  };
  // (true if an array was allocated again: the root cell in it is lost)
  auto ensure_cells = [&](int Ds) {
    return ensure_all(size_t(cells_bound(Ds)), t.cx, t.cbeg, t.ccnt, t.cchild, t.cnch, t.cparent, t.clevel, t.coct,
                      t.leaves);
  };
  const bool speculate = t.ds_hint >= 0;
  int Ds = t.ds_hint;
  // the root cell is written by the first launches: cells for the largest
  // depth the build can turn out to have (the histogram's, or the hint's)
  ensure_cells(speculate ? Ds : kHistLevels);
  const RootOut rout{root,    t.misc.p, t.lcount.p, t.lstart_d.p, t.cx.p, t.cbeg.p, t.ccnt.p, t.cparent.p,
                     t.clevel.p, n};
  if (forest) {
    hipLaunchKernelGGL(k_forest_init, dim3(256), dim3(256), 0, s, rout, hist7);
    XF_LAUNCH();
    t.forest_part.ensure(size_t(c.forest_n) * kForestShares * 6);
    hipLaunchKernelGGL(k_forest_bounds, dim3(kForestShares, c.forest_n), dim3(256), 0, s, c.bodies, c.forest_off.p,
                       t.forest_part.p, t.misc.p);
    XF_LAUNCH();
    hipLaunchKernelGGL(k_forest_roots, dim3(ceil_div(c.forest_n, 64)), dim3(64), 0, s, c.forest_off.p, t.forest_part.p,
                       c.forest_n, c.forest_roots.p);
    XF_LAUNCH();
  } else {
    hipLaunchKernelGGL(k_bounds_part, dim3(kBoundsBlocks), dim3(256), 0, s, c.bodies, n, t.bounds_part.p, hist7);
    XF_LAUNCH();
    hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(kBoundsBlocks), 0, s, t.bounds_part.p, rout);
    XF_LAUNCH();
  }

  t.key.ensure(n);
  t.key2.ensure(n);
  t.val.ensure(n);
  t.val2.ensure(n);
  // a tree expected to be deeper than the histogram takes it from the sorted keys
  const bool sorted_hist = speculate && Ds > kHistLevels;
  hipLaunchKernelGGL(sorted_hist ? k_keys<false> : k_keys<true>, dim3(ceil_div(n, kKeysThreads)), dim3(kKeysThreads), 0,
                     s, c.bodies, n, root, t.key.p, t.val.p, t.hist.p + hist_off(kHistLevels), froots,
                     forest ? c.forest_off.p : nullptr, c.forest_n, t.misc.p + 19);
  XF_LAUNCH();
  // one block per level-3 prefix (4096 level-7 bins each)
  t.hist_bmax.ensure(8 << (3 * 3));
  auto pyramid = [&] {
    hipLaunchKernelGGL(k_hist_pyramid, dim3(1 << (3 * 3)), dim3(1024), 0, s, t.hist.p, t.hist_bmax.p);
    XF_LAUNCH();
  };
  if (!sorted_hist) pyramid();

  // Sort depth Ds: the first level whose most populous prefix holds at
  // most ncrit bodies (kMaxLevel if none of levels 1..7 does).  It needs the
  // histogram on the host; instead of waiting for it here the build reuses
  // the previous call's depth and checks it at the level-size read below.
  // A depth at or above the true one builds the same tree (a cell splits
  // only above ncrit bodies, and each leaf keeps its bodies in input order),
  // so only a smaller one makes the build start over.
  c.pin_i.ensure(kPinInts);
  c.pin_d.ensure(4);
  int *hm = c.pin_i.p + kPinLevelMax;
  if (!speculate) {
    hipLaunchKernelGGL(k_hist_top, dim3(1), dim3(512), 0, s, t.hist.p, t.hist_bmax.p, t.misc.p);
    XF_LAUNCH();
    XF_HIP(hipMemcpyAsync(hm, t.misc.p, sizeof(int) * 9, hipMemcpyDeviceToHost, s));
    stream_wait(s);
    if (hm[0] & 1) fail(EXAFMM_ERR_ARG, "non-finite body coordinate or charge");
    Ds = sort_depth(hm, n, ncrit, forest, lforce);
  }

  // Bodies in the order of their top Ds octant digits: a counting sort on the
  // histogram up to its depth (2 - 3 launches where the radix sort takes three
  // per eight bits), the stable radix sort below.  Bodies in random order cost the
  // counting sort an atomic and a scattered write each, about 82 us per 10^6, a
  // radix pass 24: many of them take the radix sort as well, unless the last
  // build's came in tree order.  Builds of uniform bodies, counting / radix, random
  // order and tree order: 500,000 ncrit 64 (5 levels) 198 / 202 and 161 / 183 us, 10^6
  // ncrit 300 (5) 295 / 269 and 207 / 241, 4 x 10^6 ncrit 300 (5) 915 / 782 and 503 /
  // 595, 1.5 x 10^6 ncrit 64 (6) 386 / 383 and 266 / 297, 4 x 10^6 ncrit 64 (6) 945 /
  // 894 and 553 / 694.
  const bool place = Ds <= kHistLevels && (t.in_order || n < (Ds <= 5 ? kPlaceMax5 : kPlaceMax7));
  unsigned long long *k1 = t.key.p, *k2 = t.key2.p;
  int *v1 = t.val.p, *v2 = t.val2.p;
  if (place) {
    const int Dc = std::max(Ds, 3), bins = 1 << (3 * Dc);  // levels 1 and 2 are summed later
    t.cursor.ensure(bins);
    scan_exclusive(t.hist.p + hist_off(Dc), t.cursor.p, bins, t.scan_tmp, s);
    hipLaunchKernelGGL(k_place, dim3(ceil_div(n, 256)), dim3(256), 0, s, k1, n, 3 * (kMaxLevel - Dc), t.cursor.p, k2,
                       v1);
    XF_LAUNCH();
    k1 = k2;
  } else {
    radix_sort_pairs(k1, v1, k2, v2, int(n), 3 * (kMaxLevel - Ds), 3 * kMaxLevel, t.rs_hist, s);
    if (sorted_hist) {
      hipLaunchKernelGGL(k_hist_sorted, dim3(ceil_div(n, 256)), dim3(256), 0, s, k1, n,
                         t.hist.p + hist_off(kHistLevels));
      XF_LAUNCH();
      pyramid();
    }
  }

  // level-by-level split
  const int64_t ubtot = cells_bound(Ds);
  if (ensure_cells(Ds)) {  // (a first build deeper than the histogram: the root again)
    const RootOut again{root,    t.misc.p, t.lcount.p, t.lstart_d.p, t.cx.p, t.cbeg.p, t.ccnt.p, t.cparent.p,
                        t.clevel.p, n};
    hipLaunchKernelGGL(k_root, dim3(1), dim3(1), 0, s, again);
    XF_LAUNCH();
  }
  t.perm.ensure(n);
  t.xs.ensure(n);
  t.xq.ensure(n);
  t.body_leaf.ensure(n);
  const size_t words = size_t(ceil_div(ubtot, 1024)) + 1;
  if (t.lookback.cap < words || t.lookback_tag >= (1u << 24) - 64) {  // (a new tag per launch, 24 bits)
    t.lookback.ensure(words);
    XF_HIP(hipMemsetAsync(t.lookback.p, 0, sizeof(unsigned long long) * t.lookback.cap, s));
    t.lookback_tag = 0;
  }
  const int lfuse = std::min(Ds, kTopLevels);
  // (with a depth of 0 no level is split, but the histogram is still finished)
  hipLaunchKernelGGL(k_top_levels, dim3(1), dim3(kTopThreads), 0, s, lfuse, ncrit, lforce, t.lcount.p, t.lstart_d.p, k1,
                     t.hist.p, speculate ? t.hist_bmax.p : nullptr, t.misc.p, froots, t.cx.p, t.cbeg.p, t.ccnt.p,
                     t.cchild.p, t.cnch.p, t.cparent.p, t.clevel.p, t.coct.p, t.misc.p + 18);
  XF_LAUNCH();
  for (int l = lfuse; l < Ds; l++) {
    hipLaunchKernelGGL(k_split_level, dim3(ceil_div(level_bound(l), 1024)), dim3(1024), 0, s, l, ncrit, lforce,
                       t.lcount.p, t.lstart_d.p, k1, t.hist.p, froots, t.cx.p, t.cbeg.p, t.ccnt.p, t.cchild.p, t.cnch.p,
                       t.cparent.p, t.clevel.p, t.coct.p, t.misc.p + 18, t.misc.p + 24 + l, ++t.lookback_tag, t.lookback.p);
    XF_LAUNCH();
  }

  // Leaves, the gather into tree order and the write-back run before the
  // level sizes are read, so that read overlaps them: the counts come from
  // the device, and grids are sized from the bound ubtot.  A tree the checks
  // below reject or rebuild (flag bit 1 or 2) leaves the caller's bodies
  // untouched.
  hipLaunchKernelGGL(k_leaves, dim3(ceil_div(ubtot, 1024)), dim3(1024), 0, s, Ds, ncrit, t.lcount.p, t.lstart_d.p,
                     t.ccnt.p, t.cchild.p, t.cnch.p, t.leaves.p, t.misc.p, t.misc.p + 46, ++t.lookback_tag,
                     t.lookback.p);
  XF_LAUNCH();
  const TreeReport rep{t.lcount.p, t.misc.p, root, c.pin_i.p + kPinLevels, c.pin_i.p + kPinMisc, c.pin_d.p};
  hipLaunchKernelGGL(k_leaf_gather, dim3(int(std::min<int64_t>(ubtot, 16384))), dim3(64), sizeof(int) * ncrit, s,
                     t.leaves.p, t.misc.p + 17, t.cbeg.p, t.ccnt.p, t.cx.p, v1, c.bodies, t.perm.p, t.xs.p, t.xq.p,
                     t.body_leaf.p, ncrit, rep);
  XF_LAUNCH();
  if (c.defer_writeback)
    c.writeback_pending = true;
  else
    writeback_bodies(c, s);

  // level sizes, flags, level maxima, root
  const int *lc = c.pin_i.p + kPinLevels, *fl = c.pin_i.p + kPinMisc;
  const double *rootv = c.pin_d.p;
  stream_wait(s);
  if (fl[0] & 1) fail(EXAFMM_ERR_ARG, "non-finite body coordinate or charge");
  // The histogram fixes depths up to kHistLevels; a deeper tree was sorted
  // at the last tree's depth + 1, which is enough unless a cell of that
  // level still holds more than ncrit bodies (flag 2, below kMaxLevel).
  const int need = sort_depth(fl, n, ncrit, forest, lforce);
  const bool too_shallow = need <= kHistLevels ? need > Ds : (Ds < kMaxLevel && (fl[0] & 2));
  if (too_shallow) {  // build again at the depth the histogram gives
    t.ds_hint = need;
    tree_build(c);
    return;
  }
  for (int d = 0; d < 3; d++) t.X0[d] = rootv[d];
  t.R0 = rootv[3];
  if (fl[0] & 2) fail(EXAFMM_ERR_DEPTH, "more than ncrit bodies share a 21-level octant path");
  t.lstart.assign(1, 0);
  int depth = 0;
  for (int l = 0; l <= Ds; l++) {
    if (lc[l] == 0) break;
    depth = l;
    t.lstart.push_back(t.lstart.back() + lc[l]);
  }
  t.depth = depth;
  t.in_order = fl[20] >= 8 * int64_t(fl[19]);  // (random order: runs of one or two)
  t.ds_hint = need <= kHistLevels ? need : std::min(kMaxLevel, depth + 1);
  t.ncells = t.lstart.back();
  const int nc = int(t.ncells);
  // every cell either split or is a leaf (the scan above wrote the same
  // count to misc[17] for the kernels)
  t.nleaves = nc - fl[18];
  t.built = true;
}

// Reference numbering: the reference appends a parent's children block
// when it visits the parent, in DFS preorder (3d/build_tree.h:115-132).
void tree_ref_order(Ctx &c, std::vector<int64_t> &bfs2ref, std::vector<int64_t> &ref2bfs) {
  Tree &t = c.t;
  const int64_t nc = t.ncells;
  std::vector<int> cchild(nc), cnch(nc);
  XF_HIP(hipMemcpy(cchild.data(), t.cchild.p, sizeof(int) * nc, hipMemcpyDeviceToHost));
  XF_HIP(hipMemcpy(cnch.data(), t.cnch.p, sizeof(int) * nc, hipMemcpyDeviceToHost));
  bfs2ref.assign(nc, -1);
  ref2bfs.assign(nc, -1);
  bfs2ref[0] = 0;
  int64_t next = 1;
  std::vector<int> stack{0};
  while (!stack.empty()) {
    const int u = stack.back();
    stack.pop_back();
    if (cnch[u] == 0) continue;
    const int64_t first = next;
    next += cnch[u];
    for (int k = 0; k < cnch[u]; k++) bfs2ref[cchild[u] + k] = first + k;
    for (int k = cnch[u] - 1; k >= 0; k--) stack.push_back(cchild[u] + k);
  }
  for (int64_t i = 0; i < nc; i++) ref2bfs[bfs2ref[i]] = i;
}

void tree_export_cells(Ctx &c, exafmm_cell *out) {
  Tree &t = c.t;
  const int64_t nc = t.ncells;
  std::vector<int64_t> b2r, r2b;
  tree_ref_order(c, b2r, r2b);
  std::vector<double4> cx(nc);
  std::vector<int> cbeg(nc), ccnt(nc), cchild(nc), cnch(nc);
  XF_HIP(hipMemcpy(cx.data(), t.cx.p, sizeof(double4) * nc, hipMemcpyDeviceToHost));
  XF_HIP(hipMemcpy(cbeg.data(), t.cbeg.p, sizeof(int) * nc, hipMemcpyDeviceToHost));
  XF_HIP(hipMemcpy(ccnt.data(), t.ccnt.p, sizeof(int) * nc, hipMemcpyDeviceToHost));
  XF_HIP(hipMemcpy(cchild.data(), t.cchild.p, sizeof(int) * nc, hipMemcpyDeviceToHost));
  XF_HIP(hipMemcpy(cnch.data(), t.cnch.p, sizeof(int) * nc, hipMemcpyDeviceToHost));
  for (int64_t b = 0; b < nc; b++) {
    exafmm_cell &o = out[b2r[b]];
    o.nchild = cnch[b];
    o.nbody = ccnt[b];
    o.child = cnch[b] ? b2r[cchild[b]] : -1;
    o.body = cbeg[b];
    o.X[0] = cx[b].x;
    o.X[1] = cx[b].y;
    o.X[2] = cx[b].z;
    o.R = cx[b].w;
  }
}

}  // namespace xf
