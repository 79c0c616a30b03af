// m2l_mfma.hip -- M2L grouped by translation key, applied on MFMA.
//
// Reference: M2L 3d/kernel.h:233-260 (singular harmonics 3d/kernel.h:83-116).
//
// Radius scaling makes the translation operator of a pair depend only on
// its key (integer offset d in units of the finer radius, and the level
// difference): with M~_n^m = M_n^m / Rs^n and L~_j^k = L_j^k Rc^{j+1},
//   L~ = T(d) M~,  T = reference coefficients x I_{j+n}(d) x 2^{a(j+1) + b n},
// where Rc = Rf 2^a, Rs = Rf 2^b.  In real form (P^2 real degrees of freedom
// per expansion: Re M_n^0, Re/Im M_n^m for m > 0) T is a dense P^2 x P^2
// matrix, generated once per distinct key in FP64.
//
// Targets are grouped in tiles of 512 cells of one octant position (cells
// with the same position relative to their parent have the same key set away
// from the domain boundary and from changes of depth, whatever their level).
// For each key in a tile's key union the source columns are gathered and
// multiplied by the key's operator; all keys of a tile accumulate into the
// same MFMA accumulators, so each target's L is written once, without
// atomics, in a fixed order.
//
// Precision: FP32 uses v_mfma_f32_16x16x4_f32.  BF16X3 splits operator and
// multipoles into bf16 hi + lo parts and forms hi*hi + hi*lo + lo*hi with
// v_mfma_f32_16x16x32_bf16 (FP32 accumulate), ~16 significant bits per
// product.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "fmm_internal.h"
#include "fmm_ops.h"
#include "sk_schedule.h"

namespace xf {
using namespace xfd;

// GEMM workgroup: 16 waves over a tile of 512 target columns.  The columns
// form 32 subtiles of 16 (one MFMA column tile each); wave w takes subtiles w
// and 16 + w.  Neighbouring columns have like key sets, so a key's empty
// subtiles come in runs, and the interleaving spreads what is left over the
// waves (they meet at a barrier every round).  Two column tiles per wave keep
// the accumulators of nine row tiles within 128 registers: four waves per
// SIMD hide the gathers' latency (with four column tiles and two waves per
// SIMD they waited half their cycles).
constexpr int kGemmThreads = 1024;
constexpr int kGemmWaves = kGemmThreads / 64;
constexpr int kTileN = 512;
constexpr int kCT = kTileN / 16 / kGemmWaves;  // column tiles per wave
// tile column of a wave's column tile ct, lane l
__device__ inline int tile_col(int w, int ct, int lane) { return (ct * kGemmWaves + w) * 16 + (lane & 15); }
// Load through the scalar cache: uniform address, data written before the launch.
template <class T>
__device__ inline T uniform_load(const T *p) {
  return *reinterpret_cast<const __attribute__((address_space(4))) T *>(reinterpret_cast<uintptr_t>(p));
}
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

struct Geom {
  int P, PP, R;  // R = row tiles of 16 (rows padded to 16R)
  int K4;        // FP32 k-steps of 4
  int K32;       // BF16 k-steps of 32
};
// BF16 multipole rows: P^2 padded to a multiple of 8, plus a tail of zeros
// after the zero row that covers the last k-step's k-groups.
constexpr int kBf16Tail = 32;
static int bf16_row(const Geom &g) { return (g.PP + 7) / 8 * 8; }
// elements of each of the two BF16 cast arrays (hi, lo) of a tree of nc cells
static size_t bf16_cast_elems(const Geom &g, int64_t nc) { return size_t(nc + 1) * bf16_row(g) + kBf16Tail; }

static Geom geom(int P) {
  Geom g;
  g.P = P;
  g.PP = P * P;
  g.R = (g.PP + 15) / 16;
  g.K4 = (g.PP + 3) / 4;
  g.K32 = (g.PP + 31) / 32;
  return g;
}

// ---------------------------------------------------------------- tiles
constexpr int kTileUnroll = 8;  // list entries in flight per thread (list walks below)
// MurmurHash3's 32-bit finaliser: spreads key ids before taking the minimum.
__device__ inline unsigned mix32(unsigned h) {
  h ^= h >> 16;
  h *= 0x85ebca6bu;
  h ^= h >> 13;
  h *= 0xc2b2ae35u;
  h ^= h >> 16;
  return h;
}

// Three hashes make the sort key 56 bits, seven radix passes where one hash took
// three: a pass over the 37,449 cells of 2^20 uniform bodies takes 32 us beside P2P
// (which hides it: P2P outlasts the tile build there), over the 19,199 of 300,007
// clustered bodies 33 us.
constexpr int kMinHashes = 3;
constexpr int kGroupShift = 48, kSortBits = 56;

// Counters of the tile build (m2l_misc): group populations 0..255, then the
// plan [slots, tiles, cells in tiles, key set differs].
constexpr int kMiscPlan = 256, kMiscInts = 260;

// Sort key of a target cell: group in bits 48..55 (255 = no M2L) -- the
// octant, or (level, octant) with `by_level` -- and below it 16 bits each of the
// minima of kMinHashes hashes of its key ids: cells with similar key sets share
// such a minimum with a probability equal to the sets' Jaccard similarity, so
// sorting by them packs cells of like key sets into the same subtile (fewer
// empty GEMM columns; with one hash and ties in index order the GEMM of 1.5M
// clustered bodies took 4.80 ms, with three 4.46, beside P2P).
// One wave per cell: the lanes take the list entries in turn and the
// minimum hash is a wave reduction.
__global__ void __launch_bounds__(256) k_group_keys(int ncells, const double4 *__restrict__ cx,
                                                    const int *__restrict__ cparent, const int *__restrict__ clevel,
                                                    const int *__restrict__ m2l_beg, const int *__restrict__ m2l_cnt,
                                                    const int2 *__restrict__ list, int lmin, int by_level,
                                                    unsigned long long *__restrict__ key, int *__restrict__ val,
                                                    int *__restrict__ misc) {
  const int lane = threadIdx.x & (kWave - 1);
  const int c = blockIdx.x * (256 / kWave) + int(threadIdx.x / kWave);
  if (blockIdx.x == 0) {  // counters of the launches that follow
    misc[threadIdx.x] = 0;
    if (threadIdx.x < kMiscInts - 256) misc[256 + threadIdx.x] = 0;
  }
  if (c >= ncells) return;  // whole wave
  unsigned g = 255;
  unsigned long long mh = 0;
  // cells above level lmin take their M2L elsewhere (FP64, per pair)
  const int n = clevel[c] < lmin ? 0 : m2l_cnt[c];
  if (n > 0) {
    int o = 0;
    const int p = cparent[c];
    if (p >= 0) {
      const double4 a = cx[c], b = cx[p];
      o = (a.x > b.x) + ((a.y > b.y) << 1) + ((a.z > b.z) << 2);
    }
    g = (by_level ? unsigned(min(clevel[c], 30)) * 8 : 0u) + o;
    unsigned m[kMinHashes];
#pragma unroll
    for (int h = 0; h < kMinHashes; h++) m[h] = 0xffffffffu;
    const int b0 = m2l_beg[c];
    for (int i = lane; i < n; i += kWave) {
      const unsigned id = unsigned(list[b0 + i].y);
#pragma unroll
      for (int h = 0; h < kMinHashes; h++) m[h] = min(m[h], mix32(id + h * 0x9e3779b9u));
    }
#pragma unroll
    for (int h = 0; h < kMinHashes; h++) {
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) m[h] = min(m[h], unsigned(__shfl_xor(int(m[h]), d)));
      mh |= (unsigned long long)(m[h] >> 16) << (kGroupShift - 16 * (h + 1));
    }
  }
  if (lane == 0) {
    key[c] = (unsigned long long)g << kGroupShift | mh;
    val[c] = c;
  }
}

// Tiles from the group populations gc[0..254] (group 255 = cells without
// M2L, not tiled): each group's cells, in sorted order, are cut into tiles
// of at most kTileN.  Writes each tile's first cell and count, and plan[1] =
// tiles, plan[2] = cells in tiles.  (Launches of one workgroup like this one
// and k_tile_scan stay launches: run by the last workgroup of the launch before
// them, the agent-scope fences of every workgroup of that launch write back
// and invalidate the L2s under the P2P that runs beside it, which cost more.)
__global__ void __launch_bounds__(256) k_tile_plan(int *__restrict__ misc, int *__restrict__ tfirst,
                                                   int *__restrict__ tcount) {
  __shared__ int wt[4][2];
  const int gi = threadIdx.x, lane = gi & 63, w = gi >> 6;
  const int n = gi < 255 ? misc[gi] : 0, nt = (n + kTileN - 1) / kTileN;
  int it = nt, ic = n;
  for (int d = 1; d < 64; d <<= 1) {
    const int x = __shfl_up(it, d), y = __shfl_up(ic, d);
    if (lane >= d) {
      it += x;
      ic += y;
    }
  }
  if (lane == 63) {
    wt[w][0] = it;
    wt[w][1] = ic;
  }
  __syncthreads();
  for (int i = 0; i < w; i++) {
    it += wt[i][0];
    ic += wt[i][1];
  }
  if (gi == 255) {
    misc[kMiscPlan + 1] = it;
    misc[kMiscPlan + 2] = ic;
  }
  for (int j = 0; j * kTileN < n; j++) {
    tfirst[it - nt + j] = ic - n + j * kTileN;
    tcount[it - nt + j] = min(kTileN, n - j * kTileN);
  }
}

// The cells in sorted order and the group populations after the radix sort.
__global__ void __launch_bounds__(256) k_group_hist(int ncells, const unsigned long long *__restrict__ key,
                                                    const int *__restrict__ val, int *__restrict__ sorted,
                                                    int *__restrict__ misc) {
  __shared__ int h[256];
  h[threadIdx.x] = 0;
  __syncthreads();
  for (int c = blockIdx.x * 256 + threadIdx.x; c < ncells; c += gridDim.x * 256) {
    atomicAdd(&h[int(key[c] >> kGroupShift)], 1);
    sorted[c] = val[c];
  }
  __syncthreads();
  if (h[threadIdx.x]) atomicAdd(&misc[threadIdx.x], h[threadIdx.x]);
}

// Small trees: each cell's place is the number of cells that sort before it
// (lower key, or equal key and lower index).  A workgroup places 64 cells, its
// 16 waves counting over a sixteenth of the cells each (wave-uniform keys:
// scalar loads).  Quadratic, and one launch where the radix sort takes nine:
// at 16,384 cells it costs what they do.
constexpr int kCellRankMax = 16384;
__global__ void __launch_bounds__(1024) k_cell_rank(int n, const unsigned long long *__restrict__ key, int *__restrict__ sorted,
                                                    int *__restrict__ misc) {
  __shared__ int part[16][kWave];
  const int lane = threadIdx.x & (kWave - 1), w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int i = blockIdx.x * kWave + lane;
  const unsigned long long k = i < n ? key[i] : 0ull;
  const int j0 = w * n / 16, j1 = (w + 1) * n / 16, first = blockIdx.x * kWave;
  int r = 0;
  // before this workgroup's cells equal keys count, after them they do not
  for (int j = j0; j < min(j1, first); j++) r += key[j] <= k;
  for (int j = max(j0, first); j < min(j1, first + kWave); j++) r += key[j] < k || (key[j] == k && j < i);
  for (int j = max(j0, first + kWave); j < j1; j++) r += key[j] < k;
  part[w][lane] = r;
  __syncthreads();
  if (w == 0 && i < n) {
    r = 0;
    for (int q = 0; q < 16; q++) r += part[q][lane];
    sorted[r] = i;
    atomicAdd(&misc[int(k >> kGroupShift)], 1);
  }
}

// Tile kernels: one thread per target column walks that column's M2L list
// (entries (source << 5 | image, key id)), kTileUnroll entries in flight.

// Distinct keys of one tile: bitmap over key ids in LDS.
// Four threads per column (blockDim.x / 4 columns at a time), entries i = sub mod 4.
__device__ inline void tile_bitmap(const int *cells, int ncol, const int *beg, const int *cnt, const int2 *list,
                                   unsigned *bm, int nwords) {
  for (int i = threadIdx.x; i < nwords; i += blockDim.x) bm[i] = 0;
  __syncthreads();
  const int sub = threadIdx.x & 3;
  for (int t = threadIdx.x >> 2; t < ncol; t += blockDim.x >> 2) {
    const int c = cells[t];
    const int b = beg[c], n = cnt[c];
    for (int i0 = sub; i0 < n; i0 += 4 * kTileUnroll) {
      int id[kTileUnroll];
#pragma unroll
      for (int k = 0; k < kTileUnroll; k++) id[k] = i0 + 4 * k < n ? list[b + i0 + 4 * k].y : -1;
#pragma unroll
      for (int k = 0; k < kTileUnroll; k++)
        if (id[k] >= 0) atomicOr(&bm[id[k] >> 5], 1u << (id[k] & 31));
    }
  }
  __syncthreads();
}

// Key set and its size per tile (launched over the bound of tiles).  The
// launch also compares the key set with the one the operators were generated
// for (old_keys, null if there is none to compare with).
constexpr int kTileCountThreads = 1024;
__global__ void __launch_bounds__(kTileCountThreads)
    k_tile_count(const int *__restrict__ tfirst, const int *__restrict__ tcount, const int *__restrict__ sorted,
                 const int *__restrict__ beg, const int *__restrict__ cnt, const int2 *__restrict__ list, int nkeys,
                 int *__restrict__ misc, int *__restrict__ tU, unsigned *__restrict__ tbits,
                 const unsigned long long *__restrict__ keys, const unsigned long long *__restrict__ old_keys) {
  extern __shared__ unsigned bm[];
  __shared__ int tot;
  const int nwords = (nkeys + 31) / 32, ntiles = misc[kMiscPlan + 1];
  if (int(blockIdx.x) < ntiles) {
    const int *cells = sorted + tfirst[blockIdx.x];
    const int ncol = tcount[blockIdx.x];
    tile_bitmap(cells, ncol, beg, cnt, list, bm, nwords);
    if (threadIdx.x == 0) tot = 0;
    __syncthreads();
    int s = 0;
    for (int i = threadIdx.x; i < nwords; i += blockDim.x) {
      s += __popc(bm[i]);
      tbits[int64_t(blockIdx.x) * nwords + i] = bm[i];  // the key set, for k_tile_fill
    }
    atomicAdd(&tot, s);
    __syncthreads();
    if (threadIdx.x == 0) tU[blockIdx.x] = tot;
  }
  if (old_keys)
    for (int i = blockIdx.x * kTileCountThreads + threadIdx.x; i < nkeys; i += gridDim.x * kTileCountThreads)
      if (keys[i] != old_keys[i]) atomicOr(&misc[kMiscPlan + 3], 1);
}

// Tile bases: exclusive scan of the slot counts (one workgroup), and the plan
// for the host (pinned memory).
__global__ void __launch_bounds__(kTileCountThreads) k_tile_scan(const int *__restrict__ misc,
                                                                 const int *__restrict__ tU, int *__restrict__ tbase,
                                                                 int *host_plan) {
  __shared__ int wt[kTileCountThreads / kWave];
  const int ntiles = misc[kMiscPlan + 1];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  int carry = 0;
  for (int t0 = 0; t0 < ntiles; t0 += kTileCountThreads) {
    const int t = t0 + threadIdx.x;
    const int v = t < ntiles ? tU[t] : 0;
    int incl = v;
    for (int d = 1; d < kWave; d <<= 1) {
      const int x = __shfl_up(incl, d);
      if (lane >= d) incl += x;
    }
    if (lane == kWave - 1) wt[w] = incl;
    __syncthreads();
    int before = carry, all = 0;
    for (int i = 0; i < kTileCountThreads / kWave; i++) {
      before += i < w ? wt[i] : 0;
      all += wt[i];
    }
    if (t < ntiles) tbase[t] = before + incl - v;
    carry += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const int plan[4] = {carry, ntiles, misc[kMiscPlan + 2], misc[kMiscPlan + 3]};
    for (int i = 0; i < 4; i++) __hip_atomic_store(host_plan + i, plan[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Key list (ascending) and source matrix [U][tn] (-1 = no pair) of a tile.
// Workgroup (tile, q) owns columns 64q .. 64q + 63: it marks them empty in
// every key row, then four threads per column walk that column's M2L list
// (entries i = sub mod 4) and write the source cell into the key's row.
// The key set comes from k_tile_count's bitmap.  Byte q of a key's mask
// (tmask, 8 bytes per slot) gets one bit per subtile of 16 columns that holds
// a pair; a wave fills one subtile.
__global__ void __launch_bounds__(256) k_tile_fill(const int *__restrict__ tfirst, const int *__restrict__ tcount,
                                                   const int *__restrict__ sorted, const int *__restrict__ beg,
                                                   const int *__restrict__ cnt, const int2 *__restrict__ list,
                                                   int nkeys, const int *__restrict__ tbase,
                                                   const unsigned *__restrict__ tbits, int *__restrict__ tkeys,
                                                   int *__restrict__ tmat, unsigned char *__restrict__ tmask) {
  extern __shared__ unsigned bm[];
  constexpr int tn = kTileN;
  const int nwords = (nkeys + 31) / 32;
  unsigned *rank = bm + nwords;  // exclusive popcount prefix per word
  unsigned *hit = rank + nwords;  // [4 subtiles][nwords]: key ranks with a pair in the subtile
  for (int i = threadIdx.x; i < 4 * nwords; i += blockDim.x) hit[i] = 0;
  const int tile = blockIdx.x, q = blockIdx.y;
  const int *cells = sorted + tfirst[tile];
  const int ncol = tcount[tile];
  for (int i = threadIdx.x; i < nwords; i += blockDim.x) bm[i] = tbits[int64_t(tile) * nwords + i];
  // exclusive prefix of the word popcounts (block scan in chunks of 256 words)
  __shared__ int carry;
  __shared__ int wsum[256 / 64];
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int w0 = 0; w0 < nwords; w0 += 256) {
    const int i = w0 + threadIdx.x;
    const int v = i < nwords ? __popc(bm[i]) : 0;
    int incl = v;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int u = __shfl_up(incl, d);
      if (lane >= d) incl += u;
    }
    if (lane == 63) wsum[wv] = incl;
    __syncthreads();
    int before = carry;
    for (int k = 0; k < wv; k++) before += wsum[k];
    if (i < nwords) rank[i] = before + incl - v;
    __syncthreads();
    if (threadIdx.x == 255) carry = before + incl;
    __syncthreads();
  }
  const int base = tbase[tile];
  const int U = carry;
  if (q == 0) {
    for (int i = threadIdx.x; i < nwords; i += blockDim.x) {
      unsigned w = bm[i];
      int r = rank[i];
      while (w) {
        const int bt = __ffs(w) - 1;
        w &= w - 1;
        tkeys[base + r++] = i * 32 + bt;
      }
    }
  }
  for (int i = threadIdx.x; i < U * 64; i += blockDim.x)
    tmat[(int64_t(base) + i / 64) * tn + q * 64 + (i & 63)] = -1;
  __syncthreads();
  const int col = q * 64 + (threadIdx.x >> 2), sub = threadIdx.x & 3;
  if (col < ncol) {
    const int c = cells[col];
    const int b = beg[c], n = cnt[c];
    for (int i0 = sub; i0 < n; i0 += 4 * kTileUnroll) {
      int2 en[kTileUnroll];
#pragma unroll
      for (int k = 0; k < kTileUnroll; k++) {
        const int i = i0 + 4 * k;
        en[k] = i < n ? list[b + i] : make_int2(0, -1);
      }
#pragma unroll
      for (int k = 0; k < kTileUnroll; k++) {
        const int id = en[k].y;
        if (id < 0) continue;
        const unsigned w = bm[id >> 5];
        const int r = rank[id >> 5] + __popc(w & ((1u << (id & 31)) - 1u));
        tmat[(int64_t(base) + r) * tn + col] = en[k].x >> 5;  // source cell (the image is part of the key)
        atomicOr(&hit[(threadIdx.x >> 6) * nwords + (r >> 5)], 1u << (r & 31));
      }
    }
  }
  __syncthreads();
  for (int r = threadIdx.x; r < U; r += blockDim.x) {
    unsigned m = 0;
    for (int k = 0; k < 4; k++) m |= ((hit[k * nwords + (r >> 5)] >> (r & 31)) & 1u) << k;
    tmask[(int64_t(base) + r) * 8 + q] = (unsigned char)m;
  }
}

// Learned orders are run in a few order classes (ranges of orders, one
// GEMM launch each): of[p] = class of order p, hi[k] = highest order of
// class k.
struct OrderClasses {
  int n;
  unsigned char of[kMaxP + 1], hi[kMaxP + 1];
};

// Each tile's slots grouped by order class (ascending class, key order
// within a class), so that one GEMM launch per class covers a contiguous
// run of every tile's slots.  One wave per tile; per 64 slots, one ballot
// per class gives every slot its rank.  perm[tbase[t] + j] = slot of the
// j-th slot of tile t in that grouping; cls[o * ts + t] = tbase[t] + first
// grouped slot of class o in tile t, cls[(ncls + o) * ts + t] = their count.
__global__ void __launch_bounds__(256) k_order_partition(int ntiles, int ts, const int *__restrict__ tbase,
                                                         const int *__restrict__ tU,
                                                         const unsigned char *__restrict__ tkp, OrderClasses oc,
                                                         int *__restrict__ perm, int *__restrict__ cls) {
  const int ncls = oc.n;
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + int(threadIdx.x >> 6);
  if (t >= ntiles) return;  // whole wave
  const int b = tbase[t], U = tU[t];
  const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;
  auto cls_of = [&](int u) { return u < U ? int(oc.of[min(int(tkp[b + u]), kMaxP)]) : -1; };
  int cnt = 0;  // lane o < ncls: slots of class o
  for (int u0 = 0; u0 < U; u0 += 64) {
    const int o = cls_of(u0 + lane);
    for (int k = 0; k < ncls; k++) {
      const unsigned long long m = __ballot(o == k);
      if (lane == k) cnt += __popcll(m);
    }
  }
  // exclusive prefix of the counts over the orders
  int incl = cnt;
  for (int d = 1; d < 64; d <<= 1) {
    const int v = __shfl_up(incl, d);
    if (lane >= d) incl += v;
  }
  int run = incl - cnt;
  if (lane < ncls) {
    cls[int64_t(lane) * ts + t] = b + run;
    cls[int64_t(ncls + lane) * ts + t] = cnt;
  }
  for (int u0 = 0; u0 < U; u0 += 64) {
    const int o = cls_of(u0 + lane);
    for (int k = 0; k < ncls; k++) {
      const unsigned long long m = __ballot(o == k);
      if (!m) continue;
      const int at = __shfl(run, k);
      if (o == k) perm[b + at + __popcll(m & below)] = b + u0 + lane;
      if (lane == k) run += __popcll(m);
    }
  }
}

// Per order (wave o), the exclusive prefix over the tiles of that order's
// slot counts, and their total: the stream-K schedule of the order's launch.
__global__ void __launch_bounds__(1024) k_order_prefix(int ntiles, int ts, int ncls, int *__restrict__ cls) {
  const int lane = threadIdx.x & 63, o = int(threadIdx.x >> 6);
  if (o >= ncls) return;
  const int *cnt = cls + int64_t(ncls + o) * ts;
  int *pre = cls + int64_t(2 * ncls + o) * ts;
  int carry = 0;
  for (int t0 = 0; t0 < ntiles; t0 += 64) {
    const int t = t0 + lane;
    const int v = t < ntiles ? cnt[t] : 0;
    int incl = v;
    for (int d = 1; d < 64; d <<= 1) {
      const int u = __shfl_up(incl, d);
      if (lane >= d) incl += u;
    }
    if (t < ntiles) pre[t] = carry + incl - v;
    carry += __shfl(incl, 63);
  }
  if (lane == 0) cls[int64_t(3 * ncls) * ts + o] = carry;
}

// ---------------------------------------------------------------- operands
// GEMM operands from the scaled FP64 multipoles M~ (P^2 per cell, rows of
// KP): FP32 copy, or bf16 hi + lo split (hi = bf16(x), lo = bf16(x - hi)).
// Row ncells is the zero row; `tail` more zeros follow it, so a k-group load
// of the zero row past KP stays inside the array and reads zeros.
__global__ void __launch_bounds__(256) k_mt(int PP, int KP, int ncells, int tail, const double *__restrict__ M,
                                            float *__restrict__ mt32, __bf16 *__restrict__ mhi,
                                            __bf16 *__restrict__ mlo) {
  const int64_t g = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int c = int(g / KP), r = int(g % KP);
  if (g >= int64_t(ncells + 1) * KP + tail) return;
  // row ncells is all zeros: the GEMM's loads for empty slots read it
  const float v = (c < ncells && r < PP) ? float(M[int64_t(c) * PP + r]) : 0.0f;
  if (mt32) mt32[g] = v;
  if (mhi) {
    const __bf16 h = __bf16(v);
    mhi[g] = h;
    mlo[g] = __bf16(v - float(h));
  }
}

// One workgroup per key: singular harmonics of d in FP64, then the operator
// in MFMA fragment order.
//  FP32 (16x16x4):  op32[key][kk][r][lane], element (row, kcol):
//                   r = row/16, kk = kcol/4, lane = (kcol%4)*16 + row%16
//  BF16 (16x16x32): ophi/oplo[key][kk][r][lane][8], element (row, kcol):
//                   r = row/16, kk = kcol/32, lane = ((kcol%32)/8)*16 + row%16
__global__ void __launch_bounds__(256) k_ops_gen(int P, int fillP, int R, int K4, int K32, double R0, double cycle,
                                                 const unsigned long long *__restrict__ keys, float *__restrict__ op32,
                                                 __bf16 *__restrict__ ophi, __bf16 *__restrict__ oplo) {
  __shared__ cpx<double> I[(2 * kMaxP) * (2 * kMaxP + 1) / 2];
  const int id = blockIdx.x;
  double dx, dy, dz;
  int a, b;
  key_at(keys, id, R0, cycle, dx, dy, dz, a, b);
  if (threadIdx.x < fillP) singular_column(threadIdx.x, fillP, dx, dy, dz, I);
  __syncthreads();
  if (op32) {
    const int64_t per = int64_t(K4) * R * 64;
    for (int64_t e = threadIdx.x; e < per; e += blockDim.x) {
      const int lane = int(e % 64), r = int((e / 64) % R), kk = int(e / (64 * R));
      const int row = r * 16 + lane % 16, kc = kk * 4 + lane / 16;
      op32[id * per + e] = float(op_entry(P, fillP, row, kc, a, b, I));
    }
  }
  if (ophi) {
    const int64_t per = int64_t(K32) * R * 64 * 8;
    for (int64_t e = threadIdx.x; e < per; e += blockDim.x) {
      const int i = int(e % 8), lane = int((e / 8) % 64), r = int((e / 512) % R), kk = int(e / (512 * R));
      const int row = r * 16 + lane % 16, kc = kk * 32 + (lane / 16) * 8 + i;
      const float v = float(op_entry(P, fillP, row, kc, a, b, I));
      const __bf16 h = __bf16(v);
      ophi[id * per + e] = h;
      oplo[id * per + e] = __bf16(v - float(h));
    }
  }
}

// ---------------------------------------------------------------- GEMM
// One workgroup = one tile of up to 512 targets and a block of RTB row
// tiles (blockIdx.y); a wave holds the accumulators of its column tiles
// and all RTB row tiles, so each source multipole is fetched once per tile and
// row block.  The operators are staged global -> LDS (global_load_lds, no
// register round trip) in rounds, the next round while the current one is
// multiplied, with one wait and barrier per round; a wave loads its next
// k-step's source multipoles as soon as it has issued the current one's
// products.
constexpr int kGemmMaxRT = 9;     // row tiles per wave (8 accumulator registers each)
constexpr int kGemmMaxRTF32 = 8;  // the FP32 kernel's

template <int RH>
__device__ inline void write_locals(int PP, int rbase, int nr, const int *cells, int ncol, int w,
                                    const v4f (&acc)[RH][kCT], int lane, double *L) {
#pragma unroll
  for (int ct = 0; ct < kCT; ct++) {
    const int col = tile_col(w, ct, lane);
    if (col >= ncol) continue;
    double *Lc = L + int64_t(cells[col]) * PP;
#pragma unroll
    for (int r = 0; r < RH; r++) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int row = (rbase + r) * 16 + 4 * (lane >> 4) + i;
        // row tiles of this block only (another block owns the next ones)
        if (r < nr && row < PP) Lc[row] += double(acc[r][ct][i]);
      }
    }
  }
}

// Split-key variant: this workgroup's share of the locals, stored (each
// (cell, row) of a tile belongs to one workgroup per key slice).
template <int RH>
__device__ inline void write_partial(int PP, int rbase, int nr, const int *cells, int ncol, int w,
                                     const v4f (&acc)[RH][kCT], int lane, float *Lp) {
  // opaque: the row tests and offsets below are then computed here, not hoisted
  // out of a stream-K workgroup's segment loop into registers it lacks
  asm volatile("" : "+s"(PP), "+v"(lane));
#pragma unroll
  for (int ct = 0; ct < kCT; ct++) {
    const int col = tile_col(w, ct, lane);
    if (col >= ncol) continue;
    float *Lc = Lp + int64_t(cells ? cells[col] : col) * PP;
#pragma unroll
    for (int r = 0; r < RH; r++) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int row = (rbase + r) * 16 + 4 * (lane >> 4) + i;
        if (r < nr && row < PP) Lc[row] = acc[r][ct][i];
      }
    }
  }
}

// Adds the key slices of the split-key GEMM into the locals (fixed order).
__global__ void k_combine_slices(int PP, int64_t ncells, int nslice, const int *__restrict__ sorted, int ncell_tiled,
                                 const float *__restrict__ Lpart, double *__restrict__ L) {
  const int64_t g = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (g >= int64_t(ncell_tiled) * PP) return;
  const int c = sorted[g / PP], r = int(g % PP);
  double s = 0.0;
  for (int z = 0; z < nslice; z++) s += double(Lpart[(int64_t(z) * ncells + c) * PP + r]);
  L[int64_t(c) * PP + r] += s;
}

// s_waitcnt immediates (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt
// 6:4, lgkmcnt 11:8) that wait for vmcnt <= N and nothing else.
constexpr int waitcnt_vm(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }
constexpr int kWaitVm0 = waitcnt_vm(0);

// Row of the full operator layout [kk][row tile][lane] for run c of a
// block's staged copy (c = kk * nrt + local row tile).
__device__ inline int op_run(int c, int nrt, int RT, int rt0) {
  const int kk = c / nrt, rl = c % nrt;
  return kk * RT + rt0 + rl;
}

// FP32 form: a workgroup per tile and row block, key slices where tiles are few;
// subtiles without a pair of a key are not multiplied (tiles that mix levels have
// larger key unions).  A k-step's operator rows are read together, ahead of the
// branches on the subtile bits.  Kernel alone, us, against tiles of one level and
// every column multiplied: 131,626 uniform bodies, ncrit 32, theta 0.3, order 6 /
// 9 / 13: 1,443 / 5,045 / 16,102 -> 1,429 / 4,702 / 16,271; theta 0.4, order 9:
// 2,391 -> 2,190; 30,000, ncrit 16, order 9: 2,531 -> 1,362; 20,000, order 16: 16,733
// -> 6,461; 500,000, ncrit 64, order 8: 2,437 -> 2,571; 10^6, theta 0.5, order 8: 819
// -> 698; 131,626 clustered, order 9: 13,956 -> 7,020; 50,000 periodic, order 9:
// 4,378 -> 3,972.  (Mixed levels with every column multiplied: 6,831 where 5,045 is
// given, 20,607 for 16,102.)
template <int RH>
__global__ void __launch_bounds__(kGemmThreads) k_m2l_f32(int PP, int RT, int RTB, int K4, int KP,
                                                          const int *__restrict__ tfirst,
                                                          const int *__restrict__ tcount,
                                                          const int *__restrict__ tbase, const int *__restrict__ tU,
                                                          const int *__restrict__ sorted,
                                                          const int *__restrict__ tkeys,
                                                          const int *__restrict__ tmat,
                                                          const unsigned long long *__restrict__ tmask,
                                                          const float *__restrict__ op32,
                                                          const float *__restrict__ mt,
                                                          const unsigned char *__restrict__ tkp, int kr,
                                                          int64_t ncells, float *__restrict__ Lpart,
                                                          double *__restrict__ L) {
  extern __shared__ float As[];
  constexpr int TN = kTileN;
  // wave index read through a scalar register: the k-step and key loops
  // below then branch uniformly instead of under execution masks
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = blockIdx.x;
  const int ncol = tcount[tile];
  // keys of this workgroup: slice blockIdx.z of gridDim.z of the tile's keys
  const int Ut = tU[tile], ub = int(int64_t(Ut) * blockIdx.z / gridDim.z),
            ue = int(int64_t(Ut) * (blockIdx.z + 1) / gridDim.z);
  const int U = ue - ub, base = tbase[tile] + ub;
  const int rt0 = blockIdx.y * RTB;
  const int nrt = min(RTB, RT - rt0);
  const int kq = lane >> 4;
  v4f acc[RH][kCT];
#pragma unroll
  for (int r = 0; r < RH; r++)
#pragma unroll
    for (int ct = 0; ct < kCT; ct++) acc[r][ct] = v4f{0, 0, 0, 0};
  const int64_t per = int64_t(K4) * RT * 64;
  const int NC = K4 * nrt;  // runs of 64 floats per staged block
  const int BUF = NC * 64;  // floats per LDS buffer
  // order of key u (tkp: per-key orders of a variable-order evaluation):
  // k-steps and row tiles of this block that it needs, and its K bound
  auto kcols = [&](int u) { const int p = tkp ? tkp[base + u] : (int)__builtin_sqrtf(float(PP) + 0.5f); return p * p; };
  auto ksteps = [&](int kc) { return (kc + 3) / 4; };
  auto rtiles = [&](int kc) { return max(0, min(nrt, (kc + 15) / 16 - rt0)); };
  if (U > 0) {
    // LDS: operator slots [2 buffers][kr keys][BUF], then the keys' column
    // sources [3 buffers][kr keys][TN]; staging as in the BF16 kernel below
    int *Ts = reinterpret_cast<int *>(As + size_t(2) * kr * BUF);
    const int R = (U + kr - 1) / kr;
    auto stage_ops = [&](int r) {
      for (int u = r * kr; u < min(r * kr + kr, U); u++) {
        float *dst = As + size_t((r & 1) * kr + u - r * kr) * BUF;
        const int kc = kcols(u), ks = ksteps(kc), nr = rtiles(kc);
        const float *Ak = op32 + int64_t(tkeys[base + u]) * per;
        for (int j = w; j < ks * nr; j += kGemmWaves) {
          const int kk = j / nr, rl = j - kk * nr, c = kk * nrt + rl;
          __builtin_amdgcn_global_load_lds(Ak + int64_t(op_run(c, nrt, RT, rt0)) * 64 + lane, dst + c * 64, 4, 0, 0);
        }
      }
    };
    auto stage_src = [&](int r) {
      const int nu = min(kr, U - r * kr);
      for (int j = w; j < TN / 64 * nu; j += kGemmWaves) {
        const int ui = j / (TN / 64), q = j % (TN / 64);
        __builtin_amdgcn_global_load_lds(tmat + (int64_t(base) + r * kr + ui) * TN + q * 64 + lane,
                                         Ts + ((r % 3) * kr + ui) * TN + q * 64, 4, 0, 0);
      }
    };
    auto col_src = [&](int u, int (&sc)[kCT]) {
      const int *T = Ts + (((u / kr) % 3) * kr + u % kr) * TN;
#pragma unroll
      for (int ct = 0; ct < kCT; ct++) sc[ct] = T[tile_col(w, ct, lane)];
    };
    // empty slots and k at or past the key's K bound read the zero row
    // (index ncells): unconditional loads stay in flight until used
    auto load_b = [&](const int (&sc)[kCT], int kk, int kc, float (&bv)[kCT]) {
      const int k = kk * 4 + kq;
#pragma unroll
      for (int ct = 0; ct < kCT; ct++) bv[ct] = mt[int64_t(sc[ct] >= 0 && k < kc ? sc[ct] : ncells) * KP + k];
    };
    // bit ct: this wave's column tile ct holds a pair of key u (u < U)
    auto mask_of = [&](int u) {
      const unsigned long long m = uniform_load(tmask + base + u) >> (8 * (w >> 2) + (w & 3));
      return int((m & 1) | ((m >> 31) & 2));
    };
    stage_ops(0);
    stage_src(0);
    if (R > 1) stage_src(1);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int src[kCT], nsrc[kCT];
    int m = mask_of(0);
    float bcur[kCT], bnext[kCT];
    col_src(0, src);
    int kc = kcols(0);
    if (ksteps(kc) > 0) load_b(src, 0, kc, bnext);
    for (int r = 0; r < R; r++) {
      if (r + 1 < R) stage_ops(r + 1);
      if (r + 2 < R) stage_src(r + 2);
      __builtin_amdgcn_sched_barrier(0);
      bool b_after = false;
      const int u0 = r * kr, u1 = min(u0 + kr, U);
      for (int u = u0; u < u1; u++) {
        const float *Acur = As + size_t((r & 1) * kr + u - u0) * BUF;
        const int ks = ksteps(kc), nr = rtiles(kc);
        const int kc_next = u + 1 < U ? kcols(u + 1) : 0;
        const bool next = u + 1 < U && ksteps(kc_next) > 0;
        if (u + 1 < U) col_src(u + 1, nsrc);
        const int m_next = mask_of(min(u + 1, U - 1));
        for (int kk = 0; kk < ks; kk++) {
#pragma unroll
          for (int ct = 0; ct < kCT; ct++) bcur[ct] = bnext[ct];
          if (kk + 1 < ks) {
            load_b(src, kk + 1, kc, bnext);
            b_after = true;
          } else if (next) {
            load_b(nsrc, 0, kc_next, bnext);
            b_after = true;
          }
          if (m == 0) continue;  // uniform, as the subtile bits below
          const float *Ak = Acur + kk * nrt * 64 + lane;
          float a[RH];
#pragma unroll
          for (int r2 = 0; r2 < RH; r2++) a[r2] = Ak[min(r2, nr - 1) * 64];
#pragma unroll
          for (int ct = 0; ct < kCT; ct++)
            if (m & (1 << ct)) {
#pragma unroll
              for (int r2 = 0; r2 < RH; r2++)
                if (r2 < nr) acc[r2][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r2], bcur[ct], acc[r2][ct], 0, 0, 0);
            }
        }
        if (ks <= 0 && next) {
          load_b(nsrc, 0, kc_next, bnext);
          b_after = true;
        }
#pragma unroll
        for (int ct = 0; ct < kCT; ct++) src[ct] = nsrc[ct];
        kc = kc_next;
        m = m_next;
      }
      // staging of this round's start landed (only the kCT loads of the last
      // B prefetch are younger); then every wave is done with this round
      if (b_after)
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(kCT));
      else
        __builtin_amdgcn_s_waitcnt(kWaitVm0);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __builtin_amdgcn_s_barrier();
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (Lpart)
    write_partial<RH>(PP, rt0, nrt, sorted + tfirst[tile], ncol, w, acc, lane, Lpart + int64_t(blockIdx.z) * ncells * PP);
  else
    write_locals<RH>(PP, rt0, nrt, sorted + tfirst[tile], ncol, w, acc, lane, L);
}

// Order of one GEMM launch: pl (k bound pl^2 of every key, unless the
// per-slot orders tkp are given), the row tiles RTo and k-steps K32o it
// covers (of the RT x K32 of the operator layout, which holds order
// sqrt(PP)), and an optional slot permutation (slot u of tile t is
// perm[tbase[t] + u]).
struct OrderPass {
  int pl, RTo, K32o;
  const int *perm;
};

// What a BF16x3 GEMM launch reads of one tree: tiles and their keys, sources
// and subtile masks, operators, cast multipoles.
struct GemmIn {
  const int *tfirst, *tcount, *tU, *sorted, *tkeys, *tmat;
  const unsigned long long *tmask;
  const v8bf *ophi, *oplo;
  const __bf16 *mhi, *mlo;
  int64_t ncells;
};

// The k-steps of the tile's keys form one sequence of units (key u, k-step
// kk).  A round is G units (two LDS buffers of G units: a whole key need not
// fit, a small one takes a fraction of a round); at its start the next
// round's operators are staged into the other buffer, and the tile-matrix
// rows of the keys up to kGemmLook past them into a ring, so a wave finds its
// next key's sources in LDS.
//
// A key's subtile masks (tile fill) tell each wave, a block of 64 keys at a
// time, which keys hold a pair in its columns: the wave skips the others
// outright and the empty column tiles of the rest, and loads the multipoles
// of its next non-empty key ahead.  Clustered trees leave most subtiles of a
// tile's key union empty (200,000 bodies, 90% of them in a Plummer sphere:
// 56% with 16 columns, 87% with the whole tile).
//
// What bounds it: the waits for gathered multipoles and staged operators
// (MFMA busy a third to a half of the time; the fetch stays near 2 TB/s).
// Against eight waves of four contiguous column tiles each, whole keys per
// round, every column multiplied: 1.5M clustered bodies, order 12: 7.1 -> 3.8
// ms; 10,000 uniform bodies, order 10: 101 -> 37 us; 2^20 uniform: 0.70 -> 0.62
// ms; 12 problems of a batch graph: 6.5 -> 0.83 ms (with the stream-K launch).
//
// The body runs slots first .. first + U - 1 of a tile, row block `by`.
// Output: added into the FP64 locals L (Lpart null), or stored as FP32
// partial locals, by cell (Lpart + cell * PP, part_local false) or by tile
// column (Lpart + col * PP).
//
// VAR: learned orders (slot permutation, an order and so K bound and row
// tiles per slot).  Without it every key has the order op.pl of the operators
// and all RH row tiles are multiplied (those past a shorter last row block
// read staged bytes of other rows and are not written).
constexpr int kGemmLook = 4;
template <int RH, bool VAR>
__device__ __attribute__((always_inline)) inline void m2l_bf16x3_body(const GemmIn &g, int tile, int by, int first,
                                                                      int U, bool part_local, int PP, int RT, int RTB,
                                                                      int K32, int KP, OrderPass op,
                                                                      const unsigned char *__restrict__ tkp, int G,
                                                                      int ring, float *__restrict__ Lpart,
                                                                      double *__restrict__ L) {
  extern __shared__ v8bf Ab[];
  constexpr int TN = kTileN;
  // wave index read through a scalar register: the unit loop below then
  // branches uniformly instead of under execution masks
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ncol = g.tcount[tile];
  // a tile without keys in this launch adds nothing to the locals
  if (U <= 0 && !Lpart) return;
  const int rt0 = by * RTB;
  const int nrt = min(RTB, op.RTo - rt0);
  const int kq = lane >> 4;
  v4f acc[RH][kCT];
#pragma unroll
  for (int r = 0; r < RH; r++)
#pragma unroll
    for (int ct = 0; ct < kCT; ct++) acc[r][ct] = v4f{0, 0, 0, 0};
  const int64_t per = int64_t(K32) * RT * 64;  // v8bf per key and part
  const int KS = op.K32o;                      // units per key
  const int UE = nrt * 128;                    // v8bf per staged unit: hi rows, lo rows
  auto slot = [&](int u) { return VAR && op.perm ? uniform_load(op.perm + first + u) : first + u; };
  // order of key u (tkp: per-key orders of a variable-order evaluation):
  // k-steps and row tiles of this block that it needs, and its K bound
  auto kcols = [&](int u) {
    const int p = VAR && tkp ? int(uniform_load(tkp + slot(u))) : op.pl;
    return p * p;
  };
  auto ksteps = [&](int kc) { return VAR ? (kc + 31) / 32 : KS; };
  auto rtiles = [&](int kc) { return VAR ? max(0, min(nrt, (kc + 15) / 16 - rt0)) : nrt; };
  if (U > 0) {
    int *Ts = reinterpret_cast<int *>(Ab + size_t(2) * G * UE);
    const int N = U * KS, R = (N + G - 1) / G;
    int su = 0, sk = 0;  // the next unit to stage
    auto stage_ops = [&](int r) {
      const int n = min(G, N - r * G);
      int off = 0;
      for (int i = 0; i < n; i++) {
        const int kc = kcols(su);
        if (sk < ksteps(kc)) {
          const int nr = rtiles(kc);
          const int64_t o = int64_t(uniform_load(g.tkeys + slot(su))) * per + int64_t(sk * RT + rt0) * 64;
          v8bf *dst = Ab + size_t((r & 1) * G + i) * UE;
          for (int q = (w - off) & (kGemmWaves - 1); q < 2 * nr; q += kGemmWaves) {
            const int part = q >= nr, rl = part ? q - nr : q;
            __builtin_amdgcn_global_load_lds((part ? g.oplo : g.ophi) + o + rl * 64 + lane,
                                             dst + (part * nrt + rl) * 64, 16, 0, 0);
          }
          off += 2 * nr;
        }
        if (++sk == KS) {
          sk = 0;
          su++;
        }
      }
    };
    // rows of keys a .. b - 1 into the ring (eight waves per key, 64 columns each)
    auto stage_rows = [&](int a, int b) {
      constexpr int kRuns = TN / 64;
      const int q = w % kRuns;
      for (int u = a + w / kRuns; u < b; u += kGemmWaves / kRuns)
        __builtin_amdgcn_global_load_lds(g.tmat + int64_t(slot(u)) * TN + q * 64 + lane,
                                         Ts + (u & (ring - 1)) * TN + q * 64, 4, 0, 0);
    };
    // keys whose rows are wanted once the units before (su, sk) are staged
    auto row_end = [&]() { return min(U, su + (sk > 0) + kGemmLook); };
    // bit ct of key 64 b + lane: this wave's column tile ct holds a pair
    auto load_masks = [&](int b) {
      const int u = b * 64 + lane;
      const unsigned long long m =
          (u < U ? g.tmask[VAR && op.perm ? op.perm[first + u] : first + u] : 0ull) >> (8 * (w >> 2) + (w & 3));
      static_assert(kCT == 2 && kGemmWaves == 16, "bits w and 32 + w of a mask");
      return int((m & 1) | ((m >> 31) & 2));
    };
    // This lane's first element of its columns' source rows, in 16-byte
    // units (KP is a multiple of 8); empty slots read the zero row (index
    // ncells), so every load is unconditional and stays in flight until its
    // k-step: masking at load time would make the wave wait for the data.
    const unsigned row8 = unsigned(KP) / 8, zero8 = unsigned(g.ncells) * row8;
    auto col_src = [&](int u, unsigned (&sc)[kCT]) {
      const int *T = Ts + (u & (ring - 1)) * TN;
#pragma unroll
      for (int ct = 0; ct < kCT; ct++) {
        const int c = T[tile_col(w, ct, lane)];
        sc[ct] = (c >= 0 ? unsigned(c) * row8 : zero8) + kq;
      }
    };
    // k-groups at or past the key's K bound (the last k-step's) read the zero
    // row; the one vector that straddles a variable order's bound is masked
    // when it is used (mask_b)
    auto load_b = [&](const unsigned (&sc)[kCT], int kk, int kc, v8bf (&bh)[kCT], v8bf (&bl)[kCT]) {
      const v8bf *ph = reinterpret_cast<const v8bf *>(g.mhi) + kk * 4;
      const v8bf *pl = reinterpret_cast<const v8bf *>(g.mlo) + kk * 4;
      const bool in = kk * 32 + kq * 8 < kc;
#pragma unroll
      for (int ct = 0; ct < kCT; ct++) {
        const unsigned o = in ? sc[ct] : zero8;
        bh[ct] = ph[o];
        bl[ct] = pl[o];
      }
    };
    auto mask_b = [&](int kk, int kc, v8bf (&bh)[kCT], v8bf (&bl)[kCT]) {
      const int k0 = kk * 32 + kq * 8;
      if (k0 >= kc || k0 + 8 <= kc) return;
#pragma unroll
      for (int ct = 0; ct < kCT; ct++)
#pragma unroll
        for (int i = 0; i < 8; i++)
          if (k0 + i >= kc) {
            bh[ct][i] = __bf16(0.0f);
            bl[ct][i] = __bf16(0.0f);
          }
    };
    stage_ops(0);
    int rows = row_end();
    stage_rows(0, rows);
    int nib = load_masks(0), nib_next = load_masks(1);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    unsigned long long act = __ballot(nib != 0);
    unsigned src[kCT];
    v8bf bh[kCT], bl[kCT];
    int u = 0, kk = 0, kc = kcols(0);
    int pu = -1, pk = 0;  // the unit whose multipoles bh, bl hold (or will, once they land)
    for (int r = 0; r < R; r++) {
      const int landed = rows;
      if (r + 1 < R) {
        stage_ops(r + 1);
        const int e = row_end();
        stage_rows(rows, e);
        rows = max(rows, e);
      }
      __builtin_amdgcn_sched_barrier(0);
      // B loads issued after this round's staging: at most the last ones are
      // still in flight when the round ends
      bool b_after = false;
      const int n = min(G, N - r * G);
      for (int i = 0; i < n; i++) {
        const int m = __builtin_amdgcn_readlane(nib, u & 63);
        const int ks = ksteps(kc);
        if (m != 0 && kk < ks) {
          if (pu != u || pk != kk) {
            col_src(u, src);
            load_b(src, kk, kc, bh, bl);
          }
          // only an order below the operator's has a bound inside the padded K range
          if (VAR && kk * 32 + 32 > kc) mask_b(kk, kc, bh, bl);
          const v8bf *Ah = Ab + size_t((r & 1) * G + i) * UE + lane, *Al = Ah + nrt * 64;
          const int nr = rtiles(kc);
          // Up to seven row tiles a row tile's operator is read while the one
          // before it is multiplied, which the branches on the subtile bits keep
          // the compiler from doing (2^20 uniform bodies, order 10: 2.97 -> 2.92
          // ms); the registers of more row tiles leave no room for it.
          constexpr bool kAhead = !VAR && RH <= 7;
          v8bf a_hi = Ah[0], a_lo = Al[0];
#pragma unroll
          for (int r2 = 0; r2 < RH; r2++) {
            if (!VAR || r2 < nr) {  // uniform, as the subtile bits below
              v8bf n_hi = a_hi, n_lo = a_lo;
              if (kAhead && r2 + 1 < RH) {
                n_hi = Ah[(r2 + 1) * 64];
                n_lo = Al[(r2 + 1) * 64];
              } else if (!kAhead) {
                a_hi = Ah[r2 * 64];
                a_lo = Al[r2 * 64];
              }
#pragma unroll
              for (int ct = 0; ct < kCT; ct++) {
                if (m & (1 << ct)) {
                  acc[r2][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_hi, bh[ct], acc[r2][ct], 0, 0, 0);
                  acc[r2][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_hi, bl[ct], acc[r2][ct], 0, 0, 0);
                  acc[r2][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_lo, bh[ct], acc[r2][ct], 0, 0, 0);
                }
              }
              if (kAhead) {
                a_hi = n_hi;
                a_lo = n_lo;
              }
            }
          }
          // the next unit's multipoles into the same registers: the SIMD's other
          // waves cover the latency (a second buffer costs the fourth wave)
          if (kk + 1 < ks) {
            load_b(src, kk + 1, kc, bh, bl);
            pu = u;
            pk = kk + 1;
            b_after = true;
          } else {
            // this wave's next key, if it lies in this block of masks and its row is in LDS
            const unsigned long long rest = (u & 63) == 63 ? 0ull : act >> ((u & 63) + 1);
            const int v = u + __ffsll((long long)rest);
            if (rest && v < landed) {
              col_src(v, src);
              load_b(src, 0, kcols(v), bh, bl);
              pu = v;
              pk = 0;
              b_after = true;
            }
          }
        }
        if (++kk == KS) {
          kk = 0;
          u++;
          if (u < U) kc = kcols(u);
          if ((u & 63) == 0) {
            nib = nib_next;
            act = __ballot(nib != 0);
            nib_next = load_masks(u / 64 + 1);
          }
        }
      }
      // the staging issued at this round's start has landed (loads complete
      // in issue order; only the 2 kCT loads of the last B prefetch are
      // younger), then every wave is done with this round's buffers
      if (b_after)
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * kCT));
      else
        __builtin_amdgcn_s_waitcnt(kWaitVm0);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __builtin_amdgcn_s_barrier();
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (Lpart)
    write_partial<RH>(PP, rt0, nrt, part_local ? nullptr : g.sorted + g.tfirst[tile], ncol, w, acc, lane, Lpart);
  else
    write_locals<RH>(PP, rt0, nrt, g.sorted + g.tfirst[tile], ncol, w, acc, lane, L);
}

template <int RH, bool VAR>
__global__ void __launch_bounds__(kGemmThreads) k_m2l_bf16x3(GemmIn g, const int *__restrict__ tbase, int PP, int RT,
                                                             int RTB, int K32, int KP, OrderPass op,
                                                             const unsigned char *__restrict__ tkp, int G, int ring,
                                                             float *__restrict__ Lpart, double *__restrict__ L) {
  // keys of this workgroup: slice blockIdx.z of gridDim.z of the tile's keys
  const int Ut = g.tU[blockIdx.x];
  const int ub = int(int64_t(Ut) * blockIdx.z / gridDim.z), ue = int(int64_t(Ut) * (blockIdx.z + 1) / gridDim.z);
  m2l_bf16x3_body<RH, VAR>(g, blockIdx.x, blockIdx.y, tbase[blockIdx.x] + ub, ue - ub, false, PP, RT, RTB, K32, KP, op, tkp,
                      G, ring, Lpart ? Lpart + int64_t(blockIdx.z) * g.ncells * PP : nullptr, L);
}

// Stream-K schedule: the tiles' key slots, in tile order (slot tbase[t] + u
// is key u of tile t; S slots in all), are split evenly over the W = min(gridDim.x,
// S) active workgroups of one persistent launch (one per CU and row block;
// sk_schedule.h).  Workgroup w takes slots [w S / W, (w + 1) S / W), at least
// one, and the others return; each tile it touches gives one FP32
// partial of the tile's locals, stored by tile column in segment w + t of
// Lseg, and k_sk_combine adds a tile's segments in workgroup order.  Every
// workgroup gets the same number of slots, so none waits on a straggler.  A
// launch of one order of a learned-order evaluation schedules that order's
// slots: tbase is then the exclusive prefix of their per-tile counts tU,
// tstart[t] where tile t's run of them starts in the order-grouped slots, and
// Sdev their total.
//
// First slot of active workgroup w (slots are counted in ints), in a scalar
// register, as is everything the schedule derives from it: the GEMM body has
// no vector registers to spare.
__device__ inline int sk_first(int64_t w, int64_t S, int64_t W) {
  return __builtin_amdgcn_readfirstlane(int(sk_slot(w, S, W)));
}

template <class F>
__device__ __attribute__((always_inline)) inline void sk_segments(int ntiles, int s0, int s1, int off,
                                                                  const int *tbase, const int *tU, F &&segment) {
  // first tile holding slot s0 (slots of these tiles start at off): the last t with off + tbase[t] <= s0
  int lo = 0, hi = ntiles - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off + tbase[mid] <= s0)
      lo = mid;
    else
      hi = mid - 1;
  }
  for (int t = __builtin_amdgcn_readfirstlane(lo); t < ntiles; t++) {
    const int b = off + tbase[t];
    if (b >= s1) break;
    const int ub = __builtin_amdgcn_readfirstlane(max(s0, b) - b);
    const int n = __builtin_amdgcn_readfirstlane(min(s1, b + tU[t]) - b) - ub;
    if (n <= 0) continue;
    segment(t, ub, n);
    __syncthreads();  // the LDS of this segment is free before the next one stages
  }
}

template <int RH, bool VAR>
__global__ void __launch_bounds__(kGemmThreads) k_m2l_bf16x3_sk(GemmIn g, const int *__restrict__ tbase,
                                                                const int *__restrict__ tstart, int PP, int RT, int RTB,
                                                                int K32, int KP, OrderPass op, int ntiles, int64_t S,
                                                                const int *__restrict__ Sdev,
                                                                const unsigned char *__restrict__ tkp, int G, int ring,
                                                                float *__restrict__ Lseg) {
  if (Sdev) S = *Sdev;  // one order's slot count, summed on the device
  const int W = sk_active(gridDim.x, S), w = blockIdx.x;
  if (w >= W) return;
  const int s0 = sk_first(w, S, W), s1 = sk_first(w + 1, S, W);
  sk_segments(ntiles, s0, s1, 0, tbase, g.tU, [&](int t, int ub, int n) {
    m2l_bf16x3_body<RH, VAR>(g, t, blockIdx.y, tstart[t] + ub, n, true, PP, RT, RTB, K32, KP, op, tkp, G, ring,
                        Lseg + (w + t) * int64_t(kTileN) * PP, nullptr);
  });
}

// Sum of a tile's stream-K segments (workgroups wf .. wl in order) into the
// FP64 locals: element e = (tile column, VEC rows from VEC * (e % (rows / VEC)))
// of tile t, rows 0 .. rows - 1 (those the launch computed); slots b .. b + n -
// 1 of S belong to the tile, its segments start at seg0 + w.  Four rows per
// thread where rows and row length are multiples of four, and four segments'
// loads in flight: a small tree's few slots are spread over every workgroup, so
// that a tile has a hundred segments (10,000 uniform bodies: 392 -> 371 us).
template <int VEC>
__device__ inline void sk_combine(int64_t e, int PP, int rows, int ncol, int64_t b, int n, int64_t S, int W,
                                  int64_t seg0, const int *cells, const float *__restrict__ Lseg,
                                  double *__restrict__ L) {
  const int per = rows / VEC, col = int(e / per), row = int(e % per) * VEC;
  if (col >= ncol || n == 0) return;
  W = sk_active(W, S);
  const int wf = sk_owner(b, S, W), wl = sk_owner(b + n - 1, S, W);
  typedef float vec __attribute__((ext_vector_type(VEC)));
  const int64_t step = int64_t(kTileN) * PP;
  const float *p = Lseg + (wf + seg0) * step + int64_t(col) * PP + row;
  double acc[VEC] = {};
  int w = wf;
  for (; w + 3 <= wl; w += 4, p += 4 * step) {
    vec v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = *reinterpret_cast<const vec *>(p + k * step);
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int i = 0; i < VEC; i++) acc[i] += double(v[k][i]);
  }
  for (; w <= wl; w++, p += step) {
    const vec v = *reinterpret_cast<const vec *>(p);
#pragma unroll
    for (int i = 0; i < VEC; i++) acc[i] += double(v[i]);
  }
  double *Lc = L + int64_t(cells[col]) * PP + row;
#pragma unroll
  for (int i = 0; i < VEC; i++) Lc[i] += acc[i];
}
static int sk_combine_vec(int PP, int rows) { return PP % 4 == 0 && rows % 4 == 0 ? 4 : 1; }

template <int VEC>
__global__ void __launch_bounds__(256) k_sk_combine(int PP, int rows, int ntiles, int64_t S, const int *__restrict__ Sdev,
                                                    int W, const int *__restrict__ tfirst,
                                                    const int *__restrict__ tcount, const int *__restrict__ tbase,
                                                    const int *__restrict__ tU, const int *__restrict__ sorted,
                                                    const float *__restrict__ Lseg, double *__restrict__ L) {
  const int t = blockIdx.y;
  if (t >= ntiles) return;
  if (Sdev) S = *Sdev;
  sk_combine<VEC>(int64_t(blockIdx.x) * 256 + threadIdx.x, PP, rows, tcount[t], tbase[t], tU[t], S, W, t,
                  sorted + tfirst[t], Lseg, L);
}

// The segments of a learned-order evaluation's launches, one per order class,
// added in one pass over the locals (a pass per class read and wrote them
// again: over 300,007 bodies' cells at order 13 four passes took 97 us, this 63;
// over 2^22 bodies' 0.8 ms, 0.4 less).
constexpr int kMaxClasses = 6;
struct ClassSum {
  const int *pre, *cnt, *tot;  // per tile: first slot, slots; all slots (ClassPass)
  int W, rows;                 // workgroups, rows of the launch
  int64_t base;                // its segments in the buffer
};
struct ClassSums {
  int n;
  ClassSum c[kMaxClasses];
};
__global__ void __launch_bounds__(256) k_sk_combine_classes(int PP, int rows, int ntiles, ClassSums sums,
                                                            const int *__restrict__ tfirst,
                                                            const int *__restrict__ tcount,
                                                            const int *__restrict__ sorted,
                                                            const float *__restrict__ Lseg, double *__restrict__ L) {
  const int t = blockIdx.y;
  const int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int col = int(e / rows), row = int(e % rows);
  if (t >= ntiles || col >= tcount[t]) return;
  double *Lc = L + int64_t(sorted[tfirst[t] + col]) * PP + row;
  // every class's first two segments are loaded before the first is added
  const int64_t step = int64_t(kTileN) * PP;
  const float *p[kMaxClasses];
  int nseg[kMaxClasses];
  float v[kMaxClasses][2];
#pragma unroll
  for (int k = 0; k < kMaxClasses; k++) {
    const ClassSum &c = sums.c[k];
    nseg[k] = 0;
    v[k][0] = v[k][1] = 0.0f;
    if (k >= sums.n) continue;
    const int n = c.cnt[t];
    if (n == 0 || row >= c.rows) continue;
    const int64_t b = c.pre[t], S = *c.tot;
    const int W = sk_active(c.W, S), wf = sk_owner(b, S, W);
    nseg[k] = sk_owner(b + n - 1, S, W) - wf + 1;
    p[k] = Lseg + c.base + (wf + int64_t(t)) * step + int64_t(col) * PP + row;
    v[k][0] = p[k][0];
    if (nseg[k] > 1) v[k][1] = p[k][step];
  }
  double l = *Lc;
#pragma unroll
  for (int k = 0; k < kMaxClasses; k++) {
    if (nseg[k] == 0) continue;
    double acc = double(v[k][0]);
    if (nseg[k] > 1) acc += double(v[k][1]);
    for (int w = 2; w < nseg[k]; w++) acc += double(p[k][w * step]);
    l += acc;
  }
  *Lc = l;
}

// One problem of a grouped keyed-GEMM launch (all problems of one order in
// a batch): its tiles, operators, cast multipoles and locals.
struct GroupGemm {
  GemmIn in;
  const int *tbase;
  double *L;
  int ntiles, tile0;  // tile0: first of its tiles among the launch's
};

// All problems of one order in one stream-K launch: the slots of problem i
// are sstart[i] .. sstart[i + 1] - 1 of S = sstart[nprob], its tiles the
// launch's tiles tile0 ...  (A workgroup per tile and row block left the
// chip to the tiles with the most keys: 12 problems of up to 10^5 bodies
// have 8 tiles each.)
template <int RH>
__global__ void __launch_bounds__(kGemmThreads) k_m2l_bf16x3_grouped(const GroupGemm *__restrict__ gr,
                                                                     const int *__restrict__ sstart, int nprob, int PP,
                                                                     int RT, int RTB, int K32, int KP, int pl, int G,
                                                                     int ring, float *__restrict__ Lseg) {
  const int S = sstart[nprob], W = sk_active(gridDim.x, S), w = blockIdx.x;
  if (w >= W) return;
  const int s0 = sk_first(w, S, W), s1 = sk_first(w + 1, S, W);
  const OrderPass op{pl, RT, K32, nullptr};
  for (int i = __builtin_amdgcn_readfirstlane(group_of(sstart, nprob, s0)); i < nprob && sstart[i] < s1; i++) {
    const GroupGemm &q = gr[i];
    sk_segments(q.ntiles, max(s0, sstart[i]), min(s1, sstart[i + 1]), sstart[i], q.tbase, q.in.tU,
                [&](int t, int ub, int n) {
                  m2l_bf16x3_body<RH, false>(q.in, t, blockIdx.y, q.tbase[t] + ub, n, true, PP, RT, RTB, K32, KP, op, nullptr,
                                      G, ring, Lseg + (w + q.tile0 + t) * int64_t(kTileN) * PP, nullptr);
                });
  }
}

template <int VEC>
__global__ void __launch_bounds__(256) k_sk_combine_grouped(const GroupGemm *__restrict__ gr,
                                                            const int *__restrict__ sstart,
                                                            const int *__restrict__ tstart, int nprob, int PP, int W,
                                                            const float *__restrict__ Lseg) {
  const int gt = blockIdx.y, i = group_of(tstart, nprob, gt), t = gt - tstart[i];
  const GroupGemm &q = gr[i];
  sk_combine<VEC>(int64_t(blockIdx.x) * 256 + threadIdx.x, PP, PP, q.in.tcount[t], sstart[i] + q.tbase[t], q.in.tU[t],
             sstart[nprob], W, gt, q.in.sorted + q.in.tfirst[t], Lseg, q.L);
}

// Tile-matrix rows held in LDS for G units of KS per key: two rounds' keys
// and the look-ahead, a power of two.
static int gemm_ring(int KS, int G) {
  int n = 1;
  while (n < ceil_div(2 * G, KS) + 2 + kGemmLook) n *= 2;
  return n;
}

// Row tiles per workgroup for rounds of `kr` (FP32: keys; BF16: units, a key
// having K32 of them): two operator buffers and the column sources within the
// LDS budget, at most the accumulators of kGemmMaxRT row tiles per wave.
static int lds_limit(int device) {
  int n = 0;
  XF_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMaxSharedMemoryPerBlock, device));
  return n;
}
static int rows_per_block(const Geom &g, bool bf16, int device, int kr) {
  const int max_lds = lds_limit(device);
  const int per_rt = 2 * kr * (bf16 ? 64 * 16 * 2 : g.K4 * 64 * 4);  // both buffers
  const int avail = max_lds - (bf16 ? gemm_ring(g.K32, kr) : 3 * kr) * kTileN * 4;
  if (per_rt > avail) {
    if (kr == 1) fail(EXAFMM_ERR_UNSUPPORTED, "expansion order too large for the LDS operator stage");
    return 0;
  }
  const int rtb = std::min({g.R, bf16 ? kGemmMaxRT : kGemmMaxRTF32, avail / per_rt});
  // balance the row blocks
  const int nblk = ceil_div(g.R, rtb);
  return ceil_div(g.R, nblk);
}

static size_t gemm_lds(const Geom &g, bool bf16, int RTB, int kr) {
  return size_t(2) * kr * RTB * (bf16 ? 64 * 16 * 2 : g.K4 * 64 * 4) +
         size_t(bf16 ? gemm_ring(g.K32, kr) : 3 * kr) * kTileN * sizeof(int);
}

// One order's launch of a learned-order BF16x3 GEMM: order p over the
// slots of that order (tile t: grouped slots cb[t] .. cb[t] + cnt[t] - 1,
// slot permutation perm).
struct ClassPass {
  int p;          // highest order of the class
  bool variable;  // the class holds several orders: each slot runs at its own (tile_p)
  const int *perm;
  const int *start, *cnt;  // per tile: first order-grouped slot (tbase included) and count
  const int *pre, *tot;    // per tile: exclusive prefix of the counts; their total (stream-K)
};

static GemmIn gemm_in(const Ctx &c, const Ctx &sc, const Geom &g, const ClassPass *cp) {
  const int ts = c.m2l_tstride;
  GemmIn in{};
  in.tfirst = c.tiles.p;
  in.tcount = c.tiles.p + ts;
  in.tU = cp ? cp->cnt : c.tiles.p + 3 * ts;
  in.sorted = c.tiles.p + 4 * ts;
  in.tkeys = c.tile_keys.p;
  in.tmat = c.tile_mat.p;
  in.tmask = c.tile_mask.p;
  const size_t per = size_t(g.K32) * g.R * 64 * 8;
  in.ophi = reinterpret_cast<const v8bf *>(c.ops32.p);
  in.oplo = reinterpret_cast<const v8bf *>(reinterpret_cast<const __bf16 *>(c.ops32.p) + per * c.lists.nkeys);
  in.mhi = reinterpret_cast<const __bf16 *>(sc.mt32.p);
  in.mlo = in.mhi + bf16_cast_elems(g, sc.t.ncells);
  in.ncells = sc.t.ncells;
  return in;
}

struct GemmShape {
  int rtb, kr, ksplit;
  int sk = 0;  // stream-K: one persistent workgroup per CU over the tiles' key slots (BF16x3)
};

static int cu_count(int device) {
  int n = 0;
  XF_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device));
  return std::max(n, 1);
}

// Persistent workgroups per row block of a stream-K launch.
static int sk_groups(int device, int nblk) { return std::max(1, cu_count(device) / nblk); }

// The attribute belongs to the kernel, not to the launch: always the limit, so
// that contexts on several threads agree on it.
template <class K>
static void gemm_attr(K *kernel) {
  int device = 0;
  XF_HIP(hipGetDevice(&device));
  XF_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                             lds_limit(device)));
}

template <int RH>
static void launch_bf16(Ctx &c, const Ctx &sc, const Geom &g, int ntiles, int KPb, GemmShape sh, float *Lpart,
                        double *Lout, const ClassPass *cp, ClassSums *sums) {
  const int ts = c.m2l_tstride;
  const int *tbase = c.tiles.p + 2 * ts;
  const Geom go = cp ? geom(cp->p) : g;  // rows and k-steps this launch covers
  const GemmIn in = gemm_in(c, sc, g, cp);
  const OrderPass op{go.P, go.R, go.K32, cp ? cp->perm : nullptr};
  const unsigned char *tkp = (c.learned && (!cp || cp->variable)) ? c.tile_p.p : nullptr;
  const int nblk = ceil_div(go.R, sh.rtb), ring = gemm_ring(go.K32, sh.kr);
  const size_t lds = gemm_lds(go, true, sh.rtb, sh.kr);
  if (!sh.sk) {
    auto *k = cp ? &k_m2l_bf16x3<RH, true> : &k_m2l_bf16x3<RH, false>;
    gemm_attr(k);
    hipLaunchKernelGGL(k, dim3(ntiles, nblk, sh.ksplit), dim3(kGemmThreads), lds, c.s0, in,
                       cp ? cp->start : tbase, g.PP, g.R, sh.rtb, g.K32, KPb, op, tkp, sh.kr, ring,
                       sh.ksplit > 1 ? Lpart : nullptr, Lout);
    XF_LAUNCH();
    return;
  }
  const int W = sk_groups(c.cfg.device, nblk);
  const int64_t S = c.m2l_totalU;
  if (!sums) c.m2l_part.ensure(size_t(W + ntiles) * kTileN * g.PP);  // (else sized for every class)
  float *seg = c.m2l_part.p + (sums ? sums->c[sums->n].base : 0);
  const int *pre = cp ? cp->pre : tbase, *start = cp ? cp->start : tbase;
  const int *Sdev = cp ? cp->tot : nullptr;
  auto *k = cp ? &k_m2l_bf16x3_sk<RH, true> : &k_m2l_bf16x3_sk<RH, false>;
  gemm_attr(k);
  hipLaunchKernelGGL(k, dim3(W, nblk), dim3(kGemmThreads), lds, c.s0, in, pre, start, g.PP, g.R,
                     sh.rtb, g.K32, KPb, op, ntiles, S, Sdev, tkp, sh.kr, ring, seg);
  XF_LAUNCH();
  const int rows = std::min(g.PP, 16 * go.R);
  if (sums) {  // added with the other classes' by m2l_fast
    ClassSum &k = sums->c[sums->n++];
    k = ClassSum{pre, in.tU, Sdev, W, rows, k.base};
    return;
  }
  const int vec = sk_combine_vec(g.PP, rows);
  hipLaunchKernelGGL(vec == 4 ? k_sk_combine<4> : k_sk_combine<1>,
                     dim3(ceil_div(int64_t(kTileN) * rows / vec, 256), ntiles), dim3(256), 0, c.s0, g.PP, rows,
                     ntiles, S, Sdev, W, in.tfirst, in.tcount, pre, in.tU, in.sorted, seg, Lout);
  XF_LAUNCH();
}

template <int RH>
static void launch_f32(Ctx &c, const Ctx &sc, const Geom &g, int ntiles, int KP, GemmShape sh, float *Lpart,
                       double *Lout) {
  const int ts = c.m2l_tstride;
  const int *t = c.tiles.p;
  const size_t lds = gemm_lds(g, false, sh.rtb, sh.kr);
  gemm_attr(&k_m2l_f32<RH>);
  hipLaunchKernelGGL((k_m2l_f32<RH>), dim3(ntiles, ceil_div(g.R, sh.rtb), sh.ksplit), dim3(kGemmThreads), lds, c.s0,
                     g.PP, g.R, sh.rtb, g.K4, KP, t, t + ts, t + 2 * ts, t + 3 * ts, t + 4 * ts, c.tile_keys.p,
                     c.tile_mat.p, c.tile_mask.p, c.ops32.p, sc.mt32.p, c.learned ? c.tile_p.p : nullptr, sh.kr,
                     int64_t(c.t.ncells), sh.ksplit > 1 ? Lpart : nullptr, Lout);
  XF_LAUNCH();
}

static void run_gemm(Ctx &c, const Ctx &sc, const Geom &g, int ntiles, bool bf16, int KP, int KPb, GemmShape sh,
                     double *Lout, const ClassPass *cp = nullptr, ClassSums *sums = nullptr) {
  float *part = nullptr;
  if (sh.ksplit > 1) {
    c.m2l_part.ensure(size_t(sh.ksplit) * c.t.ncells * g.PP);
    part = c.m2l_part.p;
  }
  switch (sh.rtb) {
#define XF_GEMM_CASE(n)                                                             \
  case n:                                                                           \
    if (bf16)                                                                       \
      launch_bf16<n>(c, sc, g, ntiles, KPb, sh, part, Lout, cp, sums);              \
    else                                                                            \
      launch_f32<n <= kGemmMaxRTF32 ? n : 1>(c, sc, g, ntiles, KP, sh, part, Lout); \
    break;
    XF_GEMM_CASE(1)
    XF_GEMM_CASE(2)
    XF_GEMM_CASE(3)
    XF_GEMM_CASE(4)
    XF_GEMM_CASE(5)
    XF_GEMM_CASE(6)
    XF_GEMM_CASE(7)
    XF_GEMM_CASE(8)
    XF_GEMM_CASE(9)
#undef XF_GEMM_CASE
    default: fail(EXAFMM_ERR_UNSUPPORTED, "expansion order");
  }
  if (sh.ksplit > 1) {
    const int64_t n = int64_t(c.m2l_ncell_tiled) * g.PP;
    hipLaunchKernelGGL(k_combine_slices, dim3(ceil_div(n, 256)), dim3(256), 0, c.s0, g.PP, int64_t(c.t.ncells),
                       sh.ksplit, c.tiles.p + 4 * c.m2l_tstride, c.m2l_ncell_tiled, part, Lout);
    XF_LAUNCH();
  }
}

// Rounds the autotuners try, in units of a launch of KS units per key: whole
// keys as far as two buffers fit, else the most units that do, and half a key.
static std::vector<int> gemm_rounds(const Geom &go, int device) {
  std::vector<int> r;
  for (int n = 1; n <= 4; n++)
    if (rows_per_block(go, true, device, n * go.K32) >= std::min(go.R, ceil_div(go.R, ceil_div(go.R, kGemmMaxRT))))
      r.push_back(n * go.K32);
  for (int G = go.K32 - 1; G > 1 && r.empty(); G--)
    if (rows_per_block(go, true, device, G) >= ceil_div(go.R, ceil_div(go.R, kGemmMaxRT))) r.push_back(G);
  if (go.K32 >= 4) r.push_back(go.K32 / 2);
  if (r.empty()) r.push_back(1);
  return r;
}

// Autotuner of the GEMM shape: operator staged per LDS round (more per
// barrier hides the copy latency of short, low-order keys), stream-K, or a
// workgroup per tile with key slices (a tile's keys split over several
// workgroups whose FP32 partial locals a second kernel adds in a fixed order:
// more parallelism when tiles are few and keys many).  The first time a (order, precision, order policy, tile
// count class) is seen, every candidate (GEMM and, with key slices, the
// combining kernel) runs twice into a scratch copy of the locals, alone on
// the device, timed with HIP events; the fastest run's shape is kept for
// the context's lifetime.
static GemmShape gemm_shape(Ctx &c, const Ctx &sc, const Geom &g, int ntiles, bool bf16, int KP, int KPb,
                            const ClassPass *cp = nullptr) {
  int tclass = 0;
  while ((1 << tclass) < ntiles) tclass++;
  // a learned-order launch of one order is tuned per order (its rows, k-steps and LDS)
  const Geom go = cp ? geom(cp->p) : g;
  const long long key = ((long long)g.P << 24) | ((long long)bf16 << 20) | ((long long)c.learned << 16) |
                        ((long long)(cp ? cp->p : 0) << 32) | tclass;
  auto it = c.gemm_tuned.find(key);
  auto shape = [](int v) { return GemmShape{v & 255, (v >> 8) & 255, (v >> 16) & 255, v >> 24}; };
  if (it != c.gemm_tuned.end()) return shape(it->second);
  if (c.defer_tuning && c.cfg.autotune) {
    // the tuned class nearest in tile count (the low bits of the key), if there is one
    c.tuning_wanted = true;
    const std::pair<const long long, int> *near = nullptr;
    for (const auto &kv : c.gemm_tuned)
      if ((kv.first >> 16) == (key >> 16) &&
          (!near || std::llabs(kv.first - key) < std::llabs(near->first - key)))
        near = &kv;
    if (near) return shape(near->second);
  }
  std::vector<GemmShape> cand;
  auto slices = [&](int rtb, int kr, int nb) {
    cand.push_back(GemmShape{rtb, kr, 1});
    // key slices only where the workgroups would not fill the device (the FP32
    // form, which has no stream-K, also in thirds and sixths: 80 tiles in three
    // slices are one round of workgroups)
    const int wg = ntiles * nb;
    for (const int ks : {2, 3, 4, 6, 8})
      if ((bf16 ? ks != 3 && ks != 6 && wg * ks <= 2048 : wg * ks <= 4096) && c.m2l_totalU >= 8 * ks * ntiles) cand.push_back(GemmShape{rtb, kr, ks});
  };
  if (bf16) {
    for (const int G : gemm_rounds(go, c.cfg.device)) {
      const int r = rows_per_block(go, true, c.cfg.device, G), nb = ceil_div(go.R, r);
      slices(r, G, nb);
      if (std::getenv("EXAFMM_GEMM_NO_SK") == nullptr) cand.push_back(GemmShape{r, G, 1, 1});
    }
  } else {
    // low orders: short keys, so more of them per LDS round (481,932 clustered bodies,
    // theta 0.3, order 4: rounds of 8 or 12 instead of up to 5, whole step 1.07 -> 0.99 of what tiles of one level took)
    const int krmax = go.P <= 5 ? 12 : go.P <= 10 ? 5 : 3;
    for (int kr = 1; kr <= krmax; kr += kr < 5 ? 1 : 3 + (kr > 5)) {
      const int rmax = rows_per_block(go, false, c.cfg.device, kr);
      if (rmax < 1) continue;
      int last = -1;
      for (int nb = ceil_div(go.R, rmax); nb <= ceil_div(go.R, rmax) + 2; nb++) {
        const int r = ceil_div(go.R, nb);
        if (r != last && r <= rmax) slices(r, kr, nb);
        last = r;
      }
    }
  }
  GemmShape best = cand[0];
  if (std::getenv("EXAFMM_GEMM_SK_ONLY"))  // the stream-K candidates alone (tests, A/B timing)
    for (const GemmShape &sh : cand)
      if (sh.sk) {
        best = sh;
        break;
      }
  if (c.capturing) fail(EXAFMM_ERR_STATE, "GEMM shape not tuned before recording a graph");
  if (std::getenv("EXAFMM_GEMM_SK_ONLY")) cand.erase(std::remove_if(cand.begin(), cand.end(), [](const GemmShape &x) { return !x.sk; }), cand.end());
  if (cand.empty()) fail(EXAFMM_ERR_UNSUPPORTED, "no GEMM shape");
  if (cand.size() > 1 && c.cfg.autotune && c.defer_tuning) return best;  // (not kept: tuned by the next run)
  if (cand.size() > 1 && c.cfg.autotune) {
    hipStream_t s = c.s0;
    XF_HIP(hipStreamSynchronize(c.s1));  // tune alone on the device
    c.L_tune.ensure(size_t(c.t.ncells) * c.P * c.P);
    size_t need = 1;
    for (const GemmShape &sh : cand)
      need = std::max(need, sh.sk ? size_t(sk_groups(c.cfg.device, ceil_div(go.R, sh.rtb)) + ntiles) * kTileN * g.PP
                                  : size_t(sh.ksplit > 1 ? sh.ksplit : 0) * c.t.ncells * g.PP);
    c.m2l_part.ensure(need);  // no allocation inside the timings
    hipEvent_t e0, e1;
    XF_HIP(hipEventCreate(&e0));
    XF_HIP(hipEventCreate(&e1));
    float bt = 1e30f;
    for (const GemmShape &sh : cand) {
      for (int rep = 0; rep < 2; rep++) {  // best of two runs per candidate
        XF_HIP(hipEventRecord(e0, s));
        run_gemm(c, sc, g, ntiles, bf16, KP, KPb, sh, c.L_tune.p, cp);
        XF_HIP(hipEventRecord(e1, s));
        XF_HIP(hipEventSynchronize(e1));
        float ms = 0;
        XF_HIP(hipEventElapsedTime(&ms, e0, e1));
        if (ms < bt) {
          bt = ms;
          best = sh;
        }
      }
    }
    XF_HIP(hipEventDestroy(e0));
    XF_HIP(hipEventDestroy(e1));
  }
  c.gemm_tuned[key] = best.rtb | (best.kr << 8) | (best.ksplit << 16) | (best.sk << 24);
  return best;
}

// Whether the operators in ops32 were generated for this configuration and a
// key set of this size (the keys themselves are compared on the device).
static bool ops_comparable(const Ctx &c, int nkeys, int fillP, int bf16) {
  const bool periodic = c.cfg.images > 0;
  return c.ops_P == c.P && c.ops_fill == fillP && c.ops_bf16 == bf16 && c.ops_nkeys == nkeys &&
         (!periodic || (c.ops_R0 == c.t.R0 && c.ops_cycle == c.cfg.cycle));
}

static void ops_remember(Ctx &c, int nkeys, int fillP, int bf16, hipStream_t s) {
  c.ops_keys.ensure(std::max(nkeys, 1));
  XF_HIP(hipMemcpyAsync(c.ops_keys.p, c.lists.keys.p, sizeof(unsigned long long) * nkeys, hipMemcpyDeviceToDevice, s));
  c.ops_nkeys = nkeys;
  c.ops_P = c.P;
  c.ops_fill = fillP;
  c.ops_bf16 = bf16;
  c.ops_R0 = c.t.R0;
  c.ops_cycle = c.cfg.cycle;
}

// Whether the next keyed GEMM runs learned per-slot orders (a forest has no
// common root to scale the tolerance by: fixed order).
static bool learned_orders(const Ctx &c) {
  return c.cfg.order_policy == EXAFMM_ORDER_LEARNED && c.have_model && c.forest_n == 0;
}

// Tiles, key lists and operators: depend only on the tree and the lists,
// so they can be built on a side stream while the upward pass runs.
void m2l_prepare(Ctx &c, hipStream_t s) {
  c.m2l_ready = false;
  c.m2l_ntiles = 0;
  const Geom g = geom(c.P);
  const bool bf16 = c.cfg.m2l_precision == EXAFMM_PREC_BF16X3;
  const int fillP = c.cfg.m2l_truncation == EXAFMM_M2L_FULL ? 2 * c.P - 1 : c.P;
  const int nc = int(c.t.ncells);
  const int nkeys = c.lists.nkeys;
  if (nkeys > (1 << 16)) fail(EXAFMM_ERR_CAPACITY, "more than 65536 distinct M2L translations");

  // 1. tiles: cells with pairs grouped by octant, then key set
  c.t.key.ensure(nc);
  c.t.key2.ensure(nc);
  c.t.val.ensure(nc);
  c.t.val2.ensure(nc);
  // cells sorted by (group, min-hashes of the key set), BFS order within ties:
  // on adaptive trees this raises the fraction of non-empty GEMM slots; on
  // uniform trees, where BFS neighbours already share key sets, it changes little.
  // Tiles mix the levels (keys are scale-free: on a clustered set of 200,000
  // bodies half as many (tile, key) slots as with tiles of one level), unless
  // the keys carry the level (periodic) or the slots take one learned order
  // each, chosen for cells of one size.
  const bool by_level = c.cfg.images > 0 || learned_orders(c);
  c.m2l_by_level = by_level;
  // Tiles of at most kTileN cells per group, laid out on the device (no host
  // round trip before the per-tile counts); arrays strided by the bound
  // ntmax: [first | count | base | U] x ntmax, then the sorted cells
  const int tn = kTileN;
  const int ntmax = ceil_div(nc, tn) + 255;
  c.tiles.ensure(size_t(4) * ntmax + nc);
  int *d_first = c.tiles.p, *d_count = c.tiles.p + ntmax, *d_base = c.tiles.p + 2 * ntmax,
      *d_U = c.tiles.p + 3 * ntmax, *d_sorted = c.tiles.p + 4 * ntmax;
  c.m2l_misc.ensure(kMiscInts);
  const bool ranked = nc <= kCellRankMax;
  hipLaunchKernelGGL(k_group_keys, dim3(ceil_div(nc, 256 / kWave)), dim3(256), 0, s, nc, c.t.cx.p, c.t.cparent.p,
                     c.t.clevel.p, c.lists.m2l_beg.p, c.lists.m2l_cnt.p, c.lists.m2l.p, m2l_fp64_levels(c),
                     int(by_level), c.t.key.p, c.t.val.p, c.m2l_misc.p);
  XF_LAUNCH();
  if (ranked) {
    hipLaunchKernelGGL(k_cell_rank, dim3(ceil_div(nc, kWave)), dim3(1024), 0, s, nc, c.t.key.p, d_sorted, c.m2l_misc.p);
  } else {
    unsigned long long *k1 = c.t.key.p, *k2 = c.t.key2.p;
    int *v1 = c.t.val.p, *v2 = c.t.val2.p;
    radix_sort_pairs(k1, v1, k2, v2, nc, kGroupShift - 16 * kMinHashes, kSortBits, c.m2l_rs_hist, s);
    hipLaunchKernelGGL(k_group_hist, dim3(std::min(ceil_div(nc, 256), 64)), dim3(256), 0, s, nc, k1, v1, d_sorted,
                       c.m2l_misc.p);
  }
  XF_LAUNCH();
  hipLaunchKernelGGL(k_tile_plan, dim3(1), dim3(256), 0, s, c.m2l_misc.p, d_first, d_count);
  XF_LAUNCH();
  const int nwords = (nkeys + 31) / 32;
  c.tile_bits.ensure(size_t(ntmax) * std::max(nwords, 1));
  c.pin_i.ensure(kPinInts);
  const bool compare = ops_comparable(c, nkeys, fillP, bf16);
  hipLaunchKernelGGL(k_tile_count, dim3(ntmax), dim3(kTileCountThreads), sizeof(unsigned) * nwords, s, d_first, d_count,
                     d_sorted, c.lists.m2l_beg.p, c.lists.m2l_cnt.p, c.lists.m2l.p, nkeys, c.m2l_misc.p, d_U,
                     c.tile_bits.p, c.lists.keys.p, compare ? c.ops_keys.p : nullptr);
  XF_LAUNCH();
  hipLaunchKernelGGL(k_tile_scan, dim3(1), dim3(kTileCountThreads), 0, s, c.m2l_misc.p, d_U, d_base,
                     c.pin_i.p + kPinPlan);
  XF_LAUNCH();
  // one host round trip: slots, tiles, cells in tiles, and whether the operators still fit
  stream_wait(s);
  const int *plan = c.pin_i.p + kPinPlan;
  const int totalU = plan[0], ntiles = plan[1], off = plan[2];
  const bool cached = compare && plan[3] == 0;
  c.m2l_tstride = ntmax;
  if (ntiles == 0) {
    c.m2l_ready = true;
    return;
  }
  c.tile_keys.ensure(std::max(totalU, 1));
  c.tile_mat.ensure(size_t(std::max(totalU, 1)) * tn);
  c.tile_mask.ensure(std::max(totalU, 1));
  hipLaunchKernelGGL(k_tile_fill, dim3(ntiles, tn / 64), dim3(256), sizeof(unsigned) * 6 * nwords, s, d_first,
                     d_count, d_sorted, c.lists.m2l_beg.p, c.lists.m2l_cnt.p, c.lists.m2l.p, nkeys, d_base,
                     c.tile_bits.p, c.tile_keys.p, c.tile_mat.p, reinterpret_cast<unsigned char *>(c.tile_mask.p));
  XF_LAUNCH();

  // 2. operators (cached by key set)
  const double cyc = c.cfg.images > 0 ? c.cfg.cycle : 0.0;
  if (bf16) {
    const size_t per = size_t(g.K32) * g.R * 64 * 8;
    if (!cached) {
      c.ops32.ensure((per * nkeys * 2 + 1) / 2 + 1);
      __bf16 *ophi = reinterpret_cast<__bf16 *>(c.ops32.p);
      hipLaunchKernelGGL(k_ops_gen, dim3(nkeys), dim3(256), 0, s, c.P, fillP, g.R, g.K4, g.K32, c.t.R0, cyc,
                         c.lists.keys.p, (float *)nullptr, ophi, ophi + per * nkeys);
      XF_LAUNCH();
      ops_remember(c, nkeys, fillP, 1, s);
    }
  } else {
    const size_t per = size_t(g.K4) * g.R * 64;
    if (!cached) {
      c.ops32.ensure(per * nkeys);
      hipLaunchKernelGGL(k_ops_gen, dim3(nkeys), dim3(256), 0, s, c.P, fillP, g.R, g.K4, g.K32, c.t.R0, cyc,
                         c.lists.keys.p, c.ops32.p, (__bf16 *)nullptr, (__bf16 *)nullptr);
      XF_LAUNCH();
      ops_remember(c, nkeys, fillP, 0, s);
    }
  }
  c.m2l_ntiles = ntiles;
  c.m2l_ncell_tiled = off;
  c.m2l_totalU = totalU;
  c.m2l_ready = true;
}

// Cast the multipoles and run the keyed GEMM (after m2l_prepare, on s0).
void m2l_fast(Ctx &tc, const Ctx &sc) {
  if (&tc != &sc) fail(EXAFMM_ERR_UNSUPPORTED, "keyed M2L needs source == target tree");
  Ctx &c = tc;
  if (!c.m2l_ready) {
    if (c.capturing) fail(EXAFMM_ERR_STATE, "keyed M2L tiles missing while recording a graph");
    m2l_prepare(c, c.s0);
  }
  hipStream_t s = c.s0;
  join_upward(c);
  const Geom g = geom(c.P);
  const bool bf16 = c.cfg.m2l_precision == EXAFMM_PREC_BF16X3;
  const int nc = int(c.t.ncells);
  const int ntiles = c.m2l_ntiles;
  c.m2l_ntiles_last = ntiles;
  if (!c.graph_locks) c.m2l_ready = false;  // tiles belong to this horizontal pass (or to the graph)
  if (ntiles == 0) return;
  // BF16 rows hold P^2 coefficients padded to a multiple of 8 (one k-group
  // load), not to the MFMA's K of 32 per step: the k-groups past the row
  // read the zero row, which stays in cache
  const int KP = g.K4 * 4, KPb = bf16_row(g);
  if (bf16) {
    const size_t rows = bf16_cast_elems(g, nc);  // per part
    c.mt32.ensure(rows + 1);                     // two bf16 arrays in a float buffer
    __bf16 *mhi = reinterpret_cast<__bf16 *>(c.mt32.p);
    __bf16 *mlo = mhi + rows;
    hipLaunchKernelGGL(k_mt, dim3(ceil_div(int64_t(rows), 256)), dim3(256), 0, s, c.P * c.P, KPb, nc, kBf16Tail,
                       c.M.p, (float *)nullptr, mhi, mlo);
    XF_LAUNCH();
  } else {
    c.mt32.ensure(size_t(nc + 1) * KP);
    hipLaunchKernelGGL(k_mt, dim3(ceil_div(int64_t(nc + 1) * KP, 256)), dim3(256), 0, s, c.P * c.P, KP, nc, 0,
                       c.M.p, c.mt32.p, (__bf16 *)nullptr, (__bf16 *)nullptr);
    XF_LAUNCH();
  }

  // per-key orders of a learned-order evaluation (need the multipoles, and tiles of one level)
  c.learned = learned_orders(c) && c.m2l_by_level;
  if (c.learned)
    order_select(c, c.tiles.p, c.tiles.p + c.m2l_tstride, c.tiles.p + 2 * c.m2l_tstride,
                 c.tiles.p + 3 * c.m2l_tstride, c.tiles.p + 4 * c.m2l_tstride, ntiles, c.m2l_totalU, kTileN, s);

  // 3. GEMM over tiles, shape from the autotuner
  if (c.learned && bf16) {
    // one launch per order class over that class's slots of every tile
    // (grouped by k_order_partition), each with its own tuned shape: a
    // slot's cost then follows its order, and the launches add into the
    // locals in class sequence.  Classes: orders up to 8, then pairs (9-10,
    // 11-12, ...): few launches (each adds a partial-locals pass), each
    // class's LDS stage and row tiles sized to its highest order
    OrderClasses oc{};
    for (int p = 0; p <= kMaxP; p++) {
      const int q = std::min(std::max(p, kMlpPmin), c.P);
      const int k = q <= 8 ? 0 : (q - 7) / 2;
      oc.of[p] = (unsigned char)k;
      oc.hi[k] = (unsigned char)std::max<int>(oc.hi[k], q);
      oc.n = std::max(oc.n, k + 1);
    }
    const int ncls = oc.n;
    const int ts = c.m2l_tstride;
    c.tile_perm.ensure(std::max(c.m2l_totalU, 1));
    // tile_cls: [start | count | prefix] x order x tile stride, then the totals
    c.tile_cls.ensure(size_t(3) * ncls * ts + ncls);
    hipLaunchKernelGGL(k_order_partition, dim3(ceil_div(ntiles, 4)), dim3(256), 0, s, ntiles, ts, c.tiles.p + 2 * ts,
                       c.tiles.p + 3 * ts, c.tile_p.p, oc, c.tile_perm.p, c.tile_cls.p);
    XF_LAUNCH();
    hipLaunchKernelGGL(k_order_prefix, dim3(1), dim3(64 * ncls), 0, s, ntiles, ts, ncls, c.tile_cls.p);
    XF_LAUNCH();
    if (!c.capturing) XF_HIP(hipEventRecord(c.ev[13], s));
    std::vector<ClassPass> pass;
    std::vector<GemmShape> shape;
    // EXAFMM_GEMM_SK_ONLY=class: a sum per class (tests)
    const char *only = std::getenv("EXAFMM_GEMM_SK_ONLY");
    bool all_sk = ncls <= kMaxClasses && !(only && std::strcmp(only, "class") == 0);
    for (int o = ncls - 1; o >= 0; o--) {
      const int *cls = c.tile_cls.p;
      int lo = kMaxP;
      for (int p = kMlpPmin; p <= c.P; p++)
        if (oc.of[p] == o) lo = std::min(lo, p);
      pass.push_back(ClassPass{oc.hi[o], lo < oc.hi[o], c.tile_perm.p, cls + size_t(o) * ts, cls + size_t(ncls + o) * ts,
                               cls + size_t(2 * ncls + o) * ts, cls + size_t(3 * ncls) * ts + o});
      shape.push_back(gemm_shape(c, sc, g, ntiles, bf16, KP, KPb, &pass.back()));
      all_sk = all_sk && shape.back().sk;
    }
    // Stream-K launches leave their segments for one sum over the classes: (CUs +
    // tiles) x 512 x P^2 floats for every class at once (300,007 clustered bodies,
    // order 13: 4 x 114 MB; 2^22, order 14: 4 x 315 MB).  Where that much is not to
    // be had, a sum per class in one class's segments.
    ClassSums sums{};
    int rows = 0;
    int64_t seg = 0;
    for (size_t k = 0; all_sk && k < pass.size(); k++) {
      const Geom go = geom(pass[k].p);
      sums.c[k].base = seg;
      seg += int64_t(sk_groups(c.cfg.device, ceil_div(go.R, shape[k].rtb)) + ntiles) * kTileN * g.PP;
      rows = std::max(rows, std::min(g.PP, 16 * go.R));
    }
    if (all_sk) try {
        c.m2l_part.ensure(size_t(seg));
      } catch (const Failure &e) {
        if (e.code != EXAFMM_ERR_ALLOC) throw;
        all_sk = false;
      }
    for (size_t k = 0; k < pass.size(); k++)
      run_gemm(c, sc, g, ntiles, bf16, KP, KPb, shape[k], c.L.p, &pass[k], all_sk ? &sums : nullptr);
    if (all_sk) {
      hipLaunchKernelGGL(k_sk_combine_classes, dim3(ceil_div(int64_t(kTileN) * rows, 256), ntiles), dim3(256), 0, s,
                         g.PP, rows, ntiles, sums, c.tiles.p, c.tiles.p + ts, c.tiles.p + 4 * ts, c.m2l_part.p, c.L.p);
      XF_LAUNCH();
    }
    return;
  }
  const GemmShape sh = gemm_shape(c, sc, g, ntiles, bf16, KP, KPb);
  if (!c.capturing) XF_HIP(hipEventRecord(c.ev[13], s));
  run_gemm(c, sc, g, ntiles, bf16, KP, KPb, sh, c.L.p);
}


// ---------------------------------------------------------------- grouped (batch)
struct GroupCast {
  const double *M;
  __bf16 *mhi, *mlo;
  int64_t ncells;
  int PP, KP;
  int64_t elems;  // elements of each cast array: rows of KP, the zero row, the zero tail
};

// BF16 hi/lo cast of the multipoles of every problem of one order (row
// ncells of each problem is the zero row).
__global__ void __launch_bounds__(256) k_mt_grouped(const GroupCast *__restrict__ g, const int *__restrict__ start,
                                                    int nprob) {
  const int b = blockIdx.x, i = group_of(start, nprob, b);
  const GroupCast q = g[i];
  const int64_t e = int64_t(b - start[i]) * 256 + threadIdx.x;
  if (e >= q.elems) return;
  const int64_t c = e / q.KP;
  const int r = int(e % q.KP);
  const float v = (c < q.ncells && r < q.PP) ? float(q.M[c * q.PP + r]) : 0.0f;
  const __bf16 h = __bf16(v);
  q.mhi[e] = h;
  q.mlo[e] = __bf16(v - float(h));
}

// Descriptor tables of one order's problems (their tiles and operators from
// m2l_prepare, their cast buffers sized by an earlier evaluation) for one
// GEMM shape (rows per workgroup, units per LDS round), the same for every
// problem of the launch.
static void group_tables(const std::vector<Ctx *> &probs, GemmGroupPlan &plan, int rtb, int kr) {
  plan.nprob = 0;
  plan.ntiles = plan.cast_blocks = 0;
  if (probs.empty()) return;
  const int P = probs[0]->P;
  const Geom g = geom(P);
  const int KPb = bf16_row(g);  // the cast layout of m2l_fast: rows of KPb, zero row, zero tail
  plan.P = P;
  plan.rtb = rtb;
  plan.kr = kr;
  plan.groups = sk_groups(probs[0]->cfg.device, ceil_div(g.R, rtb));
  plan.lds = gemm_lds(g, true, rtb, kr);
  std::vector<GroupGemm> d;
  std::vector<GroupCast> cd;
  std::vector<int> st, cst;  // st: slot prefix, then tile prefix
  std::vector<int> tst;
  int64_t slots = 0, tiles = 0, cacc = 0;
  for (Ctx *cp : probs) {
    Ctx &c = *cp;
    if (c.P != P || c.cfg.m2l_precision != EXAFMM_PREC_BF16X3) fail(EXAFMM_ERR_ARG, "mixed orders in a GEMM group");
    if (!c.m2l_ready) fail(EXAFMM_ERR_STATE, "keyed M2L tiles missing");
    if (c.m2l_ntiles == 0) continue;
    const int64_t nc = c.t.ncells;
    const size_t elems = bf16_cast_elems(g, nc);
    c.mt32.ensure(elems + 1);  // two bf16 arrays in a float buffer (set-up time, not under capture)
    __bf16 *mhi = reinterpret_cast<__bf16 *>(c.mt32.p);
    d.push_back(GroupGemm{gemm_in(c, c, g, nullptr), c.tiles.p + 2 * c.m2l_tstride, c.L.p, c.m2l_ntiles, int(tiles)});
    st.push_back(int(slots));
    tst.push_back(int(tiles));
    slots += c.m2l_totalU;
    tiles += c.m2l_ntiles;
    cd.push_back(GroupCast{c.M.p, mhi, mhi + elems, nc, g.PP, KPb, int64_t(elems)});
    cst.push_back(int(cacc));
    cacc += ceil_div(int64_t(elems), 256);
  }
  if (slots > (int64_t(1) << 31) - 1 || tiles > 65535 || cacc > (int64_t(1) << 31) - 1)
    fail(EXAFMM_ERR_CAPACITY, "batch too large");
  plan.nprob = int(d.size());
  plan.ntiles = int(tiles);
  plan.cast_blocks = int(cacc);
  if (!plan.nprob) return;
  st.push_back(int(slots));
  tst.push_back(int(tiles));
  st.insert(st.end(), tst.begin(), tst.end());
  cst.push_back(int(cacc));
  plan.seg.ensure(size_t(plan.groups + tiles) * kTileN * g.PP);
  plan.desc.ensure(sizeof(GroupGemm) * d.size());
  plan.cast_desc.ensure(sizeof(GroupCast) * cd.size());
  plan.start.ensure(st.size());
  plan.cast_start.ensure(cst.size());
  XF_HIP(hipMemcpy(plan.desc.p, d.data(), sizeof(GroupGemm) * d.size(), hipMemcpyHostToDevice));
  XF_HIP(hipMemcpy(plan.cast_desc.p, cd.data(), sizeof(GroupCast) * cd.size(), hipMemcpyHostToDevice));
  XF_HIP(hipMemcpy(plan.start.p, st.data(), sizeof(int) * st.size(), hipMemcpyHostToDevice));
  XF_HIP(hipMemcpy(plan.cast_start.p, cst.data(), sizeof(int) * cst.size(), hipMemcpyHostToDevice));
}

// Autotuner of a grouped GEMM: every round size runs on the batch itself
// (alone on the device, after one untimed launch), timed with HIP events; the
// fastest is kept.  The runs add into the locals, which the graph's prologue
// clears.
void m2l_group_setup(const std::vector<Ctx *> &probs, GemmGroupPlan &plan, hipStream_t s, bool tune) {
  if (probs.empty()) return;
  const Geom g = geom(probs[0]->P);
  const int dev = probs[0]->cfg.device;
  const std::vector<int> rounds = gemm_rounds(g, dev);
  int best = rounds[0];
  if (tune && rounds.size() > 1) {
    hipEvent_t e0, e1;
    XF_HIP(hipEventCreate(&e0));
    XF_HIP(hipEventCreate(&e1));
    float bt = 1e30f;
    for (const int kr : rounds) {
      const int rtb = rows_per_block(g, true, dev, kr);
      group_tables(probs, plan, rtb, kr);
      m2l_group_launch(plan, s);  // untimed
      XF_HIP(hipEventRecord(e0, s));
      m2l_group_launch(plan, s);
      XF_HIP(hipEventRecord(e1, s));
      XF_HIP(hipEventSynchronize(e1));
      float ms = 0;
      XF_HIP(hipEventElapsedTime(&ms, e0, e1));
      plan.tuned.push_back({rtb, kr, ms});
      if (ms < bt) {
        bt = ms;
        best = kr;
      }
    }
    XF_HIP(hipEventDestroy(e0));
    XF_HIP(hipEventDestroy(e1));
  }
  group_tables(probs, plan, rows_per_block(g, true, dev, best), best);
}

template <int RH>
static void launch_group(const GemmGroupPlan &plan, const Geom &g, hipStream_t s) {
  const GroupGemm *d = reinterpret_cast<const GroupGemm *>(plan.desc.p);
  gemm_attr(&k_m2l_bf16x3_grouped<RH>);
  hipLaunchKernelGGL((k_m2l_bf16x3_grouped<RH>), dim3(plan.groups, ceil_div(g.R, plan.rtb)), dim3(kGemmThreads),
                     plan.lds, s, d, plan.start.p, plan.nprob, g.PP, g.R, plan.rtb, g.K32, bf16_row(g), g.P, plan.kr,
                     gemm_ring(g.K32, plan.kr), plan.seg.p);
  XF_LAUNCH();
  const int vec = sk_combine_vec(g.PP, g.PP);
  hipLaunchKernelGGL(vec == 4 ? k_sk_combine_grouped<4> : k_sk_combine_grouped<1>,
                     dim3(ceil_div(int64_t(kTileN) * g.PP / vec, 256), plan.ntiles), dim3(256), 0, s, d,
                     plan.start.p, plan.start.p + plan.nprob + 1, plan.nprob, g.PP, plan.groups, plan.seg.p);
  XF_LAUNCH();
}

void m2l_group_launch(const GemmGroupPlan &plan, hipStream_t s) {
  if (!plan.nprob) return;
  const Geom g = geom(plan.P);
  const GroupCast *cd = reinterpret_cast<const GroupCast *>(plan.cast_desc.p);
  hipLaunchKernelGGL(k_mt_grouped, dim3(plan.cast_blocks), dim3(256), 0, s, cd, plan.cast_start.p, plan.nprob);
  XF_LAUNCH();
  switch (plan.rtb) {
    case 1: return launch_group<1>(plan, g, s);
    case 2: return launch_group<2>(plan, g, s);
    case 3: return launch_group<3>(plan, g, s);
    case 4: return launch_group<4>(plan, g, s);
    case 5: return launch_group<5>(plan, g, s);
    case 6: return launch_group<6>(plan, g, s);
    case 7: return launch_group<7>(plan, g, s);
    case 8: return launch_group<8>(plan, g, s);
    case 9: return launch_group<9>(plan, g, s);
    default: fail(EXAFMM_ERR_UNSUPPORTED, "expansion order");
  }
}

}  // namespace xf
