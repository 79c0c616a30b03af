// traverse.hip -- dual-tree traversal emitting flat M2L / P2P lists.
//
// Reference: the dual-tree rule of 3d/traverse_eager.h:147-165 and its lazy
// list form 3d/traverse_lazy.h:27-43:
//   MAC |Xi-Xj|^2 theta^2 > (Ri+Rj)^2          -> M2L(Ci, Cj)
//   both leaves                                -> P2P(Ci, Cj)
//   Cj leaf or (Ri >= Rj and Ci not a leaf)    -> split Ci
//   otherwise                                  -> split Cj
// Target-centric, level-synchronous form: a pair (c, b) is visited iff b
// is handed down from c's parent (the parent's pair split on the target
// side) or b is a child of a pair (c, parent(b)) split on the source side.
// One wavefront per target cell works through its pairs breadth-first in
// LDS, so every target's lists are built by one wave, in a fixed order.  One
// launch per level: the entries are staged in LDS, a workgroup reserves room
// for its targets' lists with one atomic per output array, and the waves copy
// their entries there (where a list lands varies from run to run, its
// contents do not).  At 2^20 uniform bodies the lists took 365 us as a count
// launch, an exclusive scan and a fill launch per level.
// The MAC is evaluated in FP64 with contraction disabled, so each pair is
// classified exactly as the reference classifies it.
//
// Periodic boundary (3dp/traverse_lazy.h:39-57, 124-135): the source tree
// is visited in its 27 near images; every list entry carries its image
// index (packed as cell * 32 + image, image = ix+1 + 3(iy+1) + 9(iz+1)) and
// the MAC uses dX = Xc - Xb - iX * cycle.  Free space uses image 13 (0,0,0).
#include <algorithm>

#include "fmm_internal.h"
#include "list_capacity.h"

namespace xf {

constexpr int kTravWaves = 8;
// Pairs per target: the queue that fits beside the staged lists at 16 waves
// per CU, and the one a pass is repeated with when a target overflows it.
// The large one leaves room for one workgroup per CU instead of three; a context
// that needed it (theta below about 0.3) keeps it.  30,000 uniform bodies, ncrit
// 32: the lists take 298 us at theta 0.25 and 412 at 0.2, 391 and 721 as count,
// scan and fill launches on that queue.
constexpr int kQSmall = 768, kQCap = 2048;
// list entries staged per target; a longer list is walked a second time,
// straight into place
constexpr int kStageM2L = 256, kStageP2P = 128, kStageOut = 256;
// Passes at most: lists that are cut short at every level double the hand-down
// list's room each time (96 entries per cell; a target hands down fewer than
// kQCap), and the large queue and a larger key table may take one each.
constexpr int kListPasses = 16;
constexpr unsigned long long kEmpty = ~0ull;

struct TravArgs {
  // target tree
  const double4 *cx;
  const int *cnch, *clevel, *cparent;
  // source tree
  const double4 *scx;
  const int *scnch, *scchild, *sclevel;
  double theta;
  double cycle;
  int periodic;
  int lstart, lcount;
  // hand-down lists
  const int *in_beg, *in_cnt, *in;
  int *out_cnt, *out_beg, *out;
  // results
  int *m2l_cnt, *m2l_beg;
  int2 *m2l;
  int *p2p_cnt, *p2p_beg, *p2p;
  int *flags;
  unsigned long long *tot;
  int64_t cap_m2l, cap_p2p, cap_out;
  // translation keys
  unsigned long long *hslots;
  int hmask;
  int want_keys;
  int self_start;  // first level: each cell starts from (itself, no shift) -- a forest's problem roots
};

__device__ inline unsigned long long mix64(unsigned long long x) {
  x ^= x >> 33;
  x *= 0xff51afd7ed558ccdull;
  x ^= x >> 33;
  x *= 0xc4ceb9fe1a85ec53ull;
  x ^= x >> 33;
  return x;
}

// Key of the M2L translation (c <- b): integer offset (Xc - Xb) / Rf in units
// of the finer radius Rf, level difference, and -- periodic only -- the
// image and the level of Rf (the image shift is not a whole number of
// cell widths).  Under radius scaling of M and L the operator depends on
// nothing else.  Layout: dx,dy,dz 16 bits each, image 5, level 5, diff 6.
__device__ inline bool m2l_key(double4 Xc, int lc, double4 Xb, int lb, int img, int periodic,
                               unsigned long long &key) {
  // The offset is a whole number of finer radii (up to the rounding of the
  // centres), so one reciprocal serves the three components: its relative
  // error moves an offset of at most 32767 by far less than the 0.5 rint
  // tolerates.
  const double inv = 1.0 / fmin(Xc.w, Xb.w);
  const double dx = rint((Xc.x - Xb.x) * inv), dy = rint((Xc.y - Xb.y) * inv), dz = rint((Xc.z - Xb.z) * inv);
  const double lim = 32767.0;
  const int ld = lc - lb;
  if (fabs(dx) > lim || fabs(dy) > lim || fabs(dz) > lim || ld < -31 || ld > 31) return false;
  const unsigned long long ix = (unsigned long long)((long long)dx + 32768);
  const unsigned long long iy = (unsigned long long)((long long)dy + 32768);
  const unsigned long long iz = (unsigned long long)((long long)dz + 32768);
  const unsigned long long im = periodic ? unsigned(img) : 13u;
  const unsigned long long lf = periodic ? unsigned(max(lc, lb)) : 0u;
  key = (ix << 48) | (iy << 32) | (iz << 16) | (im << 11) | (lf << 6) | (unsigned long long)(ld + 32);
  return true;
}

// Slots only go from empty to a key during a pass, so the probe reads at
// workgroup scope (served from the CU's L1 once the few hundred live keys
// are there): a stale read shows either the empty value, and the CAS then
// returns the slot's real content, or another key, and the probe moves on;
// it never shows a key the slot does not hold.
__device__ inline int key_insert(unsigned long long *slots, int mask, unsigned long long key, int *flags) {
  int h = int(mix64(key) & (unsigned long long)mask);
  for (int probe = 0; probe <= mask; probe++) {
    unsigned long long v = __hip_atomic_load(&slots[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (v == key) return h;
    if (v == kEmpty) {
      const unsigned long long prev = atomicCAS(&slots[h], kEmpty, key);
      if (prev == kEmpty || prev == key) return h;
    }
    h = (h + 1) & mask;
  }
  atomicOr(flags, 8);
  return 0;
}

// Exclusive prefix over the lanes of v (0 .. 15) and the total: one ballot per
// bit of v, no trips through LDS on the walk's chain.
__device__ inline int wave_excl_scan(int v, unsigned long long lt, int &total) {
  int x = 0;
  total = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const unsigned long long m = __ballot((v >> k) & 1);
    x += __popcll(m & lt) << k;
    total += __popcll(m) << k;
  }
  return x;
}

// Hash slot of the translation of list entry `entry` (source cell << 5 | image).
__device__ inline int entry_slot(const TravArgs &a, double4 Xc, int lc, int entry) {
  const int b = entry >> 5;
  unsigned long long key;
  if (m2l_key(Xc, lc, a.scx[b], a.sclevel[b], entry & 31, a.periodic, key))
    return key_insert(a.hslots, a.hmask, key, a.flags);
  atomicOr(a.flags, 16);
  return 0;
}

// The walk of one target's pairs (a wave); q[0 .. tail) holds the initial
// ones.  emit(kind, position within that kind's list, entry) receives every
// entry, kind 0 = M2L, 1 = P2P, 2 = handed down to the children.  Returns false
// if the queue overflows.  A round is a chain -- queue, cells, ballots, queue --
// and what can be left out of it is: the translation keys are hashed when the
// lists are copied out, by full waves side by side (hashed here, the children's
// index loaded after the test and their places found by a shuffle scan, the
// levels of 1.5M clustered bodies took 0.90 ms, now 0.55).
template <int QCAP, class F>
__device__ __attribute__((always_inline)) inline bool walk(const TravArgs &a, int *q, int tail, int lane, double4 Xc,
                                                           int leafc, int &nm, int &np, int &no, F &&emit) {
  const unsigned long long lt = lane ? (~0ull >> (64 - lane)) : 0ull;
  const double th2 = a.theta;
  int head = 0;
  nm = np = no = 0;
  while (head < tail) {
    const int k = min(kWave, tail - head);
    int b = -1, kind = -1, nchb = 0, first = 0;
    double4 Xb;
    int img = 13;
    if (lane < k) {
      const int e = q[(head + lane) % QCAP];
      b = e >> 5;
      img = e & 31;
      Xb = a.scx[b];
      nchb = a.scnch[b];
      first = a.scchild[b];
      const double sx = ((img % 3) - 1) * a.cycle, sy = (((img / 3) % 3) - 1) * a.cycle,
                   sz = ((img / 9) - 1) * a.cycle;
      bool mac;
      {
#pragma clang fp contract(off)
        const double dx = Xc.x - Xb.x - sx, dy = Xc.y - Xb.y - sy, dz = Xc.z - Xb.z - sz;
        const double R2 = (dx * dx + dy * dy + dz * dz) * th2 * th2;
        const double Rs = Xc.w + Xb.w;
        mac = R2 > Rs * Rs;
      }
      if (mac)
        kind = 0;
      else if (leafc && nchb == 0)
        kind = 1;
      else if (nchb == 0 || (Xc.w >= Xb.w && !leafc))
        kind = 2;
      else
        kind = 3;
    }
    const unsigned long long mm = __ballot(kind == 0), mp = __ballot(kind == 1), mo = __ballot(kind == 2);
    if (kind == 0)
      emit(0, nm + __popcll(mm & lt), (b << 5) | img);
    else if (kind == 1)
      emit(1, np + __popcll(mp & lt), (b << 5) | img);
    else if (kind == 2)
      emit(2, no + __popcll(mo & lt), (b << 5) | img);
    nm += __popcll(mm);
    np += __popcll(mp);
    no += __popcll(mo);
    // split the source: enqueue its children
    const int nadd = kind == 3 ? nchb : 0;
    int total;
    const int off = wave_excl_scan(nadd, lt, total);
    if (tail - head - k + total > QCAP) return false;
    if (nadd) {
      for (int i = 0; i < nadd; i++) q[(tail + off + i) % QCAP] = ((first + i) << 5) | img;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    head += k;
    tail += total;
  }
  return true;
}

// Initial pairs of target c: handed down from the parent, or (root, root).
// Returns their number, -1 if they overflow the queue; 0 if the parent's list
// did not fit (its launch raised the flag that repeats the pass with more room).
template <int QCAP>
__device__ inline int start_pairs(const TravArgs &a, int c, int lane, int *q) {
  int tail;
  if (a.in) {
    const int par = a.cparent[c];
    const int ib = a.in_beg[par];
    tail = a.in_cnt[par];
    if (int64_t(ib) + tail > a.cap_out) return 0;
    if (tail > QCAP) return -1;
    for (int i = lane; i < tail; i += kWave) q[i] = a.in[ib + i];
  } else if (a.self_start) {
    tail = 1;
    if (lane == 0) q[0] = (c << 5) | 13;
  } else if (a.periodic) {
    tail = 27;
    if (lane < 27) q[lane] = lane;  // (root, image) for the 27 near images
  } else {
    tail = 1;
    if (lane == 0) q[0] = 13;  // (root, no shift)
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  return tail;
}

template <int QCAP>
__global__ void __launch_bounds__(kTravWaves *kWave) k_traverse(TravArgs a) {
  __shared__ int queue[kTravWaves][QCAP];
  __shared__ int sm[kTravWaves][kStageM2L], sp[kTravWaves][kStageP2P], so[kTravWaves][kStageOut];
  __shared__ int cnt[kTravWaves][3];
  __shared__ long long base[3];
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  const int t = blockIdx.x * kTravWaves + w;
  const int c = a.lstart + t;
  const bool in = t < a.lcount;
  int *q = queue[w];
  double4 Xc = make_double4(0, 0, 0, 0);
  int leafc = 0, lc = 0, nm = 0, np = 0, no = 0;
  if (in) {
    Xc = a.cx[c];
    leafc = a.cnch[c] == 0;
    lc = a.clevel[c];
    const int tail = start_pairs<QCAP>(a, c, lane, q);
    const bool ok = tail >= 0 && walk<QCAP>(a, q, tail, lane, Xc, leafc, nm, np, no,
                                            [&](int kind, int pos, int entry) {
                                              if (kind == 0) {
                                                if (pos < kStageM2L) sm[w][pos] = entry;
                                              } else if (kind == 1) {
                                                if (pos < kStageP2P) sp[w][pos] = entry;
                                              } else if (pos < kStageOut) {
                                                so[w][pos] = entry;
                                              }
                                            });
    if (!ok) {
      // a repeated pass with the large queue, or (that one too) an error
      if (lane == 0) atomicOr(a.flags, QCAP < kQCap ? kListQueue : 4);
      nm = np = no = 0;
    }
  }
  if (lane == 0) {
    cnt[w][0] = nm;
    cnt[w][1] = np;
    cnt[w][2] = no;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    int s = 0;
    for (int i = 0; i < kTravWaves; i++) s += cnt[i][threadIdx.x];
    const int64_t cap = threadIdx.x == 0 ? a.cap_m2l : threadIdx.x == 1 ? a.cap_p2p : a.cap_out;
    int b0 = 0;
    if (s) {  // counted in 64 bits: a total past 2^31 entries raises the flag too
      const unsigned long long first = atomicAdd(a.tot + threadIdx.x, (unsigned long long)s);
      if (list_overflows(first, s, cap)) atomicOr(a.flags, 1);
      b0 = list_place(first, cap);
    }
    base[threadIdx.x] = b0;
  }
  __syncthreads();
  if (!in) return;
  long long bm = base[0], bp = base[1], bo = base[2];
  for (int i = 0; i < w; i++) {
    bm += cnt[i][0];
    bp += cnt[i][1];
    bo += cnt[i][2];
  }
  if (lane == 0) {
    a.m2l_beg[c] = list_place(bm, a.cap_m2l);
    a.m2l_cnt[c] = nm;
    a.p2p_beg[c] = list_place(bp, a.cap_p2p);
    a.p2p_cnt[c] = np;
    a.out_beg[c] = list_place(bo, a.cap_out);
    a.out_cnt[c] = no;
  }
  auto place = [&](int kind, int pos, int entry) {
    if (kind == 0) {
      const int slot = a.want_keys ? entry_slot(a, Xc, lc, entry) : 0;
      if (bm + pos < a.cap_m2l) a.m2l[bm + pos] = make_int2(entry, slot);
    } else if (kind == 1) {
      if (bp + pos < a.cap_p2p) a.p2p[bp + pos] = entry;
    } else if (bo + pos < a.cap_out) {
      a.out[bo + pos] = entry;
    }
  };
  if (nm > kStageM2L || np > kStageP2P || no > kStageOut) {
    walk<QCAP>(a, q, start_pairs<QCAP>(a, c, lane, q), lane, Xc, leafc, nm, np, no, place);
    return;
  }
  for (int i = lane; i < np; i += kWave) place(1, i, sp[w][i]);
  for (int i = lane; i < no; i += kWave) place(2, i, so[w][i]);
  for (int i = lane; i < nm; i += kWave) place(0, i, sm[w][i]);
}

// Start of a pass: empty key table, zero totals and flags, zero locals, and
// in a forest empty lists for the cells above the problems' roots.
__global__ void __launch_bounds__(256) k_lists_init(unsigned long long *__restrict__ slots, int nslots,
                                                    int *__restrict__ tot, double *__restrict__ L, int64_t nL,
                                                    TravArgs a, int nv) {
  const int64_t i0 = int64_t(blockIdx.x) * 256 + threadIdx.x, n = int64_t(gridDim.x) * 256;
  for (int64_t i = i0; i < nslots; i += n) slots[i] = kEmpty;
  for (int64_t i = i0; i < nL; i += n) L[i] = 0.0;
  if (i0 < 8) tot[i0] = 0;
  for (int64_t i = i0; i < nv; i += n)
    a.m2l_cnt[i] = a.m2l_beg[i] = a.p2p_cnt[i] = a.p2p_beg[i] = a.out_cnt[i] = a.out_beg[i] = 0;
}

__global__ void k_hash_collect(const unsigned long long *__restrict__ slots, int n,
                               unsigned long long *__restrict__ keys, int *__restrict__ sl, int *__restrict__ count) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n && slots[i] != kEmpty) {
    const int p = atomicAdd(count, 1);
    keys[p] = slots[i];
    sl[p] = i;
  }
}

// M2L entries carry their hash slot out of the traversal; after the keys are
// sorted the slot becomes the key's rank (the id the operators are stored by).
// The count is the device total (tot: Lists::tot), capped at the list
// capacity; flags (if given) skip a pass that is repeated or ranked by the radix
// sort instead.  host_tot (if given) receives the totals and flags (pinned memory).
__global__ void k_entry_ids(int2 *__restrict__ m2l, const int *__restrict__ tot, int64_t cap,
                            const int *__restrict__ slot2id, const int *__restrict__ flags, int *host_tot) {
  if (host_tot && blockIdx.x == 0 && threadIdx.x < 8)
    __hip_atomic_store(host_tot + threadIdx.x, tot[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (flags && (*flags & (kListRetry | 32))) return;
  const int64_t n = min(*reinterpret_cast<const int64_t *>(tot), cap);
  for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256)
    m2l[i].y = slot2id[m2l[i].y];
}

// Key sort for the usual key sets (hundreds to some ten thousand distinct
// translations): a key's rank is the number of smaller keys.  A workgroup
// ranks 64 keys, its 16 waves counting over a sixteenth of the set each (the
// keys they compare with are wave-uniform: scalar loads).  Writes the sorted
// keys and the slot -> rank map.  A larger set raises bit 32 of *flags and is
// left to the radix sort.  (One workgroup over the whole set in LDS: 34 us for
// 1,164 keys, 109 us for 2,180, now 5 - 6 us.)
constexpr int kRankMax = 12288;
__global__ void __launch_bounds__(1024) k_key_rank(const unsigned long long *__restrict__ in,
                                                   const int *__restrict__ sl, const int *__restrict__ count,
                                                   unsigned long long *__restrict__ keys, int *__restrict__ slot2id,
                                                   int *__restrict__ flags) {
  __shared__ int part[16][kWave];
  const int n = *count;
  if (n > kRankMax) {
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(flags, 32);
    return;
  }
  const int lane = threadIdx.x & (kWave - 1), w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int i = blockIdx.x * kWave + lane;
  if (int(blockIdx.x) * kWave >= n) return;
  const unsigned long long k = i < n ? in[i] : 0ull;
  int r = 0;
  for (int j = w * n / 16; j < (w + 1) * n / 16; j++) r += in[j] < k;
  part[w][lane] = r;
  __syncthreads();
  if (w != 0 || i >= n) return;
  r = 0;
  for (int q = 0; q < 16; q++) r += part[q][lane];
  keys[r] = k;
  slot2id[sl[i]] = r;
}

__global__ void k_slot_ids(const int *__restrict__ sl, int n, int *__restrict__ slot2id) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) slot2id[sl[i]] = i;
}

void traverse(Ctx &tc, const Ctx &sc, const std::function<void()> &after_kernels) {
  Tree &T = tc.t;
  const Tree &S = sc.t;
  Lists &Lr = tc.lists;
  hipStream_t s = tc.s0;
  const int64_t nc = T.ncells;
  const bool keys = (&tc == &sc);
  if (S.ncells >= (int64_t(1) << 26)) fail(EXAFMM_ERR_CAPACITY, "more than 2^26 cells");
  Lr.m2l_beg.ensure(nc);
  Lr.m2l_cnt.ensure(nc);
  Lr.p2p_beg.ensure(nc);
  Lr.p2p_cnt.ensure(nc);
  Lr.out_beg.ensure(nc);
  Lr.out_cnt.ensure(nc);
  Lr.tot.ensure(8);
  tc.pin_i.ensure(kPinInts);
  tc.L.ensure(size_t(nc) * tc.P * tc.P);
  Lr.cap_m2l = std::max(Lr.cap_m2l, list_capacity(nc, 200));
  Lr.cap_p2p = std::max(Lr.cap_p2p, list_capacity(nc, 96));
  Lr.cap_out = std::max(Lr.cap_out, list_capacity(nc, 96));
  if (keys && Lr.hcap == 0) Lr.hcap = 1 << 16;

  int tot[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  uint64_t total[3] = {0, 0, 0};
  bool done = false;
  for (int attempt = 0; attempt < kListPasses; attempt++) {
    Lr.m2l.ensure(Lr.cap_m2l);
    Lr.p2p.ensure(Lr.cap_p2p);
    Lr.out.ensure(Lr.cap_out);
    if (keys) Lr.hslots.ensure(Lr.hcap);
    TravArgs a{};
    a.cx = T.cx.p;
    a.cnch = T.cnch.p;
    a.clevel = T.clevel.p;
    a.cparent = T.cparent.p;
    a.scx = S.cx.p;
    a.scnch = S.cnch.p;
    a.scchild = S.cchild.p;
    a.sclevel = S.clevel.p;
    a.theta = tc.cfg.theta;
    a.periodic = tc.cfg.images > 0;
    a.cycle = tc.cfg.images > 0 ? tc.cfg.cycle : 0.0;
    a.out_cnt = Lr.out_cnt.p;
    a.out_beg = Lr.out_beg.p;
    a.out = Lr.out.p;
    a.m2l_cnt = Lr.m2l_cnt.p;
    a.m2l_beg = Lr.m2l_beg.p;
    a.m2l = Lr.m2l.p;
    a.p2p_cnt = Lr.p2p_cnt.p;
    a.p2p_beg = Lr.p2p_beg.p;
    a.p2p = Lr.p2p.p;
    a.flags = Lr.tot.p + kTotFlags;
    a.tot = reinterpret_cast<unsigned long long *>(Lr.tot.p);
    a.cap_m2l = Lr.cap_m2l;
    a.cap_p2p = Lr.cap_p2p;
    a.cap_out = Lr.cap_out;
    a.hslots = Lr.hslots.p;
    a.hmask = Lr.hcap - 1;
    a.want_keys = keys;
    // a forest starts at its problems' roots (level lroot): the cells above
    // are never paired, their lists stay empty
    const int l0 = T.lroot;
    if (l0 > 0 && &tc != &sc) fail(EXAFMM_ERR_UNSUPPORTED, "a forest's horizontal pass needs source == target");
    a.self_start = l0 > 0;
    const int64_t nL = nc * tc.P * tc.P;
    hipLaunchKernelGGL(k_lists_init, dim3(int(std::max<int64_t>(64, std::min<int64_t>(ceil_div(nL, 256 * 4), 2048)))),
                       dim3(256), 0, s, Lr.hslots.p, keys ? Lr.hcap : 0, Lr.tot.p, tc.L.p, nL, a,
                       l0 > 0 ? T.lstart[l0] : 0);
    XF_LAUNCH();
    for (int l = l0; l <= T.depth; l++) {
      a.lstart = T.lstart[l];
      a.lcount = T.lstart[l + 1] - T.lstart[l];
      a.in = l > l0 ? Lr.out.p : nullptr;
      a.in_beg = Lr.out_beg.p;
      a.in_cnt = Lr.out_cnt.p;
      const int g = ceil_div(a.lcount, kTravWaves);
      hipLaunchKernelGGL(Lr.large_queue ? k_traverse<kQCap> : k_traverse<kQSmall>, dim3(g), dim3(kTravWaves * kWave), 0,
                         s, a);
      XF_LAUNCH();
    }
    if (after_kernels) after_kernels();
    if (keys) {
      // distinct translation keys out of the hash table (discarded if the
      // pass has to be repeated), counted into tot[kTotKeys]
      Lr.keys.ensure(size_t(Lr.hcap) * 2);
      Lr.kscratch.ensure(size_t(Lr.hcap) * 2 + 8);
      Lr.slot2id.ensure(Lr.hcap);
      hipLaunchKernelGGL(k_hash_collect, dim3(ceil_div(Lr.hcap, 256)), dim3(256), 0, s, Lr.hslots.p, Lr.hcap,
                         Lr.keys.p + Lr.hcap, Lr.kscratch.p, Lr.tot.p + kTotKeys);
      XF_LAUNCH();
      // The usual small key set is ranked, and the entries renumbered,
      // before the totals are read, so the read overlaps them (counts from
      // the device; a repeated pass redoes it all, a set above kRankMax is
      // flagged and sorted below).
      hipLaunchKernelGGL(k_key_rank, dim3(std::min(Lr.hcap, kRankMax) / kWave), dim3(1024), 0, s, Lr.keys.p + Lr.hcap,
                         Lr.kscratch.p, Lr.tot.p + kTotKeys, Lr.keys.p, Lr.slot2id.p, Lr.tot.p + kTotFlags);
      XF_LAUNCH();
      hipLaunchKernelGGL(k_entry_ids, dim3(int(std::min<int64_t>(ceil_div(Lr.cap_m2l, 256), 4096))), dim3(256), 0, s,
                         Lr.m2l.p, Lr.tot.p, Lr.cap_m2l, Lr.slot2id.p, Lr.tot.p + kTotFlags, tc.pin_i.p + kPinTot);
      XF_LAUNCH();
    }
    if (!keys) XF_HIP(hipMemcpyAsync(tc.pin_i.p + kPinTot, Lr.tot.p, sizeof(tot), hipMemcpyDeviceToHost, s));
    stream_wait(s);
    std::copy(tc.pin_i.p + kPinTot, tc.pin_i.p + kPinTot + 8, tot);
    std::memcpy(total, tot, sizeof(total));
    const int flags = tot[kTotFlags];
    // work started by after_kernels ends before a repeated pass resets the flags
    if (after_kernels && (flags & kListRetry)) stream_wait(tc.s1);
    if (flags & 4) fail(EXAFMM_ERR_CAPACITY, "traversal work queue overflow (pairs per target cell > 2048)");
    if (flags & 16) fail(EXAFMM_ERR_CAPACITY, "M2L offset out of key range");
    // what the next pass needs more of (a pass cut short shows lower bounds)
    if (flags & kListQueue) Lr.large_queue = true;
    if (flags & 1) {
      int64_t *const cap[3] = {&Lr.cap_m2l, &Lr.cap_p2p, &Lr.cap_out};
      for (int k = 0; k < 3; k++) {
        const int64_t n = list_grow(*cap[k], total[k]);
        if (!n) fail(EXAFMM_ERR_CAPACITY, "more than 2^31 - 1 entries of one kind of interaction list");
        *cap[k] = n;
      }
    }
    if (flags & 8) {
      if (Lr.hcap >= 1 << 24) fail(EXAFMM_ERR_CAPACITY, "more than 2^23 distinct M2L translations");
      Lr.hcap *= 4;
    }
    if (flags & kListRetry) continue;
    Lr.nm2l = int64_t(total[0]);
    Lr.np2p = int64_t(total[1]);
    done = true;
    break;
  }
  if (!done) fail(EXAFMM_ERR_CAPACITY, "interaction lists or key table still full");
  Lr.valid = true;
  Lr.nkeys = 0;
  if (keys) {
    unsigned long long *k1 = Lr.keys.p + Lr.hcap, *k2 = Lr.keys.p;
    int *v1 = Lr.kscratch.p, *v2 = Lr.kscratch.p + Lr.hcap;
    const int nk = tot[kTotKeys];
    if (tot[kTotFlags] & 32) {  // more keys than k_key_rank holds
      radix_sort_pairs(k1, v1, k2, v2, nk, 0, 64, T.rs_hist, s);
      hipLaunchKernelGGL(k_slot_ids, dim3(ceil_div(std::max(nk, 1), 256)), dim3(256), 0, s, v1, nk, Lr.slot2id.p);
      XF_LAUNCH();
      if (k1 != Lr.keys.p)
        XF_HIP(hipMemcpyAsync(Lr.keys.p, k1, sizeof(unsigned long long) * nk, hipMemcpyDeviceToDevice, s));
      if (Lr.nm2l > 0) {
        hipLaunchKernelGGL(k_entry_ids, dim3(std::min(ceil_div(Lr.nm2l, 256), 4096)), dim3(256), 0, s, Lr.m2l.p,
                           Lr.tot.p, Lr.cap_m2l, Lr.slot2id.p, (const int *)nullptr, (int *)nullptr);
        XF_LAUNCH();
      }
    }
    Lr.nkeys = nk;
  }
}

}  // namespace xf
