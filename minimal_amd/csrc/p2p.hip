// p2p.hip -- near-field body-body interactions and the FP64 direct sum.
//
// Reference: P2P 3d/kernel.h:122-150 over each target's P2P list
// (3d/traverse_lazy.h:56), direct 3d/traverse_eager.h:193-202.
// Both add p += q/r and F -= q*dX/r^3 (dX = x_target - x_source) and skip
// pairs at zero distance.
//
// FP32 path: one wavefront per target leaf.  The leaf's list entries
// (source leaves, with their periodic image) are staged in LDS with a prefix
// of their body counts; the sources themselves are then staged 256 at a
// time as float(X_s + shift - C_t) -- computed in FP64 from the tree-order
// coordinates and rounded once -- so a body that is both target and source
// gets the same FP32 coordinates either way and its zero distance is exact
// (also between two different trees).  Targets are float(X_t - C_t), the
// tree's leaf-relative copy.
//
// The leaf's targets go in balanced blocks of at most kP2PTC: a block's
// targets are wave-uniform (scalar registers), and lane l takes staged
// source 64k + l in round k, so each round is one LDS read per lane and TC
// interactions per lane, with no padding of the target block.  Per lane and
// target the four sums (p and the three force components) run over the
// lane's sources; at the end the 64 lane partials are added by recursive
// halving across lanes, in a fixed order.
//
// EXAFMM_PREC_FP32_NEWTON refines the hardware 1/sqrt by one Newton step
// y (3 - r^2 y^2) / 2 and compensates the sums: every kP2PFlush rounds the
// lane partials (FP32 sums of at most kP2PFlush terms) are reduced across
// the lanes and added into Kahan-compensated running sums, one per lane
// (a lane holds one target's p or force component after the reduction).
#include <algorithm>
#include <type_traits>

#include "fmm_internal.h"

namespace xf {

constexpr int kP2PWaves = 4;      // target leaves per workgroup, one wave each
constexpr int kP2PSeg = 128;      // list entries staged per segment
constexpr int kP2PChunk = 256;    // sources staged per chunk (4 rounds of 64)
constexpr int kP2PTC = 16;        // targets per block (plain)
#ifndef P2P_FLUSH
#define P2P_FLUSH 64
#endif
constexpr int kP2PFlush = P2P_FLUSH;  // rounds per compensated block (Newton + compensated)
#ifndef P2P_TC_STEP
#define P2P_TC_STEP 1
#endif
constexpr int kP2PTCStep = P2P_TC_STEP;  // block sizes are multiples of this (instantiated variants)

__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

template <int N>
constexpr int pow2ceil() {
  return N <= 1 ? 1 : 2 * pow2ceil<(N + 1) / 2>();
}

// Kahan step: s + v with the rounding error carried in c (s - c is the sum).
__device__ inline void kahan_add(float &s, float &c, float v) {
  const float y = v - c;
  const float t = s + y;
  c = (t - s) - y;
  s = t;
}

struct P2PLds {
  int pre[kP2PSeg + 1];    // prefix of the staged entries' body counts
  int beg[kP2PSeg];        // first source body of each entry
  int cnt[kP2PSeg];        // body count of each entry
  double dlx[kP2PSeg], dly[kP2PSeg], dlz[kP2PSeg];  // shift - C_t of each entry
  float4 src[kP2PChunk];   // staged sources: x, y, z in the target frame, q
};

// Stages list entries [seg, seg + ne) of the target leaf: the leaf's own
// entry (image 13) moves to position 0; returns the number of sources and
// sets *nself to the body count of the leaf's own entry (0 if absent).
__device__ inline int p2p_stage_entries(P2PLds &L, const int *__restrict__ list, int b0, int seg, int ne,
                                        int self_key, const int *__restrict__ scbeg,
                                        const int *__restrict__ sccnt, double4 Cc, double cycle, int lane,
                                        int *nself) {
  constexpr int kPer = kP2PSeg / kWave;
  wave_sync();
  int self = -1;
#pragma unroll
  for (int k = 0; k < kPer; k++) {
    const int e = lane * kPer + k;
    if (e < ne && list[b0 + seg + e] == self_key) self = e;
  }
  const unsigned long long hit = __ballot(self >= 0);
  const int sidx = hit ? __shfl(self, __ffsll((long long)hit) - 1) : -1;
#pragma unroll
  for (int k = 0; k < kPer; k++) {
    const int e = lane * kPer + k;
    if (e < ne) {
      const int pos = e == sidx ? 0 : (e == 0 && sidx > 0 ? sidx : e);
      const int en = list[b0 + seg + e];
      const int sc = en >> 5, img = en & 31;
      L.cnt[pos] = sccnt[sc];
      L.beg[pos] = scbeg[sc];
      L.dlx[pos] = ((img % 3) - 1) * cycle - Cc.x;
      L.dly[pos] = (((img / 3) % 3) - 1) * cycle - Cc.y;
      L.dlz[pos] = ((img / 9) - 1) * cycle - Cc.z;
    }
  }
  wave_sync();
  int cnt[kPer], run = 0;
#pragma unroll
  for (int k = 0; k < kPer; k++) {
    const int e = lane * kPer + k;
    cnt[k] = e < ne ? L.cnt[e] : 0;
    run += cnt[k];
  }
  int incl = run;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int v = __shfl_up(incl, d);
    if (lane >= d) incl += v;
  }
  int acc = incl - run;
  if (lane == 0) L.pre[0] = 0;
#pragma unroll
  for (int k = 0; k < kPer; k++) {
    const int e = lane * kPer + k;
    acc += cnt[k];
    if (e < ne) L.pre[e + 1] = acc;
  }
  wave_sync();
  *nself = sidx >= 0 ? L.pre[1] : 0;
  return L.pre[ne];
}

// Stages sources [c0, c0 + nsrc) of the staged entries, padded to whole
// rounds of 64 with far sources of zero charge (r^2 ~ 3e36: finite, so the
// Newton step stays finite, and the pair adds exact zeros).  e is the lane's
// entry cursor (positions only move forward).
__device__ inline void p2p_stage_sources(P2PLds &L, const double4 *__restrict__ sxs, int c0, int nsrc, int lane,
                                         int &e) {
  const int nround = (nsrc + kWave - 1) / kWave;
  const float4 far_src = make_float4(1e18f, 1e18f, 1e18f, 0.0f);
  wave_sync();  // the previous chunk has been read
#pragma unroll
  for (int k = 0; k < kP2PChunk / kWave; k++) {
    const int p = k * kWave + lane;
    if (p < nsrc) {
      const int g = c0 + p;
      while (L.pre[e + 1] <= g) e++;
      const double4 X = sxs[L.beg[e] + g - L.pre[e]];
      L.src[p] = make_float4(float(X.x + L.dlx[e]), float(X.y + L.dly[e]), float(X.z + L.dlz[e]), float(X.w));
    } else if (k < nround) {
      L.src[p] = far_src;
    }
  }
  wave_sync();
}

// One round: the lane's staged source against the TC block targets.
// CHECK skips pairs at zero distance (3d/kernel.h:139): only rounds that can
// hold such pairs use it.
template <int TC, bool CHECK, bool REFINE>
__device__ inline void p2p_round(float4 s, const float (&xt)[TC], const float (&yt)[TC], const float (&zt)[TC],
                                 float (&ap)[TC], float (&ax)[TC], float (&ay)[TC], float (&az)[TC]) {
#pragma unroll
  for (int t = 0; t < TC; t++) {
    const float dx = xt[t] - s.x, dy = yt[t] - s.y, dz = zt[t] - s.z;
    const float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
    float y = __builtin_amdgcn_rsqf(r2);
    if (REFINE) {
      const float h = (r2 * y) * y;
      y = y * fmaf(h, -0.5f, 1.5f);
    }
    if (CHECK) y = r2 > 0.0f ? y : 0.0f;
    const float qi = s.w * y;
    const float q3 = qi * (y * y);
    ap[t] += qi;
    ax[t] = fmaf(dx, q3, ax[t]);
    ay[t] = fmaf(dy, q3, ay[t]);
    az[t] = fmaf(dz, q3, az[t]);
  }
}

// Cross-lane totals of the block's four sums: halving over the targets,
// then a butterfly over the lanes that share a target.  Lane l receives
// component l % kLow (p, F_x, F_y, F_z for 0..3) of target l / kLow, with
// kLow = 64 / T2 (T2 = TC rounded up to a power of two); other lanes 0.
template <int TC, class T>
__device__ inline T p2p_lane_total(const T (&ap)[TC], const T (&ax)[TC], const T (&ay)[TC], const T (&az)[TC],
                                   int lane) {
  constexpr int T2 = pow2ceil<TC>();
  constexpr int kLow = kWave / T2;
  T vp[T2], vx[T2], vy[T2], vz[T2];
#pragma unroll
  for (int i = 0; i < T2; i++) {
    vp[i] = i < TC ? ap[i] : T(0);
    vx[i] = i < TC ? ax[i] : T(0);
    vy[i] = i < TC ? ay[i] : T(0);
    vz[i] = i < TC ? az[i] : T(0);
  }
  T rp = halving<T2>(vp, lane), rx = halving<T2>(vx, lane), ry = halving<T2>(vy, lane), rz = halving<T2>(vz, lane);
  rp = lane_sum<kLow>(rp);
  rx = lane_sum<kLow>(rx);
  ry = lane_sum<kLow>(ry);
  rz = lane_sum<kLow>(rz);
  const int comp = lane % kLow;
  return comp == 0 ? rp : comp == 1 ? rx : comp == 2 ? ry : comp == 3 ? rz : T(0);
}

// Targets t0 .. t0 + tc - 1 (tc <= TC) of a leaf (a wave) against its whole list.
// same_tree: sources and targets are one tree, so only the leaf's own entry
// can hold zero distances; otherwise every round checks.  REFINE: every
// kP2PFlush rounds the lane partials are reduced across lanes and added
// into one Kahan-compensated running sum per lane (target, component).
template <int TC, bool REFINE>
__device__ __attribute__((always_inline)) inline void p2p_block(int t0, int tc, int tb, double4 Cc, int b0, int nl,
                                                                const float4 *__restrict__ xq,
                                                                const int *__restrict__ list,
                                                                const int *__restrict__ scbeg,
                                                                const int *__restrict__ sccnt,
                                                                const double4 *__restrict__ sxs, double cycle,
                                                                int self_key, int same_tree,
                                                                exafmm_body *__restrict__ bodies, P2PLds &L) {
  const int lane = threadIdx.x & (kWave - 1);
  float xt[TC], yt[TC], zt[TC];
#pragma unroll
  for (int t = 0; t < TC; t++) {
    const float4 v = xq[tb + t0 + min(t, tc - 1)];  // wave-uniform address: scalar loads
    xt[t] = v.x;
    yt[t] = v.y;
    zt[t] = v.z;
  }
  float ap[TC], ax[TC], ay[TC], az[TC];
#pragma unroll
  for (int t = 0; t < TC; t++) ap[t] = ax[t] = ay[t] = az[t] = 0.0f;
  float ks = 0.0f, kc = 0.0f;  // compensated sum of this lane's (target, component)
  int since = 0;               // rounds since the last flush
  auto flush = [&]() {
    kahan_add(ks, kc, p2p_lane_total<TC>(ap, ax, ay, az, lane));
#pragma unroll
    for (int t = 0; t < TC; t++) ap[t] = ax[t] = ay[t] = az[t] = 0.0f;
    since = 0;
  };
  for (int seg = 0; seg < nl; seg += kP2PSeg) {
    const int ne = min(kP2PSeg, nl - seg);
    int nself = 0;
    const int total = p2p_stage_entries(L, list, b0, seg, ne, self_key, scbeg, sccnt, Cc, cycle, lane, &nself);
    // sources that can sit at zero distance: the leaf's own (staged first),
    // or all of them when the trees differ
    const int nchecked = same_tree ? nself : total;
    int e = 0;
    for (int c0 = 0; c0 < total; c0 += kP2PChunk) {
      const int nsrc = min(kP2PChunk, total - c0);
      const int nround = (nsrc + kWave - 1) / kWave;
      p2p_stage_sources(L, sxs, c0, nsrc, lane, e);
      const int nck = min(nround, max(0, (nchecked - c0 + kWave - 1) / kWave));
      int k = 0;
      for (; k < nck; k++) p2p_round<TC, true, REFINE>(L.src[k * kWave + lane], xt, yt, zt, ap, ax, ay, az);
      for (; k < nround; k++) p2p_round<TC, false, REFINE>(L.src[k * kWave + lane], xt, yt, zt, ap, ax, ay, az);
      if (REFINE) {
        since += nround;
        if (since >= kP2PFlush) flush();
      }
    }
  }
  constexpr int kLow = kWave / pow2ceil<TC>();
  const int t = lane / kLow, comp = lane % kLow;
  double v;
  if (REFINE) {
    flush();
    v = double(ks) - double(kc);
  } else {
    v = double(p2p_lane_total<TC>(ap, ax, ay, az, lane));
  }
  if (comp < 4 && t < tc) {  // slots tc .. TC - 1 repeat the last target and are not written
    exafmm_body *ob = bodies + tb + t0 + t;
    if (comp == 0)
      ob->p += v;
    else
      ob->F[comp - 1] -= v;
  }
}

// One target leaf (a wave): its targets in nb = ceil(tn / kP2PTC) blocks of
// balanced size, each run by the variant of the next multiple of
// kP2PTCStep (the extra slots repeat the block's last target).
template <bool REFINE>
__device__ __attribute__((always_inline)) inline void p2p_leaf(
    int li, const int *__restrict__ leaves, const int *__restrict__ cbeg, const int *__restrict__ ccnt,
    const double4 *__restrict__ cx, const float4 *__restrict__ xq, const int *__restrict__ lbeg,
    const int *__restrict__ lcnt, const int *__restrict__ list, const int *__restrict__ scbeg,
    const int *__restrict__ sccnt, const double4 *__restrict__ sxs, double cycle, int same_tree,
    exafmm_body *__restrict__ bodies, P2PLds &L) {
  const int c = leaves[li];
  const int tb = cbeg[c], tn = ccnt[c];
  const double4 Cc = cx[c];
  const int b0 = lbeg[c], nl = lcnt[c];
  const int self_key = same_tree ? ((c << 5) | 13) : -1;
  const int nb = (tn + kP2PTC - 1) / kP2PTC;
  const int per = (tn + nb - 1) / nb;
  for (int t0 = 0; t0 < tn; t0 += per) {
    const int tc = min(per, tn - t0);
    const int tv = (tc + kP2PTCStep - 1) / kP2PTCStep * kP2PTCStep;
#define XF_P2P_BLOCK(N)                                                                                        \
  case N:                                                                                                      \
    if (N % kP2PTCStep == 0)                                                                                   \
      p2p_block<N, REFINE>(t0, tc, tb, Cc, b0, nl, xq, list, scbeg, sccnt, sxs, cycle, self_key, same_tree, bodies, \
                           L);                                                                                 \
    break;
    switch (tv) {
      XF_P2P_BLOCK(1)
      XF_P2P_BLOCK(2)
      XF_P2P_BLOCK(3)
      XF_P2P_BLOCK(4)
      XF_P2P_BLOCK(5)
      XF_P2P_BLOCK(6)
      XF_P2P_BLOCK(7)
      XF_P2P_BLOCK(8)
      XF_P2P_BLOCK(9)
      XF_P2P_BLOCK(10)
      XF_P2P_BLOCK(11)
      XF_P2P_BLOCK(12)
      XF_P2P_BLOCK(13)
      XF_P2P_BLOCK(14)
      XF_P2P_BLOCK(15)
      XF_P2P_BLOCK(16)
      default:
        break;
    }
#undef XF_P2P_BLOCK
  }
}

// A P2P launched before the host has read the traversal's flags: it does
// nothing if that pass is to be repeated (list capacity or key table full)
// or failed (work queue overflow, offset out of key range), as its lists
// are then incomplete.
__device__ inline bool p2p_skip(const int *list_flags) {
  return list_flags && (__atomic_load_n(list_flags, __ATOMIC_RELAXED) & (kListRetry | 4 | 16));
}

template <bool REFINE>
__global__ void __launch_bounds__(kP2PWaves *kWave) __attribute__((amdgpu_waves_per_eu(REFINE ? 3 : 4))) k_p2p32(
    const int *__restrict__ leaves, const int *__restrict__ nleaves, const int *__restrict__ cbeg,
    const int *__restrict__ ccnt, const double4 *__restrict__ cx, const float4 *__restrict__ xq,
    const int *__restrict__ lbeg, const int *__restrict__ lcnt, const int *__restrict__ list,
    const int *__restrict__ scbeg, const int *__restrict__ sccnt, const double4 *__restrict__ sxs, double cycle,
    int same_tree, exafmm_body *__restrict__ bodies, const int *__restrict__ list_flags) {
  __shared__ P2PLds lds[kP2PWaves];
  // wave-uniform (scalar) leaf index: the per-leaf quantities, the block
  // targets and the loop bounds stay in scalar registers
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int li = blockIdx.x * kP2PWaves + w;
  if (li >= *nleaves || p2p_skip(list_flags)) return;  // whole wave; the kernel uses wave-level syncs only
  p2p_leaf<REFINE>(li, leaves, cbeg, ccnt, cx, xq, lbeg, lcnt, list, scbeg, sccnt, sxs, cycle, same_tree, bodies,
                   lds[w]);
}

// All problems of a batch in one launch: block b belongs to the problem i
// with start[i] <= b < start[i + 1] (each problem's own tree is source and
// target).
__global__ void __launch_bounds__(kP2PWaves *kWave) k_p2p32_grouped(const GroupTree *__restrict__ g,
                                                                    const int *__restrict__ start, int nprob) {
  __shared__ P2PLds lds[kP2PWaves];
  const int b = blockIdx.x, i = group_of(start, nprob, b);
  const GroupTree &t = g[i];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int li = (b - start[i]) * kP2PWaves + w;
  if (li >= *t.nleaves) return;
  p2p_leaf<false>(li, t.leaves, t.cbeg, t.ccnt, t.cx, t.xq, t.lbeg, t.lcnt, t.list, t.cbeg, t.ccnt, t.xs, 0.0, 1,
                  t.bodies, lds[w]);
}

// One FP64 interaction (3d/kernel.h:135-146): p += q/r, F -= q dX/r^3 (the
// caller subtracts), pairs at zero distance skipped.  The hardware's 1/sqrt
// (about 2^-23 relative) takes one third-order step
//   e = 1 - r^2 y^2,  y += y e (1/2 + 3/8 e)
// (remainder 5/16 e^3, below 2^-60), and 1/r^2 is y^2 after a Newton step of its
// own: seven FP64 operations where a divide and a square root expand to about
// forty.  The rounding is that of the divide and the root: in units of 2^-53, rms,
// 1/r 0.46 (0.46 with them), 1/r^2 0.44 (0.44; 1.03 without its step), 1/r^3 0.77
// (0.88; 1.52 without).  Squared distances outside [2^-900, 2^900) -- zero,
// overflow, NaN -- take the plain divide and root.
__device__ inline void p2p64_pair(double dx, double dy, double dz, double q, double &pot, double &ax, double &ay,
                                  double &az) {
  const double r2 = fma(dz, dz, fma(dy, dy, dx * dx));
  double y = __builtin_amdgcn_rsq(r2);
  const double t = r2 * y;
  const double e = fma(-t, y, 1.0);
  y = fma(y * e, fma(e, 0.375, 0.5), y);
  double y2 = y * y;
  y2 = fma(y2, fma(-r2, y2, 1.0), y2);
  const unsigned hi = unsigned(__double2hiint(r2));
  if (hi - (123u << 20) >= (1800u << 20)) {
    y2 = r2 != 0.0 ? 1.0 / r2 : 0.0;
    y = sqrt(y2);
  }
  const double qi = q * y;
  const double f = qi * y2;
  pot += qi;
  ax = fma(dx, f, ax);
  ay = fma(dy, f, ay);
  az = fma(dz, f, az);
}

// FP64 P2P: a workgroup per target leaf, its waves taking the leaf's targets
// in balanced blocks of at most kP2P64TC; as in the FP32 kernel a block's
// targets are wave-uniform and the lanes take the staged entries' sources,
// one load per source and block.  FP64 VALU bound (25 instructions per
// interaction, 26 with image shifts).  67,984,904 interactions (30,000 bodies): 169 us; 903 us with
// a thread per target walking its sources one by one through a divide and a
// square root each.
constexpr int kP2P64TC = 8;

template <int TC, bool PERIODIC>
__device__ __attribute__((always_inline)) inline void p2p64_block(int t0, int tc, int tb, int b0, int nl,
                                                                  const double4 *__restrict__ xs,
                                                                  const int *__restrict__ list,
                                                                  const int *__restrict__ scbeg,
                                                                  const int *__restrict__ sccnt,
                                                                  const double4 *__restrict__ sxs, double cycle,
                                                                  exafmm_body *__restrict__ bodies, P2PLds &L) {
  const int lane = threadIdx.x & (kWave - 1);
  double xt[TC], yt[TC], zt[TC], ap[TC], ax[TC], ay[TC], az[TC];
#pragma unroll
  for (int t = 0; t < TC; t++) {
    const double4 v = xs[tb + t0 + min(t, tc - 1)];  // wave-uniform address: scalar loads
    xt[t] = v.x;
    yt[t] = v.y;
    zt[t] = v.z;
    ap[t] = ax[t] = ay[t] = az[t] = 0.0;
  }
  for (int seg = 0; seg < nl; seg += kP2PSeg) {
    const int ne = min(kP2PSeg, nl - seg);
    int nself = 0;
    const int total = p2p_stage_entries(L, list, b0, seg, ne, -1, scbeg, sccnt, make_double4(0, 0, 0, 0), cycle,
                                        lane, &nself);
    // 3dp/kernel.h:133: dX = Xi - Xj - iX * cycle, the image shift last: bodies
    // that meet through an image meet exactly as they do there
    int e = 0;
    for (int g = lane; g < total; g += kWave) {
      while (L.pre[e + 1] <= g) e++;
      const double4 X = sxs[L.beg[e] + g - L.pre[e]];
#pragma unroll
      for (int t = 0; t < TC; t++) {
        double dx = xt[t] - X.x, dy = yt[t] - X.y, dz = zt[t] - X.z;
        if (PERIODIC) {
          dx -= L.dlx[e];
          dy -= L.dly[e];
          dz -= L.dlz[e];
        }
        p2p64_pair(dx, dy, dz, X.w, ap[t], ax[t], ay[t], az[t]);
      }
    }
  }
  constexpr int kLow = kWave / pow2ceil<TC>();
  const int t = lane / kLow, comp = lane % kLow;
  const double v = p2p_lane_total<TC>(ap, ax, ay, az, lane);
  if (comp < 4 && t < tc) {
    exafmm_body *ob = bodies + tb + t0 + t;
    if (comp == 0)
      ob->p += v;
    else
      ob->F[comp - 1] -= v;
  }
}

template <bool PERIODIC>
__global__ void __launch_bounds__(kP2PWaves *kWave) k_p2p64(const int *__restrict__ leaves,
                                                            const int *__restrict__ nleaves,
                                                            const int *__restrict__ cbeg, const int *__restrict__ ccnt,
                                                            const double4 *__restrict__ xs,
                                                            const int *__restrict__ lbeg,
                                                            const int *__restrict__ lcnt, const int *__restrict__ list,
                                                            const int *__restrict__ scbeg,
                                                            const int *__restrict__ sccnt,
                                                            const double4 *__restrict__ sxs, double cycle,
                                                            exafmm_body *__restrict__ bodies,
                                                            const int *__restrict__ list_flags) {
  __shared__ P2PLds lds[kP2PWaves];
  const int li = blockIdx.x;
  if (li >= *nleaves || p2p_skip(list_flags)) return;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // wave-level syncs only below
  const int c = leaves[li];
  const int tb = cbeg[c], tn = ccnt[c];
  const int b0 = lbeg[c], nl = lcnt[c];
  const int nb = (tn + kP2P64TC - 1) / kP2P64TC;
  const int per = (tn + nb - 1) / max(nb, 1);
  for (int t0 = w * per; t0 < tn; t0 += kP2PWaves * per) {
    const int tc = min(per, tn - t0);
#define XF_P2P64_BLOCK(N)                                                                          \
  case N:                                                                                          \
    p2p64_block<N, PERIODIC>(t0, tc, tb, b0, nl, xs, list, scbeg, sccnt, sxs, cycle, bodies, lds[w]);        \
    break;
    switch (tc) {
      XF_P2P64_BLOCK(1)
      XF_P2P64_BLOCK(2)
      XF_P2P64_BLOCK(3)
      XF_P2P64_BLOCK(4)
      XF_P2P64_BLOCK(5)
      XF_P2P64_BLOCK(6)
      XF_P2P64_BLOCK(7)
      XF_P2P64_BLOCK(8)
      default:
        break;
    }
#undef XF_P2P64_BLOCK
  }
}

int p2p_group_blocks(int64_t nleaves) { return ceil_div(nleaves, kP2PWaves); }

void p2p_grouped(const GroupTree *g, const int *start, int nprob, int nblocks, hipStream_t s) {
  hipLaunchKernelGGL(k_p2p32_grouped, dim3(nblocks), dim3(kP2PWaves * kWave), 0, s, g, start, nprob);
  XF_LAUNCH();
}

void p2p_apply(Ctx &tc, const Ctx &sc, hipStream_t s, const int *list_flags) {
  const Tree &T = tc.t, &S = sc.t;
  const Lists &L = tc.lists;
  const double cycle = tc.cfg.images > 0 ? tc.cfg.cycle : 0.0;
  if (tc.cfg.p2p_precision == EXAFMM_PREC_FP64) {
    auto *k = cycle != 0.0 ? k_p2p64<true> : k_p2p64<false>;
    hipLaunchKernelGGL(k, dim3(T.nleaves), dim3(kP2PWaves * kWave), 0, s, T.leaves.p, T.misc.p + 17, T.cbeg.p,
                       T.ccnt.p, T.xs.p, L.p2p_beg.p, L.p2p_cnt.p, L.p2p.p, S.cbeg.p, S.ccnt.p, S.xs.p, cycle,
                       tc.bodies, list_flags);
  } else {
    auto *k = tc.cfg.p2p_precision == EXAFMM_PREC_FP32_NEWTON ? k_p2p32<true> : k_p2p32<false>;
    hipLaunchKernelGGL(k, dim3(ceil_div(T.nleaves, kP2PWaves)), dim3(kP2PWaves * kWave), 0, s, T.leaves.p,
                       T.misc.p + 17, T.cbeg.p, T.ccnt.p, T.cx.p, T.xq.p, L.p2p_beg.p, L.p2p_cnt.p, L.p2p.p,
                       S.cbeg.p, S.ccnt.p, S.xs.p, cycle, int(&tc == &sc), tc.bodies, list_flags);
  }
  XF_LAUNCH();
}

// ---------------------------------------------------------------- direct sum
// FP64 direct sum.  Lanes take sources, targets are wave-uniform in blocks
// of kDirectTC, so each loaded source serves kDirectTC interactions and the
// per-lane sums meet across the lanes once per wave.  The sources are cut
// into shares; the four waves of a workgroup take four target blocks against
// the same share (its lines then come from L2 once), or, with fewer than
// four blocks, quarters of the share.  Each (share, target) partial is
// stored and k_direct_sum adds a target's partials in a fixed order.  FP64
// VALU bound.  1,000 targets x 2^20 sources: 0.92 ms; 2.83 ms with a workgroup
// per target (every target streaming all sources, a divide and a root each).
constexpr int kDirectTC = 8;
constexpr int kDirectWaves = 4;
constexpr int kDirectGroups = 2048;  // workgroups aimed at: eight per CU

// Sums of targets t0 .. t0 + tc - 1 over the sources first + lane, + stride, ...
// below s1: component lane % (64 / TC) of target lane / (64 / TC).
template <int TC>
__device__ __attribute__((always_inline)) inline double direct_block(const exafmm_body *__restrict__ t, int tc,
                                                                     const exafmm_body *__restrict__ s, int64_t s0,
                                                                     int64_t s1, int64_t stride, int lane) {
  double xt[TC], yt[TC], zt[TC], ap[TC], ax[TC], ay[TC], az[TC];
#pragma unroll
  for (int i = 0; i < TC; i++) {
    const exafmm_body *b = t + min(i, tc - 1);
    xt[i] = b->X[0];
    yt[i] = b->X[1];
    zt[i] = b->X[2];
    ap[i] = ax[i] = ay[i] = az[i] = 0.0;
  }
  for (int64_t j = s0 + lane; j < s1; j += stride) {
    const double sx = s[j].X[0], sy = s[j].X[1], sz = s[j].X[2], q = s[j].q;
#pragma unroll
    for (int i = 0; i < TC; i++)
      p2p64_pair(xt[i] - sx, yt[i] - sy, zt[i] - sz, q, ap[i], ax[i], ay[i], az[i]);
  }
  return p2p_lane_total<TC>(ap, ax, ay, az, lane);
}

__global__ void __launch_bounds__(kDirectWaves *kWave) k_direct(const exafmm_body *__restrict__ t, int64_t nt,
                                                                const exafmm_body *__restrict__ s, int64_t ns,
                                                                int wt, double *__restrict__ part) {
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int ws = kDirectWaves / wt;  // waves that share a target block
  const int64_t t0 = (int64_t(blockIdx.x) * wt + w % wt) * kDirectTC;
  if (t0 >= nt) return;
  const int64_t share = int64_t(blockIdx.y) * ws + w / wt, shares = int64_t(gridDim.y) * ws;
  const int64_t s0 = share * ns / shares, s1 = (share + 1) * ns / shares;
  const int tc = int(min(int64_t(kDirectTC), nt - t0));
  constexpr int kLow = kWave / kDirectTC;
  const int i = lane / kLow, comp = lane % kLow;
  const double v = direct_block<kDirectTC>(t + t0, tc, s, s0, s1, kWave, lane);
  if (comp < 4 && i < tc) part[(share * nt + t0 + i) * 4 + comp] = v;
}

// Few sources: a workgroup of 16 waves takes four targets over all of them
// and adds its waves' sums itself, in one launch.  Up to kDirectOneMax
// sources a wave has few enough rounds that the launch saved is worth more
// than the even split: 1,000 x 8,000 in 23 us, 32 in two launches (and 2,000 x
// 8,000 in 32 against 37); the gap closes beyond.  Few targets leave most CUs idle
// here and cross earlier: 1 to 100 x 8,192 in 21 - 22 us, 19 - 20 in two launches
// (8,193 sources); the rule looks at the sources alone (a workgroup per target:
// 23 - 24).
//
// Sixteen waves shorten a workgroup's chain of rounds where the workgroups do not
// fill the device.  Up to kDirectFewSources sources there are no rounds to share,
// and from kDirectManyTargets targets on the device is full of workgroups anyway:
// four waves, which start and meet sooner.  Sixteen / four waves, us: 200 x 264 15.0 /
// 14.8, 1,000 x 2,000 16.9 / 17.7, 2,000 x 8,192 33.9 / 33.9, 10,000 x 2,000 49.9 / 34.8,
// 100,000 x 264 192 / 72, 100,000 x 8,192 859 / 732.
constexpr int kDirectOneTC = 4;
constexpr int64_t kDirectOneMax = 8192, kDirectFewSources = 512, kDirectManyTargets = 2000;
template <int W>
__global__ void __launch_bounds__(W *kWave) k_direct_one(exafmm_body *__restrict__ t, int64_t nt,
                                                         const exafmm_body *__restrict__ s, int64_t ns) {
  constexpr int kLow = kWave / kDirectOneTC;
  __shared__ double red[W][kDirectOneTC * 4];
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t t0 = int64_t(blockIdx.x) * kDirectOneTC;
  const int tc = int(min(int64_t(kDirectOneTC), nt - t0));
  const double v = direct_block<kDirectOneTC>(t + t0, tc, s, w * kWave, ns, W * kWave, lane);
  if (lane % kLow < 4) red[w][lane / kLow * 4 + lane % kLow] = v;
  __syncthreads();
  const int i = threadIdx.x / 4, comp = threadIdx.x % 4;
  if (i >= tc) return;
  // the waves' sums pairwise: one after the other their roundings add up (500 to
  // 8,192 sources of one sign: p off by 1.0 - 1.2e-16 rms, 0.7 this way)
  double ws[W];
#pragma unroll
  for (int k = 0; k < W; k++) ws[k] = red[k][threadIdx.x];
#pragma unroll
  for (int o = W / 2; o > 0; o /= 2)
#pragma unroll
    for (int k = 0; k < o; k++) ws[k] += ws[k + o];
  const double sum = ws[0];
  if (comp == 0)
    t[t0 + i].p += sum;
  else
    t[t0 + i].F[comp - 1] -= sum;
}

// One wave per target: lane (h, comp) = (lane / 4, lane % 4) adds the shares
// h, h + 16, ..., then the 16 lanes of a component are added by halving.
__global__ void __launch_bounds__(256) k_direct_sum(exafmm_body *__restrict__ t, int64_t nt, int64_t shares,
                                                    const double *__restrict__ part) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t i = int64_t(blockIdx.x) * (256 / kWave) + threadIdx.x / kWave;
  if (i >= nt) return;  // whole wave
  const int comp = lane & 3;
  double v = 0.0;
  for (int64_t h = lane >> 2; h < shares; h += kWave / 4) v += part[(h * nt + i) * 4 + comp];
#pragma unroll
  for (int m = 4; m < kWave; m <<= 1) v += __shfl_xor(v, m);
  if (lane >= 4) return;
  if (comp == 0)
    t[i].p += v;
  else
    t[i].F[comp - 1] -= v;
}

void direct_sum(Ctx &c, exafmm_body *t, int64_t nt, const exafmm_body *s, int64_t ns) {
  if (nt <= 0 || ns <= 0) return;
  if (ns <= kDirectOneMax) {
    const int waves = ns <= kDirectFewSources || nt >= kDirectManyTargets ? 4 : 16;
    hipLaunchKernelGGL(waves == 4 ? k_direct_one<4> : k_direct_one<16>, dim3(ceil_div(nt, kDirectOneTC)),
                       dim3(waves * kWave), 0, c.s0, t, nt, s, ns);
    XF_LAUNCH();
    return;
  }
  const int64_t blocks = (nt + kDirectTC - 1) / kDirectTC;
  const int wt = blocks >= 4 ? 4 : blocks >= 2 ? 2 : 1;
  const int64_t groups = (blocks + wt - 1) / wt;
  // shares of at least two source rounds per wave, about kDirectGroups workgroups in all
  const int ws = kDirectWaves / wt;
  const int64_t gy = std::max<int64_t>(
      1, std::min<int64_t>((kDirectGroups + groups - 1) / groups, ns / (int64_t(2) * kWave * ws)));
  const int64_t shares = gy * ws;
  c.direct_part.ensure(size_t(shares) * nt * 4);
  hipLaunchKernelGGL(k_direct, dim3(unsigned(groups), unsigned(gy)), dim3(kDirectWaves * kWave), 0, c.s0, t, nt, s, ns,
                     wt, c.direct_part.p);
  XF_LAUNCH();
  hipLaunchKernelGGL(k_direct_sum, dim3(ceil_div(nt, 256 / kWave)), dim3(256), 0, c.s0, t, nt, shares,
                     c.direct_part.p);
  XF_LAUNCH();
}

}  // namespace xf
