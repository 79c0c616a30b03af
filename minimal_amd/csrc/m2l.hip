// m2l.hip -- multipole-to-local translation.
//
// Reference: M2L 3d/kernel.h:233-260 with singular harmonics 3d/kernel.h:83-116,
// evaluated over each target's M2L list (3d/traverse_lazy.h:46-56).
//
// Two paths:
//  * exact  (m2l_precision = FP64): the reference's sum per pair on the FP64
//    singular harmonics of the true offset.  Parity path.
//  * fast   (FP32 / BF16X3): pairs grouped by translation key; every key's
//    radius-scaled P^2 x P^2 real operator is applied to tiles of targets
//    with MFMA (m2l_mfma.hip).
// Truncation: "reference" keeps the terms the reference evaluates (its
// harmonic table is zero above degree P-1, so j+n <= P-1); "full" keeps
// every j+n <= 2P-2.
#include <algorithm>
#include <cmath>
#include <mutex>

#include "fmm_internal.h"
#include "fmm_ops.h"

namespace xf {
using namespace xfd;

// The per-pair sum as a convolution.  With the signed extensions
// X_n^{-m} = (-1)^m conj(X_n^m) of the multipoles and of the singular
// harmonics, the reference's sign cases (3d/kernel.h:241-255) collapse to
//   L_j^k = (-1)^(j+k) sum_{n, |m| <= n} M_n^m I_{j+n}^{m-k}(d),
// and with d in units of the target's radius Rc the scaled expansions enter
// directly: L~_j^k = (-1)^(j+k) sum M~_n^m (Rs/Rc)^n I_{j+n}^{m-k}(d/Rc), no
// powers of the radii themselves.
//
// A workgroup takes one target cell and one share of its list, kBatch pairs
// at a time: its threads fill the pairs' signed harmonics and multipoles in
// LDS (one thread per pair and column), then each of its four waves sums its
// own range of the outputs (j,k), several pairs side by side.  A lane sums
// two outputs of consecutive order, (j,k) and (j,k+1): the harmonic that the
// first meets at m is the second's at m + 1, so each term costs one harmonic
// and one multipole read for two outputs.  With the reference's truncation
// an output of degree j has (P-j)^2 terms, so the ranges group outputs of
// like degree (m2l64_plan): the low degrees, a handful of long sums, run many
// pairs at once.  The bound is the LDS reads (two 16-byte reads per eight
// FP64 FMAs) and, for short lists, the chain of the harmonics.
// WIDE (trees of very different size): the powers (Rs/Rc)^n and the harmonics of
// d/Rc leave the range of double while their products stay small.  A pair whose
// source is the larger cell then takes d in units of Rs:
//   L~_j^k = (-1)^(j+k) (Rc/Rs)^(j+1) sum M~_n^m I_{j+n}^{m-k}(d/Rs),
// all factors at most 1; the sum of each pair is scaled by (Rc/Rs)^j as it is
// added.
// 118,396 pairs (P = 10, reference truncation): 218 us; the periodic top
// levels of 131,072 bodies: 154 us.  (A wave per cell, one pair after
// another, a lane per output with the sign cases and powers in the inner
// loop: 3,382 and 2,469 us.)
constexpr int kM2L64Threads = 256, kM2L64Waves = kM2L64Threads / kWave;
constexpr int kM2L64Lds = 40 * 1024;  // three to four workgroups per CU
// Largest ratio of a source cell's radius to a target cell's without WIDE: its
// 15th power is 2^480, and harmonics of degree 30 of a distance as many times
// the target's radius are above 2^-1000.
constexpr double kM2L64Wide = 4294967296.0;

struct M2L64Plan {
  int batch;                 // pairs in LDS at a time
  int jb[kM2L64Waves + 1];   // wave w sums degrees jb[w] .. jb[w+1] - 1
};

// A pair's LDS row of the degrees below p, both signs: an odd number of
// 16-byte elements, so that lanes reading the same element of different
// pairs fall into different banks.
__host__ __device__ constexpr int m2l64_stride(int p) { return (p * p) | 1; }

// Lanes per pair of the degrees below j: degree j has j + 1 outputs, two
// consecutive orders k per lane.
__host__ __device__ inline int m2l64_slots(int j) { return ((j + 1) * (j + 1)) / 4; }

// Degree ranges of the waves and the pairs per batch: the split whose
// slowest wave takes the fewest steps per pair, where a range of `len`
// lanes runs 64 / len pairs side by side, takes as many steps for them as
// its lowest degree has terms, and a batch also pays for its harmonics
// (about as long as kHarmonicSteps terms).
static M2L64Plan m2l64_search(int P, int fillP) {
  constexpr double kHarmonicSteps = 40;
  const int per = int(sizeof(double2)) * (m2l64_stride(fillP) + m2l64_stride(P));
  const int bmax = std::max(1, std::min(kM2L64Lds / per, kM2L64Threads / fillP));
  auto cost = [&](int j0, int j1, int batch) {
    if (j0 >= j1) return 0;
    const int len = m2l64_slots(j1) - m2l64_slots(j0), nn = std::min(P, fillP - j0);
    if (len > kWave) return 1 << 30;
    const int side = kWave / len;
    return nn * nn * ((batch + side - 1) / side);
  };
  M2L64Plan best{};
  double least = 1e300;
  for (int n = 1; n <= bmax; n++)
    for (int a = 0; a <= P; a++)
      for (int b = a; b <= P; b++)
        for (int c = b; c <= P; c++) {
          const int w = std::max(std::max(cost(0, a, n), cost(a, b, n)), std::max(cost(b, c, n), cost(c, P, n)));
          if ((w + kHarmonicSteps) / n < least) {
            least = (w + kHarmonicSteps) / n;
            best = M2L64Plan{n, {0, a, b, c, P}};
          }
        }
  return best;
}

// The search runs once per order and truncation.
static M2L64Plan m2l64_plan(int P, int fillP) {
  static std::mutex mu;
  static M2L64Plan plans[kMaxP + 1][2] = {};
  std::lock_guard<std::mutex> lk(mu);
  M2L64Plan &pl = plans[P][fillP > P];
  if (!pl.batch) pl = m2l64_search(P, fillP);
  return pl;
}

// grid: (cells, shares of a cell's list).  part: partial locals [share][cell]
// [P^2], added in share order by k_m2l_fp64_sum; null with one share (the
// sums go straight into L).
template <int P, bool WIDE>
__global__ void __launch_bounds__(kM2L64Threads)
    k_m2l_fp64(int fillP, int ncells, M2L64Plan pl, const double4 *__restrict__ cx,
               const double4 *__restrict__ scx, const int *__restrict__ beg, const int *__restrict__ cnt,
               const int2 *__restrict__ list, const double *__restrict__ M, double *__restrict__ L,
               double *__restrict__ part, double cycle) {
  extern __shared__ double2 sm[];
  constexpr int PP = P * P;
  constexpr int MS = m2l64_stride(P);
  const int c = blockIdx.x, IS = m2l64_stride(fillP);
  const int n_all = cnt[c];
  const int p0 = int(int64_t(n_all) * blockIdx.y / gridDim.y), p1 = int(int64_t(n_all) * (blockIdx.y + 1) / gridDim.y);
  const double4 Xc = cx[c];
  if (!part && n_all == 0) return;
  double *out = part ? part + (int64_t(blockIdx.y) * ncells + c) * PP : L + int64_t(c) * PP;
  double2 *Is = sm;                      // [batch][IS], element (l, o) at l^2 + l + o
  double2 *Ms = sm + pl.batch * IS;      // [batch][MS]
  __shared__ double ratio[WIDE ? kM2L64Threads : 1];  // per pair of the batch: min(1, Rc/Rs)
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
  // this wave's outputs (a range of degrees), and this lane's output and pair slot
  int j0 = 0, j1 = 0;
#pragma unroll
  for (int k = 0; k < kM2L64Waves; k++)
    if (k == w) {
      j0 = pl.jb[k];
      j1 = pl.jb[k + 1];
    }
  const int len = m2l64_slots(j1) - m2l64_slots(j0);     // lanes per pair
  const int side = len > 0 ? kWave / len : 1;            // pairs side by side
  const int slot = len > 0 ? lane / len : 0;
  int j = j0, k = m2l64_slots(j0) + (len > 0 ? lane % len : 0);  // this lane's outputs: (j, k), (j, k + 1)
  while (j + 1 < j1 && m2l64_slots(j + 1) <= k) j++;
  k = 2 * (k - m2l64_slots(j));
  const double inv = Xc.w > 0.0 ? 1.0 / Xc.w : 0.0;
  const int b0 = beg[c];
  // this thread's multipole coefficient: pair slot bm, real-form index im = (nm, mm, imag)
  constexpr int kPairs = kM2L64Threads / PP;
  const int bm = tid / PP, im = tid % PP;
  int nm = 0;
  while ((nm + 1) * (nm + 1) <= im) nm++;
  const int rem = im - nm * nm, mm = (rem + 1) / 2;
  const bool imag = rem > 0 && rem % 2 == 0;
  const double msign = sgn(mm);
  double r0 = 0.0, i0 = 0.0, r1 = 0.0, i1 = 0.0;
  if (Xc.w > 0.0) {  // a cell of radius 0 holds its bodies at its centre: L~ is 0
    for (int q0 = p0; q0 < p1; q0 += pl.batch) {
      const int nb = min(pl.batch, p1 - q0);
      __syncthreads();
      // one thread per (pair, column m): I_l^m for l = m .. fillP - 1, both signs
      for (int t = tid; t < nb * fillP; t += kM2L64Threads) {
        const int b = t / fillP, m = t - b * fillP;
        const int2 e = list[b0 + q0 + b];
        const int img = e.x & 31;
        const double4 Xs = scx[e.x >> 5];
        // 3dp/kernel.h:200: dX = Xi - Xj - iX * cycle
        const double unit = WIDE && Xs.w > Xc.w ? 1.0 / Xs.w : inv;
        const double dx = (Xc.x - Xs.x - ((img % 3) - 1) * cycle) * unit;
        const double dy = (Xc.y - Xs.y - (((img / 3) % 3) - 1) * cycle) * unit;
        const double dz = (Xc.z - Xs.z - ((img / 9) - 1) * cycle) * unit;
        const double r2 = dx * dx + dy * dy + dz * dz;
        const double ir2 = 1.0 / r2;
        double ar = sqrt(ir2), ai = 0.0;
        if (WIDE && Xs.w > Xc.w) ar *= Xc.w * unit;
        if (WIDE && m == 0) ratio[b] = Xs.w > Xc.w ? Xc.w * unit : 1.0;
        for (int k = 1; k <= m; k++) {
          const double f = double(2 * k - 1) * ir2;
          const double tr = (ar * dx - ai * dy) * f, ti = (ar * dy + ai * dx) * f;
          ar = tr;
          ai = ti;
        }
        double2 *Ib = Is + b * IS;
        const double sg = sgn(m), dzi = dz * ir2;
        double br = 0.0, bi = 0.0;
        double c2 = double(2 * m + 1), d = 0.0;  // 2l + 1 and (l + m)(l - m): exact
        for (int l = m; l < fillP; l++) {
          Ib[l * l + l + m] = make_double2(ar, ai);
          if (m) Ib[l * l + l - m] = make_double2(sg * ar, -sg * ai);
          const double cz = c2 * dzi, di = d * ir2;
          const double nr = -fma(cz, ar, di * br), ni = -fma(cz, ai, di * bi);
          br = ar;
          bi = ai;
          ar = nr;
          ai = ni;
          d += c2;
          c2 += 2.0;
        }
      }
      // this thread's multipole coefficient of pairs bm, bm + kPairs, ...:
      // M~_n^m (Rs/Rc)^n, both signs
      if (bm < kPairs)
        for (int b = bm; b < nb; b += kPairs) {
          const int src = list[b0 + q0 + b].x >> 5;
          const double Rs = scx[src].w, x = WIDE && Rs > Xc.w ? 1.0 : Rs * inv, x2 = x * x, x4 = x2 * x2;
          double v = M[int64_t(src) * PP + im];
          v *= (nm & 1) ? x : 1.0;
          v *= (nm & 2) ? x2 : 1.0;
          v *= (nm & 4) ? x4 : 1.0;
          v *= (nm & 8) ? x4 * x4 : 1.0;
          double2 *Mb = Ms + b * MS + nm * nm + nm;
          if (mm == 0) {
            Mb[0] = make_double2(v, 0.0);
          } else if (!imag) {
            Mb[mm].x = v;
            Mb[-mm].x = msign * v;
          } else {
            Mb[mm].y = v;
            Mb[-mm].y = -msign * v;
          }
        }
      __syncthreads();
      if (len <= 0 || slot >= side) continue;
      const int nmax = min(P, fillP - j);
      for (int b = slot; b < nb; b += side) {
        const double2 *Ib = Is + b * IS;
        const double before[4] = {r0, i0, r1, i1};
        if (WIDE) r0 = i0 = r1 = i1 = 0.0;
#pragma unroll
        for (int n = 0; n < P; n++) {
          if (n >= nmax) break;
          const int i = (j + n) * (j + n + 1) - k - n;
          const double2 *Ip = Ib + i, *Mp = Ms + b * MS + n * n;
          double2 y1 = Ib[max(i - 1, 0)];  // (no second output at k = j: its sum is dropped)
#pragma unroll
          for (int m = 0; m <= 2 * n; m++) {
            const double2 a = Mp[m], y0 = Ip[m];
            r0 = fma(a.x, y0.x, r0);
            i0 = fma(a.x, y0.y, i0);
            r1 = fma(a.x, y1.x, r1);
            i1 = fma(a.x, y1.y, i1);
            r0 = fma(-a.y, y0.y, r0);
            i0 = fma(a.y, y0.x, i0);
            r1 = fma(-a.y, y1.y, r1);
            i1 = fma(a.y, y1.x, i1);
            y1 = y0;
          }
        }
        if (WIDE) {
          double f = 1.0;
          for (int q = 0; q < j; q++) f *= ratio[b];
          r0 = fma(r0, f, before[0]);
          i0 = fma(i0, f, before[1]);
          r1 = fma(r1, f, before[2]);
          i1 = fma(i1, f, before[3]);
        }
      }
    }
  }
  // the pair slots of an output, added in order
  __syncthreads();
  double2 *red = sm + w * 2 * kWave;
  red[2 * lane] = make_double2(r0, i0);
  red[2 * lane + 1] = make_double2(r1, i1);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  if (lane >= len) return;
#pragma unroll
  for (int h = 0; h < 2; h++, k++) {
    if (k > j) break;
    double sr = 0.0, si = 0.0;
    for (int q = 0; q < side; q++) {
      sr += red[2 * (q * len + lane) + h].x;
      si += red[2 * (q * len + lane) + h].y;
    }
    const double s = sgn(j + k);
    if (part) {
      out[rf(j, k, 0)] = sr * s;
      if (k > 0) out[rf(j, k, 1)] = si * s;
    } else {
      out[rf(j, k, 0)] += sr * s;
      if (k > 0) out[rf(j, k, 1)] += si * s;
    }
  }
}

// Adds the list shares of k_m2l_fp64 into the locals, in share order.
__global__ void __launch_bounds__(256) k_m2l_fp64_sum(int64_t n, int shares, const double *__restrict__ part,
                                                      double *__restrict__ L) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  double s = 0.0;
  for (int k = 0; k < shares; k++) s += part[int64_t(k) * n + i];
  L[i] += s;
}

// M2L per pair in FP64 for cells 0 .. ncells - 1 of the target tree.  Lists
// differ in length several times over (hundreds of image translations per
// cell at the top of a periodic tree), and a batch of pairs is a long chain
// (list, cell, harmonics, sums), so below 8,192 cells the lists are shared
// out over up to 16 workgroups each -- as many as the mean list has batches: a tree
// of a few cells with short lists is not worth the second launch (60 problems of
// 60 bodies each, re-evaluated by a graph: 1,822 -> 1,440 us; most have no pairs, and
// m2l_apply leaves before this).
static void m2l_fp64(Ctx &tc, const Ctx &sc, int ncells, double cycle) {
  join_upward(tc);
  const int P = tc.P, PP = P * P;
  const int fillP = tc.cfg.m2l_truncation == EXAFMM_M2L_FULL ? 2 * P - 1 : P;
  const M2L64Plan pl = m2l64_plan(P, fillP);
  const size_t lds = std::max(sizeof(double2) * size_t(pl.batch) * (m2l64_stride(fillP) + m2l64_stride(P)),
                              sizeof(double2) * 2 * kM2L64Threads);  // (the last sums)
  const int64_t mean = ceil_div(tc.lists.nm2l, int64_t(pl.batch) * std::max(ncells, 1));
  const int shares = int(std::max<int64_t>(1, std::min<int64_t>({16, 8192 / std::max(ncells, 1), mean})));
  double *part = nullptr;
  if (shares > 1) {
    tc.m2l_part64.ensure(size_t(shares) * ncells * PP);
    part = tc.m2l_part64.p;
  }
  // (one tree's cells differ by 2^21 at most)
  const bool wide = sc.t.R0 > kM2L64Wide * std::ldexp(tc.t.R0, -tc.t.depth);
  switch (P) {
#define XF_M2L64_CASE(n)                                                                                           \
  case n:                                                                                                          \
    hipLaunchKernelGGL((wide ? k_m2l_fp64<n, true> : k_m2l_fp64<n, false>), dim3(ncells, shares), dim3(kM2L64Threads), lds, tc.s0, fillP, ncells, pl,    \
                       tc.t.cx.p, sc.t.cx.p, tc.lists.m2l_beg.p, tc.lists.m2l_cnt.p, tc.lists.m2l.p, sc.M.p, tc.L.p, \
                       part, cycle);                                                                               \
    break;
    XF_M2L64_CASE(2)
    XF_M2L64_CASE(3)
    XF_M2L64_CASE(4)
    XF_M2L64_CASE(5)
    XF_M2L64_CASE(6)
    XF_M2L64_CASE(7)
    XF_M2L64_CASE(8)
    XF_M2L64_CASE(9)
    XF_M2L64_CASE(10)
    XF_M2L64_CASE(11)
    XF_M2L64_CASE(12)
    XF_M2L64_CASE(13)
    XF_M2L64_CASE(14)
    XF_M2L64_CASE(15)
    XF_M2L64_CASE(16)
#undef XF_M2L64_CASE
    default: fail(EXAFMM_ERR_UNSUPPORTED, "expansion order");
  }
  XF_LAUNCH();
  if (shares > 1) {
    const int64_t n = int64_t(ncells) * PP;
    hipLaunchKernelGGL(k_m2l_fp64_sum, dim3(ceil_div(n, 256)), dim3(256), 0, tc.s0, n, shares, part, tc.L.p);
    XF_LAUNCH();
  }
}

void m2l_fast(Ctx &tc, const Ctx &sc);  // m2l_mfma.hip

// Levels whose M2L runs per pair in FP64 beside the keyed GEMM.  Periodic:
// levels 0..2, whose cells collect hundreds of image translations that add
// up to a small difference of large terms (the neutral periodic potential),
// where FP32 accumulation would leave an offset of ~1e-5 relative.
int m2l_fp64_levels(const Ctx &c) { return c.cfg.images > 0 ? std::min(3, c.t.depth + 1) : 0; }

void m2l_apply(Ctx &tc, const Ctx &sc) {
  Tree &t = tc.t;
  const double cyc = tc.cfg.images > 0 ? tc.cfg.cycle : 0.0;
  if (tc.lists.nm2l == 0) {  // the locals are zero already
    join_upward(tc);
    return;
  }
  if (tc.cfg.m2l_precision != EXAFMM_PREC_FP64 && tc.lists.nkeys > 0) {
    const int lf = m2l_fp64_levels(tc);
    if (lf > 0) m2l_fp64(tc, sc, t.lstart[lf], cyc);  // cells of levels < lf come first in breadth-first order
    m2l_fast(tc, sc);
    return;
  }
  m2l_fp64(tc, sc, int(t.ncells), cyc);
}

}  // namespace xf
