// expansions.hip -- P2M, M2M (upward), L2L, L2P (downward).
//
// Reference operators: P2M 3d/kernel.h:187-202, M2M :204-231, L2L :262-291,
// L2P :293-322; passes 3d/traverse_lazy.h:7-24 (upward) and :65-80
// (downward).
//
// Storage: every cell's expansions are kept in radius-scaled real form,
//   M~[rf(n,m,.)] = (Re, Im) M_n^m / R^n,   L~[rf(j,k,.)] = (Re, Im) L_j^k R^(j+1),
// P^2 doubles per cell (the imaginary parts of the m = 0 coefficients are
// zero for real charges and are not stored).  In this form the child <-> parent
// shifts do not depend on the level: M2M and L2L are one fixed P^2 x P^2 FP64
// matrix per octant, generated once from the reference's shift formulas
// (m2m_coef / l2l_coef applied to unit vectors) and applied as batched
// matrix-vector products.  Harmonics come from the trig-free Cartesian
// recurrences of fmm_internal.h (same functions and normalisation as the
// reference's spherical evaluation).  P2M, M2M and L2L run in FP64; L2P
// evaluates in FP32 (FP64 in parity mode) and adds into FP64 body
// accumulators, with the force from Cartesian ladder identities of the
// solid harmonics (finite at r = 0 and on the z axis, where the reference's
// spherical form divides by zero, 3d/kernel.h:31-40).
#include <type_traits>

#include "fmm_internal.h"
#include "fmm_ops.h"

namespace xf {
using namespace xfd;

// 1/i for i <= 1024 (the harmonic recurrences need 1/(2m) and
// 1/((n+m)(n-m)), n, m < 16): correctly rounded at compile time, so a table
// read replaces an FP64 division in the kernels.
struct InvTable {
  double v[1025];
  constexpr InvTable() : v() {
    for (int i = 1; i <= 1024; i++) v[i] = 1.0 / i;
  }
};
static __constant__ InvTable kInv = InvTable();

// f(integral_constant<P>) for the order at run time: kernels whose loops over
// the degrees unroll are instantiated per order.
#define XF_ORDER_CASE(f, n)                       \
  case n:                                         \
    return f(std::integral_constant<int, n>());
#define XF_ORDER_CASES(f)                                                                                 \
  XF_ORDER_CASE(f, 2) XF_ORDER_CASE(f, 3) XF_ORDER_CASE(f, 4) XF_ORDER_CASE(f, 5) XF_ORDER_CASE(f, 6)     \
  XF_ORDER_CASE(f, 7) XF_ORDER_CASE(f, 8) XF_ORDER_CASE(f, 9) XF_ORDER_CASE(f, 10) XF_ORDER_CASE(f, 11)   \
  XF_ORDER_CASE(f, 12) XF_ORDER_CASE(f, 13) XF_ORDER_CASE(f, 14) XF_ORDER_CASE(f, 15) XF_ORDER_CASE(f, 16)
template <class F>
static void by_order(int P, F &&f) {
  switch (P) {
    XF_ORDER_CASES(f)
    default:
      fail(EXAFMM_ERR_UNSUPPORTED, "expansion order");
  }
}

// ---------------------------------------------------------------- P2M
// M~_n^m = sum_b q_b conj(Y_n^m(u_b)), u = (x_b - X_c)/R (3d/kernel.h:193
// evaluates Y at -beta, i.e. the conjugate).  One wave per leaf.  A column m
// holds P - m degrees, so a lane takes columns j and P - 1 - j, P + 1 terms
// whatever j: J = ceil(P / 2) lanes serve a body and G = 64 / J bodies run
// side by side, with no lane waiting for a longer column.  A term is
//   Y_n = a z Y_{n-1} + s r^2 Y_{n-2},  s = -1/((n+m)(n-m)),  a = (2n-1) s
// (n = m + 1: a = -1, s = 0), the factors in registers; where the second
// column begins they are 0 and its Y_m^m is added.  The G bodies' sums meet
// in LDS, in body order.  FP64 VALU bound.  (A lane per column and four bodies
// side by side waited for the longest column: the step of 2^20 uniform bodies,
// order 10, 3.13 -> 3.04 ms with this, 1.5M clustered, order 12, 8.72 -> 8.56 ms.)
constexpr int kP2MWaves = 4;

template <int P>
struct P2MShape {
  static constexpr int J = (P + 1) / 2, G = kWave / J, T = P + 1;
  static constexpr int S = kWave + J;  // LDS row: lanes reading (term, column) pairs in turn hit distinct banks
  using Lds = double[kP2MWaves][T * S];
};

template <int P>
__device__ __attribute__((always_inline)) inline void p2m_body(int bx, const int *__restrict__ leaves,
                                                               const int *__restrict__ nleaves,
                                                               const int *__restrict__ cbeg,
                                                               const int *__restrict__ ccnt,
                                                               const double4 *__restrict__ cx,
                                                               const double4 *__restrict__ xs,
                                                               double *__restrict__ M,
                                                               typename P2MShape<P>::Lds &red) {
  using Sh = P2MShape<P>;
  constexpr int J = Sh::J, G = Sh::G, T = Sh::T, S = Sh::S;
  const int lane = threadIdx.x % kWave, w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int li = bx * kP2MWaves + w;
  if (li >= *nleaves) return;  // whole wave; wave-level syncs only below
  const int c = leaves[li];
  const int beg = cbeg[c], cnt = ccnt[c];
  const double4 C = cx[c];
  const double invR = C.w > 0.0 ? 1.0 / C.w : 0.0;  // R = 0: every body at the centre
  const int j = lane % J, g = lane / J, mb = P - 1 - j;
  const int tb = P - j;  // first term of the second column (none if it is the first: P odd, j = J - 1)
  double ca = 1.0, cb = mb > j ? 1.0 : 0.0;  // 1/(2^m m!)
  for (int k = 1; k <= j; k++) ca *= kInv.v[2 * k];
  for (int k = 1; k <= mb; k++) cb *= kInv.v[2 * k];
  double fa[T], fs[T], ar[T], ai[T];
#pragma unroll
  for (int t = 0; t < T; t++) {
    const int m = t < tb ? j : mb, n = t < tb ? j + t : t - 1;
    const bool in = n > m && !(t >= tb && mb == j);
    const double s = in ? -kInv.v[(n + m) * (n - m)] : 0.0;
    fa[t] = in ? (n == m + 1 ? -1.0 : double(2 * n - 1) * s) : 0.0;
    fs[t] = n == m + 1 ? 0.0 : s;
    ar[t] = ai[t] = 0.0;
  }
  for (int b0 = 0; b0 < cnt; b0 += G) {
    const int b = b0 + g;
    const bool valid = g < G && b < cnt;
    const double4 B = xs[beg + min(b, cnt - 1)];
    const double q = valid ? B.w : 0.0;
    const double x = (B.x - C.x) * invR, y = -(B.y - C.y) * invR, z = (B.z - C.z) * invR;  // conjugate
    const double r2 = x * x + y * y + z * z;
    // (x + iy)^j, then (x + iy)^(P-1-j) = (x + iy)^j ((x + iy)^2)^(J-1-j) [(x + iy) if P is even]
    double pr = 1.0, pi = 0.0;
#pragma unroll
    for (int k = 1; k < J; k++)
      if (k <= j) {
        const double tr = pr * x - pi * y;
        pi = pr * y + pi * x;
        pr = tr;
      }
    double cr = pr * (q * ca), ci = pi * (q * ca);
    const double xr = x * x - y * y, xi = 2.0 * (x * y);
#pragma unroll
    for (int k = 1; k < J; k++)
      if (k <= J - 1 - j) {
        const double tr = pr * xr - pi * xi;
        pi = pr * xi + pi * xr;
        pr = tr;
      }
    if (P % 2 == 0) {
      const double tr = pr * x - pi * y;
      pi = pr * y + pi * x;
      pr = tr;
    }
    const double br = pr * (q * cb), bi = pi * (q * cb);
    double or_ = 0.0, oi = 0.0;  // the term before
    ar[0] += cr;
    ai[0] += ci;
#pragma unroll
    for (int t = 1; t < T; t++) {
      const double az = fa[t] * z, sr = fs[t] * r2;
      double nr = az * cr + sr * or_, ni = az * ci + sr * oi;
      if (t >= P - J + 1) {  // the second column may begin here
        const double sel = t == tb ? 1.0 : 0.0;
        nr += sel * br;
        ni += sel * bi;
      }
      or_ = cr;
      oi = ci;
      cr = nr;
      ci = ni;
      ar[t] += cr;
      ai[t] += ci;
    }
  }
  // sums over the body groups: output o = (term, column pair) by lane o % 64
  double *R = red[w];
  double *Mc = M + int64_t(c) * P * P;
#pragma unroll
  for (int part = 0; part < 2; part++) {
#pragma unroll
    for (int t = 0; t < T; t++) R[t * S + lane] = part ? ai[t] : ar[t];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int o = lane; o < T * J; o += kWave) {
      const int t = o / J, oj = o % J;
      const bool second = t >= P - oj;
      const int m = second ? P - 1 - oj : oj, n = second ? t - 1 : oj + t;
      double v = 0.0;
#pragma unroll
      for (int k = 0; k < G; k++) v += R[t * S + k * J + oj];
      if (!(second && m == oj) && (part == 0 || m > 0)) Mc[rf(n, m, part)] = v;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

template <int P>
__global__ void __launch_bounds__(kP2MWaves *kWave) k_p2m(const int *__restrict__ leaves,
                                                          const int *__restrict__ nleaves,
                                                          const int *__restrict__ cbeg, const int *__restrict__ ccnt,
                                                          const double4 *__restrict__ cx,
                                                          const double4 *__restrict__ xs, double *__restrict__ M) {
  __shared__ typename P2MShape<P>::Lds red;
  p2m_body<P>(blockIdx.x, leaves, nleaves, cbeg, ccnt, cx, xs, M, red);
}

// The problems of one order of a batch in one launch (block -> problem through start[]).
template <int P>
__global__ void __launch_bounds__(kP2MWaves *kWave) k_p2m_grouped(const GroupTree *__restrict__ g,
                                                                  const int *__restrict__ start, int nprob) {
  const int b = blockIdx.x, i = group_of(start, nprob, b);
  const GroupTree &t = g[i];
  __shared__ typename P2MShape<P>::Lds red;
  p2m_body<P>(b - start[i], t.leaves, t.nleaves, t.cbeg, t.ccnt, t.cx, t.xs, t.M, red);
}

// All problems of a small batch in one launch, each workgroup by its problem's
// order: the registers and LDS of the highest order leave room for few workgroups,
// and a launch less per order is worth more (grouped_record).
__global__ void __launch_bounds__(kP2MWaves *kWave) k_p2m_orders(const GroupTree *__restrict__ g,
                                                                 const int *__restrict__ start, int nprob) {
  __shared__ typename P2MShape<kMaxP>::Lds lds;  // every order's fits
  const int b = blockIdx.x, i = group_of(start, nprob, b);
  const GroupTree &t = g[i];
  auto run = [&](auto p) {
    p2m_body<p()>(b - start[i], t.leaves, t.nleaves, t.cbeg, t.ccnt, t.cx, t.xs, t.M,
                  reinterpret_cast<typename P2MShape<p()>::Lds &>(lds));
  };
  switch (t.P) {
    XF_ORDER_CASES(run)
  }
}


// ---------------------------------------------------------------- shift operators
// Column `col` of the scaled M2M (kind 0) or L2L (kind 1) operator of octant
// o, for a parent of radius 1 and a child of radius 1/2 centred at
// parent + (+/-1/2) per axis.  T[kind][o][col][row] (row fastest).
__global__ void k_shift_ops(int P, double *__restrict__ T) {
  const int PP = P * P, NT = P * (P + 1) / 2;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 2 * 8 * PP) return;
  const int kind = t / (8 * PP), o = (t / PP) % 8, col = t % PP;
  cpx<double> Y[kMaxP * (kMaxP + 1) / 2];
  double2 in[kMaxP * (kMaxP + 1) / 2];
  for (int i = 0; i < NT; i++) in[i] = make_double2(0, 0);
  int n = 0;
  while ((n + 1) * (n + 1) <= col) n++;
  const int rem = col - n * n, m = (rem + 1) / 2;
  const bool im = rem > 0 && rem % 2 == 0;
  const double ox = (o & 1) ? 0.5 : -0.5, oy = (o & 2) ? 0.5 : -0.5, oz = (o & 4) ? 0.5 : -0.5;
  double *out = T + ((int64_t(kind) * 8 + o) * PP + col) * PP;
  if (kind == 0) {
    // child scaled unit vector -> unscaled child M (radius 1/2), shift by Xp - Xc
    const double v = ldexp(1.0, -n);
    in[nms(n, m)] = im ? make_double2(0, v) : make_double2(v, 0);
    regular_all<double>(P, -ox, -oy, -oz, Y);
    for (int jk = 0; jk < NT; jk++) {
      int j, k;
      jk_of(jk, j, k);
      const double2 r = m2m_coef(j, k, in, Y);  // parent radius 1: scaled == unscaled
      out[rf(j, k, 0)] = r.x;
      if (k > 0) out[rf(j, k, 1)] = r.y;
    }
  } else {
    // parent scaled unit vector (radius 1: L = L~) -> child L, scaled by (1/2)^(j+1)
    in[nms(n, m)] = im ? make_double2(0, 1) : make_double2(1, 0);
    regular_all<double>(P, ox, oy, oz, Y);
    for (int jk = 0; jk < NT; jk++) {
      int j, k;
      jk_of(jk, j, k);
      const double2 r = l2l_coef(P, j, k, in, Y);
      const double s = ldexp(1.0, -(j + 1));
      out[rf(j, k, 0)] = r.x * s;
      if (k > 0) out[rf(j, k, 1)] = r.y * s;
    }
  }
}

void shift_ops(Ctx &c, hipStream_t s) {
  if (c.shift_P == c.P) return;
  const int PP = c.P * c.P;
  c.shift_T.ensure(size_t(2) * 8 * PP * PP);
  hipLaunchKernelGGL(k_shift_ops, dim3(ceil_div(2 * 8 * PP, 64)), dim3(64), 0, s, c.P, c.shift_T.p);
  XF_LAUNCH();
  c.shift_P = c.P;
}

// ---------------------------------------------------------------- M2M
// M2M and L2L as FP64 MFMA GEMMs over the cells of one level
// (v_mfma_f64_16x16x4_f64: A lane l = row l%16, k l/16; B lane l = column
// l%16, k l/16; D register i of lane l = row l/16 + 4i, column l%16).  A wave owns one
// 16-row tile of the operator and 16 parents; its operands stream straight
// from L2 into registers (no LDS round trip: every loaded value feeds a
// 16x16x4 product), four k-steps per batch so the loads of a batch overlap.
// Degree structure: an M2M row of degree j reads columns of degree <= j, an
// L2L row of degree j reads columns of degree >= j, so a row tile stops
// (starts) at the column bound of its last (first) row.
typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int kShiftWaves = 4;  // row tiles per workgroup
constexpr int kShiftBatch = 4;  // k-steps of 4 columns loaded together
// The batch graph's L2L runs alone on the device (after the GEMM), so it loads
// deeper: all 25 k-steps of order 10 in two rounds (M2M runs beside P2P, where
// more registers cost it more than the latency it saves)
constexpr int kL2LBatch = 13;

__device__ inline int degree_of(int row) {
  int j = 0;
  while ((j + 1) * (j + 1) <= row) j++;
  return j;
}

// Children of the parents p0 .. p0 + 15 of a level by octant: thread t < 128
// takes child t % 8 of parent p0 + t / 8 and files it under the octant its
// centre lies in relative to the parent's (strict >, 3d/build_tree.h:50-56);
// octants without a child keep -1.  Every load is issued at once (no walk
// over the children per octant).  `only` >= 0 keeps that octant alone, in
// row 0.  The caller fills chl with -1 and puts a barrier before and after.
__device__ inline void file_children(int tid, int p0, int lstart, int lcount, const int *__restrict__ cchild,
                                     const int *__restrict__ cnch, const double4 *__restrict__ cx, int only,
                                     int (*chl)[16]) {
  if (tid >= 128) return;
  const int q = tid >> 3, j = tid & 7;
  if (p0 + q >= lcount) return;
  const int p = lstart + p0 + q;
  const int nch = cnch[p], first = cchild[p];
  if (j >= nch) return;
  const double4 Cp = cx[p], Cc = cx[first + j];
  const int o = (Cc.x > Cp.x) + ((Cc.y > Cp.y) << 1) + ((Cc.z > Cp.z) << 2);
  if (only < 0)
    chl[o][q] = first + j;
  else if (o == only)
    chl[0][q] = first + j;
}

// M~_parent = sum over children of T_M2M[octant] M~_child (3d/kernel.h:206).
// grid: (parent tiles of 16, row tiles of 16).  The eight waves of a block
// take one octant each (K = that octant's columns), so a small level's
// launch waits for one octant's chain of loads, not eight; the eight
// partial tiles are then added in LDS in octant order.
constexpr int kM2MWaves = 8;
__device__ __attribute__((always_inline)) inline void m2m_body(int bx, int by, int P, int lstart, int lcount,
                                const int *__restrict__ cchild,
                                const int *__restrict__ cnch,
                                const double4 *__restrict__ cx,
                                const double *__restrict__ T, double *__restrict__ M) {
  __shared__ int chl[8][16];
  __shared__ v4d part[kM2MWaves][kWave];
  const int PP = P * P;
  const int lane = threadIdx.x % kWave, o = threadIdx.x / kWave;
  const int j16 = lane & 15, kq = lane >> 4;
  const int p0 = bx * 16;
  if (threadIdx.x < 128) chl[threadIdx.x / 16][threadIdx.x % 16] = -1;
  __syncthreads();
  file_children(threadIdx.x, p0, lstart, lcount, cchild, cnch, cx, -1, chl);
  __syncthreads();
  const int r0 = by * 16;  // the grid has ceil(PP / 16) row tiles: r0 < PP
  const int jmax = degree_of(min(r0 + 16, PP) - 1);
  const int ncol = (jmax + 1) * (jmax + 1);
  const int ksteps = (ncol + 3) / 4;
  const int row = min(r0 + j16, PP - 1);  // rows past PP compute garbage that is never stored
  const int ch = chl[o][j16];
  const double *To = T + int64_t(o) * PP * PP;
  const double *Mc = M + int64_t(ch < 0 ? 0 : ch) * PP;
  v4d acc = {0, 0, 0, 0};
  for (int k0 = 0; k0 < ksteps; k0 += kShiftBatch) {
    double a[kShiftBatch], b[kShiftBatch];
#pragma unroll
    for (int s = 0; s < kShiftBatch; s++) {
      const int col = (k0 + s) * 4 + kq;
      const bool in = col < ncol;
      a[s] = in ? To[int64_t(col) * PP + row] : 0.0;
      b[s] = (in && ch >= 0) ? Mc[col] : 0.0;
    }
#pragma unroll
    for (int s = 0; s < kShiftBatch; s++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], b[s], acc, 0, 0, 0);
  }
  part[o][lane] = acc;
  __syncthreads();
  if (o != 0) return;
  v4d sum = part[0][lane];
#pragma unroll
  for (int oo = 1; oo < kM2MWaves; oo++) sum += part[oo][lane];
  const int pl = p0 + j16;
  if (pl >= lcount) return;
  const int p = lstart + pl;
  if (cnch[p] == 0) return;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int r = r0 + kq + 4 * i;
    if (r < PP) M[int64_t(p) * PP + r] = sum[i];
  }
}

__global__ void __launch_bounds__(kM2MWaves *kWave) k_m2m(int P, int lstart, int lcount,
                                                          const int *__restrict__ cchild,
                                                          const int *__restrict__ cnch,
                                                          const double4 *__restrict__ cx,
                                                          const double *__restrict__ T, double *__restrict__ M) {
  m2m_body(blockIdx.x, blockIdx.y, P, lstart, lcount, cchild, cnch, cx, T, M);
}

// Row-tile form of M2M (single tree): one workgroup per 16 parents of a
// level, wave w = row tile w of the P^2 rows (ceil(P^2/16) waves), each wave
// looping over the 8 octants.  All waves that read a parent tile's children
// run in one workgroup, so those rows come from HBM once and then from that
// CU's caches.  Operator columns and the B operand are loaded kShiftBatch2
// k-steps at a time.
constexpr int kShiftBatch2 = 8;
constexpr int kRowTileMaxWaves = 16;  // P <= 16
// Levels with fewer parents run the octant-parallel kernel (k_m2m, an octant
// per wave): its chains of dependent loads are 8x shorter, and few parents
// leave the cache-sharing of the row-tile form little to share.
constexpr int kRowTileMinParents = 8192;

// waves of a row-tile workgroup: one per row tile, at least two (filing the
// children of 16 parents takes 128 threads)
static int row_tile_waves(int PP) { return std::max(2, ceil_div(PP, 16)); }

// M~_parent = sum over octants of T_M2M[octant] M~_child (3d/kernel.h:206),
// octants added in order into one accumulator per row tile.
__global__ void __launch_bounds__(kRowTileMaxWaves *kWave) k_m2m_rows(int P, int lstart, int lcount,
                                                                      const int *__restrict__ cchild,
                                                                      const int *__restrict__ cnch,
                                                                      const double4 *__restrict__ cx,
                                                                      const double *__restrict__ T,
                                                                      double *__restrict__ M) {
  __shared__ int chl[8][16];
  const int PP = P * P;
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  const int j16 = lane & 15, kq = lane >> 4;
  const int p0 = blockIdx.x * 16;
  if (threadIdx.x < 128) chl[threadIdx.x / 16][threadIdx.x % 16] = -1;
  __syncthreads();
  file_children(threadIdx.x, p0, lstart, lcount, cchild, cnch, cx, -1, chl);
  __syncthreads();
  const int r0 = w * 16;  // blockDim.x = 64 max(2, ceil(PP / 16))
  if (r0 >= PP) return;
  const int jmax = degree_of(min(r0 + 16, PP) - 1);
  const int ncol = (jmax + 1) * (jmax + 1);
  const int ksteps = (ncol + 3) / 4;
  const int row = min(r0 + j16, PP - 1);
  v4d acc = {0, 0, 0, 0};
  for (int o = 0; o < 8; o++) {
    const int ch = chl[o][j16];
    if (!__any(ch >= 0)) continue;
    const double *To = T + int64_t(o) * PP * PP;
    const double *Mc = M + int64_t(ch < 0 ? 0 : ch) * PP;
    for (int k0 = 0; k0 < ksteps; k0 += kShiftBatch2) {
      double a[kShiftBatch2], b[kShiftBatch2];
#pragma unroll
      for (int s = 0; s < kShiftBatch2; s++) {
        const int col = (k0 + s) * 4 + kq;
        const bool in = col < ncol;
        a[s] = in ? To[int64_t(col) * PP + row] : 0.0;
        b[s] = (in && ch >= 0) ? Mc[col] : 0.0;
      }
#pragma unroll
      for (int s = 0; s < kShiftBatch2; s++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], b[s], acc, 0, 0, 0);
    }
  }
  const int pl = p0 + j16;
  if (pl >= lcount) return;
  const int p = lstart + pl;
  if (cnch[p] == 0) return;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int r = r0 + kq + 4 * i;
    if (r < PP) M[int64_t(p) * PP + r] = acc[i];
  }
}

// L~_child += T_L2L[octant] L~_parent (3d/kernel.h:265-280) for the cells
// cell0 .. cell0 + nc - 1 of one level (single tree).  A workgroup keeps one
// octant's operator in registers -- wave w the row tile w, all its k-steps --
// and takes the cells of that octant in its range of the level, 16 at a time
// (grid: (ranges, octants); the octants' workgroups of a range share an XCD and
// so the parents' rows).  The operator is loaded once per workgroup where the
// row-tile form above reads it again for every 16 parents, and the waves meet
// only where a list of cells begins.  Orders above 13 have more row tiles than
// waves fit beside such registers: two passes over the row tiles.  Bound by the
// FP64 matrix rate and the cells' rows; the levels of 1.5M clustered bodies,
// order 12: 650 -> 232 us, of 300,007, order 13: 200 -> 118.
template <int P>
struct L2LShape {
  static constexpr int PP = P * P, RT = (PP + 15) / 16, Passes = RT > 11 ? 2 : 1, W = (RT + Passes - 1) / Passes;
  static constexpr int KS = (PP + 3) / 4;  // k-steps of a full row tile
  // k-steps loaded together: 4 to 7, as KS divides best
  static constexpr int batch() {
    int best = 7;
    for (int k = 6; k >= 4; k--)
      if ((KS + k - 1) / k * k < (KS + best - 1) / best * best) best = k;
    return best;
  }
  static constexpr int B = batch(), NB = (KS + B - 1) / B;
  static constexpr int PerCU = 2 * W <= 16 ? 2 : 1;  // workgroups a CU has room for
};
constexpr int kL2LChunk = 1024;  // cells filtered at a time
template <int P>
__global__ void __launch_bounds__(L2LShape<P>::W *kWave) k_l2l_oct(int cell0, int nc,
                                                                   const unsigned char *__restrict__ coct,
                                                                   const int *__restrict__ cparent,
                                                                   const double *__restrict__ T,
                                                                   double *__restrict__ L) {
  using Sh = L2LShape<P>;
  constexpr int PP = Sh::PP, NTH = Sh::W * kWave, B = Sh::B, NB = Sh::NB;
  __shared__ int cell[kL2LChunk], parent[kL2LChunk];
  __shared__ int count;
  const int lane = threadIdx.x % kWave, w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int j16 = lane & 15, kq = lane >> 4;
  const int o = blockIdx.y;
  const int first = cell0 + int(int64_t(nc) * blockIdx.x / gridDim.x);
  const int last = cell0 + int(int64_t(nc) * (blockIdx.x + 1) / gridDim.x);
  const double *To = T + (int64_t(8) + o) * PP * PP;
  for (int base = first; base < last; base += kL2LChunk) {
    const int end = min(base + kL2LChunk, last);
    __syncthreads();  // the last chunk's lists are done with
    if (threadIdx.x == 0) count = 0;
    __syncthreads();
    for (int i0 = base; i0 < end; i0 += NTH) {
      const int c = i0 + threadIdx.x;
      const bool mine = c < end && coct[c] == o;
      const unsigned long long m = __ballot(mine);
      int at = 0;
      if (lane == 0 && m) at = atomicAdd(&count, int(__popcll(m)));  // (the order of the list does not matter)
      at = __shfl(at, 0) + __popcll(m & (lane ? (~0ull >> (64 - lane)) : 0ull));
      if (mine) {
        cell[at] = c;
        parent[at] = cparent[c];
      }
    }
    __syncthreads();
    const int n = count;
    if (n == 0) continue;
    for (int pass = 0; pass < Sh::Passes; pass++) {
      const int r0 = (pass * Sh::W + w) * 16;
      if (r0 >= PP) continue;
      // the row tile's columns c0 .. PP - 1 in nb whole batches that end at the
      // last column: those before c0 have factors 0
      const int jmin = degree_of(r0), c0 = jmin * jmin;
      const int nb = (PP - c0 + 4 * B - 1) / (4 * B), cs = PP - 4 * B * nb + kq;
      const int row = min(r0 + j16, PP - 1);
      double a[NB * B];
#pragma unroll
      for (int s = 0; s < NB * B; s++) {
        const int col = cs + 4 * s;
        a[s] = col >= c0 && col < PP ? To[int64_t(col) * PP + row] : 0.0;
      }
      for (int g = 0; g < n; g += 16) {
        const bool in = g + j16 < n;
        const int at = min(g + j16, n - 1);
        const double *Lp = L + int64_t(parent[at]) * PP;
        double *Lc = L + int64_t(cell[at]) * PP;
        double old[4], b[2][B];
#pragma unroll
        for (int s = 0; s < B; s++) b[0][s] = Lp[max(cs + 4 * s, 0)];
        Lp += cs;
#pragma unroll
        for (int i = 0; i < 4; i++) old[i] = Lc[min(r0 + kq + 4 * i, PP - 1)];
        v4d acc = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < NB; k++) {
          if (k < nb) {  // uniform
            if (k + 1 < nb) {  // the next batch's loads ahead of the products
#pragma unroll
              for (int s = 0; s < B; s++) b[(k + 1) & 1][s] = Lp[4 * ((k + 1) * B + s)];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < B; s++)
              acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k * B + s], b[k & 1][s], acc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        if (in) {
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const int r = r0 + kq + 4 * i;
            if (r < PP) Lc[r] = old[i] + acc[i];
          }
        }
      }
    }
  }
}

// One level of every problem of a batch in one launch: lv[i] describes
// problem lv[i].prob's cells of this level as nbx x nby blocks.
__global__ void __launch_bounds__(kM2MWaves *kWave) k_m2m_grouped(const GroupTree *__restrict__ g,
                                                                    const GroupLevel *__restrict__ lv,
                                                                    const int *__restrict__ start, int n) {
  const int b = blockIdx.x, i = group_of(start, n, b), lb = b - start[i];
  const GroupLevel L = lv[i];
  const GroupTree &t = g[L.prob];
  m2m_body(lb % L.nbx, lb / L.nbx, t.P, L.lstart, L.lcount, t.cchild, t.cnch, t.cx, t.shift_T, t.M);
}


// L~_child += T_L2L[octant] L~_parent for the children of one level of
// parents (3d/kernel.h:265-280).  grid: (parent tiles of 16, row blocks of
// 64, octant).
__device__ __attribute__((always_inline)) inline void l2l_body(int bx, int by, int bz, int P, int lstart, int lcount,
                                const int *__restrict__ cchild,
                                const int *__restrict__ cnch,
                                const double4 *__restrict__ cx,
                                const double *__restrict__ T, double *__restrict__ L) {
  __shared__ int chl[1][16];
  const int PP = P * P;
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  const int j16 = lane & 15, kq = lane >> 4;
  const int p0 = bx * 16, o = bz;
  if (threadIdx.x < 16) chl[0][threadIdx.x] = -1;
  __syncthreads();
  file_children(threadIdx.x, p0, lstart, lcount, cchild, cnch, cx, o, chl);
  __syncthreads();
  const int r0 = (by * kShiftWaves + w) * 16;
  if (r0 >= PP) return;
  const int jmin = degree_of(r0);
  const int c0 = jmin * jmin;
  const int ksteps = (PP - c0 + 3) / 4;
  const int row = min(r0 + j16, PP - 1);
  const int ch = chl[0][j16];
  const double *To = T + (int64_t(8) + o) * PP * PP;
  const int pl = min(p0 + j16, lcount - 1);
  const double *Lp = L + int64_t(lstart + pl) * PP;
  v4d acc = {0, 0, 0, 0};
  for (int k0 = 0; k0 < ksteps; k0 += kL2LBatch) {
    double a[kL2LBatch], b[kL2LBatch];
#pragma unroll
    for (int s = 0; s < kL2LBatch; s++) {
      const int col = c0 + (k0 + s) * 4 + kq;
      const bool in = col < PP;
      a[s] = in ? To[int64_t(col) * PP + row] : 0.0;
      b[s] = (in && ch >= 0) ? Lp[col] : 0.0;
    }
#pragma unroll
    for (int s = 0; s < kL2LBatch; s++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], b[s], acc, 0, 0, 0);
  }
  if (ch < 0) return;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int r = r0 + kq + 4 * i;
    if (r < PP) L[int64_t(ch) * PP + r] += acc[i];
  }
}

// One level of parents of every problem of a batch in one launch (blocks
// nbx x nby x 8 octants per problem).
__global__ void __launch_bounds__(kShiftWaves *kWave) k_l2l_grouped(const GroupTree *__restrict__ g,
                                                                    const GroupLevel *__restrict__ lv,
                                                                    const int *__restrict__ start, int n) {
  const int b = blockIdx.x, i = group_of(start, n, b), lb = b - start[i];
  const GroupLevel L = lv[i];
  const GroupTree &t = g[L.prob];
  const int bx = lb % L.nbx, r = lb / L.nbx;
  l2l_body(bx, r % L.nby, r / L.nby, t.P, L.lstart, L.lcount, t.cchild, t.cnch, t.cx, t.shift_T, t.L);
}


// ---------------------------------------------------------------- L2P
// With u = (x - Xc)/R and Lh_n^m = w_m L_n^m R^n = w_m L~/R (w_0 = 1, w_m = 2),
// phi = Re sum_{n, m>=0} Lh_n^m Y_n^m(u) (3d/kernel.h:302-316).  The gradient uses
//   dz Y_n^m = -Y_{n-1}^m,  (dx + i dy) Y_n^m = -Y_{n-1}^{m+1},
//   (dx - i dy) Y_n^m = Y_{n-1}^{m-1} (m >= 1), = -conj(Y_{n-1}^1) (m = 0).
// Degree by degree, with the harmonics of the last two degrees in registers:
// every coefficient is read from LDS once and meets Y_{n-1}^{m-1}, Y_{n-1}^m,
// Y_{n-1}^{m+1} and Y_n^m there.  (Column by column a coefficient was read for
// each of the four, and orders without an unrolled kernel ran a loop of
// dependent LDS reads: order 12, 1.5M bodies 223 -> 90 us.)
template <int P, class T>
__device__ __attribute__((always_inline)) inline void l2p_eval(T x, T y, T z, const cpx<T> *Lh, T &pot, T &Fx2,
                                                               T &Fy2, T &Dz) {
  T r2 = x * x + y * y + z * z;
  T Ar = 0, Ai = 0, Br = 0, Bi = 0, dz = 0, ph = Lh[0].re;
  T ar[P], ai[P], br[P], bi[P];  // Y_{n-1}^m, Y_{n-2}^m
#pragma unroll
  for (int m = 0; m < P; m++) ar[m] = ai[m] = br[m] = bi[m] = 0;
  ar[0] = 1;
  int o = 0;
#pragma unroll
  for (int n = 1; n < P; n++) {
    // opaque position and offset: this degree's harmonics and coefficients are
    // made here, not all at the front, where they would take every register
    asm volatile("" : "+v"(o), "+v"(x), "+v"(y), "+v"(z), "+v"(r2), "+v"(ph), "+v"(dz), "+v"(Ar), "+v"(Ai), "+v"(Br),
                      "+v"(Bi));
    T cr[P], ci[P];  // Y_n^m
#pragma unroll
    for (int m = 0; m <= n; m++) {
      if (m == n) {
        const T inv = T(0.5 / n);
        cr[m] = (ar[n - 1] * x - ai[n - 1] * y) * inv;
        ci[m] = (ar[n - 1] * y + ai[n - 1] * x) * inv;
      } else if (m == n - 1) {
        cr[m] = -z * ar[m];
        ci[m] = -z * ai[m];
      } else {
        const T s = T(-1.0 / double((n + m) * (n - m))), cz = T(2 * n - 1) * z;
        cr[m] = (cz * ar[m] + r2 * br[m]) * s;
        ci[m] = m ? (cz * ai[m] + r2 * bi[m]) * s : T(0);
      }
      const cpx<T> l = Lh[o + nms(n, m)];
      if (m == 0) {  // real
        ph += l.re * cr[0];
        dz -= l.re * ar[0];
        if (n > 1) {
          Ar -= T(2) * (l.re * ar[1]);
          Ai -= T(2) * (l.re * ai[1]);
        }
      } else {
        ph += l.re * cr[m] - l.im * ci[m];
        if (m < n) dz -= l.re * ar[m] - l.im * ai[m];
        if (m + 1 < n) {
          Ar -= l.re * ar[m + 1] - l.im * ai[m + 1];
          Ai -= l.re * ai[m + 1] + l.im * ar[m + 1];
        }
        Br += l.re * ar[m - 1] - l.im * ai[m - 1];
        Bi += l.re * ai[m - 1] + l.im * ar[m - 1];
      }
    }
#pragma unroll
    for (int m = 0; m <= n; m++) {
      br[m] = ar[m];
      bi[m] = ai[m];
      ar[m] = cr[m];
      ai[m] = ci[m];
    }
  }
  pot = ph;
  Dz = dz;
  Fx2 = Ar + Br;  // 2 dphi/dx
  Fy2 = Ai - Bi;  // 2 dphi/dy
}

// L2P over the bodies in tree order, 64 per wave (full waves whatever the leaf
// sizes; one wave per leaf leaves half its lanes idle at 32 bodies a leaf).
// The wave's bodies fall into runs of equal leaf; up to kL2PSlots runs at a
// time have their coefficients staged in LDS (one pass for uniform trees, a
// few when many small leaves share a wave), and each lane evaluates its own
// body against its run's slot.  T = float, or double in parity mode.
constexpr int kL2PSlots = 8;
template <int P, class T>
struct L2PLds {
  cpx<T> Lh[kL2PSlots][(P * (P + 1) / 2) | 1];  // odd: the slots' equal entries lie in distinct banks
  int leaf[kL2PSlots];
};
template <int P, class T>
__device__ __attribute__((always_inline)) inline void l2p_body(int bx, int64_t n, const int *__restrict__ body_leaf,
                                                               const double4 *__restrict__ cx,
                                                               const double *__restrict__ L,
                                                               const double4 *__restrict__ xs,
                                                               exafmm_body *__restrict__ bodies,
                                                               L2PLds<P, T> &lds) {
  constexpr int NT = P * (P + 1) / 2, KE = (NT + kWave - 1) / kWave;
  auto &Lh = lds.Lh;
  auto &sleaf = lds.leaf;
  const int lane = threadIdx.x;
  const int64_t b = int64_t(bx) * kWave + lane;
  const bool valid = b < n;
  const int leaf = valid ? body_leaf[b] : -1;
  const int prev = __shfl_up(leaf, 1);
  const unsigned long long starts = __ballot(valid && (lane == 0 || prev != leaf));
  const int nruns = __popcll(starts);
  const int run = valid ? __popcll(starts & (~0ull >> (63 - lane))) - 1 : -1;
  int em[KE], er[KE];  // this lane's coefficients: order m, place of the real part
#pragma unroll
  for (int k = 0; k < KE; k++) {
    int en;
    jk_of(min(lane + k * kWave, NT - 1), en, em[k]);
    er[k] = rf(en, em[k], 0);
  }
  double4 C = make_double4(0, 0, 0, 1), B = make_double4(0, 0, 0, 0);
  if (valid) {
    C = cx[leaf];
    B = xs[b];
  }
  const double invR = C.w > 0.0 ? 1.0 / C.w : 0.0;  // R = 0: every body at the centre
  for (int g0 = 0; g0 < nruns; g0 += kL2PSlots) {
    const int ns = min(kL2PSlots, nruns - g0);
    if (valid && run >= g0 && run < g0 + ns && (lane == 0 || prev != leaf)) sleaf[run - g0] = leaf;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
#pragma unroll 4
    for (int sl = 0; sl < ns; sl++) {
      const int c = __builtin_amdgcn_readfirstlane(sleaf[sl]);
      const double Rc = cx[c].w, w = Rc > 0.0 ? 1.0 / Rc : 0.0;
      const double *Lc = L + int64_t(c) * P * P;
#pragma unroll
      for (int k = 0; k < KE; k++)
        if (lane + k * kWave < NT) {
          const double re = Lc[er[k]], im = em[k] ? Lc[er[k] + 1] : 0.0;
          const double wm = em[k] ? 2.0 * w : w;
          Lh[sl][lane + k * kWave] = {T(re * wm), T(im * wm)};
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (valid && run >= g0 && run < g0 + ns) {
      T pot, fx2, fy2, dz;
      l2p_eval<P, T>(T((B.x - C.x) * invR), T((B.y - C.y) * invR), T((B.z - C.z) * invR), Lh[run - g0], pot, fx2, fy2,
                     dz);
      exafmm_body *o = bodies + b;
      o->p += double(pot);
      o->F[0] += 0.5 * double(fx2) * invR;
      o->F[1] += 0.5 * double(fy2) * invR;
      o->F[2] += double(dz) * invR;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

template <int P, class T>
__global__ void __launch_bounds__(64) k_l2p(int64_t n, const int *__restrict__ body_leaf,
                                            const double4 *__restrict__ cx, const double *__restrict__ L,
                                            const double4 *__restrict__ xs, exafmm_body *__restrict__ bodies) {
  __shared__ L2PLds<P, T> lds;
  l2p_body<P, T>(blockIdx.x, n, body_leaf, cx, L, xs, bodies, lds);
}

// All problems of a batch in one launch, each workgroup by its problem's order
// (a launch per order: 45 us for three orders, their tails one after the other).
__global__ void __launch_bounds__(64) k_l2p_grouped(const GroupTree *__restrict__ g, const int *__restrict__ start,
                                                    int nprob) {
  __shared__ L2PLds<kMaxP, float> lds;  // every order's fits
  const int b = blockIdx.x, i = group_of(start, nprob, b);
  const GroupTree &t = g[i];
  auto run = [&](auto p) {
    l2p_body<p(), float>(b - start[i], t.n, t.body_leaf, t.cx, t.L, t.xs, t.bodies,
                         reinterpret_cast<L2PLds<p(), float> &>(lds));
  };
  switch (t.P) {
    XF_ORDER_CASES(run)
  }
}


// ---------------------------------------------------------------- grouped launches
int p2m_group_blocks(int64_t nleaves) { return ceil_div(nleaves, kP2MWaves); }
int shift_group_rows(int P) { return ceil_div(P * P, 16 * kShiftWaves); }
int m2m_group_rows(int P) { return ceil_div(P * P, 16); }

void p2m_orders(const GroupTree *g, const int *start, int nprob, int nblocks, hipStream_t s) {
  hipLaunchKernelGGL(k_p2m_orders, dim3(nblocks), dim3(kP2MWaves * kWave), 0, s, g, start, nprob);
  XF_LAUNCH();
}
void p2m_grouped(int P, const GroupTree *g, const int *start, int nprob, int nblocks, hipStream_t s) {
  by_order(P, [&](auto p) {
    hipLaunchKernelGGL((k_p2m_grouped<p()>), dim3(nblocks), dim3(kP2MWaves * kWave), 0, s, g, start, nprob);
  });
  XF_LAUNCH();
}
void m2m_grouped(const GroupTree *g, const GroupLevel *lv, const int *start, int n, int nblocks, hipStream_t s) {
  hipLaunchKernelGGL(k_m2m_grouped, dim3(nblocks), dim3(kM2MWaves * kWave), 0, s, g, lv, start, n);
  XF_LAUNCH();
}
void l2l_grouped(const GroupTree *g, const GroupLevel *lv, const int *start, int n, int nblocks, hipStream_t s) {
  hipLaunchKernelGGL(k_l2l_grouped, dim3(nblocks), dim3(kShiftWaves * kWave), 0, s, g, lv, start, n);
  XF_LAUNCH();
}
void l2p_grouped(const GroupTree *g, const int *start, int nprob, int nblocks, hipStream_t s) {
  hipLaunchKernelGGL(k_l2p_grouped, dim3(nblocks), dim3(kWave), 0, s, g, start, nprob);
  XF_LAUNCH();
}

void upward(Ctx &c, hipStream_t s, hipEvent_t wide) {
  Tree &t = c.t;
  const int P = c.P, PP = P * P;
  shift_ops(c, s);
  c.M.ensure(size_t(t.ncells) * PP);
  by_order(P, [&](auto p) {
    hipLaunchKernelGGL((k_p2m<p()>), dim3(ceil_div(t.nleaves, kP2MWaves)), dim3(kP2MWaves * kWave), 0, s, t.leaves.p,
                       t.misc.p + 17, t.cbeg.p, t.ccnt.p, t.cx.p, t.xs.p, c.M.p);
  });
  XF_LAUNCH();
  int last_wide = t.depth;  // the last level, going up, that fills the device
  for (int l = t.lroot; l < t.depth && last_wide == t.depth; l++)
    if (t.lstart[l + 1] - t.lstart[l] >= kRowTileMinParents) last_wide = l;
  if (wide && last_wide == t.depth) XF_HIP(hipEventRecord(wide, s));
  for (int l = t.depth - 1; l >= t.lroot; l--) {  // (a forest stops at its problems' roots)
    const int cnt = t.lstart[l + 1] - t.lstart[l];
    if (cnt >= kRowTileMinParents)
      hipLaunchKernelGGL(k_m2m_rows, dim3(ceil_div(cnt, 16)), dim3(row_tile_waves(PP) * kWave), 0, s, c.P,
                         t.lstart[l], cnt, t.cchild.p, t.cnch.p, t.cx.p, c.shift_T.p, c.M.p);
    else
      hipLaunchKernelGGL(k_m2m, dim3(ceil_div(cnt, 16), m2m_group_rows(P)), dim3(kM2MWaves * kWave), 0, s, c.P,
                         t.lstart[l], cnt, t.cchild.p, t.cnch.p, t.cx.p, c.shift_T.p, c.M.p);
    XF_LAUNCH();
    if (wide && l == last_wide) XF_HIP(hipEventRecord(wide, s));
  }
  c.have_M = true;
}

void l2l_pass(Ctx &c) {
  Tree &t = c.t;
  hipStream_t s = c.s0;
  shift_ops(c, s);
  by_order(c.P, [&](auto p) {
    using Sh = L2LShape<p()>;
    for (int l = t.lroot + 1; l <= t.depth; l++) {
      const int nc = t.lstart[l + 1] - t.lstart[l];
      // ranges with about 16 cells per octant, until the device is full
      const int ranges = std::min(std::max(1, nc / 128), 32 * Sh::PerCU);
      hipLaunchKernelGGL((k_l2l_oct<p()>), dim3(ranges, 8), dim3(Sh::W * kWave), 0, s, t.lstart[l], nc, t.coct.p,
                         t.cparent.p, c.shift_T.p, c.L.p);
      XF_LAUNCH();
    }
  });
}

void l2p_pass(Ctx &c) {
  Tree &t = c.t;
  // FP64 evaluation in parity mode, FP32 otherwise
  by_order(c.P, [&](auto p) {
    auto k = c.cfg.m2l_precision == EXAFMM_PREC_FP64 ? k_l2p<p(), double> : k_l2p<p(), float>;
    hipLaunchKernelGGL(k, dim3(ceil_div(t.n, kWave)), dim3(kWave), 0, c.s0, t.n, t.body_leaf.p, t.cx.p, c.L.p, t.xs.p,
                       c.bodies);
  });
  XF_LAUNCH();
}

}  // namespace xf
