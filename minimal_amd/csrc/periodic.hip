// periodic.hip -- far periodic images, dipole correction, Ewald oracle.
//
// Far images (3dp/traverse_lazy.h:75-121, eager 3dp/traverse_eager.h:46-92):
// a super-cell starts as the root (centre X0, multipole M_root); at each of
// images-1 levels the root's local expansion receives M2L from the 26 x 27
// copies at offsets (3i + c) * cycle (i != 0), then the super-cell absorbs
// its 26 neighbours by M2M and cycle triples.  Each level's M2L is one
// launch of 702 workgroups writing partial locals, summed in a fixed order;
// the M2M is one workgroup per neighbour, summed in neighbour order.
//
// Dipole correction (3dp/fmm.cxx:63-75): p -= 4 pi/(3 cycle^3) |D|^2 / N / q,
// F -= 4 pi/(3 cycle^3) D, D = sum q X.  Bodies with q = 0 keep p (the
// reference divides by q).
//
// Ewald sum (3dp/ewald.h:22-150) in FP64 on the device: wave part by
// DFT/IDFT over the half space |k| <= ksize, real part with erfc over each
// body pair's nearest image within the cutoff, self term.
#include <algorithm>
#include <cmath>

#include <mutex>
#include <string>

#include "fmm_internal.h"
#include "fmm_ops.h"

namespace xf {
using namespace xfd;

__global__ void __launch_bounds__(64) k_far_m2l(int P, int NT, int fillP, double cyc, const double2 *__restrict__ Msup,
                                                double2 *__restrict__ part) {
  __shared__ cpx<double> I[(2 * kMaxP) * (2 * kMaxP + 1) / 2];
  __shared__ double2 Ms[kMaxP * (kMaxP + 1) / 2];
  const int e = blockIdx.x;  // 26 neighbour blocks x 27 sub-images, reference loop order
  const int ib = e / 27, cidx = e % 27;
  const int nb = ib < 13 ? ib : ib + 1;  // skip the centre block
  const int ix = nb / 9 - 1, iy = (nb / 3) % 3 - 1, iz = nb % 3 - 1;
  const int cx = cidx / 9 - 1, cy = (cidx / 3) % 3 - 1, cz = cidx % 3 - 1;
  // dX = X_root - X_super - iX * cycle, with X_super = X_root
  const double dx = -(ix * 3 + cx) * cyc, dy = -(iy * 3 + cy) * cyc, dz = -(iz * 3 + cz) * cyc;
  if (threadIdx.x < fillP) singular_column(threadIdx.x, fillP, dx, dy, dz, I);
  for (int i = threadIdx.x; i < NT; i += 64) Ms[i] = Msup[i];
  __syncthreads();
  for (int jk = threadIdx.x; jk < NT; jk += 64) {
    int j, k;
    jk_of(jk, j, k);
    part[int64_t(e) * NT + jk] = m2l_coef(P, fillP, j, k, Ms, I);
  }
}

// Sum of the partial locals, added to the root's scaled L~: one workgroup
// per coefficient, the parts added by a fixed-order tree.
__global__ void __launch_bounds__(256) k_far_sum(int P, int nparts, double R0, const double2 *__restrict__ part,
                                                 double *__restrict__ Lroot) {
  __shared__ double sx[256], sy[256];
  const int NT = P * (P + 1) / 2, jk = blockIdx.x, t = threadIdx.x;
  double ax = 0, ay = 0;
  for (int e = t; e < nparts; e += 256) {
    ax += part[int64_t(e) * NT + jk].x;
    ay += part[int64_t(e) * NT + jk].y;
  }
  sx[t] = ax;
  sy[t] = ay;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (t < o) {
      sx[t] += sx[t + o];
      sy[t] += sy[t + o];
    }
    __syncthreads();
  }
  if (t == 0) {
    int j, k;
    jk_of(jk, j, k);
    const double s = pow(R0, double(j + 1));
    Lroot[rf(j, k, 0)] += sx[0] * s;
    if (k > 0) Lroot[rf(j, k, 1)] += sy[0] * s;
  }
}

// Root multipole M = M~ R0^n (complex) as the first super-cell.
__global__ void __launch_bounds__(64) k_far_init(int P, double R0, const double *__restrict__ Mroot,
                                                 double2 *__restrict__ sup) {
  const int NT = P * (P + 1) / 2;
  for (int jk = threadIdx.x; jk < NT; jk += 64) {
    int n, m;
    jk_of(jk, n, m);
    const double s = pow(R0, double(n));
    sup[jk] = make_double2(Mroot[rf(n, m, 0)] * s, m ? Mroot[rf(n, m, 1)] * s : 0.0);
  }
}

// Msup += sum over the 26 neighbours (child centre X + i*cycle) of
// M2M(Msup): one workgroup per neighbour writes its term, then the terms
// are added in neighbour order.
__global__ void __launch_bounds__(64) k_far_m2m(int P, int NT, double cyc, const double2 *__restrict__ Msup,
                                                double2 *__restrict__ part) {
  __shared__ cpx<double> Y[kMaxP * (kMaxP + 1) / 2];
  __shared__ double2 Mc[kMaxP * (kMaxP + 1) / 2];
  const int b = blockIdx.x, nb = b < 13 ? b : b + 1;  // skip the centre
  const int ix = nb / 9 - 1, iy = (nb / 3) % 3 - 1, iz = nb % 3 - 1;
  for (int i = threadIdx.x; i < NT; i += 64) Mc[i] = Msup[i];
  if (threadIdx.x == 0) regular_all<double>(P, -ix * cyc, -iy * cyc, -iz * cyc, Y);  // Xparent - Xchild
  __syncthreads();
  for (int jk = threadIdx.x; jk < NT; jk += 64) {
    int j, k;
    jk_of(jk, j, k);
    part[int64_t(b) * NT + jk] = m2m_coef(j, k, Mc, Y);
  }
}

__global__ void __launch_bounds__(64) k_far_m2m_sum(int NT, const double2 *__restrict__ part,
                                                    double2 *__restrict__ Msup) {
  for (int jk = threadIdx.x; jk < NT; jk += 64) {
    double2 acc = make_double2(0, 0);
    for (int b = 0; b < 26; b++) {
      acc.x += part[int64_t(b) * NT + jk].x;
      acc.y += part[int64_t(b) * NT + jk].y;
    }
    Msup[jk].x += acc.x;
    Msup[jk].y += acc.y;
  }
}

void periodic_far(Ctx &c) {
  const int P = c.P, NT = c.NT;
  const int fillP = c.cfg.m2l_truncation == EXAFMM_M2L_FULL ? 2 * P - 1 : P;
  if (c.cfg.images < 2) return;
  Buf<double2> &sup = c.far_sup, &part = c.far_part;
  sup.ensure(NT);
  part.ensure(size_t(702) * NT);
  hipLaunchKernelGGL(k_far_init, dim3(1), dim3(64), 0, c.s0, P, c.t.R0, c.M.p, sup.p);
  XF_LAUNCH();
  double cyc = c.cfg.cycle;
  for (int lev = 0; lev < c.cfg.images - 1; lev++) {
    hipLaunchKernelGGL(k_far_m2l, dim3(702), dim3(64), 0, c.s0, P, NT, fillP, cyc, sup.p, part.p);
    XF_LAUNCH();
    hipLaunchKernelGGL(k_far_sum, dim3(NT), dim3(256), 0, c.s0, P, 702, c.t.R0, part.p, c.L.p);
    XF_LAUNCH();
    // the 26 neighbour terms reuse the partial-local buffer (read above)
    hipLaunchKernelGGL(k_far_m2m, dim3(26), dim3(64), 0, c.s0, P, NT, cyc, sup.p, part.p);
    XF_LAUNCH();
    hipLaunchKernelGGL(k_far_m2m_sum, dim3(1), dim3(64), 0, c.s0, NT, part.p, sup.p);
    XF_LAUNCH();
    cyc *= 3;
  }
}

// ---------------------------------------------------------------- dipole
// Dipole moment sum_i q_i x_i: kDipoleBlocks workgroups sum grid-strided
// ranges, then one workgroup adds their partials in a fixed order.
constexpr int kDipoleBlocks = 256;
__device__ inline void block_sum3(double (&d)[3], double (*s)[256]) {
  for (int k = 0; k < 3; k++) s[k][threadIdx.x] = d[k];
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o)
      for (int k = 0; k < 3; k++) s[k][threadIdx.x] += s[k][threadIdx.x + o];
    __syncthreads();
  }
}

__global__ void __launch_bounds__(256) k_dipole(int64_t n, const exafmm_body *__restrict__ b, double *__restrict__ part) {
  __shared__ double s[3][256];
  double d[3] = {0, 0, 0};
  for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256)
    for (int k = 0; k < 3; k++) d[k] += b[i].X[k] * b[i].q;
  block_sum3(d, s);
  if (threadIdx.x < 3) part[blockIdx.x * 3 + threadIdx.x] = s[threadIdx.x][0];
}

__global__ void __launch_bounds__(256) k_dipole_final(const double *__restrict__ part, double *__restrict__ out) {
  __shared__ double s[3][256];
  double d[3] = {0, 0, 0};
  for (int k = 0; k < 3; k++) d[k] = part[threadIdx.x * 3 + k];
  block_sum3(d, s);
  if (threadIdx.x < 3) out[threadIdx.x] = s[threadIdx.x][0];
}

__global__ void __launch_bounds__(256) k_dipole_apply(int64_t n, double coef, const double *__restrict__ D,
                                                      exafmm_body *__restrict__ b) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const double dn = D[0] * D[0] + D[1] * D[1] + D[2] * D[2];
  if (b[i].q != 0) b[i].p -= coef * dn / double(n) / b[i].q;
  for (int k = 0; k < 3; k++) b[i].F[k] -= coef * D[k];
}

void dipole_correction(Ctx &c) {
  c.dipole_part.ensure(3 * kDipoleBlocks + 3);
  double *D = c.dipole_part.p + 3 * kDipoleBlocks;
  hipLaunchKernelGGL(k_dipole, dim3(kDipoleBlocks), dim3(256), 0, c.s0, c.t.n, c.bodies, c.dipole_part.p);
  XF_LAUNCH();
  hipLaunchKernelGGL(k_dipole_final, dim3(1), dim3(kDipoleBlocks), 0, c.s0, c.dipole_part.p, D);
  XF_LAUNCH();
  const double cyc = c.cfg.cycle;
  const double coef = 4 * M_PI / (3 * cyc * cyc * cyc);
  hipLaunchKernelGGL(k_dipole_apply, dim3(ceil_div(c.t.n, 256)), dim3(256), 0, c.s0, c.t.n, coef, D, c.bodies);
  XF_LAUNCH();
}

// ---------------------------------------------------------------- Ewald
struct Wave {
  double K[3];
  double re, im;
};

// Wave vectors k in the half space (3dp/ewald.h:54-79): l = 0..kmax,
// m = -kmax..kmax (0..kmax at l = 0), n = -kmax..kmax (1..kmax at l = m = 0),
// l^2 + m^2 + n^2 <= kmax^2, in that nested order.
//
// A row is one (l, m) with its run of n.  Largest |n| of a row; -1: no row.
__host__ __device__ inline int ewald_row_nmax(int kmax, int l, int m) {
  const int r = kmax * kmax - l * l - m * m;
  if (r < 0 || (l == 0 && m < 0)) return -1;
  int n = int(sqrt(double(r)));
  while (n * n > r) n--;
  while ((n + 1) * (n + 1) <= r) n++;
  return n;
}
__host__ __device__ inline int ewald_row_count(int kmax, int l, int m) {
  const int n = ewald_row_nmax(kmax, l, m);
  return n < 0 ? 0 : (l == 0 && m == 0) ? n : 2 * n + 1;
}
static int ewald_wave_count(int kmax) {
  int nw = 0;
  for (int l = 0; l <= kmax; l++)
    for (int m = -kmax; m <= kmax; m++) nw += ewald_row_count(kmax, l, m);
  return nw;
}

// Structure factors of the waves (3dp/ewald.h:22-34), one workgroup per row
// (l, m) and run of kEwaldRun orders |n|.  A source costs one sine/cosine
// pair for the row's phase l x + m y and one for z, in half turns (exact
// argument reduction); the orders n follow by complex multiplication, and n
// and -n share their four products, so a wave costs four FP64 operations per
// source instead of a sine and a cosine.  Every thread keeps the run's sums in
// registers; the lanes meet by recursive halving at the end.  100,003
// sources, 2,800 waves: 200 us; 1,150 us with a workgroup per wave.
constexpr int kEwaldThreads = 512, kEwaldWaves = kEwaldThreads / kWave;
// Orders per run: eight accumulator registers each, and every further run of a
// row repeats the row's sines over the sources.  Runs of 8 / 12 / 16 orders,
// 100,003 sources, two targets: ksize 5 397 / 400 / 405 us, 11 (one run of 12) 561
// / 455 / 460, 15 750 / 783 / 666, 23 1,564 / 1,577 / 1,457.
constexpr int kEwaldRun = 12;
__global__ void __launch_bounds__(kEwaldThreads) k_ewald_dft(int kmax, Wave *__restrict__ waves,
                                                             const exafmm_body *__restrict__ s, int64_t ns,
                                                             double cyc, double coef, double coef2) {
  __shared__ double red[kEwaldWaves][kWave];
  __shared__ int base;
  const int side = 2 * kmax + 1, row = blockIdx.x, l = row / side, m = row % side - kmax;
  const int nmax = ewald_row_nmax(kmax, l, m), n0 = blockIdx.y * kEwaldRun;
  if (nmax < n0) return;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
  if (tid == 0) base = 0;
  __syncthreads();
  int before = 0;  // waves of the rows before this one
  for (int r = tid; r < row; r += kEwaldThreads) before += ewald_row_count(kmax, r / side, r % side - kmax);
  if (before) atomicAdd(&base, before);
  const double u = 2.0 / cyc;
  // sums over the sources of Er c_n, Ei s_n, Er s_n, Ei c_n
  double a[kEwaldRun] = {}, b[kEwaldRun] = {}, c[kEwaldRun] = {}, d[kEwaldRun] = {};
  for (int64_t j = tid; j < ns; j += kEwaldThreads) {
    const double x = s[j].X[0], y = s[j].X[1], z = s[j].X[2] * u, q = s[j].q;
    double er, ei, zr, zi, cr = 1.0, ci = 0.0;
    sincospi(double(l) * (x * u) + double(m) * (y * u), &ei, &er);
    er *= q;
    ei *= q;
    sincospi(z, &zi, &zr);
    if (n0) sincospi(double(n0) * z, &ci, &cr);
#pragma unroll
    for (int i = 0; i < kEwaldRun; i++) {
      if (n0 + i <= nmax) {  // uniform
        a[i] = fma(er, cr, a[i]);
        b[i] = fma(ei, ci, b[i]);
        c[i] = fma(er, ci, c[i]);
        d[i] = fma(ei, cr, d[i]);
        const double tr = cr * zr - ci * zi;
        ci = cr * zi + ci * zr;
        cr = tr;
      }
    }
  }
  // lane l receives the total of the run's order l / 4 (four lanes share one)
  auto total = [&](const double (&x)[kEwaldRun]) {
    double v[16];
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = i < kEwaldRun ? x[i < kEwaldRun ? i : 0] : 0.0;
    double r = halving<16>(v, lane);
    r += __shfl_xor(r, 1);
    return r + __shfl_xor(r, 2);
  };
  const double ta = total(a), tb = total(b), tc = total(c), td = total(d);
  const int q = lane & 3;
  red[w][lane] = q == 0 ? ta : q == 1 ? tb : q == 2 ? tc : td;
  __syncthreads();
  if (tid < kWave) {
    double t = 0.0;
    for (int k = 0; k < kEwaldWaves; k++) t += red[k][tid];
    red[0][tid] = t;
  }
  __syncthreads();
  // threads 0 .. kEwaldRun - 1 write n = n0 + tid, the next kEwaldRun write -n
  const int i = tid % kEwaldRun, sg = tid < kEwaldRun ? 1 : -1, n = sg * (n0 + i);
  if (tid >= 2 * kEwaldRun || n0 + i > nmax || (sg < 0 && n == 0)) return;
  const int nmin = l == 0 && m == 0 ? 1 : -nmax;
  if (n < nmin) return;
  const double *t = red[0] + 4 * i;
  const double re = t[0] - sg * t[1], im = sg * t[2] + t[3];
  const double scale = M_PI * u;
  const double k0 = l * scale, k1 = m * scale, k2 = n * scale;
  const double KK = k0 * k0 + k1 * k1 + k2 * k2;
  const double factor = coef * exp(-KK * coef2) / KK;
  waves[base + n - nmin] = Wave{{double(l), double(m), double(n)}, re * factor, im * factor};
}

// exp(x^2) erfc(x) for x >= 0 as g(t) / (1 + 2x), t = (x - K) / (x + K),
// K = 3.75 (Shepherd and Laframboise, Math. Comp. 36, 1981, 249-253: this
// variable and weight make one polynomial serve every x).  g's coefficients:
// Chebyshev interpolation of the function computed to 100 digits, truncated
// at degree 24 (next terms below 3e-18) and expanded in powers of t; relative
// error against 40 digits on (0, 1000]: 6e-16.
constexpr double kErfcxK = 3.75;
constexpr int kErfcxDeg = 24;
static __constant__ double kErfcx[kErfcxDeg + 1] = {
    1.2375126308378275, -0.14024059858554697, 0.0035854154854644293, 0.082276738490145204, -0.10880393014174886,
    0.092304321160377484, -0.058693398589636771, 0.028362277418956406, -0.0097465795580292756,
    0.0017556258528952954, 0.00029371366559134481, -0.00029015408054084172, 5.1649098892682407e-05,
    2.2384239155082231e-05, -1.1444146237700524e-05, -9.7355989673677497e-07, 1.7516376488490621e-06,
    -5.7218230603224086e-08, -2.5866850716155884e-07, 2.3263508708859124e-08, 3.8675334242222354e-08,
    -3.7442100809620183e-09, -5.1739902140113095e-09, 3.1114333809799254e-10, 4.2514714447963895e-10};

// Per pair of the real part (3dp/ewald.h:82-102): with x = alpha r,
//   pot = erfc(x) / x,  grad = 2/sqrt(pi) exp(-x^2) / x^2 + erfc(x) / x^3,
// from one exponential, one 1/sqrt and one reciprocal.
__device__ inline void ewald_pair(double x2, double &pot, double &grad) {
  double y = __builtin_amdgcn_rsq(x2);
  const double e = fma(-(x2 * y), y, 1.0);
  y = fma(y * e, fma(e, 0.375, 0.5), y);
  double x = x2 * y;
  const unsigned hi = unsigned(__double2hiint(x2));
  if (hi - (123u << 20) >= (1800u << 20)) {  // outside the step's exponent range, denormals and infinity among it
    y = 1.0 / sqrt(x2);
    x = fmin(x2 * y, 1e6);  // (exp(-x^2) is 0 there, and the products below stay finite)
  }
  const double xk = x + kErfcxK, w = fma(2.0, x, 1.0), dd = xk * w;
  double r = __builtin_amdgcn_rcp(dd);
  const double f = fma(-dd, r, 1.0);
  r = fma(r, fma(f, f, f), r);  // 1 / ((x + K)(1 + 2x)), remainder f^3
  const double t = (x - kErfcxK) * (r * w);
  double g = kErfcx[kErfcxDeg];
#pragma unroll
  for (int i = kErfcxDeg - 1; i >= 0; i--) g = fma(g, t, kErfcx[i]);
  const double h = g * (r * xk);  // exp(x^2) erfc(x)
  const double ex = exp(-x2), hy = h * y;
  pot = ex * hy;
  grad = ex * (y * y) * (M_2_SQRTPI + hy);
}

// Two targets per workgroup, whose waves share the Ewald waves and the
// sources.  A loaded source is tested against both targets; the pairs inside
// the cutoff (about half at cutoff = cycle / 2) go into a queue per wave and
// target in LDS, and a queue is evaluated a full wave at a time, so no lane
// idles through the exponential.  FP64 VALU bound, at four waves per SIMD
// (140 registers would leave two).  1,000 targets x 100,003 sources: 400 us;
// 743 us with a workgroup per target and every lane branching over its own
// pair.
//
// Eight waves per workgroup while two workgroups per CU (all that their queues
// leave room for) take every target: up to kEwaldManyTargets.  Beyond, four, and one
// where there is a round or two of work (kEwaldFew sources and waves).  Eight /
// four / one, us: 1,000 targets x 20,000 sources, ksize 6, 124 / 139 / 271; 2,238 x
// 300, ksize 4, 35.6 / 30.3 / 28.0; 2,238 x 20,000 214 / 220 / 362; 20,000 x 256 132 /
// - / 51; 20,000 x 1,000, ksize 3, 160 / 114 / 94; 20,000 x 20,000 1,301 / 1,243 / 1,279.
constexpr int kEwaldTargets = 2;
constexpr int64_t kEwaldManyTargets = 1024, kEwaldFew = 256;
struct EwaldQueue {
  double x[2 * kWave], y[2 * kWave], z[2 * kWave], q[2 * kWave];
};
template <int W>
__global__ void __launch_bounds__(W *kWave) __attribute__((amdgpu_waves_per_eu(4)))
    k_ewald_target(int nw, const Wave *__restrict__ waves, exafmm_body *__restrict__ t, int64_t nt,
                   const exafmm_body *__restrict__ s, int64_t ns, double alpha, double cutoff, double cyc) {
  constexpr int NT = W * kWave;
  extern __shared__ EwaldQueue queues[];  // [wave][target]
  __shared__ double red[W][kEwaldTargets][4];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int64_t t0 = int64_t(blockIdx.x) * kEwaldTargets;
  double x[kEwaldTargets], y[kEwaldTargets], z[kEwaldTargets], acc[kEwaldTargets][4] = {};
  int fill[kEwaldTargets] = {};
#pragma unroll
  for (int k = 0; k < kEwaldTargets; k++) {
    const exafmm_body *b = t + min(t0 + k, nt - 1);
    x[k] = b->X[0];
    y[k] = b->X[1];
    z[k] = b->X[2];
  }
  // wave part (3dp/ewald.h:36-51), phases in half turns
  const double u = 2.0 / cyc, scale = M_PI * u;
  for (int i = tid; i < nw; i += NT) {
    const Wave wv = waves[i];
#pragma unroll
    for (int k = 0; k < kEwaldTargets; k++) {
      double sn, cs;
      sincospi(wv.K[0] * (x[k] * u) + wv.K[1] * (y[k] * u) + wv.K[2] * (z[k] * u), &sn, &cs);
      const double dt = (wv.re * sn - wv.im * cs) * scale;
      acc[k][0] += wv.re * cs + wv.im * sn;
      for (int d = 0; d < 3; d++) acc[k][1 + d] -= dt * wv.K[d];
    }
  }
  // real part (3dp/ewald.h:82-102), nearest image of each pair
  const double a2 = alpha * alpha, a3 = a2 * alpha, c2 = cutoff * cutoff, half = cyc / 2;
  const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;
  // one cycle back towards zero beyond half a cycle
  auto nearest = [&](double d) { return d - (fabs(d) > half ? copysign(cyc, d) : 0.0); };
  auto evaluate = [&](int k, int at) {
    const EwaldQueue &Q = queues[w * kEwaldTargets + k];
    const double dx = Q.x[at], dy = Q.y[at], dz = Q.z[at], q = Q.q[at];
    double pot, grad;
    ewald_pair((dx * dx + dy * dy + dz * dz) * a2, pot, grad);
    acc[k][0] += q * pot * alpha;
    const double f = q * grad * a3;
    acc[k][1] -= dx * f;
    acc[k][2] -= dy * f;
    acc[k][3] -= dz * f;
  };
  const int64_t rounds = (ns + NT - 1) / NT;
  for (int64_t r = 0; r < rounds; r++) {
    const int64_t j = r * NT + tid;
    const bool in = j < ns;
    const exafmm_body *b = s + (in ? j : 0);
    const double sx = b->X[0], sy = b->X[1], sz = b->X[2], q = b->q;
#pragma unroll
    for (int k = 0; k < kEwaldTargets; k++) {
      const double dx = nearest(x[k] - sx), dy = nearest(y[k] - sy), dz = nearest(z[k] - sz);
      const double R2 = dx * dx + dy * dy + dz * dz;
      const bool hit = in && 0 < R2 && R2 < c2;
      const unsigned long long mask = __ballot(hit);
      EwaldQueue &Q = queues[w * kEwaldTargets + k];
      if (hit) {
        const int at = fill[k] + __popcll(mask & below);
        Q.x[at] = dx;
        Q.y[at] = dy;
        Q.z[at] = dz;
        Q.q[at] = q;
      }
      fill[k] += __popcll(mask);
      if (fill[k] >= kWave) {  // uniform: a full wave of pairs from the top
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        fill[k] -= kWave;
        evaluate(k, fill[k] + lane);
        __builtin_amdgcn_wave_barrier();
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int k = 0; k < kEwaldTargets; k++)
    if (lane < fill[k]) evaluate(k, lane);
#pragma unroll
  for (int k = 0; k < kEwaldTargets; k++)
#pragma unroll
    for (int c = 0; c < 4; c++) {
      double v = acc[k][c];
#pragma unroll
      for (int m = 1; m < kWave; m <<= 1) v += __shfl_xor(v, m);
      if (lane == 0) red[w][k][c] = v;
    }
  __syncthreads();
  if (tid >= 4 * kEwaldTargets) return;
  const int k = tid / 4, c = tid % 4;
  if (t0 + k >= nt) return;
  double v = 0.0;
  for (int i = 0; i < W; i++) v += red[i][k][c];
  exafmm_body *b = t + t0 + k;
  if (c == 0)
    b->p += v - M_2_SQRTPI * b->q * alpha;  // self term (3dp/ewald.h:146-150)
  else
    b->F[c - 1] += v;
}

static void ewald_launch(Ctx &c, Wave *w, int nw, int ksize, exafmm_body *t, int64_t nt, const exafmm_body *s,
                         int64_t ns, double alpha, double sigma, double cutoff, double cyc) {
  const double coef = 2 / sigma / cyc / cyc / cyc;
  const double coef2 = 1 / (4 * alpha * alpha);
  if (nw) {
    hipLaunchKernelGGL(k_ewald_dft, dim3((ksize + 1) * (2 * ksize + 1), ksize / kEwaldRun + 1), dim3(kEwaldThreads), 0,
                       c.s0, ksize, w, s, ns, cyc, coef, coef2);
    XF_LAUNCH();
  }
  if (nt) {
    const int waves = nt <= kEwaldManyTargets ? 8 : std::max<int64_t>(ns, nw) > kEwaldFew ? 4 : 1;
    auto *k = waves == 8 ? &k_ewald_target<8> : waves == 4 ? &k_ewald_target<4> : &k_ewald_target<1>;
    const size_t lds = sizeof(EwaldQueue) * waves * kEwaldTargets;
    XF_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
    hipLaunchKernelGGL(k, dim3(ceil_div(nt, kEwaldTargets)), dim3(waves * kWave), lds, c.s0, nw, w, t, nt, s, ns, alpha,
                       cutoff, cyc);
    XF_LAUNCH();
  }
  XF_HIP(hipStreamSynchronize(c.s0));
}

void ewald_sum(Ctx &c, exafmm_body *t, int64_t nt, const exafmm_body *s, int64_t ns, int ksize, double alpha,
               double sigma, double cutoff, double cyc) {
  static_assert(sizeof(Wave) == 5 * sizeof(double), "the wave table is held as doubles");
  const int nw = ewald_wave_count(ksize);
  c.ewald_waves.ensure(size_t(5) * std::max(nw, 1));
  ewald_launch(c, reinterpret_cast<Wave *>(c.ewald_waves.p), nw, ksize, t, nt, s, ns, alpha, sigma, cutoff, cyc);
}

// ---------------------------------------------------------------- Ewald without allocation
// The wave table of exafmm_ewald_noalloc lives in this fixed device array
// (one copy per GPU, kept until the process ends).  Host code never passes
// the array's name to a kernel: it uses the address hipGetSymbolAddress
// returned for the current device (ewald_scratch).
static __device__ __align__(256) Wave scratch[kEwaldMaxWaves];

namespace {
std::mutex g_scratch_mu;
Wave *g_scratch_ptr[kMaxDevices] = {};
}  // namespace

void ewald_scratch_init(int device) {
  if (device < 0 || device >= kMaxDevices) fail(EXAFMM_ERR_ARG, "device ordinal beyond the scratch table");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[device]) return;
  void *p = nullptr;
  XF_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  g_scratch_ptr[device] = static_cast<Wave *>(p);
}

static Wave *ewald_scratch(int device) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  Wave *p = (device >= 0 && device < kMaxDevices) ? g_scratch_ptr[device] : nullptr;
  if (!p) fail(EXAFMM_ERR_STATE, "scratch of the device not initialised (no context created on it)");
  return p;
}

void ewald_sum_noalloc(Ctx &c, exafmm_body *t, int64_t nt, const exafmm_body *s, int64_t ns, int ksize,
                       double alpha, double sigma, double cutoff, double cyc) {
  const int nw = ewald_wave_count(ksize);
  if (nw > kEwaldMaxWaves)
    fail(EXAFMM_ERR_CAPACITY, "ksize " + std::to_string(ksize) + " needs " + std::to_string(nw) +
                                  " waves; the allocation-free Ewald sum holds at most " +
                                  std::to_string(kEwaldMaxWaves));
  Wave *w = ewald_scratch(c.cfg.device);
  ewald_launch(c, w, nw, ksize, t, nt, s, ns, alpha, sigma, cutoff, cyc);
}

}  // namespace xf
