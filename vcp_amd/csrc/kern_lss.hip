// Verified linear solve around R*A - I (imats::linearsolve,
// vcp/imats.hpp:292-362): every step but the product R*A (the PI form of
// k_drgemm_planes, or the batched residual's tiles).  R*mid(b), A*mx - b,
// |R*x|, the row sums of |RA - I| and |RA - I| * T with the final enclosure
// are products with few columns, in the row-serial form of vcphip_thin.h:
// each reads its matrix once, and a step's elementwise work (midpoints, the
// subtraction of b, absolute values, the unit diagonal, the enclosure) is in
// its operand conversions and its epilogue.  The host drives the sequence
// (vcphip_lss_dev, vcphip_lss_batched_dev in vcphip_host.hip).
//
// Kernels that need directed rounding run in round-toward-+inf (see
// vcphip_device.h) and form RD(x) = -RU(-x).  The R*mid(b) kernels and the
// scalar G run in the default round-to-nearest mode: the midpoint and
// R*mid(b) are nearest-rounded in the reference (no rounding mode is set
// around them), and G = T / (1 - ||RA - I||) gets its directed roundings from
// exact error terms of nearest-rounded operations.
#include "vcphip_device.h"
#include "vcphip_kernels.h"
#include "vcphip_thin.h"

namespace {

constexpr int NT = 256;

// kv's mid(): the nearest-rounded average, (lo + hi) / 2, or lo/2 + hi/2
// where lo + hi overflows; point intervals give lo.  Round-to-nearest mode.
VCPHIP_DEVINL double lss_mid(double2 v) {
  if (v.x == v.y) return v.x;
  const double s = v.x + v.y;
  return __builtin_isinf(s) ? 0.5 * v.x + 0.5 * v.y : s * 0.5;
}

// kv's abs() of an interval (imats.hpp:315, :338): exact
VCPHIP_DEVINL double2 lss_abs(double2 v) {
  if (v.x >= 0.0) return v;
  if (v.y <= 0.0) return make_double2(-v.y, -v.x);
  return make_double2(0.0, -v.x > v.y ? -v.x : v.y);
}

// b(i, i) -= 1 in interval arithmetic (imats.hpp:324-326), round-up mode
VCPHIP_DEVINL double2 lss_minus_one(double2 v) { return make_double2(-(1.0 - v.x), v.y - 1.0); }

// The midpoint matrix M of IA (n x n, as lss_mid) bordered by the identity
// to order npad: P = [[M, 0], [0, I]], whose inverse is [[inv(M), 0], [0, I]].
// In LU with partial pivoting the border rows keep zeros in M's columns
// (their multipliers are 0), so no pivot is taken from them and a singular M
// still meets a zero pivot.  n = 0 writes the identity (IA is not read).
__global__ __launch_bounds__(NT) void k_inv_pad(int n, int npad, const double* __restrict__ IA, long lda,
                                                double* __restrict__ P) {
  const long idx = (long)blockIdx.x * NT + threadIdx.x;
  if (idx >= (long)npad * npad) return;
  const int i = (int)(idx % npad), j = (int)(idx / npad);
  double m;
  if (i < n && j < n) {
    m = lss_mid(*reinterpret_cast<const double2*>(IA + 2 * (i + lda * j)));
  } else {
    m = (i == j) ? 1.0 : 0.0;
  }
  P[idx] = m;
}

// R(0:n, 0:n) = P(0:n, 0:n)
__global__ __launch_bounds__(NT) void k_copy_block(int n, const double* __restrict__ P, long ldp,
                                                   double* __restrict__ R, long ldr) {
  const long idx = (long)blockIdx.x * NT + threadIdx.x;
  if (idx >= (long)n * n) return;
  const int i = (int)(idx % n), j = (int)(idx / n);
  R[i + ldr * j] = P[i + ldp * j];
}

// X = X - b (interval subtraction, imats.hpp:308): [RD(xl - bu), RU(xu - bl)]
__global__ __launch_bounds__(NT) void k_lss_sub(int n, int ncol, double* __restrict__ X, long ldx,
                                                const double* __restrict__ b, long ldb) {
  vcphip_mode_round_up();
  const long idx = (long)blockIdx.x * NT + threadIdx.x;
  if (idx >= (long)n * ncol) return;
  const int i = (int)(idx % n), j = (int)(idx / n);
  double2* x = reinterpret_cast<double2*>(X + 2 * (i + ldx * j));
  const double2 bv = *reinterpret_cast<const double2*>(b + 2 * (i + ldb * j));
  const double2 xv = *x;
  *x = make_double2(-(bv.y - xv.x), xv.y - bv.x);
}

// kv's abs() of an interval matrix, in place
__global__ __launch_bounds__(NT) void k_lss_abs(int rows, int cols, double* __restrict__ X, long ldx) {
  const long idx = (long)blockIdx.x * NT + threadIdx.x;
  if (idx >= (long)rows * cols) return;
  const int i = (int)(idx % rows), j = (int)(idx / rows);
  double2* x = reinterpret_cast<double2*>(X + 2 * (i + ldx * j));
  *x = lss_abs(*x);
}

// ---- directed roundings from nearest-rounded operations --------------------
// next double above / below x for finite x >= 0 (x > 0 for below)
VCPHIP_DEVINL double next_up_nn(double x) { return __longlong_as_double(__double_as_longlong(x) + 1); }
VCPHIP_DEVINL double next_dn_pos(double x) { return __longlong_as_double(__double_as_longlong(x) - 1); }

// RD and RU of t / d for t >= 0 and 2^-960 <= d (here d is 1 - g with
// 0 <= g < 1, so d >= 2^-53).  q = RN(t / d); when t >= 2^-960 the
// remainder t - q d is a double and the FMA gives it exactly, and its sign
// says on which side of q the quotient lies.  Smaller t is scaled by 2^128
// first; scaling the directed results back by 2^-128 is then corrected to
// the same direction (the scaled-back product is exact unless it is
// subnormal, and multiplying it by 2^128 again is always exact).
VCPHIP_DEVINL void div_dir_core(double t, double d, double& dn, double& up) {
  const double q = t / d;
  const double r = __builtin_fma(-q, d, t);
  up = r > 0.0 ? next_up_nn(q) : q;
  dn = (r < 0.0 && q > 0.0) ? next_dn_pos(q) : q;
}

VCPHIP_DEVINL void div_dir(double t, double d, double& dn, double& up) {
  const double tiny = vcphip_pow2(-960);
  if (!(t < tiny)) {   // also t = inf or NaN: q carries it through
    div_dir_core(t, d, dn, up);
    return;
  }
  double sdn, sup;
  div_dir_core(t * vcphip_pow2(128), d, sdn, sup);
  const double s = vcphip_pow2(-128), S = vcphip_pow2(128);
  up = sup * s;
  if (up * S < sup) up = next_up_nn(up);
  dn = sdn * s;
  if (dn * S > sdn) dn = next_dn_pos(dn);
}

// 1 - g rounded down and up (TwoSum: the error of s = RN(1 - g) is exact)
VCPHIP_DEVINL void one_minus_dir(double g, double& dn, double& up) {
  const double a = 1.0, b = -g;
  const double s = a + b;
  const double bb = s - a;
  const double e = (a - (s - bb)) + (b - bb);
  up = e > 0.0 ? next_up_nn(s) : s;
  dn = e < 0.0 ? next_dn_pos(s) : s;
}

// G = T / (1 - g) as an interval (imats.hpp:341; g is ||RA - I|| with its
// lower end set to its upper end, T likewise).  When g >= 1 (verification
// failed) or g is NaN, G is [NaN, NaN].  Round-to-nearest mode.
VCPHIP_DEVINL double2 lss_bound_factor(double g, double t) {
  if (!(g < 1.0)) return make_double2(__builtin_nan(""), __builtin_nan(""));
  double ddn, dup, lo, a, b, hi;
  one_minus_dir(g, ddn, dup);
  div_dir(t, dup, lo, a);   // lower end: RD(t / RU(1 - g))
  div_dir(t, ddn, b, hi);   // upper end: RU(t / RD(1 - g))
  return make_double2(lo, hi);
}

inline dim3 grid_of(long count) { return dim3((unsigned)((count + NT - 1) / NT)); }

// ===========================================================================
// The steps of one system (P), as row-serial products: the chains and
// epilogues are those of the product tiles (k ascending, midrad on load, the
// same fused operations in the same order), so the single and the batched
// form give the same bits.
// ===========================================================================

// mx = R mid(b): nearest rounding, each element the k-ascending FMA chain
// from 0 (the rmatmul contract with nearest rounding, vblas/README.md:167-170)
struct LssMx {
  static constexpr bool A2 = false, B2 = true, PAD16 = false;
  static constexpr int AL = 1, BL = 1;
  const double* A;
  const double* B;
  long lda, ldb;
  double* mx;
  int n;
  struct Acc {
    double s;
  };
  VCPHIP_DEVINL explicit LssMx(const VcphipLssProblem& P)
      : A(P.R), B(P.b), lda(P.ldr), ldb(P.ldb), mx(P.mx), n(P.n) {}
  VCPHIP_DEVINL double2 a(double2 v, int, int) const { return v; }
  VCPHIP_DEVINL double2 b(double2 v) const { return make_double2(lss_mid(v), 0.0); }
  VCPHIP_DEVINL void init(Acc& c, int, int) const { c.s = 0.0; }
  VCPHIP_DEVINL void step(Acc& c, double2 av, double2 bv) const { c.s = __builtin_fma(av.x, bv.x, c.s); }
  VCPHIP_DEVINL void done(const Acc& c, int row, int col) const { mx[row + (long)n * col] = c.s; }
};

// x = IA mx - b (imats.hpp:305-308): [RD(xl - bu), RU(xu - bl)]
struct LssAx : VcphipThinDr<true, false> {
  const double* rhs;
  double* xi;
  long ldrhs;
  int n;
  VCPHIP_DEVINL explicit LssAx(const VcphipLssProblem& P) : rhs(P.b), xi(P.xi), ldrhs(P.ldb), n(P.n) {
    A = P.A;
    B = P.mx;
    lda = P.lda;
    ldb = P.n;
  }
  VCPHIP_DEVINL void done(const Acc& c, int row, int col) const {
    const double2 x = result(c);
    const double2 bv = *reinterpret_cast<const double2*>(rhs + 2 * (row + ldrhs * col));
    *reinterpret_cast<double2*>(xi + 2 * (row + (long)n * col)) = make_double2(-(bv.y - x.x), x.y - bv.x);
  }
};

// y = |R x| (imats.hpp:311-315)
struct LssRy : VcphipThinDr<false, true> {
  double* y;
  int n;
  VCPHIP_DEVINL explicit LssRy(const VcphipLssProblem& P) : y(P.y), n(P.n) {
    A = P.R;
    B = P.xi;
    lda = P.ldr;
    ldb = P.n;
  }
  VCPHIP_DEVINL void done(const Acc& c, int row, int col) const {
    *reinterpret_cast<double2*>(y + 2 * (row + (long)n * col)) = lss_abs(result(c));
  }
};

// upper end of the row sums of |RA - I| (mats::norminf, vcp/mats.hpp:
// 1587-1592): s = mag(c_i0), then s = RU(s + mag(c_ij)) for j = 1, 2, ...
// DIAG: C holds R A, and the unit diagonal is subtracted on load
template <bool DIAG>
struct LssRowSum {
  static constexpr bool A2 = true, B2 = false, PAD16 = false;
  static constexpr int AL = 1, BL = 0;
  const double* A;
  const double* B = nullptr;
  long lda, ldb = 0;
  double* out;
  struct Acc {
    double s;
  };
  VCPHIP_DEVINL double2 a(double2 v, int row, int kk) const {
    if (DIAG && row == kk) v = lss_minus_one(v);
    const double p = __builtin_fabs(v.x), q = __builtin_fabs(v.y);
    return make_double2(p > q ? p : q, 0.0);
  }
  VCPHIP_DEVINL double2 b(double2 v) const { return v; }
  VCPHIP_DEVINL void init(Acc& c, int, int) const { c.s = 0.0; }
  VCPHIP_DEVINL void step(Acc& c, double2 av, double2) const { c.s = c.s + av.x; }
  VCPHIP_DEVINL void done(const Acc& c, int row, int) const { out[row] = c.s; }
};

// W = |RA - I| G (the II product with the constant column G, one column for
// all right-hand sides; its lower chain is not used) and X = mx + [-u, u],
// u = RU(|y|u + Wu) (imats.hpp:343-361).  The eight column lanes carry the
// same chain and share a group of right-hand sides, a workgroup per row block
// and group: one group for all of them left 8 rows x nrhs steps to one wave (a
// whole solve of n = 64 with 4096 right-hand sides 1151 us; 118 with groups and
// the row sums of |y| spread over workgroups, 2000 with 2000 11.4 and 4.2 ms).
// DIAG: C holds R A, and the unit diagonal is subtracted on load.
__host__ __device__ inline int lss_final_group(int n) { return n > 256 ? n / 4 / 8 * 8 : 64; }   // right-hand sides of a group

template <bool DIAG>
struct LssFinal {
  static constexpr bool A2 = true, B2 = false, PAD16 = false;
  static constexpr int AL = 2, BL = 0;
  const double* A;
  const double* B = nullptr;
  long lda, ldb = 0;
  const double *y, *mx;
  double* X;
  long ldx;
  int n, j0, j1;
  double bm, br;
  struct Acc {
    double up, r1, r2;
  };
  VCPHIP_DEVINL LssFinal(const VcphipLssProblem& P, int group)
      : A(P.C), lda(P.n), y(P.y), mx(P.mx), X(P.X), ldx(P.ldx), n(P.n), j0(group * lss_final_group(P.n)) {
    const int left = P.nrhs - j0;
    j1 = j0 + (left < lss_final_group(n) ? left : lss_final_group(n));
    vcphip_midrad_ru(P.norms[2], P.norms[3], bm, br);
  }
  VCPHIP_DEVINL double2 a(double2 v, int row, int kk) const {
    if (DIAG && row == kk) v = lss_minus_one(v);
    v = lss_abs(v);
    double mm, rr;
    vcphip_midrad_ru(v.x, v.y, mm, rr);
    return make_double2(mm, rr);
  }
  VCPHIP_DEVINL double2 b(double2 v) const { return v; }
  VCPHIP_DEVINL void init(Acc& c, int, int) const { c.up = c.r1 = c.r2 = 0.0; }
  VCPHIP_DEVINL void step(Acc& c, double2 av, double2) const {
    c.up = __builtin_fma(av.x, bm, c.up);
    const double as = __builtin_fabs(av.x) + av.y;
    c.r1 = __builtin_fma(as, br, c.r1);
    c.r2 = __builtin_fma(av.y, __builtin_fabs(bm), c.r2);
  }
  VCPHIP_DEVINL void done(const Acc& c, int row, int col) const {
    const double wu = c.up + (c.r1 + c.r2);
    const double *__restrict__ yr = y + 2 * row + 1, *__restrict__ mr = mx + row;
    double* __restrict__ xr = X + 2 * row;
#pragma unroll 4
    for (int j = j0 + col; j < j1; j += VCPHIP_THIN_CL) {
      const double u = yr[2 * (long)n * j] + wu, m = mr[(long)n * j];
      *reinterpret_cast<double2*>(xr + 2 * ldx * j) = make_double2(-(u - m), u + m);
    }
  }
};

// T = ||y||_inf: upward row sums over the columns, then their maximum, by one
// workgroup of NT threads (batched form)
VCPHIP_DEVINL double lss_ynorm(const VcphipLssProblem& P, double* red, double* first) {   // round-up mode
  double best = -__builtin_inf();
  for (int i = threadIdx.x; i < P.n; i += NT) {
    double s = 0.0;
    for (int j = 0; j < P.nrhs; ++j) {
      const double2 v = *reinterpret_cast<const double2*>(P.y + 2 * (i + (long)P.n * j));
      const double a = __builtin_fabs(v.x), b = __builtin_fabs(v.y);
      const double mag = a > b ? a : b;
      s = (j == 0) ? mag : s + mag;
    }
    if (i == 0) *first = s;
    best = s > best ? s : best;
  }
  __syncthreads();
  return vcphip_block_max<NT>(best, *first, red);
}

// ---- one system ---------------------------------------------------------------
template <class Op, int CW, int CPT, bool UP>
__global__ __launch_bounds__((VcphipThin<Op, CW, CPT>::NT)) VCPHIP_THIN_WAVES
void k_lss_step(VcphipLssProblem P) {
  if (UP) vcphip_mode_round_up();
  using T = VcphipThin<Op, CW, CPT>;
  __shared__ __attribute__((aligned(16))) typename T::Lds lds;
  Op op(P);
  const int rb = vcphip_xcd_remap(blockIdx.x, gridDim.x);
  T::run(op, lds, P.n, P.nrhs, P.n, rb * T::R, blockIdx.y * T::NC, (int)((blockIdx.x >> 8) % T::NW));
}

// the row sums of |RA - I| into rows[0, n) and those of |y| into rows[n, 2n),
// row blocks of the one, then of the other
__global__ __launch_bounds__((VcphipThin<LssRowSum<true>, 1>::NT)) VCPHIP_THIN_WAVES
void k_lss_rowsum(VcphipLssProblem P, double* __restrict__ rows) {
  vcphip_mode_round_up();
  using T = VcphipThin<LssRowSum<true>, 1>;
  using Y = VcphipThin<LssRowSum<false>, 1>;
  __shared__ __attribute__((aligned(16))) typename T::Lds lds;
  static_assert(sizeof(T::Lds) == sizeof(Y::Lds), "one buffer for both");
  const int nrb = gridDim.x / 2, rot = (int)((blockIdx.x >> 8) % T::NW);
  if ((int)blockIdx.x < nrb) {
    LssRowSum<true> op;
    op.A = P.C;
    op.lda = P.n;
    op.out = rows;
    T::run(op, lds, P.n, 1, P.n, vcphip_xcd_remap(blockIdx.x, nrb) * T::R, 0, rot);
  } else {
    LssRowSum<false> op;
    op.A = P.y;
    op.lda = P.n;
    op.out = rows + P.n;
    Y::run(op, reinterpret_cast<typename Y::Lds&>(lds), P.n, 1, P.nrhs, ((int)blockIdx.x - nrb) * Y::R, 0, rot);
  }
}

// g = ||RA - I||_inf and T = ||y||_inf from their row sums, and G: norms[0 .. 3]
__global__ __launch_bounds__(NT) void k_lss_g(VcphipLssProblem P, const double* __restrict__ rows) {
  __shared__ double red[NT];
  double norm[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const double* in = rows + (long)h * P.n;
    double best = -__builtin_inf();
    for (int i = threadIdx.x; i < P.n; i += NT) {
      const double v = in[i];
      best = v > best ? v : best;
    }
    norm[h] = vcphip_block_max<NT>(best, in[0], red);
  }
  if (threadIdx.x == 0) {
    const double2 G = lss_bound_factor(norm[0], norm[1]);
    P.norms[0] = norm[0];
    P.norms[1] = norm[1];
    P.norms[2] = G.x;
    P.norms[3] = G.y;
  }
}

template <bool DIAG>
__global__ __launch_bounds__((VcphipThin<LssFinal<DIAG>, 1>::NT)) VCPHIP_THIN_WAVES
void k_lss_final(VcphipLssProblem P) {
  vcphip_mode_round_up();
  using T = VcphipThin<LssFinal<DIAG>, 1>;
  __shared__ __attribute__((aligned(16))) typename T::Lds lds;
  LssFinal<DIAG> op(P, blockIdx.y);
  const int rb = vcphip_xcd_remap(blockIdx.x, gridDim.x);
  T::run(op, lds, P.n, VCPHIP_THIN_CL, P.n, rb * T::R, 0, (int)((blockIdx.x >> 8) % T::NW));
}

// ---- many systems of uneven size -------------------------------------------------
// each stage one launch over the blocks (8 rows, 8 right-hand sides) of all
// problems: problem p's are [wb[p], wb[p + 1]), its row blocks first
VCPHIP_DEVINL int find_problem(const long* __restrict__ wb, int count, long blk) {
  int lo = 0, hi = count - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (wb[mid] <= blk) lo = mid; else hi = mid - 1;
  }
  return lo;
}

template <class Op, bool UP>
__global__ __launch_bounds__((VcphipThin<Op, 1>::NT)) VCPHIP_THIN_WAVES
void k_lssb_step(int count, const long* __restrict__ wb, const VcphipLssProblem* __restrict__ probs) {
  if (UP) vcphip_mode_round_up();
  using T = VcphipThin<Op, 1>;
  __shared__ __attribute__((aligned(16))) typename T::Lds lds;
  const long blk = vcphip_xcd_remap(blockIdx.x, gridDim.x);
  const int p = find_problem(wb, count, blk);
  const VcphipLssProblem P = probs[p];
  const int nrb = (P.n + T::R - 1) / T::R, q = (int)(blk - wb[p]);
  Op op(P);
  T::run(op, lds, P.n, P.nrhs, P.n, (q % nrb) * T::R, (q / nrb) * T::NC, (int)((blockIdx.x >> 8) % T::NW));
}

// T and G per problem (one workgroup each), into norms[1 .. 3]
__global__ __launch_bounds__(NT) void k_lssb_ynorm(const VcphipLssProblem* __restrict__ probs) {
  vcphip_mode_round_up();
  __shared__ double red[NT];
  __shared__ double first;
  const VcphipLssProblem P = probs[blockIdx.x];
  const double t = lss_ynorm(P, red, &first);
  if (threadIdx.x == 0) P.norms[1] = t;
}

__global__ __launch_bounds__(NT) void k_lssb_g(int count, const VcphipLssProblem* __restrict__ probs) {
  const int p = blockIdx.x * NT + threadIdx.x;
  if (p >= count) return;
  const VcphipLssProblem P = probs[p];
  const double2 G = lss_bound_factor(P.normub[0], P.norms[1]);
  P.norms[2] = G.x;
  P.norms[3] = G.y;
}

__global__ __launch_bounds__((VcphipThin<LssFinal<false>, 1>::NT)) VCPHIP_THIN_WAVES
void k_lssb_final(int count, const long* __restrict__ wb, const VcphipLssProblem* __restrict__ probs) {
  vcphip_mode_round_up();
  using T = VcphipThin<LssFinal<false>, 1>;
  __shared__ __attribute__((aligned(16))) typename T::Lds lds;
  const long blk = vcphip_xcd_remap(blockIdx.x, gridDim.x);
  const int p = find_problem(wb, count, blk);
  const VcphipLssProblem P = probs[p];
  const int nrb = (P.n + T::R - 1) / T::R, q = (int)(blk - wb[p]);
  const int per = lss_final_group(P.n) / VCPHIP_THIN_CL;   // blocks of 8 right-hand sides to a group
  if (q / nrb % per) return;   // the group's first block serves it
  LssFinal<false> op(P, q / nrb / per);
  T::run(op, lds, P.n, VCPHIP_THIN_CL, P.n, q % nrb * T::R, 0, (int)((blockIdx.x >> 8) % T::NW));
}

}  // namespace

int vcphip_inv_launch_pad(int n, int npad, const double* IA, long lda, double* P, hipStream_t s) {
  hipLaunchKernelGGL(k_inv_pad, grid_of((long)npad * npad), dim3(NT), 0, s, n, npad, IA, lda, P);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_inv_launch_copy(int n, const double* P, long ldp, double* R, long ldr, hipStream_t s) {
  hipLaunchKernelGGL(k_copy_block, grid_of((long)n * n), dim3(NT), 0, s, n, P, ldp, R, ldr);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_lss_launch_sub(int n, int ncol, double* X, long ldx, const double* b, long ldb, hipStream_t s) {
  hipLaunchKernelGGL(k_lss_sub, grid_of((long)n * ncol), dim3(NT), 0, s, n, ncol, X, ldx, b, ldb);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_lss_launch_abs(int rows, int cols, double* X, long ldx, hipStream_t s) {
  hipLaunchKernelGGL(k_lss_abs, grid_of((long)rows * cols), dim3(NT), 0, s, rows, cols, X, ldx);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

namespace {
// columns per workgroup: 8 up to 8 right-hand sides, 64 above, so that a row
// block of R or IA (64 n or 128 n bytes) is read once per 64 right-hand sides.
// (The single products narrow the 64 until about 150 workgroups run; here the
// step is a small part of the solve.)
template <class Op, bool UP>
void lss_step(const VcphipLssProblem& P, hipStream_t s) {
  const unsigned rb = (unsigned)((P.n + VCPHIP_THIN_R - 1) / VCPHIP_THIN_R);
  if (P.nrhs <= 8)
    hipLaunchKernelGGL((k_lss_step<Op, 1, 1, UP>), dim3(rb), dim3(VcphipThin<Op, 1, 1>::NT), 0, s, P);
  else
    hipLaunchKernelGGL((k_lss_step<Op, 4, 2, UP>), dim3(rb, (unsigned)((P.nrhs + 63) / 64)),
                       dim3(VcphipThin<Op, 4, 2>::NT), 0, s, P);
}
}  // namespace

int vcphip_lss_launch_mx(const VcphipLssProblem& P, hipStream_t s) {
  lss_step<LssMx, false>(P, s);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_lss_launch_ax(const VcphipLssProblem& P, hipStream_t s) {
  lss_step<LssAx, true>(P, s);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_lss_launch_ry(const VcphipLssProblem& P, hipStream_t s) {
  lss_step<LssRy, true>(P, s);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_lss_launch_bound(const VcphipLssProblem& P, double* rows, hipStream_t s) {
  const unsigned rb = (unsigned)((P.n + VCPHIP_THIN_R - 1) / VCPHIP_THIN_R);
  hipLaunchKernelGGL(k_lss_rowsum, dim3(2 * rb), dim3(VcphipThin<LssRowSum<true>, 1>::NT), 0, s, P, rows);
  hipLaunchKernelGGL(k_lss_g, dim3(1), dim3(NT), 0, s, P, rows);
  const int group = lss_final_group(P.n);
  hipLaunchKernelGGL(k_lss_final<true>, dim3(rb, (unsigned)(((long)P.nrhs + group - 1) / group)),
                     dim3(VcphipThin<LssFinal<true>, 1>::NT), 0, s, P);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_lss_launch_batched_rhs(int count, long blocks, const long* wb, const VcphipLssProblem* probs,
                                  hipStream_t s) {
  if (blocks > 0x7FFFFFFFL) return -7;
  const dim3 g((unsigned)blocks);
  hipLaunchKernelGGL((k_lssb_step<LssMx, false>), g, dim3(VcphipThin<LssMx, 1>::NT), 0, s, count, wb, probs);
  hipLaunchKernelGGL((k_lssb_step<LssAx, true>), g, dim3(VcphipThin<LssAx, 1>::NT), 0, s, count, wb, probs);
  hipLaunchKernelGGL((k_lssb_step<LssRy, true>), g, dim3(VcphipThin<LssRy, 1>::NT), 0, s, count, wb, probs);
  hipLaunchKernelGGL(k_lssb_ynorm, dim3(count), dim3(NT), 0, s, probs);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_lss_launch_batched_bound(int count, long blocks, const long* wb, const VcphipLssProblem* probs,
                                    hipStream_t s) {
  hipLaunchKernelGGL(k_lssb_g, grid_of(count), dim3(NT), 0, s, count, probs);
  hipLaunchKernelGGL(k_lssb_final, dim3((unsigned)blocks), dim3(VcphipThin<LssFinal<false>, 1>::NT), 0, s, count, wb,
                     probs);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
