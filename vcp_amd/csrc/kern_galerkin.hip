// Galerkin matrix producer: Legendre_Bases_Generator::uhphiphi
// (vcp/ldbase.hpp:955-1013) in interval arithmetic,
//   A(i, j) = sum over points k of ((w_k * u_k) * phi(i, k)) * phi(j, k),
// i <= j accumulated from [0, 0] in k order and mirrored to A(j, i).  Each
// product and each sum is a separately rounded interval operation (kv's
// interval *, +): a product's lower end is the smallest of the four
// downward-rounded endpoint products, its upper end the largest of the four
// upward-rounded ones.  The kernel runs in round-toward-+inf and carries
// lower ends negated (RD(x) = -RU(-x)).
//
// Tiles of the upper triangle (tiles on the diagonal write their upper part and
// its mirror), 16 points per LDS stage, two stages.  The row operand is
// s(i, k) = (w_k * u_k) * phi(i, k), formed while staging; the column operand
// is phi(j, k).  Both come from the column-major phi (m x npts), so each stage
// reads 16 contiguous columns.
#include "vcphip_device.h"
#include "vcphip_kernels.h"

namespace {

constexpr int BK = 16, NT = 256, TM = 2, BM = 16 * TM;

// interval product in round-up mode: returns {-lower, upper}
VCPHIP_DEVINL double2 imul_neg(double al, double au, double bl, double bu) {
  const double up = __builtin_fmax(__builtin_fmax(al * bl, al * bu), __builtin_fmax(au * bl, au * bu));
  const double nlo = __builtin_fmax(__builtin_fmax((-al) * bl, (-al) * bu), __builtin_fmax((-au) * bl, (-au) * bu));
  return make_double2(nlo, up);
}

// An interval operand of the inner products takes the two-product form
// below when it is finite and lies strictly on one side of zero (lo > 0 or
// hi < 0); padding elements (outside the matrix or past the last point)
// are [0, 0] in both forms.
VCPHIP_DEVINL bool sign_definite(double lo, double hi) {
  return (lo > 0.0 || hi < 0.0) && __builtin_fabs(lo) < __builtin_inf() && __builtin_fabs(hi) < __builtin_inf();
}

// A 16 x 16 thread grid, 2 x 2 outputs per thread: thread (tx, ty) holds rows
// 2 ty, 2 ty + 1 and columns tx, tx + 16 of its tile, so that a wave reads the
// column operands of a point from consecutive 16-byte LDS slots (no bank
// conflicts) and the row operands as broadcasts.  FP64 issue bounds it: 8
// instructions per output and point in the two-product form, 512 of the 646
// per wave and stage.  A stage costs one barrier: two LDS stages, w_k u_k taken
// once per point instead of per element, a point's operands read during the
// arithmetic of the one before, and marks per point, so that a point where
// some operand holds zero does not send its whole stage through the general
// form.  The next stage's loads must be global ones (a zero by address, in place
// of a value, in the bounds checks made them FLAT, which the arithmetic then
// waited for: 400 at 1600 points 249 against 232 us, 100 at 400 63 against 58,
// one context).  Against two barriers and a mark per stage, 64 x 64 tiles from
// m = 2817 on (three contexts in turn / one): m = 400 at 1600 points 103 / 232
// against 118 / 276 us, 400 at 1681 109 / 245 against 125 / 292, 900 at 3600
// 522 / 717 against 570 / 827, 3025 at 3600 5.70 / 5.68 against 5.56 / 6.42 ms.
// Wider thread tiles (4 x 2, 4 x 4) leave the chip short of waves up to m =
// 1600 (3.3 against 3.0 ms) and tie at 3025.
__global__ __launch_bounds__(NT, 2) void k_uhphiphi(int m, int npts, const double* __restrict__ phi, long ldp,
                                                    const double* __restrict__ w, const double* __restrict__ u,
                                                    double* __restrict__ A, long lda) {
  constexpr int NQ = BM * BK / NT;   // staged elements of each side per thread
  static_assert(BM * BK % NT == 0 && BM == 16 * TM && NT == 256, "tile shape");
  vcphip_mode_round_up();
  // s(i, k) and phi(j, k) as {end of smaller magnitude, end of larger magnitude}
  __shared__ double2 sS[2][BK][BM + 1], sP[2][BK][BM + 1];
  __shared__ double2 sV[2][BK];   // w_k * u_k as {-lower, upper}, a stage ahead
  // marks the points of a stage with an operand outside the two-product form:
  // the stage in work, the next one (being stored), the one being cleared
  __shared__ int s_bad[3][BK];
  // upper-triangle tile t -> (tm, tn), tm <= tn
  const int nt = (m + BM - 1) / BM;
  int t = blockIdx.x, tm = 0;
  while (t >= nt - tm) {
    t -= nt - tm;
    ++tm;
  }
  const int row0 = tm * BM, col0 = (tm + t) * BM;
  const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
  double up[TM][TM], dn[TM][TM];   // dn = -(lower end)
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      up[i][j] = 0.0;
      dn[i][j] = -0.0;
    }
  // stage k0 in registers: the global loads of the next stage are issued
  // before the current stage's arithmetic and stored to LDS after it
  double2 ga[NQ], gb[NQ];
  auto load_stage = [&](int k0) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int e = tid + NT * q, r = e % BM, k = k0 + e / BM;
      ga[q] = (k < npts && row0 + r < m) ? *reinterpret_cast<const double2*>(phi + 2 * (row0 + r + ldp * k)) : make_double2(0.0, 0.0);
      gb[q] = (k < npts && col0 + r < m) ? *reinterpret_cast<const double2*>(phi + 2 * (col0 + r + ldp * k)) : make_double2(0.0, 0.0);
    }
  };
  auto store_v = [&](int k0, int st) {
    const int k = k0 + tid;
    if (tid < BK && k < npts) {
      const double2 wk = *reinterpret_cast<const double2*>(w + 2 * k), uk = *reinterpret_cast<const double2*>(u + 2 * k);
      sV[st][tid] = imul_neg(wk.x, wk.y, uk.x, uk.y);
    }
  };
  // a negative interval's end of smaller magnitude is its upper end
  auto small_large = [](double lo, double hi) { return hi < 0.0 ? make_double2(hi, lo) : make_double2(lo, hi); };
  auto ends = [](const double2& v) { return v.y < 0.0 ? make_double2(v.y, v.x) : v; };   // its inverse
  // stores stage k0 and notes the points whose elements do not all take the
  // two-product form
  auto store_stage = [&](int k0, int st, int (&bad)[BK]) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int e = tid + NT * q, r = e % BM, kl = e / BM;
      double2 sv = make_double2(-0.0, 0.0);
      if (k0 + kl < npts && row0 + r < m) {
        const double2 v = sV[st][kl];
        sv = imul_neg(-v.x, v.y, ga[q].x, ga[q].y);   // (w_k u_k) * phi(i, k)
        if (!sign_definite(-sv.x, sv.y)) bad[kl] = 1;
      }
      if (k0 + kl < npts && col0 + r < m && !sign_definite(gb[q].x, gb[q].y)) bad[kl] = 1;
      sS[st][kl][r] = small_large(-sv.x, sv.y);
      sP[st][kl][r] = small_large(gb[q].x, gb[q].y);
    }
  };
  if (tid < 3 * BK) s_bad[tid / BK][tid % BK] = 0;
  if (npts > 0) {
    load_stage(0);
    store_v(0, 0);
    store_v(BK, 1);
    __syncthreads();
    store_stage(0, 0, s_bad[0]);
  }
  __syncthreads();
  double2 fa[2][TM], fb[2][TM];
  auto read = [&](int st, int kk, int f) {
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[f][i] = sS[st][kk][ty * TM + i];
#pragma unroll
    for (int j = 0; j < TM; ++j) fb[f][j] = sP[st][kk][tx + 16 * j];
  };
  // s(i, k) * phi(j, k) for operands strictly on one side of zero: with
  // a, A the ends of s of smaller and larger magnitude and b, B those of
  // phi, the exact product's ends are a b and A B (both of the sign of
  // the product), so its rounded ends are max(RU(a b), RU(A B)) and
  // -max(RU(-a b), RU(-A B)): four products instead of eight and no
  // comparisons of products, with the bits of imul_neg (rounding is
  // monotone, and four products of one sign give no +0 / -0 ties)
  auto two_product = [&](const double2 (&a)[TM], const double2 (&b)[TM]) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      // a row's products first, then their maxima and sums: independent
      // products in flight instead of one mul-max-add chain at a time
      double pu[TM][2], pd[TM][2];
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        pu[j][0] = a[i].x * b[j].x;
        pu[j][1] = a[i].y * b[j].y;
        pd[j][0] = (-a[i].x) * b[j].x;
        pd[j][1] = (-a[i].y) * b[j].y;
      }
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        up[i][j] = up[i][j] + __builtin_fmax(pu[j][0], pu[j][1]);
        dn[i][j] = dn[i][j] + __builtin_fmax(pd[j][0], pd[j][1]);
      }
    }
  };
  for (int k0 = 0, st = 0, sl = 0; k0 < npts; k0 += BK, st ^= 1) {
    const bool more = k0 + BK < npts;
    if (more) load_stage(k0 + BK);
    const unsigned long long bad = __builtin_amdgcn_ballot_w64((tid & 63) < BK && s_bad[sl][tid % BK] != 0);
    sl = sl == 2 ? 0 : sl + 1;
    if (tid < BK) s_bad[sl == 2 ? 0 : sl + 1][tid] = 0;   // the slot of the stage before this one
    if (!bad) {
      read(st, 0, 0);
#pragma unroll
      for (int kk = 0; kk < BK; ++kk) {
        // the next point's operands are on their way during this one's arithmetic
        if (kk + 1 < BK) read(st, kk + 1, (kk + 1) & 1);
        __builtin_amdgcn_sched_barrier(0);
        two_product(fa[kk & 1], fb[kk & 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll 1
      for (int kk = 0; kk < BK; ++kk) {
        read(st, kk, 0);
        if (!(bad >> kk & 1)) {
          two_product(fa[0], fb[0]);
          continue;
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[0][i] = ends(fa[0][i]);
#pragma unroll
        for (int j = 0; j < TM; ++j) fb[0][j] = ends(fb[0][j]);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j) {
            const double2 p = imul_neg(fa[0][i].x, fa[0][i].y, fb[0][j].x, fb[0][j].y);   // s(i, k) * phi(j, k)
            up[i][j] = up[i][j] + p.y;
            dn[i][j] = dn[i][j] + p.x;
          }
      }
    }
    if (more) {
      store_stage(k0 + BK, st ^ 1, s_bad[sl]);
      store_v(k0 + 2 * BK, st);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const int r = row0 + ty * TM + i, c = col0 + tx + 16 * j;
      if (r < m && c < m && r <= c) {
        const double2 val = make_double2(-dn[i][j], up[i][j]);
        *reinterpret_cast<double2*>(A + 2 * (r + lda * (long)c)) = val;
        *reinterpret_cast<double2*>(A + 2 * (c + lda * (long)r)) = val;
      }
    }
}

}  // namespace

int vcphip_launch_uhphiphi(int m, int npts, const double* phi, long ldp, const double* w, const double* u, double* A,
                           long lda, hipStream_t s) {
  if (m <= 0) return 0;
  const int nt = (m + BM - 1) / BM;
  hipLaunchKernelGGL(k_uhphiphi, dim3(nt * (nt + 1) / 2), dim3(NT), 0, s, m, npts, phi, ldp, w, u, A, lda);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
