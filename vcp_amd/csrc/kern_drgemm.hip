// Plain FP64 directed-rounding GEMM family (vector FMA, LDS-tiled, gfx950).
//
// The four products of the pidblas policy:
//   II  C = IA*IB        pidblas::mulmm     vcp/pidblas.hpp:239-294
//   IP  C = IA*B         pidblas::mul_im_m  vcp/pidblas.hpp:90-140
//   PI  C = B*IA         pidblas::mul_m_im  vcp/pidblas.hpp:142-196
//   PP  Cup, Cdn = A*B   rmatmul(+1/-1)     vblas/rmatmul.hpp:100-127,
//                        udmatmul           vblas/udmatmul.hpp:738-760
// Each output element carries the k-ascending chains of the reference's
// BLAS calls (the rmatmul contract, vblas/README.md:167-170) in registers:
//   up  = RU chain of mid(A)*mid(B)                       (:269-271)
//   dn  = RU chain of (-mid(A))*mid(B) = -(RD chain)      (:264-266)
//   r1  = RU chain of (|mid A|+rad A)*rad B               (:277-279)
//   r2  = RU chain of rad A*|mid B|                       (:281)
// and the epilogue applies the reference's fix-ups in its order
//   t = RU(r1 + r2); upper = RU(up + t); lower = RD(-dn - t) = -RU(dn + t).
// Three implementations share these chains: k_drgemm_planes (the single
// products), fed from midpoint-radius planes made once per operand; the tile
// function dr_tile (the batched launches), which reads the AoS {inf, sup}
// operands and converts them to midpoint-radius on their way into LDS
// (pidblas_assist::midrad, :43-60); and the row-serial k_drgemm_thin for few
// columns and small sizes (vcphip_thin.h).  The two tiled ones carry them as
// DPP multiply-adds (vcphip_dpp.h).  A single product of k = 0 is a fill.
//
// The whole kernel runs in round-toward-+inf (see vcphip_device.h).
#include "vcphip_device.h"
#include "vcphip_kernels.h"
#include "vcphip_thin.h"
#include "vcphip_dpp.h"

namespace {

constexpr int BM = 64, BN = 64, BK = 16;
constexpr int NT = 256;          // 4 waves
// the inf-sup tiles: thread (tx, ty) of 16 x 16 holds rows 4 ty .. 4 ty + 3 and
// columns tx + 16 j
constexpr int TM = 4, TN = 4;
constexpr int PAD = 2;           // doubles of row padding (keeps 16-byte alignment)
constexpr int LA = BM + PAD;     // LDS row length of an A k-slice
constexpr int LB = BN + PAD;
constexpr int A_PER_T = BM * BK / NT;   // 4 elements of A per thread per tile
constexpr int B_PER_T = BK * BN / NT;   // 4 elements of B per thread per tile

// LDS of the tile kernels: two slices of BKT k of A (rows) and B (columns),
// an element as its (mid, rad) pair (interval) or itself (point).  One
// instance per kernel, shared by every tile shape the kernel runs; a tile of
// 32 rows uses the first 32 elements of each A row.  The odd row stride
// spreads B's stores (16 lanes along k) over the banks.
template <bool AI, bool BI>
struct DrLds {
  static constexpr int BKT = AI && BI ? 8 : 16;   // k per slice
  static constexpr int AE = AI ? 2 : 1, BE = BI ? 2 : 1, LDR = BM + 1;
  double a[2][BKT * LDR * AE];
  double b[2][BKT * LDR * BE];
};

// One (16 TMR) x BN output tile at (row0, col0): TMR = 4 gives the 64 x 64
// tile, TMR = 2 the 32 x 64 tile of the batched launches' short problems and
// edge rows (each output's chains are the same in both, so are its bits).
// Operands straight from the AoS matrices, converted on their way into LDS;
// four waves of 4 TMR x 2 rows x 32 columns in the layout of vcphip_dpp.h.
// RESID: the batched residual form R*A - I, whose diagonal elements get the
// interval subtraction of 1 (imats.hpp:324-326).  Runs in the caller's
// round-up mode.
template <bool PAIR>
__device__ __forceinline__ double2 dr_load(__amdgpu_buffer_rsrc_t g, unsigned off) {
  if (PAIR) return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(g, off, 0, 0));
  return make_double2(__builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(g, off, 0, 0)), 0.0);
}

constexpr long DR_LDMAX = VCPHIP_TILE_LDMAX;

template <bool AI, bool BI, bool RESID, int TMR = 4, bool BIG = false, class Lds = DrLds<AI, BI>>
__device__ __forceinline__ void dr_tile(Lds& L, int m, int n, int k, const double* __restrict__ A,
                                        long lda, const double* __restrict__ B, long ldb, double* __restrict__ C,
                                        long ldc, int row0, int col0) {
  static_assert(AI || BI, "an interval product");
  constexpr bool II = AI && BI;
  constexpr int RPL = 4 * TMR, TBM = 4 * RPL;   // rows per lane, tile rows
  constexpr int BKT = Lds::BKT, AE = Lds::AE, BE = Lds::BE, LDR = Lds::LDR;
  constexpr int APT = TBM * BKT / NT;           // elements of A per thread per slice
  constexpr int BPT = BN * BKT / NT;
  constexpr int AKS = NT / TBM;                 // k stride of a thread's A elements
  constexpr int BCS = NT / BKT;                 // column stride of its B elements
  static_assert(TMR == 4 || TMR == 2, "tile rows");
  static_assert(APT >= 1 && AKS * APT == BKT, "slice shape");
  const int tid = threadIdx.x;

  // global-load mapping: A column-major, TBM consecutive rows per k column;
  // B column-major, BKT consecutive k per column.
  const int a_row = tid % TBM, a_kc = tid / TBM;   // k column a_kc + AKS q
  const int b_k = tid % BKT, b_col = tid / BKT;    // column b_col + BCS q
  double2 ra[APT], rb[BPT];
  // global loads of one k-slice, zeros outside the operands: buffer loads
  // from a uniform base at 32-bit lane offsets that stay the same over the
  // slices.  The resource's size ends A after column k - 1 and B after column
  // n - 1; a row of A past m, and B's rows past k in the last slice, take an
  // offset past any size.  (Leading dimensions below DR_LDMAX keep every
  // offset below 2^31; larger ones, BIG, take 64-bit addresses and checks.)
  constexpr unsigned OUT = 1u << 31;
  const unsigned a_off = row0 + a_row < m ? 8u * AE * ((unsigned)a_row + (unsigned)lda * a_kc) : OUT;
  const unsigned a_step = 8u * AE * AKS * (unsigned)lda;
  const unsigned b_off = 8u * BE * ((unsigned)b_k + (unsigned)ldb * b_col), b_step = 8u * BE * BCS * (unsigned)ldb;
  auto load_tile = [&](int k0) {
    if (BIG) {
#pragma unroll
      for (int q = 0; q < APT; ++q) {
        const int kk = k0 + a_kc + AKS * q, r = row0 + a_row;
        const bool ok = (r < m) && (kk < k);
        if (AI) ra[q] = ok ? *reinterpret_cast<const double2*>(A + 2 * (r + lda * kk)) : make_double2(0.0, 0.0);
        else ra[q].x = ok ? A[r + lda * kk] : 0.0;
      }
#pragma unroll
      for (int q = 0; q < BPT; ++q) {
        const int kk = k0 + b_k, c = col0 + b_col + BCS * q;
        const bool ok = (kk < k) && (c < n);
        if (BI) rb[q] = ok ? *reinterpret_cast<const double2*>(B + 2 * (kk + ldb * c)) : make_double2(0.0, 0.0);
        else rb[q].x = ok ? B[kk + ldb * c] : 0.0;
      }
      return;
    }
    // the last slice may start past k (k is rounded up to 16): A is then empty
    const long sa = 8 * AE * (lda * (long)(k > k0 ? k - k0 : 0)), sb = 8 * BE * (ldb * (long)(n - col0));
    const __amdgpu_buffer_rsrc_t ga = vcphip_rsrc(A + AE * (row0 + lda * k0), (int)(sa < (long)OUT ? sa : (long)OUT));
    const __amdgpu_buffer_rsrc_t gb = vcphip_rsrc(B + BE * (k0 + ldb * col0), (int)(sb < (long)OUT ? sb : (long)OUT));
    const unsigned bo = k0 + b_k < k ? b_off : OUT;
#pragma unroll
    for (int q = 0; q < APT; ++q) ra[q] = dr_load<AI>(ga, a_off + q * a_step);
#pragma unroll
    for (int q = 0; q < BPT; ++q) rb[q] = dr_load<BI>(gb, bo + q * b_step);
  };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int q = 0; q < APT; ++q) {
      double* d = &L.a[buf][((a_kc + AKS * q) * LDR + a_row) * AE];
      if (AI) {
        double mm, rr;
        vcphip_midrad_ru(ra[q].x, ra[q].y, mm, rr);
        *reinterpret_cast<double2*>(d) = make_double2(mm, rr);
      } else {
        *d = ra[q].x;
      }
    }
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
      double* d = &L.b[buf][(b_k * LDR + b_col + BCS * q) * BE];
      if (BI) {
        double mm, rr;
        vcphip_midrad_ru(rb[q].x, rb[q].y, mm, rr);
        *reinterpret_cast<double2*>(d) = make_double2(mm, rr);
      } else {
        *d = rb[q].x;
      }
    }
  };

  const int lane = tid & 63, w = tid >> 6;
  const int lrow = (w & 1) * 2 * RPL + (lane >> 5) * RPL, lcol = (w >> 1) * 32 + (lane & 31);
  const int orow = row0 + lrow, ocol = col0 + lcol;
  const int aoff = (lrow + (lane & (RPL - 1))) * AE, boff = lcol * BE;
  double up[RPL], dn[RPL], r1[RPL], r2[RPL];
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    up[i] = 0.0;
    dn[i] = 0.0;
    r1[i] = 0.0;
    r2[i] = 0.0;
  }

  // slices up to k rounded up to 16 (as the planes pad)
  const int nt = (k + 15) / 16 * 16 / BKT;
  if (nt > 0) {
    load_tile(0);
    store_tile(0);
    if (nt > 1) load_tile(BKT);
  }
  for (int t = 0; t < nt; ++t) {
    __syncthreads();   // slice t is in LDS; the reads of the other buffer (slice t - 1) are done
    if (t + 1 < nt) store_tile((t + 1) & 1);
    if (t + 2 < nt) load_tile((t + 2) * BKT);
    const double* sa = L.a[t & 1] + aoff;
    const double* sb = L.b[t & 1] + boff;
    auto rd = [&](int kk, double2& a, double2& b) {
      if (AI) a = *reinterpret_cast<const double2*>(sa + kk * LDR * AE);
      else a.x = sa[kk * LDR];
      if (BI) b = *reinterpret_cast<const double2*>(sb + kk * LDR * BE);
      else b.x = sb[kk * LDR];
    };
    vcphip_dpp_slice<BKT>(rd, [&](double2 a, double2 b) {
      vcphip_dpp_step<AI, BI>(a.x, a.y, b.x, b.y, up, dn, r1, r2);
    });
  }

  // epilogue
  if (ocol >= n) return;
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    const int r = orow + i;
    if (r >= m) break;
    const double t = II ? r1[i] + r2[i] : r1[i];   // temp = (|mA|+rA) rB + rA |mB|   (:283)
    double hi = up[i] + t;                         // uC += temp, RU                  (:284)
    double nlo = dn[i] + t;                        // lC -= temp, RD = -(RU(-lC + t)) (:285-286)
    if (RESID && r == ocol) {                      // b(i,i) -= 1 in interval arithmetic
      hi = hi - 1.0;
      nlo = nlo + 1.0;
    }
    *reinterpret_cast<double2*>(C + 2 * (r + ldc * ocol)) = make_double2(-nlo, hi);
  }
}

// The products of k = 0: every chain is 0, so the round-up and round-down
// results are +0 and -0 (an interval's ends: {-0, +0}).  C2 null: C holds
// intervals.
__global__ __launch_bounds__(NT) void k_empty_product(int m, int n, double* __restrict__ C, long ldc,
                                                      double* __restrict__ C2) {
  const int r = blockIdx.x * NT + threadIdx.x;
  if (r >= m) return;
  for (long c = blockIdx.y; c < n; c += gridDim.y) {
    if (C2) {
      C[r + ldc * c] = 0.0;
      C2[r + ldc * c] = -0.0;
    } else {
      *reinterpret_cast<double2*>(C + 2 * (r + ldc * c)) = make_double2(-0.0, 0.0);
    }
  }
}

// ---------------------------------------------------------------------------
// The single products from operand planes.
//
// pidblas_assist::midrad (:43-60) is taken once per operand element by one
// small kernel instead of once per element and tile inside the product, and
// both operands are laid out for whole, contiguous k-slices:
//   A (m x k, column-major) -> (mid, rad) pairs (interval) or A (point),
//                              kpad x mpad, rows contiguous (ld mpad)
//   B (k x n, column-major) -> pairs or B, kpad x npad, columns contiguous
// zero beyond m, n and k (mpad, npad multiples of 64, kpad of 16).  Every
// k-slice of a tile then lies in runs of 256 to 1024 contiguous bytes, which
// the product loads straight into LDS with no bounds tests, no conversions
// and no register staging, and an element's pair is one 16-byte LDS read.
// The chains and their order are those of dr_tile, so are the results' bits
// (padding adds the same zero terms the checked loads of dr_tile add past k).
// ---------------------------------------------------------------------------
// blocks [0, na): A, 64 rows x 16 k each; the rest: B, 32 x 32 tiles through
// LDS (read along k, written along n), 32-column blocks inside 32-k blocks
template <bool AI, bool BI>
__global__ __launch_bounds__(256) void k_planes(int m, int n, int k, int mpad, int npad, int kpad, unsigned na,
                                                const double* __restrict__ A, long lda, const double* __restrict__ B,
                                                long ldb, double* __restrict__ PA, double* __restrict__ PB) {
  vcphip_mode_round_up();
  __shared__ double2 s[32][33];
  if (blockIdx.x < na) {
    const unsigned rb = blockIdx.x % (unsigned)(mpad / 64), kb = blockIdx.x / (unsigned)(mpad / 64);
    const int r = (int)rb * 64 + (threadIdx.x & 63), k0 = (int)kb * 16 + (threadIdx.x >> 6);
    double2 v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int kk = k0 + 4 * q;
      v[q] = make_double2(0.0, 0.0);
      if (r < m && kk < k) {
        if (AI) v[q] = *reinterpret_cast<const double2*>(A + 2 * (r + lda * (long)kk));
        else v[q].x = A[r + lda * (long)kk];
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const long o = (long)(k0 + 4 * q) * mpad + r;
      if (AI) {
        double mm, rr;
        vcphip_midrad_ru(v[q].x, v[q].y, mm, rr);   // (0, 0) for the padding
        *reinterpret_cast<double2*>(PA + 2 * o) = make_double2(mm, rr);
      } else {
        PA[o] = v[q].x;
      }
    }
    return;
  }
  const unsigned bb = blockIdx.x - na, nj = (unsigned)(npad / 32);
  const int k0 = (int)(bb / nj) * 32, j0 = (int)(bb % nj) * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int kk = k0 + tx, j = j0 + ty + 8 * i;
    double2 v = make_double2(0.0, 0.0);
    if (kk < k && j < n) {
      if (BI) v = *reinterpret_cast<const double2*>(B + 2 * (kk + ldb * (long)j));
      else v.x = B[kk + ldb * (long)j];
    }
    s[ty + 8 * i][tx] = v;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int kk = k0 + ty + 8 * i, j = j0 + tx;
    if (kk >= kpad) continue;   // the last block of 32 k may reach past kpad
    const double2 v = s[tx][ty + 8 * i];
    const long o = (long)kk * npad + j;
    if (BI) {
      double mm, rr;
      vcphip_midrad_ru(v.x, v.y, mm, rr);
      *reinterpret_cast<double2*>(PB + 2 * o) = make_double2(mm, rr);
    } else {
      PB[o] = v.x;
    }
  }
}

// The k-slices of a (4 RPL) x 64 tile in LDS and their loads: a stage is BKS
// k of A's rows, then of B's columns, elements of AE / BE doubles.  A
// wave-wide load moves 1 KB: 1024 / (row bytes) k-rows; the workgroup's four
// waves take the stage's 1 KB pieces in turn, G each.  Two stages: the next one's loads are in flight
// under the multiply-adds of the current one.  8 k for 64-row tiles, so that
// three workgroups' stages fit a CU; 16 k for 32-row ones, whose 8 k take
// about a load's latency.  (Three or four stages of 8 k measured 0 - 3% slower
// at n = 1024 to 3072, 8 k for 32 rows 1 - 7% slower at 512 and 1024.)
template <int RPL, int AE, int BE>
struct PlaneStage {
  static constexpr int BKS = RPL == 16 ? 8 : 16, NST = 2;
  static constexpr int ROWS = 4 * RPL, ARB = ROWS * AE * 8, BRB = 64 * BE * 8;   // bytes of a k-row
  static constexpr int ABYTES = BKS * ARB, BBYTES = BKS * BRB, BYTES = ABYTES + BBYTES;
  static constexpr int NA = ABYTES / 1024, NB = BBYTES / 1024, G = (NA + NB) / 4;
  static_assert(ABYTES % 4096 == 0 && BBYTES % 4096 == 0 && 16 % BKS == 0, "stage shape");
  const char *a, *b;
  long lda, ldb;   // bytes of a k-row of the planes
  uint32_t lds;
  int w;
  VCPHIP_DEVINL PlaneStage(const double* PA, long mpad, int row0, const double* PB, long npad, int col0, const void* L) {
    const int lane = threadIdx.x & 63;
    w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lda = mpad * AE * 8;
    ldb = npad * BE * 8;
    a = (const char*)(PA + (long)row0 * AE) + (long)(16 * lane / ARB) * lda + 16 * lane % ARB;
    b = (const char*)(PB + (long)col0 * BE) + (long)(16 * lane / BRB) * ldb + 16 * lane % BRB;
    lds = vcphip_lds_addr(L);
  }
  VCPHIP_DEVINL void issue(int t) const {
    const uint32_t d = lds + (uint32_t)(t % NST) * BYTES;
    const char* ga = a + (long)t * BKS * lda;
    const char* gb = b + (long)t * BKS * ldb;
#pragma unroll
    for (int q = 0; q < G; ++q) {
      const int c = 4 * q + w;   // wave-uniform; the four waves' pieces are all A's or all B's
      if (4 * q < NA) vcphip_lds_dma16(ga + (long)c * (1024 / ARB) * lda, d + (uint32_t)c * 1024);
      else vcphip_lds_dma16(gb + (long)(c - NA) * (1024 / BRB) * ldb, d + (uint32_t)c * 1024);
    }
  }
  // slice t has landed for every wave (only its loads are in flight), and
  // every wave's reads of the other stage, slice t - 1, are done: that stage
  // takes slice t + 1
  VCPHIP_DEVINL void next(int t, int nt) const {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (t + 1 < nt) issue(t + 1);
  }
};

// A wave's 2 RPL x 32 block of a point matrix X at (row0, col0), between the
// registers (lane: RPL rows of one column, v) and memory through D doubles of
// the wave's own LDS, D / (2 RPL) columns at a time: runs of 16 RPL contiguous
// bytes of a column instead of a double per lane and column, which filled the
// lines of the two result matrices an element at a time.  RU / RD product, one
// context, element-wise against through LDS (results / results and accumulated
// values): 2048 x 2048 x 64 148 against 36 us / 100 against 44, 4096 x 4096 x
// 128 245 against 180 / 320 against 202, 2000 x 2000 x 2000 616 against 597 /
// 722 against 593.  In LDS a column's pairs of rows are exchanged by its index,
// which spreads the accesses of both directions over the banks.
template <int RPL, int D>
struct PointBlock {
  static constexpr int R = 2 * RPL, NC = D / R, T = D / 64;   // rows, columns of a pass, doubles per lane and pass
  static VCPHIP_DEVINL int pair(int c, int p) { return c * RPL + (p ^ (c & (RPL - 1))); }
  static VCPHIP_DEVINL int elem(int c, int r) { return 2 * pair(c, r / 2) + (r & 1); }
  static VCPHIP_DEVINL void store(double2* L, const double (&v)[RPL], int lane, double* __restrict__ X, long ldx,
                                  int row0, int col0, int m, int n) {
    const int lc = lane & 31, h = lane >> 5, r = lane % R;
    const double* l = reinterpret_cast<const double*>(L);
#pragma unroll
    for (int c0 = 0; c0 < 32; c0 += NC) {
      if (col0 + c0 >= n) break;   // wave-uniform
      if (lc / NC == c0 / NC) {
#pragma unroll
        for (int i = 0; i < RPL; i += 2) L[pair(lc % NC, (h * RPL + i) / 2)] = make_double2(v[i], v[i + 1]);
      }
      vcphip_wave_sync();
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int c = lane / R + 64 / R * t;
        if (row0 + r < m && col0 + c0 + c < n) X[row0 + r + ldx * (col0 + c0 + c)] = l[elem(c, r)];
      }
      vcphip_wave_sync();   // read before the next pass overwrites it
    }
  }
  // zeros outside the m x n matrix
  static VCPHIP_DEVINL void load(double2* L, double (&v)[RPL], int lane, const double* __restrict__ X, long ldx,
                                 int row0, int col0, int m, int n) {
    const int lc = lane & 31, h = lane >> 5, r = lane % R;
    double* l = reinterpret_cast<double*>(L);
#pragma unroll
    for (int g = 0; g < 2; ++g) {   // half of the columns' loads in flight
      double x[RPL / 2];
#pragma unroll
      for (int q = 0; q < RPL / 2; ++q) {
        const int c = col0 + 16 * g + q / T * NC + lane / R + 64 / R * (q % T);
        x[q] = 0.0;
        if (row0 + r < m && c < n) x[q] = X[row0 + r + ldx * c];
      }
#pragma unroll
      for (int c0 = 16 * g; c0 < 16 * g + 16; c0 += NC) {
#pragma unroll
        for (int t = 0; t < T; ++t) l[elem(lane / R + 64 / R * t, r)] = x[(c0 - 16 * g) / NC * T + t];
        vcphip_wave_sync();
        if (lc / NC == c0 / NC) {
#pragma unroll
          for (int i = 0; i < RPL; i += 2) {
            const double2 p = L[pair(lc % NC, (h * RPL + i) / 2)];
            v[i] = p.x;
            v[i + 1] = p.y;
          }
        }
        vcphip_wave_sync();
      }
    }
  }
};

// The same for a block of interval results: a lane holds the pairs v(0) ..
// v(RPL - 1) of its column, written D pairs at a time.  2048 x 2048 x 16, a pair
// per lane and column against through LDS: interval x interval 24.1 against 15.8
// us (three contexts in turn; 32 against 23 one), 1500 x 1500 x 100 39.2 against
// 37.7 (55 against 51).
template <int RPL, int D>
struct IntervalBlock {
  static constexpr int R = 2 * RPL, NC = D / R, T = D / 64;
  static VCPHIP_DEVINL int slot(int c, int r) { return c * R + (r ^ (c & (R - 1))); }
  template <class F>
  static VCPHIP_DEVINL void store(double2* L, const F& v, int lane, double* __restrict__ X, long ldx, int row0, int col0,
                                  int m, int n) {
    const int lc = lane & 31, h = lane >> 5, r = lane % R;
#pragma unroll
    for (int c0 = 0; c0 < 32; c0 += NC) {
      if (col0 + c0 >= n) break;   // wave-uniform
      if (lc / NC == c0 / NC) {
#pragma unroll
        for (int i = 0; i < RPL; ++i) L[slot(lc % NC, h * RPL + i)] = v(i);
      }
      vcphip_wave_sync();
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int c = lane / R + 64 / R * t;
        if (row0 + r < m && col0 + c0 + c < n)
          *reinterpret_cast<double2*>(X + 2 * (row0 + r + ldx * (col0 + c0 + c))) = L[slot(c, r)];
      }
      vcphip_wave_sync();
    }
  }
};

// Tiles of 4 RPL x 64 outputs, four waves of 2 RPL rows x 32 columns, RPL
// outputs of one column per lane (vcphip_dpp.h): RPL = 16 (64 rows) for grids
// that fill the device, RPL = 8 (32 rows) for small ones.  Bound by the FP64
// multiply-adds, at n = 4096 by the clock that they leave (61 TFLOP/s is 0.93
// of the rate at 2.0 GHz).  A wave whose block is all padding keeps the loads
// and barriers in a loop of its own (20000 x 32 x 2000 548 against 502 us).
// Interval x interval, planes included, against 4 x 4 outputs per lane read
// from LDS: n = 1024 205 -> 161 us, 2048 1432 -> 1107, 4096 11.0 -> 9.1 ms;
// point x interval at 2048 981 -> 817 us, at 4096 7.5 -> 6.5 - 7.2 ms.
template <bool AI, bool BI, int RPL>
__global__ __launch_bounds__(NT, RPL == 16 ? ((AI && BI) ? 3 : 4) : 4)
void k_drgemm_planes(int m, int n, int mpad, int npad, int kpad, const double* __restrict__ PA,
                     const double* __restrict__ PB, double* __restrict__ C, long ldc, double* __restrict__ C2,
                     int accumulate) {
  constexpr bool II = AI && BI;
  constexpr int AE = AI ? 2 : 1, BE = BI ? 2 : 1;
  using Stage = PlaneStage<RPL, AE, BE>;
  vcphip_mode_round_up();
  __shared__ __attribute__((aligned(16))) char sL[Stage::NST * Stage::BYTES];
  const int ntm = mpad / Stage::ROWS, ntn = npad / 64;
  const int tile = vcphip_xcd_remap(blockIdx.x, ntm * ntn);
  int tm, tn;
  vcphip_tile_coords(tile, ntm, ntn, 16, tm, tn);
  const int row0 = tm * Stage::ROWS, col0 = tn * 64;
  const Stage st(PA, mpad, row0, PB, npad, col0, sL);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // this lane's outputs: rows lrow .. lrow + RPL - 1 of column lcol of the tile;
  // lane i of its DPP row of 16 holds A's row lrow + i
  const int lrow = (w & 1) * 2 * RPL + (lane >> 5) * RPL, lcol = (w >> 1) * 32 + (lane & 31);
  const int aoff = (lrow + (lane & (RPL - 1))) * AE * 8, boff = Stage::ABYTES + lcol * BE * 8;

  double up[RPL], dn[RPL], r1[RPL], r2[RPL];
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    up[i] = 0.0;
    dn[i] = 0.0;
    r1[i] = 0.0;
    r2[i] = 0.0;
  }
  const int wrow = row0 + (w & 1) * 2 * RPL, wcol = col0 + (w >> 1) * 32;   // the wave's block
  const int nt = kpad / Stage::BKS;
  st.issue(0);
  if (!AI && !BI && accumulate) {
    // udmatmul form: the chains continue from the values already in CU / CD,
    // which come in through the second stage (its first loads are issued after
    // the barrier that follows these reads)
    double2* L = reinterpret_cast<double2*>(sL + Stage::BYTES) + 128 * w;
    PointBlock<RPL, 256>::load(L, up, lane, C, ldc, wrow, wcol, m, n);
    PointBlock<RPL, 256>::load(L, dn, lane, C2, ldc, wrow, wcol, m, n);
#pragma unroll
    for (int i = 0; i < RPL; ++i) dn[i] = -dn[i];
  }
  if (__builtin_amdgcn_readfirstlane(wrow >= m || wcol >= n)) {   // a block of padding: load and keep the barriers
    for (int t = 0; t < nt; ++t) st.next(t, nt);
    __syncthreads();
    return;
  }
  for (int t = 0; t < nt; ++t) {
    st.next(t, nt);
    const char* s0 = sL + (t % Stage::NST) * Stage::BYTES;
    auto rd = [&](int kk, double2& a, double2& b) {
      if (AI) a = *reinterpret_cast<const double2*>(s0 + aoff + kk * Stage::ARB);
      else a.x = *reinterpret_cast<const double*>(s0 + aoff + kk * Stage::ARB);
      if (BI) b = *reinterpret_cast<const double2*>(s0 + boff + kk * Stage::BRB);
      else b.x = *reinterpret_cast<const double*>(s0 + boff + kk * Stage::BRB);
    };
    vcphip_dpp_slice<Stage::BKS>(rd, [&](double2 a, double2 b) {
      vcphip_dpp_step<AI, BI>(a.x, a.y, b.x, b.y, up, dn, r1, r2);
    });
  }

  __syncthreads();   // every wave has read the last stage
  // the wave's own quarter of the stages takes D = 2^n pairs (or pairs of rows)
  constexpr int D = Stage::NST * Stage::BYTES / 64 >= 512 ? 512 : 256;
  double2* L = reinterpret_cast<double2*>(sL) + D * w;
  if (AI || BI) {
    IntervalBlock<RPL, D>::store(
        L,
        [&](int i) {
          const double tt = II ? r1[i] + r2[i] : r1[i];   // temp (:283, :129, :185)
          const double hi = up[i] + tt;                   // uC += temp, RU (:284)
          const double nlo = dn[i] + tt;                  // lC -= temp, RD = -(RU(-lC + t)) (:285-286)
          return make_double2(-nlo, hi);
        },
        lane, C, ldc, wrow, wcol, m, n);
  } else {
    PointBlock<RPL, 2 * D>::store(L, up, lane, C, ldc, wrow, wcol, m, n);
#pragma unroll
    for (int i = 0; i < RPL; ++i) dn[i] = -dn[i];
    PointBlock<RPL, 2 * D>::store(L, dn, lane, C2, ldc, wrow, wcol, m, n);
  }
}

// ---------------------------------------------------------------------------
// Batched verified residual C_p = R_p * IA_p - I (imats::linearsolve,
// vcp/imats.hpp:318-326) for many problems of uneven size in one persistent
// launch per tile shape (TMR = 4: 64 x 64, TMR = 2: 32 x 64): workgroups
// take the tiles of a list sorted by problem size (largest first) from a
// work queue, each tile being the PI form above.
// ---------------------------------------------------------------------------
// Work queue of the persistent launches: workgroup thread 0 takes the next
// tile index from the launch's counter (zeroed by k_queue_reset just before
// the launch, on the same stream), so tiles are taken in list order as
// workgroups come free.  (A fixed stride of the grid over the list was
// 15-20% slower on uneven sets: a workgroup that drew long tiles held up the
// end of the launch.)
__device__ __forceinline__ int next_tile(unsigned* __restrict__ queue, int& slot) {
  __syncthreads();   // every thread has read the previous index (and left the tile's LDS)
  if (threadIdx.x == 0) slot = (int)atomicAdd(queue, 1u);
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(slot);   // uniform: the tile's descriptors are then scalar loads
}

__global__ __launch_bounds__(64) void k_queue_reset(unsigned* __restrict__ queue) {
  if (threadIdx.x < 2) queue[threadIdx.x] = 0u;
}

template <int TMR, bool BIG>
__global__ __launch_bounds__(NT, BIG ? 2 : 3) void k_resid_tiles(int ntiles, const VcphipResidTile* __restrict__ tiles,
                                                        const VcphipResidProblem* __restrict__ probs,
                                                        unsigned* __restrict__ queue) {
  vcphip_mode_round_up();
  __shared__ __attribute__((aligned(16))) DrLds<false, true> lds;
  __shared__ int slot;
  for (int t = next_tile(queue, slot); t < ntiles; t = next_tile(queue, slot)) {
    const VcphipResidTile tl = tiles[t];
    const VcphipResidProblem p = probs[tl.problem];
    dr_tile<false, true, true, TMR, BIG>(lds, p.n, p.n, p.n, p.R, p.ldr, p.A, p.lda, p.C, p.ldc, tl.row0, tl.col0);
  }
}

// Many interval products C_p = IA_p * IB_p of uneven (m, n, k) in one
// persistent launch per tile shape (pidblas::mulmm, vcp/pidblas.hpp:239-294,
// per problem): workgroups take the tiles of a list sorted by problem size
// from a work queue, each tile the interval x interval form above, so
// every C_p is bit-identical to the single product's.
template <int TMR, bool BIG>
__global__ __launch_bounds__(NT, 2) void k_igemm_tiles(int ntiles, const VcphipResidTile* __restrict__ tiles,
                                                        const VcphipIgemmProblem* __restrict__ probs,
                                                        unsigned* __restrict__ queue) {
  vcphip_mode_round_up();
  __shared__ __attribute__((aligned(16))) DrLds<true, true> lds;
  __shared__ int slot;
  for (int t = next_tile(queue, slot); t < ntiles; t = next_tile(queue, slot)) {
    const VcphipResidTile tl = tiles[t];
    const VcphipIgemmProblem p = probs[tl.problem];
    dr_tile<true, true, false, TMR, BIG>(lds, p.m, p.n, p.k, p.A, p.lda, p.B, p.ldb, p.C, p.ldc, tl.row0, tl.col0);
  }
}

// ---------------------------------------------------------------------------
// The single products with few columns, or too small to fill the device with
// tiles: the row-serial form of vcphip_thin.h, one launch straight from the
// AoS operands.
// ---------------------------------------------------------------------------
template <bool AI, bool BI>
struct ThinProduct : VcphipThinDr<AI, BI> {
  using Base = VcphipThinDr<AI, BI>;
  double* __restrict__ C;
  double* __restrict__ C2;
  long ldc;
  int accumulate, m, n;
  VCPHIP_DEVINL void init(typename Base::Acc& c, int row, int col) const {
    Base::init(c, row, col);
    if (!AI && !BI && accumulate && row < m && col < n) {
      c.up = C[row + ldc * col];
      c.dn = -C2[row + ldc * col];
    }
  }
  VCPHIP_DEVINL void done(const typename Base::Acc& c, int row, int col) const {
    if (AI || BI) {
      *reinterpret_cast<double2*>(C + 2 * (row + ldc * col)) = this->result(c);
    } else {
      C[row + ldc * col] = c.up;
      C2[row + ldc * col] = -c.dn;
    }
  }
};

template <bool AI, bool BI, int CW, int CPT>
__global__ __launch_bounds__((VcphipThin<ThinProduct<AI, BI>, CW, CPT>::NT)) VCPHIP_THIN_WAVES void k_drgemm_thin(int m, int n, int k, const double* __restrict__ A, long lda,
                                                     const double* __restrict__ B, long ldb, double* __restrict__ C,
                                                     long ldc, double* __restrict__ C2, int accumulate) {
  vcphip_mode_round_up();
  using T = VcphipThin<ThinProduct<AI, BI>, CW, CPT>;
  __shared__ __attribute__((aligned(16))) typename T::Lds lds;
  ThinProduct<AI, BI> op;
  op.A = A;
  op.B = B;
  op.lda = lda;
  op.ldb = ldb;
  op.C = C;
  op.C2 = C2;
  op.ldc = ldc;
  op.accumulate = accumulate;
  op.m = m;
  op.n = n;
  const int rb = vcphip_xcd_remap(blockIdx.x, gridDim.x);
  T::run(op, lds, m, n, k, rb * T::R, blockIdx.y * T::NC, (int)((blockIdx.x >> 8) % T::NW));
}

// row sums of |C| (upward, in column order: mats::norminf, vcp/mats.hpp:
// 1583-1591) over 8-row blocks of the problems, in the row-serial form: each
// C_p is read once, at a cache line per row block and column (a thread per row,
// 256 rows to a workgroup, had too few loads in flight: 153 against 98 us for
// 64 problems of n in [64, 1024])
struct ResidRowSum {
  static constexpr bool A2 = true, B2 = false, PAD16 = false;
  static constexpr int AL = 1, BL = 0;
  const double* A;
  const double* B = nullptr;
  long lda, ldb = 0;
  double* out;
  struct Acc {
    double s;
  };
  VCPHIP_DEVINL double2 a(double2 v, int, int) const {
    return make_double2(fmax(__builtin_fabs(v.x), __builtin_fabs(v.y)), 0.0);
  }
  VCPHIP_DEVINL double2 b(double2 v) const { return v; }
  VCPHIP_DEVINL void init(Acc& c, int, int) const { c.s = 0.0; }
  VCPHIP_DEVINL void step(Acc& c, double2 av, double2) const { c.s = c.s + av.x; }
  VCPHIP_DEVINL void done(const Acc& c, int row, int) const { out[row] = c.s; }
};

__global__ __launch_bounds__((VcphipThin<ResidRowSum, 1>::NT)) VCPHIP_THIN_WAVES
void k_resid_rowsum(const VcphipResidTile* __restrict__ blocks, const VcphipResidProblem* __restrict__ probs,
                    double* __restrict__ rowsum) {
  vcphip_mode_round_up();
  using T = VcphipThin<ResidRowSum, 1>;
  __shared__ __attribute__((aligned(16))) typename T::Lds lds;
  const VcphipResidTile tl = blocks[vcphip_xcd_remap(blockIdx.x, gridDim.x)];
  const VcphipResidProblem p = probs[tl.problem];
  ResidRowSum op;
  op.A = p.C;
  op.lda = p.ldc;
  op.out = rowsum + p.row_base;
  T::run(op, lds, p.n, 1, p.n, tl.row0, 0, (int)((blockIdx.x >> 8) % T::NW));
}

// ||C_p||_inf upper bound: the largest row sum (mats.hpp:1592-1598), by the
// rule that the verified solve's norm follows; one workgroup per problem
__global__ __launch_bounds__(256) void k_resid_max(int count, const VcphipResidProblem* __restrict__ probs,
                                                   const double* __restrict__ rowsum, double* __restrict__ normub) {
  __shared__ double red[256];
  const int pi = blockIdx.x;
  const VcphipResidProblem p = probs[pi];
  if (p.n <= 0) {
    if (threadIdx.x == 0) normub[pi] = 0.0;
    return;
  }
  const double* in = rowsum + p.row_base;
  double best = -__builtin_inf();
  for (int i = threadIdx.x; i < p.n; i += 256) {
    const double v = in[i];
    best = v > best ? v : best;
  }
  const double norm = vcphip_block_max<256>(best, in[0], red);
  if (threadIdx.x == 0) normub[pi] = norm;
}

// ---------------------------------------------------------------------------
// A^T A forms.  IA is k x n; tiles (tm <= tn) of the upper triangle only.
//   interval (pidblas::mulltmm, vcp/pidblas.hpp:296-358):
//     up, dn  = chains of mA_i . mA_j                (dsyrk, :308-315)
//     tij     = RU chain of |mA_i| . rA_j            (|mA|^T rA, :317-321)
//     tji     = RU chain of |mA_j| . rA_i
//     sij     = RU chain of rA_i . rA_j              (rA^T rA, :323)
//     T = RU(tij + RU(tji + sij)); upper = RU(up + T); lower = -RU(dn + T)
//   point (pidblas::vmulmm, :198-236): upper = RU chain, lower = RD chain.
// Element (i, j), i <= j, is written to (i, j) and (j, i).
// ---------------------------------------------------------------------------
// From the planes of A (k x n) made by k_planes's B part: (mid, rad) pairs (or
// A), kpad x npad, columns contiguous, zero-padded.  Column i of A is then the
// contiguous run at i of every k-row, so one plane set feeds both operands.
// Tiles of 4 RPL rows x 64 columns that meet the upper triangle.
template <bool INTV, int RPL>
__global__ __launch_bounds__(NT, RPL == 16 ? (INTV ? 2 : 4) : 4) void k_drsyrk_planes(int n, int npad, int kpad,
                                                                                      const double* __restrict__ P,
                                                                                      double* __restrict__ C,
                                                                                      long ldc) {
  constexpr int E = INTV ? 2 : 1, H = 64 / (4 * RPL);   // row blocks per 64 rows
  using Stage = PlaneStage<RPL, E, E>;
  vcphip_mode_round_up();
  __shared__ __attribute__((aligned(16))) char sL[Stage::NST * Stage::BYTES];
  int b = blockIdx.x, tn = 0;   // column block tn has H (tn + 1) row blocks
  while (b >= H * (tn + 1)) {
    b -= H * (tn + 1);
    ++tn;
  }
  const int i0 = b * Stage::ROWS, j0 = tn * 64;
  const Stage st(P, npad, i0, P, npad, j0, sL);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lrow = (w & 1) * 2 * RPL + (lane >> 5) * RPL, lcol = (w >> 1) * 32 + (lane & 31);
  const int aoff = (lrow + (lane & (RPL - 1))) * E * 8, boff = Stage::ABYTES + lcol * E * 8;
  double up[RPL], dn[RPL], tij[RPL], tji[RPL], sij[RPL];
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    up[i] = 0.0;
    dn[i] = 0.0;
    tij[i] = 0.0;
    tji[i] = 0.0;
    sij[i] = 0.0;
  }
  const int nt = kpad / Stage::BKS;
  st.issue(0);
  for (int t = 0; t < nt; ++t) {
    st.next(t, nt);
    const char* s0 = sL + (t % Stage::NST) * Stage::BYTES;
    auto rd = [&](int kk, double2& x, double2& y) {
      if (INTV) {
        x = *reinterpret_cast<const double2*>(s0 + aoff + kk * Stage::ARB);
        y = *reinterpret_cast<const double2*>(s0 + boff + kk * Stage::BRB);
      } else {
        x.x = *reinterpret_cast<const double*>(s0 + aoff + kk * Stage::ARB);
        y.x = *reinterpret_cast<const double*>(s0 + boff + kk * Stage::BRB);
      }
    };
    vcphip_dpp_slice<Stage::BKS>(rd, [&](double2 x, double2 y) {
      if (INTV) vcphip_dpp_syrk_step(x.x, x.y, y.x, y.y, up, dn, tij, tji, sij);
      else vcphip_dpp_step<false, false>(x.x, 0.0, y.x, 0.0, up, dn, tij, tji);
    });
  }
  const int c = j0 + lcol;
  if (c >= n) return;
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    const int r = i0 + lrow + i;
    if (r > c) break;
    double lo, hi;
    if (INTV) {
      const double T = tij[i] + (tji[i] + sij[i]);
      hi = up[i] + T;
      lo = -(dn[i] + T);
    } else {
      hi = up[i];
      lo = -dn[i];
    }
    *reinterpret_cast<double2*>(C + 2 * (r + ldc * c)) = make_double2(lo, hi);
    *reinterpret_cast<double2*>(C + 2 * (c + ldc * r)) = make_double2(lo, hi);
  }
}

// ---------------------------------------------------------------------------
// Inf-sup interval product (pidblas_fma::mulmm, vcp/pidblas_fma.hpp:62-71,
// with the interval FMA of vcp/ifma.hpp:44-55): per output element the
// k-ascending chains
//   up <- max over a in {inf A, sup A}, b in {inf B, sup B} of RU(a b + up)
//   dn <- min over the same of RD(a b + dn),        both from 0.
// RU is monotone, so the maximum of the four rounded FMAs is the rounded FMA
// of the largest product: the same result as the reference's sign-case
// selection (ifma.hpp:58-137), without its branches.  The RD chain is carried
// negated, d = -dn, as d <- max RU((-a) b + d).
//
// The maxima are v_max_f64, whose order is total here (-0 < +0, a NaN
// operand yields the other), so the maximum of the four does not depend on
// which end of an operand comes first: the operands are staged as (end of
// smaller magnitude, end of larger magnitude).  When every operand of a
// k-slice is finite and strictly on one side of zero, the extreme products
// are those of the smaller ends and of the larger ends, so two FMAs per chain
// give the same maximum: 4 FMAs and 2 maxima per (i, j, k) instead of 8 and 6.
// ---------------------------------------------------------------------------
// finite and strictly on one side of zero
__device__ __forceinline__ bool is_sign_definite(double lo, double hi) {
  return (lo > 0.0 || hi < 0.0) && __builtin_fabs(lo) < __builtin_inf() && __builtin_fabs(hi) < __builtin_inf();
}
// (end of smaller magnitude, end of larger magnitude) of a sign-definite
// interval; other intervals keep their order
__device__ __forceinline__ double2 ends_by_magnitude(double2 v) {
  return v.y < 0.0 ? make_double2(v.y, v.x) : v;
}

__global__ __launch_bounds__(NT) void k_isgemm(int m, int n, int k, const double* __restrict__ A, long lda,
                                               const double* __restrict__ B, long ldb, double* __restrict__ C,
                                               long ldc) {
  vcphip_mode_round_up();
  __shared__ __attribute__((aligned(16))) double sAi[BK][LA];
  __shared__ __attribute__((aligned(16))) double sAs[BK][LA];
  __shared__ __attribute__((aligned(16))) double sBi[BK][LB];
  __shared__ __attribute__((aligned(16))) double sBs[BK][LB];
  const int ntm = (m + BM - 1) / BM, ntn = (n + BN - 1) / BN;
  const int tiles = ntm * ntn;
  int tm, tn;
  vcphip_tile_coords(vcphip_xcd_remap(blockIdx.x, tiles), ntm, ntn, 8, tm, tn);
  const int row0 = tm * BM, col0 = tn * BN;
  const int tid = threadIdx.x;
  const int a_row = tid % BM, a_kc = tid / BM;
  const int b_k = tid % BK, b_col = tid / BK;
  double2 ra[A_PER_T], rb[B_PER_T];
  auto load_tile = [&](int k0) {
#pragma unroll
    for (int q = 0; q < A_PER_T; ++q) {
      const int kk = k0 + a_kc + 4 * q, r = row0 + a_row;
      ra[q] = (r < m && kk < k) ? *reinterpret_cast<const double2*>(A + 2 * (r + lda * kk)) : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int q = 0; q < B_PER_T; ++q) {
      const int kk = k0 + b_k, c = col0 + b_col + 16 * q;
      rb[q] = (kk < k && c < n) ? *reinterpret_cast<const double2*>(B + 2 * (kk + ldb * c)) : make_double2(0.0, 0.0);
    }
  };
  // stores the slice at k0 (ends by magnitude) and returns whether every
  // operand of this thread's share is finite and strictly sign-definite
  // (the zero padding past m, n and k takes either loop)
  auto store_tile = [&](int k0) {
    bool ok = true;
#pragma unroll
    for (int q = 0; q < A_PER_T; ++q) {
      const int kk = k0 + a_kc + 4 * q, r = row0 + a_row;
      if (r < m && kk < k) ok = ok && is_sign_definite(ra[q].x, ra[q].y);
      const double2 v = ends_by_magnitude(ra[q]);
      sAi[a_kc + 4 * q][a_row] = v.x;
      sAs[a_kc + 4 * q][a_row] = v.y;
    }
#pragma unroll
    for (int q = 0; q < B_PER_T; ++q) {
      const int kk = k0 + b_k, c = col0 + b_col + 16 * q;
      if (kk < k && c < n) ok = ok && is_sign_definite(rb[q].x, rb[q].y);
      const double2 v = ends_by_magnitude(rb[q]);
      sBi[b_k][b_col + 16 * q] = v.x;
      sBs[b_k][b_col + 16 * q] = v.y;
    }
    return ok;
  };
  const int tx = tid % 16, ty = tid / 16;
  double up[TM][TN], dn[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      up[i][j] = 0.0;
      dn[i][j] = -0.0;   // -(+0): the RD chain starts from +0
    }
  const int ntiles = (k + BK - 1) / BK;
  load_tile(0);
  bool two = __syncthreads_and(store_tile(0)) != 0;   // the slice takes the two-FMA loop
  for (int t = 0; t < ntiles; ++t) {
    if (t + 1 < ntiles) load_tile((t + 1) * BK);
    if (two) {
      // every operand of the slice is sign-definite: the smaller ends' and
      // the larger ends' products are the extreme ones (two FMAs per chain;
      // a separate loop, since one loop with the mixed products behind a
      // uniform branch measured 25% slower)
      for (int kk = 0; kk < BK; ++kk) {
        double as[TM], ag[TM], bs[TN], bg[TN];   // ends of smaller / larger magnitude
        {
          const double2 x0 = *reinterpret_cast<const double2*>(&sAi[kk][ty * TM]);
          const double2 x1 = *reinterpret_cast<const double2*>(&sAi[kk][ty * TM + 2]);
          const double2 x2 = *reinterpret_cast<const double2*>(&sAs[kk][ty * TM]);
          const double2 x3 = *reinterpret_cast<const double2*>(&sAs[kk][ty * TM + 2]);
          as[0] = x0.x; as[1] = x0.y; as[2] = x1.x; as[3] = x1.y;
          ag[0] = x2.x; ag[1] = x2.y; ag[2] = x3.x; ag[3] = x3.y;
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            bs[j] = sBi[kk][tx + 16 * j];
            bg[j] = sBs[kk][tx + 16 * j];
          }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const double u = up[i][j], d = dn[i][j];
            up[i][j] = __builtin_fmax(__builtin_fma(as[i], bs[j], u), __builtin_fma(ag[i], bg[j], u));
            dn[i][j] = __builtin_fmax(__builtin_fma(-as[i], bs[j], d), __builtin_fma(-ag[i], bg[j], d));
          }
      }
    } else {
#pragma unroll 2
      for (int kk = 0; kk < BK; ++kk) {
        double ai[TM], as[TM], bi[TN], bs[TN];
        {
          const double2 x0 = *reinterpret_cast<const double2*>(&sAi[kk][ty * TM]);
          const double2 x1 = *reinterpret_cast<const double2*>(&sAi[kk][ty * TM + 2]);
          const double2 x2 = *reinterpret_cast<const double2*>(&sAs[kk][ty * TM]);
          const double2 x3 = *reinterpret_cast<const double2*>(&sAs[kk][ty * TM + 2]);
          ai[0] = x0.x; ai[1] = x0.y; ai[2] = x1.x; ai[3] = x1.y;
          as[0] = x2.x; as[1] = x2.y; as[2] = x3.x; as[3] = x3.y;
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            bi[j] = sBi[kk][tx + 16 * j];
            bs[j] = sBs[kk][tx + 16 * j];
          }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const double u = up[i][j], d = dn[i][j];
            up[i][j] = __builtin_fmax(__builtin_fmax(__builtin_fma(as[i], bs[j], u), __builtin_fma(ai[i], bs[j], u)),
                                      __builtin_fmax(__builtin_fma(as[i], bi[j], u), __builtin_fma(ai[i], bi[j], u)));
            dn[i][j] = __builtin_fmax(__builtin_fmax(__builtin_fma(-as[i], bs[j], d), __builtin_fma(-ai[i], bs[j], d)),
                                      __builtin_fmax(__builtin_fma(-as[i], bi[j], d), __builtin_fma(-ai[i], bi[j], d)));
          }
      }
    }
    __syncthreads();
    if (t + 1 < ntiles) two = __syncthreads_and(store_tile((t + 1) * BK)) != 0;
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int c = col0 + tx + 16 * j;
    if (c >= n) continue;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int r = row0 + ty * TM + i;
      if (r < m) *reinterpret_cast<double2*>(C + 2 * (r + ldc * (long)c)) = make_double2(-dn[i][j], up[i][j]);
    }
  }
}

// p[0..n) = v (a kernel, so that it can precede graph replays without a
// memset node)
__global__ __launch_bounds__(256) void k_fill_f64(double* __restrict__ p, long n, double v) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = v;
}

}  // namespace

int vcphip_launch_isgemm(int m, int n, int k, const double* A, long lda, const double* B, long ldb, double* C,
                         long ldc, hipStream_t s) {
  if (m <= 0 || n <= 0) return 0;
  const int tiles = ((m + BM - 1) / BM) * ((n + BN - 1) / BN);
  hipLaunchKernelGGL(k_isgemm, dim3(tiles), dim3(NT), 0, s, m, n, k, A, lda, B, ldb, C, ldc);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_launch_empty_product(int m, int n, double* C, long ldc, double* C2, hipStream_t s) {
  if (m <= 0 || n <= 0) return 0;
  const dim3 grid((unsigned)((m + NT - 1) / NT), (unsigned)(n < 65535 ? n : 65535));
  hipLaunchKernelGGL(k_empty_product, grid, dim3(NT), 0, s, m, n, C, ldc, C2);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_launch_drgemm_thin(int kind, int m, int n, int k, const double* A, long lda, const double* B, long ldb,
                              double* C, long ldc, double* C2, int accumulate, hipStream_t s) {
  if (m <= 0 || n <= 0) return 0;
  if (k <= 0) return -1;   // k = 0 is a fill
  // columns of a workgroup: few right-hand sides take the narrow shapes; else
  // the widest (64, the fewest LDS reads per multiply-add) that still gives
  // about 150 workgroups (n = k = m = 300: 19 us with 64, 24 with 32, 30 with
  // 8 columns; 96 x 80 x 160: 12, 8.5 and 6 us)
  const long rb = ((long)m + VCPHIP_THIN_R - 1) / VCPHIP_THIN_R;
  int nc = n <= 8 ? 8 : n <= 16 ? 16 : 64;
  while (nc > 8 && n > 16 && rb * ((n + nc - 1) / nc) < 150) nc /= 2;
  const long cg = ((long)n + nc - 1) / nc;
  if (cg > 65535 || rb > 0x7FFFFFFF) return -7;
  const dim3 grid((unsigned)rb, (unsigned)cg);
#define VCPHIP_THIN_SHAPE(AI, BI, CW, CPT)                                                                        \
  hipLaunchKernelGGL((k_drgemm_thin<AI, BI, CW, CPT>), grid, dim3((VcphipThin<ThinProduct<AI, BI>, CW, CPT>::NT)), \
                     0, s, m, n, k, A, lda, B, ldb, C, ldc, C2, accumulate)
#define VCPHIP_THIN_CASE(KIND, AI, BI)                    \
  case KIND:                                              \
    if (nc == 8) VCPHIP_THIN_SHAPE(AI, BI, 1, 1);         \
    else if (nc == 16) VCPHIP_THIN_SHAPE(AI, BI, 2, 1);   \
    else if (nc == 32) VCPHIP_THIN_SHAPE(AI, BI, 4, 1);   \
    else VCPHIP_THIN_SHAPE(AI, BI, 4, 2);                 \
    break;
  switch (kind) {
    VCPHIP_THIN_CASE(VCPHIP_DR_II, true, true)
    VCPHIP_THIN_CASE(VCPHIP_DR_IP, true, false)
    VCPHIP_THIN_CASE(VCPHIP_DR_PI, false, true)
    VCPHIP_THIN_CASE(VCPHIP_DR_PP, false, false)
    default: return -1;
  }
#undef VCPHIP_THIN_CASE
#undef VCPHIP_THIN_SHAPE
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_launch_planes(int kind, int m, int n, int k, const double* A, long lda, const double* B, long ldb,
                         double* PA, double* PB, hipStream_t s) {
  const int mpad = (m + BM - 1) / BM * BM, npad = (n + BN - 1) / BN * BN, kpad = (k + BK - 1) / BK * BK;
  if (m <= 0 || n <= 0 || kpad <= 0) return 0;
  const size_t na = (size_t)(mpad / 64) * (kpad / 16), nb = (size_t)((kpad + 31) / 32) * (npad / 32);
  if (na + nb > 0x7FFFFFFFu) return -7;
  const dim3 grid((unsigned)(na + nb));
#define VCPHIP_PLANES_CASE(KIND, AI, BI)                                                                             \
  case KIND:                                                                                                         \
    hipLaunchKernelGGL((k_planes<AI, BI>), grid, dim3(256), 0, s, m, n, k, mpad, npad, kpad, (unsigned)na, A, lda, B, \
                       ldb, PA, PB);                                                                                 \
    break;
  switch (kind) {
    VCPHIP_PLANES_CASE(VCPHIP_DR_II, true, true)
    VCPHIP_PLANES_CASE(VCPHIP_DR_IP, true, false)
    VCPHIP_PLANES_CASE(VCPHIP_DR_PI, false, true)
    VCPHIP_PLANES_CASE(VCPHIP_DR_PP, false, false)
    default: return -1;
  }
#undef VCPHIP_PLANES_CASE
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_launch_drgemm_planes(int kind, int m, int n, int k, const double* PA, const double* PB, double* C, long ldc,
                                double* C2, int accumulate, int rows, hipStream_t s) {
  const int mpad = (m + BM - 1) / BM * BM, npad = (n + BN - 1) / BN * BN, kpad = (k + BK - 1) / BK * BK;
  if (m <= 0 || n <= 0) return 0;
  if (kpad == 0 || (rows != 64 && rows != 32)) return -1;   // k = 0 is a fill
  const dim3 grid((mpad / rows) * (npad / BN)), block(NT);
#define VCPHIP_PLANES_CASE(KIND, AI, BI)                                                                            \
  case KIND:                                                                                                        \
    if (rows == 64)                                                                                                 \
      hipLaunchKernelGGL((k_drgemm_planes<AI, BI, 16>), grid, block, 0, s, m, n, mpad, npad, kpad, PA, PB, C, ldc, C2, \
                         accumulate);                                                                               \
    else                                                                                                            \
      hipLaunchKernelGGL((k_drgemm_planes<AI, BI, 8>), grid, block, 0, s, m, n, mpad, npad, kpad, PA, PB, C, ldc, C2, \
                         accumulate);                                                                               \
    break;
  switch (kind) {
    VCPHIP_PLANES_CASE(VCPHIP_DR_II, true, true)
    VCPHIP_PLANES_CASE(VCPHIP_DR_IP, true, false)
    VCPHIP_PLANES_CASE(VCPHIP_DR_PI, false, true)
    VCPHIP_PLANES_CASE(VCPHIP_DR_PP, false, false)
    default: return -1;
  }
#undef VCPHIP_PLANES_CASE
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_launch_drsyrk_planes(int interval, int k, int n, const double* A, long lda, double* P, double* C, long ldc,
                                int rows, hipStream_t s) {
  if (n <= 0) return 0;
  const int npad = (n + BN - 1) / BN * BN, kpad = (k + BK - 1) / BK * BK;
  if (kpad == 0 || (rows != 64 && rows != 32)) return -1;   // k = 0 is a fill
  const size_t nb = (size_t)((kpad + 31) / 32) * (npad / 32);
  if (nb > 0x7FFFFFFFu) return -7;
  const dim3 gb((unsigned)nb);
  const int nt = npad / BN;
  const dim3 grid((unsigned)((64 / rows) * (nt * (nt + 1) / 2)));
  if (interval) {
    hipLaunchKernelGGL((k_planes<true, true>), gb, dim3(256), 0, s, 0, n, k, 64, npad, kpad, 0u, A, lda, A, lda, P, P);
    if (rows == 64) hipLaunchKernelGGL((k_drsyrk_planes<true, 16>), grid, dim3(NT), 0, s, n, npad, kpad, P, C, ldc);
    else hipLaunchKernelGGL((k_drsyrk_planes<true, 8>), grid, dim3(NT), 0, s, n, npad, kpad, P, C, ldc);
  } else {
    hipLaunchKernelGGL((k_planes<false, false>), gb, dim3(256), 0, s, 0, n, k, 64, npad, kpad, 0u, A, lda, A, lda, P, P);
    if (rows == 64) hipLaunchKernelGGL((k_drsyrk_planes<false, 16>), grid, dim3(NT), 0, s, n, npad, kpad, P, C, ldc);
    else hipLaunchKernelGGL((k_drsyrk_planes<false, 8>), grid, dim3(NT), 0, s, n, npad, kpad, P, C, ldc);
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_launch_igemm_tiles(int n64, int n32, const VcphipResidTile* tiles, const VcphipIgemmProblem* probs,
                              int grid64, int grid32, bool big, unsigned* queue, hipStream_t s) {
  if (n64 > 0 || n32 > 0) hipLaunchKernelGGL(k_queue_reset, dim3(1), dim3(64), 0, s, queue);
  if (n64 > 0) {
    if (big) hipLaunchKernelGGL((k_igemm_tiles<4, true>), dim3(grid64), dim3(NT), 0, s, n64, tiles, probs, queue);
    else hipLaunchKernelGGL((k_igemm_tiles<4, false>), dim3(grid64), dim3(NT), 0, s, n64, tiles, probs, queue);
  }
  if (n32 > 0) {
    if (big) hipLaunchKernelGGL((k_igemm_tiles<2, true>), dim3(grid32), dim3(NT), 0, s, n32, tiles + n64, probs, queue + 1);
    else hipLaunchKernelGGL((k_igemm_tiles<2, false>), dim3(grid32), dim3(NT), 0, s, n32, tiles + n64, probs, queue + 1);
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_fill_f64(double* p, long n, double v, hipStream_t s) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(k_fill_f64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n, v);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_launch_resid_tiles(int n64, int n32, const VcphipResidTile* tiles, const VcphipResidProblem* probs,
                              int grid64, int grid32, bool big, unsigned* queue, hipStream_t s) {
  if (n64 > 0 || n32 > 0) hipLaunchKernelGGL(k_queue_reset, dim3(1), dim3(64), 0, s, queue);
  if (n64 > 0) {
    if (big) hipLaunchKernelGGL((k_resid_tiles<4, true>), dim3(grid64), dim3(NT), 0, s, n64, tiles, probs, queue);
    else hipLaunchKernelGGL((k_resid_tiles<4, false>), dim3(grid64), dim3(NT), 0, s, n64, tiles, probs, queue);
  }
  if (n32 > 0) {
    if (big) hipLaunchKernelGGL((k_resid_tiles<2, true>), dim3(grid32), dim3(NT), 0, s, n32, tiles + n64, probs, queue + 1);
    else hipLaunchKernelGGL((k_resid_tiles<2, false>), dim3(grid32), dim3(NT), 0, s, n32, tiles + n64, probs, queue + 1);
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int vcphip_launch_resid(int n64, int n32, const VcphipResidTile* tiles, const VcphipResidProblem* probs, int nblk,
                        const VcphipResidTile* row_block, double* rowsum, int count, double* normub, int grid64,
                        int grid32, bool big, unsigned* queue, hipStream_t s) {
  vcphip_launch_resid_tiles(n64, n32, tiles, probs, grid64, grid32, big, queue, s);
  if (nblk > 0)
    hipLaunchKernelGGL(k_resid_rowsum, dim3(nblk), dim3(VcphipThin<ResidRowSum, 1>::NT), 0, s, row_block, probs, rowsum);
  if (count > 0) hipLaunchKernelGGL(k_resid_max, dim3(count), dim3(256), 0, s, count, probs, rowsum, normub);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
