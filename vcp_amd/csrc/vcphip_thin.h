// Row-serial products with few output columns (gfx950): C(i, c) for a block
// of R = 8 rows and a few columns, every output a chain over k in ascending
// order.  Used where a 64-column tile would be mostly padding (matrix times a
// few vectors, the verified solve's row sums and bounds) or where the 64- or
// 32-row tiles of a small product leave most of the device idle.
//
// Such a product is bound by reading A once (16 or 8 bytes per element
// against a few FMAs), or by the length of the chains.  So the split is by
// rows: a workgroup takes 8 rows (128 contiguous bytes of an interval column,
// one cache line).  Loading waves (3 beside one chain wave, 2 beside two, 4
// beside four) load and convert 8 x KB elements of A and the KB x NC block of
// B into LDS, one stage ahead of the chains and with the next stage's loads in
// flight; the chain waves carry the chains: lane = row (8) x column lane (8),
// CPT columns per lane.  Loading by separate waves keeps conversions and
// global waits out of the chains' way.  (The batched forms take their pointers
// from descriptors in memory.  Their loads are then FLAT ones, which count as
// LDS operations too: the next barrier waits for them, so a stage lasts at
// least as long as the loads issued in it.)  m = 4000 rows give 500
// workgroups, two per CU; consecutive row blocks run on one XCD, so that cache
// lines that straddle two row blocks are fetched once per L2.
//
// The operation is a policy Op:
//   A2, B2      global elements of A / B are pairs (else doubles)
//   AL, BL      doubles per element in LDS (BL = 0: no B operand)
//   PAD16       the chains run over k rounded up to 16 with zero operands
//               (the tiles' k-slices: a zero term can turn -0 into +0)
//   double2 a(double2 v, int row, int kk), double2 b(double2 v)   conversions
//   struct Acc, init(Acc&, row, col), step(Acc&, double2 a, double2 b),
//   done(Acc, row, col)
#pragma once

#include "vcphip_device.h"

// Register target of the kernels built on this: up to four waves per SIMD.  The
// upper limit is also the most a SIMD will hold (the compiler reserves the
// registers of that many), so a limit of two, enough for one row block's loads
// in flight, kept the other workgroups of a batch, and those of other streams,
// off the CU: a batch of 64 solves' row sums 100 against 49 us with four, its
// bounds 88 against 66, R mid(b) 155 against 67, 4000 x 4000 times 4 vectors
// in three streams 65 against 54.  Eight: as four.
#define VCPHIP_THIN_WAVES __attribute__((amdgpu_waves_per_eu(1, 4)))

constexpr int VCPHIP_THIN_R = 8;    // rows of a workgroup
constexpr int VCPHIP_THIN_CL = 8;   // column lanes of the chain wave

template <class Op, int CW, int CPT = 1>
struct VcphipThin {
  static constexpr int R = VCPHIP_THIN_R, WC = VCPHIP_THIN_CL * CPT, NC = WC * CW;
  static constexpr int LW = CW == 1 ? 3 : CW == 2 ? 2 : 4;   // loading waves
  static constexpr int NW = CW + LW, NT = 64 * NW;           // waves and threads of the workgroup
  static constexpr int KB = CW == 1 ? 96 : NC <= 32 ? 64 : 32;   // k per stage
  static constexpr int NL = 64 * LW;
  static constexpr int NCP = NC + 1;                   // LDS row of B: an odd stride spreads its column-wise stores
  static constexpr int APT = KB * R / NL, BPT = Op::BL ? KB * NC / NL : 0;
  static constexpr int BLN = Op::BL ? Op::BL : 1;
  static_assert(KB % 16 == 0 && APT * NL == KB * R && (!Op::BL || BPT * NL == KB * NC) && NL % KB == 0, "stage shape");
  struct Lds {
    double a[2][KB * R * Op::AL];
    double b[2][Op::BL ? KB * NCP * BLN : 2];
  };

  static constexpr int U = CPT == 1 ? 16 : 8;   // k per register set of the chains
  struct Set {   // the LDS operands of U consecutive k
    double2 a[U], b[U][CPT];
  };

  // rows row0 .. row0 + 7 and columns col0 .. col0 + NC - 1 of the m x n
  // output; the chain waves are rot .. rot + CW - 1 (mod NW)
  static VCPHIP_DEVINL void run(Op& op, Lds& L, int m, int n, int k, int row0, int col0, int rot) {
    const int kp = Op::PAD16 ? (k + 15) / 16 * 16 : k;
    const int nt = (kp + KB - 1) / KB;
    const int w0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) - rot;
    const int cw = w0 < 0 ? w0 + NW : w0, lane = threadIdx.x & 63;
    if (cw >= CW) {
      // loader: thread = one row (rows past m re-read the last one, nothing
      // of them is stored) and APT k; and BPT elements of B along k, columns
      // past n skipped (a thread's columns differ by NL / KB)
      const int tid = 64 * (cw - CW) + lane;
      const int lrow = row0 + (tid & (R - 1)) < m ? row0 + (tid & (R - 1)) : m - 1;
      const int lk = tid / R, bk = tid % KB, bc = tid / KB;
      const double* pa = op.A + (Op::A2 ? 2 : 1) * (long)lrow;
      struct Regs {
        double2 a[APT], b[BPT ? BPT : 1];
      };
      auto load = [&](Regs& g, int k0) {
        if (k0 >= kp) return;
        const bool whole = k0 + KB <= k;
#pragma unroll
        for (int q = 0; q < APT; ++q) {
          int kk = k0 + lk + (NL / R) * q;
          if (!whole && kk >= k) kk = k - 1;   // past k: zeroed in store()
          if (Op::A2) g.a[q] = *reinterpret_cast<const double2*>(pa + 2 * op.lda * kk);
          else g.a[q].x = pa[op.lda * kk];
        }
#pragma unroll
        for (int q = 0; q < BPT; ++q) {
          const int c = col0 + bc + (NL / KB) * q;
          if (c >= n) break;
          int kk = k0 + bk;
          if (!whole && kk >= k) kk = k - 1;
          if (Op::B2) g.b[q] = *reinterpret_cast<const double2*>(op.B + 2 * (kk + op.ldb * c));
          else g.b[q].x = op.B[kk + op.ldb * c];
        }
      };
      auto store = [&](const Regs& g, int buf, int k0) {
        if (k0 >= kp) return;
        const bool whole = k0 + KB <= k;
#pragma unroll
        for (int q = 0; q < APT; ++q) {
          const int e = tid + NL * q, kk = k0 + lk + (NL / R) * q;
          double2 v = op.a(g.a[q], row0 + (tid & (R - 1)), kk);
          if (!whole && kk >= k) v = make_double2(0.0, 0.0);
          if (Op::AL == 2) *reinterpret_cast<double2*>(&L.a[buf][2 * e]) = v;
          else L.a[buf][e] = v.x;
        }
#pragma unroll
        for (int q = 0; q < BPT; ++q) {
          const int c = bc + (NL / KB) * q;
          if (col0 + c >= n) break;   // lanes past n read what was there and store nothing
          double2 v = op.b(g.b[q]);
          if (!whole && k0 + bk >= k) v = make_double2(0.0, 0.0);
          if (Op::BL == 2) *reinterpret_cast<double2*>(&L.b[buf][2 * (bk * NCP + c)]) = v;
          else L.b[buf][bk * NCP + c] = v.x;
        }
      };
      Regs g;
      load(g, 0);
      store(g, 0, 0);
      load(g, KB);
      for (int t = 0; t < nt; ++t) {
        __syncthreads();   // stage t is in LDS; the other buffer's reads (stage t - 1) are done
        store(g, (t + 1) & 1, (t + 1) * KB);
        load(g, (t + 2) * KB);
      }
      return;
    }
    const int row = lane & (R - 1), cl = cw * WC + lane / R;
    typename Op::Acc acc[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) op.init(acc[j], row0 + row, col0 + cl + VCPHIP_THIN_CL * j);
    const bool some = col0 + cw * WC < n;   // else this wave only keeps the barriers
    for (int t = 0; t < nt; ++t) {
      __syncthreads();
      if (!some) continue;
      const double* la = L.a[t & 1] + Op::AL * row;
      const double* lb = L.b[t & 1] + Op::BL * cl;
      const int kc = kp - t * KB < KB ? kp - t * KB : KB;
      auto rd = [&](double2& av, double2 (&bv)[CPT], int kk) {
        if (Op::AL == 2) av = *reinterpret_cast<const double2*>(la + 2 * R * kk);
        else av.x = la[R * kk];
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
          if (Op::BL == 2) bv[j] = *reinterpret_cast<const double2*>(lb + 2 * (kk * NCP + VCPHIP_THIN_CL * j));
          else if (Op::BL == 1) bv[j].x = lb[kk * NCP + VCPHIP_THIN_CL * j];
        }
      };
      auto read = [&](Set& s, int kk) {
#pragma unroll
        for (int u = 0; u < U; ++u) rd(s.a[u], s.b[u], kk + u);
      };
      auto chains = [&](const Set& s) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < CPT; ++j) op.step(acc[j], s.a[u], s.b[u][j]);
      };
      int kk = 0;
      for (; kk + U <= kc; kk += U) {
        Set s0;
        read(s0, kk);
        chains(s0);
      }
      for (; kk < kc; ++kk) {
        double2 av, bv[CPT];
        rd(av, bv, kk);
#pragma unroll
        for (int j = 0; j < CPT; ++j) op.step(acc[j], av, bv[j]);
      }
    }
    if (!some) return;
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const int r = row0 + row, c = col0 + cl + VCPHIP_THIN_CL * j;
      if (r < m && c < n) op.done(acc[j], r, c);
    }
  }
};

// the chains of the plain products (the tiles': the same operations in the
// same order, so the same bits); round-up mode
template <bool AI, bool BI>
struct VcphipThinDr {
  static constexpr bool A2 = AI, B2 = BI, PAD16 = true;
  static constexpr int AL = AI ? 2 : 1, BL = BI ? 2 : 1;
  const double* __restrict__ A;
  const double* __restrict__ B;
  long lda, ldb;
  struct Acc {
    double up, dn, r1, r2;
  };
  VCPHIP_DEVINL double2 a(double2 v, int, int) const {
    if (AI) {
      double mm, rr;
      vcphip_midrad_ru(v.x, v.y, mm, rr);
      return make_double2(mm, rr);
    }
    return v;
  }
  VCPHIP_DEVINL double2 b(double2 v) const {
    if (BI) {
      double mm, rr;
      vcphip_midrad_ru(v.x, v.y, mm, rr);
      return make_double2(mm, rr);
    }
    return v;
  }
  VCPHIP_DEVINL void init(Acc& c, int, int) const { c.up = c.dn = c.r1 = c.r2 = 0.0; }
  VCPHIP_DEVINL void step(Acc& c, double2 av, double2 bv) const {
    c.up = __builtin_fma(av.x, bv.x, c.up);
    c.dn = __builtin_fma(-av.x, bv.x, c.dn);
    if (AI && BI) {
      const double as = __builtin_fabs(av.x) + av.y;
      c.r1 = __builtin_fma(as, bv.y, c.r1);
      c.r2 = __builtin_fma(av.y, __builtin_fabs(bv.x), c.r2);
    } else if (AI) {
      c.r1 = __builtin_fma(av.y, __builtin_fabs(bv.x), c.r1);
    } else if (BI) {
      c.r1 = __builtin_fma(__builtin_fabs(av.x), bv.y, c.r1);
    }
  }
  // {lower, upper} from the chains, the reference's fix-ups in its order
  VCPHIP_DEVINL double2 result(const Acc& c) const {
    const double t = AI && BI ? c.r1 + c.r2 : c.r1;
    const double hi = c.up + t;
    const double nlo = c.dn + t;
    return make_double2(-nlo, hi);
  }
};
