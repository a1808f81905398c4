// The chains of the plain products as DPP multiply-adds (gfx950).
//
// v_fmac_f64 takes its first factor through a DPP row broadcast: lane i of
// every row of 16 lanes to the whole row.  A lane therefore needs one
// register pair of A per chain operand for all the rows of its outputs (lane
// i of its DPP row holds A's row i) and one of B (its own column), and one k
// of an RPL x 1 block of outputs is RPL multiply-adds per chain on those
// operands.  Per k a wave reads two 16-byte LDS operands per lane (a (mid,
// rad) pair of A and one of B) for 4 RPL multiply-adds, against 16 / RPL = 8
// reads per 64 multiply-adds with a 4 x 4 block of outputs per lane, whose
// LDS time equalled the multiply-adds' and held the kernels at 0.53 - 0.65 of
// the FP64 rate.  The instruction's rate is the plain multiply-add's (measured
// on MI355X, two waves per SIMD: 64.6 against 68.7 TFLOP/s), it rounds by the
// MODE register, and its sign and magnitude modifiers apply to both factors.
//
// Each block of multiply-adds is one asm statement: the factors' last VALU
// writes and the first DPP read of them need two wait states, which the
// leading s_nop gives whatever the compiler put before it.  The statement
// writes accumulators before it has read its last factor, so they are early
// clobbers: without that an accumulator whose value equals a factor's may share
// its registers.
#pragma once

#include "vcphip_device.h"

#define VCPHIP_DPP_1(acc, i, a, b) \
  "v_fmac_f64_dpp %[" #acc #i "], " a ", " b " row_newbcast:" #i " row_mask:0xf bank_mask:0xf\n\t"
#define VCPHIP_DPP_8(acc, a, b)                                                                         \
  VCPHIP_DPP_1(acc, 0, a, b) VCPHIP_DPP_1(acc, 1, a, b) VCPHIP_DPP_1(acc, 2, a, b)                      \
  VCPHIP_DPP_1(acc, 3, a, b) VCPHIP_DPP_1(acc, 4, a, b) VCPHIP_DPP_1(acc, 5, a, b)                      \
  VCPHIP_DPP_1(acc, 6, a, b) VCPHIP_DPP_1(acc, 7, a, b)
#define VCPHIP_DPP_16(acc, a, b)                                                                        \
  VCPHIP_DPP_8(acc, a, b)                                                                               \
  VCPHIP_DPP_1(acc, 8, a, b) VCPHIP_DPP_1(acc, 9, a, b) VCPHIP_DPP_1(acc, 10, a, b)                     \
  VCPHIP_DPP_1(acc, 11, a, b) VCPHIP_DPP_1(acc, 12, a, b) VCPHIP_DPP_1(acc, 13, a, b)                   \
  VCPHIP_DPP_1(acc, 14, a, b) VCPHIP_DPP_1(acc, 15, a, b)
#define VCPHIP_DPP_O1(acc, i) [acc##i] "+&v"(acc[i])
#define VCPHIP_DPP_O8(acc)                                                                              \
  VCPHIP_DPP_O1(acc, 0), VCPHIP_DPP_O1(acc, 1), VCPHIP_DPP_O1(acc, 2), VCPHIP_DPP_O1(acc, 3),           \
      VCPHIP_DPP_O1(acc, 4), VCPHIP_DPP_O1(acc, 5), VCPHIP_DPP_O1(acc, 6), VCPHIP_DPP_O1(acc, 7)
#define VCPHIP_DPP_O16(acc)                                                                             \
  VCPHIP_DPP_O8(acc), VCPHIP_DPP_O1(acc, 8), VCPHIP_DPP_O1(acc, 9), VCPHIP_DPP_O1(acc, 10),             \
      VCPHIP_DPP_O1(acc, 11), VCPHIP_DPP_O1(acc, 12), VCPHIP_DPP_O1(acc, 13), VCPHIP_DPP_O1(acc, 14),   \
      VCPHIP_DPP_O1(acc, 15)

// one k of the chains of RPL rows x this lane's column.  (am, ar): this
// lane's row of A within its DPP row (mid and rad, or the point in am);
// (bm, br): its column of B.
//   up += am bm, dn += (-am) bm                                     (all forms)
//   II: r1 += (|am| + ar) br, r2 += ar |bm|;  IP: r1 += ar |bm|;  PI: r1 += |am| br
#define VCPHIP_DPP_STEP(RPL)                                                                                       \
  template <bool AI, bool BI>                                                                                      \
  VCPHIP_DEVINL void vcphip_dpp_step(double am, double ar, double bm, double br, double (&up)[RPL],                \
                                     double (&dn)[RPL], double (&r1)[RPL], double (&r2)[RPL]) {                    \
    if (AI && BI) {                                                                                                \
      const double as = __builtin_fabs(am) + ar;                                                                   \
      asm("s_nop 1\n\t" VCPHIP_DPP_##RPL(up, "%[am]", "%[bm]") VCPHIP_DPP_##RPL(dn, "-%[am]", "%[bm]")             \
              VCPHIP_DPP_##RPL(r2, "%[ar]", "|%[bm]|") VCPHIP_DPP_##RPL(r1, "%[as]", "%[br]")                      \
          : VCPHIP_DPP_O##RPL(up), VCPHIP_DPP_O##RPL(dn), VCPHIP_DPP_O##RPL(r1), VCPHIP_DPP_O##RPL(r2)             \
          : [am] "v"(am), [ar] "v"(ar), [as] "v"(as), [bm] "v"(bm), [br] "v"(br));                                 \
    } else if (AI) {                                                                                               \
      asm("s_nop 1\n\t" VCPHIP_DPP_##RPL(up, "%[am]", "%[bm]") VCPHIP_DPP_##RPL(dn, "-%[am]", "%[bm]")             \
              VCPHIP_DPP_##RPL(r1, "%[ar]", "|%[bm]|")                                                             \
          : VCPHIP_DPP_O##RPL(up), VCPHIP_DPP_O##RPL(dn), VCPHIP_DPP_O##RPL(r1)                                    \
          : [am] "v"(am), [ar] "v"(ar), [bm] "v"(bm));                                                             \
    } else if (BI) {                                                                                               \
      asm("s_nop 1\n\t" VCPHIP_DPP_##RPL(up, "%[am]", "%[bm]") VCPHIP_DPP_##RPL(dn, "-%[am]", "%[bm]")             \
              VCPHIP_DPP_##RPL(r1, "|%[am]|", "%[br]")                                                             \
          : VCPHIP_DPP_O##RPL(up), VCPHIP_DPP_O##RPL(dn), VCPHIP_DPP_O##RPL(r1)                                    \
          : [am] "v"(am), [bm] "v"(bm), [br] "v"(br));                                                             \
    } else {                                                                                                       \
      asm("s_nop 1\n\t" VCPHIP_DPP_##RPL(up, "%[am]", "%[bm]") VCPHIP_DPP_##RPL(dn, "-%[am]", "%[bm]")             \
          : VCPHIP_DPP_O##RPL(up), VCPHIP_DPP_O##RPL(dn)                                                           \
          : [am] "v"(am), [bm] "v"(bm));                                                                           \
    }                                                                                                              \
  }                                                                                                                \
  /* one k of the A^T A chains: up += im jm, dn += (-im) jm, tij += |im| jr, tji += |jm| ir, sij += ir jr */       \
  VCPHIP_DEVINL void vcphip_dpp_syrk_step(double im, double ir, double jm, double jr, double (&up)[RPL],           \
                                          double (&dn)[RPL], double (&tij)[RPL], double (&tji)[RPL],               \
                                          double (&sij)[RPL]) {                                                    \
    asm("s_nop 1\n\t" VCPHIP_DPP_##RPL(up, "%[im]", "%[jm]") VCPHIP_DPP_##RPL(dn, "-%[im]", "%[jm]")               \
            VCPHIP_DPP_##RPL(tij, "|%[im]|", "%[jr]") VCPHIP_DPP_##RPL(tji, "%[ir]", "|%[jm]|")                    \
                VCPHIP_DPP_##RPL(sij, "%[ir]", "%[jr]")                                                            \
        : VCPHIP_DPP_O##RPL(up), VCPHIP_DPP_O##RPL(dn), VCPHIP_DPP_O##RPL(tij), VCPHIP_DPP_O##RPL(tji),            \
          VCPHIP_DPP_O##RPL(sij)                                                                                   \
        : [im] "v"(im), [ir] "v"(ir), [jm] "v"(jm), [jr] "v"(jr));                                                 \
  }
VCPHIP_DPP_STEP(8)
VCPHIP_DPP_STEP(16)

// BKS k of a slice in LDS: rd(kk, a, b) reads the operands of one k, step(a, b)
// is its block of multiply-adds.  The reads run two k ahead (a block of 8 rows
// takes about an LDS read's latency); the scheduling barriers keep them there.
template <int BKS, class Rd, class Step>
VCPHIP_DEVINL void vcphip_dpp_slice(const Rd& rd, const Step& step) {
  double2 a[BKS], b[BKS];
  rd(0, a[0], b[0]);
  rd(1, a[1], b[1]);
#pragma unroll
  for (int kk = 0; kk < BKS; ++kk) {
    if (kk + 2 < BKS) rd(kk + 2, a[kk + 2], b[kk + 2]);
    __builtin_amdgcn_sched_barrier(0);
    step(a[kk], b[kk]);
    __builtin_amdgcn_sched_barrier(0);
  }
}
