// Exact symmetric Chinese-remainder reconstruction for the Ozaki scheme II
// kernels (interval and double-double forms).
//
// The residues u_t = X mod m_t (t < N) of an integer X with |X| < M/2 - the
// splitting parameter beta guarantees |X| <= (M/2) 2^-1e-6 (interval) or
// |X| < M/4 (dd) - determine X as
//     S = sum_t u_t w_t,   w_t = (M/m_t) ((M/m_t)^-1 mod m_t),
//     X = S - q M,         q = round(S / M) = floor(sum_t u_t (w_t / M) + 1/2).
// Both sums are byte-column sums, formed on the matrix cores:
//     col_c = sum_t u_t * byte c of w_t             (c < N, w_t < M < 2^(8 N))
//     fc_b  = sum_t u_t * byte b of F_t,   F_t = floor(2^48 w_t / M)   (b < 6)
// so S = sum_c col_c 2^(8c) and q = floor((sum_b fc_b 2^(8b) + 2^47) / 2^48).
// Each F_t is within 2^-48 of w_t / M, so with u_t < 256 and N <= 32 the
// fixed-point quotient is within 2^-35 of S / M, which stays at least 3.4e-7
// (interval) or 1/4 (dd) away from a half-integer: q is exact.  X is formed
// modulo 2^(32 NL), which suffices because |X| < 2^(32 NL - 1).
//
// The column sums are integer matrix products of int8 operands:
// sum_t u_t v_t = sum_t (u_t - 128)(v_t - 128) + 128 sum_t u_t + K, with
// K = 128 sum_t v_t - 128^2 N a per-column constant.  One
// v_mfma_i32_32x32x32_i8 handles the 64 elements of a wave (one per lane)
// against 16 columns and 16 residues: output row r holds column
// 4 (r / 8) + r % 4 of element group (r / 4) % 2, so a lane's accumulator
// register v is column v of its own element.  Its B operand is the lane's own
// 16 centred residues (k-slots of lane half h carry element group h), and the
// A operand of lane half h is zero in the rows of the other group, which
// keeps the two groups apart.  The table's columns are the six quotient
// bytes (0 .. 5), a column of ones (6), which gives sum_t (u_t - 128), and
// the N weight bytes (7 .. N + 6).  This replaces O(N^2 / 4) byte dot
// products and N double-precision multiply-adds per element by
// ceil((N + 7) / 16) x ceil(N / 16) matrix instructions per 64 elements.
// Every lane of the wave must execute them (the kernels keep all lanes
// through them and mask their stores).
#pragma once

#include "vcphip_device.h"
#include "vcphip_kernels.h"

typedef int vcphip_v4i __attribute__((ext_vector_type(4)));
typedef int vcphip_v16i __attribute__((ext_vector_type(16)));

// The per-lane A operands (weights) of the CRT products.
template <int N>
struct VcphipCrtOps {
  static constexpr int NC = N + 7;           // 6 quotient bytes, the residue sum, N weight bytes
  static constexpr int CH = (NC + 15) / 16;  // 16-column groups
  static constexpr int RH = (N + 15) / 16;   // 16-residue groups
  static_assert(16 * CH <= VCPHIP_OZ_CRTCOL && 4 * RH <= VCPHIP_OZ_MAXMOD / 4, "CRT table");
  vcphip_v4i a[CH][RH];
};

template <int N>
VCPHIP_DEVINL void vcphip_crt_ops_load(const VcphipOzParams& P, VcphipCrtOps<N>& T) {
  const unsigned lane = threadIdx.x & 63u;
  const unsigned h = lane >> 5, r = lane & 31u;
  const bool mine = ((r >> 2) & 1u) == h;
  const unsigned cl = 4 * (r >> 3) + (r & 3u);
#pragma unroll
  for (int ch = 0; ch < T.CH; ++ch)
#pragma unroll
    for (int rh = 0; rh < T.RH; ++rh)
      T.a[ch][rh] = mine ? *reinterpret_cast<const vcphip_v4i*>(&P.crt_a[16 * ch + cl][4 * rh]) : vcphip_v4i{0, 0, 0, 0};
}

// The B operands (centred residues) of elements e0 .. e0 + EL - 1 of the four
// elements 4 lane .. 4 lane + 3 that this lane reads of a 16 x 16 plane block
// (rows 4 (lane / 16) .. + 3 of column lane % 16): EL = 4 (e0 = 0), or EL = 1
// with a wave-uniform e0.  One word per plane, from a scalar resource at the
// lane's offset (U: the block's base in the first plane, wave-uniform), and
// 4 x 4 byte transposes of four planes' words.
template <int N, int EL>
VCPHIP_DEVINL void vcphip_crt_operands(const uint8_t* __restrict__ U, long plane, unsigned lane, int e0,
                                       vcphip_v4i (&b)[EL][VcphipCrtOps<N>::RH]) {
  constexpr int RH = VcphipCrtOps<N>::RH;
  static_assert(EL == 1 || EL == 4, "elements per lane");
  unsigned w[16 * RH];
#pragma unroll
  for (int t = 0; t < 16 * RH; ++t)   // bytes past N meet zero weights
    w[t] = t < N ? __builtin_amdgcn_raw_buffer_load_b32(vcphip_rsrc(U + (long)t * plane, 256), 4 * lane, 0, 0) : 0u;
  constexpr unsigned LO = 0x05010400u, HI = 0x07030602u, EVEN = 0x05040100u, ODD = 0x07060302u;
  const unsigned s1 = e0 & 2 ? HI : LO, s2 = e0 & 1 ? ODD : EVEN;   // EL = 1
#pragma unroll
  for (int t = 0; t < 16 * RH; t += 4) {
    if (t >= N) {
#pragma unroll
      for (int e = 0; e < EL; ++e) b[e][t / 16][t % 16 / 4] = 0;
      continue;
    }
    if (EL == 1) {
      const unsigned x01 = __builtin_amdgcn_perm(w[t + 1], w[t], s1), x23 = __builtin_amdgcn_perm(w[t + 3], w[t + 2], s1);
      b[0][t / 16][t % 16 / 4] = (int)(__builtin_amdgcn_perm(x23, x01, s2) ^ 0x80808080u);   // u - 128 as int8
      continue;
    }
#pragma unroll
    for (int y = 0; y < 4; ++y) w[t + y] ^= 0x80808080u;
    const unsigned l01 = __builtin_amdgcn_perm(w[t + 1], w[t], LO), h01 = __builtin_amdgcn_perm(w[t + 1], w[t], HI);
    const unsigned l23 = __builtin_amdgcn_perm(w[t + 3], w[t + 2], LO), h23 = __builtin_amdgcn_perm(w[t + 3], w[t + 2], HI);
#pragma unroll
    for (int e = 0; e < EL; ++e)
      b[e][t / 16][t % 16 / 4] = (int)__builtin_amdgcn_perm(e < 2 ? l23 : h23, e < 2 ? l01 : h01, e & 1 ? ODD : EVEN);
  }
}

// From the residues of this lane's X (its operands b): returns the sign of X
// and its magnitude in NL little-endian 32-bit limbs.
template <int N, int NL>
VCPHIP_DEVINL bool vcphip_crt_limbs(const vcphip_v4i (&b)[VcphipCrtOps<N>::RH], const VcphipCrtOps<N>& T,
                                    const VcphipOzParams& P, unsigned (&mag)[NL]) {
  static_assert(N <= 4 * NL, "byte columns beyond the limbs");
  constexpr int CH = VcphipCrtOps<N>::CH, RH = VcphipCrtOps<N>::RH;
  // column group 0 first: its columns 0..6 are the quotient bytes and the
  // residue sum, so q is known before the weight columns (7 .. N + 6) of the
  // later groups are formed, and one group's accumulators are live at a time
  vcphip_v16i acc = vcphip_v16i{};
#pragma unroll
  for (int rh = 0; rh < RH; ++rh) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a[0][rh], b[rh], acc, 0, 0, 0);
  const unsigned s128 = 128u * (unsigned)(acc[6] + 128 * N);   // 128 sum_t u_t
  // two byte columns at a time: col_c + 2^8 col_(c+1) < 2^30, with the centring
  // terms of both added at once
  const unsigned s2 = s128 * 257u;
  auto pair = [&](int g, int v) {
    const unsigned kk = (unsigned)P.crt_k[16 * g + v] + ((unsigned)P.crt_k[16 * g + v + 1] << 8);
    return (((unsigned)acc[v + 1] << 8) + (unsigned)acc[v]) + (s2 + kk);
  };
  // q = floor((sum_b fc_b 2^(8b) + 2^47) / 2^48)
  const unsigned q = (pair(0, 4) + 0x8000u + ((pair(0, 2) + (pair(0, 0) >> 16)) >> 16)) >> 16;
  // limb l = low pair + 2^16 high pair - q M_l
  long long limb[NL];
#pragma unroll
  for (int l = 0; l < NL; ++l) limb[l] = -(long long)((unsigned long long)q * P.Mlimb[l]);
  unsigned half[2 * NL];
#pragma unroll
  for (int h = 0; h < 2 * NL; ++h) half[h] = 0;
#pragma unroll
  for (int ch = 0; ch < CH; ++ch) {
    unsigned last = 0;   // the column that a pair split over two groups begins with
    if (ch > 0) {
      last = (unsigned)acc[15] + s128 + (unsigned)P.crt_k[16 * ch - 1];
      acc = vcphip_v16i{};
#pragma unroll
      for (int rh = 0; rh < RH; ++rh) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a[ch][rh], b[rh], acc, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int c = 16 * ch + v - 7;   // weight byte c
      if (c < 0 || c >= N) continue;
      if (c % 2 == 0 && c + 1 < N && v + 1 < 16) half[c >> 1] = pair(ch, v);
      else if (c % 2 == 0 && c + 1 >= N) half[c >> 1] = (unsigned)acc[v] + s128 + (unsigned)P.crt_k[16 * ch + v];
      else if (c % 2 == 1 && v == 0) half[c >> 1] = last + (((unsigned)acc[v] + s128 + (unsigned)P.crt_k[16 * ch]) << 8);
    }
  }
#pragma unroll
  for (int l = 0; l < NL; ++l)
    limb[l] += (long long)((unsigned long long)half[2 * l] + ((unsigned long long)half[2 * l + 1] << 16));
  long long carry = 0;
#pragma unroll
  for (int l = 0; l < NL; ++l) {
    const long long acc_l = limb[l] + carry;
    mag[l] = (unsigned)acc_l;
    carry = acc_l >> 32;
  }
  const bool neg = (int)mag[NL - 1] < 0;
  if (neg) {
    unsigned long long c = 1;
#pragma unroll
    for (int l = 0; l < NL; ++l) {
      const unsigned long long v = (unsigned long long)(~mag[l]) + c;
      mag[l] = (unsigned)v;
      c = v >> 32;
    }
  }
  return neg;
}

// A 16 x 16 block of results, EL of its four rows of a column per lane, to C
// through the block's LDS copy: 256 contiguous bytes per column instead of 16
// scattered ones per lane.  EL = 4: a wave's own block; EL = 1: the block of
// the workgroup's four waves, wave e0 holding element e0 of each lane.
struct VcphipBlockOut {
  static constexpr int LD = 17;   // an odd column stride in 16-byte slots
  double2 v[16 * LD];
};
template <int EL>
VCPHIP_DEVINL void vcphip_block_store(VcphipBlockOut& L, const double2 (&v)[EL], unsigned lane, int e0,
                                      double* __restrict__ C, long ldc, int i0, int j0, int m, int n) {
#pragma unroll
  for (int e = 0; e < EL; ++e) L.v[(lane & 15) * VcphipBlockOut::LD + 4 * (lane >> 4) + e0 + e] = v[e];
  if (EL == 4) __builtin_amdgcn_wave_barrier();   // LDS operations of a wave stay in order
  else __syncthreads();
  const int i = i0 + (int)(lane & 15);
#pragma unroll
  for (int e = 0; e < EL; ++e) {
    const int c = 4 * (e0 + e) + (int)(lane >> 4), j = j0 + c;
    if (i < m && j < n)
      *reinterpret_cast<double2*>(C + 2 * (i + ldc * (long)j)) = L.v[c * VcphipBlockOut::LD + (lane & 15)];
  }
}

// Blocks up to which a reconstruction gives each block four waves (EL = 1)
// instead of one.  One wave shares the weights, tables and scalar work of a
// block's elements, four fill the chip and shorten the chain; interval / dd
// form, one against four waves: n = 500 12.4 / 12.4 against 9.2 / 9.9 us, 1000
// 20 / 24 against 18 / 19, 1300 (7744 blocks) 32 / 33 against 28 / 30, 2000
// (16384) 68 / 71 against 73 / 75.
constexpr long VCPHIP_CRT_SPLIT_BLOCKS = 8192;
