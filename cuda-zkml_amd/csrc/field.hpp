// BN254 base field Fq and scalar field Fr for gfx950.
//
// Representation (device and host-math builds alike)
// ---------------------------------------------------
// An element is 9 limbs of 29 bits (uint32 each, limb < 2^29), little endian,
// holding a value in the lazy range [0, 2m) for modulus m.  The Montgomery
// radix inside kernels is R' = 2^261 (= 2^(29*9)), not the reference's 2^256:
// with 29-bit limbs every limb product is one v_mad_u64_u32 into a 64-bit
// column accumulator and no carry has to be propagated until the column is
// finished (mont_columns_fit below: at most 61 of 2^64's 64 units of 2^58).  On
// gfx950 the 32x32->64 mad issues at full rate, so the instruction count of
// the multiply is what matters; this layout needs 169 mads and 22 other ops
// (a square 133 and 30) against ~560 instructions for a compiler-lowered
// 8x32-bit CIOS.
//
// At the memory boundary elements are the reference's 32-byte little-endian
// form (4 x u64 = 8 x u32 words), Montgomery form with R = 2^256
// (reference: src/field/montgomery.cuh:33-60, src/field/fp.cuh:322-349).
// from_mont256/to_mont256 convert between the two radices with one multiply
// by a constant (2^266 mod m in, 2^256 mod m out).  For maps that are linear
// over the field (NTT, scaling by a constant prepared in the internal radix)
// the radix cancels and a plain limb repack suffices (repack_in/repack_out).
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#include "const_mul_asm.hpp"
#include "mont_asm.hpp"
#define ZK_HD __host__ __device__ __forceinline__
#else
#define ZK_HD static inline
#endif

namespace zk {

constexpr int NL = 9;
constexpr uint32_t LMASK = (1u << 29) - 1u;

// BN254 base field q = 0x30644e72e131a029b85045b68181585d97816a916871ca8d3c208c16d87cfd47
// (reference src/field/montgomery.cuh:33-38).
struct FqP {
  static constexpr uint32_t MOD[9] = {0x187cfd47u, 0x010460b6u, 0x1c72a34fu, 0x02d522d0u, 0x1585d978u,
                                      0x02db40c0u, 0x00a6e141u, 0x0e5c2634u, 0x0030644eu};
  static constexpr uint32_t MOD2[9] = {0x10f9fa8eu, 0x0208c16du, 0x18e5469eu, 0x05aa45a1u, 0x0b0bb2f0u,
                                       0x05b68181u, 0x014dc282u, 0x1cb84c68u, 0x0060c89cu};
  static constexpr uint32_t MOD3[9] = {0x0976f7d5u, 0x030d2224u, 0x1557e9edu, 0x087f6872u, 0x00918c68u,
                                       0x0891c242u, 0x01f4a3c3u, 0x0b14729cu, 0x00912cebu};
  static constexpr uint32_t MOD4[9] = {0x01f3f51cu, 0x041182dbu, 0x11ca8d3cu, 0x0b548b43u, 0x161765e0u,
                                       0x0b6d0302u, 0x029b8504u, 0x197098d0u, 0x00c19139u};
  static constexpr uint32_t MOD6[9] = {0x12edefaau, 0x061a4448u, 0x0aafd3dau, 0x10fed0e5u, 0x012318d0u,
                                       0x11238484u, 0x03e94786u, 0x1628e538u, 0x012259d6u};
  static constexpr uint32_t MOD8[9] = {0x03e7ea38u, 0x082305b6u, 0x03951a78u, 0x16a91687u, 0x0c2ecbc0u,
                                       0x16da0605u, 0x05370a08u, 0x12e131a0u, 0x01832273u};
  static constexpr uint32_t INV = 0x04866389u;  // -q^-1 mod 2^29
  static constexpr uint32_t EDIG[9] = {0x02e38790u, 0x0d1e68dcu, 0x148e556bu, 0x10c54699u, 0x0f93f7a8u,
                                       0x02d6db27u, 0x05f64f9au, 0x1010b67bu, 0x015995e9u};  // (q k + 1) / 2^29, k = -q^-1 mod 2^32
  static constexpr uint32_t ONE[9] = {0x157ccc21u, 0x141c2758u, 0x185230d3u, 0x014c0419u, 0x0aa36fb9u,
                                      0x1d4240ceu, 0x11d54c07u, 0x052ac7a8u, 0x000dc836u};  // 2^261 mod q
  static constexpr uint32_t R2[9] = {0x059bac10u, 0x0d1503a3u, 0x018016b8u, 0x10ab0ca8u, 0x02632639u,
                                     0x02c0169fu, 0x169bfd53u, 0x11869d4cu, 0x002a11a6u};  // 2^522 mod q
  static constexpr uint32_t K_IN[9] = {0x13349ca1u, 0x1a5d84a8u, 0x0a3e5cacu, 0x100249e0u, 0x12b951e8u,
                                       0x0e92d304u, 0x14cb95b3u, 0x041b9d3du, 0x00058003u};  // 2^266 mod q
  static constexpr uint32_t K_OUT[9] = {0x058f0d9du, 0x1aea1c6eu, 0x11c2cf74u, 0x11d651ebu, 0x1462c0a7u,
                                        0x11b7bc3cu, 0x1cbd99bau, 0x183340fbu, 0x000e0a77u};  // 2^256 mod q
};

// BN254 scalar field r = 0x30644e72e131a029b85045b68181585d2833e84879b9709143e1f593f0000001
// (reference src/field/fp.cuh:329-335).
struct FrP {
  static constexpr uint32_t MOD[9] = {0x10000001u, 0x1f0fac9fu, 0x0e5c2450u, 0x07d090f3u, 0x1585d283u,
                                      0x02db40c0u, 0x00a6e141u, 0x0e5c2634u, 0x0030644eu};
  static constexpr uint32_t MOD2[9] = {0x00000002u, 0x1e1f593fu, 0x1cb848a1u, 0x0fa121e6u, 0x0b0ba506u,
                                       0x05b68181u, 0x014dc282u, 0x1cb84c68u, 0x0060c89cu};
  static constexpr uint32_t MOD3[9] = {0x10000003u, 0x1d2f05deu, 0x0b146cf2u, 0x1771b2dau, 0x00917789u,
                                       0x0891c242u, 0x01f4a3c3u, 0x0b14729cu, 0x00912cebu};
  static constexpr uint32_t MOD4[9] = {0x00000004u, 0x1c3eb27eu, 0x19709143u, 0x1f4243cdu, 0x16174a0cu,
                                       0x0b6d0302u, 0x029b8504u, 0x197098d0u, 0x00c19139u};
  static constexpr uint32_t MOD6[9] = {0x00000006u, 0x1a5e0bbdu, 0x1628d9e5u, 0x0ee365b4u, 0x0122ef13u,
                                       0x11238484u, 0x03e94786u, 0x1628e538u, 0x012259d6u};
  static constexpr uint32_t MOD8[9] = {0x00000008u, 0x187d64fcu, 0x12e12287u, 0x1e84879bu, 0x0c2e9419u,
                                       0x16da0605u, 0x05370a08u, 0x12e131a0u, 0x01832273u};
  static constexpr uint32_t INV = 0x0fffffffu;  // -r^-1 mod 2^29
  static constexpr uint32_t EDIG[9] = {0x08f05368u, 0x1a996a5bu, 0x13e27f6bu, 0x15166c9eu, 0x1e906a17u,
                                       0x04c58463u, 0x16877334u, 0x0b82ba37u, 0x016af04cu};  // (r k + 1) / 2^29, k = -r^-1 mod 2^32
  static constexpr uint32_t NEGMOD[9] = {0x0fffffffu, 0x00f05360u, 0x11a3dbafu, 0x182f6f0cu, 0x0a7a2d7cu,
                                         0x1d24bf3fu, 0x1f591ebeu, 0x11a3d9cbu, 0x1fcf9bb1u};  // 2^261 - r
  static constexpr uint32_t NINV[9] = {0x0fffffffu, 0x170fac9fu, 0x1a446cf0u, 0x0d0c9698u, 0x02391658u,
                                       0x0c144c83u, 0x06cb8e6au, 0x03a1b068u, 0x1273f82fu};  // -r^-1 mod 2^261
  static constexpr uint32_t ONE[9] = {0x0fffff57u, 0x1ea70ab4u, 0x052c068bu, 0x17504f49u, 0x0aa8075bu,
                                      0x1d4240ceu, 0x11d54c07u, 0x052ac7a8u, 0x000dc836u};  // 2^261 mod r
  static constexpr uint32_t R2[9] = {0x05b69bd4u, 0x06170a5au, 0x020cddceu, 0x1db6310bu, 0x0e54d0ffu,
                                     0x1cf855e3u, 0x1c15e103u, 0x07d09161u, 0x000a054au};  // 2^522 mod r
  static constexpr uint32_t K_IN[9] = {0x0fffead7u, 0x1d5444f4u, 0x04438aa5u, 0x03b4d096u, 0x134c84dau,
                                       0x0e92d304u, 0x14cb95b3u, 0x041b9d3du, 0x00058003u};  // 2^266 mod r
  static constexpr uint32_t K_OUT[9] = {0x0ffffffbu, 0x04b1a0e2u, 0x18334a6bu, 0x18ed2b3eu, 0x1462e36fu,
                                        0x11b7bc3cu, 0x1cbd99bau, 0x183340fbu, 0x000e0a77u};  // 2^256 mod r
};

template <class P>
struct fe {
  uint32_t l[NL];
};

using fq = fe<FqP>;
using fr = fe<FrP>;

template <class P>
ZK_HD fe<P> fe_zero() {
  fe<P> r;
#pragma unroll
  for (int i = 0; i < NL; i++) r.l[i] = 0;
  return r;
}

template <class P>
ZK_HD fe<P> fe_const(const uint32_t (&c)[NL]) {
  fe<P> r;
#pragma unroll
  for (int i = 0; i < NL; i++) r.l[i] = c[i];
  return r;
}

template <class P>
ZK_HD fe<P> fe_one() {
  return fe_const<P>(P::ONE);
}

// Montgomery products sum_t a[t] b[t] 2^-261 mod m in column (product-scanning)
// order, the reduction interleaved.  acc holds one column of 29 bits plus what
// the columns below carried into it.
//   Columns 0..6: the digit is the column's low 32 bits as they are.  With
//   k = -m^-1 mod 2^32, q (m k) clears them, and q (m k + 1) = q 2^29 EDIG adds
//   q EDIG_j to column K + 1 + j; what is left of the column, its high 32
//   bits, goes on as 8 hi (2^32 = 8 * 2^29).  No multiply and no mask for the
//   digit.  Digit 6 counts at most 2^(32 + 174) m k < 2^(238) m in the sum that
//   is divided by 2^261, so these digits add less than m / 2^22 to the result.
//   Columns 7, 8: the ordinary digit q = acc (-m^-1) mod 2^29 with multiplier
//   m; digit 8 adds less than m to the result.
//   Columns 9..16: output limbs.
// Columns stay below 2^64: the operands' products (limbs below 2^29: up to
// 9 N of 2^58; one operand's or the square's limbs may be below 2^30), the
// digits' 2^32 EDIG_j (column 8 has the most, 22.8 * 2^58 for q and 34.3 *
// 2^58 for r), two digit products below 2^58 and the carry: for q at most
// 36 + 22.8 + 2.1 (four products, or one square of limbs below 2^30), for r
// 18 + 34.3 + 2.1, in units of 2^58 of 64 (mont_columns_fit).
constexpr int MONT_ND = 7;  // columns with a 32-bit digit

template <class P>
constexpr bool mont_columns_fit(int products_2p58) {
  bool ok = true;
  for (int K = 0; K < 2 * NL - 1; K++) {
    unsigned __int128 s = (unsigned __int128)products_2p58 << 58;
    for (int i = 0; i < MONT_ND && i < K; i++)
      if (K - 1 - i < NL) s += (unsigned __int128)0xffffffffu * P::EDIG[K - 1 - i];
    s += (unsigned __int128)2 << 58;  // digits 7 and 8
    s += (unsigned __int128)1 << 36;  // carry
    ok = ok && (s >> 64) == 0;
  }
  return ok;
}
static_assert(mont_columns_fit<FqP>(36), "Fq column accumulator bound");
static_assert(mont_columns_fit<FrP>(18), "Fr column accumulator bound");

#if !defined(__HIP_DEVICE_COMPILE__)
// cols(K): the sum of the operands' products of column K.  Every loop has constant
// bounds, so that all of it unrolls into straight-line code: with the columns' own
// bounds a product took 109 ns (now 59) on the host that prepares calls.
template <class P, class Cols>
static inline fe<P> mont_columns(Cols&& cols) {
  uint32_t q[NL];
  fe<P> r;
  uint64_t acc = 0;
#pragma unroll
  for (int k = 0; k < 2 * NL - 1; k++) {
    acc += cols(k);
#pragma unroll
    for (int i = 0; i < NL; i++) {
      if (i < MONT_ND && i < k && k - 1 - i < NL) acc += (uint64_t)q[i] * P::EDIG[k - 1 - i];
      if (i >= MONT_ND && i < k && k - i < NL) acc += (uint64_t)q[i] * P::MOD[k - i];
    }
    if (k < MONT_ND) {
      q[k] = (uint32_t)acc;
      acc = (acc >> 32) * 8;
      continue;
    }
    if (k < NL) {
      q[k] = ((uint32_t)acc * P::INV) & LMASK;
      acc += (uint64_t)q[k] * P::MOD[0];
    } else {
      r.l[k - NL] = (uint32_t)acc & LMASK;
    }
    acc >>= 29;
  }
  r.l[NL - 1] = (uint32_t)acc;
  return r;
}
#endif

// Montgomery product a*b*2^-261 mod m.  Inputs: limbs < 2^29, of one operand
// < 2^30 (of both over Fq).  Output: limbs < 2^29, value < a*b/2^261 + m +
// m/2^22, so below 2m for values < 8m, and also when one operand is below m
// and the other anywhere below 2^261 - 2^239.
template <class P>
ZK_HD fe<P> fmul(const fe<P>& a, const fe<P>& b) {
#if defined(__HIP_DEVICE_COMPILE__)
  fe<P> r = a;  // in place when a is dead after the product
  mont_mul_asm<P>(r.l, b.l);
  return r;
#else
  return mont_columns<P>([&](int k) {
    uint64_t s = 0;
#pragma unroll
    for (int i = 0; i < NL; i++)
      if (k - i >= 0 && k - i < NL) s += (uint64_t)a.l[i] * b.l[k - i];
    return s;
  });
#endif
}

// sum_t a[t]*b[t] * 2^-261 mod q, N = 2 or 4, with one Montgomery reduction
// for all products.  Inputs: normalized limbs (< 2^29), with N = 2 of one
// factor below 2^30 (fneg_wide); the sum of the products below 100 q^2.  The
// result is below 100 q^2 / 2^261 + q + q/2^22 < 1.6 q.
template <class P, int N>
ZK_HD fe<P> fmul_sum(const fe<P> (&a)[N], const fe<P> (&b)[N]) {
  static_assert(N == 2 || N == 4, "products of one reduction");
  static_assert(mont_columns_fit<P>(N == 2 ? 27 : 36), "column accumulator bound");
#if defined(__HIP_DEVICE_COMPILE__)
  fe<P> r = a[0];  // in place when a[0] is dead after the products
  if constexpr (N == 2)
    mont_mul2_asm<P>(r.l, b[0].l, a[1].l, b[1].l);
  else
    mont_mul4_asm<P>(r.l, b[0].l, a[1].l, b[1].l, a[2].l, b[2].l, a[3].l, b[3].l);
  return r;
#else
  return mont_columns<P>([&](int k) {
    uint64_t s = 0;
#pragma unroll
    for (int t = 0; t < N; t++) {
#pragma unroll
      for (int i = 0; i < NL; i++)
        if (k - i >= 0 && k - i < NL) s += (uint64_t)a[t].l[i] * b[t].l[k - i];
    }
    return s;
  });
#endif
}

// (a*b + c*e) * 2^-261 mod m: fmul_sum of two products (values < 4m).
template <class P>
ZK_HD fe<P> fmul2(const fe<P>& a, const fe<P>& b, const fe<P>& c, const fe<P>& e) {
  const fe<P> x[2] = {a, c}, y[2] = {b, e};
  return fmul_sum<P, 2>(x, y);
}

// Squaring: every cross product once, by the doubled limb (limbs < 2^30 over
// Fq, < 2^29 over Fr).
template <class P>
ZK_HD fe<P> fsqr(const fe<P>& a) {
#if defined(__HIP_DEVICE_COMPILE__)
  fe<P> r;
  mont_sqr_asm<P>(r.l, a.l);
  return r;
#else
  return mont_columns<P>([&](int k) {
    uint64_t s = 0;
#pragma unroll
    for (int i = 0; i < NL; i++)
      if (2 * i < k && k - i < NL) s += (uint64_t)a.l[i] * (2 * a.l[k - i]);
    if (k % 2 == 0) s += (uint64_t)a.l[k / 2] * a.l[k / 2];
    return s;
  });
#endif
}

// a w mod m for a constant w (canonical, not Montgomery) with its quotient wq =
// floor(w 2^261 / m): q = floor(a wq / 2^261) from the columns 7 and up of a wq,
// then a w - q m from the low nine columns, modulo 2^261.  The dropped columns
// and the two floors leave q short by less than 2 + 2^-22, so the result is in
// [0, 2m + m / 2^22), limbs normalized.  a: any value below 2^261 with limbs
// below LU 2^29 (not normalized).  Columns stay below 2^64: a's products 9 LU
// 2^58, the quotient's 5.6 * 2^58, with LU <= 5.  Up to LU = 3 the quotient
// digits may be the columns' low 32 bits as they are (8 * hi goes on, as in the
// Montgomery products): their products take 36.9 * 2^58 in column 7 (in column 8
// only the low bits count).
template <int LU, class P>
ZK_HD fe<P> fmul_const(const fe<P>& a, const fe<P>& w, const fe<P>& wq) {
  static_assert(LU >= 1 && LU <= 5, "limb bound");
#if defined(__HIP_DEVICE_COMPILE__)
  fe<P> r = wq;
  if constexpr (LU <= 3)
    const_mul32_asm<P>(r.l, a.l, w.l);
  else
    const_mul29_asm<P>(r.l, a.l, w.l);
  return r;
#else
  uint32_t q[NL];
  fe<P> r;
  uint64_t acc = 0;
  for (int k = NL - 2; k < 2 * NL - 1; k++) {
    for (int i = k < NL ? 0 : k - NL + 1; i < NL && i <= k; i++) acc += (uint64_t)a.l[i] * wq.l[k - i];
    if (k < NL) {
      acc >>= 29;
    } else if (LU <= 3) {
      q[k - NL] = (uint32_t)acc;
      acc = (acc >> 32) * 8;
    } else {
      q[k - NL] = (uint32_t)acc & LMASK;
      acc >>= 29;
    }
  }
  q[NL - 1] = (uint32_t)acc;
  acc = 0;
  for (int k = 0; k < NL; k++) {
    for (int i = 0; i <= k; i++) acc += (uint64_t)a.l[i] * w.l[k - i] + (uint64_t)q[i] * P::NEGMOD[k - i];
    r.l[k] = (uint32_t)acc & LMASK;
    acc >>= 29;
  }
  return r;
#endif
}

// wq = floor(w 2^261 / m) for w in internal form wi = w 2^261 mod m (canonical):
// w 2^261 = wq m + wi, so wq = wi (-m^-1) modulo 2^261.
template <class P>
ZK_HD fe<P> const_quotient(const fe<P>& wi) {
  fe<P> r;
  uint64_t acc = 0;
  for (int k = 0; k < NL; k++) {
    for (int i = 0; i <= k; i++) acc += (uint64_t)wi.l[i] * P::NINV[k - i];
    r.l[k] = (uint32_t)acc & LMASK;
    acc >>= 29;
  }
  return r;
}

// keep ? a : b.  On the device nine v_cndmask with the mask in a scalar register
// pair: the compiler's form of nine selects on one condition reads it from VCC
// back to back, where each takes 15 to 23 cycles on gfx950 instead of 4.  (s_nop:
// the two wait states between a compare that writes the pair and its first
// reader, which the compiler does not place before an assembly block.)
template <class P>
ZK_HD fe<P> fselect(bool keep, const fe<P>& a, const fe<P>& b) {
#if defined(__HIP_DEVICE_COMPILE__)
  fe<P> r = b;
  const uint64_t mask = __ballot(keep);
  asm("s_nop 1\n"
      "v_cndmask_b32_e64 %0, %0, %9, %18\n"
      "v_cndmask_b32_e64 %1, %1, %10, %18\n"
      "v_cndmask_b32_e64 %2, %2, %11, %18\n"
      "v_cndmask_b32_e64 %3, %3, %12, %18\n"
      "v_cndmask_b32_e64 %4, %4, %13, %18\n"
      "v_cndmask_b32_e64 %5, %5, %14, %18\n"
      "v_cndmask_b32_e64 %6, %6, %15, %18\n"
      "v_cndmask_b32_e64 %7, %7, %16, %18\n"
      "v_cndmask_b32_e64 %8, %8, %17, %18\n"
      : "+&v"(r.l[0]), "+&v"(r.l[1]), "+&v"(r.l[2]), "+&v"(r.l[3]), "+&v"(r.l[4]), "+&v"(r.l[5]), "+&v"(r.l[6]),
        "+&v"(r.l[7]), "+&v"(r.l[8])
      : "v"(a.l[0]), "v"(a.l[1]), "v"(a.l[2]), "v"(a.l[3]), "v"(a.l[4]), "v"(a.l[5]), "v"(a.l[6]), "v"(a.l[7]),
        "v"(a.l[8]), "s"(mask));
  return r;
#else
  return keep ? a : b;
#endif
}

// (a + b) mod m into [0, 2m).  Inputs normalized, values < 2m.
template <class P>
ZK_HD fe<P> fadd(const fe<P>& a, const fe<P>& b) {
  fe<P> s, t;
  uint32_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    uint32_t v = a.l[i] + b.l[i] + c;
    c = v >> 29;
    s.l[i] = v & LMASK;
  }
  int32_t br = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    int32_t v = (int32_t)s.l[i] - (int32_t)P::MOD2[i] + br;
    br = v >> 29;
    t.l[i] = (uint32_t)v & LMASK;
  }
  return fselect(br != 0, s, t);  // br == -1: s < 2m, keep s
}

// (a - b) mod m into [0, 2m).  Inputs normalized, values < 2m.
template <class P>
ZK_HD fe<P> fsub(const fe<P>& a, const fe<P>& b) {
  fe<P> d;
  int32_t br = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    int32_t v = (int32_t)a.l[i] - (int32_t)b.l[i] + br;
    br = v >> 29;
    d.l[i] = (uint32_t)v & LMASK;
  }
  const uint32_t mask = (uint32_t)br;  // all ones when a < b
  uint32_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    uint32_t v = d.l[i] + (P::MOD2[i] & mask) + c;
    c = v >> 29;
    d.l[i] = v & LMASK;
  }
  return d;
}

// a - b + 2m without the final correction: value in (0, 4m) for a, b in
// [0, 2m), normalized limbs.  Valid only as a multiplication input.
template <class P>
ZK_HD fe<P> fsub_lazy(const fe<P>& a, const fe<P>& b) {
  fe<P> d;
  int32_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    int32_t v = (int32_t)a.l[i] + (int32_t)P::MOD2[i] - (int32_t)b.l[i] + c;
    c = v >> 29;
    d.l[i] = (uint32_t)v & LMASK;
  }
  return d;
}

// 2m - a for a in [0, 2m]: value in [0, 2m], normalized limbs (congruent to
// -a; not reduced, so a valid multiplication input only).
template <class P>
ZK_HD fe<P> fneg_lazy(const fe<P>& a) {
  fe<P> d;
  int32_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    int32_t v = (int32_t)P::MOD2[i] - (int32_t)a.l[i] + c;
    c = v >> 29;
    d.l[i] = (uint32_t)v & LMASK;
  }
  return d;
}

// 4m with 2^29 moved down into every limb below the top one: digit by digit not
// less than any normalized value below 2m, so KWIDE_i - a_i needs no borrow.
template <class P>
constexpr uint32_t kwide(int i) {
  return i == 0 ? P::MOD4[0] + LMASK + 1u : i < NL - 1 ? P::MOD4[i] + LMASK : P::MOD4[NL - 1] - 1u;
}

// 4m - a for a in [0, 2m), limbs below 2^30 without a carry pass: an operand of
// a two-product sum or of fmul only.
template <class P>
ZK_HD fe<P> fneg_wide(const fe<P>& a) {
  fe<P> d;
#pragma unroll
  for (int i = 0; i < NL; i++) d.l[i] = kwide<P>(i) - a.l[i];
  return d;
}

// a - b + 4m limb by limb, no carry pass, for a normalized b below 2m + m / 2^22:
// limbs at most 2^30 above a's.
template <class P>
ZK_HD fe<P> fsub_wide(const fe<P>& a, const fe<P>& b) {
  fe<P> d;
#pragma unroll
  for (int i = 0; i < NL; i++) d.l[i] = a.l[i] + (kwide<P>(i) - b.l[i]);
  return d;
}

// Carry pass: the same value (below 2^261) with normalized limbs; limbs at most
// 2^32 - 8 in.
template <class P>
ZK_HD fe<P> fcarry(const fe<P>& a) {
  fe<P> s;
  uint32_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    const uint32_t v = a.l[i] + c;
    s.l[i] = v & LMASK;
    c = v >> 29;
  }
  return s;
}

// neg ? 4m - a : a under a mask, as fneg_wide.
template <class P>
ZK_HD fe<P> fneg_wide_mask(const fe<P>& a, uint32_t mask) {
  fe<P> d;
#pragma unroll
  for (int i = 0; i < NL; i++) d.l[i] = (a.l[i] ^ mask) + (mask & (kwide<P>(i) + 1u));
  return d;
}

// neg ? m - a : a for a canonical (in [0, m)); m - a is in (0, m], a valid
// value of the lazy range [0, 2m).  -a is ~a + 1 limb by limb under a mask,
// not a select: nine selects in a row through VCC take 15-23 cycles each on
// gfx950 (a mask operation 2.4 to 4.4).
template <class P>
ZK_HD fe<P> fneg_canon_if(const fe<P>& a, bool neg) {
  const uint32_t mask = neg ? ~0u : 0u;
  fe<P> d;
  int32_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    int32_t v = (int32_t)((a.l[i] ^ mask) + (mask & (P::MOD[i] + 1u))) + c;
    c = v >> 29;
    d.l[i] = (uint32_t)v & LMASK;
  }
  return d;
}

template <class P>
ZK_HD fe<P> fneg(const fe<P>& a) {
  return fsub(fe_zero<P>(), a);
}

// a + b with carries and no reduction: normalized limbs, value in [0, 4m) for
// a, b in [0, 2m).
template <class P>
ZK_HD fe<P> fadd_wide(const fe<P>& a, const fe<P>& b) {
  fe<P> s;
  uint32_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    uint32_t v = a.l[i] + b.l[i] + c;
    c = v >> 29;
    s.l[i] = v & LMASK;
  }
  return s;
}

// Limb-wise sum without normalization: limbs < 2^30, value < 4m.  Valid only
// as a direct input of fmul/fsqr.
template <class P>
ZK_HD fe<P> fadd_lazy(const fe<P>& a, const fe<P>& b) {
  fe<P> s;
#pragma unroll
  for (int i = 0; i < NL; i++) s.l[i] = a.l[i] + b.l[i];
  return s;
}

// Reduce [0, 2m) to the canonical [0, m).
template <class P>
ZK_HD fe<P> fcanon(const fe<P>& a) {
  fe<P> t;
  int32_t br = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    int32_t v = (int32_t)a.l[i] - (int32_t)P::MOD[i] + br;
    br = v >> 29;
    t.l[i] = (uint32_t)v & LMASK;
  }
  return fselect(br != 0, a, t);
}

// a == 0 mod m for a in [0, 2m): a is 0 or m.
template <class P>
ZK_HD bool fis_zero(const fe<P>& a) {
  uint32_t z = 0, e = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    z |= a.l[i];
    e |= a.l[i] ^ P::MOD[i];
  }
  return z == 0 || e == 0;
}

// a == 0 mod m for a in [0, 4m): a is 0, m, 2m or 3m.
template <class P>
ZK_HD bool fis_zero4(const fe<P>& a) {
  uint32_t z = 0, e1 = 0, e2 = 0, e3 = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    z |= a.l[i];
    e1 |= a.l[i] ^ P::MOD[i];
    e2 |= a.l[i] ^ P::MOD2[i];
    e3 |= a.l[i] ^ P::MOD3[i];
  }
  return z == 0 || e1 == 0 || e2 == 0 || e3 == 0;
}

// t - K if t >= K (K normalized limbs), else t.
template <class P>
ZK_HD fe<P> fcsub(const fe<P>& t, const uint32_t (&K)[NL]) {
  fe<P> u;
  int32_t br = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    int32_t v = (int32_t)t.l[i] - (int32_t)K[i] + br;
    br = v >> 29;
    u.l[i] = (uint32_t)v & LMASK;
  }
  return fselect(br != 0, t, u);
}

// a - b - 2c + 4m, exact (normalized limbs), for a value that stays positive:
// b + 2c < 4m.
template <class P>
ZK_HD fe<P> fsub3_lazy(const fe<P>& a, const fe<P>& b, const fe<P>& c) {
  fe<P> t;
  int32_t cy = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    int32_t v = (int32_t)a.l[i] + (int32_t)P::MOD4[i] - (int32_t)b.l[i] - 2 * (int32_t)c.l[i] + cy;
    cy = v >> 29;
    t.l[i] = (uint32_t)v & LMASK;
  }
  return t;
}

// 3a with carries and no reduction (normalized limbs, value below 2^261).
template <class P>
ZK_HD fe<P> ftriple_wide(const fe<P>& a) {
  fe<P> s;
  uint32_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    uint32_t v = 3u * a.l[i] + c;
    c = v >> 29;
    s.l[i] = v & LMASK;
  }
  return s;
}

// 6m - a for a in [0, 6m]: value in [0, 6m], normalized limbs.
template <class P>
ZK_HD fe<P> fneg_lazy6(const fe<P>& a) {
  fe<P> d;
  int32_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    int32_t v = (int32_t)P::MOD6[i] - (int32_t)a.l[i] + c;
    c = v >> 29;
    d.l[i] = (uint32_t)v & LMASK;
  }
  return d;
}

// mask ? KM*m - a : a with carries (mask all ones or zero; KM = 2 or 6, a <= KM*m).
template <int KM, class P>
ZK_HD fe<P> fneg_mask(const fe<P>& a, uint32_t mask) {
  static_assert(KM == 2 || KM == 6, "offset multiple");
  const uint32_t(&K)[NL] = KM == 2 ? P::MOD2 : P::MOD6;
  fe<P> d;
  int32_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    int32_t v = (int32_t)((a.l[i] ^ mask) + (mask & (K[i] + 1u))) + c;
    c = v >> 29;
    d.l[i] = (uint32_t)v & LMASK;
  }
  return d;
}

// a - b + KM*m with carries (KM in {2, 4, 6, 8}): for b < KM*m the value is
// a - b + KM*m > 0 with normalized limbs (valid while below 2^261).
template <int KM, class P>
ZK_HD fe<P> fsub_off(const fe<P>& a, const fe<P>& b) {
  static_assert(KM == 2 || KM == 4 || KM == 6 || KM == 8, "offset multiple");
  const uint32_t(&K)[NL] = KM == 2 ? P::MOD2 : KM == 4 ? P::MOD4 : KM == 6 ? P::MOD6 : P::MOD8;
  fe<P> d;
  int32_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    int32_t v = (int32_t)a.l[i] + (int32_t)K[i] - (int32_t)b.l[i] + c;
    c = v >> 29;
    d.l[i] = (uint32_t)v & LMASK;
  }
  return d;
}

// Canonical value of x (normalized limbs, any value below 2^261).  Both
// moduli have top limb M8 = 0x30644e; q = (l8 * floor(2^40 / (M8 + 1))) >> 40
// never exceeds floor(x / m) and falls short of it by at most 2, so
// x - q m < 3m and two conditional subtractions finish.
template <class P>
ZK_HD fe<P> freduce(const fe<P>& x) {
  static_assert(P::MOD[NL - 1] == 0x0030644eu, "quotient estimate assumes the BN254 top limb");
  const uint32_t q = (uint32_t)(((uint64_t)x.l[NL - 1] * 346695ull) >> 40);
  fe<P> r;
  int64_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    const int64_t t = (int64_t)x.l[i] - (int64_t)q * (int64_t)P::MOD[i] + c;
    r.l[i] = (uint32_t)t & LMASK;
    c = t >> 29;
  }
  return fcsub(fcsub(r, P::MOD2), P::MOD);
}

template <class P>
ZK_HD bool feq(const fe<P>& a, const fe<P>& b) {
  return fis_zero(fsub(a, b));
}

// Bit repack of a 256-bit little-endian word array into 29-bit limbs (no change
// of value).
template <class P>
ZK_HD fe<P> repack_in(const uint32_t w[8]) {
  fe<P> r;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    const int bit = 29 * i;
    const int wd = bit >> 5;
    const int sh = bit & 31;
    uint64_t v = w[wd];
    if (wd + 1 < 8) v |= (uint64_t)w[wd + 1] << 32;
    r.l[i] = (uint32_t)(v >> sh) & LMASK;
  }
  return r;
}

// Canonicalize and repack into 8 little-endian 32-bit words.
template <class P>
ZK_HD void repack_out(const fe<P>& a, uint32_t w[8]) {
  fe<P> c = fcanon(a);
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const int bit = 32 * j;
    const int i = bit / 29;
    const int sh = bit % 29;
    uint64_t v = c.l[i];
    if (i + 1 < NL) v |= (uint64_t)c.l[i + 1] << 29;
    if (i + 2 < NL && sh > 26) v |= (uint64_t)c.l[i + 2] << 58;
    w[j] = (uint32_t)(v >> sh);
  }
}

// Reference Montgomery form (R = 2^256) <-> internal form (R' = 2^261).
template <class P>
ZK_HD fe<P> from_mont256(const uint32_t w[8]) {
  return fmul(repack_in<P>(w), fe_const<P>(P::K_IN));
}

template <class P>
ZK_HD void to_mont256(const fe<P>& a, uint32_t w[8]) {
  repack_out(fmul(a, fe_const<P>(P::K_OUT)), w);
}

// Plain integer (standard form) <-> internal form.
template <class P>
ZK_HD fe<P> from_std(const uint32_t w[8]) {
  return fmul(repack_in<P>(w), fe_const<P>(P::R2));
}

template <class P>
ZK_HD void to_std(const fe<P>& a, uint32_t w[8]) {
  fe<P> one_plain = fe_zero<P>();
  one_plain.l[0] = 1;
  repack_out(fmul(a, one_plain), w);
}

// Square-and-multiply with a 256-bit plain exponent (little-endian words).
template <class P>
ZK_HD fe<P> fpow(const fe<P>& a, const uint32_t e[8]) {
  fe<P> r = fe_one<P>();
  for (int bit = 255; bit >= 0; bit--) {
    r = fsqr(r);
    if ((e[bit >> 5] >> (bit & 31)) & 1u) r = fmul(r, a);
  }
  return r;
}

}  // namespace zk
