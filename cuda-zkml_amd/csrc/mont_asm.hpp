// Montgomery products of the device as one assembly block each (gfx950).
//
// field.hpp states the algorithm (mont_columns, which the host build runs):
// 17 product columns of 29 bits, each one serial chain of v_mad_u64_u32 into a
// 64-bit accumulator, the reduction interleaved.  The blocks below run the
// same columns in the same order:
//   columns 0..6   the low 32 bits of the column are the digit q_K as they are
//                  (no multiply, no mask); the high 32 bits go on as 8 * hi,
//                  seeded by one multiply-add;
//   columns 7, 8   29-bit digits q = acc * (-m^-1) mod 2^29;
//   columns 9..16  output limbs.
// Whole products in one block, because the compiler places a wait state
// (s_nop) after every assembly block whose result the next instruction reads:
// with one block per column it put about 36 of them into a product, which cost
// a wave alone on its SIMD about 3 cycles each (measured: a dependent
// v_mad_u64_u32 6.5 cycles, with s_nop 9.5; no difference from 2 waves on).
// Instructions per product (square): 191 (163), where a 29-bit digit in every
// column with its own multiply took 205 (176).
//
// The temporaries are fixed registers (an assembly operand cannot name the
// halves of a 64-bit register pair): column K's accumulator is the pair
// v[40+2K : 41+2K] for K < 7, whose low half stays as q_K, and v[54:55] from
// column 7 on; q_7 and q_8 take v41 and v43, dead by then.  The carry-out of
// the multiply-adds (VCC) is not used: the column bounds (field.hpp) keep every
// partial sum below 2^64.
#pragma once
#include <stdint.h>

// clang-format off
#define ZK_MAD(d, x, y) "v_mad_u64_u32 " d ", vcc, " x ", " y ", " d "\n"
#define ZK_MAD0(d, x, y) "v_mad_u64_u32 " d ", vcc, " x ", " y ", 0\n"
#define ZK_T(S, i) "%[" S #i "]"
// a_i b_j of the operand sets A, B (named a0..a8 and so on)
#define ZK_P(d, A, i, B, j) ZK_MAD(d, ZK_T(A, i), ZK_T(B, j))
// products of column K

#define ZK_C0(A, B) ZK_MAD0("v[40:41]", ZK_T(A, 0), ZK_T(B, 0))
#define ZK_D0(A, B) ZK_P("v[40:41]", A, 0, B, 0)
#define ZK_C1(A, B) ZK_P("v[42:43]", A, 0, B, 1) ZK_P("v[42:43]", A, 1, B, 0)
#define ZK_C2(A, B) ZK_P("v[44:45]", A, 0, B, 2) ZK_P("v[44:45]", A, 1, B, 1) ZK_P("v[44:45]", A, 2, B, 0)
#define ZK_C3(A, B) ZK_P("v[46:47]", A, 0, B, 3) ZK_P("v[46:47]", A, 1, B, 2) ZK_P("v[46:47]", A, 2, B, 1) \
    ZK_P("v[46:47]", A, 3, B, 0)
#define ZK_C4(A, B) ZK_P("v[48:49]", A, 0, B, 4) ZK_P("v[48:49]", A, 1, B, 3) ZK_P("v[48:49]", A, 2, B, 2) \
    ZK_P("v[48:49]", A, 3, B, 1) ZK_P("v[48:49]", A, 4, B, 0)
#define ZK_C5(A, B) ZK_P("v[50:51]", A, 0, B, 5) ZK_P("v[50:51]", A, 1, B, 4) ZK_P("v[50:51]", A, 2, B, 3) \
    ZK_P("v[50:51]", A, 3, B, 2) ZK_P("v[50:51]", A, 4, B, 1) ZK_P("v[50:51]", A, 5, B, 0)
#define ZK_C6(A, B) ZK_P("v[52:53]", A, 0, B, 6) ZK_P("v[52:53]", A, 1, B, 5) ZK_P("v[52:53]", A, 2, B, 4) \
    ZK_P("v[52:53]", A, 3, B, 3) ZK_P("v[52:53]", A, 4, B, 2) ZK_P("v[52:53]", A, 5, B, 1) \
    ZK_P("v[52:53]", A, 6, B, 0)
#define ZK_C7(A, B) ZK_P("v[54:55]", A, 0, B, 7) ZK_P("v[54:55]", A, 1, B, 6) ZK_P("v[54:55]", A, 2, B, 5) \
    ZK_P("v[54:55]", A, 3, B, 4) ZK_P("v[54:55]", A, 4, B, 3) ZK_P("v[54:55]", A, 5, B, 2) \
    ZK_P("v[54:55]", A, 6, B, 1) ZK_P("v[54:55]", A, 7, B, 0)
#define ZK_C8(A, B) ZK_P("v[54:55]", A, 0, B, 8) ZK_P("v[54:55]", A, 1, B, 7) ZK_P("v[54:55]", A, 2, B, 6) \
    ZK_P("v[54:55]", A, 3, B, 5) ZK_P("v[54:55]", A, 4, B, 4) ZK_P("v[54:55]", A, 5, B, 3) \
    ZK_P("v[54:55]", A, 6, B, 2) ZK_P("v[54:55]", A, 7, B, 1) ZK_P("v[54:55]", A, 8, B, 0)
#define ZK_C9(A, B) ZK_P("v[54:55]", A, 1, B, 8) ZK_P("v[54:55]", A, 2, B, 7) ZK_P("v[54:55]", A, 3, B, 6) \
    ZK_P("v[54:55]", A, 4, B, 5) ZK_P("v[54:55]", A, 5, B, 4) ZK_P("v[54:55]", A, 6, B, 3) \
    ZK_P("v[54:55]", A, 7, B, 2) ZK_P("v[54:55]", A, 8, B, 1)
#define ZK_C10(A, B) ZK_P("v[54:55]", A, 2, B, 8) ZK_P("v[54:55]", A, 3, B, 7) ZK_P("v[54:55]", A, 4, B, 6) \
    ZK_P("v[54:55]", A, 5, B, 5) ZK_P("v[54:55]", A, 6, B, 4) ZK_P("v[54:55]", A, 7, B, 3) \
    ZK_P("v[54:55]", A, 8, B, 2)
#define ZK_C11(A, B) ZK_P("v[54:55]", A, 3, B, 8) ZK_P("v[54:55]", A, 4, B, 7) ZK_P("v[54:55]", A, 5, B, 6) \
    ZK_P("v[54:55]", A, 6, B, 5) ZK_P("v[54:55]", A, 7, B, 4) ZK_P("v[54:55]", A, 8, B, 3)
#define ZK_C12(A, B) ZK_P("v[54:55]", A, 4, B, 8) ZK_P("v[54:55]", A, 5, B, 7) ZK_P("v[54:55]", A, 6, B, 6) \
    ZK_P("v[54:55]", A, 7, B, 5) ZK_P("v[54:55]", A, 8, B, 4)
#define ZK_C13(A, B) ZK_P("v[54:55]", A, 5, B, 8) ZK_P("v[54:55]", A, 6, B, 7) ZK_P("v[54:55]", A, 7, B, 6) \
    ZK_P("v[54:55]", A, 8, B, 5)
#define ZK_C14(A, B) ZK_P("v[54:55]", A, 6, B, 8) ZK_P("v[54:55]", A, 7, B, 7) ZK_P("v[54:55]", A, 8, B, 6)
#define ZK_C15(A, B) ZK_P("v[54:55]", A, 7, B, 8) ZK_P("v[54:55]", A, 8, B, 7)
#define ZK_C16(A, B) ZK_P("v[54:55]", A, 8, B, 8)
// cross products a_i (2 a_j), i < j (2 a_j held in the output registers r_j), and the square a_(K/2)^2
#define ZK_S0 ZK_MAD0("v[40:41]", "%[a0]", "%[a0]")
#define ZK_S1 ZK_MAD("v[42:43]", "%[a0]", "%[r1]")
#define ZK_S2 ZK_MAD("v[44:45]", "%[a0]", "%[r2]") ZK_MAD("v[44:45]", "%[a1]", "%[a1]")
#define ZK_S3 ZK_MAD("v[46:47]", "%[a0]", "%[r3]") ZK_MAD("v[46:47]", "%[a1]", "%[r2]")
#define ZK_S4 ZK_MAD("v[48:49]", "%[a0]", "%[r4]") ZK_MAD("v[48:49]", "%[a1]", "%[r3]") \
    ZK_MAD("v[48:49]", "%[a2]", "%[a2]")
#define ZK_S5 ZK_MAD("v[50:51]", "%[a0]", "%[r5]") ZK_MAD("v[50:51]", "%[a1]", "%[r4]") \
    ZK_MAD("v[50:51]", "%[a2]", "%[r3]")
#define ZK_S6 ZK_MAD("v[52:53]", "%[a0]", "%[r6]") ZK_MAD("v[52:53]", "%[a1]", "%[r5]") \
    ZK_MAD("v[52:53]", "%[a2]", "%[r4]") ZK_MAD("v[52:53]", "%[a3]", "%[a3]")
#define ZK_S7 ZK_MAD("v[54:55]", "%[a0]", "%[r7]") ZK_MAD("v[54:55]", "%[a1]", "%[r6]") \
    ZK_MAD("v[54:55]", "%[a2]", "%[r5]") ZK_MAD("v[54:55]", "%[a3]", "%[r4]")
#define ZK_S8 ZK_MAD("v[54:55]", "%[a0]", "%[r8]") ZK_MAD("v[54:55]", "%[a1]", "%[r7]") \
    ZK_MAD("v[54:55]", "%[a2]", "%[r6]") ZK_MAD("v[54:55]", "%[a3]", "%[r5]") ZK_MAD("v[54:55]", "%[a4]", "%[a4]")
#define ZK_S9 ZK_MAD("v[54:55]", "%[a1]", "%[r8]") ZK_MAD("v[54:55]", "%[a2]", "%[r7]") \
    ZK_MAD("v[54:55]", "%[a3]", "%[r6]") ZK_MAD("v[54:55]", "%[a4]", "%[r5]")
#define ZK_S10 ZK_MAD("v[54:55]", "%[a2]", "%[r8]") ZK_MAD("v[54:55]", "%[a3]", "%[r7]") \
    ZK_MAD("v[54:55]", "%[a4]", "%[r6]") ZK_MAD("v[54:55]", "%[a5]", "%[a5]")
#define ZK_S11 ZK_MAD("v[54:55]", "%[a3]", "%[r8]") ZK_MAD("v[54:55]", "%[a4]", "%[r7]") \
    ZK_MAD("v[54:55]", "%[a5]", "%[r6]")
#define ZK_S12 ZK_MAD("v[54:55]", "%[a4]", "%[r8]") ZK_MAD("v[54:55]", "%[a5]", "%[r7]") \
    ZK_MAD("v[54:55]", "%[a6]", "%[a6]")
#define ZK_S13 ZK_MAD("v[54:55]", "%[a5]", "%[r8]") ZK_MAD("v[54:55]", "%[a6]", "%[r7]")
#define ZK_S14 ZK_MAD("v[54:55]", "%[a6]", "%[r8]") ZK_MAD("v[54:55]", "%[a7]", "%[a7]")
#define ZK_S15 ZK_MAD("v[54:55]", "%[a7]", "%[r8]")
#define ZK_S16 ZK_MAD("v[54:55]", "%[a8]", "%[a8]")
// reduction of column K before its products (the carry of column K - 1 < 7: 8 * its high half) ...
#define ZK_B1 ZK_MAD0("v[42:43]", "v41", "8")
#define ZK_B2 ZK_MAD0("v[44:45]", "v43", "8")
#define ZK_B3 ZK_MAD0("v[46:47]", "v45", "8")
#define ZK_B4 ZK_MAD0("v[48:49]", "v47", "8")
#define ZK_B5 ZK_MAD0("v[50:51]", "v49", "8")
#define ZK_B6 ZK_MAD0("v[52:53]", "v51", "8")
#define ZK_B7 ZK_MAD0("v[54:55]", "v53", "8")
// ... and after them: the digits of the columns below, then the column's own digit or output limb
#define ZK_R0
#define ZK_R1 ZK_MAD("v[42:43]", "v40", "%[e0]")
#define ZK_R2 ZK_MAD("v[44:45]", "v40", "%[e1]") ZK_MAD("v[44:45]", "v42", "%[e0]")
#define ZK_R3 ZK_MAD("v[46:47]", "v40", "%[e2]") ZK_MAD("v[46:47]", "v42", "%[e1]") ZK_MAD("v[46:47]", "v44", "%[e0]")
#define ZK_R4 ZK_MAD("v[48:49]", "v40", "%[e3]") ZK_MAD("v[48:49]", "v42", "%[e2]") \
    ZK_MAD("v[48:49]", "v44", "%[e1]") ZK_MAD("v[48:49]", "v46", "%[e0]")
#define ZK_R5 ZK_MAD("v[50:51]", "v40", "%[e4]") ZK_MAD("v[50:51]", "v42", "%[e3]") \
    ZK_MAD("v[50:51]", "v44", "%[e2]") ZK_MAD("v[50:51]", "v46", "%[e1]") ZK_MAD("v[50:51]", "v48", "%[e0]")
#define ZK_R6 ZK_MAD("v[52:53]", "v40", "%[e5]") ZK_MAD("v[52:53]", "v42", "%[e4]") \
    ZK_MAD("v[52:53]", "v44", "%[e3]") ZK_MAD("v[52:53]", "v46", "%[e2]") ZK_MAD("v[52:53]", "v48", "%[e1]") \
    ZK_MAD("v[52:53]", "v50", "%[e0]")
#define ZK_R7 ZK_MAD("v[54:55]", "v40", "%[e6]") ZK_MAD("v[54:55]", "v42", "%[e5]") \
    ZK_MAD("v[54:55]", "v44", "%[e4]") ZK_MAD("v[54:55]", "v46", "%[e3]") ZK_MAD("v[54:55]", "v48", "%[e2]") \
    ZK_MAD("v[54:55]", "v50", "%[e1]") \
    ZK_MAD("v[54:55]", "v52", "%[e0]") "v_mul_lo_u32 v41, v54, %[inv]\n" "v_and_b32_e32 v41, 0x1fffffff, v41\n" \
    ZK_MAD("v[54:55]", "v41", "%[m0]") "v_lshrrev_b64 v[54:55], 29, v[54:55]\n"
#define ZK_R8 ZK_MAD("v[54:55]", "v40", "%[e7]") ZK_MAD("v[54:55]", "v42", "%[e6]") \
    ZK_MAD("v[54:55]", "v44", "%[e5]") ZK_MAD("v[54:55]", "v46", "%[e4]") ZK_MAD("v[54:55]", "v48", "%[e3]") \
    ZK_MAD("v[54:55]", "v50", "%[e2]") ZK_MAD("v[54:55]", "v52", "%[e1]") \
    ZK_MAD("v[54:55]", "v41", "%[m1]") "v_mul_lo_u32 v43, v54, %[inv]\n" "v_and_b32_e32 v43, 0x1fffffff, v43\n" \
    ZK_MAD("v[54:55]", "v43", "%[m0]") "v_lshrrev_b64 v[54:55], 29, v[54:55]\n"
#define ZK_R9 ZK_MAD("v[54:55]", "v40", "%[e8]") ZK_MAD("v[54:55]", "v42", "%[e7]") \
    ZK_MAD("v[54:55]", "v44", "%[e6]") ZK_MAD("v[54:55]", "v46", "%[e5]") ZK_MAD("v[54:55]", "v48", "%[e4]") \
    ZK_MAD("v[54:55]", "v50", "%[e3]") ZK_MAD("v[54:55]", "v52", "%[e2]") ZK_MAD("v[54:55]", "v41", "%[m2]") \
    ZK_MAD("v[54:55]", "v43", "%[m1]") "v_and_b32_e32 %[r0], 0x1fffffff, v54\n" "v_lshrrev_b64 v[54:55], 29, v[54:55]\n"
#define ZK_R10 ZK_MAD("v[54:55]", "v42", "%[e8]") ZK_MAD("v[54:55]", "v44", "%[e7]") \
    ZK_MAD("v[54:55]", "v46", "%[e6]") ZK_MAD("v[54:55]", "v48", "%[e5]") ZK_MAD("v[54:55]", "v50", "%[e4]") \
    ZK_MAD("v[54:55]", "v52", "%[e3]") ZK_MAD("v[54:55]", "v41", "%[m3]") \
    ZK_MAD("v[54:55]", "v43", "%[m2]") "v_and_b32_e32 %[r1], 0x1fffffff, v54\n" "v_lshrrev_b64 v[54:55], 29, v[54:55]\n"
#define ZK_R11 ZK_MAD("v[54:55]", "v44", "%[e8]") ZK_MAD("v[54:55]", "v46", "%[e7]") \
    ZK_MAD("v[54:55]", "v48", "%[e6]") ZK_MAD("v[54:55]", "v50", "%[e5]") ZK_MAD("v[54:55]", "v52", "%[e4]") \
    ZK_MAD("v[54:55]", "v41", "%[m4]") \
    ZK_MAD("v[54:55]", "v43", "%[m3]") "v_and_b32_e32 %[r2], 0x1fffffff, v54\n" "v_lshrrev_b64 v[54:55], 29, v[54:55]\n"
#define ZK_R12 ZK_MAD("v[54:55]", "v46", "%[e8]") ZK_MAD("v[54:55]", "v48", "%[e7]") \
    ZK_MAD("v[54:55]", "v50", "%[e6]") ZK_MAD("v[54:55]", "v52", "%[e5]") ZK_MAD("v[54:55]", "v41", "%[m5]") \
    ZK_MAD("v[54:55]", "v43", "%[m4]") "v_and_b32_e32 %[r3], 0x1fffffff, v54\n" "v_lshrrev_b64 v[54:55], 29, v[54:55]\n"
#define ZK_R13 ZK_MAD("v[54:55]", "v48", "%[e8]") ZK_MAD("v[54:55]", "v50", "%[e7]") \
    ZK_MAD("v[54:55]", "v52", "%[e6]") ZK_MAD("v[54:55]", "v41", "%[m6]") \
    ZK_MAD("v[54:55]", "v43", "%[m5]") "v_and_b32_e32 %[r4], 0x1fffffff, v54\n" "v_lshrrev_b64 v[54:55], 29, v[54:55]\n"
#define ZK_R14 ZK_MAD("v[54:55]", "v50", "%[e8]") ZK_MAD("v[54:55]", "v52", "%[e7]") \
    ZK_MAD("v[54:55]", "v41", "%[m7]") \
    ZK_MAD("v[54:55]", "v43", "%[m6]") "v_and_b32_e32 %[r5], 0x1fffffff, v54\n" "v_lshrrev_b64 v[54:55], 29, v[54:55]\n"
#define ZK_R15 ZK_MAD("v[54:55]", "v52", "%[e8]") ZK_MAD("v[54:55]", "v41", "%[m8]") \
    ZK_MAD("v[54:55]", "v43", "%[m7]") "v_and_b32_e32 %[r6], 0x1fffffff, v54\n" "v_lshrrev_b64 v[54:55], 29, v[54:55]\n"
#define ZK_R16 \
    ZK_MAD("v[54:55]", "v43", "%[m8]") "v_and_b32_e32 %[r7], 0x1fffffff, v54\n" "v_alignbit_b32 %[r8], v55, v54, 29\n"

#define ZK_CLOBBER "vcc", "v40", "v41", "v42", "v43", "v44", "v45", "v46", "v47", "v48", "v49", "v50", "v51", "v52", \
    "v53", "v54", "v55"
#define ZK_IN9(S, x) [S##0] "v"(x[0]), [S##1] "v"(x[1]), [S##2] "v"(x[2]), [S##3] "v"(x[3]), [S##4] "v"(x[4]), \
    [S##5] "v"(x[5]), [S##6] "v"(x[6]), [S##7] "v"(x[7]), [S##8] "v"(x[8])
#define ZK_OUT9(x) [r0] "=&v"(x[0]), [r1] "=&v"(x[1]), [r2] "=&v"(x[2]), [r3] "=&v"(x[3]), [r4] "=&v"(x[4]), \
    [r5] "=&v"(x[5]), [r6] "=&v"(x[6]), [r7] "=&v"(x[7]), [r8] "=&v"(x[8])
#define ZK_IO9(x) [r0] "+&v"(x[0]), [r1] "+&v"(x[1]), [r2] "+&v"(x[2]), [r3] "+&v"(x[3]), [r4] "+&v"(x[4]), \
    [r5] "+&v"(x[5]), [r6] "+&v"(x[6]), [r7] "+&v"(x[7]), [r8] "+&v"(x[8])
// digit multipliers: uniform, in scalar registers
#define ZK_MODULUS(P) [inv] "s"(P::INV), \
    [e0] "s"(P::EDIG[0]), [e1] "s"(P::EDIG[1]), [e2] "s"(P::EDIG[2]), [e3] "s"(P::EDIG[3]), [e4] "s"(P::EDIG[4]), \
    [e5] "s"(P::EDIG[5]), [e6] "s"(P::EDIG[6]), [e7] "s"(P::EDIG[7]), [e8] "s"(P::EDIG[8]), \
    [m0] "s"(P::MOD[0]), [m1] "s"(P::MOD[1]), [m2] "s"(P::MOD[2]), [m3] "s"(P::MOD[3]), [m4] "s"(P::MOD[4]), \
    [m5] "s"(P::MOD[5]), [m6] "s"(P::MOD[6]), [m7] "s"(P::MOD[7]), [m8] "s"(P::MOD[8])

namespace zk {

// r = r b 2^-261 mod m.  In place: output limb r_j is written in column j + 9,
// after operand limb r_j was last read (column j + 8), so a product takes no
// registers for its result when one operand is dead after it.
template <class P>
__device__ __forceinline__ void mont_mul_asm(uint32_t* r, const uint32_t* b) {
  asm(
      ZK_C0("r", "b") ZK_R0
      ZK_B1 ZK_C1("r", "b") ZK_R1
      ZK_B2 ZK_C2("r", "b") ZK_R2
      ZK_B3 ZK_C3("r", "b") ZK_R3
      ZK_B4 ZK_C4("r", "b") ZK_R4
      ZK_B5 ZK_C5("r", "b") ZK_R5
      ZK_B6 ZK_C6("r", "b") ZK_R6
      ZK_B7 ZK_C7("r", "b") ZK_R7
      ZK_C8("r", "b") ZK_R8
      ZK_C9("r", "b") ZK_R9
      ZK_C10("r", "b") ZK_R10
      ZK_C11("r", "b") ZK_R11
      ZK_C12("r", "b") ZK_R12
      ZK_C13("r", "b") ZK_R13
      ZK_C14("r", "b") ZK_R14
      ZK_C15("r", "b") ZK_R15
      ZK_C16("r", "b") ZK_R16
      : ZK_IO9(r)
      : ZK_IN9(b, b), ZK_MODULUS(P)
      : ZK_CLOBBER);
}

// r = a^2 2^-261 mod m
template <class P>
__device__ __forceinline__ void mont_sqr_asm(uint32_t* r, const uint32_t* a) {
  asm(
      "v_lshlrev_b32_e32 %[r1], 1, %[a1]\n" "v_lshlrev_b32_e32 %[r2], 1, %[a2]\n" "v_lshlrev_b32_e32 %[r3], 1, %[a3]\n" "v_lshlrev_b32_e32 %[r4], 1, %[a4]\n" "v_lshlrev_b32_e32 %[r5], 1, %[a5]\n" "v_lshlrev_b32_e32 %[r6], 1, %[a6]\n" "v_lshlrev_b32_e32 %[r7], 1, %[a7]\n" "v_lshlrev_b32_e32 %[r8], 1, %[a8]\n"
      ZK_S0 ZK_R0
      ZK_B1 ZK_S1 ZK_R1
      ZK_B2 ZK_S2 ZK_R2
      ZK_B3 ZK_S3 ZK_R3
      ZK_B4 ZK_S4 ZK_R4
      ZK_B5 ZK_S5 ZK_R5
      ZK_B6 ZK_S6 ZK_R6
      ZK_B7 ZK_S7 ZK_R7
      ZK_S8 ZK_R8
      ZK_S9 ZK_R9
      ZK_S10 ZK_R10
      ZK_S11 ZK_R11
      ZK_S12 ZK_R12
      ZK_S13 ZK_R13
      ZK_S14 ZK_R14
      ZK_S15 ZK_R15
      ZK_S16 ZK_R16
      : ZK_OUT9(r)
      : ZK_IN9(a, a), ZK_MODULUS(P)
      : ZK_CLOBBER);
}

// r = (r b + c d) 2^-261 mod m
template <class P>
__device__ __forceinline__ void mont_mul2_asm(uint32_t* r, const uint32_t* b, const uint32_t* c, const uint32_t* d) {
  asm(
      ZK_C0("r", "b") ZK_D0("c", "d") ZK_R0
      ZK_B1 ZK_C1("r", "b") ZK_C1("c", "d") ZK_R1
      ZK_B2 ZK_C2("r", "b") ZK_C2("c", "d") ZK_R2
      ZK_B3 ZK_C3("r", "b") ZK_C3("c", "d") ZK_R3
      ZK_B4 ZK_C4("r", "b") ZK_C4("c", "d") ZK_R4
      ZK_B5 ZK_C5("r", "b") ZK_C5("c", "d") ZK_R5
      ZK_B6 ZK_C6("r", "b") ZK_C6("c", "d") ZK_R6
      ZK_B7 ZK_C7("r", "b") ZK_C7("c", "d") ZK_R7
      ZK_C8("r", "b") ZK_C8("c", "d") ZK_R8
      ZK_C9("r", "b") ZK_C9("c", "d") ZK_R9
      ZK_C10("r", "b") ZK_C10("c", "d") ZK_R10
      ZK_C11("r", "b") ZK_C11("c", "d") ZK_R11
      ZK_C12("r", "b") ZK_C12("c", "d") ZK_R12
      ZK_C13("r", "b") ZK_C13("c", "d") ZK_R13
      ZK_C14("r", "b") ZK_C14("c", "d") ZK_R14
      ZK_C15("r", "b") ZK_C15("c", "d") ZK_R15
      ZK_C16("r", "b") ZK_C16("c", "d") ZK_R16
      : ZK_IO9(r)
      : ZK_IN9(b, b), ZK_IN9(c, c), ZK_IN9(d, d), ZK_MODULUS(P)
      : ZK_CLOBBER);
}

// r = (r b + c d + f g + h k) 2^-261 mod m
template <class P>
__device__ __forceinline__ void mont_mul4_asm(uint32_t* r, const uint32_t* b, const uint32_t* c, const uint32_t* d,
                                             const uint32_t* f, const uint32_t* g, const uint32_t* h,
                                             const uint32_t* k) {
  asm(
      ZK_C0("r", "b") ZK_D0("c", "d") ZK_D0("f", "g") ZK_D0("h", "k") ZK_R0
      ZK_B1 ZK_C1("r", "b") ZK_C1("c", "d") ZK_C1("f", "g") ZK_C1("h", "k") ZK_R1
      ZK_B2 ZK_C2("r", "b") ZK_C2("c", "d") ZK_C2("f", "g") ZK_C2("h", "k") ZK_R2
      ZK_B3 ZK_C3("r", "b") ZK_C3("c", "d") ZK_C3("f", "g") ZK_C3("h", "k") ZK_R3
      ZK_B4 ZK_C4("r", "b") ZK_C4("c", "d") ZK_C4("f", "g") ZK_C4("h", "k") ZK_R4
      ZK_B5 ZK_C5("r", "b") ZK_C5("c", "d") ZK_C5("f", "g") ZK_C5("h", "k") ZK_R5
      ZK_B6 ZK_C6("r", "b") ZK_C6("c", "d") ZK_C6("f", "g") ZK_C6("h", "k") ZK_R6
      ZK_B7 ZK_C7("r", "b") ZK_C7("c", "d") ZK_C7("f", "g") ZK_C7("h", "k") ZK_R7
      ZK_C8("r", "b") ZK_C8("c", "d") ZK_C8("f", "g") ZK_C8("h", "k") ZK_R8
      ZK_C9("r", "b") ZK_C9("c", "d") ZK_C9("f", "g") ZK_C9("h", "k") ZK_R9
      ZK_C10("r", "b") ZK_C10("c", "d") ZK_C10("f", "g") ZK_C10("h", "k") ZK_R10
      ZK_C11("r", "b") ZK_C11("c", "d") ZK_C11("f", "g") ZK_C11("h", "k") ZK_R11
      ZK_C12("r", "b") ZK_C12("c", "d") ZK_C12("f", "g") ZK_C12("h", "k") ZK_R12
      ZK_C13("r", "b") ZK_C13("c", "d") ZK_C13("f", "g") ZK_C13("h", "k") ZK_R13
      ZK_C14("r", "b") ZK_C14("c", "d") ZK_C14("f", "g") ZK_C14("h", "k") ZK_R14
      ZK_C15("r", "b") ZK_C15("c", "d") ZK_C15("f", "g") ZK_C15("h", "k") ZK_R15
      ZK_C16("r", "b") ZK_C16("c", "d") ZK_C16("f", "g") ZK_C16("h", "k") ZK_R16
      : ZK_IO9(r)
      : ZK_IN9(b, b), ZK_IN9(c, c), ZK_IN9(d, d), ZK_IN9(f, f), ZK_IN9(g, g), ZK_IN9(h, h), ZK_IN9(k, k),
        ZK_MODULUS(P)
      : ZK_CLOBBER);
}

}  // namespace zk
// clang-format on
