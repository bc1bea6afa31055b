// Host build of the device field / curve headers (cuda-zkml_amd/csrc/field.hpp,
// curve.hpp) for CPU unit tests: the same source that the kernels inline,
// compiled by g++ and driven from Python with big-integer expectations.
#include <stdint.h>
#include <string.h>

#include "curve.hpp"

using namespace zk;

static fq ld(const uint32_t* p) {
  fq r;
  memcpy(r.l, p, sizeof(r.l));
  return r;
}
static void st(uint32_t* p, const fq& a) { memcpy(p, a.l, sizeof(a.l)); }
static fq2 ld2(const uint32_t* p) { return fq2{ld(p), ld(p + NL)}; }
static void st2(uint32_t* p, const fq2& a) {
  st(p, a.c0);
  st(p + NL, a.c1);
}

extern "C" {

// Field operations on 9-limb Fq elements.
int fh_op(int op, const uint32_t* a, const uint32_t* b, const uint32_t* c, const uint32_t* d, uint32_t* out) {
  fq A = ld(a), B = ld(b), C = ld(c), D = ld(d), r;
  switch (op) {
    case 0: r = fmul(A, B); break;
    case 1: r = fsqr(A); break;
    case 2: r = fmul2(A, B, C, D); break;
    case 3: r = fsub_lazy(A, B); break;
    case 4: r = fneg_lazy(A); break;
    case 5: r = fadd(A, B); break;
    case 6: r = fsub(A, B); break;
    case 7: r = fmul_sub(A, B, C, D); break;
    case 9: r = freduce_x(fsub_off<4>(fsub_lazy(A, B), fadd_wide(C, C))); break;  // a - b - 2c
    case 10: r = fsub_off<4>(A, B); break;
    case 11: r = fsub_off<4>(fe_zero<FqP>(), A); break;
    case 12: r = fe_zero<FqP>(); r.l[0] = fis_zero<FqP>(A) ? 1u : 0u; break;
    case 13: r = fe_zero<FqP>(); r.l[0] = fis_zero4<FqP>(A) ? 1u : 0u; break;
    case 14: r = fadd_wide(A, B); break;
    case 15: r = fcsub(A, FqP::MOD2); break;
    case 8: {  // four products: a*b + c*d + a*d + c*b
      const fq x[4] = {A, C, A, C}, y[4] = {B, D, D, B};
      r = fmul_sum<FqP, 4>(x, y);
      break;
    }
    default: return -1;
  }
  st(out, r);
  return 0;
}

// The NTT butterfly's Fr operations (the same templates over the scalar
// field): 0 fmul, 1 fadd_wide, 2 fcsub(a, 2r), 3 fsub_lazy (a + 2r - b),
// 4 / 5 / 7: a - b + 4r / 8r / 2r, 6 freduce (canonical value).
int fh_fr_op(int op, const uint32_t* a, const uint32_t* b, uint32_t* out) {
  fr A, B, r;
  memcpy(A.l, a, sizeof(A.l));
  memcpy(B.l, b, sizeof(B.l));
  switch (op) {
    case 0: r = fmul(A, B); break;
    case 1: r = fadd_wide(A, B); break;
    case 2: r = fcsub(A, FrP::MOD2); break;
    case 3: r = fsub_lazy(A, B); break;
    case 4: r = fsub_off<4>(A, B); break;
    case 5: r = fsub_off<8>(A, B); break;
    case 6: r = freduce(A); break;
    case 7: r = fsub_off<2>(A, B); break;
    default: return -1;
  }
  memcpy(out, r.l, sizeof(r.l));
  return 0;
}

// XYZZ operations, X reduced below 2q afterwards; G1 points are 36 words (x, y,
// zz, zzz), G2 points 72.
// op 0: p += (qx, qy) affine   1: p += q   2: p = 2p   3: p = 2 (qx, qy)
int fh_xyzz(int g2, int op, const uint32_t* p, const uint32_t* q, uint32_t* out) {
  if (!g2) {
    xyzz<fq> P{ld(p), ld(p + 9), ld(p + 18), ld(p + 27)}, Q{ld(q), ld(q + 9), ld(q + 18), ld(q + 27)};
    switch (op) {
      case 0: xyzz_madd(P, Q.x, Q.y); break;
      case 1: xyzz_add_lx(P, Q); break;
      case 2: xyzz_dbl_lx(P); break;
      case 3: xyzz_mdbl_lx(P, Q.x, Q.y); break;
      default: return -1;
    }
    st(out, freduce_x(P.x));
    st(out + 9, P.y);
    st(out + 18, P.zz);
    st(out + 27, P.zzz);
  } else {
    xyzz<fq2> P{ld2(p), ld2(p + 18), ld2(p + 36), ld2(p + 54)}, Q{ld2(q), ld2(q + 18), ld2(q + 36), ld2(q + 54)};
    switch (op) {
      case 0: xyzz_madd(P, Q.x, Q.y); break;
      case 1: xyzz_add_lx(P, Q); break;
      case 2: xyzz_dbl_lx(P); break;
      case 3: xyzz_mdbl_lx(P, Q.x, Q.y); break;
      default: return -1;
    }
    st2(out, freduce_x(P.x));
    st2(out + 18, P.y);
    st2(out + 36, P.zz);
    st2(out + 54, P.zzz);
  }
  return 0;
}

// The lazy-X forms (X in [0, 6q) in and out): op 0: p += (qx, qy) affine, p
// finite   1: p += q   2: p = 2p   3: p = 2 (qx, qy).  Returns 1 where op 0
// reports the point at infinity.
int fh_xyzz_lx(int g2, int op, const uint32_t* p, const uint32_t* q, uint32_t* out) {
  int inf = 0;
  if (!g2) {
    xyzz<fq> P{ld(p), ld(p + 9), ld(p + 18), ld(p + 27)}, Q{ld(q), ld(q + 9), ld(q + 18), ld(q + 27)};
    switch (op) {
      case 0: inf = xyzz_madd_fin_lx(P, Q.x, Q.y); break;
      case 1: xyzz_add_lx(P, Q); break;
      case 2: xyzz_dbl_lx(P); break;
      case 3: xyzz_mdbl_lx(P, Q.x, Q.y); break;
      default: return -1;
    }
    st(out, P.x);
    st(out + 9, P.y);
    st(out + 18, P.zz);
    st(out + 27, P.zzz);
  } else {
    xyzz<fq2> P{ld2(p), ld2(p + 18), ld2(p + 36), ld2(p + 54)}, Q{ld2(q), ld2(q + 18), ld2(q + 36), ld2(q + 54)};
    switch (op) {
      case 0: inf = xyzz_madd_fin_lx(P, Q.x, Q.y); break;
      case 1: xyzz_add_lx(P, Q); break;
      case 2: xyzz_dbl_lx(P); break;
      case 3: xyzz_mdbl_lx(P, Q.x, Q.y); break;
      default: return -1;
    }
    st2(out, P.x);
    st2(out + 18, P.y);
    st2(out + 36, P.zz);
    st2(out + 54, P.zzz);
  }
  return inf;
}

// Products by a constant over Fr: limbs of a below lu 2^29 (lu 1, 3 or 5).
int fh_fr_const(int lu, const uint32_t* a, const uint32_t* w, const uint32_t* wq, uint32_t* out) {
  fr A, W, Q, r;
  memcpy(A.l, a, sizeof(A.l));
  memcpy(W.l, w, sizeof(W.l));
  memcpy(Q.l, wq, sizeof(Q.l));
  switch (lu) {
    case 1: r = fmul_const<1>(A, W, Q); break;
    case 3: r = fmul_const<3>(A, W, Q); break;
    case 5: r = fmul_const<5>(A, W, Q); break;
    default: return -1;
  }
  memcpy(out, r.l, sizeof(r.l));
  return 0;
}

// 0 const_quotient(a), 1 fsub_wide(a, b), 2 fadd_lazy(a, b), 3 fcarry(a)
int fh_fr_wide(int op, const uint32_t* a, const uint32_t* b, uint32_t* out) {
  fr A, B, r;
  memcpy(A.l, a, sizeof(A.l));
  memcpy(B.l, b, sizeof(B.l));
  switch (op) {
    case 0: r = const_quotient(A); break;
    case 1: r = fsub_wide(A, B); break;
    case 2: r = fadd_lazy(A, B); break;
    case 3: r = fcarry(A); break;
    default: return -1;
  }
  memcpy(out, r.l, sizeof(r.l));
  return 0;
}
}
