// BN254 G1 (over Fq) and G2 (over Fq2 = Fq[u]/(u^2+1)) group arithmetic for
// the MSM kernels, in XYZZ coordinates: (X, Y, ZZ, ZZZ) with x = X/ZZ,
// y = Y/ZZZ, ZZ^3 = ZZZ^2; ZZ = 0 encodes the point at infinity.  Formulas are
// the a = 0 cases of the EFD "xyzz" family: madd-2008-s (8M+2S),
// add-2008-s (12M+2S), dbl-2008-s-1 (6M+3S) and mdbl-2008-s-1.  The reference
// uses Jacobian coordinates (src/curve/g1.cuh:89-187) and affine G2 formulas
// (src/curve/g2.cuh:103-146); every one of them computes the same group law,
// and results leave the device as canonical affine points.
//
// All functions are generic over the coordinate field F (fq or fq2) through
// the overloads fmul/fsqr/fis_zero and the like below.
//
// The *_lx forms leave X in (0, 6m) ("lazy X") instead of reducing it: X3 = R^2 -
// PPP - 2Q + 4m is one carry pass, where a reduced X3 takes two conditional
// subtractions more (about 90 of a mixed addition's 2300 instructions, a third of
// them selects).  X is only ever a product's operand or subtracted with an offset,
// so no other step changes its cost.  Y, ZZ, ZZZ stay below 2m.  xyzz_madd gives X
// below 2m, too.  Bounds, per coordinate and in units of m (a product
// of a and b is below ab / 169.2 + 1.0000003; an Fq2 product is one of sums
// a0 b0 + (4 - a1) b1 with a the reduced factor; an Fq2 square (a0 + a1)(a0 -
// a1 + 8) and (2 a0) a1):
//   mixed addition: U2, S2 < 1.1; P = U2 - X + 6 in (0, 7.1), R = S2 - Y + 2 in
//   (0, 3.1); P^2 < 1.8, R^2 < 1.4; PPP, Q < 1.25 (Fq2: 1 + (1.73 + 4) 7.1 / 169.2);
//   X3 = R^2 - PPP - 2Q + 4 in (0.25, 5.4); Q - X3 + 6 in (0.6, 7), so Y3 < 1.5; ZZ3,
//   ZZZ3 < 1.1.
//   addition: P, R in (0, 4), P^2, R^2 < 1.4, then as above.
//   doubling: U = 2Y < 4, V = U^2 < 1.4, W, S < 1.2, X^2 < 1.99, M = 3 X^2 < 6,
//   M^2 < 1.99, X3 = M^2 - 2S + 4 in (1.6, 6), S - X3 + 6 in (0, 5.6), Y3 < 1.6.
// P = 0 mod m is tested on the reduced square (two comparisons, four for the
// wider Fq2 one) instead of on P, which has more representatives.
#pragma once
#include "field.hpp"

namespace zk {

// ------------------------------------------------------------------ Fq2
struct fq2 {
  fq c0, c1;
};

ZK_HD fq fneg_canon_if(const fq& a, bool neg) { return fneg_canon_if<FqP>(a, neg); }
ZK_HD fq2 fneg_canon_if(const fq2& a, bool neg) { return fq2{fneg_canon_if(a.c0, neg), fneg_canon_if(a.c1, neg)}; }
// (a0 + a1 u)(b0 + b1 u) = (a0 b0 - a1 b1) + (a0 b1 + a1 b0) u, each
// coordinate one fmul_sum (4 limb products, 2 reductions; the reference uses
// Karatsuba, src/field/fp2.cuh:73-78: 3 multiplies, each with its own
// reduction).  -a1 enters as 4q - a1 (no carry pass), so a must be reduced (a1 <
// 2q); b may be a lazy value (< 8q).
ZK_HD fq2 fmul(const fq2& a, const fq2& b) {
  const fq x0[2] = {a.c0, fneg_wide(a.c1)}, y0[2] = {b.c0, b.c1};
  const fq x1[2] = {a.c0, a.c1}, y1[2] = {b.c1, b.c0};
  return fq2{fmul_sum<FqP, 2>(x0, y0), fmul_sum<FqP, 2>(x1, y1)};
}
// (a + bu)^2 = (a+b)(a-b) + (2a)b u; a may be a lazy value (< 8q; the result is
// below 2q for a < 6q, its real part below 2.3q up to 7q).
ZK_HD fq2 fsqr(const fq2& a) {
  return fq2{fmul(fadd_lazy(a.c0, a.c1), fsub_off<8>(a.c0, a.c1)), fmul(fadd_lazy(a.c0, a.c0), a.c1)};
}
ZK_HD bool fis_zero(const fq2& a) { return fis_zero(a.c0) && fis_zero(a.c1); }

ZK_HD void fset_zero(fq& a) { a = fe_zero<FqP>(); }
ZK_HD void fset_zero(fq2& a) { a = fq2{fe_zero<FqP>(), fe_zero<FqP>()}; }
ZK_HD void fset_one(fq& a) { a = fe_one<FqP>(); }
ZK_HD void fset_one(fq2& a) { a = fq2{fe_one<FqP>(), fe_zero<FqP>()}; }

// x b for a lazy x (< 6m) and a reduced b.
ZK_HD fq fmul_x(const fq& x, const fq& b) { return fmul(x, b); }
ZK_HD fq2 fmul_x(const fq2& x, const fq2& b) { return fmul(b, x); }

// a*b - c*d with one Montgomery reduction per coordinate (fmul_sum, the
// subtracted products entering as (km - x) * y).  a and b may be lazy values
// (a < 6m, b < 7m); c and d are reduced (< 2m).
ZK_HD fq fmul_sub(const fq& a, const fq& b, const fq& c, const fq& d) { return fmul2(a, b, c, fneg_wide(d)); }
ZK_HD fq2 fmul_sub(const fq2& a, const fq2& b, const fq2& c, const fq2& d) {
  // real: a0 b0 - a1 b1 - c0 d0 + c1 d1, imaginary: a0 b1 + a1 b0 - c0 d1 - c1 d0
  const fq na1 = fneg_lazy6(a.c1), nc0 = fneg_lazy(c.c0), nc1 = fneg_lazy(c.c1);
  const fq x0[4] = {a.c0, na1, nc0, c.c1}, y0[4] = {b.c0, b.c1, d.c0, d.c1};
  const fq x1[4] = {a.c0, a.c1, nc0, nc1}, y1[4] = {b.c1, b.c0, d.c1, d.c0};
  return fq2{fmul_sum<FqP, 4>(x0, y0), fmul_sum<FqP, 4>(x1, y1)};
}
// a - b left in (0, 4m) for reduced a, b: only as an fmul_sub factor or an
// fsqr input.
ZK_HD fq fsub_m(const fq& a, const fq& b) { return fsub_lazy(a, b); }
ZK_HD fq2 fsub_m(const fq2& a, const fq2& b) { return fq2{fsub_lazy(a.c0, b.c0), fsub_lazy(a.c1, b.c1)}; }
// a - b + 6m for a lazy b (< 6m), with the same uses.
ZK_HD fq fsub_x(const fq& a, const fq& b) { return fsub_off<6>(a, b); }
ZK_HD fq2 fsub_x(const fq2& a, const fq2& b) { return fq2{fsub_off<6>(a.c0, b.c0), fsub_off<6>(a.c1, b.c1)}; }
ZK_HD fq2 fsub3_lazy(const fq2& a, const fq2& b, const fq2& c) {
  return fq2{fsub3_lazy(a.c0, b.c0, c.c0), fsub3_lazy(a.c1, b.c1, c.c1)};
}
ZK_HD fq2 ftriple_wide(const fq2& a) { return fq2{ftriple_wide(a.c0), ftriple_wide(a.c1)}; }
ZK_HD fq2 fadd_wide(const fq2& a, const fq2& b) { return fq2{fadd_wide(a.c0, b.c0), fadd_wide(a.c1, b.c1)}; }
// a^2 = 0 mod m for a square of a value below 7m (fsqr's bounds above)
ZK_HD bool fis_zero_sqr(const fq& a) { return fis_zero<FqP>(a); }
ZK_HD bool fis_zero_sqr(const fq2& a) { return fis_zero4<FqP>(a.c0) && fis_zero<FqP>(a.c1); }
// lazy X (< 6m) into [0, 2m)
ZK_HD fq freduce_x(const fq& a) { return fcsub(fcsub(a, FqP::MOD4), FqP::MOD2); }
ZK_HD fq2 freduce_x(const fq2& a) { return fq2{freduce_x(a.c0), freduce_x(a.c1)}; }

// ------------------------------------------------------------------ XYZZ
template <class F>
struct xyzz {
  F x, y, zz, zzz;
};

template <class F>
ZK_HD void xyzz_set_inf(xyzz<F>& p) {
  fset_zero(p.x);
  fset_zero(p.y);
  fset_zero(p.zz);
  fset_zero(p.zzz);
}

template <class F>
ZK_HD bool xyzz_is_inf(const xyzz<F>& p) {
  return fis_zero(p.zz);
}

template <class F>
ZK_HD void xyzz_set_affine(xyzz<F>& p, const F& x, const F& y) {
  p.x = x;
  p.y = y;
  fset_one(p.zz);
  fset_one(p.zzz);
}

// Shared tail of the doublings: y below 2m, x lazy; w = U V, zz = V (times the
// old ZZ, ZZZ by the caller).
template <class F>
ZK_HD void xyzz_dbl_xy(const F& x, const F& y, F& x3, F& y3, F& v, F& w) {
  const F u = fadd_wide(y, y);
  v = fsqr(u);
  w = fmul(v, u);
  const F s = fmul(v, x);
  const F m = ftriple_wide(fsqr(x));
  F zero;
  fset_zero(zero);
  x3 = fsub3_lazy(fsqr(m), zero, s);
  y3 = fmul_sub(m, fsub_x(s, x3), w, y);
}

// p = 2 * (x, y) for an affine point (mdbl-2008-s-1)
template <class F>
ZK_HD void xyzz_mdbl_lx(xyzz<F>& p, const F& x, const F& y) {
  F x3, y3, v, w;
  xyzz_dbl_xy(x, y, x3, y3, v, w);
  p.x = x3;
  p.y = y3;
  p.zz = v;
  p.zzz = w;
}

// p = 2p (dbl-2008-s-1)
template <class F>
ZK_HD void xyzz_dbl_lx(xyzz<F>& p) {
  if (xyzz_is_inf(p)) return;
  F x3, y3, v, w;
  xyzz_dbl_xy(p.x, p.y, x3, y3, v, w);
  p.x = x3;
  p.y = y3;
  p.zz = fmul(p.zz, v);
  p.zzz = fmul(p.zzz, w);
}

// p += (x2, y2), affine and finite, for a finite p (madd-2008-s); returns true
// when the sum is the point at infinity (then p is set to it).  Ordered for few
// live values: x2 and y2 are dead after P and R (equal points double p itself),
// X after Q, PP and P after PPP, and R^2 comes last.
template <class F>
ZK_HD bool xyzz_madd_fin_lx(xyzz<F>& p, const F& x2, const F& y2) {
  const F P = fsub_x(fmul(x2, p.zz), p.x);
  const F R = fsub_m(fmul(y2, p.zzz), p.y);
  const F pp = fsqr(P);
  if (__builtin_expect(fis_zero_sqr(pp), 0)) {
    if (fis_zero_sqr(fsqr(R))) {
      xyzz_dbl_lx(p);
      return false;
    }
    xyzz_set_inf(p);
    return true;
  }
  const F q = fmul_x(p.x, pp);
  p.zz = fmul(p.zz, pp);
  const F ppp = fmul(pp, P);
  p.zzz = fmul(p.zzz, ppp);
  p.x = fsub3_lazy(fsqr(R), ppp, q);
  p.y = fmul_sub(R, fsub_x(q, p.x), p.y, ppp);
  return false;
}

// p += q (add-2008-s)
template <class F>
ZK_HD void xyzz_add_lx(xyzz<F>& p, const xyzz<F>& q) {
  if (xyzz_is_inf(q)) return;
  if (xyzz_is_inf(p)) {
    p = q;
    return;
  }
  const F u1 = fmul(q.zz, p.x);
  const F P = fsub_m(fmul(p.zz, q.x), u1);
  const F s1 = fmul(p.y, q.zzz);
  const F R = fsub_m(fmul(q.y, p.zzz), s1);
  const F pp = fsqr(P);
  if (__builtin_expect(fis_zero(pp), 0)) {
    if (fis_zero(fsqr(R))) xyzz_dbl_lx(p);
    else xyzz_set_inf(p);
    return;
  }
  const F qq = fmul(u1, pp);
  p.zz = fmul(fmul(p.zz, q.zz), pp);
  const F ppp = fmul(pp, P);
  p.zzz = fmul(fmul(p.zzz, q.zzz), ppp);
  p.x = fsub3_lazy(fsqr(R), ppp, qq);
  p.y = fmul_sub(R, fsub_x(qq, p.x), s1, ppp);
}

// p += (x2, y2) affine and finite, every coordinate below 2m.
template <class F>
ZK_HD void xyzz_madd(xyzz<F>& p, const F& x2, const F& y2) {
  if (xyzz_is_inf(p)) {
    xyzz_set_affine(p, x2, y2);
    return;
  }
  (void)xyzz_madd_fin_lx(p, x2, y2);
  p.x = freduce_x(p.x);
}

// a^-1 = a^(q-2) (Fermat); Fq2 through the norm: (c0 - c1 u) / (c0^2 + c1^2)
ZK_HD fq finv(const fq& a) {
  const uint32_t qm2[8] = {0xd87cfd45u, 0x3c208c16u, 0x6871ca8du, 0x97816a91u,
                           0x8181585du, 0xb85045b6u, 0xe131a029u, 0x30644e72u};  // q - 2
  return fpow(a, qm2);
}
ZK_HD fq2 finv(const fq2& a) {
  fq n = finv(fadd(fsqr(a.c0), fsqr(a.c1)));
  return fq2{fmul(a.c0, n), fneg(fmul(a.c1, n))};
}

// Affine forms x = X / ZZ, y = Y / ZZZ of PER points with one inversion of
// the product of every ZZ * ZZZ (Montgomery's trick); inf[j] marks the point
// at infinity (x, y then unset).  X may be lazy.
template <class F, int PER>
ZK_HD void xyzz_to_affine_batch(const xyzz<F> (&p)[PER], F (&x)[PER], F (&y)[PER], bool (&inf)[PER]) {
  F pre[PER], d[PER];
  F prod;
  fset_one(prod);
  for (int j = 0; j < PER; j++) {
    pre[j] = prod;
    inf[j] = xyzz_is_inf(p[j]);
    if (!inf[j]) {
      d[j] = fmul(p[j].zz, p[j].zzz);
      prod = fmul(prod, d[j]);
    }
  }
  F inv = finv(prod);
  for (int j = PER - 1; j >= 0; j--) {
    if (inf[j]) continue;
    F di = fmul(inv, pre[j]);  // 1 / (ZZ_j ZZZ_j)
    inv = fmul(inv, d[j]);
    x[j] = fmul_x(p[j].x, fmul(di, p[j].zzz));
    y[j] = fmul(p[j].y, fmul(di, p[j].zz));
  }
}

}  // namespace zk
