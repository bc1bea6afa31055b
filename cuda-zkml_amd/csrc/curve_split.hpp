// Fq2 split over a lane pair, for the latency-bound G2 kernels (chunk
// combine, bucket reduction).  There a few waves each run a long chain of
// dependent point additions, so the chain's length in instructions is the
// time.  With fq2h the two coordinates of every Fq2 value live in two
// adjacent lanes (even lane: c0, odd lane: c1): additions are one Fq
// operation per lane, and a product takes the partner's coordinates through a
// DPP lane swap and then needs a single fmul_sum per lane instead of two.
// The XYZZ formulas of curve.hpp run unchanged on fq2h.
//
// Both lanes of a pair must execute together: every branch inside these
// operations is taken on values both lanes agree on (fis_zero combines the
// two halves), and the kernels index work by pair.
#pragma once
#include "curve.hpp"

namespace zk {

struct fq2h {
  fq c;  // this lane's coordinate: c0 (even lane) or c1 (odd lane)
};

__device__ __forceinline__ bool lane_odd() { return (threadIdx.x & 1) != 0; }

// the partner lane's value (DPP quad_perm [1, 0, 3, 2])
__device__ __forceinline__ uint32_t swap_pair(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false);
}
__device__ __forceinline__ fq swap_pair(const fq& a) {
  fq r;
#pragma unroll
  for (int i = 0; i < NL; i++) r.l[i] = swap_pair(a.l[i]);
  return r;
}
__device__ __forceinline__ fq fsel(bool odd, const fq& a, const fq& b) {
  fq r;
#pragma unroll
  for (int i = 0; i < NL; i++) r.l[i] = odd ? a.l[i] : b.l[i];
  return r;
}

__device__ __forceinline__ fq2h fneg_canon_if(const fq2h& a, bool neg) { return fq2h{fneg_canon_if(a.c, neg)}; }
__device__ __forceinline__ fq2h fsub_m(const fq2h& a, const fq2h& b) { return fq2h{fsub_lazy(a.c, b.c)}; }
__device__ __forceinline__ fq2h fsub_x(const fq2h& a, const fq2h& b) { return fq2h{fsub_off<6>(a.c, b.c)}; }
__device__ __forceinline__ fq2h fsub3_lazy(const fq2h& a, const fq2h& b, const fq2h& c) {
  return fq2h{fsub3_lazy(a.c, b.c, c.c)};
}
__device__ __forceinline__ fq2h ftriple_wide(const fq2h& a) { return fq2h{ftriple_wide(a.c)}; }
__device__ __forceinline__ fq2h fadd_wide(const fq2h& a, const fq2h& b) { return fq2h{fadd_wide(a.c, b.c)}; }

__device__ __forceinline__ bool fis_zero(const fq2h& a) {
  const uint32_t z = fis_zero(a.c) ? 1u : 0u;
  return (z & swap_pair(z)) != 0;
}
__device__ __forceinline__ bool fis_zero_sqr(const fq2h& a) {
  const uint32_t z = fis_zero4<FqP>(a.c) ? 1u : 0u;
  return (z & swap_pair(z)) != 0;
}
__device__ __forceinline__ void fset_zero(fq2h& a) { a.c = fe_zero<FqP>(); }
__device__ __forceinline__ void fset_one(fq2h& a) { a.c = lane_odd() ? fe_zero<FqP>() : fe_one<FqP>(); }

// The even / odd lane's coordinate on both lanes of the pair (DPP quad_perm
// [0, 0, 2, 2] and [1, 1, 3, 3]).  The operations below take their operands by
// these moves and by negations under a lane mask instead of selects.  (A move may
// read a register two wait states after its write at the earliest, and the
// compiler does not see the writes inside a product's assembly block: the limbs go
// in order, the block writes the last ones last.  A test looks at every move of
// the built library.)
template <int CTRL>
__device__ __forceinline__ fq dpp_fq(const fq& a) {
  fq r;
#pragma unroll
  for (int i = 0; i < NL; i++) r.l[i] = (uint32_t)__builtin_amdgcn_mov_dpp((int)a.l[i], CTRL, 0xF, 0xF, false);
  return r;
}
__device__ __forceinline__ fq even_both(const fq2h& a) { return dpp_fq<0xA0>(a.c); }
__device__ __forceinline__ fq odd_both(const fq2h& a) { return dpp_fq<0xF5>(a.c); }
// all ones on even lanes; opaque, so that the compiler does not keep the masked
// modulus limbs of every operation in registers across a loop (36 of them, which
// the G2 accumulation spilled)
__device__ __forceinline__ uint32_t even_mask() {
  uint32_t m = (threadIdx.x & 1u) - 1u;
  asm volatile("" : "+v"(m));
  return m;
}

// (a0 + a1 u)(b0 + b1 u): even lane a0 b0 + (-a1) b1, odd lane a0 b1 + a1 b0
// (the pairs of the fq2 fmul of curve.hpp, with the same operand bounds).
__device__ __forceinline__ fq2h fmul(const fq2h& a, const fq2h& b) {
  const fq x[2] = {even_both(a), fneg_wide_mask(odd_both(a), even_mask())};
  const fq y[2] = {b.c, swap_pair(b.c)};
  return fq2h{fmul_sum<FqP, 2>(x, y)};
}
__device__ __forceinline__ fq2h fmul_x(const fq2h& x, const fq2h& b) { return fmul(b, x); }

// (a + bu)^2: even lane (a0 + a1)(a0 - a1 + 8q), odd lane (a0 + a0) a1; each
// first factor is the partner's coordinate plus a0.
__device__ __forceinline__ fq2h fsqr(const fq2h& a) {
  const uint32_t mask = even_mask();
  const fq pa = swap_pair(a.c);
  fq w;  // even: a0 - a1 + 8q, odd: a1
  int32_t c = 0;
#pragma unroll
  for (int i = 0; i < NL; i++) {
    int32_t v = (int32_t)(a.c.l[i] + (mask & (FqP::MOD8[i] - pa.l[i]))) + c;
    c = v >> 29;
    w.l[i] = (uint32_t)v & LMASK;
  }
  return fq2h{fmul(fadd_lazy(pa, even_both(a)), w)};
}

// a b - c d (fq2 fmul_sub of curve.hpp): even lane a0 b0 - a1 b1 - c0 d0 +
// c1 d1, odd lane a0 b1 + a1 b0 - c0 d1 - c1 d0.
__device__ __forceinline__ fq2h fmul_sub(const fq2h& a, const fq2h& b, const fq2h& c, const fq2h& d) {
  const uint32_t mask = even_mask();
  const fq x[4] = {even_both(a), fneg_mask<6>(odd_both(a), mask), fneg_lazy(even_both(c)),
                   fneg_mask<2>(odd_both(c), ~mask)};
  const fq y[4] = {b.c, swap_pair(b.c), d.c, swap_pair(d.c)};
  return fq2h{fmul_sum<FqP, 4>(x, y)};
}

// Point loads and stores between the fq2 memory layout (c0 then c1 for each
// coordinate) and the lane-pair registers: each lane moves its half.
__device__ __forceinline__ xyzz<fq2h> load_half(const xyzz<fq2>& p) {
  const int r = lane_odd() ? 1 : 0;
  const fq* w = (const fq*)&p;
  return xyzz<fq2h>{fq2h{w[0 + r]}, fq2h{w[2 + r]}, fq2h{w[4 + r]}, fq2h{w[6 + r]}};
}
__device__ __forceinline__ void store_half(xyzz<fq2>& p, const xyzz<fq2h>& v) {
  const int r = lane_odd() ? 1 : 0;
  fq* w = (fq*)&p;
  w[0 + r] = v.x.c;
  w[2 + r] = v.y.c;
  w[4 + r] = v.zz.c;
  w[6 + r] = v.zzz.c;
}

// Register form of the latency-bound kernels: fq stays one lane per point,
// fq2 becomes a lane pair.
template <class F>
struct Lanes {
  typedef F R;
  typedef xyzz<F> Pt;
  static constexpr int N = 1;
  __device__ static xyzz<F> load(const xyzz<F>& p) { return p; }
  __device__ static void store(xyzz<F>& p, const xyzz<F>& v) { p = v; }
};
template <>
struct Lanes<fq2> {
  typedef fq2h R;
  typedef xyzz<fq2h> Pt;
  static constexpr int N = 2;
  __device__ static xyzz<fq2h> load(const xyzz<fq2>& p) { return load_half(p); }
  __device__ static void store(xyzz<fq2>& p, const xyzz<fq2h>& v) { store_half(p, v); }
};

}  // namespace zk

namespace zk {

// ------------------------------------------------------------------ split point operations
// One point operation of a latency-bound chain dealt to two lane groups
// ("roles"): G1 to a lane pair (E = fq, role = lane bit 0), G2 to two lane
// pairs (E = fq2h, role = lane bit 1, each pair holding the two Fq2 halves).
// Role 0 holds x and zz of the point, role 1 y and zzz: the independent
// products of the formulas then take their operands from the role's own half
//   U1, U2, ZZ1 ZZ2, P, P^2   |   S1, S2, ZZZ1 ZZZ2, R, R^2
// and only five values cross between the roles (U1, P^2, R^2, PPP, Q), each
// as one broadcast lane move per limb.  An addition's 12 products, 2 squares
// and one two-product sum become 5 products, a square and the sum deep; it
// issues about 0.6 of the instructions of the one-lane form on each lane.
// Holding the whole point in both roles instead took 12 nine-limb selects to
// pick each role's operands (and the selects ran through VCC back to back, 15
// to 23 cycles each).  The roles branch together (every branch tests values
// both hold).
template <class E>
struct xyzz_half {
  E a, b;  // role 0: x (lazy, as in the *_lx forms), zz; role 1: y, zzz
};

template <class E>
struct SplitRole;
template <>
struct SplitRole<fq> {
  static constexpr uint32_t BIT = 1;
  static constexpr int FROM0 = 0xA0, FROM1 = 0xF5;  // quad_perm [0, 0, 2, 2], [1, 1, 3, 3]
};
template <>
struct SplitRole<fq2h> {
  static constexpr uint32_t BIT = 2;
  static constexpr int FROM0 = 0x44, FROM1 = 0xEE;  // quad_perm [0, 1, 0, 1], [2, 3, 2, 3]
};

template <class E>
__device__ __forceinline__ bool split_role1() {
  return (threadIdx.x & SplitRole<E>::BIT) != 0;
}

template <int CTRL>
__device__ __forceinline__ fq2h dpp_fq(const fq2h& a) {
  return fq2h{dpp_fq<CTRL>(a.c)};
}
// role 0's / role 1's value of a, on both roles
template <class E>
__device__ __forceinline__ E from0(const E& a) {
  return dpp_fq<SplitRole<E>::FROM0>(a);
}
template <class E>
__device__ __forceinline__ E from1(const E& a) {
  return dpp_fq<SplitRole<E>::FROM1>(a);
}
__device__ __forceinline__ fq pick(bool c, const fq& a, const fq& b) { return fsel(c, a, b); }
__device__ __forceinline__ fq2h pick(bool c, const fq2h& a, const fq2h& b) { return fq2h{fsel(c, a.c, b.c)}; }

template <class E>
__device__ __forceinline__ void xyzz_set_inf(xyzz_half<E>& p) {
  fset_zero(p.a);
  fset_zero(p.b);
}

// zz and zzz are 0 mod m together, so both roles find the same answer
template <class E>
__device__ __forceinline__ bool xyzz_is_inf(const xyzz_half<E>& p) {
  return fis_zero(p.b);
}

// p = 2p (dbl-2008-s-1): X^2 | V = U^2, S = X V | W = U V, M^2 and X3 on both,
// ZZ3 = V ZZ | ZZZ3 = W ZZZ, then Y3 = M (S - X3) - W Y on role 1.
template <class E>
__device__ __forceinline__ void xyzz_dbl_lx(xyzz_half<E>& p) {
  if (xyzz_is_inf(p)) return;
  const bool r1 = split_role1<E>();
  const E s = pick(r1, fadd_wide(p.a, p.a), p.a);  // X | U = 2 Y
  const E t = fsqr(s);
  const E V = from1(t), M = ftriple_wide(from0(t));
  const E w = fmul(V, s);  // S | W
  p.b = fmul(pick(r1, w, V), p.b);
  const E S = from0(w);
  E zero;
  fset_zero(zero);
  const E X3 = fsub3_lazy(fsqr(M), zero, S);
  const E d = fmul_sub(M, fsub_x(S, X3), w, p.a);
  p.a = pick(r1, d, X3);
}

// p += q (add-2008-s)
template <class E>
__device__ __forceinline__ void xyzz_add_lx(xyzz_half<E>& p, const xyzz_half<E>& q) {
  if (xyzz_is_inf(q)) return;
  if (xyzz_is_inf(p)) {
    p = q;
    return;
  }
  const bool r1 = split_role1<E>();
  const E a = fmul(q.b, p.a);                // U1 | S1
  const E PR = fsub_m(fmul(p.b, q.a), a);    // P | R, lazy, (0, 4m)
  const E t = fsqr(PR);                      // PP | RR
  const E PP = from0(t);
  if (__builtin_expect(fis_zero(PP), 0)) {
    if (fis_zero(from1(t))) xyzz_dbl_lx(p);
    else xyzz_set_inf(p);
    return;
  }
  const E v = fmul(PP, pick(r1, from0(a), PR));        // PPP | Q = U1 PP
  const E PPP = from0(v);
  p.b = fmul(fmul(p.b, q.b), pick(r1, PPP, PP));       // ZZ3 | ZZZ3
  const E Q = from1(v);
  const E X3 = fsub3_lazy(from1(t), PPP, Q);
  const E d = fmul_sub(PR, fsub_x(Q, X3), a, PPP);     // | Y3 = R (Q - X3) - S1 PPP
  p.a = pick(r1, d, X3);
}

// The point in the register form of each layout: Lanes (and one lane per
// point): xyzz<R>; SplitLanes: xyzz_half<E>, the coordinates moved by the role
// that holds them.
template <class F>
struct SplitLanes;
template <>
struct SplitLanes<fq> {
  typedef xyzz_half<fq> Pt;
  static constexpr int N = 2;
  __device__ static Pt load(const xyzz<fq>& p) {
    const int r = split_role1<fq>() ? 1 : 0;
    const fq* w = (const fq*)&p;
    return Pt{w[r], w[2 + r]};
  }
  __device__ static void store(xyzz<fq>& p, const Pt& v) {
    const int r = split_role1<fq>() ? 1 : 0;
    fq* w = (fq*)&p;
    w[r] = v.a;
    w[2 + r] = v.b;
  }
};
template <>
struct SplitLanes<fq2> {
  typedef xyzz_half<fq2h> Pt;
  static constexpr int N = 4;
  // fq words of p: x0 x1 y0 y1 zz0 zz1 zzz0 zzz1; this lane's are at 2 role + half
  __device__ static int word() { return (int)(threadIdx.x & 3); }
  __device__ static Pt load(const xyzz<fq2>& p) {
    const fq* w = (const fq*)&p;
    return Pt{fq2h{w[word()]}, fq2h{w[4 + word()]}};
  }
  __device__ static void store(xyzz<fq2>& p, const Pt& v) {
    fq* w = (fq*)&p;
    w[word()] = v.a.c;
    w[4 + word()] = v.b.c;
  }
};

}  // namespace zk
