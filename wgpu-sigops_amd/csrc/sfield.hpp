// sfield.hpp -- the field arithmetic of the point ladders: 9 limbs of 29 bits as in field.hpp, but
// signed throughout, for the three field primes (Montgomery form, R = 2^261).
//
// field.hpp keeps every value and every column non-negative: a subtraction adds a biased multiple
// of M, sums are folded back (fnorm_red, 29-41 instructions), and the columns of a product start at
// offsets that the compiler adds one by one (14 64-bit adds in a secp256k1 product). Here values
// lie in (-kM, kM), a limb is any i32, products are v_mad_i64_i32 on signed columns and carries are
// arithmetic shifts, so:
//   * a difference is one 32-bit subtraction per limb and needs neither a bias nor a fold;
//   * a product has no offsets: 167 VALU instructions against 189 (secp256k1);
//   * scaling by 2 or 3 and the subtraction of an unreduced value happen inside the final carry
//     chain, which returns normalised limbs either way;
//   * a b + c d takes one reduction (s_dot), which removes one of 7 (doubling) and of 11 (addition).
// Normalised here: limbs 0..7 in [0, 2^29), limb 8 signed and small; every product returns that.
// What may enter a product is bounded by its columns alone: each must lie in [-2^63, 2^63) where it
// is shifted. Host builds with SIGOPS_HOST_CHECK=1 carry limb and value intervals through every
// operation and check that for the worst case, as field.hpp does for its own bounds.
#pragma once
#include "field.hpp"

namespace sigops {

struct sfe {
  i32 v[NL];
#if SIGOPS_BOUNDS
  i64 lo = 0, hi = LMASK;          // limbs 0..7
  i64 tlo = 0, thi = 1 << 25;      // limb 8
  long double vlo = 0, vhi = 231584178474632390847141970017375815706539969331281128078915168015826259279872.0L;
#endif
};

#if SIGOPS_BOUNDS
inline long double sfe_ld(const sfe& a) {
  long double x = 0;
  for (int k = NL - 1; k >= 0; k--) x = ldexpl(x, 29) + a.v[k];
  return x;
}
inline void s_check(const sfe& a, const char* what) {
  for (int k = 0; k < NL - 1; k++) BCHECK(a.v[k] >= a.lo && a.v[k] <= a.hi, what);
  BCHECK(a.v[NL - 1] >= a.tlo && a.v[NL - 1] <= a.thi, what);
  const long double x = sfe_ld(a), slack = p2(200);
  BCHECK(x >= a.vlo - slack && x <= a.vhi + slack, what);
}
inline void s_limbs_fit(const sfe& a) {
  BCHECK(a.lo >= -(1ll << 31) && a.hi < (1ll << 31) && a.tlo >= -(1ll << 31) && a.thi < (1ll << 31), "limb outside i32");
}
// an interval, for the worst case of a column
struct ival {
  long double lo = 0, hi = 0;
  void add(long double l, long double h) {
    lo += l;
    hi += h;
  }
  void mac(i64 al, i64 ah, i64 bl, i64 bh) {
    const long double p[4] = {(long double)al * bl, (long double)al * bh, (long double)ah * bl, (long double)ah * bh};
    long double l = p[0], h = p[0];
    for (long double x : p) {
      l = x < l ? x : l;
      h = x > h ? x : h;
    }
    add(l, h);
  }
  void fits() const { BCHECK(lo >= -p2(63) && hi < p2(63), "signed column out of range"); }
};
inline void s_range(const sfe& a, int k, i64& l, i64& h) {
  l = k == NL - 1 ? a.tlo : a.lo;
  h = k == NL - 1 ? a.thi : a.hi;
}
// columns of sum (+-) a b over the given pairs, Montgomery steps, shifts; then the final chain
// (times `scale`, less `sub` when given); sets the bounds of the result r and checks it
struct spair {
  const sfe* a;
  const sfe* b;
};
template <class F>
inline void s_bounds(std::initializer_list<spair> plus, const sfe* minus_sq, int scale, const sfe* sub, int sub_c, sfe& r) {
  ival col[2 * NL - 1];
  long double vl = 0, vh = 0;
  for (const spair& p : plus) {
    s_check(*p.a, "signed product input");
    s_check(*p.b, "signed product input");
    for (int i = 0; i < NL; i++)
      for (int j = 0; j < NL; j++) {
        i64 al, ah, bl, bh;
        s_range(*p.a, i, al, ah);
        s_range(*p.b, j, bl, bh);
        col[i + j].mac(al, ah, bl, bh);
      }
    ival v;
    const long double q[4] = {p.a->vlo * p.b->vlo, p.a->vlo * p.b->vhi, p.a->vhi * p.b->vlo, p.a->vhi * p.b->vhi};
    v.lo = v.hi = q[0];
    for (long double x : q) {
      v.lo = x < v.lo ? x : v.lo;
      v.hi = x > v.hi ? x : v.hi;
    }
    if (p.a == p.b && v.lo < 0) v.lo = 0;
    vl += v.lo;
    vh += v.hi;
  }
  if (minus_sq) {
    s_check(*minus_sq, "signed product input");
    for (int i = 0; i < NL; i++)
      for (int j = 0; j < NL; j++) {
        i64 al, ah, bl, bh;
        s_range(*minus_sq, i, al, ah);
        s_range(*minus_sq, j, bl, bh);
        col[i + j].mac(-ah, -al, bl, bh);
      }
    const long double m = minus_sq->vhi > -minus_sq->vlo ? minus_sq->vhi : -minus_sq->vlo;
    vl -= m * m;
  }
  const long double MM = (long double)LMASK;
  for (int i = 0; i < NL; i++) {
    if (i) col[i].add(floorl(col[i - 1].lo / p2(29)), floorl(col[i - 1].hi / p2(29)));
    for (int t = 0; t < F::SP_N; t++) {
      const long double c = (long double)F::SP_COEF[t] * MM;
      if (t == 0 && F::SP_COEF[t] == -1) continue;
      col[i + F::SP_OFF[t]].add(c < 0 ? c : 0, c > 0 ? c : 0);
    }
    col[i].fits();
  }
  long double cl = floorl(col[NL - 1].lo / p2(29)) * scale, ch = floorl(col[NL - 1].hi / p2(29)) * scale;
  for (int k = 0; k < NL - 1; k++) {
    ival t;
    t.lo = col[NL + k].lo * scale + cl;
    t.hi = col[NL + k].hi * scale + ch;
    if (sub) t.add(-(long double)sub_c * sub->hi, -(long double)sub_c * sub->lo);
    t.fits();
    cl = floorl(t.lo / p2(29));
    ch = floorl(t.hi / p2(29));
  }
  const long double M = mod_ld<F>();
  r.vlo = vl / p2(261) * scale;
  r.vhi = (vh / p2(261) + M) * scale;
  if (sub) {
    s_check(*sub, "subtrahend");
    const long double a = r.vlo, b = r.vhi;
    r.vlo = a - sub_c * sub->vhi;
    r.vhi = b - sub_c * sub->vlo;
  }
  r.lo = 0;
  r.hi = LMASK;
  r.tlo = (i64)floorl(r.vlo / p2(232)) - 1;
  r.thi = (i64)floorl(r.vhi / p2(232)) + 1;
  s_limbs_fit(r);
  s_check(r, "signed product output");
}
#endif

// ---- limbwise operations ----
DEV sfe s_from(const fe& a) {  // a non-negative value
  sfe r;
#pragma unroll
  for (int k = 0; k < NL; k++) r.v[k] = (i32)a.v[k];
#if SIGOPS_BOUNDS
  r.lo = 0;
  r.hi = (i64)a.lmax;
  r.tlo = 0;
  r.thi = (i64)a.tmax;
  r.vlo = 0;
  r.vhi = a.vmax;
  s_limbs_fit(r);
#endif
  return r;
}

DEV sfe s_add(const sfe& a, const sfe& b) {
  sfe r;
#pragma unroll
  for (int k = 0; k < NL; k++) r.v[k] = a.v[k] + b.v[k];
#if SIGOPS_BOUNDS
  r.lo = a.lo + b.lo, r.hi = a.hi + b.hi, r.tlo = a.tlo + b.tlo, r.thi = a.thi + b.thi;
  r.vlo = a.vlo + b.vlo, r.vhi = a.vhi + b.vhi;
  s_limbs_fit(r);
#endif
  return r;
}

DEV sfe s_sub(const sfe& a, const sfe& b) {
  sfe r;
#pragma unroll
  for (int k = 0; k < NL; k++) r.v[k] = a.v[k] - b.v[k];
#if SIGOPS_BOUNDS
  r.lo = a.lo - b.hi, r.hi = a.hi - b.lo, r.tlo = a.tlo - b.thi, r.thi = a.thi - b.tlo;
  r.vlo = a.vlo - b.vhi, r.vhi = a.vhi - b.vlo;
  s_limbs_fit(r);
#endif
  return r;
}

DEV sfe s_dbl(const sfe& a) { return s_add(a, a); }

DEV sfe s_neg(const sfe& a) {
  sfe r;
#pragma unroll
  for (int k = 0; k < NL; k++) r.v[k] = -a.v[k];
#if SIGOPS_BOUNDS
  r.lo = -a.hi, r.hi = -a.lo, r.tlo = -a.thi, r.thi = -a.tlo, r.vlo = -a.vhi, r.vhi = -a.vlo;
#endif
  return r;
}

DEV sfe s_neg_if(bool neg, const sfe& a) {  // two 32-bit operations per limb
  const i32 m = (i32)lane_mask(neg);
  sfe r;
#pragma unroll
  for (int k = 0; k < NL; k++) r.v[k] = (a.v[k] ^ m) - m;
#if SIGOPS_BOUNDS
  const i64 x = a.hi > -a.lo ? a.hi : -a.lo, t = a.thi > -a.tlo ? a.thi : -a.tlo;
  const long double y = a.vhi > -a.vlo ? a.vhi : -a.vlo;
  r.lo = -x, r.hi = x, r.tlo = -t, r.thi = t, r.vlo = -y, r.vhi = y;
#endif
  return r;
}

DEV sfe s_sel(u32 mask, const sfe& a, const sfe& b) {  // mask ? a : b, limbwise
  sfe r;
#pragma unroll
  for (int k = 0; k < NL; k++) r.v[k] = (i32)(((u32)a.v[k] & mask) | ((u32)b.v[k] & ~mask));
#if SIGOPS_BOUNDS
  r.lo = a.lo < b.lo ? a.lo : b.lo, r.hi = a.hi > b.hi ? a.hi : b.hi;
  r.tlo = a.tlo < b.tlo ? a.tlo : b.tlo, r.thi = a.thi > b.thi ? a.thi : b.thi;
  r.vlo = a.vlo < b.vlo ? a.vlo : b.vlo, r.vhi = a.vhi > b.vhi ? a.vhi : b.vhi;
#endif
  return r;
}

// the same value with normalised limbs (one carry chain)
DEV sfe s_carry(const sfe& a) {
  sfe r;
  i32 c = 0;
#pragma unroll
  for (int k = 0; k < NL - 1; k++) {
    const i32 x = a.v[k] + c;
    r.v[k] = (i32)((u32)x & LMASK);
    c = x >> SIGOPS_LIMB_BITS;
  }
  r.v[NL - 1] = a.v[NL - 1] + c;
#if SIGOPS_BOUNDS
  s_check(a, "s_carry input");
  BCHECK(a.lo >= -(1ll << 31) + 8 && a.hi <= (1ll << 31) - 8, "s_carry limbs");
  r.lo = 0, r.hi = LMASK, r.vlo = a.vlo, r.vhi = a.vhi;
  r.tlo = a.tlo - 4, r.thi = a.thi + 4;
#endif
  return r;
}

// ---- products ----
DEV i64 s_mac(i32 x, i32 y, i64 c) { return (i64)((u64)c + (u64)((i64)x * (i64)y)); }

template <class F>
DEV void s_step(i64 (&acc)[2 * NL - 1], int i) {
  static_assert(F::SPARSE, "signed arithmetic is for the field primes");
  if (i > 0) acc[i] += acc[i - 1] >> SIGOPS_LIMB_BITS;
  const i32 m = (i32)(((u32)acc[i] * F::N0) & LMASK);
#pragma unroll
  for (int t = 0; t < F::SP_N; t++) {
    i32 coef = F::SP_COEF[t];
    if (t == 0 && coef == -1) continue;  // only clears bits that the carry shift drops (field.hpp)
#if defined(__HIP_DEVICE_COMPILE__)
    coef = g_sp_coef.v[sp_base<F>() + t];
#endif
    acc[i + F::SP_OFF[t]] = s_mac(coef, m, acc[i + F::SP_OFF[t]]);
  }
}

// the carry chain over columns 8..16: SCALE times the value, less SUBC times sub
template <int SCALE, int SUBC>
DEV sfe s_final(const i64 (&acc)[2 * NL - 1], const sfe* sub) {
  static_assert(SCALE >= 1 && SCALE <= 3, "scales 1, 2, 3");
  sfe r;
  i64 c = acc[NL - 1] >> SIGOPS_LIMB_BITS;
  if (SCALE > 1) c *= SCALE;
#pragma unroll
  for (int k = 0; k < NL - 1; k++) {
    i64 t = acc[NL + k];
    if (SUBC) t = SCALE == 1 ? s_mac(sub->v[k], -SUBC, t) : t;
    if (SCALE == 2) t = (i64)((u64)t << 1);
    if (SCALE == 3) t = (i64)(((u64)t << 1) + (u64)t);
    t = (i64)((u64)t + (u64)c);
    r.v[k] = (i32)((u32)t & LMASK);
    c = t >> SIGOPS_LIMB_BITS;
  }
  r.v[NL - 1] = (i32)c - (SUBC ? SUBC * sub->v[NL - 1] : 0);
  return r;
}

// SCALE a b 2^-261
template <class F, int SCALE = 1>
DEV_MUL sfe s_mul(const sfe& a, const sfe& b) {
  i64 acc[2 * NL - 1] = {};
#pragma unroll
  for (int i = 0; i < NL; i++) {
#pragma unroll
    for (int j = 0; j < NL; j++) acc[i + j] = s_mac(a.v[i], b.v[j], acc[i + j]);
    s_step<F>(acc, i);
  }
  sfe r = s_final<SCALE, 0>(acc, nullptr);
#if SIGOPS_BOUNDS
  s_bounds<F>({{&a, &b}}, nullptr, SCALE, nullptr, 0, r);
#endif
  return r;
}

template <class F>
DEV void s_sqr_acc(const sfe& a, i64 (&acc)[2 * NL - 1]) {
  i32 a2[NL];
#pragma unroll
  for (int k = 0; k < NL; k++) a2[k] = (i32)((u32)a.v[k] << 1);
#pragma unroll
  for (int i = 0; i < NL; i++) {
    acc[2 * i] = s_mac(a.v[i], a.v[i], acc[2 * i]);
#pragma unroll
    for (int j = i + 1; j < NL; j++) acc[i + j] = s_mac(a.v[i], a2[j], acc[i + j]);
    s_step<F>(acc, i);
  }
#if SIGOPS_BOUNDS
  BCHECK(a.lo > -(1ll << 30) && a.hi < (1ll << 30), "square: doubled limb");
#endif
}

// SCALE a^2 2^-261
template <class F, int SCALE = 1>
DEV_MUL sfe s_sqr(const sfe& a) {
  i64 acc[2 * NL - 1] = {};
  s_sqr_acc<F>(a, acc);
  sfe r = s_final<SCALE, 0>(acc, nullptr);
#if SIGOPS_BOUNDS
  s_bounds<F>({{&a, &a}}, nullptr, SCALE, nullptr, 0, r);
#endif
  return r;
}

// a^2 2^-261 - SUBC s
template <class F, int SUBC>
DEV_MUL sfe s_sqr_sub(const sfe& a, const sfe& s) {
  i64 acc[2 * NL - 1] = {};
  s_sqr_acc<F>(a, acc);
  sfe r = s_final<1, SUBC>(acc, &s);
#if SIGOPS_BOUNDS
  s_bounds<F>({{&a, &a}}, nullptr, 1, &s, SUBC, r);
#endif
  return r;
}

// SCALE (a b + c d) 2^-261 with one reduction
template <class F, int SCALE = 1>
DEV_MUL sfe s_dot(const sfe& a, const sfe& b, const sfe& c, const sfe& d) {
  i64 acc[2 * NL - 1] = {};
#pragma unroll
  for (int i = 0; i < NL; i++) {
#pragma unroll
    for (int j = 0; j < NL; j++) {
      acc[i + j] = s_mac(a.v[i], b.v[j], acc[i + j]);
      acc[i + j] = s_mac(c.v[i], d.v[j], acc[i + j]);
    }
    s_step<F>(acc, i);
  }
  sfe r = s_final<SCALE, 0>(acc, nullptr);
#if SIGOPS_BOUNDS
  s_bounds<F>({{&a, &b}, {&c, &d}}, nullptr, SCALE, nullptr, 0, r);
#endif
  return r;
}

// (a b - c^2) 2^-261 with one reduction
template <class F>
DEV_MUL sfe s_dot_sqr(const sfe& a, const sfe& b, const sfe& c) {
  i32 nc[NL], c2[NL];
#pragma unroll
  for (int k = 0; k < NL; k++) {
    nc[k] = -c.v[k];
    c2[k] = (i32)((u32)c.v[k] << 1);
  }
  i64 acc[2 * NL - 1] = {};
#pragma unroll
  for (int i = 0; i < NL; i++) {
    acc[2 * i] = s_mac(nc[i], c.v[i], acc[2 * i]);
#pragma unroll
    for (int j = 0; j < NL; j++) {
      acc[i + j] = s_mac(a.v[i], b.v[j], acc[i + j]);
      if (j > i) acc[i + j] = s_mac(nc[i], c2[j], acc[i + j]);
    }
    s_step<F>(acc, i);
  }
  sfe r = s_final<1, 0>(acc, nullptr);
#if SIGOPS_BOUNDS
  BCHECK(c.lo > -(1ll << 30) && c.hi < (1ll << 30), "square: doubled limb");
  s_bounds<F>({{&a, &b}}, &c, 1, nullptr, 0, r);
#endif
  return r;
}

// x to a fixed exponent along an addition chain (field.hpp, fpow_chain)
template <class F, class CH, int S>
DEV void s_chain_steps(sfe* t) {
  if constexpr (S < CH::N) {
    sfe v = t[CH::SRC[S]];
#pragma unroll 1
    for (int k = 0; k < CH::NSQ[S]; k++) v = s_sqr<F>(v);
    if constexpr (CH::MUL[S] >= 0) v = s_mul<F>(v, t[CH::MUL[S]]);
    t[CH::DST[S]] = v;
    s_chain_steps<F, CH, S + 1>(t);
  }
}
template <class F, class CH>
DEV sfe s_pow_chain(const sfe& x) {
  sfe t[CH::SLOTS];
  t[0] = x;
  s_chain_steps<F, CH, 0>(t);
  return t[CH::RESULT];
}

// SCALE (a^2 - b^2) 2^-261 with one reduction
template <class F, int SCALE = 1>
DEV_MUL sfe s_sqr_diff(const sfe& a, const sfe& b) {
  i32 nb[NL], a2[NL], b2[NL];
#pragma unroll
  for (int k = 0; k < NL; k++) {
    nb[k] = -b.v[k];
    a2[k] = (i32)((u32)a.v[k] << 1);
    b2[k] = (i32)((u32)b.v[k] << 1);
  }
  i64 acc[2 * NL - 1] = {};
#pragma unroll
  for (int i = 0; i < NL; i++) {
    acc[2 * i] = s_mac(a.v[i], a.v[i], acc[2 * i]);
    acc[2 * i] = s_mac(nb[i], b.v[i], acc[2 * i]);
#pragma unroll
    for (int j = i + 1; j < NL; j++) {
      acc[i + j] = s_mac(a.v[i], a2[j], acc[i + j]);
      acc[i + j] = s_mac(nb[i], b2[j], acc[i + j]);
    }
    s_step<F>(acc, i);
  }
  sfe r = s_final<SCALE, 0>(acc, nullptr);
#if SIGOPS_BOUNDS
  BCHECK(a.lo > -(1ll << 30) && a.hi < (1ll << 30) && b.lo > -(1ll << 30) && b.hi < (1ll << 30), "square: doubled limb");
  s_bounds<F>({{&a, &a}}, &b, SCALE, nullptr, 0, r);
#endif
  return r;
}

// the limbs as they are, for tables held as fe
DEV fe s_raw(const sfe& a) {
  fe r;
#pragma unroll
  for (int k = 0; k < NL; k++) r.v[k] = (u32)a.v[k];
  return r;
}
// back from s_raw, with the bounds of any value in (-4M, 4M) with folded limbs
template <class F>
DEV sfe s_unraw(const fe& a) {
  sfe r;
#pragma unroll
  for (int k = 0; k < NL; k++) r.v[k] = (i32)a.v[k];
#if SIGOPS_BOUNDS
  r.lo = -(1 << 25);
  r.hi = (i64)LMASK + (1 << 25);
  r.vhi = 4.0L * mod_ld<F>();
  r.vlo = -r.vhi;
  r.thi = (i64)(r.vhi / p2(232)) + 1;
  r.tlo = -r.thi;
  s_check(r, "s_unraw");
#endif
  return r;
}

// a normalised value in (-K M, K' M), K + K' <= 24, to field.hpp's normalised form, < (1 + 2^-19) M
template <class F, u32 K>
DEV fe s_to_fe(const sfe& a) {
  constexpr limbs9 B = sub_bias<F, K, 1>();  // every limb at least 2^29 - 1: a may be folded (s_fold)
  fe r;
#pragma unroll
  for (int k = 0; k < NL; k++) r.v[k] = (u32)a.v[k] + B.v[k];
#if SIGOPS_BOUNDS
  s_check(a, "s_to_fe input");
  BCHECK(a.lo > -(i64)LMASK && a.hi < 2ll * LMASK && a.vlo > -(long double)K * mod_ld<F>() && a.tlo + (i64)B.v[NL - 1] >= 0, "s_to_fe range");
  BOUNDS_SET(r, (u64)a.hi + 2ull * LMASK + 1, (u64)(a.thi + (i64)B.v[NL - 1]), a.vhi + K * mod_ld<F>());
#endif
  return fnorm_red<F>(r);
}

// the value mod M brought to [0, 2^TOP) plus a few units of its low limbs (TOP = 256, or 255 for
// 2^255 - 19): the signed bits above 2^TOP, read from limb 8, folded with the prime's identity (see
// fnorm_red) into the limbs they belong to, without a carry chain (4 to 7 instructions). |a| < 2^261.
template <class F>
DEV sfe s_fold(const sfe& a) {
  constexpr int TB = F::SP_N == 2 ? 23 : 24;
  sfe r = a;
  const i32 q = a.v[NL - 1] >> TB;
  r.v[NL - 1] = a.v[NL - 1] & ((1 << TB) - 1);
  if constexpr (F::SP_N == 2) {
    r.v[0] += 19 * q;
  } else if constexpr (F::SP_N == 3) {
    r.v[0] += 977 * q;
    r.v[1] += q * 8;
  } else {
    r.v[0] += q;
    r.v[3] -= q * (1 << 9);
    r.v[6] -= q * (1 << 18);
    r.v[7] += q * (1 << 21);
  }
#if SIGOPS_BOUNDS
  s_check(a, "s_fold input");
  const i64 ql = a.tlo >> TB, qh = a.thi >> TB;
  const i64 qm = qh > -ql ? qh : -ql;
  BCHECK(qm < 16, "s_fold range");
  const i64 w = F::SP_N == 5 ? (1 << 21) : 977;
  r.lo = a.lo - w * qm;
  r.hi = a.hi + w * qm;
  r.tlo = 0;
  r.thi = (1 << TB) - 1;
  // the lower limbs add at most (hi - LMASK) 2^203 and a few units beyond 2^TOP
  const long double e = p2(F::SP_N == 2 ? 255 : 256);
  r.vlo = -p2(229);
  r.vhi = e + p2(229);
  s_limbs_fit(r);
  s_check(r, "s_fold output");
#endif
  return r;
}

// whether SCALE h^2 2^-261 (normalised, below 2 SCALE M) may be 0 mod M: true for every multiple of
// M, and false otherwise but for a chance of 2^-56, as only the two lowest limbs are compared with
// those of 0 and SCALE M. A false positive sends its item to the careful path, whose
// result is the same.
template <class F, int SCALE>
DEV bool s_sqr_maybe_zero(const sfe& a) {
  bool any = false;
#pragma unroll
  for (u32 j = 0; j < 2; j++) {
    const u64 m = ((u64)F::M[0] + ((u64)F::M[1] << SIGOPS_LIMB_BITS)) * (u64)(j * SCALE);
    const u32 l0 = (u32)m & LMASK, l1 = (u32)(m >> SIGOPS_LIMB_BITS) & LMASK;
    any = any || (((u32)a.v[0] ^ l0) | ((u32)a.v[1] ^ l1)) == 0;
  }
#if SIGOPS_BOUNDS
  BCHECK(a.lo >= 0 && a.hi <= LMASK && a.vlo >= 0 && a.vhi < 2.0L * SCALE * mod_ld<F>(), "s_sqr_maybe_zero input");
#endif
  return any;
}

}  // namespace sigops
