// quad.hpp -- point arithmetic spread over four lanes, for calls too small to fill the GPU.
//
// One lane per signature leaves a call of a few thousand items with one wavefront on some SIMDs and
// the others idle, and its time is one item's serial chain of instructions. Here the four lanes of
// a quad hold the four coordinates of one point, one field element each, and the independent
// products of a formula run side by side: a doubling takes 3 products in sequence instead of 6 to 8, an
// addition 4 instead of 10 (secp, XYZZ coordinates), an Edwards operation 2 instead of 7 or 8
// (Hisil, Wong, Carter, Dawson 2008, section 4: four processors). Operands move between the lanes
// with DPP quad permutations, which cost no memory access.
// Instructions in sequence (secp256k1): doubling 720 against 1,055, addition 900 against 1,740.
//
// Host builds (tests) hold the four lanes in an array and check the bounds of every lane.
#pragma once
#include "ed25519.hpp"

namespace sigops {

constexpr int Q0 = 1, Q1 = 2, Q2 = 4, Q3 = 8;  // lane masks

#if defined(__HIP_DEVICE_COMPILE__)
typedef sfe qfe;  // this lane's element
DEV u32 q_lane() { return threadIdx.x & 3u; }
template <int MASK>
DEV u32 q_mask() {
  return lane_mask((MASK >> q_lane()) & 1);
}
// lane k takes the element of lane A, B, C, D (k = 0, 1, 2, 3)
template <int A, int B, int C, int D>
DEV qfe q_perm(const qfe& x) {
  qfe r;
#pragma unroll
  for (int k = 0; k < NL; k++)
    r.v[k] = __builtin_amdgcn_mov_dpp(x.v[k], A | (B << 2) | (C << 4) | (D << 6), 0xf, 0xf, true);
  return r;
}
#define Q_EACH(expr) \
  {                  \
    return expr;     \
  }
#define Q_AT(x) x
#else
struct qfe {
  sfe l[4];
};
template <int A, int B, int C, int D>
DEV qfe q_perm(const qfe& x) {
  return qfe{{x.l[A], x.l[B], x.l[C], x.l[D]}};
}
#define Q_EACH(expr)                         \
  {                                          \
    qfe r_;                                  \
    for (int q = 0; q < 4; q++) r_.l[q] = expr; \
    return r_;                               \
  }
#define Q_AT(x) x.l[q]
#endif

template <int K>
DEV qfe q_bcast(const qfe& x) {
  return q_perm<K, K, K, K>(x);
}
DEV qfe q_add(const qfe& a, const qfe& b) Q_EACH(s_add(Q_AT(a), Q_AT(b)))
DEV qfe q_sub(const qfe& a, const qfe& b) Q_EACH(s_sub(Q_AT(a), Q_AT(b)))
DEV qfe q_dbl(const qfe& a) Q_EACH(s_dbl(Q_AT(a)))
DEV qfe q_carry(const qfe& a) Q_EACH(s_carry(Q_AT(a)))
template <class F>
DEV qfe q_fold(const qfe& a) Q_EACH(s_fold<F>(Q_AT(a)))
template <class F, int SCALE = 1>
DEV qfe q_mul(const qfe& a, const qfe& b) Q_EACH((s_mul<F, SCALE>(Q_AT(a), Q_AT(b))))
template <class F>
DEV qfe q_sqr(const qfe& a) Q_EACH(s_sqr<F>(Q_AT(a)))

// lanes in MASK take a, the others b
template <int MASK>
DEV qfe q_sel(const qfe& a, const qfe& b) {
#if defined(__HIP_DEVICE_COMPILE__)
  return s_sel(q_mask<MASK>(), a, b);
#else
  qfe r;
  for (int q = 0; q < 4; q++) r.l[q] = ((MASK >> q) & 1) ? a.l[q] : b.l[q];
  return r;
#endif
}
// zero outside MASK
template <int MASK>
DEV qfe q_keep(const qfe& a) {
  qfe r = a;
#if defined(__HIP_DEVICE_COMPILE__)
  const u32 m = q_mask<MASK>();
#pragma unroll
  for (int k = 0; k < NL; k++) r.v[k] = (i32)((u32)r.v[k] & m);
#else
  for (int q = 0; q < 4; q++)
    if (!((MASK >> q) & 1)) r.l[q] = s_from(fe_zero());
#endif
  return r;
}
// negated on the lanes in MASK
template <int MASK>
DEV qfe q_neg(const qfe& a) {
#if defined(__HIP_DEVICE_COMPILE__)
  return s_neg_if((MASK >> q_lane()) & 1, a);
#else
  qfe r = a;
  for (int q = 0; q < 4; q++)
    if ((MASK >> q) & 1) r.l[q] = s_neg(a.l[q]);
  return r;
#endif
}

// ---- secp: XYZZ coordinates with W = 2Y: lanes X, W, ZZ, ZZZ (x = X / ZZ, y = W / (2 ZZZ)) ----
// doubling: V = W^2, S = X V, M = 3X^2 + a ZZ^2, X3 = M^2 - 2S, W3 = 2 M (S - X3) - V^2, ZZ3 = V ZZ,
// ZZZ3 = W V ZZZ. a = 0 or -3. The state's W may have signed limbs, the others are normalised.
template <class C>
DEV qfe q_sdbl(const qfe& s) {
  typedef typename C::Fp F;
  const qfe r1 = q_sqr<F>(s);                        // X^2, V, ZZ^2, -
  qfe t = q_perm<1, 0, 1, 1>(r1);                    // V, X^2, V, V
  if constexpr (C::A_IS_M3) t = q_sub(t, q_keep<Q1>(q_bcast<2>(r1)));
  t = q_carry(q_add(t, q_dbl(q_keep<Q1>(t))));       // V, M, V, V
  const qfe r2 = q_mul<F>(q_sel<Q0>(s, t), q_sel<Q0 | Q1>(t, q_perm<0, 1, 2, 1>(s)));  // S, M^2, ZZ3, W V
  const qfe S = q_bcast<0>(r2);
  const qfe X3 = q_carry(q_sub(q_sub(q_bcast<1>(r2), S), S));
  const qfe y = q_perm<1, 0, 2, 3>(t);               // M, V, -, -
  const qfe r3 = q_mul<F>(q_sel<Q3>(r2, y), q_sel<Q0>(q_dbl(q_sub(S, X3)), q_sel<Q1>(y, s)));
  // 2 M (S - X3), V^2, -, ZZZ3
  return q_sel<Q0>(X3, q_sel<Q1>(q_sub(q_bcast<0>(r3), r3), q_sel<Q2>(r2, r3)));
}

// + the affine (x2, w2 = 2 y2), given on lanes 2 and 3 of e: P = x2 ZZ - X, r = w2 ZZZ - W, then, all
// scaled by 2: J = 4 P^3, Q = 4 X P^2, X3 = r^2 - J - 2Q, W3 = 2 (r (Q - X3) - W J), ZZ3 = 4 ZZ P^2,
// ZZZ3 = 2 ZZZ J. exc is set (on every lane of the quad's lane 0) when P == 0.
template <class C>
DEV qfe q_smadd(const qfe& s, const qfe& e, bool& exc) {
  typedef typename C::Fp F;
  const qfe r1 = q_mul<F>(e, s);                                 // -, -, x2 ZZ, w2 ZZZ
  const qfe d = q_carry(q_sub(q_perm<2, 3, 2, 3>(r1), s));       // P, r, -, -
  const qfe r2 = q_sqr<F>(d);                                    // P^2, r^2
#if defined(__HIP_DEVICE_COMPILE__)
  exc = exc || (s_sqr_maybe_zero<F, 1>(r2) && q_lane() == 0);
#else
  exc = exc || s_sqr_maybe_zero<F, 1>(r2.l[0]);
#endif
  const qfe r3 = q_mul<F, 2>(q_dbl(q_bcast<0>(r2)), q_sel<Q1>(q_bcast<0>(d), s));  // Q, J, ZZ3, -
  const qfe J = q_bcast<1>(r3), Q = q_bcast<0>(r3);
  const qfe X3 = q_fold<F>(q_carry(q_sub(q_sub(q_sub(q_bcast<1>(r2), J), Q), Q)));
  const qfe r4 = q_mul<F, 2>(q_sel<Q0>(q_bcast<1>(d), J), q_sel<Q0>(q_sub(r3, X3), s));
  // 2 r (Q - X3), 2 W J, -, ZZZ3
  return q_sel<Q0>(X3, q_sel<Q1>(q_sub(q_bcast<0>(r4), r4), q_sel<Q2>(r3, r4)));
}

// ---- Edwards (a = -1): lanes X, Y, Z, T, normalised ----
DEV qfe q_edbl(const qfe& s) {
  const qfe r1 = q_mul<Fe>(q_sel<Q3>(q_bcast<0>(s), s), q_sel<Q3>(q_bcast<1>(s), s));  // XX, YY, ZZ, XY
  const qfe a = q_bcast<0>(r1), b = q_bcast<1>(r1);
  const qfe g = q_add(b, a), h = q_sub(b, a);
  const qfe tc = q_sub(q_dbl(q_bcast<2>(r1)), h);
  const qfe e = q_dbl(q_bcast<3>(r1));
  return q_mul<Fe>(q_sel<Q0 | Q3>(e, q_sel<Q1>(g, h)), q_carry(q_sel<Q0 | Q2>(tc, q_sel<Q1>(h, g))));
}

// + the point given as lanes Y - X, Y + X, Z, 2dT of c
DEV qfe q_eadd(const qfe& s, const qfe& c) {
  // Y - X, Y + X, Z, T
  const qfe a = q_add(q_keep<Q0 | Q1>(q_perm<1, 0, 2, 3>(s)), q_neg<Q0>(s));
  const qfe r1 = q_mul<Fe>(a, c);
  const qfe mm = q_bcast<0>(r1), pp = q_bcast<1>(r1), zz = q_dbl(q_bcast<2>(r1)), tt = q_bcast<3>(r1);
  const qfe e = q_sub(pp, mm), g = q_add(pp, mm), h = q_add(zz, tt), tc = q_sub(zz, tt);
  return q_mul<Fe>(q_sel<Q0 | Q3>(e, q_sel<Q1>(g, h)), q_carry(q_sel<Q0 | Q2>(tc, q_sel<Q1>(h, g))));
}

#undef Q_EACH
#undef Q_AT

}  // namespace sigops
