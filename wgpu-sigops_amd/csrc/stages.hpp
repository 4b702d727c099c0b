// stages.hpp -- the stages of a large secp call, whose inversions are shared between items.
//
// A recovery inverts r modulo n and the result's Z modulo p, 20,000 VALU instructions each, of about
// 400,000 for the item. Both are shared: a lane of the stages before and after the ladder takes
// every lanes-th item, inverts the product of their values once and multiplies back (Montgomery's
// trick: 3 products of 170-220 instructions per item). The stages pass 64 and 112 bytes per item
// through the Scratch: put<N>(p, words), get<N, A = 0>(p, words), N 16-byte chunks of position p.
// Host builds (tests) provide uint4 and make_uint4.
#pragma once
#include "secp.hpp"

namespace sigops {

constexpr u32 STAGE_LANES = 65536;  // lanes of those stages: one wavefront per SIMD

// u1, u2 of the positions first, first + step, ... below end. Src: sig(p, words) and digest(p,
// words), sig false where the position holds no item. VERIFY: u1 = z/s, u2 = r/s; else -z/r, s/r.
template <class C, bool VERIFY, class Src, class Scratch>
DEV void secp_scalars_lane(u32 first, u32 step, u32 end, const Src& src, const Scratch& sc) {
  typedef typename C::Fn Fn;
  if (first >= end) return;
  const fe one = fe_from_const(Fn::ONE);
  auto denominator = [&](u32 p, secp_sig& g) {
    u32 sr[16];
    if (!src.sig(p, sr) || secp_decode_sig<C>(sr, g) != ST_OK) return one;
    return to_mont<Fn>(fe_from_words(VERIFY ? g.s : g.r));
  };
  fe run = one;
  u32 p = first;
#pragma unroll 1
  for (;;) {
    u32 w[12];
#pragma unroll
    for (int k = 0; k < NL; k++) w[k] = run.v[k];
    w[9] = w[10] = w[11] = 0;
    sc.template put<3>(p, w);
    secp_sig g;
    run = mont_mul<Fn>(run, denominator(p, g));
    if (end - p <= step) break;
    p += step;
  }
  fe inv = finv<Fn>(run);
#pragma unroll 1
  for (;;) {
    u32 w[16], dr[8];
    sc.template get<3>(p, w);
    fe before;
#pragma unroll
    for (int k = 0; k < NL; k++) before.v[k] = w[k];
    secp_sig g;
    const fe d = denominator(p, g);
    const fe di = mont_mul<Fn>(inv, before);
    inv = mont_mul<Fn>(inv, d);
    if (src.digest(p, dr)) {
      secp_decode_digest<C>(dr, g);
      const fe zd = mont_mul<Fn>(to_mont<Fn>(fe_from_words(g.z)), di);
      const fe u1m = VERIFY ? zd : fneg<Fn>(zd);
      const fe u2m = mont_mul<Fn>(to_mont<Fn>(fe_from_words(VERIFY ? g.r : g.s)), di);
      fe_to_words(from_mont<Fn>(u1m), w);
      fe_to_words(from_mont<Fn>(u2m), w + 8);
      sc.template put<4>(p, w);
    }
    if (p == first) break;
    p -= step;
  }
}

// Q = u1 G + u2 P of position p (u1, u2 from secp_scalars_lane)
template <class C, class Scratch, class Tab, class Comb>
DEV jac secp_point(u32 p, const fe& x, const fe& y, const Scratch& sc, Tab& tab, const Comb& comb, bool& exc) {
  u32 w[16];
  sc.template get<4>(p, w);
  secp_pro pro;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    pro.u1[k] = w[k];
    pro.u2[k] = w[8 + k];
  }
  secp_carriers<C, true>(pro, x, y);
  return secp_ladder_wide<C>(pro, tab, comb, exc);
}

// the recovery at position p up to its Jacobian result, left in the scratch with the status
template <class C, class Scratch, class Tab, class Comb>
DEV u32 secp_recover_point(const u32 sr[16], u32 p, const Scratch& sc, Tab& tab, const Comb& comb) {
  secp_sig g;
  u32 st = secp_decode_sig<C>(sr, g);
  u32 w[28];  // without a point only the status is set (secp_finish_lane)
  if (st == ST_OK) {
    fe x, y;
    if (!secp_lift<C>(g.r, g.y_odd, x, y)) st = ST_NO_POINT;
    if (st == ST_OK) {
      bool exc = false;
      const jac Q = secp_point<C>(p, x, y, sc, tab, comb, exc);
      if (exc) st = ST_PENDING;
#pragma unroll
      for (int k = 0; k < NL; k++) {
        w[k] = Q.X.v[k]; w[9 + k] = Q.Y.v[k]; w[18 + k] = Q.Z.v[k];
      }
    }
  }
  w[27] = st;
  sc.template put<7>(p, w);
  return st;
}

// affine keys of the positions first, first + step, ... below end, from the scratch. Dst: out(p),
// the item's 64 output bytes (null where the position holds no item; they carry the running products
// in between), and status(p, st).
template <class C, class Dst, class Scratch>
DEV void secp_finish_lane(u32 first, u32 step, u32 end, const Dst& dst, const Scratch& sc) {
  typedef typename C::Fp F;
  if (first >= end) return;
  auto z_of = [&](const u32* w) {
    const fe one = fe_from_const(F::ONE);
    fe z;
#pragma unroll
    for (int k = 0; k < NL; k++) z.v[k] = w[27] == ST_OK ? w[18 + k] : one.v[k];
    return z;
  };
  fe run = fe_from_const(F::ONE);
  u32 p = first;
#pragma unroll 1
  for (;;) {
    uint4* o = dst.out(p);
    if (o) {
      u32 w[28];
      sc.template get<3, 4>(p, w);
      o[0] = make_uint4(run.v[0], run.v[1], run.v[2], run.v[3]);
      o[1] = make_uint4(run.v[4], run.v[5], run.v[6], run.v[7]);
      o[2] = make_uint4(run.v[8], 0, 0, 0);
      run = mont_mul<F>(run, z_of(w));
    }
    if (end - p <= step) break;
    p += step;
  }
  fe inv = finv<F>(run);
#pragma unroll 1
  for (;;) {
    uint4* o = dst.out(p);
    if (o) {
      u32 w[28], res[16];
      sc.template get<7>(p, w);
      fe before;
      const uint4 b0 = o[0], b1 = o[1], b2 = o[2];
      before.v[0] = b0.x; before.v[1] = b0.y; before.v[2] = b0.z; before.v[3] = b0.w;
      before.v[4] = b1.x; before.v[5] = b1.y; before.v[6] = b1.z; before.v[7] = b1.w;
      before.v[8] = b2.x;
      const fe zi = mont_mul<F>(inv, before);
      inv = mont_mul<F>(inv, z_of(w));
      const u32 keep = lane_mask(w[27] == ST_OK);
      fe X, Y;
#pragma unroll
      for (int k = 0; k < NL; k++) { X.v[k] = w[k] & keep; Y.v[k] = w[9 + k] & keep; }
      secp_store_affine<C>(X, Y, zi, res);
#pragma unroll
      for (int c = 0; c < 4; c++)
        o[c] = make_uint4(res[4 * c] & keep, res[4 * c + 1] & keep, res[4 * c + 2] & keep, res[4 * c + 3] & keep);
      dst.status(p, w[27]);
    }
    if (p == first) break;
    p -= step;
  }
}

}  // namespace sigops
