// ed25519.hpp -- Ed25519 verification with ed25519-dalek `VerifyingKey::verify` semantics, one
// signature per lane.
//
// Reference flow: src/wgsl/ed25519_eddsa.wgsl:6-63 (-A, [s]B + [k](-A)),
// src/wgsl/ed25519_utils.wgsl:27-118 (pow_p58, sqrt_ratio_i, decompression),
// src/wgsl/main/ed25519_eddsa_main_0.wgsl:23-86 (decoding, A.y mod p, preimage) and _5.wgsl:20-46
// (compress and byte-compare with R). Acceptance rules follow dalek (the reference test oracle,
// src/tests/ed25519_eddsa.rs:26) rather than the WGSL, which skips the s < l check (src/wgsl/main/ed25519_eddsa_main_0.wgsl:51-54):
//   s >= l -> reject; A must decompress (y taken mod p, sign bit applied also to x = 0);
//   k = SHA-512(R || A || M) mod l over the given bytes; accept iff compress([s]B - [k]A) == R.
//
// Group law: extended twisted Edwards (a = -1) with the unified formulas of Hisil-Wong-Carter-
// Dawson 2008 in the completed-point form used by curve25519-dalek; they are complete on the
// whole curve (d is a non-square), so torsion components of A need no special handling and there
// is no exceptional path. Scalar multiplication shares one doubling chain (Strauss-Shamir):
//   [s]B: w = 8 signed odd digits over an LDS-staged table of (2j+1)B in affine Niels form;
//   [k](-A): w = 4 signed odd digits over a per-lane table of odd multiples in cached form.
// The kernels run the lattice-reduced form of the final check (a 136-bit chain, same results) with
// [v]B from wide tables (ed_check_lattice_wide), or from 8-bit ones for a caller's table; the
// full-length form is left for challenges without a short pair.
#pragma once
#include "secp.hpp"  // nibble / byte8 helpers and status codes
#include "sha512.hpp"

namespace sigops {

typedef ModPed Fe;
typedef ModL Fl;

struct ext {
  fe X, Y, Z, T;
};
struct cached {  // (Y+X, Y-X, Z, 2d*T)
  fe ypx, ymx, z, t2d;
};

DEV ext ext_identity() {
  ext r;
  r.X = fe_zero();
  r.Y = fe_from_const(Fe::ONE);
  r.Z = r.Y;
  r.T = fe_zero();
  return r;
}

// Group law on lazy field arithmetic (field.hpp). Inputs: coordinates normalised with value < 2M;
// cached ypx / ymx normalised, z and t2d products (t2d possibly a lazy negation [2, 2]).
// Bounds of intermediates as [limb bound in units of 2^29, value bound in units of M]; a product
// needs La*Lb < 7.1 and Va*Vb < 64 (M = 2^255 - 19, R = 2^261).
DEV cached to_cached(const ext& P) {
  cached c;
  c.ypx = fnorm_red<Fe>(fadd_nr(P.Y, P.X));
  c.ymx = fnorm_red<Fe>(fsub_nr<Fe, 3, 1>(P.Y, P.X));  // P.X may be any value < 2M
  c.z = P.Z;
  c.t2d = mont_mul<Fe>(P.T, fe_from_const(ED_D2));
  return c;
}

// completed point (E:G:H:Tc) with x = E/Tc, y = G/H -> extended; each pair product within bounds
DEV ext completed_to_ext(const fe& E, const fe& G, const fe& H, const fe& Tc, bool want_t) {
  ext r;
  r.X = mont_mul<Fe>(E, Tc);
  r.Y = mont_mul<Fe>(G, H);
  r.Z = mont_mul<Fe>(H, Tc);
  r.T = want_t ? mont_mul<Fe>(E, G) : fe_zero();
  return r;
}

// doubling (a = -1); T of the input is not used
DEV ext edbl(const ext& P, bool want_t) {
  const fe XX = mont_sqr<Fe>(P.X);
  const fe YY = mont_sqr<Fe>(P.Y);
  const fe ZZ = mont_sqr<Fe>(P.Z);
  const fe XpY2 = mont_sqr<Fe>(fadd_nr(P.X, P.Y));           // [2, 4]^2
  const fe G = fadd_nr(YY, XX);                               // YY + XX: [2, 2.2]
  const fe H = fsub_nr<Fe, 2, 1>(YY, XX);                     // YY - XX: [3, 3.1]
  const fe E = fnorm_red<Fe>(fsub_nr<Fe, 3, 2>(XpY2, G));     // 2XY
  const fe Tc = fnorm_red<Fe>(fsub_nr<Fe, 2, 1>(fadd_nr(fscale_nr(ZZ, 2), XX), YY));  // 2ZZ - (YY - XX)
  return completed_to_ext(E, G, H, Tc, want_t);               // [1]x[1], [2]x[3], [3]x[1], [1]x[2]
}

DEV ext eadd_cached(const ext& P, const cached& Q, bool want_t) {
  const fe PP = mont_mul<Fe>(fadd_nr(P.Y, P.X), Q.ypx);
  const fe MM = mont_mul<Fe>(fsub_nr<Fe, 3, 1>(P.Y, P.X), Q.ymx);  // P.X: any value < 2M
  const fe TT2d = mont_mul<Fe>(P.T, Q.t2d);
  const fe ZZ2 = mont_mul<Fe>(fscale_nr(P.Z, 2), Q.z);
  const fe E = fnorm_red<Fe>(fsub_nr<Fe, 2, 1>(PP, MM));
  const fe G = fadd_nr(PP, MM);                               // [2, 2.x]
  const fe H = fadd_nr(ZZ2, TT2d);                            // [2, 2.x]
  const fe Tc = fsub_nr<Fe, 2, 1>(ZZ2, TT2d);                 // [3, 3.x]
  return completed_to_ext(E, G, H, Tc, want_t);               // [1]x[3], [2]x[2], [2]x[3], [1]x[2]
}

// affine Niels (y+x, y-x, 2d*x*y); t2d possibly a lazy negation
DEV ext eadd_niels(const ext& P, const fe& ypx, const fe& ymx, const fe& t2d, bool want_t) {
  const fe PP = mont_mul<Fe>(fadd_nr(P.Y, P.X), ypx);
  const fe MM = mont_mul<Fe>(fsub_nr<Fe, 3, 1>(P.Y, P.X), ymx);
  const fe TT2d = mont_mul<Fe>(P.T, t2d);
  const fe ZZ2 = fscale_nr(P.Z, 2);                           // [2, 4]
  const fe E = fnorm_red<Fe>(fsub_nr<Fe, 2, 1>(PP, MM));
  const fe G = fadd_nr(PP, MM);                               // [2, 2.x]
  const fe H = fadd_nr(ZZ2, TT2d);                            // [3, 5.x]
  const fe Tc = fnorm_red<Fe>(fsub_nr<Fe, 2, 1>(ZZ2, TT2d));
  return completed_to_ext(E, G, H, Tc, want_t);               // [1]x[1], [2]x[3], [3]x[1], [1]x[2]
}

// ---- the ladders' group law, on signed arithmetic (sfield.hpp): no folds and no biases; a doubling
// takes 1,070 VALU instructions against edbl's 1,250 ----
struct sext {
  sfe X, Y, Z, T;  // normalised
};
struct scached {  // (Y+X, Y-X, Z, 2d*T); t2d may be negated
  sfe ypx, ymx, z, t2d;
};

DEV sext sext_identity() {
  const sfe zero = s_from(fe_zero()), one = s_from(fe_from_const(Fe::ONE));
  return sext{zero, one, one, zero};
}

DEV sext s_completed(const sfe& E, const sfe& G, const sfe& H, const sfe& Tc, bool want_t) {
  sext r;
  r.X = s_mul<Fe>(E, Tc);
  r.Y = s_mul<Fe>(G, H);
  r.Z = s_mul<Fe>(H, Tc);
  r.T = want_t ? s_mul<Fe>(E, G) : s_from(fe_zero());
  return r;
}

// doubling; E = 2XY as a product
DEV sext sedbl(const sext& P, bool want_t) {
  const sfe XX = s_sqr<Fe>(P.X), YY = s_sqr<Fe>(P.Y), ZZ2 = s_sqr<Fe, 2>(P.Z);
  const sfe H = s_sub(YY, XX);
  return s_completed(s_mul<Fe, 2>(P.X, P.Y), s_add(YY, XX), H, s_sub(ZZ2, H), want_t);
}

DEV sext seadd(const sext& P, const scached& Q, bool want_t) {
  const sfe PP = s_mul<Fe>(s_add(P.Y, P.X), Q.ypx), MM = s_mul<Fe>(s_sub(P.Y, P.X), Q.ymx);
  const sfe TT = s_mul<Fe>(P.T, Q.t2d), ZZ2 = s_mul<Fe, 2>(P.Z, Q.z);
  return s_completed(s_sub(PP, MM), s_add(PP, MM), s_add(ZZ2, TT), s_sub(ZZ2, TT), want_t);
}

// + an affine point given as (y + x)/2, (y - x)/2, d x y (the wide table's entries)
DEV sext seadd_half(const sext& P, const sfe& ypx, const sfe& ymx, const sfe& td, bool want_t) {
  const sfe PP = s_mul<Fe>(s_add(P.Y, P.X), ypx), MM = s_mul<Fe>(s_sub(P.Y, P.X), ymx);
  const sfe TT = s_mul<Fe>(P.T, td);
  return s_completed(s_sub(PP, MM), s_add(PP, MM), s_add(P.Z, TT), s_sub(P.Z, TT), want_t);
}

// + an affine point given as y + x, y - x, 2dxy
DEV sext seadd_niels(const sext& P, const sfe& ypx, const sfe& ymx, const sfe& t2d, bool want_t) {
  const sfe PP = s_mul<Fe>(s_add(P.Y, P.X), ypx), MM = s_mul<Fe>(s_sub(P.Y, P.X), ymx);
  const sfe TT = s_mul<Fe>(P.T, t2d), ZZ2 = s_carry(s_dbl(P.Z));
  return s_completed(s_sub(PP, MM), s_add(PP, MM), s_add(ZZ2, TT), s_sub(ZZ2, TT), want_t);
}

DEV scached s_to_cached(const sext& P) {
  scached c;
  c.ypx = s_carry(s_add(P.Y, P.X));
  c.ymx = s_carry(s_sub(P.Y, P.X));
  c.z = P.Z;
  c.t2d = s_mul<Fe>(P.T, s_from(fe_from_const(ED_D2)));
  return c;
}
DEV cached s_raw(const scached& c) { return cached{s_raw(c.ypx), s_raw(c.ymx), s_raw(c.z), s_raw(c.t2d)}; }

// a table entry as stored, or its negative: Y+X and Y-X swapped, 2dT negated
DEV scached s_entry(const cached& c, bool neg) {
  const u32 m = lane_mask(neg);
  const sfe a = s_unraw<Fe>(c.ypx), b = s_unraw<Fe>(c.ymx);
  return scached{s_sel(m, b, a), s_sel(m, a, b), s_unraw<Fe>(c.z), s_neg_if(neg, s_unraw<Fe>(c.t2d))};
}

// dalek FieldElement::sqrt_ratio_i (field.rs): returns was_nonzero_square, r = nonnegative root
DEV bool sqrt_ratio_i(const fe& u, const fe& v, fe& r_out) {
  const fe v3 = mont_mul<Fe>(mont_sqr<Fe>(v), v);
  const fe v7 = mont_mul<Fe>(mont_sqr<Fe>(v3), v);
  fe r = mont_mul<Fe>(mont_mul<Fe>(u, v3), s_to_fe<Fe, 1>(s_pow_chain<Fe, CH_ED_P58>(s_from(mont_mul<Fe>(u, v7)))));
  const fe check = mont_mul<Fe>(v, mont_sqr<Fe>(r));
  const fe i = fe_from_const(ED_SQRTM1);
  const fe neg_u = fneg<Fe>(u);
  const bool correct = feq<Fe>(check, u);
  const bool flipped = feq<Fe>(check, neg_u);
  const bool flipped_i = feq<Fe>(check, mont_mul<Fe>(neg_u, i));
  const fe r_prime = mont_mul<Fe>(i, r);
  r = fsel(flipped || flipped_i, r_prime, r);
  const bool r_neg = (from_mont<Fe>(r).v[0] & 1u) != 0;
  r = fsel(r_neg, fneg<Fe>(r), r);
  r_out = r;
  return correct || flipped;
}

// ED_BAD_R and ED_SMALL_ORDER come from verify_strict only
enum : u32 { ED_OK = 0, ED_BAD_S = 1, ED_BAD_KEY = 2, ED_MISMATCH = 3, ED_BAD_R = 4, ED_SMALL_ORDER = 5 };

// dalek CompressedEdwardsY::decompress: y = the 255 low bits taken mod p (non-canonical y is
// accepted), x = sqrt_ratio_i(y^2 - 1, d y^2 + 1), negated when the sign bit is set (also for
// x = 0). enc: 8 raw little-endian words. Returns false if there is no such x.
DEV bool ed_decompress(const u32 enc[8], fe& x, fe& y) {
  u32 yw[8];
#pragma unroll
  for (int i = 0; i < 8; i++) yw[i] = enc[i];
  const bool x_sign = (yw[7] >> 31) != 0;
  yw[7] &= 0x7fffffffu;
  if (!words_lt(yw, ED_P32)) {
    u32 t[8];
    words_sub(yw, ED_P32, t);
#pragma unroll
    for (int i = 0; i < 8; i++) yw[i] = t[i];
  }
  y = to_mont<Fe>(fe_from_words(yw));
  const fe one = fe_from_const(Fe::ONE);
  const fe yy = mont_sqr<Fe>(y);
  const fe u = fsub<Fe>(yy, one);
  const fe v = fadd<Fe>(mont_mul<Fe>(yy, fe_from_const(ED_D)), one);
  const bool ok = sqrt_ratio_i(u, v, x);
  if (x_sign) x = fneg<Fe>(x);
  return ok;
}

// dalek EdwardsPoint::is_small_order: [8]P is the identity (X = 0 and Y = Z after three doublings)
DEV bool ed_small_order(const fe& x, const fe& y) {
  ext P;
  P.X = x;
  P.Y = y;
  P.Z = fe_from_const(Fe::ONE);
  P.T = fe_zero();  // doubling does not read T
#pragma unroll 1
  for (int i = 0; i < 3; i++) P = edbl(P, false);
  return fis_zero<Fe>(P.X) && feq<Fe>(P.Y, P.Z);
}

// k = the 512-bit little-endian digest h (16 words) mod l, as 8 little-endian words
DEV void ed25519_k_from_digest(const u32 h[16], u32 k[8]) {
  const fe hi = mont_mul<Fl>(fe_from_words(h + 8), fe_from_const(L_C256));
  const fe lo = mont_mul<Fl>(fe_from_words(h), fe_from_const(L_C0));
  fe_to_words(fcanon<Fl>(fadd<Fl>(hi, lo)), k);
}

// sig_raw: 16 raw words (R || s); pk_raw: 8 raw words; message in mem at msg_off, len bytes.
// k = SHA-512(R || A || M) mod l as 8 little-endian words
template <class Mem>
DEV void ed25519_challenge(const u32 sig_raw[16], const u32 pk_raw[8], const Mem& mem, u64 msg_off, u32 len,
                           u32 k[8]) {
  u32 hdr[16], h[16];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    hdr[i] = sig_raw[i];
    hdr[8 + i] = pk_raw[i];
  }
  sha512_ed(hdr, mem, msg_off, len, h);
  ed25519_k_from_digest(h, k);
}

// verify_strict's extra rules (dalek VerifyingKey::verify_strict): R must decompress and neither R
// nor A may have small order. The rules on R are evaluated in a pass of their own between the hash
// and the verifier (registers to spare): this returns ED_OK, ED_BAD_R or ED_SMALL_ORDER, which
// travels to the verifier in bits 29..31 of the challenge's top word (k < l < 2^253 leaves those
// bits zero). The rule on A runs in the verifier, which decompresses A anyway.
DEV u32 ed25519_strict_r_checks(const u32 sig_raw[16]) {
  fe rx, ry;
  if (!ed_decompress(sig_raw, rx, ry)) return ED_BAD_R;
  return ed_small_order(rx, ry) ? ED_SMALL_ORDER : ED_OK;
}
constexpr u32 ED_K_STRICT_SHIFT = 29;

// ---- lattice-reduced check (T. Pornin, "Optimized Lattice Basis Reduction In Dimension 2, and
// Fast Schnorr and EdDSA Signature Verification", IACR ePrint 2020/454) ----
// dalek's test compress([s]B - [k]A) == R bytes runs a 253-bit doubling chain. With a pair
// (c0, c1) such that c0 = c1 k (mod 8l), c1 odd and |c0|, c1 < 2^136, the check becomes
//     [c1 s mod l] B - [c0] A - [c1] R == identity
// over a 136-bit chain, with R decoded from its bytes. The left side is [c1]([s]B - [k]A - R):
// [c1 k] A = [c0] A since the order of A divides 8l, and [c1 s] B = [c1 s mod l] B since B has
// order l. c1 is odd and below l, so it is prime to every order in the group, and the point is the
// identity exactly when [s]B - [k]A == R. R must decode canonically (y < p, and no sign bit on
// x = 0): compress never produces another encoding, so dalek rejects those bytes, and so does this
// check. The high half of c1 s mod l runs on its own table of odd multiples of [2^136] B.
constexpr int ED_LAT_BITS = SIGOPS_ED_LAT_BITS;
static_assert(ED_LAT_BITS == 136, "carriers, windows and the split of c1 s assume 136 bits");
constexpr int ED_LAT_MAX_STEPS = 320;  // Euclid steps from 2^255 to 2^128: at most 183, plus corrections
constexpr u32 ED_BTAB_HI = 1u << (SIGOPS_WG - 1);  // index of (2j+1) [2^136] B is ED_BTAB_HI + j

#if defined(SIGOPS_HOST_CHECK) && SIGOPS_HOST_CHECK && !defined(__HIP_DEVICE_COMPILE__)
// host check build only: send every item through the full-length check
inline bool& ed_force_full() {
  static bool f = false;
  return f;
}
#endif

// R decoded as compress() could have produced it: y < p and no sign bit on x = 0
DEV bool ed_decode_canonical(const u32 enc[8], fe& x, fe& y) {
  u32 yw[8];
#pragma unroll
  for (int i = 0; i < 8; i++) yw[i] = enc[i];
  yw[7] &= 0x7fffffffu;
  const bool canon = words_lt(yw, ED_P32);
  const bool ok = ed_decompress(enc, x, y);
  return ok && canon && !((enc[7] >> 31) != 0 && fis_zero<Fe>(x));
}

template <int NW>
DEV double words_f64(const u32* w) {  // nearest-ish double of a multi-word value (7 roundings at most)
  double d = (double)w[NW - 1];
#pragma unroll
  for (int i = NW - 2; i >= 0; i--) d = d * 4294967296.0 + (double)w[i];
  return d;
}

// r = a - q b over N words (a, b unsigned or two's complement); returns the high part that the
// product and the borrow left above the top word (0 when a - q b is in [0, 2^(32N)))
template <int N>
DEV u64 words_submul(const u32* a, const u32* b, u32 q, u32* r) {
  u32 hi = 0, br = 0;
#pragma unroll
  for (int i = 0; i < N; i++) {
    const u64 p = (u64)q * b[i] + hi;
    hi = (u32)(p >> 32);
    const u64 d = (u64)a[i] - (u32)p - br;
    r[i] = (u32)d;
    br = (u32)(d >> 63);
  }
  return (u64)hi + br;
}

template <int N>
DEV void words_neg_if(bool c, u32* w) {  // two's complement negation when c
  const u32 m = lane_mask(c);
  u32 cy = c ? 1u : 0u;
#pragma unroll
  for (int i = 0; i < N; i++) {
    const u64 x = (u64)(w[i] ^ m) + cy;
    w[i] = (u32)x;
    cy = (u32)(x >> 32);
  }
}

// (c0, c1) from Euclid's remainder sequence on (8l, k). Every remainder is r_j = t_j k (mod 8l); the
// first one below 2^128 has |t_j| <= 8l / r_(j-1) < 2^127. When t_j is even, t_(j-1) is odd (two
// consecutive t are coprime) and the pair is (r_(j-1) - m r_j, t_(j-1) - m t_j) with the m that
// balances the two coordinates. Quotients come from double-precision estimates (relative error
// below 2^-49, so off by at most one below 2^32), corrected exactly: one too large is undone, one
// too small leaves a remainder >= b for the next step. Every update is exact integer arithmetic,
// so c0 = c1 k (mod 8l) holds whatever the estimates, and the bounds are checked at the end.
// Returns false when no pair within 2^136 was found (about 3 in 10^6 random k) or a quotient
// reached 2^32 (about 2 in 10^8); the caller then runs the full-length check. c0 >= 0 comes out
// with its sign apart (c0_neg), c1 > 0.
DEV bool ed_lattice(const u32 k[8], u32 c0[5], u32 c1[5], bool& c0_neg) {
  u32 a[8], b[8], ta[5], tb[5];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    a[i] = (ED_L32[i] << 3) | (i > 0 ? ED_L32[i - 1] >> 29 : 0u);  // 8l < 2^256
    b[i] = k[i];
  }
#pragma unroll
  for (int i = 0; i < 5; i++) {
    ta[i] = 0;
    tb[i] = i == 0 ? 1u : 0u;
  }
  bool ok = true;
  int steps = 0;
#pragma unroll 1
  while ((b[4] | b[5] | b[6] | b[7]) != 0) {  // a >= b >= 2^128 here
    if (++steps > ED_LAT_MAX_STEPS) {
      ok = false;
      break;
    }
    const double qd = __builtin_floor(words_f64<8>(a) / words_f64<8>(b));
    if (!(qd < 4294967295.0)) {  // a quotient of 2^32 or more (about 2^-32 per step for random k)
      ok = false;
      break;
    }
    u32 q = qd > 1.0 ? (u32)qd : 1u;
    u32 r[8];
    const u64 over = words_submul<8>(a, b, q, r);
    if (over != 0) {  // q was one too large: add b back, which must bring the value to [0, 2^256)
      const u32 cy = words_add(r, b, r);
      q -= 1;
      if ((u64)cy != over) {
        ok = false;
        break;
      }
    }
    u32 tr[5];
    words_submul<5>(ta, tb, q, tr);  // |t| < 2^128 throughout: no overflow of 160 bits
    const bool lt = words_lt(r, b);  // a full step (else a partial one: a <- r)
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const u32 nb = lt ? r[i] : b[i];
      a[i] = lt ? b[i] : r[i];
      b[i] = nb;
    }
#pragma unroll
    for (int i = 0; i < 5; i++) {
      const u32 nt = lt ? tr[i] : tb[i];
      ta[i] = lt ? tb[i] : tr[i];
      tb[i] = nt;
    }
  }
#if defined(SIGOPS_HOST_CHECK) && SIGOPS_HOST_CHECK && !defined(__HIP_DEVICE_COMPILE__)
  if (ed_force_full()) ok = false;
#endif
  u32 w0[8];
  if (tb[0] & 1u) {
#pragma unroll
    for (int i = 0; i < 8; i++) w0[i] = b[i];
#pragma unroll
    for (int i = 0; i < 5; i++) c1[i] = tb[i];
  } else {
    u32 ua[5], ub[5];
#pragma unroll
    for (int i = 0; i < 5; i++) {
      ua[i] = ta[i];
      ub[i] = tb[i];
    }
    words_neg_if<5>((ta[4] >> 31) != 0, ua);
    words_neg_if<5>((tb[4] >> 31) != 0, ub);
    const double md = __builtin_floor((words_f64<8>(a) - words_f64<5>(ua)) / (words_f64<8>(b) + words_f64<5>(ub)));
    if (!(md < 4294967296.0)) ok = false;
    const u32 m = (ok && md > 0.0) ? (u32)md : 0u;
    if (words_submul<8>(a, b, m, w0) != 0) ok = false;  // m above the quotient a / b
    words_submul<5>(ta, tb, m, c1);  // |c1| < 2^160; a wrapped value fails the bound below
  }
  c0_neg = (c1[4] >> 31) != 0;
  words_neg_if<5>(c0_neg, c1);
#pragma unroll
  for (int i = 0; i < 5; i++) c0[i] = w0[i];
  const u32 hi0 = w0[5] | w0[6] | w0[7] | (w0[4] >> (ED_LAT_BITS - 128));
  return ok && hi0 == 0 && (c1[4] >> (ED_LAT_BITS - 128)) == 0;
}

// table of the odd multiples (2e+1) P, e = 0..7, of P = (x, y) in cached form (raw signed limbs) at
// entries e0..e0+7
template <class Tab>
DEV void ed_table_odd(Tab& tab, int e0, const fe& x, const fe& y) {
  sext P;
  P.X = s_from(x);
  P.Y = s_from(y);
  P.Z = s_from(fe_from_const(Fe::ONE));
  P.T = s_mul<Fe>(P.X, P.Y);
  const scached P2 = s_to_cached(sedbl(P, true));
  sext T = P;
  tab.store(e0, s_raw(s_to_cached(P)));
#pragma unroll 1
  for (int e = 1; e < 8; e++) {
    T = seadd(T, P2, true);
    tab.store(e0 + e, s_raw(s_to_cached(T)));
  }
}

// acc + (digit's odd multiple of the table's point, negated per digit and stream sign); the table
// holds (2j+1) B at entries base + j in affine Niels form
template <class BTab>
DEV sext ed_add_b(const sext& acc, const BTab& bt, u32 base, u32 digit, bool neg_stream, bool want_t) {
  const bool neg = (digit < 128) != neg_stream;
  fe ypx, ymx, t2d;
  bt.load(base + (((digit < 128) ? ~digit : digit) & 127u), ypx, ymx, t2d);
  const u32 m = lane_mask(neg);
  const sfe a = s_from(ypx), b = s_from(ymx);
  return seadd_niels(acc, s_sel(m, b, a), s_sel(m, a, b), s_neg_if(neg, s_from(t2d)), want_t);
}

// the cached identity (Y+X, Y-X, Z, 2dT) = (1, 1, 1, 0), or entry e of the table when use
template <class Tab>
DEV scached ed_entry_or_identity(const Tab& tab, u32 e, bool neg, bool use) {
  const scached c = s_entry(tab.load(e), neg);
  const u32 m = lane_mask(use);
  const sfe one = s_from(fe_from_const(Fe::ONE));
  return scached{s_sel(m, c.ypx, one), s_sel(m, c.ymx, one), s_sel(m, c.z, one), s_sel(m, c.t2d, s_from(fe_zero()))};
}

// the wide table's entry (ed_comb): (y + x)/2, (y - x)/2, dxy as 8 little-endian words each,
// canonical Montgomery form
struct ed_comb_entry {
  u32 v[24];
};

// acc + [v]B from the wide table: the 16 digits of the carrier c of an odd v (b_neg: negated). Comb:
// load(i, j, entry&) for the odd multiple (2j + 1) 2^(16 i) B.
template <class Comb>
DEV sext ed_comb(sext acc, const u32 c[8], bool b_neg, const Comb& comb) {
  auto digit = [&](int i) { return (c[i >> 1] >> ((i & 1) * 16)) & 0xFFFFu; };
  auto load = [&](int i, ed_comb_entry& e) {
    const u32 d = digit(i);
    comb.load(i, ((d < COMB_ENTRIES) ? ~d : d) & (COMB_ENTRIES - 1u), e);
  };
  ed_comb_entry e;
  load(0, e);
#pragma unroll 1
  for (int i = 0; i < COMB_WINDOWS; i++) {
    const bool neg = (digit(i) < COMB_ENTRIES) != b_neg;
    const u32 m = lane_mask(neg);
    const sfe a = s_from(fe_from_words(e.v)), b = s_from(fe_from_words(e.v + 8)), t = s_from(fe_from_words(e.v + 16));
    if (i + 1 < COMB_WINDOWS) load(i + 1, e);
    acc = seadd_half(acc, s_sel(m, b, a), s_sel(m, a, b), s_neg_if(neg, t), i + 1 < COMB_WINDOWS);
  }
  return acc;
}

// the scalars of the lattice-reduced check, as digit carriers of odd values: c0 and c1 (136 bits), and
// v = c1 s mod l
struct ed_lat {
  u32 ca[5], cr[5];
  u32 v[8];              // v, or l - v when v is even
  bool a_neg, a_fix;     // c0 is negative; |c0| was even and one was added
  bool b_neg;            // v was even
};

// false when k has no short pair (the full-length check then decides)
DEV bool ed_lat_scalars(const u32 k[8], const u32 s[8], ed_lat& o) {
  u32 c0[5], c1[5];
  o.a_neg = false;
  const bool ok = ed_lattice(k, c0, c1, o.a_neg);
  u32 cw[8], t[8];
#pragma unroll
  for (int i = 0; i < 8; i++) cw[i] = i < 5 ? c1[i] : 0u;
  fe_to_words(fcanon<Fl>(to_mont<Fl>(mont_mul<Fl>(fe_from_words(cw), fe_from_words(s)))), o.v);
  o.b_neg = (o.v[0] & 1u) == 0;
  words_sub(ED_L32, o.v, t);
#pragma unroll
  for (int i = 0; i < 8; i++) o.v[i] = o.b_neg ? t[i] : o.v[i];
  o.a_fix = (c0[0] & 1u) == 0;
  c0[0] |= 1u;
  glv_carrier<ED_LAT_BITS>(c0, o.ca);
  glv_carrier<ED_LAT_BITS>(c1, o.cr);
  return ok;
}
// carrier of the odd v < 2^253 over 256 bits, for ed_comb
DEV void ed_v_carrier(const u32 v[8], u32 c[8]) {
#pragma unroll
  for (int i = 0; i < 8; i++) c[i] = (v[i] >> 1) | (i < 7 ? v[i + 1] << 31 : 0x80000000u);
}

// One 136-bit chain: [c0](-A) + [c1](-R), the A digits at tab's entries 0..7 and the R digits at 8..15,
// four doublings and one addition of each per 4-bit window; add_b(acc, i) adds what belongs to an
// even window i (the B digits of the 8-bit tables, or nothing).
template <class Tab, class AddB>
DEV sext ed_lat_ladder(const ed_lat& o, const Tab& tab, const AddB& add_b) {
  constexpr int W = ED_LAT_BITS / 4;
  // top windows: the digits are positive; the A stream's sign applies
  sext acc = seadd(sext_identity(), s_entry(tab.load(nibble(o.ca, W - 1) - 8), o.a_neg), true);
  acc = seadd(acc, s_entry(tab.load(8 + nibble(o.cr, W - 1) - 8), false), false);
#pragma unroll 1
  for (int i = W - 2; i >= 0; i--) {
    const u32 da = nibble(o.ca, i), dr = nibble(o.cr, i);
    const cached ea = tab.load((da < 8 ? ~da : da) & 7u);
#pragma unroll 1
    for (int d = 0; d < 4; d++) acc = sedbl(acc, d == 3);  // T is needed only by an addition that follows
    const cached er = tab.load(8 + ((dr < 8 ? ~dr : dr) & 7u));
    acc = seadd(acc, s_entry(ea, (da < 8) != o.a_neg), true);
    acc = add_b(seadd(acc, s_entry(er, dr < 8), (i & 1) == 0), i);
  }
  return acc;
}

// X == 0 and Y == Z
DEV bool s_is_identity(const sext& P) {
  return fis_zero<Fe>(s_to_fe<Fe, 8>(P.X)) && fis_zero<Fe>(s_to_fe<Fe, 8>(s_carry(s_sub(P.Y, P.Z))));
}

// the 136-bit check with 8-bit windows of B: [v0](+-B) + [v1](+-[2^136]B) + [a](+-(-A)) + [c1](-R) (-
// the +-(-A) that made an even |c0| odd) == identity
template <class Tab, class BTab>
DEV bool ed_check_lattice(const ed_lat& o, const Tab& tab, const BTab& bt) {
  // v split at bit 136; an even high half takes one more: v = (v_lo - 2^136) + 2^136 (v_hi + 1), the
  // low stream then negated
  const u32(&v)[8] = o.v;
  u32 lo[5] = {v[0], v[1], v[2], v[3], v[4] & 0xffu};
  u32 hi[5] = {(v[4] >> 8) | (v[5] << 24), (v[5] >> 8) | (v[6] << 24), (v[6] >> 8) | (v[7] << 24), v[7] >> 8, 0u};
  const bool hi_even = (hi[0] & 1u) == 0;
  hi[0] |= 1u;
  const u32 top[5] = {0, 0, 0, 0, 1u << (ED_LAT_BITS - 128)};
  u32 t[5], br = 0;
#pragma unroll
  for (int i = 0; i < 5; i++) {
    const u64 d = (u64)top[i] - lo[i] - br;
    t[i] = (u32)d;
    br = (u32)(d >> 63);
  }
#pragma unroll
  for (int i = 0; i < 5; i++) lo[i] = hi_even ? t[i] : lo[i];
  u32 cb0[5], cb1[5];
  glv_carrier<ED_LAT_BITS>(lo, cb0);
  glv_carrier<ED_LAT_BITS>(hi, cb1);
  const bool b0_neg = o.b_neg != hi_even, b1_neg = o.b_neg;
  sext acc = ed_lat_ladder(o, tab, [&](const sext& a, int i) {
    if (i & 1) return a;
    const sext b = ed_add_b(a, bt, 0, byte8(cb0, i >> 1), b0_neg, true);
    return ed_add_b(b, bt, ED_BTAB_HI, byte8(cb1, i >> 1), b1_neg, i == 0);
  });
  // the A stream ran on |c0| + 1 when |c0| was even: take its point off once
  return s_is_identity(seadd(acc, ed_entry_or_identity(tab, 0, !o.a_neg, o.a_fix), false));
}

// the same with [v]B from the wide table
template <class Tab, class Comb>
DEV bool ed_check_lattice_wide(const ed_lat& o, const Tab& tab, const Comb& comb) {
  u32 c[8];
  ed_v_carrier(o.v, c);
  sext acc = ed_lat_ladder(o, tab, [](const sext& a, int) { return a; });
  acc = seadd(acc, ed_entry_or_identity(tab, 0, !o.a_neg, o.a_fix), true);
  return s_is_identity(ed_comb(acc, c, o.b_neg, comb));
}

// the full-length check: compress([s]B + [k](-A)) == R bytes, tab entries 0..7 = -A's odd multiples
template <class Tab, class BTab>
DEV bool ed_check_full(const u32 s[8], const u32 k[8], const u32 sig_raw[16], const Tab& tab, const BTab& bt) {
  // odd representatives: s even -> l - s with B negated; k even -> k + 1 and a final +A
  const bool b_neg = (s[0] & 1u) == 0;
  const bool k_even = (k[0] & 1u) == 0;
  u32 s1[8], k1[8];
  {
    u32 t[8];
    words_sub(ED_L32, s, t);  // only used when s < l (else the result is discarded)
    u32 c = k_even ? 1u : 0u;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      s1[i] = b_neg ? t[i] : s[i];
      const u64 kk = (u64)k[i] + c;
      k1[i] = (u32)kk;
      c = (u32)(kk >> 32);
    }
  }
  u32 c1[8], c2[8];
  ed_v_carrier(s1, c1);
  ed_v_carrier(k1, c2);
  sext acc = seadd(sext_identity(), s_entry(tab.load(nibble(c2, 63) - 8), false), true);
#pragma unroll 1
  for (int i = 62; i >= 0; i--) {
    const u32 c = nibble(c2, i);
    const cached E = tab.load((c < 8 ? ~c : c) & 7u);
#pragma unroll 1
    for (int d = 0; d < 4; d++) acc = sedbl(acc, d == 3);
    acc = seadd(acc, s_entry(E, c < 8), (i & 1) == 0);
    if ((i & 1) == 0) acc = ed_add_b(acc, bt, 0, byte8(c1, i >> 1), b_neg, i == 0);
  }
  // + A when k was made odd by adding one, else + identity (complete formulas)
  acc = seadd(acc, ed_entry_or_identity(tab, 0, true, k_even), false);
  // compress and compare with R
  const fe zi = finv<Fe>(s_to_fe<Fe, 8>(acc.Z));
  const fe xa = from_mont<Fe>(mont_mul<Fe>(s_to_fe<Fe, 8>(acc.X), zi));
  const fe ya = from_mont<Fe>(mont_mul<Fe>(s_to_fe<Fe, 8>(acc.Y), zi));
  u32 enc[8];
  fe_to_words(ya, enc);
  enc[7] ^= (xa.v[0] & 1u) << 31;
  u32 diff = 0;
#pragma unroll
  for (int i = 0; i < 8; i++) diff |= enc[i] ^ sig_raw[i];
  return diff == 0;
}

// Verification given the challenge k (from ed25519_challenge). lattice(k, s, tab): the lattice-reduced
// check on tab's entries 0..7 (-A) and 8..15 (-R), or false in `found` when k has no short pair.
// STRICT: dalek VerifyingKey::verify_strict; the status of its rules on R arrives in the top bits
// of k (ed25519_strict_r_checks) and A's small order is checked here.
template <bool STRICT, class Tab, class BTab, class Lattice>
DEV u32 ed25519_verify_with(const u32 sig_raw[16], const u32 pk_raw[8], const u32 k_in[8], Tab& tab, const BTab& bt,
                            const Lattice& lattice) {
  u32 k[8];
#pragma unroll
  for (int i = 0; i < 8; i++) k[i] = k_in[i];
  u32 strict_status = ED_OK;
  if constexpr (STRICT) {
    strict_status = k[7] >> ED_K_STRICT_SHIFT;
    k[7] &= (1u << ED_K_STRICT_SHIFT) - 1u;
  }
  u32 status = ED_OK;
  // s (little-endian bytes = little-endian words)
  u32 s[8];
#pragma unroll
  for (int i = 0; i < 8; i++) s[i] = sig_raw[8 + i];
  if (!words_lt(s, ED_L32)) status = ED_BAD_S;
  fe x, y;
  const bool ok = ed_decompress(pk_raw, x, y);
  if (!ok && status == ED_OK) status = ED_BAD_KEY;
  if (STRICT && status == ED_OK) status = strict_status;
  // verify_strict: A of small order (checked after R's rules, as dalek checks R first)
  if (STRICT && status == ED_OK && ed_small_order(x, y)) status = ED_SMALL_ORDER;
  ed_table_odd(tab, 0, fneg<Fe>(x), y);
  bool found = false;
  bool equal = lattice(k, s, found);
  if (!found) equal = ed_check_full(s, k, sig_raw, tab, bt);
  if (status == ED_OK && !equal) status = ED_MISMATCH;
  return status;
}

// R decoded and its table built, then `check` on the scalars
template <class Tab, class Check>
DEV bool ed_with_lattice(const u32 sig_raw[16], const u32 k[8], const u32 s[8], Tab& tab, bool& found,
                         const Check& check) {
  ed_lat o;
  found = ed_lat_scalars(k, s, o);
  if (!found) return false;
  fe rx, ry;
  const bool r_ok = ed_decode_canonical(sig_raw, rx, ry);
  ed_table_odd(tab, 8, fneg<Fe>(rx), ry);
  return check(o) && r_ok;
}

// the same with the resident or a caller's 8-bit table of B.
// LATTICE: the lattice-reduced check (and the full-length one for challenges without a short
// pair); otherwise the full-length check only.
// BTab: load(idx, ypx, ymx, t2d) for (2 idx + 1) B at idx < ED_BTAB_HI and, with LATTICE,
// (2 j + 1) [2^136] B at idx = ED_BTAB_HI + j. Tab: per-lane store(e, cached) / load(e), 8 entries
// (16 with LATTICE).
template <bool STRICT = false, bool LATTICE = false, class Tab, class BTab>
DEV u32 ed25519_verify_core(const u32 sig_raw[16], const u32 pk_raw[8], const u32 k_in[8], Tab& tab,
                            const BTab& bt) {
  return ed25519_verify_with<STRICT>(sig_raw, pk_raw, k_in, tab, bt, [&](const u32* k, const u32* s, bool& found) {
    if constexpr (LATTICE)
      return ed_with_lattice(sig_raw, k, s, tab, found, [&](const ed_lat& o) { return ed_check_lattice(o, tab, bt); });
    else
      return false;
  });
}

// the challenge, with the status of verify_strict's rules on R in its top bits
template <bool STRICT, class Mem>
DEV void ed25519_challenge_strict(const u32 sig_raw[16], const u32 pk_raw[8], const Mem& mem, u64 msg_off, u32 len,
                                  u32 k[8]) {
  ed25519_challenge(sig_raw, pk_raw, mem, msg_off, len, k);
  if constexpr (STRICT) k[7] |= ed25519_strict_r_checks(sig_raw) << ED_K_STRICT_SHIFT;
}

template <bool STRICT = false, bool LATTICE = false, class Tab, class BTab, class Mem>
DEV u32 ed25519_verify_item(const u32 sig_raw[16], const u32 pk_raw[8], const Mem& mem, u64 msg_off, u32 len,
                            Tab& tab, const BTab& bt) {
  u32 k[8];
  ed25519_challenge_strict<STRICT>(sig_raw, pk_raw, mem, msg_off, len, k);
  return ed25519_verify_core<STRICT, LATTICE>(sig_raw, pk_raw, k, tab, bt);
}

// the lattice-reduced check with the wide table of B; bt: the 8-bit table, for the full-length check
template <bool STRICT, class Tab, class BTab, class Comb, class Mem>
DEV u32 ed25519_verify_wide(const u32 sig_raw[16], const u32 pk_raw[8], const Mem& mem, u64 msg_off, u32 len,
                            Tab& tab, const BTab& bt, const Comb& comb) {
  u32 k8[8];
  ed25519_challenge_strict<STRICT>(sig_raw, pk_raw, mem, msg_off, len, k8);
  return ed25519_verify_with<STRICT>(sig_raw, pk_raw, k8, tab, bt, [&](const u32* k, const u32* s, bool& found) {
    return ed_with_lattice(sig_raw, k, s, tab, found,
                           [&](const ed_lat& o) { return ed_check_lattice_wide(o, tab, comb); });
  });
}

}  // namespace sigops
