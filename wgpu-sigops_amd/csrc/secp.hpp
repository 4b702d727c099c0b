// secp.hpp -- secp256k1 / secp256r1 public-key recovery, one signature per lane.
//
// Reference semantics: src/wgsl/secp256k1_ecdsa.wgsl:7-130 and src/wgsl/secp256r1_ecdsa.wgsl:7-130
// (decode, lift R, u1 = -z/r, u2 = s/r, Q = u1*G + u2*R, affine output), with the acceptance rules
// of the reference's CPU path (fuel-crypto over libsecp256k1 / ecdsa 0.16): r, s in [1, n-1],
// z = digest mod n, R must exist, Q != infinity. Errors write 64 zero bytes and a status code.
//
// Algorithm (gfx950-oriented; the reference uses plain double-and-add, src/wgsl/secp256k1_curve.wgsl:277-294,
// and a w=4 fixed-base loop, :388-447, with Strauss-Shamir disabled, :336-383):
//   * one shared doubling chain (Strauss-Shamir) for u1*G + u2*R;
//   * both scalars in the signed all-odd digit form k = sum (2c_i - (2^w-1)) 2^(wi) with
//     C = (k >> 1) | 2^255 for odd k (even k: use n - k and negate the base), so every window
//     performs exactly one addition and no lane ever branches on a zero digit;
//   * u2*R: w = 4, table of odd multiples R..15R in per-lane memory, made affine (secp256k1: up to an
//     isomorphism) so that every addition of the R stream is a mixed addition;
//   * u1*G: 16 additions from wide tables of G after the chain (secp_comb); with a caller's table of
//     G, w = 8 on the chain, odd multiples G..255G staged in LDS by the kernel;
//   * Jacobian formulas dbl-2009-l (a = 0) / dbl-2001-b (a = -3), add-2007-bl, madd-2007-bl.
//     These are incomplete: an addition of P and +-P is detected (H == 0) and the lane is marked
//     for the careful path, which redoes the item with complete, branching formulas.
#pragma once
#include "inv.hpp"
#include "sfield.hpp"

namespace sigops {

enum : u32 {
  ST_OK = 0,
  ST_BAD_R = 1,
  ST_BAD_S = 2,
  ST_NO_POINT = 3,
  ST_INFINITY = 4,    // recovery: Q = infinity; verification: u1 G + u2 Q = infinity
  ST_HIGH_S = 5,      // verification, secp256k1: s > (n-1)/2
  ST_BAD_KEY = 6,     // verification: the key is not a curve point with X, Y < p
  ST_MISMATCH = 7,    // verification: x(u1 G + u2 Q) mod n != r
  ST_PENDING = 0xFF,  // exceptional addition met: the careful path finishes the item
};

struct CurveK1 {
  typedef ModPk1 Fp;
  typedef ModNk1 Fn;
  static constexpr bool A_IS_M3 = false;
  static constexpr bool GLV = true;    // phi(x, y) = (beta x, y) = [lambda](x, y)
  static constexpr bool LOW_S = true;  // verification accepts s <= (n-1)/2 only (libsecp256k1)
  DEV static fe b() { return fe_from_const(K1_B); }
  DEV static const u32 (&n32())[8] { return K1_N32; }
  DEV static const u32 (&p32())[8] { return K1_P32; }
  DEV static const u32 (&pmn32())[8] { return K1_PMN32; }
  DEV static const u32 (&nhalf32())[8] { return K1_NHALF32; }
  typedef CH_K1_SQRT SqrtChain;  // x^((p+1)/4)
};
struct CurveR1 {
  typedef ModPr1 Fp;
  typedef ModNr1 Fn;
  static constexpr bool A_IS_M3 = true;
  static constexpr bool GLV = false;
  static constexpr bool LOW_S = false;  // p256 / ecdsa 0.16 verification accepts either s
  DEV static fe b() { return fe_from_const(R1_B); }
  DEV static const u32 (&n32())[8] { return R1_N32; }
  DEV static const u32 (&p32())[8] { return R1_P32; }
  DEV static const u32 (&pmn32())[8] { return R1_PMN32; }
  DEV static const u32 (&nhalf32())[8] { return R1_N32; }  // unused (LOW_S is false)
  typedef CH_R1_SQRT SqrtChain;
};

struct jac {
  fe X, Y, Z;
};

// Point formulas on lazy field arithmetic (field.hpp). Inputs: coordinates normalised with value
// < 2M. Outputs: X3, Y3 from fnorm_red (value < (1+2^-19) M), Z3 from a multiplication (< 2M).
// Intermediate bounds are noted as [limb bound in units of 2^29, value bound in units of M];
// a product needs La*Lb < 7.1 and Va*Vb < 32.

template <class C>
DEV jac jdbl(const jac& P) {
  typedef typename C::Fp F;
  jac R;
  if (!C::A_IS_M3) {
    // a = 0, 3M + 4S: S = 4XY^2, M = 3X^2, X3 = M^2 - 2S, Y3 = M(S - X3) - 8Y^4, Z3 = 2YZ
    const fe XX = mont_sqr<F>(P.X);
    const fe YY = mont_sqr<F>(P.Y);                           // [1, 1.13]
    const fe S = mont_mul<F>(fscale_nr(P.X, 4), YY);          // [4, 8] x [1, 1.13] -> [1, 1.29]
    const fe Mn = fnorm_red<F>(fscale_nr(XX, 3));              // [1, 1+]
    R.X = fnorm_red<F>(fsub_nr<F, 3, 2>(mont_sqr<F>(Mn), fscale_nr(S, 2)));
    const fe Y4x4 = mont_sqr<F>(fscale_nr(YY, 2));            // 4 Y^4: [2, 2.26]^2 -> [1, 1.16]
    const fe MSX = mont_mul<F>(Mn, fsub_nr<F, 2, 1>(S, R.X));  // [1, 1+] x [3, 3.29]
    R.Y = fnorm_red<F>(fsub_nr<F, 3, 2>(MSX, fscale_nr(Y4x4, 2)));
    R.Z = mont_mul<F>(fscale_nr(P.Y, 2), P.Z);                // [2, 4] x [1, 2]
  } else {
    // a = -3, dbl-2001-b with 4beta and 2YZ taken as products:
    //   alpha = 3(X - Z^2)(X + Z^2), X3 = alpha^2 - 8beta, Y3 = alpha(4beta - X3) - 8Y^4, Z3 = 2YZ
    const fe delta = mont_sqr<F>(P.Z);
    const fe gamma = mont_sqr<F>(P.Y);
    const fe beta4 = mont_mul<F>(fscale_nr(P.X, 4), gamma);   // [4, 8] x [1, 1.13]
    const fe t = mont_mul<F>(fsub_nr<F, 2, 1>(P.X, delta), fadd_nr(P.X, delta));  // [3, 4] x [2, 3.13]
    const fe alpha = fnorm_red<F>(fscale_nr(t, 3));
    R.X = fnorm_red<F>(fsub_nr<F, 3, 2>(mont_sqr<F>(alpha), fscale_nr(beta4, 2)));
    const fe g4 = mont_sqr<F>(fscale_nr(gamma, 2));            // 4 gamma^2
    const fe aBX = mont_mul<F>(alpha, fsub_nr<F, 2, 1>(beta4, R.X));
    R.Y = fnorm_red<F>(fsub_nr<F, 3, 2>(aBX, fscale_nr(g4, 2)));
    R.Z = mont_mul<F>(fscale_nr(P.Y, 2), P.Z);
  }
  return R;
}

// add-2007-bl: 11M + 5S. exc is set when H == 0 (P == +-Q). Q.Y may be a lazy negation [2, 3].
template <class C>
DEV jac jadd(const jac& P, const jac& Q, bool& exc) {
  typedef typename C::Fp F;
  const fe Z1Z1 = mont_sqr<F>(P.Z);
  const fe Z2Z2 = mont_sqr<F>(Q.Z);
  const fe U1 = mont_mul<F>(P.X, Z2Z2);
  const fe U2 = mont_mul<F>(Q.X, Z1Z1);
  const fe S1 = mont_mul<F>(mont_mul<F>(P.Y, Q.Z), Z2Z2);
  const fe S2 = mont_mul<F>(mont_mul<F>(Q.Y, P.Z), Z1Z1);
  const fe H = fnorm_red<F>(fsub_nr<F, 2, 1>(U2, U1));
  exc = exc || fis_zero<F>(H);
  const fe I = mont_sqr<F>(fscale_nr(H, 2));
  const fe J = mont_mul<F>(H, I);
  const fe r = fnorm_red<F>(fscale_nr(fsub_nr<F, 2, 1>(S2, S1), 2));  // [6, 6.x] -> [1, 1+]
  const fe V = mont_mul<F>(U1, I);
  jac R;
  R.X = fnorm_red<F>(fsub_nr<F, 4, 3>(mont_sqr<F>(r), fadd_nr(J, fscale_nr(V, 2))));
  const fe rVX = mont_mul<F>(r, fsub_nr<F, 2, 1>(V, R.X));
  R.Y = fnorm_red<F>(fsub_nr<F, 2, 1>(rVX, mont_mul<F>(fscale_nr(S1, 2), J)));
  // ((Z1 + Z2)^2 - Z1Z1 - Z2Z2) H = 2 Z1 Z2 H
  const fe Zs = mont_sqr<F>(fadd_nr(P.Z, Q.Z));             // [2, 4]^2
  R.Z = mont_mul<F>(fsub_nr<F, 3, 2>(Zs, fadd_nr(Z1Z1, Z2Z2)), H);  // [4, 4.x] x [1, 1+]
  return R;
}

// madd-2007-bl (Q affine, y2 possibly a lazy negation [2, 3]): 8M + 3S
template <class C>
DEV jac jmadd(const jac& P, const fe& x2, const fe& y2, bool& exc) {
  typedef typename C::Fp F;
  const fe Z1Z1 = mont_sqr<F>(P.Z);
  const fe U2 = mont_mul<F>(x2, Z1Z1);
  const fe S2 = mont_mul<F>(mont_mul<F>(y2, P.Z), Z1Z1);
  const fe H = fnorm_red<F>(fsub_nr<F, 2, 1>(U2, P.X));
  exc = exc || fis_zero<F>(H);
  const fe I4 = fscale_nr(mont_sqr<F>(H), 4);               // I = 4 H^2: [4, 4.x]
  const fe J = mont_mul<F>(H, I4);
  const fe r = fnorm_red<F>(fscale_nr(fsub_nr<F, 2, 1>(S2, P.Y), 2));
  const fe V = mont_mul<F>(P.X, I4);
  jac R;
  R.X = fnorm_red<F>(fsub_nr<F, 4, 3>(mont_sqr<F>(r), fadd_nr(J, fscale_nr(V, 2))));
  const fe rVX = mont_mul<F>(r, fsub_nr<F, 2, 1>(V, R.X));
  R.Y = fnorm_red<F>(fsub_nr<F, 2, 1>(rVX, mont_mul<F>(fscale_nr(P.Y, 2), J)));
  R.Z = mont_mul<F>(P.Z, fscale_nr(H, 2));                  // (Z1 + H)^2 - Z1Z1 - HH = 2 Z1 H
  return R;
}

// ---- the ladder's formulas, on signed arithmetic (sfield.hpp) ----
// Points carry W = 2Y in place of Y: the doubling's 4XY^2 = X W^2 and 8Y^4 = W^4 / 2 then need no
// scaling, and W3 = 2 M (S - X3) - W^4 is a difference of two products that takes one reduction, as
// the addition's W3 = 2 (r (V - X3) - W1 J) is. The subtractions of X3 and the factors 2 and 3 are
// part of the products' carry chains. VALU instructions (secp256k1): doubling 1,055 against jdbl's
// 1,280, mixed addition 1,740 against jmadd's 2,018.
struct jacs {
  sfe X, W, Z;
};

// 3M + 4S (a = 0) or 4M + 4S (a = -3), one reduction less: S = X W^2, M = 3X^2 + aZ^4,
// X3 = M^2 - 2S, W3 = 2 M (S - X3) - W^4, Z3 = W Z
template <class C>
DEV jacs sdbl(const jacs& P) {
  typedef typename C::Fp F;
  const sfe WW = s_sqr<F>(P.W);
  const sfe S = s_mul<F>(P.X, WW);
  sfe Mn;
  if constexpr (C::A_IS_M3)
    Mn = s_sqr_diff<F, 3>(P.X, s_sqr<F>(P.Z));  // 3 (X^2 - Z^4)
  else
    Mn = s_sqr<F, 3>(P.X);
  jacs R;
  R.X = s_sqr_sub<F, 2>(Mn, S);
  R.W = s_dot_sqr<F>(Mn, s_dbl(s_sub(S, R.X)), WW);
  R.Z = s_mul<F>(P.W, P.Z);
  return R;
}

// madd-2007-bl on (X, W, Z) with the affine (x2, w2 = 2 y2), 8M + 3S with one reduction less:
// r = w2 Z1^3 - W1. exc is set when H == 0 (P == +-Q). za: the Z that x2 and w2 are scaled by (P.Z,
// or P.Z times the factor between the accumulator's curve and the table's).
template <class C>
DEV jacs smadd_z(const jacs& P, const sfe& za, const sfe& x2, const sfe& w2, bool& exc) {
  typedef typename C::Fp F;
  const sfe ZZ = s_sqr<F>(za);
  const sfe U2 = s_mul<F>(x2, ZZ);
  const sfe S2 = s_mul<F>(s_mul<F>(w2, za), ZZ);
  const sfe H = s_sub(U2, P.X);
  const sfe HH2 = s_sqr<F, 2>(H);
  exc = exc || s_sqr_maybe_zero<F, 2>(HH2);
  const sfe J = s_mul<F, 2>(H, HH2);    // 4 H^3
  const sfe V = s_mul<F, 2>(P.X, HH2);  // 4 X1 H^2
  const sfe r = s_sub(S2, P.W);
  jacs R;
  R.X = s_fold<F>(s_sqr_sub<F, 1>(r, s_add(J, s_dbl(V))));
  R.W = s_dot<F, 2>(r, s_sub(V, R.X), s_neg(P.W), J);
  R.Z = s_mul<F, 2>(P.Z, H);
  return R;
}
template <class C>
DEV jacs smadd(const jacs& P, const sfe& x2, const sfe& w2, bool& exc) {
  return smadd_z<C>(P, P.Z, x2, w2, exc);
}

// (X, W, Z) -> (X, Y, Z) of the same point in field.hpp's form: Y = W / 2, so scaled by 2:
// (4X, 4W, 2Z)
template <class C>
DEV jac s_to_jac(const jacs& P) {
  typedef typename C::Fp F;
  jac R;
  R.X = fnorm_red<F>(fscale_nr(s_to_fe<F, 4>(P.X), 4));
  R.Y = fnorm_red<F>(fscale_nr(s_to_fe<F, 4>(P.W), 4));
  R.Z = fnorm_red<F>(fscale_nr(s_to_fe<F, 4>(P.Z), 2));
  return R;
}

// -y as a lazy value [2, 3] when neg, y otherwise (no carries, no v_cndmask). y < 2M can have a
// top limb up to (2M >> 232), one above the top limb of 2M's LB = 1 bias, hence K = 3.
template <class F>
DEV fe fneg_if(bool neg, const fe& y) {
  return fsel(neg, fsub_nr<F, 3, 1>(fe_zero(), y), y);
}

// ---- complete (branching) group law for the careful path ----
struct jacf {
  jac P;
  bool inf;
};

template <class C>
DEV jacf jdbl_c(const jacf& P) {
  typedef typename C::Fp F;
  if (P.inf || fis_zero<F>(P.P.Y)) return jacf{P.P, true};
  return jacf{jdbl<C>(P.P), false};
}

template <class C>
DEV jacf jadd_c(const jacf& P, const jacf& Q) {
  typedef typename C::Fp F;
  if (P.inf) return Q;
  if (Q.inf) return P;
  const fe Z1Z1 = mont_sqr<F>(P.P.Z);
  const fe Z2Z2 = mont_sqr<F>(Q.P.Z);
  const fe U1 = mont_mul<F>(P.P.X, Z2Z2);
  const fe U2 = mont_mul<F>(Q.P.X, Z1Z1);
  const fe S1 = mont_mul<F>(mont_mul<F>(P.P.Y, Q.P.Z), Z2Z2);
  const fe S2 = mont_mul<F>(mont_mul<F>(Q.P.Y, P.P.Z), Z1Z1);
  if (feq<F>(U1, U2)) {
    if (feq<F>(S1, S2)) return jdbl_c<C>(P);
    return jacf{P.P, true};
  }
  bool exc = false;
  return jacf{jadd<C>(P.P, Q.P, exc), false};
}

// ---- integer words (little-endian u32) for the GLV split ----
// r = a * b mod 2^(32 NR); every step a[i]*b[j] + r + carry < 2^64
template <int NA, int NB, int NR>
DEV void wmul(const u32* a, const u32* b, u32* r) {
#pragma unroll
  for (int k = 0; k < NR; k++) r[k] = 0;
#pragma unroll
  for (int i = 0; i < NA; i++) {
    u64 c = 0;
#pragma unroll
    for (int j = 0; j < NB; j++) {
      if (i + j < NR) {
        const u64 t = (u64)a[i] * b[j] + r[i + j] + c;
        r[i + j] = (u32)t;
        c = t >> 32;
      }
    }
    if (i + NB < NR) r[i + NB] = (u32)c;
  }
}

DEV void wadd8(u32 a[8], const u32 b[8]) {  // a += b mod 2^256
  u64 c = 0;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const u64 t = (u64)a[i] + b[i] + c;
    a[i] = (u32)t;
    c = t >> 32;
  }
}

DEV void wsub8(u32 a[8], const u32 b[8]) {  // a -= b mod 2^256
  u32 t[8];
  words_sub(a, b, t);
#pragma unroll
  for (int i = 0; i < 8; i++) a[i] = t[i];
}

// GLV split for secp256k1 (constants and their derivation: gen_consts.py glv_k1). For k < n:
//   c1 = round(k g1 / 2^384) = round(k b2 / n), c2 = round(k |b1| / n)  (both < 2^128)
//   (k1, k2) = (k, 0) - c1 (a1, b1) - c2 (a2, b2), so k1 + k2 lambda = k (mod n), |k_i| < 2^128
//   then one lattice vector v1 = (a1, b1) (flips both parities), v2 = (a2, b2) (flips k2) or
//   v1 + v2 (flips k1) makes both halves odd: |k_i| < 2^129.
// Output: magnitudes h1, h2 (5 words) and signs, k = (-1)^n1 h1 + (-1)^n2 h2 lambda (mod n).
DEV void glv_split(const u32 k[8], u32 h1[5], u32 h2[5], bool& n1, bool& n2) {
  u32 p[16], c1[4], c2[4];
#pragma unroll
  for (int pass = 0; pass < 2; pass++) {
    wmul<8, 8, 16>(k, pass == 0 ? GLV_G1 : GLV_G2, p);
    u64 cy = p[11] >> 31;  // + 2^383: round to nearest
    u32* c = pass == 0 ? c1 : c2;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      cy += p[12 + i];
      c[i] = (u32)cy;
      cy >>= 32;
    }
  }
  u32 k1[8], k2[8], t[8];
#pragma unroll
  for (int i = 0; i < 8; i++) k1[i] = k[i];
  wmul<4, 8, 8>(c1, GLV_A1, t);
  wsub8(k1, t);
  wmul<4, 8, 8>(c2, GLV_A2, t);
  wsub8(k1, t);
  wmul<4, 8, 8>(c1, GLV_B1N, k2);
  wmul<4, 8, 8>(c2, GLV_B2, t);
  wsub8(k2, t);
  // parity correction: both even -> v1, k2 even -> v2, k1 even -> v1 + v2
  const bool e1 = (k1[0] & 1u) == 0, e2 = (k2[0] & 1u) == 0;
  const int sel = e1 ? (e2 ? 0 : 2) : 1;
  const u32 any = lane_mask(e1 || e2);
  u32 f1[8], f2[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    u32 a = GLV_FIX_K1[i], b = GLV_FIX_K2[i];
    if (sel == 1) { a = GLV_FIX_K1[8 + i]; b = GLV_FIX_K2[8 + i]; }
    if (sel == 2) { a = GLV_FIX_K1[16 + i]; b = GLV_FIX_K2[16 + i]; }
    f1[i] = a & any;
    f2[i] = b & any;
  }
  wadd8(k1, f1);
  wadd8(k2, f2);
  n1 = (k1[7] >> 31) != 0;
  n2 = (k2[7] >> 31) != 0;
  u32 z[8] = {0, 0, 0, 0, 0, 0, 0, 0}, m1[8], m2[8];
  words_sub(z, k1, m1);
  words_sub(z, k2, m2);
#pragma unroll
  for (int i = 0; i < 5; i++) {
    h1[i] = n1 ? m1[i] : k1[i];
    h2[i] = n2 ? m2[i] : k2[i];
  }
}

// digit carrier of an odd h < 2^B over 5 words: C = (h >> 1) | 2^(B-1); the w-bit digits c_i of C
// give h = sum (2 c_i - (2^w - 1)) 2^(w i), every digit odd and the top one positive
template <int B>
DEV void glv_carrier(const u32 h[5], u32 c[5]) {
#pragma unroll
  for (int i = 0; i < 5; i++) c[i] = (h[i] >> 1) | (i < 4 ? h[i + 1] << 31 : 0u);
  c[(B - 1) >> 5] |= 1u << ((B - 1) & 31);
}

constexpr int GLV_BR = 132;  // R streams: 33 windows of 4 bits (halves < 2^129)
constexpr int GLV_BG = 136;  // G streams: 17 windows of 8 bits

// ---- per-item recovery ----
// sig_raw: the 64 signature bytes as 16 little-endian u32 loads; dig_raw: 8 words of the digest.
// Prologue results shared by the fast and careful ladders.
struct secp_pro {
  u32 status;
  fe rx, ry;         // R affine, Montgomery form of p; ry = -y when ry_neg
  bool ry_neg;
  u32 c1[8], c2[8];  // digit carriers C = (k' >> 1) | 2^255 for u1 (G) and u2 (R) (no GLV)
  bool g_neg;        // G digits must be negated (u1 replaced by n - u1) (no GLV)
  u32 cg1[5], cg2[5], cr1[5], cr2[5];  // GLV: carriers of the halves of u1 (G) and u2 (R)
  bool sg1, sg2, sr1, sr2;             // GLV: signs of those halves
  u32 u1[8], u2[8];  // plain u1, u2 (for the careful path)
};

// odd representative of a scalar k and its digit carrier: k, or n - k when k is even (neg: the digits
// then spell -k), C = (k' >> 1) | 2^255
template <class C>
DEV bool odd_carrier(const u32 k[8], u32 c[8]) {
  const bool neg = (k[0] & 1u) == 0;
  u32 t[8];
  words_sub(C::n32(), k, t);
#pragma unroll
  for (int i = 0; i < 8; i++) t[i] = neg ? t[i] : k[i];
#pragma unroll
  for (int i = 0; i < 8; i++) c[i] = (t[i] >> 1) | (i < 7 ? t[i + 1] << 31 : 0x80000000u);
  return neg;
}

// Q = u1 G + u2 P ladder set-up shared by recovery (P = R) and verification (P = the key), from the
// plain o.u1, o.u2: the digit carriers of the ladder (GLV halves for secp256k1, odd representatives
// otherwise). WIDE: u1 for the wide fixed-base tables (secp_comb) instead of the ladder's G streams.
// P affine (x, y).
template <class C, bool WIDE = false>
DEV void secp_carriers(secp_pro& o, const fe& x, const fe& y) {
  typedef typename C::Fp Fp;
  o.rx = x;
  o.ry = y;
  o.ry_neg = false;
  o.g_neg = false;
  if constexpr (WIDE || !C::GLV) o.g_neg = odd_carrier<C>(o.u1, o.c1);
  if constexpr (C::GLV) {
    u32 h1[5], h2[5];
    if constexpr (!WIDE) {
      glv_split(o.u1, h1, h2, o.sg1, o.sg2);
      glv_carrier<GLV_BG>(h1, o.cg1);
      glv_carrier<GLV_BG>(h2, o.cg2);
    }
    glv_split(o.u2, h1, h2, o.sr1, o.sr2);
    glv_carrier<GLV_BR>(h1, o.cr1);
    glv_carrier<GLV_BR>(h2, o.cr2);
  } else {
    o.ry_neg = odd_carrier<C>(o.u2, o.c2);
    if (o.ry_neg) o.ry = fneg<Fp>(y);
  }
}

// the same from u1m, u2m in Montgomery form of n
template <class C, bool WIDE = false>
DEV void secp_scalars(secp_pro& o, const fe& u1m, const fe& u2m, const fe& x, const fe& y) {
  typedef typename C::Fn Fn;
  fe_to_words(from_mont<Fn>(u1m), o.u1);
  fe_to_words(from_mont<Fn>(u2m), o.u2);
  secp_carriers<C, WIDE>(o, x, y);
}

// a signature's r, s, its recovery parity, and z = digest mod n; ST_OK, ST_BAD_R or ST_BAD_S
struct secp_sig {
  u32 r[8], s[8], z[8];
  bool y_odd;
};
template <class C>
DEV u32 secp_decode_sig(const u32 sig_raw[16], secp_sig& o) {
  const u32(&n)[8] = C::n32();
  u32 sraw[8];
#pragma unroll
  for (int i = 0; i < 8; i++) sraw[i] = sig_raw[8 + i];
  o.y_odd = (sraw[0] & 0x80u) != 0;  // first byte of s
  sraw[0] &= ~0x80u;
  words_from_be_bytes(sig_raw, o.r);
  words_from_be_bytes(sraw, o.s);
  if (words_is_zero(o.r) || !words_lt(o.r, n)) return ST_BAD_R;
  if (words_is_zero(o.s) || !words_lt(o.s, n)) return ST_BAD_S;
  return ST_OK;
}
template <class C>
DEV void secp_decode_digest(const u32 dig_raw[8], secp_sig& o) {
  const u32(&n)[8] = C::n32();
  words_from_be_bytes(dig_raw, o.z);
  if (!words_lt(o.z, n)) {
    u32 t[8];
    words_sub(o.z, n, t);
#pragma unroll
    for (int i = 0; i < 8; i++) o.z[i] = t[i];
  }
}

// x^3 + a x + b
template <class C>
DEV fe secp_rhs(const fe& x) {
  typedef typename C::Fp Fp;
  fe rhs = mont_mul<Fp>(mont_sqr<Fp>(x), x);
  if (C::A_IS_M3) rhs = fsub<Fp>(rhs, fadd<Fp>(fdbl<Fp>(x), x));
  return fadd<Fp>(rhs, C::b());
}

// the curve point with x-coordinate r and the given parity of y; false if there is none
template <class C>
DEV bool secp_lift(const u32 r[8], bool y_odd, fe& x, fe& y) {
  typedef typename C::Fp Fp;
  x = to_mont<Fp>(fe_from_words(r));
  const fe rhs = secp_rhs<C>(x);
  y = s_to_fe<Fp, 1>(s_pow_chain<Fp, typename C::SqrtChain>(s_from(rhs)));
  const bool ok = feq<Fp>(mont_sqr<Fp>(y), rhs);
  const fe yc = from_mont<Fp>(y);
  if ((bool)(yc.v[0] & 1u) != y_odd) y = fneg<Fp>(y);
  return ok;
}

template <class C, bool WIDE = false>
DEV void secp_prologue(const u32 sig_raw[16], const u32 dig_raw[8], secp_pro& o) {
  typedef typename C::Fn Fn;
  secp_sig g;
  o.status = secp_decode_sig<C>(sig_raw, g);
  secp_decode_digest<C>(dig_raw, g);
  fe x, y;
  const bool ok = secp_lift<C>(g.r, g.y_odd, x, y);
  if (o.status == ST_OK && !ok) o.status = ST_NO_POINT;
  // u1 = -z/r, u2 = s/r (mod n)
  const fe rn = to_mont<Fn>(fe_from_words(g.r));
  const fe rinv = finv<Fn>(rn);
  const fe u1m = fneg<Fn>(mont_mul<Fn>(to_mont<Fn>(fe_from_words(g.z)), rinv));
  const fe u2m = mont_mul<Fn>(to_mont<Fn>(fe_from_words(g.s)), rinv);
  secp_scalars<C, WIDE>(o, u1m, u2m, x, y);
}

// ---- verification with a known public key (fuel Signature::verify) ----
// Rules of the reference's CPU stack (fuel-crypto 0.49 over libsecp256k1 for secp256k1, p256 /
// ecdsa 0.16 verify_prehash for secp256r1): r, s in [1, n-1] after clearing the recid bit (which
// verification ignores); secp256k1 also s <= (n-1)/2; the key X || Y with X, Y < p on the curve;
// z = digest mod n, u1 = z/s, u2 = r/s, P = u1 G + u2 Q != infinity, accept iff x(P) mod n == r.
// pub_raw: the 64 key bytes as 16 little-endian u32 loads. The same ladders then run with the key
// in place of R.
// the key as an affine point and the checks that do not need the scalars
template <class C>
DEV u32 secp_decode_verify(const u32 sig_raw[16], const u32 pub_raw[16], secp_sig& g, fe& x, fe& y) {
  typedef typename C::Fp Fp;
  u32 xw[8], yw[8];
  words_from_be_bytes(pub_raw, xw);
  words_from_be_bytes(pub_raw + 8, yw);
  u32 st = secp_decode_sig<C>(sig_raw, g);
  if (st == ST_OK && C::LOW_S && words_lt(C::nhalf32(), g.s)) st = ST_HIGH_S;
  if (st == ST_OK && (!words_lt(xw, C::p32()) || !words_lt(yw, C::p32()))) st = ST_BAD_KEY;
  x = to_mont<Fp>(fe_from_words(xw));
  y = to_mont<Fp>(fe_from_words(yw));
  if (st == ST_OK && !feq<Fp>(mont_sqr<Fp>(y), secp_rhs<C>(x))) st = ST_BAD_KEY;
  return st;
}

template <class C, bool WIDE = false>
DEV void secp_prologue_verify(const u32 sig_raw[16], const u32 dig_raw[8], const u32 pub_raw[16], secp_pro& o) {
  typedef typename C::Fn Fn;
  secp_sig g;
  fe x, y;
  o.status = secp_decode_verify<C>(sig_raw, pub_raw, g, x, y);
  secp_decode_digest<C>(dig_raw, g);
  // u1 = z/s, u2 = r/s (mod n)
  const fe sinv = finv<Fn>(to_mont<Fn>(fe_from_words(g.s)));
  const fe u1m = mont_mul<Fn>(to_mont<Fn>(fe_from_words(g.z)), sinv);
  const fe u2m = mont_mul<Fn>(to_mont<Fn>(fe_from_words(g.r)), sinv);
  secp_scalars<C, WIDE>(o, u1m, u2m, x, y);
}

// the verifier's final check on P = (X : Y : Z) (Jacobian) without an inversion: x(P) < p < 2n,
// so x(P) mod n == r means X == r Z^2, or X == (r + n) Z^2 when r + n < p. sig_raw: the signature
// as loaded (r is decoded again here rather than kept live through the ladder).
template <class C>
DEV u32 secp_verify_x(const jac& P, const u32 sig_raw[16]) {
  typedef typename C::Fp F;
  u32 r[8], rn[8];
  words_from_be_bytes(sig_raw, r);
  words_add(r, C::n32(), rn);  // meaningful only when r < p - n
  const fe z2 = mont_sqr<F>(P.Z);
  const bool eq1 = feq<F>(P.X, mont_mul<F>(to_mont<F>(fe_from_words(r)), z2));
  const bool eq2 = feq<F>(P.X, mont_mul<F>(to_mont<F>(fe_from_words(rn)), z2));
  if (fis_zero<F>(P.Z)) return ST_INFINITY;
  return (eq1 || (eq2 && words_lt(r, C::pmn32()))) ? ST_OK : ST_MISMATCH;
}

DEV u32 nibble(const u32 c[8], int i) { return (c[i >> 3] >> ((i & 7) * 4)) & 15u; }
DEV u32 byte8(const u32 c[8], int j) { return (c[j >> 2] >> ((j & 3) * 8)) & 255u; }
// 9-bit digit j of a carrier (bits 9j .. 9j + 8, which may straddle two words)
DEV u32 digit9(const u32* c, int j) {
  const int b = 9 * j, w = b >> 5, sh = b & 31;
  u32 v = c[w] >> sh;
  if (sh > 23) v |= c[w + 1] << (32 - sh);
  return v & 511u;
}

// fixed-base windows of 9 bits (the host check's second form): 256 odd multiples of G, 4 fewer G
// additions per secp256k1 item and 3 per P-256 item than 8 bits. The carriers come from the 8-bit ones: a carrier is
// (h >> 1) | 2^(B-1) for the odd h it spells, so moving the marker bit re-spells h over B' bits.
constexpr int GLV_BG9 = 135;  // G streams of secp256k1: 15 windows of 9 bits
constexpr int R1_BG9 = 261;   // the G stream of P-256: 29 windows of 9 bits

// acc + the entry of the per-lane table that the 4-bit digit d spells (negated per digit and stream
// sign); PHI: phi(entry) = (beta x, y). e: the entry, loaded ahead by r_load.
struct r_entry {
  fe x, w;
};
template <bool PHI, class Tab>
DEV r_entry r_load(const Tab& tab, u32 d) {
  r_entry e;
  const u32 idx = ((d < 8) ? ~d : d) & 7u;
  if constexpr (PHI)
    tab.load_affine_phi(idx, e.x, e.w);
  else
    tab.load_affine(idx, e.x, e.w);
  return e;
}
template <class C>
DEV jacs r_add(const jacs& acc, const r_entry& e, bool neg, bool& exc) {
  typedef typename C::Fp F;
  return smadd<C>(acc, s_unraw<F>(e.x), s_neg_if(neg, s_unraw<F>(e.w)), exc);
}

// acc + the odd multiple of the G table's point that the digit d of WGB bits spells; zeta: the
// accumulator's coordinates are those of the curve isomorphic by zeta (secp_build_table)
template <class C, int WGB, bool PHI, class GTab>
DEV jacs g_add(const jacs& acc, const GTab& gt, u32 d, bool neg_stream, const sfe& zeta, bool& exc) {
  typedef typename C::Fp F;
  constexpr u32 HALF = 1u << (WGB - 1);
  fe gx, gy;
  const u32 idx = ((d < HALF) ? ~d : d) & (HALF - 1u);
  if constexpr (PHI)
    gt.load_phi(idx, gx, gy);
  else
    gt.load(idx, gx, gy);
  const sfe w = s_neg_if((d < HALF) != neg_stream, s_dbl(s_from(gy)));
  if constexpr (C::GLV) return smadd_z<C>(acc, s_mul<F>(acc.Z, zeta), s_from(gx), w, exc);
  return smadd<C>(acc, s_from(gx), w, exc);
}

// Per-lane table of the odd multiples (2e + 1) P, e = 0..7, as affine (x, w = 2y) on a curve where
// all of them are, so that the ladder adds its entries with the mixed formula (8M + 3S instead of
// 11M + 5S per addition).
// The entries are built on an isomorphic curve where 2P is affine, so the seven additions are
// mixed ones too: with 2P = (X2, W2, Z2), the map (x, y) -> (Z2^2 x, Z2^3 y) takes the curve to
// y^2 = x^3 + a Z2^4 x + b Z2^6, 2P to the affine (X2, W2) and P to (Z2^2 x, Z2^3 y). The addition
// formulas do not involve a or b. A Jacobian (X, W, Z) there is (X, W, Z Z2) on the curve.
// Then, from the last entry down, with the factors zr_e = Z_e / Z_(e-1) that the additions give:
//   * a = 0 (secp256k1): the entries are scaled to the last one's Z, (X rho^2, W rho^3) with
//     rho = Z_7 / Z_e, which makes them affine on the curve isomorphic by zeta = Z2 Z_7. The ladder
//     runs there (the doubling does not involve b) and multiplies its Z by zeta at the end, so no
//     inversion is needed (a divstep inversion is 20,000 instructions, 7% of an item). beta x is
//     stored beside each entry for the phi(R) stream.
//   * a = -3 (P-256): the doubling needs a, so the entries are made affine on the curve itself by
//     one inversion of Z2 Z_7 (Montgomery's trick, with the same factors).
// Tab: store_full(e, (X, W, zr), unused) / load_full and store_affine(e, x, w) / load_affine (and
// the _phi forms with beta x); sync() if other lanes read what one lane stores: it orders the stores
// before it with the other lanes' loads after it, and loads with stores likewise. Returns zeta (1 for
// P-256).
template <class Tab>
DEV auto tab_sync(Tab& tab, int) -> decltype(tab.sync()) {
  tab.sync();
}
template <class Tab>
DEV void tab_sync(Tab&, long) {}

template <class C, class Tab>
DEV sfe secp_build_table(const secp_pro& o, Tab& tab, bool& exc) {
  typedef typename C::Fp F;
  jacs P;
  P.X = s_from(o.rx);
  P.W = s_from(fnorm_red<F>(fscale_nr(o.ry, 2)));
  P.Z = s_from(fe_from_const(F::ONE));
  const jacs P2 = sdbl<C>(P);
  const sfe beta = s_from(C::GLV ? fe_from_const(K1_BETA) : fe_zero());
  const sfe zz = s_sqr<F>(P2.Z);
  jacs T;
  T.X = s_mul<F>(P.X, zz);
  T.W = s_mul<F>(P.W, s_mul<F>(zz, P2.Z));
  T.Z = P.Z;
  tab.store_full(0, jac{s_raw(T.X), s_raw(T.W), s_raw(T.Z)}, fe_zero());
#pragma unroll 1
  for (int e = 1; e < 8; e++) {
    // smadd with Z1 = 1 tracked apart: Z_e = Z_(e-1) zr_e with zr_e = 2H
    const sfe ZZ = s_sqr<F>(T.Z);
    const sfe H = s_sub(s_mul<F>(P2.X, ZZ), T.X);
    const sfe r = s_sub(s_mul<F>(s_mul<F>(P2.W, T.Z), ZZ), T.W);
    const sfe HH2 = s_sqr<F, 2>(H);
    exc = exc || s_sqr_maybe_zero<F, 2>(HH2);
    const sfe J = s_mul<F, 2>(H, HH2);
    const sfe V = s_mul<F, 2>(T.X, HH2);
    // 2H as a normalised value: 2H times R times R^-1
    const sfe zr = s_mul<F, 2>(H, P.Z);
    T.X = s_fold<F>(s_sqr_sub<F, 1>(r, s_add(J, s_dbl(V))));
    T.W = s_dot<F, 2>(r, s_sub(V, T.X), s_neg(T.W), J);
    T.Z = s_mul<F>(T.Z, zr);
    tab.store_full(e, jac{s_raw(T.X), s_raw(T.W), s_raw(zr)}, fe_zero());
  }
  tab_sync(tab, 0);
  sfe zeta = s_mul<F>(T.Z, P2.Z);  // Z2 Z_7
  sfe rho;
  if constexpr (C::GLV)
    rho = P.Z;
  else
    rho = s_from(finv<F>(s_to_fe<F, 4>(zeta)));  // 1 / (Z2 Z_7)
#pragma unroll 1
  for (int e = 7; e >= 0; e--) {
    jac E;  // (X, W, zr)
    fe unused;
    tab.load_full(e, E, unused);
    tab_sync(tab, 0);
    const sfe r2 = s_sqr<F>(rho);
    const sfe ax = s_mul<F>(s_unraw<F>(E.X), r2);
    const sfe aw = s_mul<F>(s_unraw<F>(E.Y), s_mul<F>(r2, rho));
    rho = s_mul<F>(rho, s_unraw<F>(E.Z));
    if constexpr (C::GLV)
      tab.store_affine_phi(e, s_raw(ax), s_raw(aw), s_raw(s_mul<F>(ax, beta)));
    else
      tab.store_affine(e, s_raw(ax), s_raw(aw));
  }
  return zeta;
}

// the ladder's first point: the entry of the top digit (always positive), with the stream's sign
template <class C, class Tab>
DEV jacs r_first(const Tab& tab, u32 d, bool neg) {
  typedef typename C::Fp F;
  fe x, w;
  tab.load_affine(d - 8, x, w);
  return jacs{s_unraw<F>(x), s_carry(s_neg_if(neg, s_unraw<F>(w))), s_from(fe_from_const(F::ONE))};
}

// Q = h1 G + h2 phi(G) + h3 R + h4 phi(R) on one doubling chain of 132 bits (secp256k1; phi(x, y) =
// (beta x, y), both tables store beta x beside x), or u1 G + u2 R on one of 256 bits (P-256). R
// streams: 33 (64) windows of 4 bits over the per-lane table of odd multiples of R. G streams: WGB
// = 8 or 9 bits over the table gt of odd multiples of G, or WGB = 0: none, the caller adds u1 G
// (secp_comb). Every window adds exactly one entry.
template <class C, int WGB, class Tab, class GTab>
DEV jacs secp_ladder_s(const secp_pro& o, Tab& tab, const GTab& gt, bool& exc) {
  typedef typename C::Fp F;
  static_assert(WGB == 0 || WGB == 8 || WGB == 9, "fixed-base windows of 8 or 9 bits, or none");
  const sfe zeta = secp_build_table<C>(o, tab, exc);
  jacs acc;
  if constexpr (C::GLV) {
    u32 cg1[5], cg2[5];
#pragma unroll
    for (int i = 0; i < 5; i++) {
      cg1[i] = o.cg1[i];
      cg2[i] = o.cg2[i];
    }
    if constexpr (WGB == 9) {  // marker bit GLV_BG - 1 = 135 -> GLV_BG9 - 1 = 134 (the halves are below 2^130)
      cg1[4] = (cg1[4] & ~(1u << 7)) | (1u << 6);
      cg2[4] = (cg2[4] & ~(1u << 7)) | (1u << 6);
    }
    acc = r_first<C>(tab, nibble(o.cr1, 32), o.sr1);
    {
      const u32 d = nibble(o.cr2, 32);
      acc = r_add<C>(acc, r_load<true>(tab, d), o.sr2, exc);
    }
    if constexpr (WGB == 8) {
      acc = g_add<C, WGB, false>(acc, gt, byte8(cg1, 16), o.sg1, zeta, exc);
      acc = g_add<C, WGB, true>(acc, gt, byte8(cg2, 16), o.sg2, zeta, exc);
    }
    // the first table load of a window is issued before its doublings and the second before the
    // first addition; each is hidden behind that work without keeping both entries live
    if constexpr (WGB == 9) {  // one doubling per trip: R digits at multiples of 4, G digits at multiples of 9
      r_entry e1;
      u32 c1 = 0;
#pragma unroll 1
      for (int p = 127; p >= 0; p--) {
        if ((p & 3) == 3) {
          c1 = nibble(o.cr1, p >> 2);
          e1 = r_load<false>(tab, c1);
        }
        acc = sdbl<C>(acc);
        if ((p & 3) == 0) {
          const u32 c2 = nibble(o.cr2, p >> 2);
          const r_entry e2 = r_load<true>(tab, c2);
          acc = r_add<C>(acc, e1, (c1 < 8) != o.sr1, exc);
          acc = r_add<C>(acc, e2, (c2 < 8) != o.sr2, exc);
        }
        if (p % 9 == 0) {
          acc = g_add<C, WGB, false>(acc, gt, digit9(cg1, p / 9), o.sg1, zeta, exc);
          acc = g_add<C, WGB, true>(acc, gt, digit9(cg2, p / 9), o.sg2, zeta, exc);
        }
      }
    } else {
#pragma unroll 1
      for (int i = 31; i >= 0; i--) {
        const u32 c1 = nibble(o.cr1, i), c2 = nibble(o.cr2, i);
        const r_entry e1 = r_load<false>(tab, c1);
#pragma unroll 1
        for (int d = 0; d < 4; d++) acc = sdbl<C>(acc);
        const r_entry e2 = r_load<true>(tab, c2);
        acc = r_add<C>(acc, e1, (c1 < 8) != o.sr1, exc);
        acc = r_add<C>(acc, e2, (c2 < 8) != o.sr2, exc);
        if constexpr (WGB == 8) {
          if ((i & 1) == 0) {
            acc = g_add<C, WGB, false>(acc, gt, byte8(cg1, i >> 1), o.sg1, zeta, exc);
            acc = g_add<C, WGB, true>(acc, gt, byte8(cg2, i >> 1), o.sg2, zeta, exc);
          }
        }
      }
    }
    acc.Z = s_mul<F>(acc.Z, zeta);
  } else {
    u32 cg[9];
#pragma unroll
    for (int i = 0; i < 8; i++) cg[i] = o.c1[i];
    cg[8] = 0;
    if constexpr (WGB == 9) {
      cg[7] &= 0x7fffffffu;  // marker bit 255 -> R1_BG9 - 1 = 260 (u1 < n < 2^256)
      cg[8] = 1u << (R1_BG9 - 1 - 256);
    }
    acc = r_first<C>(tab, nibble(o.c2, 63), false);
    if constexpr (WGB == 9) {
      acc = g_add<C, WGB, false>(acc, gt, digit9(cg, 28), o.g_neg, zeta, exc);
      r_entry e;
      u32 c = 0;
#pragma unroll 1
      for (int p = 251; p >= 0; p--) {
        if ((p & 3) == 3) {
          c = nibble(o.c2, p >> 2);
          e = r_load<false>(tab, c);
        }
        acc = sdbl<C>(acc);
        if ((p & 3) == 0) acc = r_add<C>(acc, e, c < 8, exc);
        if (p % 9 == 0) acc = g_add<C, WGB, false>(acc, gt, digit9(cg, p / 9), o.g_neg, zeta, exc);
      }
    } else {
#pragma unroll 1
      for (int i = 62; i >= 0; i--) {
        // the HBM load of this window's entry is issued before the doublings, which hide its latency
        const u32 c = nibble(o.c2, i);
        const r_entry e = r_load<false>(tab, c);
#pragma unroll 1
        for (int d = 0; d < 4; d++) acc = sdbl<C>(acc);
        acc = r_add<C>(acc, e, c < 8, exc);
        if constexpr (WGB == 8) {
          if ((i & 1) == 0) acc = g_add<C, WGB, false>(acc, gt, byte8(cg, i >> 1), o.g_neg, zeta, exc);
        }
      }
    }
  }
  return acc;
}

// ---- u1 G from wide fixed-base tables ----
// For every 16-bit window i of a scalar the 32,768 odd multiples (2j + 1) 2^(16 i) G, affine as
// (x, w = 2y), 64 bytes each: 33.5 MB per curve, built on the GPU once per device (kern_comb.hip).
// u1 G then takes 16 mixed additions and no doubling, against 30 (secp256k1) or 29 (P-256) additions
// from 9-bit windows on the ladder's chain.
constexpr int COMB_BITS = 16;
constexpr int COMB_WINDOWS = 256 / COMB_BITS;
constexpr u32 COMB_ENTRIES = 1u << (COMB_BITS - 1);

struct comb_entry {
  u32 v[16];  // x, w as 8 little-endian words each, canonical Montgomery form
};

// acc + the 16 entries that u1's digits spell (o.c1, o.g_neg from secp_carriers<C, true>). Comb:
// load(i, j, comb_entry&). The next entry's load is issued before an addition that does not need it.
template <class C, class Comb>
DEV jacs secp_comb(jacs acc, const secp_pro& o, const Comb& comb, bool& exc) {
  auto digit = [&](int i) { return (o.c1[i >> 1] >> ((i & 1) * 16)) & 0xFFFFu; };
  auto load = [&](int i, comb_entry& e) {
    const u32 d = digit(i);
    comb.load(i, ((d < COMB_ENTRIES) ? ~d : d) & (COMB_ENTRIES - 1u), e);
  };
  comb_entry e;
  load(0, e);
#pragma unroll 1
  for (int i = 0; i < COMB_WINDOWS; i++) {
    const sfe x = s_from(fe_from_words(e.v)), w = s_from(fe_from_words(e.v + 8));
    const bool neg = (digit(i) < COMB_ENTRIES) != o.g_neg;
    if (i + 1 < COMB_WINDOWS) load(i + 1, e);
    acc = smadd<C>(acc, x, s_neg_if(neg, w), exc);
  }
  return acc;
}

// secp_ladder_s with its result in field.hpp's form. R-table stored per lane (secp_build_table).
// GTab provides load(idx, fe& x, fe& y) for the odd multiples (2 idx + 1) G: 128 of them for
// fixed-base windows of WGB = 8 bits, 256 for 9.
template <class C, int WGB = 8, class Tab, class GTab>
DEV jac secp_ladder(const secp_pro& o, Tab& tab, const GTab& gt, bool& exc) {
  return s_to_jac<C>(secp_ladder_s<C, WGB>(o, tab, gt, exc));
}

// careful path: Q = u1*G + u2*R by double-and-add with the complete law (slow, branching)
template <class C, class GTab>
DEV jacf secp_ladder_careful(const secp_pro& o, const GTab& gt) {
  typedef typename C::Fp F;
  jacf G, R, GR, acc;
  fe gx, gy;
  gt.load(0, gx, gy);
  G.P.X = gx; G.P.Y = gy; G.P.Z = fe_from_const(F::ONE); G.inf = false;
  // o.u2 is the true u2; undo the negation of o.ry that came with the fast ladder's n - u2
  R.P.X = o.rx; R.P.Y = o.ry_neg ? fneg<F>(o.ry) : o.ry; R.P.Z = fe_from_const(F::ONE); R.inf = false;
  GR = jadd_c<C>(G, R);
  acc.inf = true;
  acc.P = G.P;
  for (int i = 255; i >= 0; i--) {
    acc = jdbl_c<C>(acc);
    const bool b1 = (o.u1[i >> 5] >> (i & 31)) & 1u;
    const bool b2 = (o.u2[i >> 5] >> (i & 31)) & 1u;
    if (b1 && b2) acc = jadd_c<C>(acc, GR);
    else if (b1) acc = jadd_c<C>(acc, G);
    else if (b2) acc = jadd_c<C>(acc, R);
  }
  return acc;
}

// affine x, y (Montgomery form) from X, Y, Z and 1 / Z, as big-endian X || Y (16 words as stored)
template <class C>
DEV void secp_store_affine(const fe& X, const fe& Y, const fe& zi, u32 out_raw[16]) {
  typedef typename C::Fp F;
  const fe zi2 = mont_sqr<F>(zi);
  const fe x = from_mont<F>(mont_mul<F>(X, zi2));
  const fe y = from_mont<F>(mont_mul<F>(Y, mont_mul<F>(zi2, zi)));
  u32 w[8];
  fe_to_words(x, w);
  words_to_be_bytes(w, out_raw);
  fe_to_words(y, w);
  words_to_be_bytes(w, out_raw + 8);
}

// Jacobian -> affine
template <class C>
DEV void secp_output(const jac& Q, u32 out_raw[16]) {
  secp_store_affine<C>(Q.X, Q.Y, finv<typename C::Fp>(Q.Z), out_raw);
}

// u1 G + u2 P on the wide tables (o from secp_carriers<C, true>)
template <class C, class Tab, class Comb>
DEV jac secp_ladder_wide(const secp_pro& pro, Tab& tab, const Comb& comb, bool& exc) {
  const jacs Q = secp_ladder_s<C, 0>(pro, tab, comb, exc);
  return s_to_jac<C>(secp_comb<C>(Q, pro, comb, exc));
}

// one recovery by itself, its inversions not shared: the status (ST_PENDING when the ladder met an
// exceptional addition and the careful pass must redo the item) and the key X || Y (zeros unless
// ST_OK)
template <class C, class Tab, class Comb>
DEV u32 secp_item(const u32 sr[16], const u32 dr[8], Tab& tab, const Comb& comb, u32 o[16]) {
  secp_pro pro;
  secp_prologue<C, true>(sr, dr, pro);
  u32 st = pro.status;
  if (st == ST_OK) {
    bool exc = false;
    const jac Q = secp_ladder_wide<C>(pro, tab, comb, exc);
    if (exc)
      st = ST_PENDING;
    else
      secp_output<C>(Q, o);
  }
  if (st != ST_OK) {
#pragma unroll
    for (int k = 0; k < 16; k++) o[k] = 0;
  }
  return st;
}

}  // namespace sigops
