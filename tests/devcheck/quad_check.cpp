// quad_check.cpp -- host (g++) build of the four-lane point formulas (csrc/quad.hpp): the lanes of a
// quad held in an array, with the bound checker on for each. Test infrastructure only.
#include <cstring>

#include "quad.hpp"

using namespace sigops;

namespace {
template <class F>
sfe load(const unsigned char* be) {
  u32 raw[8], w[8];
  memcpy(raw, be, 32);
  words_from_be_bytes(raw, w);
  const fe m = fcanon<F>(fnorm_red<F>(to_mont<F>(fe_from_words(w))));
  return s_from(m);
}
template <class F>
void store(const fe& x, unsigned char* be) {
  u32 w[8], raw[8];
  fe_to_words(from_mont<F>(x), w);
  words_to_be_bytes(w, raw);
  memcpy(be, raw, 32);
}

// starts at P, then for each step 'd' doubles and 'a' / 's' adds / subtracts the affine Q
template <class C>
int secp(const char* prog, const unsigned char* p, const unsigned char* q, unsigned char* out) {
  typedef typename C::Fp F;
  const sfe one = s_from(fe_from_const(F::ONE));
  const sfe qx = load<F>(q), qw = s_carry(s_dbl(load<F>(q + 32)));
  qfe s{{load<F>(p), s_carry(s_dbl(load<F>(p + 32))), one, one}};
  bool exc = false;
  for (; *prog; prog++) {
    if (*prog == 'd') s = q_sdbl<C>(s);
    else s = q_smadd<C>(s, qfe{{qx, qx, qx, *prog == 'a' ? qw : s_neg(qw)}}, exc);
  }
  const fe zi = finv<F>(s_to_fe<F, 4>(s.l[3]));
  const fe zz = mont_sqr<F>(mont_mul<F>(s_to_fe<F, 4>(s.l[2]), zi));
  store<F>(mont_mul<F>(s_to_fe<F, 4>(s.l[0]), zz), out);
  store<F>(mont_mul<F>(s_to_fe<F, 4>(s_carry(s.l[1])), zi), out + 32);  // 2y
  return exc;
}
}  // namespace

extern "C" {
int qc_secp(int curve, const char* prog, const unsigned char* p, const unsigned char* q, unsigned char* out) {
  return curve == 0 ? secp<CurveK1>(prog, p, q, out) : secp<CurveR1>(prog, p, q, out);
}

// the same on Edwards points (x, y); out: x, y
void qc_ed(const char* prog, const unsigned char* p, const unsigned char* q, unsigned char* out) {
  const sfe one = s_from(fe_from_const(Fe::ONE)), d2 = s_from(fe_from_const(ED_D2));
  const sfe x = load<Fe>(q), y = load<Fe>(q + 32);
  const sfe px = load<Fe>(p), py = load<Fe>(p + 32);
  const sfe t = s_mul<Fe>(s_mul<Fe>(x, y), d2);
  const sfe ypx = s_carry(s_add(y, x)), ymx = s_carry(s_sub(y, x));
  qfe s{{px, py, one, s_mul<Fe>(px, py)}};
  for (; *prog; prog++) {
    if (*prog == 'd') s = q_edbl(s);
    else if (*prog == 'a') s = q_eadd(s, qfe{{ymx, ypx, one, t}});
    else s = q_eadd(s, qfe{{ypx, ymx, one, s_neg(t)}});
  }
  const fe zi = finv<Fe>(s_to_fe<Fe, 8>(s.l[2]));
  store<Fe>(mont_mul<Fe>(s_to_fe<Fe, 8>(s.l[0]), zi), out);
  store<Fe>(mont_mul<Fe>(s_to_fe<Fe, 8>(s.l[1]), zi), out + 32);
}
}
