// sfield_check.cpp -- host (g++) build of the signed field arithmetic (csrc/sfield.hpp), exposed on
// raw limbs so that tests compare it with Python integers at the edges of its limb ranges. Bound
// checker on: an operand outside what the columns hold aborts. Test infrastructure only.
#include "secp.hpp"

using namespace sigops;

namespace {
sfe in(const int* v, int lo, int hi) {  // limbs 0..7 in [lo, hi], limb 8 as small as the ladder's
  sfe r;
  for (int k = 0; k < NL; k++) r.v[k] = v[k];
  r.lo = lo;
  r.hi = hi;
  r.thi = 1 << 26;
  r.tlo = -r.thi;
  r.vhi = ldexpl((long double)r.thi + 4, 232);
  r.vlo = -r.vhi;
  return r;
}

template <class F>
void run(int op, const int* a, const int* b, const int* c, const int* d, int* out, unsigned* canon) {
  const int N = (int)LMASK;
  sfe r;
  switch (op) {
    case 0: r = s_mul<F>(in(a, -N, N), in(b, -N, N)); break;
    case 1: r = s_mul<F, 2>(in(a, -N, N), in(b, -N, N)); break;
    case 2: r = s_sqr<F>(in(a, -N, N)); break;
    case 3: r = s_sqr<F, 3>(in(a, -N, N)); break;
    case 4: r = s_sqr_sub<F, 2>(in(a, -N, N), in(b, -N, N)); break;
    case 5: r = s_dot<F, 2>(in(a, -N, N), in(b, -N, N), in(c, -N, N), in(d, -N, N)); break;
    case 6: r = s_dot_sqr<F>(in(a, -N, N), in(b, -2 * N, 2 * N), in(c, -N, N)); break;
    case 7: r = s_sqr_diff<F, 3>(in(a, 0, N), in(b, 0, N)); break;
    case 8: r = s_fold<F>(in(a, 0, N)); break;
    default: r = s_carry(in(a, -3 * N, 3 * N)); break;
  }
  for (int k = 0; k < NL; k++) out[k] = r.v[k];
  if (op < 8) {  // small enough for the conversion: r > -20 M
    const fe f = s_to_fe<F, 20>(r);
    for (int k = 0; k < NL; k++) canon[k] = f.v[k];
  }
}
}  // namespace

extern "C" {
// op on limb vectors modulo secp256k1 p (0), P-256 p (1) or 2^255 - 19 (2); out: the result's limbs,
// canon: the same value as field.hpp's normalised limbs (ops 0..7)
void sc_op(int op, int mod, const int* a, const int* b, const int* c, const int* d, int* out, unsigned* canon) {
  if (mod == 0) run<ModPk1>(op, a, b, c, d, out, canon);
  else if (mod == 1) run<ModPr1>(op, a, b, c, d, out, canon);
  else run<ModPed>(op, a, b, c, d, out, canon);
}

// s_sqr_maybe_zero on the square of H = U2 - X given as limbs
int sc_maybe_zero(int mod, const int* h) {
  const int N = (int)LMASK;
  sfe x = in(h, -N, N);
  x.thi = 1 << 26;
  x.tlo = -x.thi;
  x.vhi = ldexpl((long double)x.thi, 232);
  x.vlo = -x.vhi;
  if (mod == 0) return s_sqr_maybe_zero<ModPk1, 2>(s_sqr<ModPk1, 2>(x));
  return s_sqr_maybe_zero<ModPr1, 2>(s_sqr<ModPr1, 2>(x));
}
}
