// wide_check.cpp -- host (g++) build, bound checker on, of what the kernels run by default: the ladders with
// the wide fixed-base tables, one item at a time, through the stages that share inversions, and on the four
// lanes of a quad. The tables' entries come from the caller, entry by entry. Test infrastructure only.
#include <cstring>
#include <vector>

#include <cstdint>
struct uint4 {
  uint32_t x, y, z, w;
};
inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return uint4{x, y, z, w}; }

#include "quad.hpp"
#include "stages.hpp"

using namespace sigops;

namespace {
// entry j of window `win` of a curve's wide table (0 secp256k1, 1 secp256r1, 2 Ed25519): the words as stored
typedef void (*entry_fn)(int curve, int win, unsigned j, u32* words);
entry_fn g_entry;

template <class C>
constexpr int curve_id() {
  return C::GLV ? 0 : 1;
}
template <class C>
struct CombHost {
  void load(int i, u32 j, comb_entry& e) const { g_entry(curve_id<C>(), i, j, e.v); }
};
struct EdCombHost {
  void load(int i, u32 j, ed_comb_entry& e) const { g_entry(2, i, j, e.v); }
};
template <class F>
fe canonical(const u32* w) {
  fe x;
  for (int k = 0; k < NL; k++) x.v[k] = w[k];
  BOUNDS_SET(x, LMASK, F::M[NL - 1], mod_ld<F>());
  return x;
}
template <class C>
struct GTabHost {
  void load(u32 idx, fe& x, fe& y) const {
    const u32* e = (C::GLV ? K1_GTABLE : R1_GTABLE) + idx * 20;
    x = canonical<typename C::Fp>(e);
    y = canonical<typename C::Fp>(e + 9);
  }
};
struct BTabHost {
  void load(u32 idx, fe& ypx, fe& ymx, fe& t2d) const {
    const u32* e = ED_BTABLE + idx * 28;
    ypx = canonical<Fe>(e);
    ymx = canonical<Fe>(e + 9);
    t2d = canonical<Fe>(e + 18);
  }
};
// the per-lane table as the kernels keep it: raw limbs
fe words_of(const fe& x) {
  fe r;
  for (int k = 0; k < NL; k++) r.v[k] = x.v[k];
  return r;
}
struct STabHost {
  jac t[8];
  fe x[8], w[8], bx[8];
  void store_full(int e, const jac& p, const fe&) { t[e] = jac{words_of(p.X), words_of(p.Y), words_of(p.Z)}; }
  void load_full(u32 e, jac& p, fe&) const { p = t[e]; }
  void store_affine(int e, const fe& a, const fe& b) { x[e] = words_of(a), w[e] = words_of(b); }
  void load_affine(u32 e, fe& a, fe& b) const { a = x[e], b = w[e]; }
  void store_affine_phi(int e, const fe& a, const fe& b, const fe& c) { store_affine(e, a, b), bx[e] = words_of(c); }
  void load_affine_phi(u32 e, fe& a, fe& b) const { a = bx[e], b = w[e]; }
};
struct CTabHost {
  cached t[16];
  void store(int e, const cached& p) { t[e] = cached{words_of(p.ypx), words_of(p.ymx), words_of(p.z), words_of(p.t2d)}; }
  cached load(u32 e) const { return t[e]; }
};
struct MemHost {
  const u32* w;
  u32 word(u64 i) const { return w[i]; }
};

template <class C>
u32 careful(const u32* sr, const u32* dr, unsigned char* out) {
  secp_pro pro;
  secp_prologue<C>(sr, dr, pro);
  const jacf Q = secp_ladder_careful<C>(pro, GTabHost<C>{});
  if (Q.inf) return ST_INFINITY;
  u32 o[16];
  secp_output<C>(Q.P, o);
  memcpy(out, o, 64);
  return ST_OK;
}

// ---- four lanes: the tables' entries as the lanes read them, then the formulas of quad.hpp ----
template <class C>
struct Quad {
  typedef typename C::Fp F;
  STabHost tab;
  sfe zero = s_from(fe_zero());
  // x on lane 2, w on lane 3 with its sign
  qfe entry(u32 d, bool phi, bool neg) const {
    const u32 e = ((d < 8) ? ~d : d) & 7u;
    return qfe{{zero, zero, s_unraw<F>(phi ? tab.bx[e] : tab.x[e]), s_neg_if((d < 8) != neg, s_unraw<F>(tab.w[e]))}};
  }
  // lanes X, W, ZZ, ZZZ of u1 G + u2 P
  qfe ladder(const secp_pro& pro, bool& exc) {
    const sfe zeta = secp_build_table<C>(pro, tab, exc);
    const sfe one = s_from(fe_from_const(F::ONE));
    constexpr int TOP = C::GLV ? 32 : 63;
    const u32* c1 = C::GLV ? pro.cr1 : pro.c2;
    const bool s1 = C::GLV && pro.sr1;
    qfe acc = q_sel<Q2 | Q3>(qfe{{one, one, one, one}}, q_perm<2, 3, 2, 3>(entry(nibble(c1, TOP), false, s1)));
    if (C::GLV) acc = q_smadd<C>(acc, entry(nibble(pro.cr2, TOP), true, pro.sr2), exc);
    for (int i = TOP - 1; i >= 0; i--) {
      for (int d = 0; d < 4; d++) acc = q_sdbl<C>(acc);
      acc = q_smadd<C>(acc, entry(nibble(c1, i), false, s1), exc);
      if (C::GLV) acc = q_smadd<C>(acc, entry(nibble(pro.cr2, i), true, pro.sr2), exc);
    }
    if (C::GLV) {
      const sfe z2 = s_sqr<F>(zeta), z3 = s_mul<F>(z2, zeta);
      acc.l[2] = s_mul<F>(acc.l[2], z2);
      acc.l[3] = s_mul<F>(acc.l[3], z3);
    }
    for (int i = 0; i < COMB_WINDOWS; i++) {
      const u32 d = (pro.c1[i >> 1] >> ((i & 1) * 16)) & 0xFFFFu;
      comb_entry e;
      g_entry(curve_id<C>(), i, ((d < COMB_ENTRIES) ? ~d : d) & (COMB_ENTRIES - 1u), e.v);
      const sfe w = s_from(fe_from_words(e.v + 8));
      acc = q_smadd<C>(acc, qfe{{zero, zero, s_from(fe_from_words(e.v)),
                                 s_neg_if((d < COMB_ENTRIES) != pro.g_neg, w)}}, exc);
    }
    return acc;
  }
};

// the point of an item with status ST_OK so far, on four lanes: x and y, or an exceptional addition
template <class C>
u32 quad_point(const secp_pro& pro, unsigned char* out) {
  typedef typename C::Fp F;
  Quad<C> q;
  bool exc = false;
  const qfe a = q.ladder(pro, exc);
  if (exc) return ST_PENDING;
  const sfe zi = s_from(finv<F>(s_to_fe<F, 4>(a.l[3])));
  const sfe zz = s_sqr<F>(s_mul<F>(a.l[2], zi));
  const fe half = fnorm_red<F>(s_to_fe<F, 4>(s_mul<F>(a.l[1], zi)));  // 2y
  const fe two = fnorm_red<F>(fscale_nr(fe_from_const(F::ONE), 2));
  u32 w[8], o[16];
  fe_to_words(from_mont<F>(s_to_fe<F, 4>(s_mul<F>(a.l[0], zz))), w);
  words_to_be_bytes(w, o);
  fe_to_words(from_mont<F>(mont_mul<F>(half, finv<F>(two))), w);
  words_to_be_bytes(w, o + 8);
  memcpy(out, o, 64);
  return ST_OK;
}

template <class C>
int recover(const unsigned char* sig, const unsigned char* dig, unsigned char* out, int quad) {
  u32 sr[16], dr[8], o[16];
  memcpy(sr, sig, 64);
  memcpy(dr, dig, 32);
  memset(out, 0, 64);
  u32 st;
  if (quad) {
    secp_pro pro;
    secp_prologue<C, true>(sr, dr, pro);
    st = pro.status;
    if (st == ST_OK) st = quad_point<C>(pro, out);
  } else {
    STabHost tab;
    st = secp_item<C>(sr, dr, tab, CombHost<C>{}, o);
    memcpy(out, o, 64);
  }
  return st == ST_PENDING ? (int)careful<C>(sr, dr, out) | 0x100 : (int)st;
}

template <class C>
int verify(const unsigned char* sig, const unsigned char* dig, const unsigned char* pub) {
  u32 sr[16], dr[8], pr[16];
  memcpy(sr, sig, 64);
  memcpy(dr, dig, 32);
  memcpy(pr, pub, 64);
  secp_pro pro;
  secp_prologue_verify<C, true>(sr, dr, pr, pro);
  if (pro.status != ST_OK) return (int)pro.status;
  STabHost tab;
  bool exc = false;
  const jac P = secp_ladder_wide<C>(pro, tab, CombHost<C>{}, exc);
  if (!exc) return (int)secp_verify_x<C>(P, sr);
  secp_prologue_verify<C>(sr, dr, pr, pro);
  const jacf Q = secp_ladder_careful<C>(pro, GTabHost<C>{});
  return (Q.inf ? (int)ST_INFINITY : (int)secp_verify_x<C>(Q.P, sr)) | 0x100;
}

// the stages' scratch and items; item i at position p of `at`, ~0: none
struct Scratch {
  std::vector<u32>& w;
  template <int N>
  void put(u32 p, const u32* v) const { memcpy(&w[28 * p], v, 16 * N); }
  template <int N, int A = 0>
  void get(u32 p, u32* v) const { memcpy(v + 4 * A, &w[28 * p + 4 * A], 16 * N); }
};
struct Items {
  const u32* at;
  const unsigned char *sigs, *digs;
  uint4* outs;
  unsigned char* st;
  bool item(u32 p) const { return at[p] != ~0u; }
  bool sig(u32 p, u32* w) const { return item(p) && memcpy(w, sigs + 64 * at[p], 64); }
  bool digest(u32 p, u32* w) const { return item(p) && memcpy(w, digs + 32 * at[p], 32); }
  uint4* out(u32 p) const { return item(p) ? outs + 4 * at[p] : nullptr; }
  void status(u32 p, u32 s) const { st[at[p]] = (unsigned char)s; }
};

template <class C, bool VERIFY>
void stages(u32 positions, const u32* at, u32 lanes, const unsigned char* sigs, const unsigned char* digs,
            const unsigned char* pubs, unsigned char* out, unsigned char* st) {
  std::vector<u32> mem(28 * (positions + 1), 0xDEADBEEFu);
  const Scratch sc{mem};
  const Items it{at, sigs, digs, (uint4*)out, st};
  for (u32 l = 0; l < lanes; l++) secp_scalars_lane<C, VERIFY>(l, lanes, positions, it, sc);
  for (u32 p = 0; p < positions; p++) {
    if (!it.item(p)) continue;
    STabHost tab;
    u32 sr[16];
    it.sig(p, sr);
    if constexpr (VERIFY) {
      u32 pr[16];
      memcpy(pr, pubs + 64 * at[p], 64);
      secp_sig g;
      fe x, y;
      u32 s = secp_decode_verify<C>(sr, pr, g, x, y);
      bool exc = false;
      if (s == ST_OK) {
        const jac P = secp_point<C>(p, x, y, sc, tab, CombHost<C>{}, exc);
        s = exc ? (u32)ST_PENDING : secp_verify_x<C>(P, sr);
      }
      st[at[p]] = (unsigned char)s;
    } else {
      secp_recover_point<C>(sr, p, sc, tab, CombHost<C>{});
    }
  }
  if constexpr (!VERIFY)
    for (u32 l = 0; l < lanes; l++) secp_finish_lane<C>(l, lanes, positions, it, sc);
}

// [v]B - [c0]A - [c1]R == identity on four lanes
bool ed_quad(const ed_lat& o, const CTabHost& tab) {
  constexpr int W = ED_LAT_BITS / 4;
  const sfe one = s_from(fe_from_const(Fe::ONE)), zero = s_from(fe_zero());
  fe f = fe_zero();  // 1/2 in Montgomery form
  f.v[0] = 608;
  BOUNDS_SET(f, 608, 0, 609.0L);
  const sfe half = s_from(f);
  auto load = [&](u32 e, bool neg) {
    const cached& c = tab.t[e];
    const sfe a = s_unraw<Fe>(c.ypx), b = s_unraw<Fe>(c.ymx);
    return qfe{{neg ? a : b, neg ? b : a, s_unraw<Fe>(c.z), s_neg_if(neg, s_unraw<Fe>(c.t2d))}};
  };
  auto entry = [&](int base, const u32* c, int i, bool neg) {
    const u32 d = nibble(c, i);
    return load(base + (((d < 8) ? ~d : d) & 7u), (d < 8) != neg);
  };
  qfe acc = q_eadd(qfe{{zero, one, one, zero}}, entry(0, o.ca, W - 1, o.a_neg));
  acc = q_eadd(acc, entry(8, o.cr, W - 1, false));
  for (int i = W - 2; i >= 0; i--) {
    for (int d = 0; d < 4; d++) acc = q_edbl(acc);
    acc = q_eadd(acc, entry(0, o.ca, i, o.a_neg));
    acc = q_eadd(acc, entry(8, o.cr, i, false));
  }
  acc = q_eadd(acc, o.a_fix ? load(0, !o.a_neg) : qfe{{one, one, one, zero}});
  u32 c[8];
  ed_v_carrier(o.v, c);
  for (int i = 0; i < COMB_WINDOWS; i++) {
    const u32 d = (c[i >> 1] >> ((i & 1) * 16)) & 0xFFFFu;
    const bool neg = (d < COMB_ENTRIES) != o.b_neg;
    ed_comb_entry e;
    g_entry(2, i, ((d < COMB_ENTRIES) ? ~d : d) & (COMB_ENTRIES - 1u), e.v);
    const sfe p = s_from(fe_from_words(e.v)), m = s_from(fe_from_words(e.v + 8)), t = s_from(fe_from_words(e.v + 16));
    acc = q_eadd(acc, qfe{{neg ? p : m, neg ? m : p, half, s_neg_if(neg, t)}});
  }
  return fis_zero<Fe>(s_to_fe<Fe, 4>(s_carry(acc.l[0]))) &&
         fis_zero<Fe>(s_to_fe<Fe, 4>(s_carry(s_sub(acc.l[1], acc.l[2]))));
}
}  // namespace

extern "C" {
void wc_entries(entry_fn f) { g_entry = f; }

// status, bit 8 when the careful path decided; quad: the ladder on four lanes
int wc_recover(int curve, const unsigned char* sig, const unsigned char* dig, unsigned char* out, int quad) {
  return curve == 0 ? recover<CurveK1>(sig, dig, out, quad) : recover<CurveR1>(sig, dig, out, quad);
}
int wc_verify(int curve, const unsigned char* sig, const unsigned char* dig, const unsigned char* pub) {
  return curve == 0 ? verify<CurveK1>(sig, dig, pub) : verify<CurveR1>(sig, dig, pub);
}
// items through the stages; 0xFF where an exceptional addition leaves an item to the careful path
void wc_stages(int curve, int verify, unsigned positions, const u32* at, unsigned lanes, const unsigned char* sigs,
               const unsigned char* digs, const unsigned char* pubs, unsigned char* out, unsigned char* st) {
  const auto run = curve == 0 ? (verify ? stages<CurveK1, true> : stages<CurveK1, false>)
                              : (verify ? stages<CurveR1, true> : stages<CurveR1, false>);
  run(positions, at, lanes, sigs, digs, pubs, out, st);
}
// flags: bit 0 verify_strict rules, bit 1 the check on four lanes (of items that have a short pair)
int wc_ed25519(const unsigned char* sig, const unsigned char* pk, const unsigned char* msg, unsigned len, int flags) {
  u32 sr[16], pr[8], k8[8];
  memcpy(sr, sig, 64);
  memcpy(pr, pk, 32);
  std::vector<u32> buf((len + 16) / 4 + 4);
  memcpy(buf.data(), msg, len);
  const MemHost mem{buf.data()};
  CTabHost tab;
  if (!(flags & 2))
    return (int)((flags & 1) ? ed25519_verify_wide<true>(sr, pr, mem, 0, len, tab, BTabHost{}, EdCombHost{})
                             : ed25519_verify_wide<false>(sr, pr, mem, 0, len, tab, BTabHost{}, EdCombHost{}));
  auto check = [&](const u32* k, const u32* s, bool& found) {
    return ed_with_lattice(sr, k, s, tab, found, [&](const ed_lat& o) { return ed_quad(o, tab); });
  };
  if (flags & 1) {
    ed25519_challenge_strict<true>(sr, pr, mem, 0, len, k8);
    return (int)ed25519_verify_with<true>(sr, pr, k8, tab, BTabHost{}, check);
  }
  ed25519_challenge_strict<false>(sr, pr, mem, 0, len, k8);
  return (int)ed25519_verify_with<false>(sr, pr, k8, tab, BTabHost{}, check);
}
}
