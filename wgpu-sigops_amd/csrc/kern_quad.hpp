// kern_quad.hpp -- signature items spread over the four lanes of a quad (quad.hpp), 16 items per
// workgroup of two wavefronts, for calls that would otherwise leave SIMDs idle.
//
// One wavefront (the point wave) lifts the points, builds their tables in LDS and runs the ladder;
// the other (the scalar wave) meanwhile hashes, inverts, splits and recodes the scalars, and hands
// the digits over through LDS. The point wave runs several times as long, so two of them should not
// share a SIMD while another has none: the workgroup makes its point wave the one on the SIMD with
// fewer of them (QuadRole). Fixed roles met on SIMDs from some 500 workgroups on, which ones
// depending on the launch (16,384 recoveries took 864 us instead of 551).
#pragma once
#include "kernels_impl.hpp"
#include "quad.hpp"

namespace sigops {

constexpr u32 QUAD_ITEMS = 16;    // items per workgroup
constexpr u32 QUAD_THREADS = 128;

#if defined(__HIP_DEVICE_COMPILE__)

// this lane's item of the workgroup's, the same for the point and the scalar wave
DEV u32 quad_item() { return (threadIdx.x & 63u) >> 2; }

// The point waves running on every SIMD of the device, counted by the workgroups themselves (load: 4
// words per compute unit, by the hardware's ids; zero when nothing runs).
struct QuadRole {
  u32* mine;    // the counter of this workgroup's point wave
  bool points;  // whether this wavefront is the point wave
  DEV static u32 hw_id() { return __builtin_amdgcn_s_getreg(4 | (31 << 11)); }          // HW_ID
  DEV static u32 xcc_id() { return __builtin_amdgcn_s_getreg(20 | (3 << 11)); }         // XCC_ID, 4 bits
  DEV QuadRole(u32* load, u32* sh) {  // sh: 3 words of LDS; every thread of the workgroup calls
    const u32 w = threadIdx.x >> 6, hw = hw_id();
    if ((threadIdx.x & 63u) == 0) sh[w] = (hw >> 4) & 3u;
    __syncthreads();
    u32* cu = load + 4 * ((xcc_id() & 15u) * 256 + ((hw >> 8) & 255u));
    if (threadIdx.x == 0) {
      const u32 c0 = atomicAdd(cu + sh[0], 1u);
      u32 pick = 0;
      if (c0) {
        const u32 c1 = atomicAdd(cu + sh[1], 1u);
        pick = c1 < c0 ? 1u : 0u;
        atomicSub(cu + sh[1 - pick], 1u);
      }
      sh[2] = pick;
    }
    __syncthreads();
    points = w == sh[2];
    mine = cu + sh[sh[2]];
  }
  DEV void done() const {  // after the workgroup's last work
    if (points && (threadIdx.x & 63u) == 0) atomicSub(mine, 1u);
  }
};

// a table in LDS, as the per-lane tables' interface; lane 0 of the quad writes, all four read
struct QuadSecpTab {
  u32* t;  // this item's 8 entries: x, w, then (building) the factor of Z or (secp256k1) beta x
  static constexpr u32 ENTRY = 27, ITEM = 8 * ENTRY + 1;  // + 1: the items' entries on different banks
  // The quad is within one wavefront, whose LDS accesses execute in their order in the code: what is
  // needed is that the compiler keeps that order across lanes. No instruction comes of it.
  DEV void sync() const {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  DEV void put(u32 e, int f, const fe& x) {
    if (q_lane() == 0) {
#pragma unroll
      for (int k = 0; k < NL; k++) t[e * ENTRY + f * NL + k] = x.v[k];
    }
  }
  DEV fe get(u32 e, int f) const {
    fe r;
#pragma unroll
    for (int k = 0; k < NL; k++) r.v[k] = t[e * ENTRY + f * NL + k];
    return r;
  }
  DEV void store_full(int e, const jac& p, const fe&) {
    put(e, 0, p.X);
    put(e, 1, p.Y);
    put(e, 2, p.Z);
  }
  DEV void load_full(u32 e, jac& p, fe&) const {
    p.X = get(e, 0);
    p.Y = get(e, 1);
    p.Z = get(e, 2);
  }
  DEV void store_affine(int e, const fe& x, const fe& w) {
    put(e, 0, x);
    put(e, 1, w);
  }
  DEV void store_affine_phi(int e, const fe& x, const fe& w, const fe& bx) {
    put(e, 0, x);
    put(e, 1, w);
    put(e, 2, bx);
  }
};

constexpr u32 QUAD_SCALAR_WORDS = 27;  // per item, from the scalar wave; odd, for the banks
struct QuadShared {
  u32 role[4];
  u32 sc[QUAD_ITEMS * QUAD_SCALAR_WORDS];
  u32 tab[QUAD_ITEMS * (16 * 36 + 1)];  // secp: QuadSecpTab; Ed25519: 16 cached entries of 36 words
};

// 4-bit digit of a carrier in LDS, 16-bit digit
DEV u32 quad_digit4(const u32* c, int i) { return (c[i >> 3] >> ((i & 7) * 4)) & 15u; }
DEV u32 quad_digit16(const u32* c, int i) { return (c[i >> 1] >> ((i & 1) * 16)) & 0xFFFFu; }

DEV u32 quad_flags(u32 f, int from) {  // lane `from`'s word on every lane of the quad
  const u32 a = (u32)__builtin_amdgcn_mov_dpp((int)f, 0x00, 0xf, 0xf, true);
  const u32 b = (u32)__builtin_amdgcn_mov_dpp((int)f, 0x55, 0xf, 0xf, true);
  const u32 c = (u32)__builtin_amdgcn_mov_dpp((int)f, 0xAA, 0xf, 0xf, true);
  return from == 0 ? a : (from == 1 ? b : c);
}

// the scalar wave of a secp item: words 0..7 the carrier of u1, 8.. those of u2 (secp256k1: two of 5
// words), 18 the signs (bit 0 G, bits 1 and 2 the R streams)
template <class C, bool VERIFY>
DEV void quad_secp_scalars(const u32 sr[16], const u32 dr[8], u32* sc) {
  typedef typename C::Fn Fn;
  secp_sig g;
  (void)secp_decode_sig<C>(sr, g);  // an invalid signature's scalars are not used
  secp_decode_digest<C>(dr, g);
  const fe inv = finv<Fn>(to_mont<Fn>(fe_from_words(VERIFY ? g.s : g.r)));
  const fe zd = mont_mul<Fn>(to_mont<Fn>(fe_from_words(g.z)), inv);
  const fe u2m = mont_mul<Fn>(to_mont<Fn>(fe_from_words(VERIFY ? g.r : g.s)), inv);
  secp_pro o;
  secp_scalars<C, true>(o, VERIFY ? zd : fneg<Fn>(zd), u2m, fe_zero(), fe_zero());
  if (q_lane() == 0) {
#pragma unroll
    for (int k = 0; k < 8; k++) sc[k] = o.c1[k];
    if constexpr (C::GLV) {
#pragma unroll
      for (int k = 0; k < 5; k++) {
        sc[8 + k] = o.cr1[k];
        sc[13 + k] = o.cr2[k];
      }
      sc[18] = (u32)o.g_neg | ((u32)o.sr1 << 1) | ((u32)o.sr2 << 2);
    } else {
#pragma unroll
      for (int k = 0; k < 8; k++) sc[8 + k] = o.c2[k];
      sc[18] = (u32)o.g_neg | ((u32)o.ry_neg << 1);
    }
  }
}

// a table entry for q_smadd: x (field fx) on lane 2, w on lane 3 with its sign
DEV qfe quad_entry(const QuadSecpTab& tab, u32 d, int fx, bool neg) {
  const u32 e = ((d < 8) ? ~d : d) & 7u;
  const bool w = q_lane() == 3;
  const u32* p = tab.t + e * QuadSecpTab::ENTRY + (w ? (u32)NL : (u32)fx * NL);
  qfe r;
#pragma unroll
  for (int k = 0; k < NL; k++) r.v[k] = (i32)p[k];
  return s_neg_if(w && ((d < 8) != neg), r);
}

// Q = u1 G + u2 P as lanes X, W, ZZ, ZZZ
template <class C>
DEV qfe quad_secp_ladder(const sfe& zeta, const QuadSecpTab& tab, const u32* sc, const uint4* comb, bool& exc) {
  typedef typename C::Fp F;
  const u32 sg = sc[18], q = q_lane();
  const bool g_neg = sg & 1u, r1 = (sg >> 1) & 1u, r2 = (sg >> 2) & 1u;
  const qfe one = s_from(fe_from_const(F::ONE));
  constexpr int TOP = C::GLV ? 32 : 63;
  qfe acc;
  {  // lanes x, w, 1, 1 from an entry's x on lane 2 and w on lane 3
    const qfe e = quad_entry(tab, quad_digit4(sc + 8, TOP), 0, r1);
    acc = q_sel<Q2 | Q3>(one, q_perm<2, 3, 2, 3>(e));
  }
  if constexpr (C::GLV) acc = q_smadd<C>(acc, quad_entry(tab, quad_digit4(sc + 13, TOP), 2, r2), exc);
#pragma unroll 1
  for (int i = TOP - 1; i >= 0; i--) {
    const qfe e1 = quad_entry(tab, quad_digit4(sc + 8, i), 0, r1);
#pragma unroll 1
    for (int d = 0; d < 4; d++) acc = q_sdbl<C>(acc);
    acc = q_smadd<C>(acc, e1, exc);
    if constexpr (C::GLV) acc = q_smadd<C>(acc, quad_entry(tab, quad_digit4(sc + 13, i), 2, r2), exc);
  }
  if constexpr (C::GLV) {  // back from the table's curve: ZZ zeta^2, ZZZ zeta^3
    const sfe z2 = s_sqr<F>(zeta), z3 = s_mul<F>(z2, zeta);
    acc = q_sel<Q2 | Q3>(s_mul<F>(acc, q_sel<Q2>(z2, z3)), acc);
  }
  auto entry = [&](int i, u32* w) {
    const u32 d = quad_digit16(sc, i);
    const u32 j = ((d < COMB_ENTRIES) ? ~d : d) & (COMB_ENTRIES - 1u);
    const uint4* p = comb + 4 * ((u64)i * COMB_ENTRIES + j) + (q == 3 ? 2 : 0);
    const uint4 a = p[0], b = p[1];
    w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w; w[4] = b.x; w[5] = b.y; w[6] = b.z; w[7] = b.w;
  };
  u32 w[8];
  entry(0, w);
#pragma unroll 1
  for (int i = 0; i < COMB_WINDOWS; i++) {
    const sfe x = s_from(fe_from_words(w));
    const bool neg = (quad_digit16(sc, i) < COMB_ENTRIES) != g_neg;
    if (i + 1 < COMB_WINDOWS) entry(i + 1, w);
    acc = q_smadd<C>(acc, s_neg_if(neg && q == 3, x), exc);
  }
  return acc;
}

// the point wave of a recovery: status (ST_PENDING: exceptional addition) and the key, on every lane
template <class C>
DEV u32 quad_recover_out(u32 st, const qfe& acc, bool exc, u32 o[16]) {
  typedef typename C::Fp F;
  if (st == ST_OK && quad_flags(exc, 0)) st = ST_PENDING;
  const sfe X = q_bcast<0>(acc), W = q_bcast<1>(acc), ZZ = q_bcast<2>(acc), ZZZ = q_bcast<3>(acc);
  const sfe zi = s_from(finv<F>(s_to_fe<F, 4>(ZZZ)));
  const sfe zz = s_sqr<F>(s_mul<F>(ZZ, zi));  // 1 / ZZ, as ZZ^3 = ZZZ^2
  const fe x = from_mont<F>(s_to_fe<F, 4>(s_mul<F>(X, zz)));
  const fe w = from_mont<F>(s_to_fe<F, 4>(s_mul<F>(W, zi)));  // 2y
  u32 t[8];
  fe_to_words(x, t);
  words_to_be_bytes(t, o);
  // y = w / 2: (w + p) / 2 for odd w
  fe_to_words(w, t);
  const u32 m = lane_mask(t[0] & 1u);
  u32 c = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const u64 v = (u64)t[k] + (C::p32()[k] & m) + c;
    t[k] = (u32)v;
    c = (u32)(v >> 32);
  }
#pragma unroll
  for (int k = 0; k < 8; k++) t[k] = (t[k] >> 1) | ((k < 7 ? t[k + 1] : c) << 31);
  words_to_be_bytes(t, o + 8);
  const u32 keep = lane_mask(st == ST_OK);
#pragma unroll
  for (int k = 0; k < 16; k++) o[k] &= keep;
  return st;
}

// secp_verify_x on X, ZZ
template <class C>
DEV u32 quad_verify_out(u32 st, const qfe& acc, bool exc, const u32 r[8]) {
  typedef typename C::Fp F;
  if (st != ST_OK) return st;
  if (quad_flags(exc, 0)) return ST_PENDING;
  u32 rn[8];
  words_add(r, C::n32(), rn);  // meaningful only when r < p - n
  const fe X = s_to_fe<F, 4>(q_bcast<0>(acc)), zz = s_to_fe<F, 4>(q_bcast<2>(acc));
  const bool eq1 = feq<F>(X, mont_mul<F>(to_mont<F>(fe_from_words(r)), zz));
  const bool eq2 = feq<F>(X, mont_mul<F>(to_mont<F>(fe_from_words(rn)), zz));
  if (fis_zero<F>(zz)) return ST_INFINITY;
  return (eq1 || (eq2 && words_lt(r, C::pmn32()))) ? ST_OK : ST_MISMATCH;
}

// 16 items of one curve by one workgroup. points: the wavefront's role; valid, i: this quad's item; VERIFY: pubs, status only.
// pend: called with the item that needs the careful pass.
template <class C, bool VERIFY, class Pend>
DEV void quad_secp_tile(QuadShared& sh, bool points, bool valid, u32 i, const uint4* sigs, const uint4* digs, const uint4* pubs,
                        uint4* out, u8* status, const uint4* comb, const Pend& pend) {
  const u32 item = quad_item();
  u32* sc = sh.sc + item * QUAD_SCALAR_WORDS;
  QuadSecpTab tab{sh.tab + item * QuadSecpTab::ITEM};
  u32 sr[16];
  u32 st = ST_OK;
  bool exc = false;
  secp_sig g;
  sfe zeta;
  if (valid) {
    load_words(sigs + 4 * (u64)i, sr, 4);
    if (points) {
      secp_pro pro;
      if constexpr (VERIFY) {
        u32 pr[16];
        load_words(pubs + 4 * (u64)i, pr, 4);
        st = secp_decode_verify<C>(sr, pr, g, pro.rx, pro.ry);
      } else {
        st = secp_decode_sig<C>(sr, g);
        if (!secp_lift<C>(g.r, g.y_odd, pro.rx, pro.ry) && st == ST_OK) st = ST_NO_POINT;
      }
      zeta = secp_build_table<C>(pro, tab, exc);
    } else {
      u32 dr[8];
      load_words(digs + 2 * (u64)i, dr, 2);
      quad_secp_scalars<C, VERIFY>(sr, dr, sc);
    }
  }
  __syncthreads();
  if (!valid || !points) return;
  const qfe acc = quad_secp_ladder<C>(zeta, tab, sc, comb, exc);
  if constexpr (VERIFY) {
    st = quad_verify_out<C>(st, acc, exc, g.r);
  } else {
    u32 o[16];
    st = quad_recover_out<C>(st, acc, exc, o);
    const u32 q = q_lane();
    uint4* po = out + 4 * (u64)i;
    // lane q stores 16 bytes
    u32 w[4];
#pragma unroll
    for (int k = 0; k < 4; k++) w[k] = q == 0 ? o[k] : (q == 1 ? o[4 + k] : (q == 2 ? o[8 + k] : o[12 + k]));
    po[q] = make_uint4(w[0], w[1], w[2], w[3]);
  }
  if (q_lane() == 0) {
    if (st == ST_PENDING) pend(i);
    status[i] = (u8)st;
  }
}

// ---- Ed25519 ----
struct QuadEdTab {  // cached odd multiples in LDS: -A at entries 0..7 (written by lane 0), -R at 8..15 (lane 2)
  u32* t;
  static constexpr u32 ENTRY = 36, ITEM = 16 * ENTRY + 1;
  DEV void store(int e, const cached& p) {
    if ((q_lane() & 1u) == 0) {
      u32* w = t + (e + (q_lane() ? 8 : 0)) * ENTRY;
#pragma unroll
      for (int k = 0; k < NL; k++) {
        w[k] = p.ypx.v[k]; w[9 + k] = p.ymx.v[k]; w[18 + k] = p.z.v[k]; w[27 + k] = p.t2d.v[k];
      }
    }
  }
  // this lane's field of entry e, for q_eadd: Y - X, Y + X, Z, 2dT, or of its negative
  DEV qfe load(u32 e, bool neg) const {
    const u32 q = q_lane();
    const u32 f = q < 2 ? ((1u - q) ^ (u32)neg) : q;
    const u32* w = t + e * ENTRY + f * NL;
    qfe r;
#pragma unroll
    for (int k = 0; k < NL; k++) r.v[k] = (i32)w[k];
    return s_neg_if(neg && q == 3, r);
  }
};

// the scalar wave: words 0..7 the carrier of v = c1 s mod l (odd representative), 8..12 that of c0,
// 13..17 that of c1, 18 flags (bit 0 B negated, 1 the A stream negated, 2 c0 made odd, 3 a short pair
// was found), 19..26 the challenge
template <class Mem>
DEV void quad_ed_scalars(const u32 sr[16], const u32 pr[8], const Mem& mem, u64 off, u32 len, u32* sc) {
  u32 k[8], s[8], cv[8];
  ed25519_challenge(sr, pr, mem, off, len, k);
#pragma unroll
  for (int i = 0; i < 8; i++) s[i] = sr[8 + i];
  ed_lat o;
  const bool ok = ed_lat_scalars(k, s, o);
  ed_v_carrier(o.v, cv);
  if (q_lane() == 0) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      sc[i] = cv[i];
      sc[19 + i] = k[i];
    }
#pragma unroll
    for (int i = 0; i < 5; i++) {
      sc[8 + i] = o.ca[i];
      sc[13 + i] = o.cr[i];
    }
    sc[18] = (u32)o.b_neg | ((u32)o.a_neg << 1) | ((u32)o.a_fix << 2) | ((u32)ok << 3);
  }
}

// [v]B - [c0]A - [c1]R == identity (ed_check_lattice_wide), on every lane
DEV bool quad_ed_check(const QuadEdTab& tab, const u32* sc, const uint4* comb) {
  constexpr int W = ED_LAT_BITS / 4;
  const u32 sg = sc[18], q = q_lane();
  const bool b_neg = sg & 1u, a_neg = (sg >> 1) & 1u, a_fix = (sg >> 2) & 1u;
  const qfe one = s_from(fe_from_const(Fe::ONE));
  const qfe identity = q_keep<Q1 | Q2>(one);
  qfe half = s_from(fe_zero());  // 2^260 mod p
  half.v[0] = 608;
  auto entry = [&](int base, const u32* c, int i, bool neg) {
    const u32 d = quad_digit4(c, i);
    return tab.load(base + (((d < 8) ? ~d : d) & 7u), (d < 8) != neg);
  };
  qfe acc = q_eadd(identity, entry(0, sc + 8, W - 1, a_neg));
  acc = q_eadd(acc, entry(8, sc + 13, W - 1, false));
#pragma unroll 1
  for (int i = W - 2; i >= 0; i--) {
#pragma unroll 1
    for (int d = 0; d < 4; d++) acc = q_edbl(acc);
    acc = q_eadd(acc, entry(0, sc + 8, i, a_neg));
    acc = q_eadd(acc, entry(8, sc + 13, i, false));
  }
  // the A stream ran on |c0| + 1 when |c0| was even: take its point off once, else add the identity
  {
    const qfe id = q_keep<Q0 | Q1 | Q2>(one), e = tab.load(0, !a_neg);
    acc = q_eadd(acc, s_sel(lane_mask(a_fix), e, id));
  }
  auto load = [&](int i, u32* w) {
    const u32 d = quad_digit16(sc, i);
    const u32 j = ((d < COMB_ENTRIES) ? ~d : d) & (COMB_ENTRIES - 1u);
    const bool neg = (d < COMB_ENTRIES) != b_neg;
    // lanes (y - x)/2, (y + x)/2, -, dxy of entries stored as (y + x)/2, (y - x)/2, dxy; lane 2 takes
    // 1/2, so that q_eadd's doubled Z product is Z
    const u32 f = q < 2 ? ((1u - q) ^ (u32)neg) : 2u;
    const uint4* p = comb + ED_COMB_UINT4 * ((u64)i * COMB_ENTRIES + j) + 2 * f;
    const uint4 a = p[0], b = p[1];
    w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w; w[4] = b.x; w[5] = b.y; w[6] = b.z; w[7] = b.w;
  };
  u32 w[8];
  load(0, w);
#pragma unroll 1
  for (int i = 0; i < COMB_WINDOWS; i++) {
    const sfe x = s_from(fe_from_words(w));
    const bool neg = (quad_digit16(sc, i) < COMB_ENTRIES) != b_neg;
    if (i + 1 < COMB_WINDOWS) load(i + 1, w);
    acc = q_eadd(acc, q_sel<Q2>(half, s_neg_if(neg && q == 3, x)));
  }
  // X == 0 (lane 0) and Y == Z (lane 1)
  const qfe z = s_carry(s_sub(acc, q_keep<Q1>(q_bcast<2>(acc))));
  const bool zero = fis_zero<Fe>(s_to_fe<Fe, 4>(z));
  return quad_flags(zero, 0) && quad_flags(zero, 1);
}

// QUAD_ITEMS Ed25519 items by one workgroup; ct, bt: the full-length check's tables (challenges without a
// short pair, about 3 in 10^6)
template <bool STRICT>
DEV void quad_ed_tile(QuadShared& sh, bool points, bool valid, u32 i, const uint4* sigs, const uint4* aux, const u32* msgs,
                      const u64* msg_off, u8* status, const uint4* comb, CTabDev& ct, const BTabGlobal& bt) {
  const u32 item = quad_item();
  u32* sc = sh.sc + item * QUAD_SCALAR_WORDS;
  QuadEdTab tab{sh.tab + item * QuadEdTab::ITEM};
  u32 sr[16], pr[8];
  u32 flags = 0;  // of this lane's point: bit 0 decodes, 1 as compress would have encoded it, 2 small order
  if (valid) {
    load_words(sigs + 4 * (u64)i, sr, 4);
    load_words(aux + 2 * (u64)i, pr, 2);
    if (points) {
      // lanes 0 and 1 take A, lanes 2 and 3 take R
      const u32 m = q_mask<Q2 | Q3>();
      u32 enc[8];
#pragma unroll
      for (int k = 0; k < 8; k++) enc[k] = (sr[k] & m) | (pr[k] & ~m);
      fe x, y;
      flags = ed_decompress(enc, x, y);
      u32 yw[8];
#pragma unroll
      for (int k = 0; k < 8; k++) yw[k] = enc[k];
      yw[7] &= 0x7fffffffu;
      if (words_lt(yw, ED_P32) && !((enc[7] >> 31) != 0 && fis_zero<Fe>(x))) flags |= 2u;
      if (STRICT && ed_small_order(x, y)) flags |= 4u;
      ed_table_odd(tab, 0, fneg<Fe>(x), y);
    } else {
      const u64 off = msg_off[i];
      quad_ed_scalars(sr, pr, MemDev{msgs}, off, (u32)(msg_off[i + 1] - off), sc);
    }
  }
  __syncthreads();
  if (!valid || !points) return;
  const u32 fa = quad_flags(flags, 0), fr = quad_flags(flags, 2);
  u32 s[8];
#pragma unroll
  for (int k = 0; k < 8; k++) s[k] = sr[8 + k];
  u32 st = ED_OK;
  if (!words_lt(s, ED_L32)) st = ED_BAD_S;
  else if (!(fa & 1u)) st = ED_BAD_KEY;
  else if (STRICT && !(fr & 1u)) st = ED_BAD_R;
  else if (STRICT && ((fr | fa) & 4u)) st = ED_SMALL_ORDER;
  bool equal = quad_ed_check(tab, sc, comb) && (fr & 3u) == 3u;
  if (!((sc[18] >> 3) & 1u)) {  // no short pair: the full-length check, the same on the quad's lanes
    u32 k[8];
#pragma unroll
    for (int j = 0; j < 8; j++) k[j] = sc[19 + j];
    equal = ed25519_verify_core<false, false>(sr, pr, k, ct, bt) == ED_OK;
  }
  if (st == ED_OK && !equal) st = ED_MISMATCH;
  if (q_lane() == 0) status[i] = (u8)st;
}

#endif  // __HIP_DEVICE_COMPILE__

}  // namespace sigops
