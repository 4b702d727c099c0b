// quad_table_check.cpp -- host (g++) build of secp_build_table over a table that one lane of a quad writes
// and all four read (csrc/kern_quad.hpp keeps it in LDS), with the memory model of that hand-off: what a
// lane wrote reaches the others at the next sync(), and a word may be written again only if a sync()
// lies between the others' reads and the write. Test infrastructure only.
#include <cstring>

#include "secp.hpp"

using namespace sigops;

namespace {
struct SharedTab {
  struct entry {
    fe f[3];
  };
  entry written[8], visible[8];
  bool read_since[8] = {};  // read by the other lanes after the last sync()
  bool race = false;
  bool writer;              // whether this lane sees its own writes at once
  explicit SharedTab(bool w) : writer(w) {}
  void put(int e, const fe& a, const fe& b, const fe& c) {
    race = race || read_since[e];
    written[e] = entry{{a, b, c}};
  }
  void sync() {
    memcpy((void*)visible, (void*)written, sizeof visible);
    memset(read_since, 0, sizeof read_since);
  }
  void store_full(int e, const jac& p, const fe&) { put(e, p.X, p.Y, p.Z); }
  void load_full(u32 e, jac& p, fe&) {
    const entry& x = writer ? written[e] : visible[e];
    read_since[e] = true;
    p.X = x.f[0];
    p.Y = x.f[1];
    p.Z = x.f[2];
  }
  void store_affine(int e, const fe& x, const fe& w) { put(e, x, w, fe_zero()); }
  void store_affine_phi(int e, const fe& x, const fe& w, const fe& bx) { put(e, x, w, bx); }
};

template <class F>
fe load(const unsigned char* be) {
  u32 raw[8], w[8];
  memcpy(raw, be, 32);
  words_from_be_bytes(raw, w);
  return to_mont<F>(fe_from_words(w));
}

// bit 0: a word was written while another lane may still read it; bit 1: the lanes that do not write
// made other entries than the lane that does
template <class C>
int check(const unsigned char* p) {
  secp_pro o;
  o.rx = load<typename C::Fp>(p);
  o.ry = load<typename C::Fp>(p + 32);
  SharedTab a(true), b(false);
  bool exc = false;
  secp_build_table<C>(o, a, exc);
  secp_build_table<C>(o, b, exc);
  bool same = true;
  for (int e = 0; e < 8; e++)
    for (int f = 0; f < 3; f++) same = same && !memcmp(a.written[e].f[f].v, b.written[e].f[f].v, sizeof(u32) * NL);
  return (a.race || b.race ? 1 : 0) | (same ? 0 : 2);
}
}  // namespace

extern "C" int qt_check(int curve, const unsigned char* p) {
  bounds_enabled() = false;  // the words of a lane that reads too early are not a field element
  return curve == 0 ? check<CurveK1>(p) : check<CurveR1>(p);
}
