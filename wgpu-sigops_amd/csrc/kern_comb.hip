// kern_comb.hip -- builds the wide fixed-base tables (secp.hpp, secp_comb) on the GPU: for every
// 16-bit window i the 32,768 odd multiples of 2^(16 i) G as affine (x, w = 2y).
#include "kernels_impl.hpp"

namespace sigops {

constexpr u32 RUN = 32;                         // entries a lane builds by successive additions
constexpr u32 RUNS = COMB_ENTRIES / RUN;        // lanes per window
constexpr u32 COMB_LANES = COMB_WINDOWS * RUNS;
static_assert(COMB_LANES % 256 == 0, "whole workgroups");

// Lane (i, r): B = 2^(16 i) G by doublings, D = 2B, the run's first entry (2 RUN r + 1) B by double
// and add with the complete law, then RUN - 1 mixed additions of D. T = (2j + 1) B is never +-D
// (2j + 1 is odd and below n), so the incomplete addition is safe. The run's Jacobian points and
// running Z products wait in tmp until one inversion makes them affine.
template <class C>
__global__ __launch_bounds__(256, SIGOPS_WAVES_PER_EU) void k_comb_build(const uint4* __restrict__ gtab,
                                                                    uint4* __restrict__ comb,
                                                                    uint4* __restrict__ tmp_base) {
  typedef typename C::Fp F;
  const u32 lane = blockIdx.x * blockDim.x + threadIdx.x;
  const u32 win = lane / RUNS, r = lane % RUNS;
  LaneTab<9> tmp;
  tmp.base = tmp_base;
  tmp.slots = COMB_LANES;
  tmp.slot = lane;
  jacf B, S;
  fe gx, gy;
  GTabLds{gtab}.load(0, gx, gy);
  B.P.X = gx;
  B.P.Y = gy;
  B.P.Z = fe_from_const(F::ONE);
  B.inf = false;
#pragma unroll 1
  for (u32 d = 0; d < COMB_BITS * win; d++) B = jdbl_c<C>(B);
  S = B;
  const u32 k = 2 * RUN * r + 1;
#pragma unroll 1
  for (int b = 30 - __builtin_clz(k); b >= 0; b--) {
    S = jdbl_c<C>(S);
    if ((k >> b) & 1u) S = jadd_c<C>(S, B);
  }
  fe dx, dy;
  {
    const jacf D = jdbl_c<C>(B);
    const fe zi = finv<F>(D.P.Z), zi2 = mont_sqr<F>(zi);
    dx = mont_mul<F>(D.P.X, zi2);
    dy = mont_mul<F>(D.P.Y, mont_mul<F>(zi2, zi));
  }
  fe run = fe_from_const(F::ONE);
  jac T = S.P;
  bool exc = false;
#pragma unroll 1
  for (u32 e = 0; e < RUN; e++) {
    if (e) {
      T.X = fnorm_red<F>(T.X);
      T.Y = fnorm_red<F>(T.Y);
      T = jmadd<C>(T, dx, dy, exc);
    }
    u32 w[36];
#pragma unroll
    for (int c = 0; c < NL; c++) {
      w[c] = T.X.v[c]; w[9 + c] = T.Y.v[c]; w[18 + c] = T.Z.v[c]; w[27 + c] = run.v[c];
    }
    tmp.put(e, w);
    run = mont_mul<F>(run, T.Z);
  }
  fe inv = finv<F>(run);
#pragma unroll 1
  for (u32 e = RUN; e-- > 0;) {
    u32 w[36];
    tmp.get(e, w);
    fe X, Y, Z, before;
#pragma unroll
    for (int c = 0; c < NL; c++) {
      X.v[c] = w[c]; Y.v[c] = w[9 + c]; Z.v[c] = w[18 + c]; before.v[c] = w[27 + c];
    }
    const fe zi = mont_mul<F>(inv, before);
    inv = mont_mul<F>(inv, Z);
    const fe zi2 = mont_sqr<F>(zi);
    const fe x = mont_mul<F>(X, zi2), y = mont_mul<F>(Y, mont_mul<F>(zi2, zi));
    u32 o[16];
    fe_to_words(fcanon<F>(x), o);
    fe_to_words(fcanon<F>(fnorm_red<F>(fscale_nr(y, 2))), o + 8);
    uint4* p = comb + 4 * ((u64)win * COMB_ENTRIES + RUN * r + e);
#pragma unroll
    for (int c = 0; c < 4; c++) p[c] = make_uint4(o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]);
  }
}

// the same for Ed25519's B, entries ((y + x)/2, (y - x)/2, dxy): every formula is complete
__global__ __launch_bounds__(256, SIGOPS_WAVES_PER_EU) void k_comb_build_ed(const uint4* __restrict__ btab,
                                                                       uint4* __restrict__ comb,
                                                                       uint4* __restrict__ tmp_base) {
  const u32 lane = blockIdx.x * blockDim.x + threadIdx.x;
  const u32 win = lane / RUNS, r = lane % RUNS;
  LaneTab<9> tmp;
  tmp.base = tmp_base;
  tmp.slots = COMB_LANES;
  tmp.slot = lane;
  fe ypx, ymx, t2d;
  BTabLds{btab}.load(0, ypx, ymx, t2d);
  ext B = eadd_niels(ext_identity(), ypx, ymx, t2d, true);
#pragma unroll 1
  for (u32 d = 0; d < COMB_BITS * win; d++) B = edbl(B, true);
  ext S = B;
  const cached Bc = to_cached(B), Dc = to_cached(edbl(B, true));
  const u32 k = 2 * RUN * r + 1;
#pragma unroll 1
  for (int b = 30 - __builtin_clz(k); b >= 0; b--) {
    S = edbl(S, true);
    if ((k >> b) & 1u) S = eadd_cached(S, Bc, true);
  }
  fe run = fe_from_const(Fe::ONE);
#pragma unroll 1
  for (u32 e = 0; e < RUN; e++) {
    if (e) S = eadd_cached(S, Dc, true);
    u32 w[36];
#pragma unroll
    for (int c = 0; c < NL; c++) {
      w[c] = S.X.v[c]; w[9 + c] = S.Y.v[c]; w[18 + c] = S.Z.v[c]; w[27 + c] = run.v[c];
    }
    tmp.put(e, w);
    run = mont_mul<Fe>(run, S.Z);
  }
  fe inv = finv<Fe>(run);
#pragma unroll 1
  for (u32 e = RUN; e-- > 0;) {
    u32 w[36];
    tmp.get(e, w);
    fe X, Y, Z, before;
#pragma unroll
    for (int c = 0; c < NL; c++) {
      X.v[c] = w[c]; Y.v[c] = w[9 + c]; Z.v[c] = w[18 + c]; before.v[c] = w[27 + c];
    }
    const fe zi = mont_mul<Fe>(inv, before);
    inv = mont_mul<Fe>(inv, Z);
    const fe x = mont_mul<Fe>(X, zi), y = mont_mul<Fe>(Y, zi);
    u32 o[24];
    fe half = fe_zero();  // 1/2 in Montgomery form: 2^260 = 32 * 2^255 = 608 (mod p)
    half.v[0] = 608;
    fe_to_words(fcanon<Fe>(mont_mul<Fe>(fadd<Fe>(y, x), half)), o);
    fe_to_words(fcanon<Fe>(mont_mul<Fe>(fsub<Fe>(y, x), half)), o + 8);
    fe_to_words(fcanon<Fe>(mont_mul<Fe>(mont_mul<Fe>(x, y), fe_from_const(ED_D))), o + 16);
    uint4* p = comb + 6 * ((u64)win * COMB_ENTRIES + RUN * r + e);
#pragma unroll
    for (int c = 0; c < 6; c++) p[c] = make_uint4(o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]);
  }
}

size_t comb_bytes(int curve) { return (size_t)COMB_WINDOWS * COMB_ENTRIES * (curve == 2 ? 96 : 64); }
size_t comb_tmp_bytes() { return (size_t)COMB_LANES * RUN * 9 * 16; }

hipError_t launch_comb_build(int curve, const void* gtab, void* comb, void* tmp, hipStream_t s) {
  if (curve == 0)
    k_comb_build<CurveK1><<<COMB_LANES / 256, 256, 0, s>>>((const uint4*)gtab, (uint4*)comb, (uint4*)tmp);
  else if (curve == 1)
    k_comb_build<CurveR1><<<COMB_LANES / 256, 256, 0, s>>>((const uint4*)gtab, (uint4*)comb, (uint4*)tmp);
  else
    k_comb_build_ed<<<COMB_LANES / 256, 256, 0, s>>>((const uint4*)gtab, (uint4*)comb, (uint4*)tmp);
  return hipGetLastError();
}

}  // namespace sigops
