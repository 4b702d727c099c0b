// kern_secp.hip -- instantiates the secp recovery kernels for one curve (SIGOPS_CURVE = CurveK1
// or CurveR1, set by the build) and provides its launch helper.
#include "kernels_impl.hpp"

#ifndef SIGOPS_CURVE
#error "build with -DSIGOPS_CURVE=CurveK1 or -DSIGOPS_CURVE=CurveR1"
#endif
#define SIGOPS_CAT2(a, b) a##b
#define SIGOPS_CAT(a, b) SIGOPS_CAT2(a, b)

namespace sigops {

static constexpr int CURVE_ID = std::is_same<SIGOPS_CURVE, CurveK1>::value ? 0 : 1;

static u32 stage_blocks(u32 n) { return ((n < STAGE_LANES ? n : STAGE_LANES) + 255) / 256; }

hipError_t SIGOPS_CAT(launch_secp_recover_, SIGOPS_CURVE)(const SecpLaunch& L, const void* sigs, const void* digs,
                                                         void* out, void* status, u32 n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const u32 want = (n + 255) / 256;
  const u32 g = want < L.grid ? want : L.grid;
  const bool quad = !L.gtab8 && n <= QUAD_MAX_ITEMS;
  if (!quad) k_fill_u32<<<1, 64, 0, s>>>(L.pend_count, 0u, 1u);
  if (quad) {
    const hipError_t e = launch_quad_secp(CURVE_ID, false, L, sigs, digs, nullptr, out, status, n, s);
    if (e != hipSuccess) return e;
  } else if (L.gtab8) {
    k_secp_recover<SIGOPS_CURVE><<<g, 256, 0, s>>>((const uint4*)sigs, (const uint4*)digs, (uint4*)out, (u8*)status, n,
                                                  (const uint4*)L.gtab8, (uint4*)L.lane_tab, L.slots, L.pend_list,
                                                  L.pend_count);
  } else {
    const bool shared = n >= SECP_SHARED_FROM;
    const ItemScratch sc{(uint4*)L.scratch, L.scratch_stride};
    if (shared)
      k_secp_scalars<SIGOPS_CURVE, false><<<stage_blocks(n), 256, 0, s>>>((const uint4*)sigs, (const uint4*)digs, n, sc);
    const auto points = shared ? k_secp_points<SIGOPS_CURVE, true> : k_secp_points<SIGOPS_CURVE, false>;
    points<<<g, 256, 0, s>>>((const uint4*)sigs, (const uint4*)digs, (uint4*)out, (u8*)status, n, sc,
                             (const uint4*)L.comb, (uint4*)L.lane_tab, L.slots, L.pend_list, L.pend_count);
    if (shared) k_secp_finish<SIGOPS_CURVE><<<stage_blocks(n), 256, 0, s>>>((uint4*)out, (u8*)status, n, sc);
  }
  k_secp_careful<SIGOPS_CURVE><<<64, 64, 0, s>>>((const uint4*)sigs, (const uint4*)digs, (uint4*)out, (u8*)status,
                                                (const uint4*)(L.gtab8 ? L.gtab8 : L.gtab), L.pend_list, L.pend_count);
  return hipGetLastError();
}

hipError_t SIGOPS_CAT(launch_secp_verify_, SIGOPS_CURVE)(const SecpLaunch& L, const void* sigs, const void* digs,
                                                        const void* pubs, void* status, u32 n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const u32 want = (n + 255) / 256;
  const u32 g = want < L.grid ? want : L.grid;
  if (n <= QUAD_MAX_ITEMS) {
    const hipError_t e = launch_quad_secp(CURVE_ID, true, L, sigs, digs, pubs, nullptr, status, n, s);
    if (e != hipSuccess) return e;
  } else {
    const bool shared = n >= SECP_SHARED_FROM;
    const ItemScratch sc{(uint4*)L.scratch, L.scratch_stride};
    k_fill_u32<<<1, 64, 0, s>>>(L.pend_count, 0u, 1u);
    if (shared)
      k_secp_scalars<SIGOPS_CURVE, true><<<stage_blocks(n), 256, 0, s>>>((const uint4*)sigs, (const uint4*)digs, n, sc);
    const auto verify = shared ? k_secp_verify<SIGOPS_CURVE, true> : k_secp_verify<SIGOPS_CURVE, false>;
    verify<<<g, 256, 0, s>>>((const uint4*)sigs, (const uint4*)digs, (const uint4*)pubs, (u8*)status, n, sc,
                             (const uint4*)L.comb, (uint4*)L.lane_tab, L.slots, L.pend_list, L.pend_count);
  }
  k_secp_verify_careful<SIGOPS_CURVE><<<64, 64, 0, s>>>((const uint4*)sigs, (const uint4*)digs, (const uint4*)pubs,
                                                       (u8*)status, (const uint4*)L.gtab, L.pend_list, L.pend_count);
  return hipGetLastError();
}

}  // namespace sigops
