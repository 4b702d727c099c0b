// kern_quad.hip -- the plain entry points' kernels for small calls (kern_quad.hpp): one workgroup per 16
// items, no other launch but the careful pass.
#include "kern_quad.hpp"

namespace sigops {

template <class C, bool VERIFY>
__global__ __launch_bounds__(QUAD_THREADS, 2) void k_quad_secp(const uint4* __restrict__ sigs,
                                                           const uint4* __restrict__ digs,
                                                           const uint4* __restrict__ pubs, uint4* __restrict__ out,
                                                           u8* __restrict__ status, u32 n,
                                                           const uint4* __restrict__ comb, u32* __restrict__ pend_list,
                                                           u32* __restrict__ pend_count, u32* __restrict__ load) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ QuadShared sh;
  const QuadRole role(load, sh.role);
  const u32 i = blockIdx.x * QUAD_ITEMS + quad_item();
  quad_secp_tile<C, VERIFY>(sh, role.points, i < n, i, sigs, digs, pubs, out, status, comb,
                            [&](u32 p) { pend_list[atomicAdd(pend_count, 1u)] = p; });
  role.done();
#endif
}

template <bool STRICT>
__global__ __launch_bounds__(QUAD_THREADS, 2) void k_quad_ed(const uint4* __restrict__ sigs,
                                                         const uint4* __restrict__ keys,
                                                         const u32* __restrict__ msgs,
                                                         const u64* __restrict__ msg_off, u8* __restrict__ status,
                                                         u32 n, const uint4* __restrict__ comb,
                                                         const uint4* __restrict__ gb, uint4* __restrict__ lane_tab,
                                                         u32 slots, u32* __restrict__ load) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ QuadShared sh;
  const QuadRole role(load, sh.role);
  const u32 i = blockIdx.x * QUAD_ITEMS + quad_item();
  CTabDev ct;
  ct.base = lane_tab;
  ct.slots = slots;
  ct.slot = blockIdx.x * 64 + (threadIdx.x & 63u);  // the point wave's lanes
  quad_ed_tile<STRICT>(sh, role.points, i < n, i, sigs, keys, msgs, msg_off, status, comb, ct, BTabGlobal{gb});
  role.done();
#endif
}

static __global__ void k_clear_u32(u32* p) { *p = 0; }

// u32 words of the pending list are free from an earlier call: only the count is cleared
hipError_t launch_quad_secp(int curve, bool verify, const SecpLaunch& L, const void* sigs, const void* digs,
                            const void* pubs, void* out, void* status, uint32_t n, hipStream_t s) {
  const u32 g = (n + QUAD_ITEMS - 1) / QUAD_ITEMS;
  k_clear_u32<<<1, 1, 0, s>>>(L.pend_count);
  auto go = [&](auto kernel) {
    kernel<<<g, QUAD_THREADS, 0, s>>>((const uint4*)sigs, (const uint4*)digs, (const uint4*)pubs, (uint4*)out,
                                      (u8*)status, n, (const uint4*)L.comb, L.pend_list, L.pend_count, L.quad_load);
  };
  if (curve == 0)
    verify ? go(k_quad_secp<CurveK1, true>) : go(k_quad_secp<CurveK1, false>);
  else
    verify ? go(k_quad_secp<CurveR1, true>) : go(k_quad_secp<CurveR1, false>);
  return hipGetLastError();
}

hipError_t launch_quad_ed(bool strict, const EdQuadLaunch& L, uint32_t n, hipStream_t s) {
  const u32 g = (n + QUAD_ITEMS - 1) / QUAD_ITEMS;
  auto go = [&](auto kernel) {
    kernel<<<g, QUAD_THREADS, 0, s>>>((const uint4*)L.sigs, (const uint4*)L.keys, (const u32*)L.msgs, L.msg_off,
                                      (u8*)L.status, n, (const uint4*)L.comb, (const uint4*)L.gb, (uint4*)L.lane_tab,
                                      L.slots, L.quad_load);
  };
  strict ? go(k_quad_ed<true>) : go(k_quad_ed<false>);
  return hipGetLastError();
}

}  // namespace sigops
