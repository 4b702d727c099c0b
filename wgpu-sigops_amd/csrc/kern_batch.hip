// kern_batch.hip -- mixed-scheme batch: device-side bucketing plus one persistent kernel.
//
// A batch mixes secp256k1 recoveries, secp256r1 recoveries and Ed25519 verifications with messages
// of any length. The reference has one kernel chain per scheme and fixed 32-byte messages; here:
//   1. k_bucket_hist / k_bucket_scan / k_bucket_scatter sort item indices into buckets (k1, r1, and
//      Ed25519 by SHA-512 block count, so the lanes of a wavefront hash equally long messages), each
//      scheme padded to whole tiles; the buckets are processed in the context's order (its rank
//      table: secp256r1, secp256k1, then Ed25519 by decreasing block count);
//   2. k_batch_run is persistent: every wavefront takes tiles (64 x tile_rounds items of one scheme,
//      claims.hpp), so the scheme is uniform across the wavefront and load balances dynamically; it
//      runs the same per-item code as the plain kernels;
//   3. k_batch_careful finishes secp items whose fast ladder met an exceptional addition.
// A large batch (BATCH_SHARED_FROM) shares its inversions between items: k_batch_scalars computes u1 and
// u2 of the secp items before k_batch_run, several per lane with one inversion, and k_batch_finish makes
// the recovered keys affine after it in the same way. A small one runs on four lanes per item.
// The batch's buffers and n are read from device memory (BatchIO), so the captured graph of these
// launches replays for any buffers and any n up to the context capacity.
#include "claims.hpp"
#include "kern_quad.hpp"

namespace sigops {

static_assert(BATCH_QUAD_LANES == BATCH_QUAD_BLOCKS * 64 && BATCH_QUAD_TILE == QUAD_ITEMS,
              "kernels.hpp's launch shape of a small batch");
static_assert(BATCH_FIRST_TILES == FIRST_TILES_MAX && (4 * NBUCKETS + 4) % 2 == 0, "claims as 64-bit words");

constexpr u32 DUMMY = 0xFFFFFFFFu;

struct BatchArgs {
  const u8* scheme;
  const uint4* sigs;
  const uint4* aux;  // digest (secp) or public key (Ed25519), 32 bytes per item
  const u32* msgs;
  const u64* msg_off;
  uint4* out;
  u8* status;
  u32 n;
  const BatchIO* io;  // the call's buffers and n in device memory; bind_io copies them into the fields above
  u32* counts;      // [NB]
  u32* cursor;      // [NB]
  u32* tile_start;  // [NB + 1] in processing order
  u32* bucket_of;   // [NB] processing rank -> bucket
  u32* order;       // padded item lists, bucket-major in processing order
  u32* tile_counter;  // tiles taken beyond the launch's first
  u32* tile_taken;    // bit per first tile (ClaimWave)
  u32* pend_list;
  u32* pend_count;
  const u8* rank;   // bucket -> processing rank
  u32 tile_items;   // 64 * tile_rounds
  u32 cus;          // compute units if the persistent kernel's grid is a multiple of them, else 0
  ItemScratch sc;   // secp items, by position in `order`
};

// Every kernel starts with bind_io: the per-call buffers come from device memory (written on the
// stream before the launches), the rest of BatchArgs is fixed per context and passed by value, so a
// captured graph of these launches is the same for every call.
DEV void bind_io(BatchArgs& a) {
  const BatchIO& v = *a.io;
  a.scheme = (const u8*)v.scheme;
  a.sigs = (const uint4*)v.sigs;
  a.aux = (const uint4*)v.aux;
  a.msgs = (const u32*)v.msgs;
  a.msg_off = v.msg_off;
  a.out = (uint4*)v.out;
  a.status = (u8*)v.status;
  a.n = v.n;
}

// scheme == NULL: every item is an Ed25519 verification (the plain Ed25519 path hashes through
// the same bucketing, so that its wavefronts hash equally long messages)
DEV u32 item_scheme(const BatchArgs& a, u32 i) { return a.scheme ? a.scheme[i] : 2u; }

DEV u32 item_bucket(const BatchArgs& a, u32 i) {
  const u32 s = item_scheme(a, i);
  if (s == 0) return BUCKET_K1;
  if (s == 1) return BUCKET_R1;
  const u64 len = a.msg_off[i + 1] - a.msg_off[i];
  u64 nb = (64 + len + 17 + 127) >> 7;
  if (nb > ED_BINS) nb = ED_BINS;
  return BUCKET_ED0 + (u32)nb - 1;
}

__global__ __launch_bounds__(256) void k_bucket_hist(BatchArgs a) {
  bind_io(a);
  __shared__ u32 h[NBUCKETS];
  for (u32 t = threadIdx.x; t < NBUCKETS; t += blockDim.x) h[t] = 0;
  __syncthreads();
  const u32 n = a.n;
  for (u32 i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    if (item_scheme(a, i) > 2) continue;
    atomicAdd(&h[item_bucket(a, i)], 1u);
  }
  __syncthreads();
  for (u32 t = threadIdx.x; t < NBUCKETS; t += blockDim.x)
    if (h[t]) atomicAdd(&a.counts[t], h[t]);
}

// By one wavefront (the block's first): tile offsets in processing order from the buckets' counts c
// (LDS), each bucket's first position (start, LDS) and DUMMY padding. Ed25519 buckets that follow each
// other share tiles: a tile belongs to the bucket of its first position, and one that spans two hashes
// a block more on some lanes (5,000 VALU instructions of 340,000). With every bucket padded to whole
// tiles instead, 65,536 items in 9 buckets were 1,029 tiles for 1,024 SIMDs, so that a few took two
// (a host call 2,774 us; 2,157 us with shared tiles).
// One thread walking the ranks took 29 us, longer than the sort's other passes.
DEV void bucket_scan(const BatchArgs& a, const u32* c, u32* start, u32* bucket_of) {
  static_assert(NBUCKETS < 64, "one lane per bucket");
  const u32 lane = threadIdx.x;
  if (lane < 64) {
    if (lane < NBUCKETS) bucket_of[a.rank[lane]] = lane;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const u32 b = lane < NBUCKETS ? bucket_of[lane] : 0;
    const u32 cnt = lane < NBUCKETS ? c[b] : 0;
    auto prefix = [&](u32 v) {  // inclusive, over the ranks
#pragma unroll
      for (u32 d = 1; d < 64; d <<= 1) {
        const u32 u = __shfl_up(v, d);
        if (lane >= d) v += u;
      }
      return v;
    };
    // runs of buckets that share tiles: heads, and the items from the run's head up to this bucket's end
    const u64 ed = __ballot(lane < NBUCKETS && b >= BUCKET_ED0), heads = ~(ed & (ed << 1));
    const u32 items = prefix(cnt), head = 63u - (u32)__builtin_clzll(heads & (~0ull >> (63u - lane)));
    const u32 head_items = __shfl(items - cnt, head), run = items - head_items;
    const bool tail = lane + 1 == NBUCKETS || ((heads >> 1 >> lane) & 1u);
    const u32 tiles = tail && lane < NBUCKETS ? (run + a.tile_items - 1) / a.tile_items : 0;
    const u32 end = prefix(tiles), first = (end - tiles) * a.tile_items + run - cnt;
    if (lane < NBUCKETS) {
      a.tile_start[lane] = (first + a.tile_items - 1) / a.tile_items;
      if (lane == NBUCKETS - 1) a.tile_start[NBUCKETS] = end;
      start[b] = first;
      a.bucket_of[lane] = b;
    }
    if (tiles)
      for (u32 k = first + cnt; k < end * a.tile_items; k++) a.order[k] = DUMMY;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

__global__ __launch_bounds__(64) void k_bucket_scan(BatchArgs a) {
  bind_io(a);
  __shared__ u32 c[NBUCKETS], start[NBUCKETS], bucket_of[NBUCKETS];
  if (threadIdx.x < NBUCKETS) c[threadIdx.x] = a.counts[threadIdx.x];
  __syncthreads();
  bucket_scan(a, c, start, bucket_of);
  if (threadIdx.x < NBUCKETS) a.cursor[threadIdx.x] = start[threadIdx.x];
}

// the whole bucketing of a small batch in one workgroup (clear, histogram, scan, scatter: four
// launches otherwise)
__global__ __launch_bounds__(1024) void k_bucket_small(BatchArgs a) {
  bind_io(a);
  __shared__ u32 c[NBUCKETS], start[NBUCKETS], bucket_of[NBUCKETS];
  if (threadIdx.x < NBUCKETS) c[threadIdx.x] = 0;
  if (threadIdx.x == 0) *a.pend_count = 0;
  __syncthreads();
  const u32 n = a.n;
  for (u32 i = threadIdx.x; i < n; i += blockDim.x) {
    if (item_scheme(a, i) > 2)
      a.status[i] = 0xFD;  // unknown scheme: reported as a canary failure by the host
    else
      atomicAdd(&c[item_bucket(a, i)], 1u);
  }
  __syncthreads();
  bucket_scan(a, c, start, bucket_of);
  __syncthreads();
  for (u32 i = threadIdx.x; i < n; i += blockDim.x)
    if (item_scheme(a, i) <= 2) a.order[atomicAdd(&start[item_bucket(a, i)], 1u)] = i;
}

// the bucket of tile t, the same on every lane of the wavefront
DEV u32 tile_bucket(const BatchArgs& a, u32 t) {
  const u32 lane = threadIdx.x & 63u;
  const bool here = lane < NBUCKETS && a.tile_start[lane] <= t && t < a.tile_start[lane + 1];
  const u64 m = __ballot(here);
  return __builtin_amdgcn_readfirstlane(a.bucket_of[__ffsll((unsigned long long)m) - 1]);
}

// Each workgroup ranks its chunk of 1024 items (4 per thread) per bucket with LDS atomics,
// reserves one range per bucket with a single global atomic, then writes the indices: one global
// atomic per bucket and chunk instead of one per item, on a handful of counters shared by every
// workgroup.
__global__ __launch_bounds__(256) void k_bucket_scatter(BatchArgs a) {
  bind_io(a);
  constexpr u32 PER = 4;
  __shared__ u32 cnt[NBUCKETS];
  __shared__ u32 base[NBUCKETS];
  const u32 n = a.n;
  for (u32 c0 = blockIdx.x * blockDim.x * PER; c0 < n; c0 += gridDim.x * blockDim.x * PER) {
    for (u32 t = threadIdx.x; t < NBUCKETS; t += blockDim.x) cnt[t] = 0;
    __syncthreads();
    u32 bq[PER], rq[PER];
#pragma unroll
    for (u32 q = 0; q < PER; q++) {
      const u32 i = c0 + q * blockDim.x + threadIdx.x;
      bq[q] = NBUCKETS;
      rq[q] = 0;
      if (i < n) {
        if (item_scheme(a, i) > 2) {
          a.status[i] = 0xFD;  // unknown scheme: reported as a canary failure by the host
        } else {
          bq[q] = item_bucket(a, i);
          rq[q] = atomicAdd(&cnt[bq[q]], 1u);
        }
      }
    }
    __syncthreads();
    for (u32 t = threadIdx.x; t < NBUCKETS; t += blockDim.x)
      if (cnt[t]) base[t] = atomicAdd(&a.cursor[t], cnt[t]);
    __syncthreads();
#pragma unroll
    for (u32 q = 0; q < PER; q++)
      if (bq[q] < NBUCKETS) a.order[base[bq[q]] + rq[q]] = c0 + q * blockDim.x + threadIdx.x;
    __syncthreads();
  }
}

DEV void store16(uint4* p, const u32 o[16]) {
#pragma unroll
  for (int c = 0; c < 4; c++) p[c] = make_uint4(o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]);
}

// a secp item; SHARED: up to its Jacobian result in the scratch (k_batch_finish makes it affine)
template <class C, bool SHARED>
DEV void batch_secp_item(const BatchArgs& a, u32 i, u32 pos, STabDev& tab, const CombDev& comb) {
  u32 sr[16], st;
  load_words(a.sigs + 4 * (u64)i, sr, 4);
  if constexpr (SHARED) {
    st = secp_recover_point<C>(sr, pos, a.sc, tab, comb);
  } else {
    u32 dr[8], o[16];
    load_words(a.aux + 2 * (u64)i, dr, 2);
    st = secp_item<C>(sr, dr, tab, comb, o);
    store16(a.out + 4 * (u64)i, o);
    a.status[i] = (u8)st;
  }
  if (st == ST_PENDING) a.pend_list[atomicAdd(a.pend_count, 1u)] = i;
}

// the positions of one curve's tiles as items of the stages around the persistent kernel
struct OrderItems {
  const BatchArgs& a;
  DEV bool sig(u32 p, u32* w) const {
    const u32 i = a.order[p];
    if (i == DUMMY) return false;
    load_words(a.sigs + 4 * (u64)i, w, 4);
    return true;
  }
  DEV bool digest(u32 p, u32* w) const {
    const u32 i = a.order[p];
    if (i == DUMMY) return false;
    load_words(a.aux + 2 * (u64)i, w, 2);
    return true;
  }
  DEV uint4* out(u32 p) const {
    const u32 i = a.order[p];
    return i == DUMMY ? nullptr : a.out + 4 * (u64)i;
  }
  DEV void status(u32 p, u32 st) const { a.status[a.order[p]] = (u8)st; }
};

// u1, u2 of every secp item (secp_scalars_lane), after the bucketing
__global__ __launch_bounds__(256, SIGOPS_WAVES_PER_EU) void k_batch_scalars(BatchArgs a) {
  bind_io(a);
  const u32 id = blockIdx.x * blockDim.x + threadIdx.x, lanes = gridDim.x * blockDim.x;
  const u32 rk = a.rank[BUCKET_K1], rr = a.rank[BUCKET_R1];
  secp_scalars_lane<CurveK1, false>(a.tile_start[rk] * a.tile_items + id, lanes, a.tile_start[rk + 1] * a.tile_items,
                                    OrderItems{a}, a.sc);
  secp_scalars_lane<CurveR1, false>(a.tile_start[rr] * a.tile_items + id, lanes, a.tile_start[rr + 1] * a.tile_items,
                                    OrderItems{a}, a.sc);
}

// affine keys and statuses of every secp item, after the persistent kernel
__global__ __launch_bounds__(256, SIGOPS_WAVES_PER_EU) void k_batch_finish(BatchArgs a) {
  bind_io(a);
  const u32 id = blockIdx.x * blockDim.x + threadIdx.x, lanes = gridDim.x * blockDim.x;
  const u32 rk = a.rank[BUCKET_K1], rr = a.rank[BUCKET_R1];
  secp_finish_lane<CurveK1>(a.tile_start[rk] * a.tile_items + id, lanes, a.tile_start[rk + 1] * a.tile_items,
                            OrderItems{a}, a.sc);
  secp_finish_lane<CurveR1>(a.tile_start[rr] * a.tile_items + id, lanes, a.tile_start[rr + 1] * a.tile_items,
                            OrderItems{a}, a.sc);
}

// a wavefront's view of the launch's tile claims (claims.hpp)
struct ClaimWave {
  u64* taken;    // bit per first tile
  u32* counter;  // tiles taken beyond the first
  u64 free;      // this lane's 64 first tiles as last seen: bits of those not taken
  DEV explicit ClaimWave(const BatchArgs& a) : taken((u64*)a.tile_taken), counter(a.tile_counter), free(0) {}
  DEV static u32 lane() { return threadIdx.x & 63u; }
  DEV u64 take(u32 l, u32 b) { return atomicOr((unsigned long long*)taken + l, 1ull << b); }
  DEV bool own(u32 t) { return __ballot(lane() == 0 && !((take(t >> 6, t & 63) >> (t & 63)) & 1u)) != 0; }
  DEV void look(u32 n) {
    const u32 l0 = 64 * lane();
    const u64 in = n >= l0 + 64 ? ~0ull : (n > l0 ? ~0ull >> (64 - (n - l0)) : 0);
    free = in ? ~__hip_atomic_load(taken + lane(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & in : 0;
  }
  DEV u64 words() const { return __ballot(free != 0); }
  DEV u32 first(u32 l) const { return (u32)__builtin_amdgcn_readlane((int)__builtin_ctzll(free | (1ull << 63)), (int)l); }
  DEV bool claim(u32 l, u32 b) {
    bool won = false;
    if (lane() == l) {
      const u64 old = take(l, b);
      won = !((old >> b) & 1u);
      free &= ~(old | (1ull << b));
    }
    return __ballot(won) != 0;
  }
  DEV u32 beyond() {
    u32 t = 0;
    if (lane() == 0) t = atomicAdd(counter, 1u);
    return __builtin_amdgcn_readfirstlane(t);
  }
};

// The schemes a persistent launch serves (template mask): the mixed batch serves all three; the
// plain Ed25519 entry points serve only Ed25519 (dalek `verify`, or `verify_strict` rules, or `verify`
// with a caller's table of B staged in LDS), so they run the same tile loop, with the challenge
// hashed inside it.
constexpr u32 RUN_K1 = 1, RUN_R1 = 2, RUN_ED = 4, RUN_ED_STRICT = 8, RUN_ED_TABLE = 16;
constexpr u32 RUN_MIXED = RUN_K1 | RUN_R1 | RUN_ED;

// WAVES: waves per SIMD the kernel is built for, which sets its register budget per lane (512 /
// WAVES): 2 by default (256 registers, some values spilled to scratch memory); 1 lets the
// compiler keep them in registers (accumulation registers included) with half the waves to hide
// latencies. The autotuner measures them. SHARED: between k_batch_scalars and k_batch_finish.
template <u32 MASK, int WAVES = SIGOPS_WAVES_PER_EU, bool SHARED = false>
__global__ __launch_bounds__(256, WAVES) void k_batch_run(BatchArgs a, const uint4* __restrict__ comb_k1,
                                                   const uint4* __restrict__ comb_r1,
                                                   const uint4* __restrict__ comb_ed, const uint4* __restrict__ gb,
                                                   uint4* __restrict__ lane_tab, u32 slots) {
  constexpr bool K1 = MASK & RUN_K1, R1 = MASK & RUN_R1, TABLE = MASK & RUN_ED_TABLE;
  constexpr bool ED = MASK & (RUN_ED | RUN_ED_STRICT | RUN_ED_TABLE);
  bind_io(a);
  __shared__ uint4 s_b[TABLE ? BTAB_UINT4 : 1];
  if constexpr (TABLE) {
    for (int t = threadIdx.x; t < BTAB_UINT4; t += blockDim.x) s_b[t] = gb[t];
    __syncthreads();
  }
  const u32 slot = blockIdx.x * blockDim.x + threadIdx.x;
  const u32 lane = threadIdx.x & 63u;
  STabDev jt;
  jt.base = lane_tab;
  jt.slots = slots;
  jt.slot = slot;
  CTabDev ct;
  ct.base = lane_tab;
  ct.slots = slots;
  ct.slot = slot;
  TileClaims claims(a.tile_start[NBUCKETS], a.cus, gridDim.x,
                    __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6)));
  ClaimWave wave(a);
  for (u32 t; (t = claims.next(wave)) != NO_TILE;) {
    const u32 b = tile_bucket(a, t);
    for (u32 k = 0; k < a.tile_items; k += 64) {
      const u32 pos = t * a.tile_items + k + lane;
      const u32 i = a.order[pos];
      if (i == DUMMY) continue;
      if (K1 && b == BUCKET_K1) {
        if constexpr (K1) batch_secp_item<CurveK1, SHARED>(a, i, pos, jt, CombDev{comb_k1});
      } else if (R1 && b == BUCKET_R1) {
        if constexpr (R1) batch_secp_item<CurveR1, SHARED>(a, i, pos, jt, CombDev{comb_r1});
      } else if constexpr (ED) {
        // the challenge is hashed here, inside the persistent kernel: the tile's items have equal
        // SHA-512 block counts (bucketed), and the hash's memory latency hides behind the other
        // waves' field arithmetic instead of idling the GPU in a pass of its own
        u32 sr[16], pr[8];
        load_words(a.sigs + 4 * (u64)i, sr, 4);
        load_words(a.aux + 2 * (u64)i, pr, 2);
        const u64 off = a.msg_off[i];
        const u32 len = (u32)(a.msg_off[i + 1] - off);
        if constexpr (TABLE)
          a.status[i] = (u8)ed25519_verify_item<false, true>(sr, pr, MemDev{a.msgs}, off, len, ct, BTabLds{s_b});
        else
          a.status[i] = (u8)ed25519_verify_wide<(MASK & RUN_ED_STRICT) != 0>(sr, pr, MemDev{a.msgs}, off, len, ct,
                                                                            BTabGlobal{gb}, EdCombDev{comb_ed});
        if (a.out) {
          const u32 zero[16] = {0};
          store16(a.out + 4 * (u64)i, zero);
        }
      }
    }
  }
}

// A small mixed batch: one workgroup per tile of 16 items, four lanes per item (kern_quad.hpp). The
// grid is that of the largest such batch; workgroups beyond the tiles end at once.
__global__ __launch_bounds__(QUAD_THREADS, 2) void k_batch_quad(BatchArgs a, const uint4* __restrict__ comb_k1,
                                                            const uint4* __restrict__ comb_r1,
                                                            const uint4* __restrict__ comb_ed,
                                                            const uint4* __restrict__ gb,
                                                            uint4* __restrict__ lane_tab, u32 slots,
                                                            u32* __restrict__ load) {
#if defined(__HIP_DEVICE_COMPILE__)
  bind_io(a);
  __shared__ QuadShared sh;
  const u32 t = blockIdx.x;
  if (t >= a.tile_start[NBUCKETS]) return;
  const QuadRole role(load, sh.role);
  const u32 b = tile_bucket(a, t);
  const u32 i = a.order[t * QUAD_ITEMS + quad_item()];
  const bool valid = i != DUMMY;
  const auto pend = [&](u32 p) { a.pend_list[atomicAdd(a.pend_count, 1u)] = p; };
  if (b == BUCKET_K1) {
    quad_secp_tile<CurveK1, false>(sh, role.points, valid, i, a.sigs, a.aux, nullptr, a.out, a.status, comb_k1, pend);
  } else if (b == BUCKET_R1) {
    quad_secp_tile<CurveR1, false>(sh, role.points, valid, i, a.sigs, a.aux, nullptr, a.out, a.status, comb_r1, pend);
  } else {
    if (valid && role.points) a.out[4 * (u64)i + q_lane()] = make_uint4(0, 0, 0, 0);
    CTabDev ct;
    ct.base = lane_tab;
    ct.slots = slots;
    ct.slot = blockIdx.x * 64 + (threadIdx.x & 63u);  // the point wave's lanes
    quad_ed_tile<false>(sh, role.points, valid, i, a.sigs, a.aux, a.msgs, a.msg_off, a.status, comb_ed, ct,
                        BTabGlobal{gb});
  }
  role.done();
#endif
}

__global__ __launch_bounds__(64) void k_batch_careful(BatchArgs a, const uint4* __restrict__ gk1,
                                                      const uint4* __restrict__ gr1) {
  bind_io(a);
  const u32 cnt = *a.pend_count;
  for (u32 j = blockIdx.x * blockDim.x + threadIdx.x; j < cnt; j += gridDim.x * blockDim.x) {
    const u32 i = a.pend_list[j];
    u32 sr[16], dr[8], o[16];
    load_words(a.sigs + 4 * (u64)i, sr, 4);
    load_words(a.aux + 2 * (u64)i, dr, 2);
    secp_pro pro;
    jacf Q;
    if (a.scheme[i] == 0) {
      secp_prologue<CurveK1>(sr, dr, pro);
      Q = secp_ladder_careful<CurveK1>(pro, GTabGlobal{gk1});
      if (!Q.inf) secp_output<CurveK1>(Q.P, o);
    } else {
      secp_prologue<CurveR1>(sr, dr, pro);
      Q = secp_ladder_careful<CurveR1>(pro, GTabGlobal{gr1});
      if (!Q.inf) secp_output<CurveR1>(Q.P, o);
    }
    if (Q.inf) {
#pragma unroll
      for (int k = 0; k < 16; k++) o[k] = 0;
    }
    store16(a.out + 4 * (u64)i, o);
    a.status[i] = (u8)(Q.inf ? ST_INFINITY : ST_OK);
  }
}

static __global__ void k_set_io(BatchIO* d, BatchIO v) { *d = v; }

hipError_t launch_set_batch_io(BatchIO* d_io, const BatchIO& v, hipStream_t s) {
  k_set_io<<<1, 1, 0, s>>>(d_io, v);
  return hipGetLastError();
}

static __global__ void k_zero_u32(u32* p, u32 n) {
  for (u32 i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}

static BatchArgs batch_args(const BatchLaunch& L) {
  BatchArgs a{};
  a.io = L.io;
  a.counts = L.work;                    // NBUCKETS
  a.cursor = L.work + NBUCKETS;         // NBUCKETS
  a.tile_start = L.work + 2 * NBUCKETS;  // NBUCKETS + 1
  a.tile_counter = L.work + 3 * NBUCKETS + 1;
  a.pend_count = L.work + 3 * NBUCKETS + 2;
  a.bucket_of = L.work + 3 * NBUCKETS + 4;
  a.tile_taken = L.work + 4 * NBUCKETS + 4;
  a.pend_list = L.pend_list;
  a.order = L.order;
  a.rank = L.rank;
  a.tile_items = 64u * L.tile_rounds;
  const bool whole = L.stage_grid && L.grid % L.stage_grid == 0 && L.grid * 4 <= BATCH_FIRST_TILES;
  a.cus = whole ? L.stage_grid : 0;
  a.sc = ItemScratch{(uint4*)L.scratch, L.scratch_stride};
  return a;
}

// plain Ed25519 verification (io->scheme == NULL, every item Ed25519): the bucketing by SHA-512
// block count, then the persistent kernel serving only Ed25519 tiles, each of which hashes its
// items' challenges and verifies them (dalek `verify`, or `verify_strict` rules)
hipError_t launch_ed_verify(const BatchLaunch& L, bool strict, hipStream_t s) {
  const BatchArgs a = batch_args(L);
  k_zero_u32<<<1, 256, 0, s>>>(L.work, BATCH_WORK_WORDS);
  k_bucket_hist<<<L.aux_grid, 256, 0, s>>>(a);
  k_bucket_scan<<<1, 64, 0, s>>>(a);
  k_bucket_scatter<<<L.aux_grid, 256, 0, s>>>(a);
  const auto run = L.caller_gb ? k_batch_run<RUN_ED_TABLE> : (strict ? k_batch_run<RUN_ED_STRICT> : k_batch_run<RUN_ED>);
  run<<<L.grid, 256, 0, s>>>(a, nullptr, nullptr, (const uint4*)L.comb_ed,
                             (const uint4*)(L.caller_gb ? L.caller_gb : L.gb), (uint4*)L.lane_tab, L.slots);
  return hipGetLastError();
}

// a batch of at most BATCH_QUAD_MAX_ITEMS items; L.lane_tab holds at least
// BATCH_QUAD_LANES lanes
hipError_t launch_batch_small(const BatchLaunch& L, hipStream_t s) {
  BatchArgs a = batch_args(L);
  a.tile_items = QUAD_ITEMS;
  auto mark = [&](int i) -> hipError_t { return L.stage_ev ? hipEventRecord(L.stage_ev[i], s) : hipSuccess; };
  hipError_t e;
  if ((e = mark(0)) != hipSuccess) return e;
  k_bucket_small<<<1, 1024, 0, s>>>(a);
  if ((e = mark(1)) != hipSuccess || (e = mark(2)) != hipSuccess) return e;
  k_batch_quad<<<BATCH_QUAD_BLOCKS, QUAD_THREADS, 0, s>>>(a, (const uint4*)L.comb_k1, (const uint4*)L.comb_r1,
                                                          (const uint4*)L.comb_ed, (const uint4*)L.gb,
                                                          (uint4*)L.lane_tab, L.slots, L.quad_load);
  if ((e = mark(3)) != hipSuccess) return e;
  k_batch_careful<<<64, 64, 0, s>>>(a, (const uint4*)L.gk1, (const uint4*)L.gr1);
  if ((e = mark(4)) != hipSuccess) return e;
  return hipGetLastError();
}

hipError_t launch_batch(const BatchLaunch& L, bool shared, hipStream_t s) {
  const BatchArgs a = batch_args(L);
  // stage events exist only on the eager (timed) path, never under graph capture
  auto mark = [&](int i) -> hipError_t { return L.stage_ev ? hipEventRecord(L.stage_ev[i], s) : hipSuccess; };
  hipError_t e;
  if ((e = mark(0)) != hipSuccess) return e;
  // counters are cleared with a kernel (not a memset node) so the sequence is safe to capture
  k_zero_u32<<<1, 256, 0, s>>>(L.work, BATCH_WORK_WORDS);
  k_bucket_hist<<<L.aux_grid, 256, 0, s>>>(a);
  k_bucket_scan<<<1, 64, 0, s>>>(a);
  k_bucket_scatter<<<L.aux_grid, 256, 0, s>>>(a);
  if ((e = mark(1)) != hipSuccess) return e;
  // (the Ed25519 challenges are hashed inside k_batch_run; the stage stays empty, so that the
  // stage indices of earlier measurements keep their meaning)
  if ((e = mark(2)) != hipSuccess) return e;
  if (shared) k_batch_scalars<<<L.stage_grid, 256, 0, s>>>(a);
  const auto run = !shared        ? k_batch_run<RUN_MIXED>
                   : L.waves == 1 ? k_batch_run<RUN_MIXED, 1, true>
                                  : k_batch_run<RUN_MIXED, SIGOPS_WAVES_PER_EU, true>;
  run<<<L.grid, 256, 0, s>>>(a, (const uint4*)L.comb_k1, (const uint4*)L.comb_r1, (const uint4*)L.comb_ed,
                             (const uint4*)L.gb, (uint4*)L.lane_tab, L.slots);
  if (shared) k_batch_finish<<<L.stage_grid, 256, 0, s>>>(a);
  if ((e = mark(3)) != hipSuccess) return e;
  k_batch_careful<<<64, 64, 0, s>>>(a, (const uint4*)L.gk1, (const uint4*)L.gr1);
  if ((e = mark(4)) != hipSuccess) return e;
  return hipGetLastError();
}

}  // namespace sigops
