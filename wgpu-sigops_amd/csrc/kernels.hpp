// kernels.hpp -- launch helpers shared by the runtime (internal to libsigops).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace sigops {

typedef uint8_t u8;

constexpr uint32_t GTAB_ENTRIES = 1u << (8 - 1);  // odd multiples 1..255 of G
constexpr uint32_t BTAB_ENTRIES = 1u << (8 - 1);  // odd multiples 1..255 of B (and as many of [2^136] B)
// the Ed25519 fixed-base tables as held in HBM and LDS: odd multiples of B, then of [2^136] B,
// 7 uint4 per entry
constexpr uint32_t BTAB_UINT4 = 2 * BTAB_ENTRIES * 7;
constexpr uint32_t SECP_LANE_TAB_BYTES = 8 * 7 * 16;  // 8 entries x 7 uint4 (Jacobian, then affine)
constexpr uint32_t ED_LANE_TAB_BYTES = 16 * 9 * 16;   // 16 cached entries (-A, then -R) x 9 uint4

constexpr uint32_t ITEM_SCRATCH_BYTES = 7 * 16;       // per position of a secp call (ItemScratch)

// what the secp launches use of a context. gtab8: a caller's converted table (128 odd multiples), or
// null for the resident tables: the wide ones (comb) and, for the careful pass, gtab.
struct SecpLaunch {
  const void* gtab;
  const void* gtab8;
  const void* comb;
  void* scratch;
  uint32_t scratch_stride;  // positions the scratch holds, at least n
  void* lane_tab;
  uint32_t slots, grid;
  uint32_t* pend_list;
  uint32_t* pend_count;
  uint32_t* quad_load;  // QUAD_LOAD_WORDS, shared by every launch on the device
};
hipError_t launch_secp_recover_CurveK1(const SecpLaunch& L, const void* sigs, const void* digs, void* out,
                                      void* status, uint32_t n, hipStream_t s);
hipError_t launch_secp_recover_CurveR1(const SecpLaunch& L, const void* sigs, const void* digs, void* out,
                                      void* status, uint32_t n, hipStream_t s);

// verification with a known public key (64 bytes X || Y per item); status only; resident tables
hipError_t launch_secp_verify_CurveK1(const SecpLaunch& L, const void* sigs, const void* digs, const void* pubs,
                                     void* status, uint32_t n, hipStream_t s);
hipError_t launch_secp_verify_CurveR1(const SecpLaunch& L, const void* sigs, const void* digs, const void* pubs,
                                     void* status, uint32_t n, hipStream_t s);

// Small calls (kern_quad.hpp) take four lanes per item: up to this many items the point waves are at
// most one per SIMD, and the call is as long as one item. Measured (us per device call, four lanes
// against one lane per item): secp256k1 recovery 473 / 807 at 1,000 items, 551 / 812 at 16,384, 1,015
// / 812 at 20,011; secp256r1 verification 563 / 1,140, 656 / 1,148, 1,255 / 1,148; Ed25519 with
// messages up to 200 bytes 320 / 990, 543 / 1,000 (one lane per item with its bucketing). Beside other calls
// four lanes take more of the GPU: on three streams secp256r1 recovery 386 us a call at 6,000 items, 598 at
// 12,000 and 808 at 16,384, one lane per item 651 at each; the line is for calls alone.
constexpr uint32_t QUAD_MAX_ITEMS = 16384;
// Plain secp calls from this size on share their inversions between items, in a stage before and one after
// the ladders (65,536 lanes; below that a lane has one item and shares nothing). us per call, shared / not:
// secp256r1 recovery alone 1,282 / 1,245 at 20,011 items, 1,312 / 1,273 at 65,536, 2,284 / 2,278 at 131,072,
// 9,089 / 9,196 at 524,288; secp256k1 3,077 / 3,165 at 200,000, 5,912 / 6,104 at 524,288. On three streams
// secp256r1 852 / 654 at 20,011, 2,094 / 2,115 at 131,072, 3,302 / 3,370 at 200,000.
constexpr uint32_t SECP_SHARED_FROM = 3u << 16;
// the counters that keep point waves apart (kern_quad.hpp, QuadRole), zero at first
constexpr uint32_t QUAD_LOAD_WORDS = 16 * 256 * 4;
// pend_count is cleared; the careful pass is the caller's (launch_secp_*_careful)
hipError_t launch_quad_secp(int curve, bool verify, const SecpLaunch& L, const void* sigs, const void* digs,
                            const void* pubs, void* out, void* status, uint32_t n, hipStream_t s);
struct EdQuadLaunch {
  const void* sigs;
  const void* keys;
  const void* msgs;
  const uint64_t* msg_off;
  void* status;
  const void* comb;
  const void* gb;     // resident table, for the full-length check
  void* lane_tab;
  uint32_t slots;     // at least QUAD_MAX_ITEMS / 16 * 64
  uint32_t* quad_load;
};
hipError_t launch_quad_ed(bool strict, const EdQuadLaunch& L, uint32_t n, hipStream_t s);

// the wide fixed-base table of a curve (0 secp256k1, 1 secp256r1, 2 Ed25519) from its resident table; tmp:
// comb_tmp_bytes() that may be freed once the stream has passed the launch
size_t comb_bytes(int curve);
size_t comb_tmp_bytes();
hipError_t launch_comb_build(int curve, const void* gtab, void* comb, void* tmp, hipStream_t s);

// ---- mixed batch ----
constexpr uint32_t BUCKET_K1 = 0, BUCKET_R1 = 1, BUCKET_ED0 = 2;
constexpr uint32_t ED_BINS = 40;  // Ed25519 buckets by SHA-512 block count 1..40 (40 = "40 or more")
constexpr uint32_t NBUCKETS = 2 + ED_BINS;
constexpr uint32_t BATCH_FIRST_TILES = 4096;  // bits of the first tiles' claims: 1,024 workgroups
// counts, cursors, tile starts, tile ctr, pending ctr, (one unused, to align the claims), buckets, claims
constexpr uint32_t BATCH_WORK_WORDS = 4 * NBUCKETS + 4 + BATCH_FIRST_TILES / 32;
constexpr uint32_t MAX_TILE_ROUNDS = 4;

// The buffers of one batch call and its size. The host writes them into device memory
// (launch_set_batch_io, stream-ordered) before the launches, and the kernels read them from
// there, so one captured graph per context serves every call whatever buffers it passes.
struct BatchIO {
  const void* scheme;  // NULL: every item is an Ed25519 verification
  const void* sigs;
  const void* aux;
  const void* msgs;
  const uint64_t* msg_off;
  void* out;  // NULL for the plain Ed25519 path
  void* status;
  uint32_t n;
};
hipError_t launch_set_batch_io(BatchIO* d_io, const BatchIO& v, hipStream_t s);

struct BatchLaunch {
  const BatchIO* io;    // device copy of the call's buffers
  uint32_t* work;       // BATCH_WORK_WORDS
  uint32_t* order;      // capacity max_batch + NBUCKETS * 64 * tile_rounds
  uint32_t* pend_list;  // capacity max_batch
  const uint8_t* rank;  // NBUCKETS
  const void* gk1;
  const void* gr1;
  const void* gb;
  const void* comb_k1;
  const void* comb_r1;
  const void* comb_ed;
  const void* caller_gb;    // plain Ed25519 only: a caller's converted table of B, or null
  uint32_t* quad_load;
  void* scratch;            // ItemScratch of the secp items, by position in `order`
  uint32_t scratch_stride;  // its positions: the capacity of `order`
  void* lane_tab;
  uint32_t slots, grid, aux_grid, tile_rounds;
  uint32_t stage_grid;   // compute units: blocks of the stages that share an inversion between items
  uint32_t waves;        // mixed batch: waves per SIMD the persistent kernel is built for (1 or 2); 1: shared only
  hipEvent_t* stage_ev;  // null, or 5 events recorded before, between and after the 4 stages
};

// shared: the secp items' inversions are shared between items, in a stage before and one after the
// persistent kernel
hipError_t launch_batch(const BatchLaunch& L, bool shared, hipStream_t s);
// Batches from this size on share their inversions. A lane of the stages takes n / 65,536 items, and what
// that saves has to pay for two launches: each waits for the GPU to drain, and beside other batches for
// wavefronts to end. us per batch (messages up to 4 KB), shared / not: alone 1,371 / 1,294 at 20,000 items,
// 1,744 / 1,572 at 65,536, 2,502 / 2,323 at 131,072, 4,174 / 4,138 at 262,144, 7,915 / 7,533 at 524,288,
// 11,464 / 11,195 at 800,000, 13,801 / 14,451 at 2^20; on three streams at once 786 / 499, 1,029 / 890,
// 1,862 / 1,722, 3,717 / 3,386, 6,949 / 6,718, 10,383 / 10,272, 13,362 / 13,507.
constexpr uint32_t BATCH_SHARED_FROM = 13u << 16;
// A small mixed batch: four lanes per item, one workgroup per tile of 16 items of one bucket. Measured
// (us per device call, four lanes against one lane per item, messages up to 4 KB): 690 / 1,303 at 2,000
// items, 705 / 1,325 at 8,000, 1,182 / 1,326 at 16,000, 1,200 / 1,337 at 20,000, 1,451 / 1,364 at 24,000.
constexpr uint32_t BATCH_QUAD_MAX_ITEMS = 20480;
// The same beside other batches, which four lanes per item take more of the GPU from: per batch on three
// streams 363 / 453 at 6,000, 409 / 469 at 10,000, 463 / 475 at 12,000, 534 / 477 at 14,000, 751 / 493 at 20,000.
constexpr uint32_t BATCH_QUAD_MAX_BESIDE = 12288;
constexpr uint32_t BATCH_QUAD_TILE = 16;
// The launch's grid holds more items than the rules send: cut to 20,480 items, a burst of 24 requests on
// the server took longer (p90 2,302 us against 2,236; the reason was not found).
constexpr uint32_t BATCH_QUAD_CAPACITY = 24576;
static_assert(BATCH_QUAD_MAX_ITEMS <= BATCH_QUAD_CAPACITY && BATCH_QUAD_MAX_BESIDE <= BATCH_QUAD_CAPACITY, "grid");
constexpr uint32_t BATCH_QUAD_BLOCKS = BATCH_QUAD_CAPACITY / BATCH_QUAD_TILE + NBUCKETS;
constexpr uint32_t BATCH_QUAD_LANES = BATCH_QUAD_BLOCKS * 64;  // point lanes
hipError_t launch_batch_small(const BatchLaunch& L, hipStream_t s);
// plain Ed25519 verification of an all-Ed25519 batch (io->scheme == NULL, io->out == NULL): the
// bucketing, then the persistent kernel on Ed25519 tiles with the challenges hashed inside it;
// strict: ed25519-dalek verify_strict rules (resident table only)
hipError_t launch_ed_verify(const BatchLaunch& L, bool strict, hipStream_t s);

// ---- streamed tiles: the host packs tiles into pinned, device-mapped memory while one persistent
// launch drains them (layout in stream_host.hpp). A streamed batch fills positions 0.. of the
// layout once; a serving ring reuses positions base + t (mod positions) for the launch's tile t ----
constexpr uint32_t STREAM_CLOSED = 1u << 31;  // in the published count: no tile beyond it will come
// A launch drains up to STREAM_QUEUES queues of tiles (a serving ring: one per scheme; a batch: one).
// Device words of a streamed launch, cleared by the launch: u32 [q] the claim counter of queue q,
// [STREAM_CTR_PENDING] the pending count; u64 at byte 64 the wall-clock time of the last read of
// the pinned counts, at byte 72 the stop flag seen there; STREAM_MIRRORS copies of the pinned
// counts (u64 per queue) from byte 256 on, 256 bytes apart
constexpr uint32_t STREAM_QUEUES = 3;
constexpr uint32_t STREAM_CTR_PENDING = 4;
constexpr uint32_t STREAM_MIRRORS = 8;
constexpr uint32_t STREAM_CTR_BYTES = 256 + STREAM_MIRRORS * 256;
struct StreamLaunch {
  const void* desc;      // 16-byte tile descriptors, one per position (pinned, or an HBM copy)
  const void* in;        // inputs, [position][6][64] 16-byte chunks (pinned, or an HBM copy)
  const uint32_t* mrel;  // per position lane, message start relative to the tile's
  const uint32_t* mlen;  // per position lane, message length
  const void* hmsgs;     // the tiles' messages: pinned, copied by each tile to dmsgs; or equal to dmsgs
                         // when the host has copied them to HBM before publishing the tile
  void* dmsgs;           // device: the messages the hash reads (same offsets)
  uint64_t msg_cap;      // bytes of hmsgs and dmsgs: a tile's region [m0, m0 + bytes + 16) lies within
  void* out;             // pinned: results, [position][4][64] 16-byte chunks
  uint8_t* st;           // pinned: statuses, [position][64]
  uint64_t* tile_done;   // pinned: per position, seq << 32 | the descriptor's tag once the tile's results are written
  const uint64_t* ready; // pinned, per queue: seq << 32 | tiles published so far, | STREAM_CLOSED at the end
  const uint32_t* qpos;  // pinned: per queue, mask + 1 entries: position of the queue's tile t (t & mask);
                         // null: one queue whose tile t sits at position (base + t) & mask
  uint32_t nq;           // queues (1 .. STREAM_QUEUES)
  uint32_t split0, split1;  // home queue of block b: 0 if b % 256 < split0, 1 if < split1, else 2
  const uint32_t* stop;  // pinned: nonzero makes waiting waves give up
  uint32_t* err;         // pinned: set to 1 by a wave that gave up waiting
  uint32_t* ctr;         // device: STREAM_CTR_BYTES of counters and polling state (cleared by the launch)
  uint32_t* pend_list;   // device: position lanes (position * 64 + lane) the careful pass redoes
  uint32_t pend_cap;     // entries pend_list holds (further pending lanes are not recorded)
  const void* gk1;       // resident tables, for the careful pass
  const void* gr1;
  const void* gb;
  const void* comb_k1;   // wide tables
  const void* comb_r1;
  const void* comb_ed;
  void* lane_tab;
  uint32_t slots;        // tiles a wavefront may take at most
  uint32_t base, mask;   // see qpos (a batch: 0 and ~0)
  uint32_t seq, lane_slots, grid;
  uint64_t poll_ticks;   // wall-clock ticks between reads of the pinned count (device-wide)
  uint64_t limit_ticks;  // a wave that waits this long for a tile gives up
};
hipError_t launch_stream(const StreamLaunch& L, hipStream_t s);
// the polling interval (2 us) and the give-up time (15 s) of a streamed launch in the device's
// wall-clock ticks
inline void stream_poll_ticks(int device, StreamLaunch& L) {
  int khz = 0;
  if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device) != hipSuccess || khz <= 0) khz = 100000;
  L.poll_ticks = (uint64_t)khz * 2 / 1000;
  L.limit_ticks = (uint64_t)khz * 15000;
}

// what a serving ring borrows from a context: the resident tables, the lane tables and the launch
// shape they are sized for, the processing order of the buckets, and the context's stream
struct RingResources {
  const void* gk1;
  const void* gr1;
  const void* gb;
  const void* comb_k1;
  const void* comb_r1;
  const void* comb_ed;
  void* lane_tab;
  uint32_t lane_slots, grid;
  const uint32_t* bucket_order;  // processing rank -> bucket, NBUCKETS entries
  hipStream_t stream;
};


// SHA-256: digests of messages (Fuel Message::new) and addresses of 64-byte public keys.
// work: MSG_WORK_WORDS device words (cleared by the launch); order: n words, the longest-first
// processing order of the messages
constexpr uint32_t MSG_BINS = 66;  // message ordering bins by SHA-256 block count (66 = "66 or more")
constexpr uint32_t MSG_WORK_WORDS = 1 + 2 * MSG_BINS;
hipError_t launch_message_new(const void* msgs, const uint64_t* off, uint32_t n, void* out, uint32_t* work,
                              uint32_t* order, uint32_t grid, uint32_t cus, hipStream_t s);
hipError_t launch_fuel_address(const void* pubs, const void* status, uint32_t n, void* out, uint32_t grid,
                               hipStream_t s);

// caller-supplied generator tables in the reference's layout -> this engine's table (flags[0] = 0
// when the table passes its checks); lbits in 11..15
hipError_t launch_table_secp(int curve, const uint32_t* limbs, uint32_t lbits, void* gtab_out, uint32_t* flags,
                             hipStream_t s);
hipError_t launch_table_ed(const uint32_t* limbs, uint32_t lbits, void* btab_out, uint32_t* flags, hipStream_t s);

hipError_t launch_gen_secp(int curve, uint64_t seed, uint32_t n, uint32_t ppm, const void* gtab, void* sigs,
                           void* digs, void* pubs, void* corrupted, uint32_t grid, hipStream_t s);
hipError_t launch_gen_ed25519(uint64_t seed, uint32_t n, uint32_t ppm, const void* btab, const uint64_t* msg_off,
                              void* msgs, void* sigs, void* pks, void* corrupted, uint32_t grid, hipStream_t s);

}  // namespace sigops

// the resources of a context that a serving ring launches with (sigops_api.hip); SIGOPS_OK or an
// error code
struct sigops_ctx;
int sigops_ring_resources(sigops_ctx* c, sigops::RingResources* r);
// whether the next mixed batches on this context run beside others (a server's other slots)
void sigops_set_beside(sigops_ctx* c, bool beside);

