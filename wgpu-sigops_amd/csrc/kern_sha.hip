// kern_sha.hip -- SHA-256 on the device: Fuel's Message::new over raw data, and addresses of
// recovered public keys (SHA-256 of the 64-byte X || Y).
#include "kernels_impl.hpp"
#include "sha256.hpp"

namespace sigops {

// Longest messages first. Lanes take message positions by grid stride, so the launch ends with
// the last round of positions; in index order a lane that got a long message in that round kept
// the launch running, alone, for its remaining blocks. A counting sort by block count therefore
// orders the positions longest first: bin 0 holds messages of MSG_BINS or more blocks, bin b > 0
// those of MSG_BINS - b blocks. The work words hold the bin counts, the bin cursors and a word of
// flags: MSG_SORTED when more than one bin is used (with a single block count the index order is
// kept and the scatter does nothing), MSG_PAIRS when the launch is bound by its longest messages.
constexpr u32 MW_COUNT = 0, MW_CURSOR = MSG_BINS, MW_FLAG = 2 * MSG_BINS;
constexpr u32 MSG_SORTED = 1, MSG_PAIRS = 2;

// Two wavefronts to a message halve the instructions on a message's chain and add to the launch's
// total (LDS, barriers). The longest message takes `longest` steps of a wavefront's time per block, all
// messages together total / (256 cus) of them. Measured, one wavefront against two (us; 256 compute
// units, log-uniform lengths), at total / (256 cus longest) = 0.4: 245 / 161 (209,715 messages of up to
// 4,096 bytes); 1.1: 318 / 268 (524,288 of them); 1.4: 51 / 49 (300,000 of up to 200 bytes); 1.6: 103 / 102
// (524,288 of up to 700 bytes); 2.4: 68 / 74 (524,288 of up to 200 bytes).
DEV u32 msg_flags(u32 used, u64 total, u32 longest, u32 cus) {
  return (used > 1 ? MSG_SORTED : 0) | (2 * total < 3 * (u64)longest * (256 * cus) ? MSG_PAIRS : 0);
}

DEV u32 msg_bin(const u64* off, u32 i) {
  const u64 nb = (off[i + 1] - off[i] + 8) / 64 + 1;  // SHA-256 blocks, padding included
  return nb >= MSG_BINS ? 0u : MSG_BINS - (u32)nb;
}

static __global__ __launch_bounds__(256) void k_msg_hist(const u64* __restrict__ off, u32 n, u32* __restrict__ work) {
  __shared__ u32 h[MSG_BINS];
  for (u32 t = threadIdx.x; t < MSG_BINS; t += blockDim.x) h[t] = 0;
  __syncthreads();
  for (u32 i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    atomicAdd(&h[msg_bin(off, i)], 1u);
  __syncthreads();
  for (u32 t = threadIdx.x; t < MSG_BINS; t += blockDim.x)
    if (h[t]) atomicAdd(&work[MW_COUNT + t], h[t]);
}

// Exclusive scan of the bin counts (LDS) by the first wavefront, in place; returns the flags there.
DEV u32 msg_scan(u32* count, u32 cus) {
  static_assert(MSG_BINS <= 128, "two bins per lane");
  const u32 b = 2 * (threadIdx.x & 63u);
  const u32 c0 = b < MSG_BINS ? count[b] : 0, c1 = b + 1 < MSG_BINS ? count[b + 1] : 0;
  u32 pos = c0 + c1;
  u64 total = (u64)c0 * (MSG_BINS - b) + (u64)c1 * (MSG_BINS - 1 - b);  // in blocks
  const u64 m0 = __ballot(c0 != 0), m1 = __ballot(c1 != 0);
#pragma unroll
  for (u32 d = 1; d < 64; d *= 2) {
    const u32 p = __shfl_up(pos, d);
    pos += (threadIdx.x & 63u) >= d ? p : 0;
    total += __shfl_xor(total, d);
  }
  pos -= c0 + c1;
  if (b < MSG_BINS) count[b] = pos;
  if (b + 1 < MSG_BINS) count[b + 1] = pos + c0;
  const u32 f0 = m0 ? 2 * (u32)__builtin_ctzll(m0) : MSG_BINS, f1 = m1 ? 2 * (u32)__builtin_ctzll(m1) + 1 : MSG_BINS;
  return msg_flags(__popcll(m0) + __popcll(m1), total, MSG_BINS - (f0 < f1 ? f0 : f1), cus);
}

// the whole order by one workgroup, for n <= MSG_SMALL: one launch in place of
// three (5 us each; 1,000 messages of up to 64 bytes 21 -> 12 us). A message's rank in its bin is what its count returned.
constexpr u32 MSG_SMALL = 8192;
static __global__ __launch_bounds__(1024) void k_msg_order_small(const u64* __restrict__ off, u32 n,
                                                                u32* __restrict__ work, u32* __restrict__ order,
                                                                u32 cus) {
  constexpr u32 PER = MSG_SMALL / 1024;
  __shared__ u32 cnt[MSG_BINS];
  __shared__ u32 flags;
  if (threadIdx.x < MSG_BINS) cnt[threadIdx.x] = 0;
  u32 bq[PER], rq[PER];
#pragma unroll
  for (u32 q = 0; q < PER; q++) {
    const u32 i = q * 1024 + threadIdx.x;
    bq[q] = i < n ? msg_bin(off, i) : MSG_BINS;
  }
  __syncthreads();
#pragma unroll
  for (u32 q = 0; q < PER; q++) rq[q] = bq[q] < MSG_BINS ? atomicAdd(&cnt[bq[q]], 1u) : 0;
  __syncthreads();
  if (threadIdx.x < 64) {
    const u32 f = msg_scan(cnt, cus);
    if (threadIdx.x == 0) work[MW_FLAG] = flags = f;
  }
  __syncthreads();
  if ((flags & MSG_SORTED) == 0) return;
#pragma unroll
  for (u32 q = 0; q < PER; q++)
    if (bq[q] < MSG_BINS) order[cnt[bq[q]] + rq[q]] = q * 1024 + threadIdx.x;
}

// ranks within each workgroup's chunk of 1024 messages (4 per thread) by LDS atomics, then one
// global atomic per bin and chunk reserves the chunk's range in that bin (the chunks are large
// because those atomics, on 66 counters shared by every workgroup, are what the scatter waits on).
// Every workgroup scans the counts for itself: a launch between the two took 5 us.
static __global__ __launch_bounds__(256) void k_msg_scatter(const u64* __restrict__ off, u32 n, u32* __restrict__ work,
                                                           u32* __restrict__ order, u32 cus) {
  constexpr u32 PER = 4;
  __shared__ u32 cnt[MSG_BINS];
  __shared__ u32 base[MSG_BINS];
  __shared__ u32 first[MSG_BINS];
  __shared__ u32 flags;
  if (threadIdx.x < MSG_BINS) first[threadIdx.x] = work[MW_COUNT + threadIdx.x];
  __syncthreads();
  if (threadIdx.x < 64) {
    const u32 f = msg_scan(first, cus);
    if (threadIdx.x == 0) flags = f;
    if (threadIdx.x == 0 && blockIdx.x == 0) work[MW_FLAG] = f;
  }
  __syncthreads();
  if ((flags & MSG_SORTED) == 0) return;
  for (u32 c0 = blockIdx.x * blockDim.x * PER; c0 < n; c0 += gridDim.x * blockDim.x * PER) {
    for (u32 t = threadIdx.x; t < MSG_BINS; t += blockDim.x) cnt[t] = 0;
    __syncthreads();
    u32 bq[PER], rq[PER];
#pragma unroll
    for (u32 q = 0; q < PER; q++) {
      const u32 i = c0 + q * blockDim.x + threadIdx.x;
      bq[q] = MSG_BINS;
      rq[q] = 0;
      if (i < n) {
        bq[q] = msg_bin(off, i);
        rq[q] = atomicAdd(&cnt[bq[q]], 1u);
      }
    }
    __syncthreads();
    for (u32 t = threadIdx.x; t < MSG_BINS; t += blockDim.x)
      if (cnt[t]) base[t] = first[t] + atomicAdd(&work[MW_CURSOR + t], cnt[t]);
    __syncthreads();
#pragma unroll
    for (u32 q = 0; q < PER; q++)
      if (bq[q] < MSG_BINS) order[base[bq[q]] + rq[q]] = c0 + q * blockDim.x + threadIdx.x;
    __syncthreads();
  }
}

// digest i = SHA-256(msgs[off[i] .. off[i+1])); msgs 4-byte aligned with slack after the last byte.
// Messages differ in length, so no lane owns one message for the whole launch: a lane whose message
// is done takes its next position by grid stride and the message at that position of the
// longest-first order. In that order each lane takes one message from every round of similar
// lengths, so the lanes stay balanced. (A shared work counter handing out positions instead was
// the bottleneck: one contended atomic on every message's critical path, 2.4x slower on 2^20 64-byte
// messages.) X4: msgs is 16-byte aligned.
// MSG_PAIRS: a workgroup's two wavefronts share 64 messages. One reads a block of each and expands
// its schedule (K[t] + W[t]) into LDS, 32 words at a time; the other runs the rounds on the 32 words
// before. A message then advances one block per 900 instructions instead of 1,700, which is what
// bounds a launch whose longest messages outlast the rest: 65 blocks one after the other, on a
// wavefront that is alone on its SIMD by then. Both wavefronts follow the same lane states.
// 209,715 messages of 0..4096 bytes (log-uniform): 245 us with one wavefront per message, 161 us with two
// (274 us before either, the order in four launches and in index order among the SIMDs).
constexpr u32 MSG_THREADS = 128;

// a lane's place: block b of message i
struct MsgLane {
  u32 i, b, nblk, len, next;
  u64 o;
  bool live;
  // to the next block, or the next message's first
  DEV void advance(const u64* off, u32 n, u32 stride, const u32* order) {
    if (!live || ++b < nblk) return;
    live = next < n;
    if (!live) return;
    i = order ? order[next] : next;
    next = n - next > stride ? next + stride : n;
    o = off[i];
    len = (u32)(off[i + 1] - o);
    nblk = sha256_nblocks(len);
    b = 0;
  }
};

template <bool X4>
DEV void msg_block(const MemDev& mem, u64 o, u32 len, u32 b, u32 nblk, u32 w[16]) {
  if constexpr (X4)
    sha256_block_words_x4(mem, o, len, b, nblk, w);
  else
    sha256_block_words(mem, o, len, b, nblk, w);
}

DEV void msg_store(uint4* out, u32 i, const u32 h[8]) {
  out[2 * (u64)i] = make_uint4(bswap32(h[0]), bswap32(h[1]), bswap32(h[2]), bswap32(h[3]));
  out[2 * (u64)i + 1] = make_uint4(bswap32(h[4]), bswap32(h[5]), bswap32(h[6]), bswap32(h[7]));
}

// flags0: the flags where work is null (then there is no order either); pair_blocks: workgroups used
// with MSG_PAIRS
template <bool X4>
static __global__ __launch_bounds__(MSG_THREADS) void k_message_new(const u32* __restrict__ msgs,
                                                                   const u64* __restrict__ off, u32 n,
                                                                   uint4* __restrict__ out,
                                                                   const u32* __restrict__ work,
                                                                   const u32* __restrict__ order, u32 flags0,
                                                                   u32 pair_blocks, u32 cus) {
  __shared__ uint4 kw[2][8][64];
  const MemDev mem{msgs};
  const u32 flags = work ? work[MW_FLAG] : flags0;
  if ((flags & MSG_SORTED) == 0) order = nullptr;
  const u32 lane = threadIdx.x & 63u;
  u32 w[16], h[8], v[8];
  if ((flags & MSG_PAIRS) == 0) {
    const u32 stride = gridDim.x * MSG_THREADS;
    // a long position with a short one: consecutive workgroups of a compute unit overlap on one SIMD
    u32 next = (threadIdx.x < 64 ? blockIdx.x : 2 * gridDim.x - 1 - blockIdx.x) * 64 + lane;
    u32 i = 0, b = 0, nblk = 0, len = 0;
    u64 o = 0;
    for (;;) {
      const bool need = b == nblk;
      if (__ballot(need) != 0) {
        if (need) {
          const u32 j = next;
          next += stride;
          if (j >= n) break;
          i = order ? order[j] : j;
          o = off[i];
          len = (u32)(off[i + 1] - o);
          nblk = sha256_nblocks(len);
          b = 0;
#pragma unroll
          for (int k = 0; k < 8; k++) h[k] = SHA256_IV[k];
        }
      }
      msg_block<X4>(mem, o, len, b, nblk, w);
      sha256_compress(h, w);
      if (++b == nblk) msg_store(out, i, h);
    }
    return;
  }
  if (blockIdx.x >= pair_blocks) return;
  const u32 stride = pair_blocks * 64;
  const bool expands = threadIdx.x < 64;
  // Workgroups go round the compute units, and a unit's j-th starts j SIMDs further on, so the even j
  // lie on SIMDs of their own: they take positions from the front, the odd ones from the back.
  const u32 j = blockIdx.x / cus, r = (j >> 1) * cus + blockIdx.x % cus;
  MsgLane s;
  s.live = true;
  s.b = s.nblk = 0;
  s.next = ((j & 1) ? pair_blocks - 1 - r : r) * 64 + lane;
  s.advance(off, n, stride, order);
  MsgLane prev = s;
  prev.live = false;
  u32 raw[X4 ? 20 : 17];
  auto load = [&](const MsgLane& m) {
    if constexpr (X4)
      sha256_block_load_x4(mem, m.o, m.len, m.b, raw);
    else
      sha256_block_load(mem, m.o, m.len, m.b, raw);
  };
  if (expands && s.live) load(s);
  for (;;) {
    if (expands) {
      if (s.live) {
        if constexpr (X4)
          sha256_block_place_x4(raw, s.o, s.len, s.b, s.nblk, w);
        else
          sha256_block_assemble(raw, (u32)(s.o & 3u) * 8u, s.len, s.b, s.nblk, w);
        sha256_expand<0>(w, [&](int q, u32 x, u32 y, u32 z, u32 t) { kw[0][q][lane] = make_uint4(x, y, z, t); });
      }
    } else if (prev.live) {
      sha256_rounds<8>(v, [&](int q) { return kw[1][q][lane]; });
#pragma unroll
      for (int k = 0; k < 8; k++) h[k] += v[k];
      if (prev.b + 1 == prev.nblk) msg_store(out, prev.i, h);
    }
    if (__ballot(s.live) == 0) break;  // the same on both wavefronts
    __syncthreads();
    prev = s;
    s.advance(off, n, stride, order);
    if (prev.live) {
      if (expands) {
        if (s.live) load(s);  // the next block's words arrive during the expansion
        sha256_expand<1>(w, [&](int q, u32 x, u32 y, u32 z, u32 t) { kw[1][q][lane] = make_uint4(x, y, z, t); });
      } else {
#pragma unroll
        for (int k = 0; k < 8; k++) {
          if (prev.b == 0) h[k] = SHA256_IV[k];
          v[k] = h[k];
        }
        sha256_rounds<8>(v, [&](int q) { return kw[0][q][lane]; });
      }
    }
    __syncthreads();
  }
}

// pair workgroups per compute unit: 16 KB of LDS each
constexpr u32 MSG_PAIRS_PER_CU = 8;

// address i = SHA-256(pub i), or 32 zero bytes where status[i] != 0 (a failed recovery)
static __global__ __launch_bounds__(256) void k_fuel_address(const uint4* __restrict__ pubs,
                                                            const u8* __restrict__ status, u32 n,
                                                            uint4* __restrict__ out) {
  for (u32 i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    u32 pk[16], d[8];
    load_words(pubs + 4 * (u64)i, pk, 4);
    sha256_64(pk, d);
    const u32 keep = (status == nullptr || status[i] == 0) ? ~0u : 0u;
    out[2 * (u64)i] = make_uint4(d[0] & keep, d[1] & keep, d[2] & keep, d[3] & keep);
    out[2 * (u64)i + 1] = make_uint4(d[4] & keep, d[5] & keep, d[6] & keep, d[7] & keep);
  }
}

static u32 grid_for(u32 n, u32 grid) {
  const u32 want = (n + 255) / 256;
  return want < grid ? want : grid;
}

// grid: blocks of 256; cus: compute units
hipError_t launch_message_new(const void* msgs, const u64* off, u32 n, void* out, u32* work, u32* order, u32 grid,
                              u32 cus, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const u32 groups = (n + 63) / 64;
  if (groups == 1) {
    work = order = nullptr;
  } else if (n <= MSG_SMALL) {
    k_msg_order_small<<<1, 1024, 0, s>>>(off, n, work, order, cus);
  } else {
    k_fill_u32<<<1, 256, 0, s>>>(work, 0u, MSG_WORK_WORDS);
    k_msg_hist<<<grid_for(n, cus), 256, 0, s>>>(off, n, work);
    k_msg_scatter<<<grid_for(n, grid), 256, 0, s>>>(off, n, work, order, cus);
  }
  // a workgroup per 64 messages if they may go to pairs, else per 128
  const u32 pairs = groups < MSG_PAIRS_PER_CU * cus ? groups : MSG_PAIRS_PER_CU * cus;
  const u32 singles = (groups + 1) / 2 < 2 * grid ? (groups + 1) / 2 : 2 * grid;
  const auto run = ((uintptr_t)msgs & 15u) == 0 ? k_message_new<true> : k_message_new<false>;
  run<<<pairs > singles ? pairs : singles, MSG_THREADS, 0, s>>>((const u32*)msgs, off, n, (uint4*)out, work, order,
                                                               MSG_PAIRS, pairs, cus);
  return hipGetLastError();
}

hipError_t launch_fuel_address(const void* pubs, const void* status, u32 n, void* out, u32 grid, hipStream_t s) {
  if (n == 0) return hipSuccess;
  k_fuel_address<<<grid_for(n, grid), 256, 0, s>>>((const uint4*)pubs, (const u8*)status, n, (uint4*)out);
  return hipGetLastError();
}

}  // namespace sigops
