// claims.hpp -- how the wavefronts of the mixed batch's persistent launch share its tiles (kern_batch.hip).
//
// Workgroups of 4 wavefronts go round the compute units, one wavefront to a SIMD, so wavefront w of each
// round of workgroups shares its SIMD with wavefront w of the others. A wavefront's first tile is given by
// its place, odd rounds in reverse: neighbours run the same code (they share the instruction cache), and
// as the tiles come longest first (secp256r1), a launch of less than two rounds doubles up the SIMDs with
// the shortest tiles. The tiles beyond come from a counter, and so do all tiles where they fill at most half of
// the SIMDs: wavefronts that share a SIMD with another launch's then come last, while places would lie on
// SIMDs in use (us per batch on three streams, from the counter / by place: 20,000 items 499 / 653, 30,000
// 588 / 672, 45,000 712 / 715; alone 1,332 / 1,294, 1,372 / 1,325, 1,394 / 1,340).
// A first tile is claimed by its bit, so that those of workgroups which another launch keeps from starting
// go to the wavefronts that end. A wavefront claims one tile at a time, when it is about to run it: none
// holds tiles that another could run.
// us, all tiles from one counter / so (mixed, messages up to 1 KB): 50,000 items 1,510 / 1,430, 80,000
// 2,070 / 1,850, 100,003 2,180 / 1,820, 131,072 2,360 / 2,260, 300,000 5,000 / 4,630, 400,000 6,790 /
// 6,720, 2^20 13,980 / 14,170: above four tiles per wavefront all come from the counter.
//
// Host builds (tests) run the same code over many wavefronts in turn.
#pragma once
#include "field.hpp"

namespace sigops {

constexpr u32 NO_TILE = 0xFFFFFFFFu;
constexpr u32 FIRST_TILES_MAX = 64 * 64;  // a 64-bit word of claims to each lane

// Wave: own(t): claims first tile t, false if it was taken; look(n): reads the claims of the first n
// tiles, lane l's those of tiles 64 l ..; words(): the lanes that see a free tile; first(l): the lowest
// free one of lane l's; claim(l, b): claims it, false if it was taken, and either way lane l sees it as
// taken from then on; beyond(): the next number of the counter. Results are the same on every lane.
struct TileClaims {
  u32 ntiles, first_tiles, mine;
  bool others;  // first tiles may be left over
  // cus: compute units, the grid's workgroups a multiple of them; 0: all tiles from the counter. at:
  // this wavefront among the grid's, 4 to a workgroup
  DEV TileClaims(u32 tiles, u32 cus, u32 workgroups, u32 at) : ntiles(tiles), mine(NO_TILE) {
    first_tiles = ntiles > 2 * cus && ntiles <= 16 * workgroups && cus ? workgroups * 4 : 0;
    others = first_tiles != 0;
    if (first_tiles) {
      const u32 round = 4 * cus, r = at / round, w = at % round;
      mine = r * round + ((r & 1) ? round - 1 - w : w);
    }
    first_tiles = first_tiles < ntiles ? first_tiles : ntiles;
    at_ = mine;
  }
  // the next tile to run; NO_TILE when none is left
  template <class Wave>
  DEV u32 next(Wave& w) {
    if (mine != NO_TILE) {
      const u32 t = mine;
      mine = NO_TILE;
      if (t >= ntiles) return NO_TILE;  // the rest is others' first tiles
      if (w.own(t)) return t;
    }
    if (others) {
      w.look(first_tiles);
      // from this wavefront's own place on, so that those which look at the same time do not all try
      // the same tile. Every trip takes a tile away from what this wavefront sees as free.
      const u32 from = (at_ >> 6) & 63u;
      for (u64 words; (words = w.words()) != 0;) {
        const u64 turned = (words >> from) | (words << ((64u - from) & 63u));
        const u32 l = (from + (u32)__builtin_ctzll(turned)) & 63u;
        const u32 b = w.first(l);
        if (w.claim(l, b)) return 64 * l + b;
      }
      others = false;
    }
    const u32 t = first_tiles + w.beyond();
    return t < ntiles ? t : NO_TILE;
  }

 private:
  u32 at_;
};

}  // namespace sigops
