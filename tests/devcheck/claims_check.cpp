// claims_check.cpp -- host build of the tile claims (csrc/claims.hpp) under a schedule: workgroups start
// in order while there is room, a wavefront takes tiles until none is left, a workgroup leaves its room
// when all its wavefronts have ended. Test infrastructure only.
#include <queue>
#include <tuple>
#include <vector>

#include "claims.hpp"

using namespace sigops;

namespace {
struct Launch {
  u64 taken[64] = {};
  u32 counter = 0;
};
struct Wave {
  Launch& m;
  u64 free[64];
  bool own(u32 t) {
    const u64 bit = 1ull << (t & 63), old = m.taken[t >> 6];
    m.taken[t >> 6] |= bit;
    return !(old & bit);
  }
  void look(u32 n) {
    for (u32 l = 0; l < 64; l++) {
      const u64 in = n >= 64 * l + 64 ? ~0ull : (n > 64 * l ? ~0ull >> (64 - (n - 64 * l)) : 0);
      free[l] = ~m.taken[l] & in;
    }
  }
  u64 words() const {
    u64 r = 0;
    for (u32 l = 0; l < 64; l++) r |= (u64)(free[l] != 0) << l;
    return r;
  }
  u32 first(u32 l) const { return (u32)__builtin_ctzll(free[l]); }
  bool claim(u32 l, u32 b) {
    const u64 bit = 1ull << b, old = m.taken[l];
    m.taken[l] |= bit;
    free[l] &= ~(old | bit);
    return !(old & bit);
  }
  u32 beyond() { return m.counter++; }
};
}  // namespace

// room: workgroups that may run at a time until `until`, all of them afterwards; the first `slow` ones run at
// a tenth of the others' speed (their SIMDs are in use) and reach their first tile 5 time units later. A tile
// takes 100 time units and a little that depends on it. done: how often each tile was run. Returns the time
// of the last.
extern "C" long tc_run(u32 ntiles, u32 cus, u32 workgroups, u32 room, long until, u32 slow, unsigned* done) {
  Launch m;
  std::vector<TileClaims> claims;
  std::vector<u32> running(workgroups, 4);
  for (u32 w = 0; w < 4 * workgroups; w++) claims.emplace_back(ntiles, cus, workgroups, w);
  typedef std::tuple<long, u32> ev;  // time, wavefront
  std::priority_queue<ev, std::vector<ev>, std::greater<ev>> q;
  u32 started = 0, resident = 0;
  long end = 0;
  auto start = [&](long t) {
    while (started < workgroups && (resident < room || t >= until)) {
      for (u32 k = 0; k < 4; k++) q.push(ev(started < slow ? t + 5 : t, 4 * started + k));
      started++;
      resident++;
    }
  };
  start(0);
  bool opened = false;
  while (!q.empty()) {
    const auto [t, w] = q.top();
    if (!opened && t >= until) {
      opened = true;
      start(t);
    }
    q.pop();
    Wave wave{m, {}};
    const u32 tile = claims[w].next(wave);
    if (tile == NO_TILE) {
      if (--running[w / 4] == 0) {
        resident--;
        start(t);
      }
      continue;
    }
    if (tile >= ntiles) return -1;
    done[tile]++;
    const long e = t + (100 + (tile * 7919u) % 13) * (w / 4 < slow ? 10 : 1);
    end = e > end ? e : end;
    q.push(ev(e, w));
  }
  return end;
}
