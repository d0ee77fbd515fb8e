// Host-side check of the rule by which the workgroups of a radix-sort pass take their tiles
// (thrust_amd/csrc/sort_tickets.hpp, the very function the kernel calls):
//   1. with `tiles` workgroups, workgroup i drawing the next ticket of class i % 8, every tile
//      is taken exactly once and the tiles of a class rise with its tickets -- for every tile
//      count up to 20000 and a few large ones;
//   2. no schedule of two dispatcher models leaves the pass stuck.  A tile can finish once every
//      lower tile has been taken (its look-back then finds their counts).  Model A: the
//      workgroups of class k run on XCD k only, each XCD dispatching its own in order at its own
//      pace into any number of slots.  Model B: workgroups are dispatched in order of their index
//      into at least 64 slots anywhere.  Random paces and finishing orders, many seeds;
//   3. several passes in one launch (onesweep_rest_kernel) end with any number of workgroups resident: no pass begins
//      before every tile of the one before is written, every tile is written once, and a tile that gives up ends the
//      launch with no later pass begun.
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#include "../../thrust_amd/csrc/sort_tickets.hpp"

using namespace ta;

static bool bijection(uint32_t tiles) {
  std::vector<uint8_t> seen(tiles, 0);
  uint32_t next[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  int64_t last[8] = {-1, -1, -1, -1, -1, -1, -1, -1};
  for (uint32_t i = 0; i < tiles; ++i) {
    const uint32_t k = i % 8, t = class_tile(k, next[k]++, tiles);
    if (t >= tiles || seen[t]) return false;
    if ((int64_t)t <= last[k]) return false;
    last[k] = t;
    seen[t] = 1;
  }
  return true;
}

// One run of a dispatcher model; false when it gets stuck.
static bool finishes(uint32_t tiles, bool bound_to_xcd, uint32_t slots_per_xcd, uint32_t seed) {
  std::mt19937 rnd(seed);
  std::vector<uint8_t> taken(tiles, 0);
  uint32_t next_ticket[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  uint32_t next_of_class[8] = {0, 1, 2, 3, 4, 5, 6, 7};  // model A: next workgroup index of each XCD
  uint32_t next_index = 0;                                // model B
  std::vector<std::vector<uint32_t>> resident(8);
  uint32_t lowest_untaken = 0, finished = 0;
  auto take = [&](uint32_t i) {
    const uint32_t k = i % 8, t = class_tile(k, next_ticket[k]++, tiles);
    taken[t] = 1;
    return t;
  };
  while (finished < tiles) {
    bool could_dispatch = false, could_finish = false, moved = false;
    if (bound_to_xcd) {
      for (uint32_t x = 0; x < 8; ++x)
        while (resident[x].size() < slots_per_xcd && next_of_class[x] < tiles) {
          could_dispatch = true;
          if (rnd() % 4 == 0) break;  // this XCD falls behind for a while
          resident[x].push_back(take(next_of_class[x]));
          next_of_class[x] += 8;
          moved = true;
        }
    } else {
      while (next_index < tiles) {
        std::vector<uint32_t> room;
        for (uint32_t x = 0; x < 8; ++x)
          if (resident[x].size() < slots_per_xcd) room.push_back(x);
        if (room.empty()) break;
        could_dispatch = true;
        if (rnd() % 8 == 0) break;
        resident[room[rnd() % room.size()]].push_back(take(next_index++));
        moved = true;
      }
    }
    while (lowest_untaken < tiles && taken[lowest_untaken]) ++lowest_untaken;
    for (uint32_t x = 0; x < 8; ++x) {
      std::vector<uint32_t> keep;
      for (uint32_t t : resident[x]) {
        if (t < lowest_untaken) {  // every lower tile is taken
          could_finish = true;
          if (rnd() % 3 != 0) {
            ++finished;
            moved = true;
            continue;
          }
        }
        keep.push_back(t);
      }
      resident[x].swap(keep);
    }
    if (!moved && !could_dispatch && !could_finish) return false;  // nothing can ever move again
  }
  return true;
}

// Several passes in one launch: each workgroup draws tiles of a pass until there are none, then waits until the counters
// of the pass hold what is due.  A tile is written once all lower ones of its pass have been drawn (its look-back finds
// their counts then).  `bad` (pass, tile): a tile that gives up.  False when stuck or out of turn.
static bool shares_launch(uint32_t tiles, uint32_t passes, uint32_t slots, uint32_t seed, int bad_pass, uint32_t bad_tile) {
  std::mt19937 rnd(seed);
  struct Group {
    uint32_t pass;
    int64_t tile;  // -1: has to draw; -2: waits for the pass before
  };
  std::vector<uint32_t> ticket(passes, 0);
  std::vector<std::vector<uint32_t>> held(passes, std::vector<uint32_t>(COUNTERS, 0));
  std::vector<std::vector<uint8_t>> written(passes, std::vector<uint8_t>(tiles, 0));
  auto state_of = [&](uint32_t pass) {  // 1 complete, 0 not yet, -1 never
    bool complete = true;
    for (uint32_t c = 0; c < COUNTERS; ++c) {
      if (held[pass][c] >= COUNT_GAVE_UP) return -1;
      complete = complete && held[pass][c] == due_on(c, tiles);
    }
    return complete ? 1 : 0;
  };
  std::vector<Group> resident;
  uint32_t started = 0, ended = 0;
  while (ended < tiles) {
    bool can_move = false;
    while (resident.size() < slots && started < tiles) {
      resident.push_back(Group{0, -2});
      ++started;
      can_move = true;
    }
    std::vector<Group> keep;
    for (Group g : resident) {
      bool ends = false;
      if (g.tile == -2) {
        const int before = g.pass == 0 ? 1 : state_of(g.pass - 1);
        if (before != 0) {
          can_move = true;
          if (rnd() % 2) {
            if (before < 0) ends = true;
            else g.tile = -1;
          }
        }
      } else if (g.tile == -1) {
        can_move = true;
        if (rnd() % 2) {
          const uint32_t t = ticket[g.pass]++;
          if (t < tiles) {
            g.tile = t;
          } else {
            g.tile = -2;
            if (++g.pass == passes) ends = true;
          }
        }
      } else {
        can_move = true;  // every lower tile has been drawn before this one, by a workgroup that runs or is through
        if (rnd() % 3) {
          const uint32_t t = (uint32_t)g.tile;
          if (written[g.pass][t]++) return false;
          held[g.pass][counter_of(t)] += (int)g.pass == bad_pass && t == bad_tile ? COUNT_GAVE_UP : 1u;
          g.tile = -1;
        }
      }
      if (ends) ++ended;
      else keep.push_back(g);
    }
    resident.swap(keep);
    if (!can_move) return false;
  }
  for (uint32_t p = 0; p < passes; ++p)
    for (uint32_t t = 0; t < tiles; ++t)
      if (written[p][t] != (bad_pass < 0 || (int)p <= bad_pass ? 1 : 0)) return false;
  return true;
}

// Every written tile is counted on a counter of its own slot, and the counters hold what is due exactly when all are.
static bool counts(uint32_t tiles) {
  std::vector<uint32_t> held(COUNTERS, 0);
  for (uint32_t t = 0; t < tiles; ++t) {
    bool complete = true;
    for (uint32_t c = 0; c < COUNTERS; ++c) complete = complete && held[c] == due_on(c, tiles);
    if (complete || counter_of(t) >= COUNTERS) return false;  // complete too early, or no such counter
    ++held[counter_of(t)];
  }
  // a pass of which any tile gave up is never complete, and its counters say so
  for (uint32_t bad : {0u, tiles / 2, tiles - 1}) {
    const uint32_t c = counter_of(bad), with = held[c] - 1 + COUNT_GAVE_UP;
    if (with == due_on(c, tiles) || with < COUNT_GAVE_UP || due_on(c, tiles) >= COUNT_GAVE_UP) return false;
  }
  for (uint32_t c = 0; c < COUNTERS; ++c) {
    if (held[c] != due_on(c, tiles)) return false;
    // apart from the word that hands the tiles out, from each other, and inside the slot
    if (counter_word(c) < TICKET_STRIDE || counter_word(c) % TICKET_STRIDE != 0 || counter_word(c) >= TICKET_CLASSES * TICKET_STRIDE) return false;
  }
  return true;
}

int main() {
  for (uint32_t tiles = 1; tiles <= 2000; ++tiles)
    if (!counts(tiles)) {
      std::printf("tiles=%u: the counters of a pass do not say when it is complete\n", tiles);
      return 1;
    }
  for (uint32_t tiles = 1; tiles <= 20000; ++tiles)
    if (!bijection(tiles)) {
      std::printf("tiles=%u: not every tile exactly once, or not rising inside a class\n", tiles);
      return 1;
    }
  for (uint32_t tiles : {65535u, 65536u, 65537u, 1u << 20, (1u << 20) + 13u, 3000001u})
    if (!bijection(tiles)) {
      std::printf("tiles=%u: not every tile exactly once, or not rising inside a class\n", tiles);
      return 1;
    }
  const uint32_t counts[] = {1, 7, 8, 9, 63, 64, 65, 127, 500, 513, 1000, 4097, 14564};
  for (uint32_t tiles : counts)
    for (uint32_t seed = 1; seed <= 8; ++seed) {
      for (uint32_t slots : {1u, 2u, 3u, 64u})  // per XCD
        if (!finishes(tiles, true, slots, seed)) {
          std::printf("stuck: tiles=%u bound to XCDs, %u slots per XCD, seed %u\n", tiles, slots, seed);
          return 1;
        }
      for (uint32_t slots : {8u, 16u, 64u})  // per XCD: 64, 128, 512 in all
        if (!finishes(tiles, false, slots, seed)) {
          std::printf("stuck: tiles=%u dispatched in order, %u slots, seed %u\n", tiles, 8 * slots, seed);
          return 1;
        }
    }
  for (uint32_t tiles : {1u, 2u, 6u, 7u, 8u, 50u, 171u})
    for (uint32_t slots : {1u, 2u, 5u, 64u, 171u})
      for (uint32_t seed = 1; seed <= 6; ++seed)
        for (int bad = -1; bad < 3; ++bad)
          if (!shares_launch(tiles, 3, slots, seed, bad, seed * 13 % tiles)) {
            std::printf("passes in one launch: tiles=%u, %u slots, seed %u, gives up in pass %d\n", tiles, slots, seed, bad);
            return 1;
          }
  std::printf("PASSED\n");
  return 0;
}
