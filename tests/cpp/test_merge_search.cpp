// Host-side check of the searches for a merge's tile boundaries (include/thrust/system/hip/detail/merge_search.h, the
// steps the kernels take): on keys in order every way of searching finds the boundary, and on keys in no order -- NaN
// among them, where the boundaries themselves run backward -- what a tile reads stays inside both ranges.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <limits>
#include <random>
#include <vector>

#include "../../include/thrust/system/hip/detail/merge_search.h"

using namespace thrust::system::hip::prim;
using Keys = std::vector<float>;

static bool from_a(const Keys& a, const Keys& b, uint64_t diag, uint64_t mid) { return !(b.at(diag - 1 - mid) < a.at(mid)); }

// group_merge_path (merge_kernels.h) with a loop in place of the lanes
template <int BITS>
static uint64_t by_group(const Keys& a, const Keys& b, uint64_t diag) {
  SplitInterval in(diag, a.size(), b.size());
  for (int bit = GroupRound<BITS>::first_bit(a.size(), b.size()); bit >= 0; bit -= BITS) {
    const GroupRound<BITS> round(in, bit);
    uint32_t yes = 0;
    for (uint32_t lane = 0; lane < (1u << BITS); ++lane) {
      const uint64_t mid = round.probe(lane);
      if (mid < in.hi && from_a(a, b, diag, mid)) ++yes;
    }
    round.narrow(in, yes);
  }
  return in.lo;
}

static uint64_t by_one(const Keys& a, const Keys& b, uint64_t diag) {
  const SplitInterval in(diag, a.size(), b.size());
  return aligned_partition_point(in.lo, in.hi, [&](uint64_t mid) { return from_a(a, b, diag, mid); });
}

static int failures = 0;

// Returns how many tiles have boundaries that the ranges do not allow as they are.
template <typename Search>
static int check(const char* what, const Keys& a, const Keys& b, uint64_t tile, bool in_order, Search search) {
  const uint64_t total = a.size() + b.size();
  int bad = 0;
  for (uint64_t d0 = 0; d0 < total; d0 += tile) {
    const uint64_t d1 = std::min(total, d0 + tile);
    const uint64_t s0 = search(a, b, d0), s1 = search(a, b, d1);
    if (in_order) {
      // among the first d0 outputs, ties from A first: the last one taken from A is not behind the next of B, and so on
      const uint64_t j = d0 - s0;
      const bool right = (s0 == 0 || j == b.size() || !(b[j] < a[s0 - 1])) && (j == 0 || s0 == a.size() || b[j - 1] < a[s0]);
      if (!right && ++failures) std::printf("FAILED: %s, boundary %llu\n", what, (unsigned long long)d0);
    }
    bad += s1 < s0 || s1 - s0 > d1 - d0;
    const TileSplit split(s0, s1, d1 - d0);
    const uint64_t b0 = d0 - split.a0, b1 = d1 - split.a1;
    const bool inside = split.a0 <= split.a1 && split.a1 <= a.size() && b0 <= b1 && b1 <= b.size() && split.a0 <= d0 &&
                        split.a1 <= d1 && (split.a1 - split.a0) + (b1 - b0) == d1 - d0;
    if (!inside && ++failures) std::printf("FAILED: %s, tile at %llu leaves the ranges\n", what, (unsigned long long)d0);
    if (in_order && (split.a0 != s0 || split.a1 != s1) && ++failures) std::printf("FAILED: %s, a good split changed\n", what);
  }
  return bad;
}

int main() {
  std::mt19937 rng(7);
  std::uniform_real_distribution<float> uniform(-1000.f, 1000.f);
  const float nan = std::numeric_limits<float>::quiet_NaN();
  enum Kind { SORTED, EQUAL, NAN_FIRST, NAN_SOME, NAN_MANY, UNSORTED, REVERSED, KINDS };
  int bad[KINDS][4] = {};
  const uint64_t all_sizes[][2] = {{40000, 40000}, {50021, 20011}, {33, 60000}, {60000, 1}, {0, 5000}, {4096, 0}};
  for (const auto& sizes : all_sizes) {
    for (int kind = 0; kind < KINDS; ++kind) {
      Keys r[2];
      for (int s = 0; s < 2; ++s) {
        r[s].resize(sizes[s]);
        for (float& x : r[s]) x = kind == EQUAL ? 1.f : uniform(rng);
        if (kind != UNSORTED) std::sort(r[s].begin(), r[s].end());
        if (kind == REVERSED) std::reverse(r[s].begin(), r[s].end());
        for (uint64_t i = 0; i < r[s].size(); ++i) {
          if (kind == NAN_FIRST && s == 0 && i < r[s].size() / 10) r[s][i] = nan;
          if (kind == NAN_SOME && rng() % 1000 == 0) r[s][i] = nan;
          if (kind == NAN_MANY && rng() % (s == 0 ? 2 : 4) == 0) r[s][i] = nan;
        }
      }
      const bool in_order = kind <= EQUAL;
      for (const uint64_t tile : {64, 1000, 4096}) {
        bad[kind][0] += check("one lane", r[0], r[1], tile, in_order, by_one);
        bad[kind][1] += check("4 lanes", r[0], r[1], tile, in_order, by_group<2>);
        bad[kind][2] += check("8 lanes", r[0], r[1], tile, in_order, by_group<3>);
        bad[kind][3] += check("32 lanes", r[0], r[1], tile, in_order, by_group<5>);
      }
    }
  }
  // the inputs are what the rule is for: with NaN every search has boundaries that lead out of the ranges
  for (int search = 0; search < 4; ++search) {
    if ((bad[SORTED][search] || bad[EQUAL][search]) && ++failures) std::printf("FAILED: keys in order, search %d\n", search);
    if (!bad[NAN_MANY][search] && ++failures) std::printf("FAILED: search %d has met no boundary out of order\n", search);
  }
  if (failures == 0) std::printf("PASSED\n");
  return failures != 0;
}
