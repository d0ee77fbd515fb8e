// Tile boundaries on the path of a merge: the steps of the searches for them, apart from the reads of the keys, and
// what a tile makes of their results.  Plain C++ (also compiled for the host by tests/cpp/test_merge_search.cpp, which
// plays the searches through on keys in order and in no order).
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define THRUST_AMD_SEARCH_FN __host__ __device__ inline __attribute__((always_inline))
#else
#define THRUST_AMD_SEARCH_FN inline
#endif

namespace thrust {
namespace system {
namespace hip {
namespace prim {

// First index in [lo, hi] at which a monotone predicate turns false (hi when it is true throughout), probing at every
// step the index of its interval that is a multiple of the
// largest power of two.  It needs as many steps as the bisection at worst, but the probes of the
// first steps are the same few indices for every thread that searches the same arrays (the
// nodes of one implicit tree over the index range), so they come from the caches instead of
// each being a miss of its own: the searches for the tile boundaries of a merge of 2 x 2^27 keys
// (65537 threads, 27 dependent steps each) took 108 us with the plain bisection.
template <typename Pred>
THRUST_AMD_SEARCH_FN uint64_t aligned_partition_point(uint64_t lo, uint64_t hi, Pred pred) {
  while (lo < hi) {
    const uint64_t last = hi - 1;
    const uint64_t differ = lo ^ last;
    const uint64_t mid = differ ? (last & ~((1ull << (63 - __builtin_clzll(differ))) - 1ull)) : lo;
    if (pred(mid)) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// How many of the first `diag` outputs can come from range A.
struct SplitInterval {
  uint64_t lo, hi;
  THRUST_AMD_SEARCH_FN SplitInterval(uint64_t diag, uint64_t na, uint64_t nb)
      : lo(diag > nb ? diag - nb : 0), hi(diag < na ? diag : na) {}
};

// A round of the search by 2^BITS lanes probes the multiples of 2^(BITS k) in the interval, at most 2^BITS of them, so
// that an interval below 2^(BITS (k + 1)) shrinks below 2^(BITS k).
template <int BITS>
struct GroupRound {
  uint64_t unit, first;
  // the exponent BITS k of the first round; the next ones are BITS lower each, down to 0
  static THRUST_AMD_SEARCH_FN int first_bit(uint64_t na, uint64_t nb) {
    const uint64_t longest = na < nb ? na : nb;  // no interval is longer
    return longest > 1 ? (63 - __builtin_clzll(longest)) / BITS * BITS : 0;
  }
  THRUST_AMD_SEARCH_FN GroupRound(const SplitInterval& in, int bit)
      : unit(1ull << bit), first((in.lo + unit - 1) & ~(unit - 1)) {}
  THRUST_AMD_SEARCH_FN uint64_t probe(uint32_t lane) const { return first + (uint64_t)lane * unit; }  // below in.hi, or none
  // yes: how many probes belong to range A (with keys in order the lowest ones; a count in any case)
  THRUST_AMD_SEARCH_FN void narrow(SplitInterval& in, uint32_t yes) const {
    const uint64_t no = first + (uint64_t)yes * unit;  // the first probe that said no, if it was one
    if (yes > 0) in.lo = no - unit + 1;
    if (yes < (1u << BITS) && no < in.hi) in.hi = no;
  }
};

// The elements of A that a tile of `outputs` outputs takes, [a0, a1), from the splits found for its two ends.  In keys
// that are in no order (NaN among them) the second split may lie before the first or too far behind it: what the tile
// reads stays inside the ranges all the same, and it always has its number of elements.
struct TileSplit {
  uint64_t a0, a1;
  THRUST_AMD_SEARCH_FN TileSplit(uint64_t first, uint64_t second, uint64_t outputs) : a0(first), a1(second) {
    if (a1 < a0) a1 = a0;
    if (a1 - a0 > outputs) a1 = a0 + outputs;
  }
};

}  // namespace prim
}  // namespace hip
}  // namespace system
}  // namespace thrust
