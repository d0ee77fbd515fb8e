// What the launches of a radix sort do, decided on the device from the digit histograms.  Plain C++ (also compiled
// for the host by tests/cpp/test_sort_ctl.cpp, which checks what is left to do behind a pass that gave up).
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define TA_CTL_FN __host__ __device__ inline
#else
#define TA_CTL_FN inline
#endif

namespace ta {

constexpr int MAX_PASSES = 8;  // pass launches of a sort: one per digit
constexpr int TOP_SLOTS = 2;   // passes in front of the last step of the short way, at most

// A sort through all digits uses every launch; one that takes the short way the first one or two.
struct SortCtl {
  enum : uint32_t { SKIP, RUN };
  uint32_t slot[MAX_PASSES];  // action, digit, source buffer, whether it encodes / decodes the keys
  uint32_t final_in_alt;      // result sits in the alternate buffer after the last slot
  uint32_t gave_up;           // a tile stopped waiting for its predecessors (see LOOKBACK_SPIN_LIMIT)
  uint32_t fast;              // the short way is taken, with this many digits
  uint32_t fast_src_alt;      // its last step reads the alternate buffer
  uint32_t prefix_bit;        // lowest bit of the digits the array is ordered by then
  uint32_t window;            // positions per workgroup of the last step
  uint32_t long_windows;      // windows the last step left because they do not fit a workgroup

  static TA_CTL_FN uint32_t pack(uint32_t action, uint32_t digit, uint32_t src_alt, bool encodes, bool decodes) {
    return action | digit << 4 | src_alt << 8 | (encodes ? 1u << 9 : 0u) | (decodes ? 1u << 10 : 0u);
  }
  static TA_CTL_FN bool runs(uint32_t s) { return (s & 15u) == RUN; }
  static TA_CTL_FN uint32_t digit(uint32_t s) { return s >> 4 & 15u; }
  static TA_CTL_FN bool src_alt(uint32_t s) { return (s >> 8 & 1u) != 0; }
  static TA_CTL_FN bool encodes(uint32_t s) { return (s >> 9 & 1u) != 0; }
  static TA_CTL_FN bool decodes(uint32_t s) { return (s >> 10 & 1u) != 0; }

  TA_CTL_FN bool finishes() const { return fast != 0; }
  TA_CTL_FN bool copies_back() const { return final_in_alt != 0; }

  // What a tile of the pass in slot `at` does when it stops waiting.  The array is not in the order, and does not hold
  // the keys, that the launches behind it count on -- their positions could leave it -- so they are struck out: the
  // call ends with an unfinished sort.  store(address, value) has to reach the next launch; fields that the
  // running launch reads stay as they are.  A launch of several passes reads every slot, so it strikes out none
  // (at = MAX_PASSES - 1): there a pass begins only behind a complete one, and one of which a tile gave up never is.
  template <typename Store>
  TA_CTL_FN void strike_out(int at, Store store) {
    for (int s = at + 1; s < MAX_PASSES; ++s) store(&slot[s], (uint32_t)SKIP);
    store(&fast, 0u);
    store(&final_in_alt, 0u);
    store(&gave_up, 1u);
  }
};

}  // namespace ta
