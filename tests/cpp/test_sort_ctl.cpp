// Host-side check of the control block of a radix sort (thrust_amd/csrc/sort_ctl.hpp, the functions the kernels
// call): whichever pass gives up, no launch behind it touches the array any more, and the launch itself still reads what
// it read before.
#include <cstdint>
#include <cstdio>

#include "../../thrust_amd/csrc/sort_ctl.hpp"

using namespace ta;

// The control block of a sort of `passes` digits that takes the short way with `fast` of them (0: all digits' passes).
static SortCtl plan(int passes, uint32_t fast) {
  SortCtl c{};
  const int run = fast ? (int)fast : passes;
  for (int i = 0; i < run; ++i)
    c.slot[i] = SortCtl::pack(SortCtl::RUN, (uint32_t)(passes - run + i), (uint32_t)i & 1, i == 0, !fast && i == run - 1);
  c.fast = fast;
  c.final_in_alt = fast ? 0 : passes & 1;
  return c;
}

int main() {
  int failures = 0;
  auto expect = [&](bool ok, const char* what, int passes, uint32_t fast, int at) {
    if (!ok) {
      std::printf("FAILED: %s (%d digits, short way %u, slot %d)\n", what, passes, fast, at);
      ++failures;
    }
  };
  for (int passes = 1; passes <= MAX_PASSES; ++passes) {
    for (uint32_t fast = 0; fast <= (uint32_t)TOP_SLOTS && (int)fast <= passes; ++fast) {
      for (int at = 0; at < MAX_PASSES; ++at) {
        SortCtl c = plan(passes, fast);
        const SortCtl before = c;
        if (!SortCtl::runs(c.slot[at])) continue;
        c.strike_out(at, [](uint32_t* p, uint32_t x) { *p = x; });
        expect(c.gave_up == 1, "the flag is set", passes, fast, at);
        for (int s = 0; s <= at; ++s) expect(c.slot[s] == before.slot[s], "the running launch reads its slot", passes, fast, at);
        for (int s = at + 1; s < MAX_PASSES; ++s) expect(!SortCtl::runs(c.slot[s]), "no later pass runs", passes, fast, at);
        expect(!c.finishes(), "the last step does nothing", passes, fast, at);
        expect(!c.copies_back(), "nothing is copied back", passes, fast, at);
      }
    }
  }
  // a launch of several passes: whatever it still reads of the slots stays, the launches behind it are struck out
  for (int passes = 1; passes <= MAX_PASSES; ++passes) {
    SortCtl c = plan(passes, 0);
    const SortCtl before = c;
    c.strike_out(MAX_PASSES - 1, [](uint32_t* p, uint32_t x) { *p = x; });
    for (int s = 0; s < MAX_PASSES; ++s) expect(c.slot[s] == before.slot[s], "the running launch reads all slots", passes, 0, s);
    expect(c.gave_up == 1 && !c.finishes() && !c.copies_back(), "nothing runs behind a launch of several passes", passes, 0, MAX_PASSES - 1);
  }
  if (failures == 0) std::printf("PASSED\n");
  return failures != 0;
}
