// Host-side check of the rule by which a sort of 8-byte keys takes the two-digit way (thrust_amd/csrc/top_digits.hpp,
// the function the plan kernel calls), fed with what the samples of several kinds of keys would say:
//   random keys take it at every size it is meant for, for the length their longest stretches have;
//   keys whose stretches do not fit (copies by the hundred where stretches are long anyway, one key in twenty equal) do not.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#include "../../thrust_amd/csrc/top_digits.hpp"

constexpr float STRETCH_MAX = 2560;

// Keys are drawn by draw(rnd); as the plan kernel counts them.  hot_share: share of one key among them.
static float longest_stretch(double n, uint32_t bins, double values, double hot_share, uint32_t seed) {
  std::mt19937_64 rnd(seed);
  const uint32_t samples = (uint32_t)std::min(n / 64, 16384.0);
  std::vector<uint32_t> count(bins, 0);
  std::vector<bool> seen(ta::TWIN_PLACES, false);
  double pairs = 0, twins = 0, peak = 0;
  std::uniform_real_distribution<double> u(0, 1);
  for (uint32_t i = 0; i < samples; ++i) {
    uint64_t value = u(rnd) < hot_share ? 0 : (uint64_t)(u(rnd) * values);
    uint64_t mixed = (value + seed) * 0x9e3779b97f4a7c15ull;
    mixed ^= mixed >> 31;
    mixed *= 0xbf58476d1ce4e5b9ull;
    mixed ^= mixed >> 29;
    uint32_t& c = count[mixed % bins];
    pairs += c;
    peak = std::max(peak, (double)++c);
    const uint64_t place = mixed * 0x94d049bb133111ebull >> 44;
    twins += seen[place] ? 1 : 0;
    seen[place] = true;
  }
  // the fullest of 256 bins of a digit, as a share: a few deviations above the mean
  const double share = 1.0 / 256 + 3 * std::sqrt(1.0 / 256 / n);
  const double even = bins == 65536 ? n * share * share : n / bins;
  return ta::top_two_digits((float)n, (float)samples, (float)even, (float)pairs, even > STRETCH_MAX / 4 ? (float)twins : 0.0f, (float)peak, STRETCH_MAX);
}

int main() {
  int failures = 0;
  const double random_values = 1e18;
  for (double n : {9e3, 3e4, 1e5, 1e6, 4e6, 1.6e7, 3.3e7, 6.7e7, 1.34e8, 1.5e8}) {
    int declined = 0;
    for (uint32_t seed = 1; seed <= 40; ++seed) {
      const float longest = longest_stretch(n, 65536, random_values, 0, seed);
      const double expected = n / 65536 + 3.5 * std::sqrt(n / 65536);
      if (longest == 0) ++declined;
      else if (longest < expected) {
        std::printf("FAILED: %g random keys: stretches of %g expected, not %g\n", n, expected, longest);
        ++failures;
      }
    }
    if (declined > 1) {
      std::printf("FAILED: %g random keys declined %d times of 40\n", n, declined);
      ++failures;
    }
  }
  struct Case {
    double n, values, hot;
    const char* what;
  };
  for (const Case& c : {Case{1.34e8, 1.34e6, 0, "100 copies of each key"}, Case{1.34e8, 1.34e5, 0, "1000 copies of each key"},
                        Case{6.7e7, 6.7e4, 0, "1000 copies of each key"}, Case{1e6, random_values, 0.05, "a key that is one in twenty"},
                        Case{1e6, random_values, 0.005, "a key that is one in 200"}, Case{1.34e8, random_values, 0.01, "a key that is one in 100"}}) {
    int taken = 0;
    for (uint32_t seed = 1; seed <= 40; ++seed) taken += longest_stretch(c.n, 65536, c.values, c.hot, seed) > 0 ? 1 : 0;
    if (taken > 2) {
      std::printf("FAILED: %g keys, %s: taken %d times of 40\n", c.n, c.what, taken);
      ++failures;
    }
  }
  if (failures == 0) std::printf("PASSED\n");
  return failures != 0;
}
