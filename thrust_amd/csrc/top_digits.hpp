// When a radix sort of 8-byte keys may order the array by its top two digits only.  Plain C++ (also compiled for the
// host by tests/cpp/test_top_digits.cpp, which plays it through for several kinds of keys).
#pragma once

#if defined(__HIPCC__)
#define TA_RULE_FN __host__ __device__ inline
#else
#define TA_RULE_FN inline
#endif

namespace ta {

constexpr unsigned TWIN_PLACES = 1u << 20;

// What the samples say about the stretches of equal top two digits.  All in keys of the whole array; 0: don't take them.
//   even   size of a stretch if digits were independent
//   pairs  pairs of samples that share both digits: the mean size of the stretch a key finds itself in.  What that is
//          above `even` (and above its own scatter) is how many keys come together: copies of one key, or neighbours
//   twins  samples that find their hash's one of TWIN_PLACES taken: copies among the samples, where stretches are so
//          long that `pairs` says little about them.  (S^2 / 2 / TWIN_PLACES samples do so without being equal.)
//   peak   samples in the fullest stretch: one hot key among others
// Returns the length to expect of the longest stretches but for a few in ten thousand.
TA_RULE_FN float top_two_digits(float n, float samples, float even, float pairs, float twins, float peak, float stretch_max) {
  const float per_pair = 2.0f * n / (samples * samples);
  const float mean = pairs * per_pair, scatter = pairs > 0 ? mean / __builtin_sqrtf(pairs) : 0.0f;
  const float chance = samples * samples / (2.0f * TWIN_PLACES);
  const float copies = twins - chance - 3.0f * __builtin_sqrtf(chance);
  const float of_one_key = 1.0f + (copies > 0 ? copies * per_pair : 0.0f);
  float clump = mean - even - 3.0f * scatter;
  clump = clump > of_one_key ? clump : of_one_key;
  const float typical = even > mean - clump ? even : mean - clump;
  float longest = typical + 3.5f * __builtin_sqrtf(typical * clump) + 3.0f * clump;
  if (longest > stretch_max) return 0.0f;
  const float share = samples / n;
  const float expected = longest * share, allowed = stretch_max * share;
  const float usual = expected + 4.5f * __builtin_sqrtf(expected) + 4.5f;
  const float most = allowed - __builtin_sqrtf(allowed);
  if (peak > usual) {
    if (peak > most) return 0.0f;
    const float hot = (peak + 3.0f * __builtin_sqrtf(peak)) / share;  // few samples would say nothing: most > usual here
    longest = longest > hot ? longest : hot < stretch_max ? hot : stretch_max;
  }
  return longest;
}

}  // namespace ta
