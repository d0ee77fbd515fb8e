// The sort of a few thousand keys in one workgroup: one launch instead of the chained passes.
//
// What bounds a sort of this size is latency: the launches, and inside the kernel the barriers and
// the ranking of a pass.  So the keys stay in registers and LDS from the one load to the one
// store, and as few passes as possible run:
//   - Only the bits in which the keys differ count (OR of all keys' differences to the first one).
//   - If those span more than two digits, stable passes over their TOP 2, 3 or 4 digits come first.
//     A few thousand keys then rarely share all of those bits; each key counts the keys of its group
//     that belong before it (equal ones keep their order) and moves there.  How many digits: every wave
//     counts how many pairs of 64 of its keys agree in the top 16, 24 and 32 bits, and the fewest
//     digits are taken for which a key should share them with SMALL_GROUP_MEAN others at most.
//     Should a group turn out larger than SMALL_GROUP_MAX, all digits get their pass, from the lowest
//     (the arrangement so far is a stable one, so equal keys still come out in their original order).
// One copy and one sort, back to back, against the same through the chained passes (eight launches):
// 3001 uint32 53.7 -> 12.0 us, 8192 uint32 56.7 -> 20.9, 8192 float32 58.7 -> 24.3, 3001 (uint64, uint32)
// 81.0 -> 15.7, 8192 float64 79.6 -> 28.3.  (All loads in flight at the start, the values' too, instead of one after
// the other and the values behind the sort: 8192 uint32 23.0 -> 20.9, with uint32 values 29.1 -> 25.0.)  All digits of
// the float64 take 93 us: the passes' ranking is what
// the time goes into, hence the effort to leave passes out.  Beyond 8192 keys one CU is no longer
// fast enough (its ranking alone takes 3 us per pass and 8192 keys).
// Values do not travel with the keys: every key carries its 16-bit index, the values wait in registers, are
// staged in LDS at the end and picked up by it.
#pragma once
#include "common.hpp"
#include "launch.hpp"
#include "radix_rank.hpp"
#include "sort_codec.hpp"

namespace ta {

constexpr int SMALL_ITEMS = 8;  // keys per thread at most
constexpr int SMALL_GROUP_MAX = 24;
constexpr uint32_t SMALL_GROUP_MEAN = 4;
constexpr int SMALL_TOP_DIGITS_MAX = 4;

template <typename K, typename V, bool HAS_VALUES, int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK) void small_sort_kernel(K* __restrict__ keys, V* __restrict__ vals, uint32_t n,
                                                           KeyCodec<K> codec, int begin_bit, int end_bit) {
  constexpr int WAVES = BLOCK / WAVE;
  constexpr int CAP = BLOCK * ITEMS;
  constexpr int SAMPLE_WAVES = WAVES < 8 ? WAVES : 8;  // two per SIMD: more cost time, fewer see too little
  constexpr size_t ITEM = (HAS_VALUES && sizeof(V) > sizeof(K)) ? sizeof(V) : sizeof(K);
  static_assert(BLOCK >= RADIX_SIZE && CAP <= 65536, "a thread per digit; 16-bit indices");
  __shared__ __attribute__((aligned(16))) unsigned char s_items[CAP * ITEM];
  __shared__ uint16_t s_idx[HAS_VALUES ? CAP : 1];
  __shared__ uint32_t s_cnt[WAVES * RADIX_SIZE];
  __shared__ uint32_t s_digit_wave[RADIX_SIZE / WAVE];
  __shared__ uint64_t s_vary[WAVES];
  __shared__ uint32_t s_pairs[SMALL_TOP_DIGITS_MAX + 1];
  __shared__ uint32_t s_large;
  K* s_keys = reinterpret_cast<K*>(s_items);
  V* s_vals = reinterpret_cast<V*>(s_items);

  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int rounds = (int)((n + BLOCK - 1) / BLOCK);                    // uniform, <= ITEMS
  const uint32_t span = (uint32_t)wave * (WAVE * rounds) + lane;       // wave-striped: + r * WAVE
  uint32_t* my_cnt = s_cnt + wave * RADIX_SIZE;
  const K range = (K)((end_bit - begin_bit >= (int)sizeof(K) * 8 ? ~(K)0 : (K)(((K)1 << (end_bit - begin_bit)) - 1)) << begin_bit);

  // ---- load, keys and values, all in flight together: without predicates (a predicated load is waited for before
  // the next is issued), the last element in the place of those behind it; slots past the end sort last
  K e[ITEMS];
  V v[HAS_VALUES ? ITEMS : 1];
  uint32_t idx[ITEMS];
  K first = keys[0];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) e[r] = keys[span + r * WAVE < n ? span + r * WAVE : n - 1];
  if constexpr (HAS_VALUES) {
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) v[r] = vals[span + r * WAVE < n ? span + r * WAVE : n - 1];
  }
  first = codec.encode(first);
  K differ = 0;
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t pos = span + r * WAVE;
    idx[r] = pos;
    e[r] = codec.encode(e[r]);
    differ |= e[r] ^ first;
    if (r >= rounds || pos >= n) e[r] = (K)~(K)0;
  }
  {
    struct Or {
      TA_DEVICE uint64_t operator()(uint64_t a, uint64_t b) const { return a | b; }
    };
    const uint64_t w = wave_reduce((uint64_t)(K)(differ & range), Or{});
    if (lane == 0) s_vary[wave] = w;
  }
  for (int i = threadIdx.x; i < WAVES * RADIX_SIZE; i += BLOCK) s_cnt[i] = 0;
  if (threadIdx.x == 0) s_large = 0;
  if (threadIdx.x <= SMALL_TOP_DIGITS_MAX) s_pairs[threadIdx.x] = 0;
  __syncthreads();
  uint64_t vary = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) vary |= s_vary[w];
  vary = wave_uniform(vary);

  // One stable pass over bits [lo, lo + nbits): afterwards e / idx hold, and s_keys / s_idx mirror, the
  // new arrangement.  s_cnt is all zero at entry and at exit.
  auto pass = [&](int lo, int nbits) {
    uint32_t rank[ITEMS];
    auto digit_of = [&](K x) { return (uint32_t)(x >> lo) & ((1u << nbits) - 1u); };
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
      if (r < rounds) rank[r] = wave_rank_round(digit_of(e[r]), my_cnt);
    __syncthreads();
    uint32_t sum = 0, incl = 0;
    if (threadIdx.x < RADIX_SIZE) {
      const int d = threadIdx.x;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        const uint32_t c = s_cnt[w * RADIX_SIZE + d];
        s_cnt[w * RADIX_SIZE + d] = sum;
        sum += c;
      }
      incl = wave_inclusive_scan(sum, OpPlus{});
      if (lane == WAVE - 1) s_digit_wave[wave] = incl;
    }
    __syncthreads();
    if (threadIdx.x < RADIX_SIZE) {
      const int d = threadIdx.x;
      uint32_t base = incl - sum;
      for (int w = 0; w < wave; ++w) base += s_digit_wave[w];
#pragma unroll
      for (int w = 0; w < WAVES; ++w) s_cnt[w * RADIX_SIZE + d] += base;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      if (r < rounds) {
        const uint32_t p = my_cnt[digit_of(e[r])] + rank[r];
        s_keys[p] = e[r];
        if constexpr (HAS_VALUES) s_idx[p] = (uint16_t)idx[r];
      }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < WAVES * RADIX_SIZE; i += BLOCK) s_cnt[i] = 0;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      if (r < rounds) {
        e[r] = s_keys[span + r * WAVE];
        if constexpr (HAS_VALUES) idx[r] = s_idx[span + r * WAVE];
      }
    }
    __syncthreads();
  };
  if (vary != 0) {
    const int lo = __builtin_ctzll(vary), hi = 63 - __builtin_clzll(vary);
    int digits = (hi - lo + RADIX_BITS) / RADIX_BITS;  // how many get a pass
    const int all_digits = digits;
    if (digits > 2) {
      // pairs among the first 64 keys of a few waves that agree in the top 2, 3, .. digits
      if (wave < SAMPLE_WAVES) {
        const uint64_t live = __builtin_amdgcn_ballot_w64(span < n);
        uint32_t peers_lo = (uint32_t)live, peers_hi = (uint32_t)(live >> 32);
#pragma unroll
        for (int t = 1; t <= SMALL_TOP_DIGITS_MAX; ++t) {
          const int from = hi + 1 - t * RADIX_BITS;
          wave_match_digit((uint32_t)(from >= 0 ? e[0] >> from : e[0] << -from) & (RADIX_SIZE - 1), peers_lo, peers_hi);
          if (t >= 2) {
            const uint32_t group = (uint32_t)__builtin_popcount(peers_lo) + (uint32_t)__builtin_popcount(peers_hi);
            const uint32_t w = wave_reduce(span < n ? group - 1 : 0u, OpPlus{});
            if (lane == 0) atomicAdd(&s_pairs[t], w);
          }
        }
      }
      __syncthreads();
      // (twice the) pairs compared: every whole wave 64 * 63
      const uint32_t whole_waves = n / (WAVE * rounds);
      const uint64_t compared = (uint64_t)(whole_waves < 1 ? 1 : whole_waves < SAMPLE_WAVES ? whole_waves : SAMPLE_WAVES) * (WAVE * (WAVE - 1));
      digits = all_digits;
      for (int t = SMALL_TOP_DIGITS_MAX; t >= 2; --t)
        if (t < all_digits && (uint64_t)s_pairs[t] * n <= SMALL_GROUP_MEAN * compared) digits = t;
    }
    const int top = digits == all_digits ? lo : hi + 1 - digits * RADIX_BITS;
    bool whole = digits == all_digits;  // the passes at hand cover every bit that varies
    int at = top;
    for (;;) {
      const int nbits = hi + 1 - at < RADIX_BITS ? hi + 1 - at : RADIX_BITS;
      pass(at, nbits);
      at += nbits;
      if (at <= hi) continue;
      if (whole) break;
      // groups of keys that share bits [top, hi] (and the constant bits above)
      const K upper = (K)(range & ~(((K)1 << top) - 1)), lower = (K)(range & (((K)1 << top) - 1));
      uint32_t dest[ITEMS];
      bool large = false;
#pragma unroll
      for (int r = 0; r < ITEMS; ++r) {
        const uint32_t p = span + r * WAVE;
        dest[r] = p;
        if (r < rounds && p < n) {
          const K mine_up = e[r] & upper, mine_lo = e[r] & lower;
          uint32_t q = p, after = p + 1;
          uint32_t before = 0, ahead = 0;  // keys of the group in front of this one that belong behind it, and the reverse
          int steps = 0;
          while (q > 0 && steps <= SMALL_GROUP_MAX) {
            const K x = s_keys[q - 1];
            if ((x & upper) != mine_up) break;
            before += (x & lower) > mine_lo ? 1u : 0u;
            --q;
            ++steps;
          }
          while (after < n && steps <= SMALL_GROUP_MAX) {
            const K x = s_keys[after];
            if ((x & upper) != mine_up) break;
            ahead += (x & lower) < mine_lo ? 1u : 0u;
            ++after;
            ++steps;
          }
          large = large || steps > SMALL_GROUP_MAX;
          dest[r] = p - before + ahead;
        }
      }
      if (__builtin_amdgcn_ballot_w64(large) != 0 && lane == 0) s_large = 1;
      __syncthreads();
      if (s_large) {
        whole = true;
        at = lo;
        continue;
      }
#pragma unroll
      for (int r = 0; r < ITEMS; ++r) {
        if (r < rounds) {
          s_keys[dest[r]] = e[r];
          if constexpr (HAS_VALUES) s_idx[dest[r]] = (uint16_t)idx[r];
        }
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < ITEMS; ++r) {
        if (r < rounds) {
          e[r] = s_keys[span + r * WAVE];
          if constexpr (HAS_VALUES) idx[r] = s_idx[span + r * WAVE];
        }
      }
      __syncthreads();
      break;
    }
  }

  // ---- store
  if constexpr (HAS_VALUES) {
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const uint32_t pos = span + r * WAVE;
      if (r < rounds && pos < n) s_vals[pos] = v[r];
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t pos = span + r * WAVE;
    if (r < rounds && pos < n) {
      keys[pos] = codec.decode(e[r]);
      if constexpr (HAS_VALUES) vals[pos] = s_vals[idx[r]];
    }
  }
}

constexpr uint64_t SMALL_SORT_MAX = 1024 * SMALL_ITEMS;

// Sorts n <= SMALL_SORT_MAX keys (and values, if value_bytes is not 0) in place with one launch.
int small_sort(void* keys, void* values, uint32_t n, int key_dtype, size_t value_bytes, int descending, int begin_bit,
               int end_bit, hipStream_t stream);

}  // namespace ta
