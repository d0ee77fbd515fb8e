// The last step of a radix sort whose passes covered the top digits only: the array is in stable order of a
// prefix of the keys, and every stretch of equal prefixes is short enough to be ordered in one workgroup.
//
//   bounds  for every window of `window` positions the first place at or behind its start where a new prefix begins
//           (two digits; stretches of one begin where the histogram says, which finish looks up itself)
//   finish  a workgroup takes the stretches that begin inside its window, orders them by the whole key in registers
//           and LDS and writes them to their place in the caller's array.  More than CAP keys (a stretch that the plan
//           did not expect) are left to the
//   tail    where a workgroup sorts such a window with stable passes through memory
//
// Inside a workgroup the keys go to as many bins as there are places (key minus smallest key, shifted so that the
// largest falls into the last bins): one LDS atomic per key counts a bin and tells the key its place in it, a scan
// turns counts into starts, the keys are laid out by bin, and each key counts the keys of its bin that belong in front
// of it -- the smaller ones and, among equal ones, those that stood in front -- so the atomics' order does not show.
// What bounds it: the latency of its ten steps for the 2000 keys of a workgroup, three workgroups to a CU, and vector
// instructions.  2^27 pairs of (uint64, uint32): 0.69 ms (4.7 TB/s) in place of six passes of 0.69; keys alone 0.56 in place
// of six of 0.48.  Workgroups that loop over windows
// save their dispatch where the chained passes do the sort (40 us for 2^27 keys), but cost registers (0.85 -> 1.19 ms).
// A bin of more than FINISH_BIN_MAX keys (many equal keys, values in clusters) makes the workgroup run stable passes
// over the digits that vary instead: three times as long for 2^27 uint64 that repeat 30 times (the sort still takes 0.8
// of the time of all passes).
#pragma once
#include "common.hpp"
#include "launch.hpp"
#include "radix_rank.hpp"
#include "sort_codec.hpp"
#include "sort_ctl.hpp"

namespace ta {

constexpr uint32_t FINISH_BIN_MAX = 24;

template <typename K, typename V, bool HAS_VALUES>
struct FinishShape {
  static constexpr bool BIG = sizeof(K) == 8 || (HAS_VALUES && sizeof(V) == 8);
  static constexpr int BLOCK = BIG ? 512 : 1024;
  static constexpr int ITEMS = 8;
  static constexpr int CAP = BLOCK * ITEMS;
  static constexpr int WAVES_PER_SIMD = (BIG ? 3 : 2) * BLOCK / WAVE / 4;
  static constexpr uint32_t WINDOW_MIN = BIG ? 1536 : 2048;
  static constexpr uint32_t STRETCH_MAX = CAP - WINDOW_MIN;  // longest stretch of one prefix that can be promised a place
};

// window: see above; sorted: the array in order of its keys' bits from prefix_bit on; bounds[ceil(n / window) + 1]
template <typename K>
__global__ __launch_bounds__(256) void sort_bounds_kernel(const K* __restrict__ keys_a, const K* __restrict__ keys_b, uint32_t n,
                                                          uint32_t cap, uint32_t* __restrict__ bounds, const SortCtl* __restrict__ ctl) {
  if (!ctl->finishes()) return;
  const uint32_t window = ctl->window;
  const uint32_t windows = (n + window - 1) / window;
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i > windows) return;
  if (i == 0 || i == windows) {
    bounds[i] = i == 0 ? 0 : n;
    return;
  }
  const K* __restrict__ x = ctl->fast_src_alt ? keys_b : keys_a;
  const int bit = (int)ctl->prefix_bit;
  const uint32_t edge = i * window;
  const uint32_t reach = cap - window;  // a new prefix is expected at edge + reach at the latest
  const K here = x[edge - 1] >> bit;
  uint32_t lo = edge, hi = n - edge < reach ? n : edge + reach;  // the answer lies in [lo, hi]
  if (hi < n && (x[hi] >> bit) == here) {
    lo = hi + 1;
    hi = n;
  }
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if ((x[mid] >> bit) == here) lo = mid + 1;
    else hi = mid;
  }
  bounds[i] = lo;
}

// Inclusive sum over each row of 16 lanes.
TA_DEVICE uint32_t row_inclusive_scan(uint32_t x) {
  x += dpp_move<DPP_ROW_SHR1>(0u, x);
  x += dpp_move<DPP_ROW_SHR2>(0u, x);
  x += dpp_move<DPP_ROW_SHR4>(0u, x);
  x += dpp_move<DPP_ROW_SHR8>(0u, x);
  return x;
}

template <typename K, typename V, bool HAS_VALUES>
__global__ __launch_bounds__((FinishShape<K, V, HAS_VALUES>::BLOCK), (FinishShape<K, V, HAS_VALUES>::WAVES_PER_SIMD)) void sort_finish_kernel(
    K* __restrict__ keys_a, const K* __restrict__ keys_b, V* __restrict__ vals_a, const V* __restrict__ vals_b, uint32_t n,
    KeyCodec<K> codec, const uint32_t* __restrict__ bounds,  // (8-byte keys)
    const uint32_t* __restrict__ hist, const SortCtl* __restrict__ ctl, uint32_t* __restrict__ long_windows,
    uint32_t* __restrict__ long_list,  // windows for the tail, *long_windows of them
    uint32_t* __restrict__ status, uint64_t status_words) {
  using Shape = FinishShape<K, V, HAS_VALUES>;
  constexpr int BLOCK = Shape::BLOCK, ITEMS = Shape::ITEMS, CAP = Shape::CAP, WAVES = BLOCK / WAVE;
  constexpr int BINS = CAP;                // 16-bit counts, two to a word
  constexpr int BIN_WORDS = BINS / 2;
  constexpr int LOG_BINS = __builtin_ctz(BINS);
  constexpr int MY_WORDS = BIN_WORDS / BLOCK;
  constexpr int TRASH = 32;
  constexpr int SIDE = 7;                  // places looked at on either side of a key
  // 8-byte keys are told apart by 32 bits; they are then moved like values, by the 16-bit place they had before
  constexpr bool KEYS_MOVE = sizeof(K) == 8;
  constexpr bool HAS_IDX = KEYS_MOVE || HAS_VALUES;
  constexpr size_t ITEM = (HAS_VALUES && sizeof(V) > sizeof(K)) ? sizeof(V) : sizeof(K);
  constexpr size_t CODE_BYTES = (CAP + 2 * (SIDE + 1)) * sizeof(uint32_t);
  constexpr size_t REST_BYTES = KEYS_MOVE ? CAP * sizeof(uint32_t) : 0;  // what the codes leave out of a key
  constexpr size_t FRONT_BYTES = CODE_BYTES + REST_BYTES > CAP * ITEM ? CODE_BYTES + REST_BYTES : CAP * ITEM;
  static_assert(BLOCK >= RADIX_SIZE && (CAP & (CAP - 1)) == 0 && CAP <= 8192 && MY_WORDS % 4 == 0, "shape");
  static_assert(WAVES * RADIX_SIZE <= BIN_WORDS, "the passes' counters lie over the bins");

  if (!ctl->finishes()) {
    // the chained passes do the sort: their tile descriptors are cleared here, not by every call's first kernel
    const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
    for (uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; i < status_words; i += stride) status[i] = 0;
    return;
  }
  const uint32_t window = ctl->window;
  const uint32_t windows = (n + window - 1) / window;
  __shared__ __attribute__((aligned(16))) unsigned char s_items[FRONT_BYTES];
  __shared__ uint16_t s_idx[HAS_IDX ? CAP : 1];
  __shared__ __attribute__((aligned(16))) uint32_t s_bin[BIN_WORDS + 4 + TRASH];  // behind the bins: where lanes without a key count
  __shared__ uint32_t s_wave[WAVES];
  __shared__ uint32_t s_digit_wave[RADIX_SIZE / WAVE];
  __shared__ K s_differ[WAVES];
  __shared__ uint32_t s_most;
  uint32_t* s_code = reinterpret_cast<uint32_t*>(s_items) + SIDE + 1;
  uint32_t* s_rest = reinterpret_cast<uint32_t*>(s_items + CODE_BYTES);
  K* s_keys = reinterpret_cast<K*>(s_items);
  V* s_vals = reinterpret_cast<V*>(s_items);

  const uint32_t w = blockIdx.x;
  if (w >= windows) return;
  uint32_t first, count;
  if constexpr (sizeof(K) == 8) {
    first = bounds[w];
    count = bounds[w + 1] - first;
  } else {
    // one digit: its stretches begin where the histogram says
    const uint4 starts = reinterpret_cast<const uint4*>(hist + (ctl->prefix_bit / RADIX_BITS) * RADIX_SIZE)[threadIdx.x % WAVE];
    auto start_behind = [&](uint32_t edge) {
      uint32_t at = n;
      for (const uint32_t s : {starts.x, starts.y, starts.z, starts.w}) at = s >= edge && s < at ? s : at;
      return wave_reduce(at, OpMin{});
    };
    first = start_behind(w * window);
    count = (w + 1 == windows ? n : start_behind((w + 1) * window)) - first;
  }
  if (count == 0) return;
  const uint32_t tid = threadIdx.x;
  if (count > (uint32_t)CAP) {
    if (tid == 0) long_list[atomicAdd(long_windows, 1u)] = w;
    return;
  }
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const int rounds = (int)((count + BLOCK - 1) / BLOCK);
  const K* __restrict__ keys_in = (ctl->fast_src_alt ? keys_b : keys_a) + first;
  const V* __restrict__ vals_in = HAS_VALUES ? (ctl->fast_src_alt ? vals_b : vals_a) + first : nullptr;
  K* __restrict__ keys_out = keys_a + first;
  V* __restrict__ vals_out = HAS_VALUES ? vals_a + first : nullptr;
  // f(r, the place r * BLOCK + tid) for all rounds, each behind a branch of its own (in pairs, without a branch inside,
  // the loads of two are in flight together, but an odd round more is computed, and with values registers spill: 0.97
  // against 0.73 ms for 2^27 pairs of (uint64, uint32), 0.63 against 0.56 for keys alone, which spill neither way)
  // (opaque copy: what a sweep derives from the place is not kept in registers for the next)
  auto each_round = [&](auto f) {
    uint32_t t = tid;
    asm volatile("" : "+v"(t));
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      if (r < rounds) f(r, (uint32_t)r * BLOCK + t);
    }
  };

  // ---- load; lanes without a key repeat the last one
  K e[ITEMS];
  V v[HAS_VALUES ? ITEMS : 1];
  each_round([&](int r, uint32_t p) { e[r] = keys_in[p < count ? p : count - 1]; });
  auto load_values = [&] {
    each_round([&](int r, uint32_t p) { v[r] = vals_in[p < count ? p : count - 1]; });
  };
  // the prefixes are in order, so the first and the last one say where all keys lie
  const int prefix_bit = (int)ctl->prefix_bit;
  const K lo = keys_in[0] >> prefix_bit << prefix_bit;
  const K range = (keys_in[count - 1] | (((K)1 << prefix_bit) - 1)) - lo;
  const int width = 64 - __builtin_clzll((uint64_t)range);  // prefix_bit >= 8
  const int shift = width > LOG_BINS ? width - LOG_BINS : 0;
  // what tells keys apart, in 32 bits, and a key's bin from that
  const int code_shift = KEYS_MOVE && width > 32 ? width - 32 : 0;
  const int bin_shift = shift - code_shift;
  auto decoded = [&](K x) { return codec.plain ? x : codec.decode(x); };  // (uniform)
  auto code_of = [&](K x) { return (uint32_t)((K)(x - lo) >> code_shift); };
#pragma unroll
  for (int i = 0; i < MY_WORDS / 4; ++i) reinterpret_cast<uint4*>(s_bin)[(uint32_t)i * BLOCK + tid] = uint4{0, 0, 0, 0};
  if (tid == 0) s_most = 4;
  __syncthreads();

  // ---- bins
  uint32_t slot[ITEMS];
  auto forget = [](K& x) { asm volatile("" : "+v"(x)); };  // ... nor what it derives from a key
  each_round([&](int r, uint32_t p) {
    const uint32_t b = code_of(e[r]) >> bin_shift;
    const uint32_t word = p < count ? b >> 1 : (uint32_t)(BIN_WORDS + 4) + lane % TRASH;
    slot[r] = __hip_atomic_fetch_add(&s_bin[word], (b & 1u) ? 1u << 16 : 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    forget(e[r]);
  });
  __syncthreads();
  {
    typedef uint16_t Two __attribute__((ext_vector_type(2)));
    uint32_t c[MY_WORDS];
#pragma unroll
    for (int i = 0; i < MY_WORDS / 4; ++i) *reinterpret_cast<uint4*>(c + 4 * i) = reinterpret_cast<const uint4*>(s_bin)[tid * (MY_WORDS / 4) + i];
    uint32_t sums = 0;  // no half exceeds the number of keys
    Two most2 = {0, 0};
#pragma unroll
    for (int i = 0; i < MY_WORDS; ++i) {
      sums += c[i];
      most2 = __builtin_elementwise_max(most2, __builtin_bit_cast(Two, c[i]));
    }
    const uint32_t sum = (sums & 0xffffu) + (sums >> 16);
    const uint32_t most = most2.x > most2.y ? most2.x : most2.y;
    if (most > 4) atomicMax(&s_most, most);  // few lanes
    const uint32_t incl = wave_inclusive_scan(sum, OpPlus{});
    if (lane == WAVE - 1) s_wave[wave] = incl;
    __syncthreads();
    static_assert(WAVES <= 16, "one DPP row holds the waves' sums");
    const uint32_t before = row_inclusive_scan(s_wave[lane % WAVES]);
    uint32_t at = incl - sum + (wave > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)before, __builtin_amdgcn_readfirstlane(wave - 1) & (WAVES - 1)) : 0u);
    at |= at << 16;
#pragma unroll
    for (int i = 0; i < MY_WORDS; ++i) {
      const uint32_t both = c[i] + __builtin_amdgcn_alignbit(c[i], c[i], 16);  // in either half
      c[i] = at + (c[i] << 16);
      at += both;
    }
#pragma unroll
    for (int i = 0; i < MY_WORDS / 4; ++i) reinterpret_cast<uint4*>(s_bin)[tid * (MY_WORDS / 4) + i] = *reinterpret_cast<const uint4*>(c + 4 * i);
  }
  __syncthreads();

  const uint32_t most = s_most;  // keys in the fullest bin, or 4
  const bool place_by_place = most > (uint32_t)SIDE + 1;
  if (most <= FINISH_BIN_MAX) {
    const uint16_t* s_start = reinterpret_cast<const uint16_t*>(s_bin);
    each_round([&](int r, uint32_t) {
      const uint32_t b = code_of(e[r]) >> bin_shift;
      slot[r] = ((b & 1u) ? slot[r] >> 16 : slot[r] & 0xffffu) + s_start[b];
      forget(e[r]);
    });
    each_round([&](int r, uint32_t p) {
      if (p < count) {
        s_code[slot[r]] = code_of(e[r]);
        if constexpr (HAS_IDX) s_idx[slot[r]] = (uint16_t)p;
      }
      forget(e[r]);
    });
    if constexpr (KEYS_MOVE) {
      if (place_by_place) {
        each_round([&](int r, uint32_t p) {
          if (p < count) s_rest[slot[r]] = (uint32_t)e[r] - (uint32_t)lo;
        });
      }
    }
    if (tid < SIDE) {  // what lies outside belongs outside
      s_code[-1 - (int)tid] = 0;
      s_code[count + tid] = ~0u;
    }
    __syncthreads();
    // not earlier: the registers hold the keys until here (asked for with the 8-byte keys, values cost 32 bytes of
    // spills: 2^27 pairs 0.73 against 0.69 ms, 1.6e7 109 against 82 us)
    if constexpr (HAS_VALUES) load_values();
    // ---- inside the bins: keys of lower bins are smaller and lie in front, so a lane counts the keys on the wrong
    // side of its own, without asking for their bins, as far as the fullest bin can reach.  4-byte keys leave
    // straight for their places: a wave's lie next to each other but for those steps.
    uint32_t move[HAS_IDX ? ITEMS : 1];  // place now, and in the workgroup before << 16
    auto settle = [&](auto side, auto by_place) {
      auto place = [&](uint32_t p, uint32_t& packed) {
        const uint32_t mine = s_code[p];
        const uint32_t my_idx = HAS_IDX ? s_idx[p] : 0u;
        uint32_t q = p;
        bool equal = false;
#pragma unroll
        for (int j = 1; j <= side(); ++j) {
          const uint32_t left = s_code[(int)p - j], right = s_code[(int)p + j];
          q -= left > mine ? 1u : 0u;
          q += right < mine ? 1u : 0u;
          if constexpr (HAS_IDX) equal = equal || left == mine || right == mine;
        }
        if (p < count) {
          if (by_place() || equal) {
            // place by place in the key's own bin: equal codes by what they leave out of the key (from LDS where many
            // are asked for it) and then in the order before
            const uint32_t b = mine >> bin_shift;
            const uint32_t from = s_start[b], to = b + 1 < (uint32_t)BINS ? s_start[b + 1] : count;
            const uint32_t my_rest = KEYS_MOVE && by_place() ? s_rest[p] : 0u;
            q = from;
            for (uint32_t j = from; j < to; ++j) {
              const uint32_t x = s_code[j];
              const uint32_t i = HAS_IDX ? s_idx[j] : j;
              bool front = i < (HAS_IDX ? my_idx : p);
              if constexpr (KEYS_MOVE && by_place()) {
                const uint32_t rest = s_rest[j];
                front = rest < my_rest || (rest == my_rest && front);
              } else if constexpr (KEYS_MOVE) {
                if (x == mine && code_shift != 0) {
                  const K a = keys_in[i], whole = keys_in[my_idx];
                  front = a < whole || (a == whole && front);
                }
              }
              q += x < mine || (x == mine && front) ? 1u : 0u;
            }
          }
          if constexpr (!KEYS_MOVE) keys_out[q] = decoded((K)(lo + mine));
        }
        packed = q | my_idx << 16;
      };
      if constexpr (HAS_IDX) {
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
          if (r < rounds) place((uint32_t)r * BLOCK + tid, move[r]);
        }
      } else {
        uint32_t unused;
#pragma unroll 2
        for (int r = 0; r < rounds; ++r) place((uint32_t)r * BLOCK + tid, unused);
      }
    };
    if (most <= 4) settle(std::integral_constant<int, 3>{}, std::false_type{});
    else if (most <= 6) settle(std::integral_constant<int, 5>{}, std::false_type{});
    else if (most <= SIDE + 1) settle(std::integral_constant<int, SIDE>{}, std::false_type{});
    else settle(std::integral_constant<int, 0>{}, std::true_type{});
    if constexpr (KEYS_MOVE) {
      __syncthreads();  // the codes have been read out of the room the keys take now
      each_round([&](int r, uint32_t p) { s_keys[p] = e[r]; });
      __syncthreads();
      each_round([&](int r, uint32_t p) {
        if (p < count) keys_out[move[r] & 0xffffu] = decoded(s_keys[move[r] >> 16]);
      });
    }
    if constexpr (HAS_VALUES) {
      __syncthreads();
      each_round([&](int r, uint32_t p) { s_vals[p] = v[r]; });
      __syncthreads();
      each_round([&](int r, uint32_t p) {
        if (p < count) vals_out[move[r] & 0xffffu] = s_vals[move[r] >> 16];
      });
    }
    return;
  }

  // ---- stable passes over the digits that vary.  A lane's keys are 64 places apart now (loaded again), slots past
  // the end sort last.  The keys move through LDS with their 16-bit place in the workgroup, by which the values
  // are picked up at the end.
  const uint32_t span = (uint32_t)wave * (WAVE * rounds) + lane;  // + r * WAVE
  uint32_t* s_cnt = s_bin;                                        // [WAVES][RADIX_SIZE]
  uint32_t* my_cnt = s_cnt + wave * RADIX_SIZE;
  K differ = 0;
  uint32_t idx_rank[ITEMS];  // place before, and the rank in a pass << 16
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t p = span + r * WAVE;
    idx_rank[r] = p;
    if (r < rounds) {
      const K x = keys_in[p < count ? p : count - 1];
      differ |= x ^ lo;
      e[r] = p < count ? x : (K)~(K)0;
    }
  }
  struct Or {
    TA_DEVICE K operator()(K a, K b) const { return a | b; }
  };
  differ = wave_reduce(differ, Or{});
  __syncthreads();
  if (lane == 0) s_differ[wave] = differ;
  for (int i = tid; i < WAVES * RADIX_SIZE; i += BLOCK) s_cnt[i] = 0;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < WAVES; ++w) differ |= s_differ[w];
  const uint64_t vary = wave_uniform((uint64_t)differ);
  for (int at = 0; at < (int)sizeof(K) * 8; at += RADIX_BITS) {
    if (((vary >> at) & (RADIX_SIZE - 1)) == 0) continue;
    auto digit_of = [&](K x) { return (uint32_t)(x >> at) & (RADIX_SIZE - 1u); };
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      if (r < rounds) {
        idx_rank[r] |= wave_rank_round(digit_of(e[r]), my_cnt) << 16;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
    uint32_t sum = 0, incl = 0;
    if (tid < RADIX_SIZE) {
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        const uint32_t c = s_cnt[w * RADIX_SIZE + tid];
        s_cnt[w * RADIX_SIZE + tid] = sum;
        sum += c;
      }
      incl = wave_inclusive_scan(sum, OpPlus{});
      if (lane == WAVE - 1) s_digit_wave[wave] = incl;
    }
    __syncthreads();
    if (tid < RADIX_SIZE) {
      uint32_t base = incl - sum;
      for (int w = 0; w < wave; ++w) base += s_digit_wave[w];
#pragma unroll
      for (int w = 0; w < WAVES; ++w) s_cnt[w * RADIX_SIZE + tid] += base;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      if (r < rounds) {
        const uint32_t p = my_cnt[digit_of(e[r])] + (idx_rank[r] >> 16);
        s_keys[p] = e[r];
        if constexpr (HAS_VALUES) s_idx[p] = (uint16_t)idx_rank[r];
      }
    }
    __syncthreads();
    for (int i = tid; i < WAVES * RADIX_SIZE; i += BLOCK) s_cnt[i] = 0;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      if (r < rounds) {
        e[r] = s_keys[span + r * WAVE];
        idx_rank[r] = HAS_VALUES ? s_idx[span + r * WAVE] : 0u;
      }
    }
    __syncthreads();
  }
  if constexpr (HAS_VALUES) {
    __syncthreads();
    for (uint32_t p = tid; p < count; p += BLOCK) s_vals[p] = vals_in[p];
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t p = span + r * WAVE;
    if (r < rounds && p < count) {
      keys_out[p] = codec.decode(e[r]);
      if constexpr (HAS_VALUES) vals_out[p] = s_vals[idx_rank[r] & 0xffffu];
    }
  }
}

// The windows that do not fit a workgroup of the last step: stable passes over the digits that vary in the window,
// between the place of the window in the two buffers (its own in either, so nobody else reads or writes them).
// Tiles of TAIL_BLOCK * TAIL_ITEMS keys are ranked as in a chained pass, one after the other, so the order of the tiles
// needs no look-back.  Bound by latency: one workgroup has nothing else to do meanwhile.  A sort of 2^27 uint64 with one
// value 1e4 times takes 2.09 ms, 1.96 without it, 4.14 with all digits' passes.  The plan bounds a window's keys: c equal
// prefixes weigh c / n in both digits, and the product of the heaviest shares times n fits a workgroup.
// Where no window is left over it copies the result back if it sits in the alternate buffer, or does nothing.
constexpr int TAIL_BLOCK = 1024;
constexpr int TAIL_ITEMS = 8;

template <typename K, typename V, bool HAS_VALUES>
__global__ __launch_bounds__(TAIL_BLOCK) void sort_tail_kernel(K* keys_a, K* keys_b, V* vals_a, V* vals_b, uint32_t n,
                                                               KeyCodec<K> codec, const uint32_t* __restrict__ bounds,
                                                               const uint32_t* __restrict__ long_list,
                                                               const SortCtl* __restrict__ ctl) {
  constexpr int WAVES = TAIL_BLOCK / WAVE;
  constexpr int DIGITS = (int)sizeof(K);
  constexpr uint32_t TILE = TAIL_BLOCK * TAIL_ITEMS;
  __shared__ uint32_t s_hist[DIGITS][RADIX_SIZE];
  __shared__ uint32_t s_cnt[WAVES * RADIX_SIZE];
  __shared__ uint32_t s_base[RADIX_SIZE];  // where the next key of a digit goes
  __shared__ uint32_t s_digit_wave[RADIX_SIZE / WAVE];
  __shared__ uint32_t s_constant;          // digits that all keys share, one bit each
  const uint32_t tid = threadIdx.x;
  if (ctl->copies_back()) {
    // 2^27 uint64: 418 us with four keys of a lane in flight, 446 with one; with uint32 values 689 and 607 us
    constexpr int COPIES = HAS_VALUES ? 1 : 4;
    const uint64_t stride = (uint64_t)gridDim.x * TAIL_BLOCK;
    for (uint64_t i = (uint64_t)blockIdx.x * TAIL_BLOCK + tid; i < n; i += COPIES * stride) {
      K k[COPIES];
      V v[HAS_VALUES ? COPIES : 1];
#pragma unroll
      for (int c = 0; c < COPIES; ++c) {
        const uint64_t j = i + c * stride, from = j < n ? j : i;
        k[c] = keys_b[from];
        if constexpr (HAS_VALUES) v[c] = vals_b[from];
      }
#pragma unroll
      for (int c = 0; c < COPIES; ++c) {
        const uint64_t j = i + c * stride;
        if (j < n) {
          keys_a[j] = k[c];
          if constexpr (HAS_VALUES) vals_a[j] = v[c];
        }
      }
    }
    return;
  }
  if (!ctl->finishes()) return;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  uint32_t* my_cnt = s_cnt + wave * RADIX_SIZE;
  for (uint32_t item = blockIdx.x; item < ctl->long_windows; item += gridDim.x) {
    const uint32_t w = long_list[item];
    const uint32_t first = bounds[w], count = bounds[w + 1] - first;
    bool in_alt = ctl->fast_src_alt != 0;  // where the keys are now
    __syncthreads();                       // the window before is done with the LDS
    for (uint32_t i = tid; i < (uint32_t)(DIGITS * RADIX_SIZE); i += TAIL_BLOCK) (&s_hist[0][0])[i] = 0;
    for (uint32_t i = tid; i < (uint32_t)(WAVES * RADIX_SIZE); i += TAIL_BLOCK) s_cnt[i] = 0;
    if (tid == 0) s_constant = 0;
    __syncthreads();
    {
      const K* x = (in_alt ? keys_b : keys_a) + first;
#pragma unroll 4
      for (uint32_t p = tid; p < count; p += TAIL_BLOCK) {
        const K k = x[p];
#pragma unroll
        for (int d = 0; d < DIGITS; ++d)
          __hip_atomic_fetch_add(&s_hist[d][(uint32_t)(k >> (d * RADIX_BITS)) & (RADIX_SIZE - 1u)], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
    __syncthreads();
    if (tid < RADIX_SIZE) {
#pragma unroll
      for (int d = 0; d < DIGITS; ++d)
        if (s_hist[d][tid] == count) atomicOr(&s_constant, 1u << d);
    }
    __syncthreads();
    const uint32_t constant = __builtin_amdgcn_readfirstlane(s_constant);
    for (int d = 0; d < DIGITS; ++d) {
      if (constant >> d & 1u) continue;
      const int at = d * RADIX_BITS;
      auto digit_of = [&](K x) { return (uint32_t)(x >> at) & (RADIX_SIZE - 1u); };
      const K* keys_in = (in_alt ? keys_b : keys_a) + first;
      K* keys_out = (in_alt ? keys_a : keys_b) + first;
      const V* vals_in = HAS_VALUES ? (in_alt ? vals_b : vals_a) + first : nullptr;
      V* vals_out = HAS_VALUES ? (in_alt ? vals_a : vals_b) + first : nullptr;
      uint32_t c = 0, incl = 0;
      if (tid < RADIX_SIZE) {
        c = s_hist[d][tid];
        incl = wave_inclusive_scan(c, OpPlus{});
        if (lane == WAVE - 1) s_digit_wave[wave] = incl;
      }
      __syncthreads();
      if (tid < RADIX_SIZE) {
        uint32_t base = incl - c;
        for (int v = 0; v < wave; ++v) base += s_digit_wave[v];
        s_base[tid] = base;
      }
      for (uint32_t tile = 0; tile < count; tile += TILE) {
        K e[TAIL_ITEMS];
        V v[HAS_VALUES ? TAIL_ITEMS : 1];
        uint32_t rank[TAIL_ITEMS];
        const uint32_t span = tile + (uint32_t)wave * (WAVE * TAIL_ITEMS) + lane;
        // slots past the end (of the last tile) repeat the last key and count as all ones: they come last
#pragma unroll
        for (int r = 0; r < TAIL_ITEMS; ++r) {
          const uint32_t p = span + r * WAVE, q = p < count ? p : count - 1;
          e[r] = keys_in[q];
          if constexpr (HAS_VALUES) v[r] = vals_in[q];
        }
#pragma unroll
        for (int r = 0; r < TAIL_ITEMS; ++r) {
          rank[r] = wave_rank_round(span + r * WAVE < count ? digit_of(e[r]) : RADIX_SIZE - 1u, my_cnt);
          __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        if (tid < RADIX_SIZE) {
          uint32_t sum = s_base[tid];
#pragma unroll
          for (int k = 0; k < WAVES; ++k) {
            const uint32_t t = s_cnt[k * RADIX_SIZE + tid];
            s_cnt[k * RADIX_SIZE + tid] = sum;
            sum += t;
          }
          s_base[tid] = sum;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < TAIL_ITEMS; ++r) {
          if (span + r * WAVE < count) {
            const uint32_t q = my_cnt[digit_of(e[r])] + rank[r];
            keys_out[q] = e[r];
            if constexpr (HAS_VALUES) vals_out[q] = v[r];
          }
        }
        // a wave's counters are its own until the next barrier
#pragma unroll
        for (int i = 0; i < RADIX_SIZE / WAVE; ++i) my_cnt[i * WAVE + lane] = 0;
      }
      __syncthreads();  // the next pass reads what this one has written
      in_alt = !in_alt;
    }
    if (in_alt || !codec.plain) {
      for (uint32_t p = tid; p < count; p += TAIL_BLOCK) {
        const uint32_t i = first + p;
        keys_a[i] = codec.decode(in_alt ? keys_b[i] : keys_a[i]);
        if constexpr (HAS_VALUES)
          if (in_alt) vals_a[i] = vals_b[i];
      }
    }
  }
}

}  // namespace ta
