// thrust_amd_sort_keys / thrust_amd_sort_pairs: onesweep least-significant-digit radix sort (up to 8192
// keys: one workgroup, small_sort.hpp).
//
//   init       zeroes the digit histograms, the tickets and the tile descriptors of the passes (of the first one or two,
//              where the short way is open: the last step clears the others if they are needed)
//   histogram  one read of the keys builds the 256-bin histogram of EVERY 8-bit digit
//   plan       exclusive scan of each histogram -> global digit offsets; a digit whose one
//              bin holds all n keys is marked "skip" (the reference's sequential radix
//              sort does the same, thrust/system/detail/sequential/stable_radix_sort.inl:
//              264-283), and the ping-pong source of every pass is derived from that.  Where the
//              top one or two digits leave short stretches of equal prefixes, only their passes run
//              and radix_finish.hpp orders the stretches
//   pass x P   chained digit-binning pass ("onesweep"): a tile ranks its keys by digit,
//              learns the global offset of each of its 256 digit runs by decoupled
//              look-back over the tiles before it, and scatters keys (and values)
//   copy-back  only if an odd number of passes ran (8-byte keys: in the launch of the short way's tail)
//   rest       behind the short way of a short array: the passes left over and the copy back in one launch
//
// Ranking inside a tile uses the wave64 match pattern (radix_rank.hpp): rank = wave-private LDS counter
// + number of peers in lower lanes.  Lanes hold keys wave-striped (lane l of wave w holds
// keys l, 64+l, ... of the wave's span), so (round, lane) order is memory order and the
// pass is stable.  Keys and values are then exchanged through LDS so that global stores
// are contiguous per digit run.
//
// Tile order is a dynamic ticket, so the look-back only waits for tiles that have
// started: one ticket counter per class of blockIdx % 8, so that neighbouring tiles run on
// the same XCD (sort_tickets.hpp).  Tile descriptors are one word per (tile, digit): 2 status bits above a count,
// 32-bit words for n < 2^30 keys and 64-bit words up to the limit of 2^32 - 1 keys per call
// (positions and histogram counts are 32-bit).
//
// Algorithmic HBM traffic for K-byte keys, V-byte values and P digits that vary: K*n (histogram) + P * 2*(K+V)*n;
// by the short way with one or two digits D: K*n + (D + 1) * 2*(K+V)*n.  Replaces cub::DeviceRadixSort as called from
// thrust/system/cuda/detail/sort.h:1326-1508.
#include "common.hpp"
#include "dispatch.hpp"
#include "launch.hpp"
#include "radix_finish.hpp"
#include "radix_rank.hpp"
#include "small_sort.hpp"
#include "sort_codec.hpp"
#include "sort_tickets.hpp"
#include "top_digits.hpp"

namespace ta {

constexpr uint64_t SORT_MAX_N = (1ull << 32) - 1;       // positions and counts are 32-bit
constexpr uint64_t SORT_MAX_N_NARROW = (1ull << 30) - 1;  // ... and fit 30 bits up to here

// Tile descriptor word: 2 status bits above a count.  32-bit words (30-bit counts) serve
// sorts of fewer than 2^30 keys, 64-bit words the larger ones.
template <typename D>
struct Descriptor {
  static constexpr int SHIFT = (int)sizeof(D) * 8 - 2;
  static constexpr D VALUE_MASK = ((D)1 << SHIFT) - 1;
  static constexpr D PARTIAL = (D)1 << SHIFT;
  static constexpr D INCLUSIVE = (D)2 << SHIFT;
};

constexpr uint32_t TICKET_WORDS = MAX_PASSES * TICKET_CLASSES * TICKET_STRIDE;

// A tile waits for its predecessors' counts in a loop.  Every predecessor is taken by a running
// workgroup as long as every class keeps receiving its workgroups while slots are free -- which
// holds when workgroups are bound to XCDs in turn, and when they are dispatched in order to at
// least 64 slots.  Should neither hold, a tile that has polled this often stops waiting: it
// uses what it has summed so far (its positions stay inside the array: a prefix can only be too
// small), sets SortCtl::gave_up, and every tile that sees the flag does the same, so the
// kernel ends instead of hanging.  The launches behind it do nothing then (SortCtl::strike_out): the
// call ends with an unfinished sort, keys out of order and in their encoded form.
constexpr uint32_t LOOKBACK_SPIN_LIMIT = 1u << 21;

struct SortGeometry {
  int passes;
  int begin_bit;
  int end_bit;
};

// ------------------------------------------------------------------ init
__global__ __launch_bounds__(256) void sort_init_kernel(uint32_t* __restrict__ words, uint64_t count) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride)
    words[i] = 0;
}

// ------------------------------------------------------------------ histogram
// One workgroup per CU with up to 128 KiB of LDS: every bin exists in COPIES copies and
// lane l only ever touches copy l % COPIES, so with 32 copies the 64 lanes of an LDS
// atomic fall on 32 distinct banks whatever the digits are (random digits on a single
// copy serialise about five-fold on bank conflicts).  Keys are read with 16-byte loads;
// their order does not matter here.
// WHOLE_BYTES: the keys need no encoding and the sorted bits are NP whole bytes starting
// at bit 0 (the usual full-range sort of unsigned keys), so every digit is a bit-field
// extract at a constant position.
constexpr int HIST_BLOCK = 1024;
constexpr int HIST_UNROLL = 4;  // 16-byte vectors in flight per lane
constexpr uint32_t SAMPLES = 16384;  // keys the plan looks at, at most

// Keys taken from all over the array, one from each stretch of `step` at a place that follows no pattern.
// The workgroups of the histogram kernel fetch them on the side: 16384 loads from as many pages take one
// workgroup 40 us.
template <typename K>
struct Sampling {
  K* out;              // [count], encoded
  uint32_t per_block;  // taken by each workgroup, <= HIST_BLOCK (0: none)
  uint32_t count;
  uint32_t step;
  TA_DEVICE uint32_t position(uint32_t j) const {
    return j * step + (uint32_t)(((uint64_t)(j * 2654435769u) * step) >> 32);
  }
};

template <typename K, int NP, bool WHOLE_BYTES>
__global__ __launch_bounds__(HIST_BLOCK) void sort_histogram_kernel(const K* __restrict__ keys,
                                                                     uint64_t n, KeyCodec<K> codec,
                                                                     SortGeometry geo,
                                                                     uint32_t* __restrict__ hist,
                                                                     Sampling<K> sampling) {
  constexpr int COPIES = NP <= 4 ? 32 : 16;
  constexpr int BINS = NP * RADIX_SIZE;
  constexpr int VEC = Vec16<K>::N;
  __shared__ uint32_t s_hist[BINS * COPIES];
  for (int i = threadIdx.x; i < BINS * COPIES; i += HIST_BLOCK) s_hist[i] = 0;
  __syncthreads();
  uint32_t* my_copy = s_hist + (threadIdx.x % COPIES);
  // its address says nothing yet about what is counted below: the load is on its way meanwhile
  const bool takes_sample = threadIdx.x < sampling.per_block;
  K sample = 0;
  if (takes_sample) sample = keys[sampling.position(blockIdx.x * sampling.per_block + threadIdx.x)];

  auto count = [&](K k) {
    const K e = (WHOLE_BYTES || codec.plain) ? k : codec.encode(k);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int lo = WHOLE_BYTES ? p * RADIX_BITS : geo.begin_bit + p * RADIX_BITS;
      const int nb = (WHOLE_BYTES || p < NP - 1) ? RADIX_BITS : (geo.end_bit - lo);
      const uint32_t d = (uint32_t)(e >> lo) & ((1u << nb) - 1u);
      __hip_atomic_fetch_add(my_copy + (p * RADIX_SIZE + d) * COPIES, 1u, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  };

  // head: elements before the first 16-byte boundary; tail: what the vectors leave over
  const uint64_t mis = (reinterpret_cast<uintptr_t>(keys) & 15u) / sizeof(K);
  const uint64_t head = mis ? ((VEC - mis) < n ? (VEC - mis) : n) : 0;
  const uint64_t vecs = (n - head) / VEC;
  const uint64_t tail_begin = head + vecs * VEC;
  if (blockIdx.x == 0) {
    if (threadIdx.x < head) count(keys[threadIdx.x]);
    if (tail_begin + threadIdx.x < n) count(keys[tail_begin + threadIdx.x]);
  }
  const Vec16<K>* body = reinterpret_cast<const Vec16<K>*>(keys + head);
  constexpr uint64_t TILE_VECS = (uint64_t)HIST_BLOCK * HIST_UNROLL;
  // Whole tiles: no predicates, and the next tile's vectors are in flight while this
  // tile's are counted (two register buffers in turn; the loop body always loads, so
  // the waits before counting only cover the older buffer).
  const uint64_t whole_tiles = vecs / TILE_VECS;
  const uint64_t step = gridDim.x;
  uint64_t tile = blockIdx.x;
  Vec16<K> buf_a[HIST_UNROLL], buf_b[HIST_UNROLL];
  auto load_tile = [&](Vec16<K>(&x)[HIST_UNROLL], uint64_t t) {
#pragma unroll
    for (int u = 0; u < HIST_UNROLL; ++u) x[u] = body[t * TILE_VECS + threadIdx.x + (uint64_t)u * HIST_BLOCK];
  };
  auto count_tile = [&](const Vec16<K>(&x)[HIST_UNROLL]) {
#pragma unroll
    for (int u = 0; u < HIST_UNROLL; ++u) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) count(x[u].v[i]);
    }
  };
  if (tile < whole_tiles) load_tile(buf_a, tile);
  while (tile + 2 * step < whole_tiles) {
    load_tile(buf_b, tile + step);
    count_tile(buf_a);
    load_tile(buf_a, tile + 2 * step);
    count_tile(buf_b);
    tile += 2 * step;
  }
  if (tile < whole_tiles) {
    if (tile + step < whole_tiles) {
      load_tile(buf_b, tile + step);
      count_tile(buf_a);
      count_tile(buf_b);
    } else {
      count_tile(buf_a);
    }
  }
  // the ragged tile after them, if any, goes to the workgroup whose turn it would be
  if (whole_tiles * TILE_VECS < vecs && whole_tiles % gridDim.x == blockIdx.x) {
#pragma unroll
    for (int u = 0; u < HIST_UNROLL; ++u) {
      const uint64_t i = whole_tiles * TILE_VECS + threadIdx.x + (uint64_t)u * HIST_BLOCK;
      if (i < vecs) {
        const Vec16<K> x = body[i];
#pragma unroll
        for (int j = 0; j < VEC; ++j) count(x.v[j]);
      }
    }
  }
  if (takes_sample) sampling.out[blockIdx.x * sampling.per_block + threadIdx.x] = codec.encode(sample);
  __syncthreads();
  // fold the copies; thread t starts at copy t so that a wave spreads over all banks
  for (int bin = threadIdx.x; bin < BINS; bin += HIST_BLOCK) {
    uint32_t c = 0;
#pragma unroll 8
    for (int j = 0; j < COPIES; ++j) c += s_hist[bin * COPIES + ((j + threadIdx.x) % COPIES)];
    if (c) atomicAdd(&hist[bin], c);
  }
}

template <typename K>
static void launch_histogram(int passes, uint32_t blocks, hipStream_t stream, const K* keys,
                             uint64_t n, const KeyCodec<K>& codec, const SortGeometry& geo,
                             uint32_t* hist, const Sampling<K>& sampling) {
  const bool whole = codec.plain && geo.begin_bit == 0 && geo.end_bit == passes * RADIX_BITS;
#define TA_HIST_CASE(NP)                                                                       \
  case NP:                                                                                     \
    if (whole)                                                                                 \
      TA_LAUNCH("sort_histogram", stream, (sort_histogram_kernel<K, NP, true>), dim3(blocks),  \
                dim3(HIST_BLOCK), keys, n, codec, geo, hist, sampling);                                 \
    else                                                                                       \
      TA_LAUNCH("sort_histogram", stream, (sort_histogram_kernel<K, NP, false>), dim3(blocks), \
                dim3(HIST_BLOCK), keys, n, codec, geo, hist, sampling);                                 \
    break;
  switch (passes) {
    TA_HIST_CASE(1) TA_HIST_CASE(2) TA_HIST_CASE(3) TA_HIST_CASE(4)
    TA_HIST_CASE(5) TA_HIST_CASE(6) TA_HIST_CASE(7) TA_HIST_CASE(8)
    default: break;
  }
#undef TA_HIST_CASE
}

// ------------------------------------------------------------------ scan of the histograms, and the plan
// One workgroup; a group of 256 threads takes every fourth digit, a thread owns a bin.  hist[p][d] becomes the
// exclusive prefix (the global offset of digit d in pass p), and ctl says what each of the launches behind this
// one does (SortCtl).
//
// The short way (one or two launches over the top digits, then radix_finish.hpp) is taken when the stretches of equal
// top digits can be expected to fit a workgroup, stretch_max keys:
//   one digit   its largest bin, known exactly
//   two digits  (8-byte keys) by the product of the two largest bins' shares, exact for independent digits, and, as digits
//               need not be independent and keys may repeat, by SAMPLES keys: see top_two_digits
// A stretch that is longer all the same costs its own sort by one workgroup (sort_tail_kernel), not the array's.
constexpr int PLAN_BLOCK = 1024;

template <typename K>
__global__ __launch_bounds__(PLAN_BLOCK) void sort_plan_kernel(uint32_t n, Sampling<K> sampling, uint32_t* __restrict__ hist,
                                                               SortGeometry geo, int top_slots, uint32_t cap,
                                                               uint32_t stretch_max,  // 0: the short way is not open
                                                               SortCtl* __restrict__ ctl) {
  constexpr int GROUPS = PLAN_BLOCK / RADIX_SIZE;
  constexpr int PER_THREAD = SAMPLES / PLAN_BLOCK;
  __shared__ uint32_t s_wave[MAX_PASSES][RADIX_SIZE / WAVE];
  __shared__ uint32_t s_most[MAX_PASSES];
  constexpr uint32_t PLAN_WORDS = sizeof(K) == 8 ? 1u << (2 * RADIX_BITS - 1) : 1u;
  static_assert(PLAN_WORDS == 1 || PLAN_WORDS * 32 == TWIN_PLACES, "a bit for every place");
  __shared__ uint32_t s_bins[PLAN_WORDS];  // 16-bit counts, two to a word; then bits
  __shared__ uint32_t s_pairs, s_peak, s_twins;
  const int group = threadIdx.x / RADIX_SIZE, d = threadIdx.x % RADIX_SIZE;
  const int wave = d / WAVE, lane = d % WAVE;
  if (threadIdx.x < MAX_PASSES) s_most[threadIdx.x] = 0;
  if (threadIdx.x == 0) s_pairs = s_peak = s_twins = 0;
  __syncthreads();
  uint32_t excl[MAX_PASSES / GROUPS];
#pragma unroll
  for (int i = 0; i < MAX_PASSES / GROUPS; ++i) {
    const int p = i * GROUPS + group;
    if (p < geo.passes) {
      const uint32_t c = hist[p * RADIX_SIZE + d];
      const uint32_t incl = wave_inclusive_scan(c, OpPlus{});
      const uint32_t most = wave_reduce(c, OpMax{});
      excl[i] = incl - c;
      if (lane == WAVE - 1) {
        s_wave[p][wave] = incl;
        atomicMax(&s_most[p], most);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MAX_PASSES / GROUPS; ++i) {
    const int p = i * GROUPS + group;
    if (p < geo.passes) {
      for (int w = 0; w < wave; ++w) excl[i] += s_wave[p][w];
      hist[p * RADIX_SIZE + d] = excl[i];
    }
  }
  int moving = 0, top = 0;  // digits whose pass moves something, and the highest of them
  for (int p = 0; p < geo.passes; ++p) {
    if (s_most[p] != n) {
      ++moving;
      top = p;
    }
  }
  uint32_t fast = 0;
  float longest = 0;  // stretch expected
  if (stretch_max != 0 && moving >= 3 && s_most[top] <= stretch_max) {
    fast = 1;
    longest = (float)s_most[top];
  }
  if constexpr (sizeof(K) == 8) {
    const float even = (float)s_most[top] / (float)n * (float)s_most[top > 0 ? top - 1 : 0];
    if (!fast && top_slots == 2 && moving >= 4 && even <= (float)stretch_max) {  // (uniform for the workgroup)
      const uint32_t samples = sampling.count;
      K sample[PER_THREAD];
#pragma unroll
      for (int i = 0; i < PER_THREAD; ++i) {
        const uint32_t j = (uint32_t)i * PLAN_BLOCK + threadIdx.x;
        sample[i] = j < samples ? sampling.out[j] : (K)0;
      }
      auto clear = [&] {
        for (uint32_t i = threadIdx.x; i < PLAN_WORDS; i += PLAN_BLOCK) s_bins[i] = 0;
        __syncthreads();
      };
      clear();
      const int bit = (top - 1) * RADIX_BITS;
      uint32_t pairs = 0, peak = 0, twins = 0;
#pragma unroll
      for (int i = 0; i < PER_THREAD; ++i) {
        if ((uint32_t)i * PLAN_BLOCK + threadIdx.x < samples) {
          const uint32_t bin = (uint32_t)(sample[i] >> bit) & 0xffffu;
          const uint32_t half = (bin & 1u) * 16;
          const uint32_t old = (__hip_atomic_fetch_add(&s_bins[bin >> 1], 1u << half, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >> half) & 0xffffu;
          pairs += old;
          peak = old + 1 > peak ? old + 1 : peak;
        }
      }
      if (even > (float)stretch_max / 4) {
        // samples whose bit, one of TWIN_PLACES by a hash of the key, another one has set before
        __syncthreads();
        clear();
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) {
          if ((uint32_t)i * PLAN_BLOCK + threadIdx.x < samples) {
            const uint64_t h = ((uint64_t)sample[i] ^ (uint64_t)sample[i] >> 29) * 0x9e3779b97f4a7c15ull;
            const uint32_t place = (uint32_t)(h >> 40) % TWIN_PLACES, bit_of = 1u << place % 32;
            const uint32_t old = __hip_atomic_fetch_or(&s_bins[place / 32], bit_of, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            twins += (old & bit_of) != 0 ? 1u : 0u;
          }
        }
      }
      pairs = wave_reduce(pairs, OpPlus{});
      peak = wave_reduce(peak, OpMax{});
      twins = wave_reduce(twins, OpPlus{});
      if (lane == 0) {
        atomicAdd(&s_pairs, pairs);
        atomicMax(&s_peak, peak);
        atomicAdd(&s_twins, twins);
      }
      __syncthreads();
      longest = top_two_digits((float)n, (float)samples, even, (float)s_pairs, (float)s_twins, (float)s_peak, (float)stretch_max);
      if (longest > 0) fast = 2;
    }
  }
  if (threadIdx.x != 0) return;
  uint32_t parity = 0;
  int slot = 0;
  bool first = true;
  auto put = [&](uint32_t action, int p, bool last) {
    ctl->slot[slot++] = SortCtl::pack(action, (uint32_t)p, parity, first, last);
    if (action != SortCtl::SKIP) {
      parity ^= 1u;
      first = false;
    }
  };
  ctl->fast = fast;
  ctl->gave_up = 0;
  ctl->long_windows = 0;
  if (fast) {
    for (int p = top + 1 - (int)fast; p <= top; ++p) put(s_most[p] == n ? SortCtl::SKIP : SortCtl::RUN, p, false);
    ctl->fast_src_alt = parity;
    parity = 0;  // the last step writes the caller's array
    // a window and the longest stretch that may cross its end fill a workgroup: leave room beyond the stretch expected
    const float room = fast == 1 ? longest : longest + __builtin_sqrtf(longest) + 0.02f * longest;
    uint32_t reach = (uint32_t)room + 1;
    reach = reach < cap / 8 ? cap / 8 : reach > stretch_max ? stretch_max : reach;
    // ... and take smaller windows than that where they would leave CUs without work
    const uint32_t even = n / (4 * NUM_CU) > cap - stretch_max ? n / (4 * NUM_CU) : cap - stretch_max;
    ctl->window = even < cap - reach ? even : cap - reach;
    ctl->prefix_bit = (uint32_t)((top + 1 - (int)fast) * RADIX_BITS);
  } else {
    for (int p = 0; p < geo.passes; ++p) put(s_most[p] == n ? SortCtl::SKIP : SortCtl::RUN, p, p == top);
  }
  while (slot < MAX_PASSES) put(SortCtl::SKIP, 0, false);
  ctl->final_in_alt = parity;
}

// ------------------------------------------------------------------ onesweep pass
template <typename K, typename V, bool HAS_VALUES, int BLOCK, int ITEMS>
struct PassShape {
  static constexpr int WAVES = BLOCK / WAVE;
  static constexpr int TILE = BLOCK * ITEMS;
  static constexpr size_t EXCH_ITEM = (HAS_VALUES && sizeof(V) > sizeof(K)) ? sizeof(V) : sizeof(K);
  static constexpr size_t EXCH_BYTES = (size_t)TILE * EXCH_ITEM;
  static constexpr size_t CNT_BYTES = (size_t)WAVES * RADIX_SIZE * sizeof(uint32_t);
  static constexpr size_t UNION_BYTES = EXCH_BYTES > CNT_BYTES ? EXCH_BYTES : CNT_BYTES;
};

// Tile descriptors fetched together per look-back round by each digit thread.
constexpr int LOOKBACK_WINDOW = 4;

// OFF32: every key and value of the call lies within 4 GiB of its array's start, so that
// global addresses are a scalar base plus a 32-bit byte offset (one vector instruction per
// access less than with 64-bit address arithmetic).
template <typename K, typename V, bool HAS_VALUES, int BLOCK, int ITEMS, typename D, bool OFF32>
__global__ __launch_bounds__(BLOCK) void onesweep_pass_kernel(
    K* __restrict__ keys_a, K* __restrict__ keys_b, V* __restrict__ vals_a, V* __restrict__ vals_b,
    uint32_t n, int slot, SortGeometry geo, KeyCodec<K> codec,
    const uint32_t* __restrict__ hist,      // [passes][RADIX_SIZE] global digit offsets
    D* __restrict__ status,                 // [tiles][RADIX_SIZE]
    uint32_t* __restrict__ ticket,          // [TICKET_CLASSES] counters of this pass, TICKET_STRIDE words apart
    const SortCtl* __restrict__ ctl,
    SortCtl* __restrict__ ctl_out) {        // the same block: fields that only a pass that gives up writes
  using Shape = PassShape<K, V, HAS_VALUES, BLOCK, ITEMS>;
  using Desc = Descriptor<D>;
  constexpr int WAVES = Shape::WAVES;
  constexpr int TILE = Shape::TILE;
  static_assert(BLOCK >= RADIX_SIZE, "one thread per digit is required");

  const uint32_t todo = ctl->slot[slot];
  if (!SortCtl::runs(todo)) return;
  const int pass = (int)SortCtl::digit(todo);
  const uint32_t* __restrict__ bin_base = hist + pass * RADIX_SIZE;
  const bool from_alt = SortCtl::src_alt(todo);
  const K* __restrict__ keys_in = from_alt ? keys_b : keys_a;
  K* __restrict__ keys_out = from_alt ? keys_a : keys_b;
  const V* __restrict__ vals_in = from_alt ? vals_b : vals_a;
  V* __restrict__ vals_out = from_alt ? vals_a : vals_b;

  __shared__ __attribute__((aligned(16))) unsigned char s_union[Shape::UNION_BYTES];
  __shared__ uint32_t s_scatter_base[RADIX_SIZE];  // global offset - local offset, per digit
  __shared__ uint32_t s_digit_wave[RADIX_SIZE / WAVE];
  __shared__ uint32_t s_tile;
  uint32_t* s_cnt = reinterpret_cast<uint32_t*>(s_union);  // [WAVES][RADIX_SIZE]
  K* s_keys = reinterpret_cast<K*>(s_union);
  V* s_vals = reinterpret_cast<V*>(s_union);

  if (threadIdx.x == 0) {
    const uint32_t k = blockIdx.x % TICKET_CLASSES;
    s_tile = class_tile(k, atomicAdd(ticket + k * TICKET_STRIDE, 1u), gridDim.x);
  }
  for (int i = threadIdx.x; i < WAVES * RADIX_SIZE; i += BLOCK) s_cnt[i] = 0;
  __syncthreads();
  const uint32_t tile = __builtin_amdgcn_readfirstlane(s_tile);
#define TA_PASS_LOAD(item) (item)
#define TA_PASS_STORE(item, value) (item) = (value)
#define TA_PASS_GIVES_UP() strike_out(slot)
  auto strike_out = [&](int at) {
    ctl_out->strike_out(at, [](uint32_t* p, uint32_t x) { __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); });
  };
#include "radix_pass_tile.inc"
#undef TA_PASS_LOAD
#undef TA_PASS_STORE
#undef TA_PASS_GIVES_UP
}

// ------------------------------------------------------------------ several passes in one launch
// The passes of the slots [first_slot, slots) and, if `copies`, the copy back: what stands behind the short way, and
// mostly finds nothing to do.  A workgroup takes tiles of a pass in rising order until there are none left and
// then waits until the others have written theirs.  Whoever waits, waits only for workgroups that run and wait for
// nobody but earlier tiles of the same pass, so this works with any number of workgroups resident.
// What one pass writes and another XCD's workgroup reads in the next goes past the caches that are not coherent
// (agent scope): a write-back of the L2 per tile took 35 us a pass.  Short runs leave as partial lines then, and every
// pass ends with a trip to memory for its count and one for the next pass's wait, so longer arrays keep a launch per pass.
// Copy and sort, us, a launch per pass (and the bounds of the short way in a launch) against this: short way taken, 65536
// uint32 40.0 -> 25.9, 2^20 47.5 -> 36.6, 65536 (uint32, uint32) 48.0 -> 30.3, 30011 uint64 48.9 -> 36.8, with uint64 values
// 49.4 -> 38.5; not taken (90 % one key), 65536 uint32 46.1 -> 43.6, 2^20 65.7 -> 62.3, 1.5e6 72 -> 79, 7.9e5 (uint32, uint32)
// 65.7 -> 63.2, 5.2e5 (uint32, uint64) 62.4 -> 62.1, 30011 uint64 70.5 -> 70.4, with uint64 values 78.7 -> 78.9, 10007 of
// them 74.5 -> 76 (waited for 94 -> 89).  The line is drawn where a sort that declines would pay: 65536 uint64 72.6 -> 74.5,
// with uint64 values 80.8 -> 84.8, 98304 84.1 -> 87.7, permuted 7.9e5 (uint32, uint64) 66.4 -> 68.0.
// (One counter for the tiles written instead of seven: 2^20 uint32 66.9, permuted 61.2 against 55.9; flag and slot asked for
// behind every pass, and the loads of the copy back one after the other, cost another us each.)
// tickets[slot]: word 0 counts the tiles taken, those at counter_word() the tiles written.
template <typename K, typename V, bool HAS_VALUES>
constexpr uint64_t REST_MAX = sizeof(K) == 8 ? 1u << 15 : !HAS_VALUES ? 1u << 20 : sizeof(V) == 8 ? 1u << 19 : 3u << 18;

template <typename K, typename V, bool HAS_VALUES, int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK) void onesweep_rest_kernel(
    K* keys_a, K* keys_b, V* vals_a, V* vals_b,
    uint32_t n, int first_slot, int slots, uint32_t tiles, SortGeometry geo, KeyCodec<K> codec, const uint32_t* __restrict__ hist,
    uint32_t* __restrict__ statuses, uint64_t slot_words,
    uint32_t* __restrict__ tickets, const SortCtl* __restrict__ ctl, SortCtl* __restrict__ ctl_out, bool copies) {
  if (ctl->finishes()) return;
  using Shape = PassShape<K, V, HAS_VALUES, BLOCK, ITEMS>;
  using D = uint32_t;
  using Desc = Descriptor<D>;
  constexpr bool OFF32 = true;
  constexpr int WAVES = Shape::WAVES;
  constexpr int TILE = Shape::TILE;
  __shared__ __attribute__((aligned(16))) unsigned char s_union[Shape::UNION_BYTES];
  __shared__ uint32_t s_scatter_base[RADIX_SIZE];
  __shared__ uint32_t s_digit_wave[RADIX_SIZE / WAVE];
  __shared__ uint32_t s_tile, s_go, s_gave_up;
  uint32_t* s_cnt = reinterpret_cast<uint32_t*>(s_union);
  K* s_keys = reinterpret_cast<K*>(s_union);
  V* s_vals = reinterpret_cast<V*>(s_union);
  // What there is to do is read from ctl->slot, which nothing in this launch writes; whether a pass is complete, and
  // whether one of its tiles gave up, from its counters alone.  A pass begins, and the copy back does, only behind the
  // complete pass before, so nothing works on keys that a pass left out of place.
  uint32_t* written = nullptr;  // the counters of the pass before
  // (the launches behind this one; no slot is struck out)
  auto strike_out = [&] {
    ctl_out->strike_out(MAX_PASSES - 1, [](uint32_t* p, uint32_t x) { __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); });
  };
  // The first wave, until the pass before is complete: true, or false if a tile of it gave up or this wait did.
  auto is_complete = [&]() -> bool {
    const uint32_t lane = threadIdx.x;
    const uint32_t due = lane < COUNTERS ? due_on(lane, tiles) : 0;
    for (uint32_t spins = 0; written != nullptr;) {
      uint32_t have = due;
      if (lane < COUNTERS) have = __hip_atomic_load(written + counter_word(lane), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (__builtin_amdgcn_ballot_w64(have >= COUNT_GAVE_UP) != 0) return false;
      if (__builtin_amdgcn_ballot_w64(have != due) == 0) break;
      __builtin_amdgcn_s_sleep(2);
      ++spins;
      if (spins % 1024u == 0 &&
          __builtin_amdgcn_readfirstlane(__hip_atomic_load(&ctl_out->gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0)
        return false;
      if (spins >= LOOKBACK_SPIN_LIMIT) {
        strike_out();
        return false;
      }
    }
    return true;
  };
  auto clear_counters = [&] {
    for (int i = threadIdx.x; i < WAVES * RADIX_SIZE; i += BLOCK) s_cnt[i] = 0;
  };
  if (threadIdx.x == 0) s_gave_up = 0;
  bool odd = false;  // an odd number of passes leaves the result in the alternate buffer
  for (int slot = 0; slot < slots; ++slot) odd = odd != SortCtl::runs(ctl->slot[slot]);
  for (int slot = first_slot; slot < slots; ++slot) {
    const uint32_t todo = ctl->slot[slot];
    if (!SortCtl::runs(todo)) continue;
    uint32_t* ticket = tickets + (size_t)slot * TICKET_CLASSES * TICKET_STRIDE;
    if (threadIdx.x < WAVE) {
      uint32_t first = 0;
      if (threadIdx.x == 0) first = atomicAdd(ticket, 1u);  // (on its way while the pass before ends)
      const bool go = is_complete();
      if (threadIdx.x == 0) {
        s_tile = first;
        s_go = go ? 1u : 0u;
      }
    }
    clear_counters();
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(s_go) == 0) return;
    written = ticket;
    const int pass = (int)SortCtl::digit(todo);
    const uint32_t* __restrict__ bin_base = hist + pass * RADIX_SIZE;
    const bool from_alt = SortCtl::src_alt(todo);
    // (not __restrict__: the next pass reads what this one writes)
    const K* keys_in = from_alt ? keys_b : keys_a;
    K* keys_out = from_alt ? keys_a : keys_b;
    const V* vals_in = from_alt ? vals_b : vals_a;
    V* vals_out = from_alt ? vals_a : vals_b;
    D* status = statuses + (size_t)slot * slot_words;
    // what the last pass writes stays for the next launch, unless it is copied back here
    const bool nobody_reads = SortCtl::decodes(todo) && !(copies && odd);
    for (;;) {
      const uint32_t tile = __builtin_amdgcn_readfirstlane(s_tile);
      if (tile >= tiles) break;
#define TA_PASS_LOAD(item) __hip_atomic_load(&(item), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
#define TA_PASS_STORE(item, value) (nobody_reads ? (void)((item) = (value)) : __hip_atomic_store(&(item), value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
#define TA_PASS_GIVES_UP() (s_gave_up = 1, strike_out())
#include "radix_pass_tile.inc"
#undef TA_PASS_LOAD
#undef TA_PASS_STORE
#undef TA_PASS_GIVES_UP
      // counted in when all of the workgroup's stores have been acknowledged
      uint32_t next = 0;
      if (threadIdx.x == 0) next = atomicAdd(ticket, 1u);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (threadIdx.x == 0) {
        __hip_atomic_fetch_add(ticket + counter_word(counter_of(tile)), s_gave_up != 0 ? COUNT_GAVE_UP : 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_tile = next;
      }
      clear_counters();
      __syncthreads();
    }
    __syncthreads();  // everybody has seen that there are no more tiles
  }
  if (!copies || !odd) return;
  if (threadIdx.x < WAVE) {
    // (no pass of this launch: one of an earlier launch may have given up)
    const bool go = written != nullptr ? is_complete() : ctl->gave_up == 0;
    if (threadIdx.x == 0) s_go = go ? 1u : 0u;
  }
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(s_go) != 0) {
    // (all loads in flight together, the last element in the place of those behind it)
    const uint32_t first = blockIdx.x * BLOCK + threadIdx.x, stride = gridDim.x * BLOCK;
    K k[ITEMS];
    V v[HAS_VALUES ? ITEMS : 1];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const uint32_t i = first + r * stride < n ? first + r * stride : n - 1;
      k[r] = __hip_atomic_load(keys_b + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if constexpr (HAS_VALUES) v[r] = __hip_atomic_load(vals_b + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const uint32_t i = first + r * stride;
      if (i >= n) break;
      keys_a[i] = k[r];
      if constexpr (HAS_VALUES) vals_a[i] = v[r];
    }
  }
}

// ------------------------------------------------------------------ copy-back
template <typename K, typename V, bool HAS_VALUES>
__global__ __launch_bounds__(256) void sort_copy_back_kernel(K* __restrict__ keys,
                                                             const K* __restrict__ keys_alt,
                                                             V* __restrict__ vals,
                                                             const V* __restrict__ vals_alt,
                                                             uint64_t n,
                                                             const SortCtl* __restrict__ ctl) {
  if (!ctl->copies_back()) return;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    keys[i] = keys_alt[i];
    if constexpr (HAS_VALUES) vals[i] = vals_alt[i];
  }
}

// ------------------------------------------------------------------ host side
template <typename K, typename V, bool HAS_VALUES>
struct SortPlan {
  // Large tiles (14K-18K keys of 4 bytes) keep the number of tiles in flight, and with it
  // the length of every look-back, small; two blocks of 1024 threads fill a CU (64 VGPRs,
  // 80 KB of LDS each).  8-byte keys or values halve the tile to fit LDS.  4-byte keys with values: 14 keys per lane are
  // what 64 registers hold.  With 16, 74 registers and one workgroup per CU, or 64 and 36 bytes of spills: a pass over
  // 8e6 pairs 36.9 us (with spills) -> 34.8, 1.6e7 72.9 -> 57.5, 2.4e7 114 -> 94, 6.4e7 249 -> 235, 1.34e8 486 -> 463; with 12
  // 35.2, 59.6, 94, 235, 474.
  static constexpr int BLOCK = 1024;
  static constexpr int ITEMS = (sizeof(K) == 8 || (HAS_VALUES && sizeof(V) == 8)) ? 8
                               : sizeof(K) == 4                                  ? (HAS_VALUES ? 14 : 18)
                                                                                 : 16;
  static constexpr int TILE = BLOCK * ITEMS;
  // Arrays of 4 GiB and more need 64-bit addresses, with which one workgroup of either size fills a CU's registers.
  static constexpr int FAR_ITEMS = ITEMS == 14 ? 16 : ITEMS;
  // Where tiles of this size are fewer than the CUs: a third or half of it.  The time is that of one or two tiles
  // then, and shorter with smaller ones.  Sort of 1e6 and 2.6e6 random keys, large tiles against small ones: float32 76 -> 65,
  // 97 -> 93 us; with uint32 values (tiles of 16384) 86 -> 75, 102 -> 94; uint8 29.4 -> 27.5, 34.3 -> 34.3; uint16 42.6 -> 38.8,
  // 50.6 -> 50.5; (uint16, uint64) 47 -> 45, and 51.5 -> 51.7 at 1.6e6; float64 137 -> 130 at 1e6.  Float32 at 4e6: 106 -> 110.
  static constexpr int FINE_ITEMS = ITEMS == 8 ? 4 : 6;
  static constexpr uint64_t FINE_MAX = (uint64_t)TILE * NUM_CU * 5 / 8;
  static constexpr int FINE_TILE = BLOCK * FINE_ITEMS;
  // 4-byte keys, as long as tiles of 10 keys per lane all run at once, two to a CU: copy and sort of 3.2e6, 4e6 and 5.2e6
  // keys 101 -> 96, 104 -> 103, 115 -> 106 us, with uint32 values 108 -> 108, 114 -> 115, 154 -> 126 (14 keys per lane: 134),
  // and in a second round the others are better: 6e6 keys 119.6 against 121, pairs 136 against 148.  8-byte keys with 6 per
  // lane: 4e6 118 against 124.
  static constexpr bool HAS_MID = sizeof(K) == 4 && ITEMS != 8;
  static constexpr int MID_ITEMS = HAS_MID ? 10 : ITEMS;
  static constexpr int MID_TILE = BLOCK * MID_ITEMS;
  static constexpr uint64_t MID_MAX = HAS_MID ? (uint64_t)MID_TILE * NUM_CU * 2 : 0;
};

template <typename K, typename V, bool HAS_VALUES>
static int sort_impl(void* temp, size_t* temp_bytes, void* keys, void* values, uint64_t n, int dtype,
                     int descending, int begin_bit, int end_bit, hipStream_t stream) {
  using Plan = SortPlan<K, V, HAS_VALUES>;
  const int key_bits = (int)sizeof(K) * 8;
  if (begin_bit < 0 || end_bit > key_bits || begin_bit > end_bit) return (int)hipErrorInvalidValue;
  if (n > SORT_MAX_N) return (int)hipErrorInvalidValue;
  SortGeometry geo;
  geo.begin_bit = begin_bit;
  geo.end_bit = end_bit;
  geo.passes = (end_bit - begin_bit + RADIX_BITS - 1) / RADIX_BITS;
  const bool fine = n <= Plan::FINE_MAX;
  const bool mid = !fine && n <= Plan::MID_MAX;
  const bool wide = n > SORT_MAX_N_NARROW;  // prefixes need more than 30 bits: 64-bit descriptors
  // every key and value within 4 GiB of its array's start: 32-bit byte offsets
  const bool off32 = !wide && n * (uint64_t)((HAS_VALUES && sizeof(V) > sizeof(K)) ? sizeof(V) : sizeof(K)) <= (1ull << 32);
  const uint64_t tile = fine ? Plan::FINE_TILE : mid ? Plan::MID_TILE : off32 ? Plan::TILE : Plan::BLOCK * Plan::FAR_ITEMS;
  const uint64_t tiles = (n + tile - 1) / tile;

  TempLayout lay;
  const size_t off_ctl = lay.add(sizeof(SortCtl));
  // contiguous zero-initialised region: tickets, histograms, tile descriptors
  // The short way, over whole keys only.  Against all digits' passes, sort of random keys:
  //   8-byte keys      1e4 keys 84 -> 32 us, 1e6 135 -> 79, 8e6 309 -> 166, 1.34e8 4130 -> 1880; with 4-byte values
  //                    92 -> 36, 157 -> 85, 363 -> 180, 5790 -> 2430 us; where keys repeat 10 to 30 times 0.66-0.85 of the
  //                    time, where the plan declines 1.00-1.05 (5 to 10 us up to 8e6 keys, 1 % at 1.34e8; 1.04-1.09 where
  //                    one digit varies): two launches that do nothing, one of them of a workgroup per window
  //   4-byte integers  by one digit (as long as its bins can fit at all) 1e4 keys 68 -> 22 us, 1e6 75 -> 35; with
  //                    values 70 -> 26, 85 -> 50.  Never by two digits: that saves two passes and costs the last step,
  //                    0.95-1.06 times as fast for random keys of 2^25 and more, and where keys repeat (ten times or a
  //                    thousand) the stretches outgrow a workgroup: 2^28 keys 2170 -> 3220 us when all passes follow.
  //   floats           share few exponents: 4-byte ones outgrow a workgroup at some 20000 keys, 8-byte ones (four
  //                    bits of mantissa in two digits) at a few 100000.
  // It ends where random keys' stretches of two digits come near STRETCH_MAX (1.5e8 keys); a third digit would carry on.
  using Finish = FinishShape<K, V, HAS_VALUES>;
  const bool is_float = dtype == THRUST_AMD_F32 || dtype == THRUST_AMD_F64;
  const bool two_digits = sizeof(K) == 8 && (!is_float || n <= (1u << 19));
  const bool one_digit = n <= (is_float ? 8 : 256) * (uint64_t)Finish::STRETCH_MAX;
  const bool hybrid = sizeof(K) >= 4 && begin_bit == 0 && end_bit == key_bits && n > SMALL_SORT_MAX &&
                      n / 65536 <= Finish::STRETCH_MAX * 9 / 10 && (one_digit || two_digits);
  const int top_slots = !hybrid ? 0 : two_digits ? TOP_SLOTS : 1;
  const int slots = geo.passes;
  const uint64_t max_windows = (n + Finish::WINDOW_MIN - 1) / Finish::WINDOW_MIN;
  // descriptor words of a slot; the first kernel clears those of `cleared_slots` slots, the finish kernel the others
  const size_t slot_words = (size_t)tiles * RADIX_SIZE * (wide ? 2 : 1);
  const int cleared_slots = hybrid ? top_slots : slots;
  const size_t zero_words = (size_t)TICKET_WORDS + (size_t)MAX_PASSES * RADIX_SIZE + (size_t)cleared_slots * slot_words;
  const size_t off_zero = lay.add((zero_words + (size_t)(slots - cleared_slots) * slot_words) * sizeof(uint32_t));
  const size_t off_bounds = lay.add(hybrid ? (max_windows + 1) * sizeof(uint32_t) : 0);
  const size_t off_long = lay.add(hybrid ? (n / Finish::CAP + 1) * sizeof(uint32_t) : 0);
  const size_t off_samples = lay.add(top_slots == 2 ? SAMPLES * sizeof(K) : 0);
  const size_t off_keys = lay.add((size_t)n * sizeof(K));
  const size_t off_vals = lay.add(HAS_VALUES ? (size_t)n * sizeof(V) : 0);
  if (temp == nullptr) {
    *temp_bytes = lay.total;
    return 0;
  }
  if (*temp_bytes < lay.total) return (int)hipErrorInvalidValue;
  if (n <= 1 || geo.passes == 0) return 0;
  if (!keys || (HAS_VALUES && !values)) return (int)hipErrorInvalidValue;
  if (n <= SMALL_SORT_MAX)
    return small_sort(keys, values, (uint32_t)n, dtype, HAS_VALUES ? sizeof(V) : 0, descending, begin_bit, end_bit, stream);

  char* base = static_cast<char*>(temp);
  SortCtl* ctl = reinterpret_cast<SortCtl*>(base + off_ctl);
  uint32_t* zero = reinterpret_cast<uint32_t*>(base + off_zero);
  uint32_t* tickets = zero;
  uint32_t* hist = zero + TICKET_WORDS;
  uint32_t* status = hist + MAX_PASSES * RADIX_SIZE;
  K* keys_a = static_cast<K*>(keys);
  K* keys_b = reinterpret_cast<K*>(base + off_keys);
  V* vals_a = static_cast<V*>(values);
  V* vals_b = reinterpret_cast<V*>(base + off_vals);
  const KeyCodec<K> codec = make_codec<K>(dtype, descending);

  {
    uint64_t blocks = (zero_words + 255) / 256;
    if (blocks > (uint64_t)NUM_CU * 8) blocks = (uint64_t)NUM_CU * 8;
    TA_LAUNCH("sort_init", stream, sort_init_kernel, dim3((uint32_t)blocks), dim3(256), zero, (uint64_t)zero_words);
    TA_CHECK_LAUNCH();
  }
  Sampling<K> sampling{};
  {
    constexpr uint64_t HT = (uint64_t)HIST_BLOCK * HIST_UNROLL * Vec16<K>::N;
    uint64_t blocks = (n + HT - 1) / HT;
    if (blocks > (uint64_t)NUM_CU) blocks = NUM_CU;
    if (top_slots == 2) {
      sampling.out = reinterpret_cast<K*>(base + off_samples);
      const uint64_t wanted = n / 64 < SAMPLES ? n / 64 : SAMPLES;
      const uint64_t each = wanted / blocks < (uint64_t)HIST_BLOCK ? wanted / blocks : (uint64_t)HIST_BLOCK;
      sampling.per_block = (uint32_t)(each > 0 ? each : 1);
      sampling.count = sampling.per_block * (uint32_t)blocks;
      sampling.step = (uint32_t)(n / sampling.count);
    }
    launch_histogram<K>(geo.passes, (uint32_t)blocks, stream, (const K*)keys_a, n, codec, geo, hist, sampling);
    TA_CHECK_LAUNCH();
  }
  TA_LAUNCH("sort_plan", stream, sort_plan_kernel<K>, dim3(1), dim3(PLAN_BLOCK), (uint32_t)n, sampling, hist, geo, top_slots, (uint32_t)Finish::CAP, hybrid ? Finish::STRETCH_MAX : 0u, ctl);
  TA_CHECK_LAUNCH();
  uint32_t* bounds = reinterpret_cast<uint32_t*>(base + off_bounds);
  uint32_t* long_list = reinterpret_cast<uint32_t*>(base + off_long);
  const bool tail = top_slots == 2;  // (8-byte keys)
  const int single_launches = hybrid && n <= REST_MAX<K, V, HAS_VALUES> ? top_slots : slots;  // passes with a launch of their own
  for (int slot = 0; slot < slots; ++slot) {
    if constexpr (sizeof(K) >= 4) {
      if (hybrid && slot == top_slots) {
        // (stretches of one digit begin where the histogram says)
        if constexpr (sizeof(K) == 8) {
          TA_LAUNCH("sort_bounds", stream, sort_bounds_kernel<K>, dim3((uint32_t)(max_windows / 256 + 1)), dim3(256), (const K*)keys_a, (const K*)keys_b, (uint32_t)n, (uint32_t)Finish::CAP, bounds, (const SortCtl*)ctl);
          TA_CHECK_LAUNCH();
        }
        TA_LAUNCH("sort_finish", stream, (sort_finish_kernel<K, V, HAS_VALUES>), dim3((uint32_t)max_windows), dim3(Finish::BLOCK), keys_a, (const K*)keys_b, vals_a, (const V*)vals_b, (uint32_t)n, codec, (const uint32_t*)bounds, (const uint32_t*)hist, (const SortCtl*)ctl, &ctl->long_windows, long_list, status + (size_t)top_slots * slot_words, (uint64_t)((slots - top_slots) * slot_words));
        TA_CHECK_LAUNCH();
      }
    }
    if constexpr (sizeof(K) >= 4) {
      if (slot >= single_launches) {
        static_assert(REST_MAX<K, V, HAS_VALUES> <= Plan::FINE_MAX, "tiles as in the passes before, 32-bit offsets");
        TA_LAUNCH("onesweep_rest", stream, (onesweep_rest_kernel<K, V, HAS_VALUES, Plan::BLOCK, Plan::FINE_ITEMS>), dim3((uint32_t)tiles), dim3(Plan::BLOCK), keys_a, keys_b, vals_a, vals_b, (uint32_t)n, slot, slots, (uint32_t)tiles, geo, codec, (const uint32_t*)hist, status, (uint64_t)slot_words, tickets, (const SortCtl*)ctl, ctl, !tail);
        TA_CHECK_LAUNCH();
        if (!tail) return 0;
        break;
      }
    }
    const char* label = hybrid && slot >= top_slots ? "onesweep_rest" : "onesweep_pass";
    uint32_t* slot_status = status + (size_t)slot * slot_words;
    uint32_t* slot_tickets = tickets + (size_t)slot * TICKET_CLASSES * TICKET_STRIDE;
    auto launch = [&](auto kernel, auto* descriptors) {
      TA_LAUNCH(label, stream, kernel, dim3((uint32_t)tiles), dim3(Plan::BLOCK), keys_a, keys_b, vals_a, vals_b, (uint32_t)n, slot, geo, codec, (const uint32_t*)hist, descriptors, slot_tickets, (const SortCtl*)ctl, ctl);
    };
    if (fine) launch(onesweep_pass_kernel<K, V, HAS_VALUES, Plan::BLOCK, Plan::FINE_ITEMS, uint32_t, true>, slot_status);
    else if (mid) launch(onesweep_pass_kernel<K, V, HAS_VALUES, Plan::BLOCK, Plan::MID_ITEMS, uint32_t, true>, slot_status);
    else if (off32) launch(onesweep_pass_kernel<K, V, HAS_VALUES, Plan::BLOCK, Plan::ITEMS, uint32_t, true>, slot_status);
    else if (wide) launch(onesweep_pass_kernel<K, V, HAS_VALUES, Plan::BLOCK, Plan::FAR_ITEMS, uint64_t, false>, reinterpret_cast<uint64_t*>(slot_status));
    else launch(onesweep_pass_kernel<K, V, HAS_VALUES, Plan::BLOCK, Plan::FAR_ITEMS, uint32_t, false>, slot_status);
    TA_CHECK_LAUNCH();
  }
  if constexpr (sizeof(K) == 8) {
    if (top_slots == 2) {
      uint64_t blocks = (n + TAIL_BLOCK - 1) / TAIL_BLOCK;
      if (blocks > (uint64_t)NUM_CU * 2) blocks = (uint64_t)NUM_CU * 2;
      TA_LAUNCH("sort_tail", stream, (sort_tail_kernel<K, V, HAS_VALUES>), dim3((uint32_t)blocks), dim3(TAIL_BLOCK), keys_a, keys_b, vals_a, vals_b, (uint32_t)n, codec, (const uint32_t*)bounds, (const uint32_t*)long_list, (const SortCtl*)ctl);
      TA_CHECK_LAUNCH();
      return 0;
    }
  }
  {
    uint64_t blocks = (n + 255) / 256;
    if (blocks > (uint64_t)NUM_CU * 8) blocks = (uint64_t)NUM_CU * 8;
    TA_LAUNCH("sort_copy_back", stream, (sort_copy_back_kernel<K, V, HAS_VALUES>), dim3((uint32_t)blocks), dim3(256), keys_a, (const K*)keys_b, vals_a, (const V*)vals_b, n, (const SortCtl*)ctl);
    TA_CHECK_LAUNCH();
  }
  return 0;
}

}  // namespace ta

TA_EXPORT int thrust_amd_sort_keys(void* temp, size_t* temp_bytes, void* keys, uint64_t n,
                                   int key_dtype, int descending, int begin_bit, int end_bit,
                                   void* stream) {
  using namespace ta;
  if (!temp_bytes || !valid_dtype(key_dtype)) return (int)hipErrorInvalidValue;
  return with_item_bytes(thrust_amd_dtype_size(key_dtype), [&](auto kt) {
    using K = typename decltype(kt)::type;
    return sort_impl<K, uint32_t, false>(temp, temp_bytes, keys, nullptr, n, key_dtype, descending,
                                         begin_bit, end_bit, (hipStream_t)stream);
  });
}

TA_EXPORT int thrust_amd_sort_pairs(void* temp, size_t* temp_bytes, void* keys, void* values,
                                    uint64_t n, int key_dtype, size_t value_bytes, int descending,
                                    int begin_bit, int end_bit, void* stream) {
  using namespace ta;
  if (!temp_bytes || !valid_dtype(key_dtype) || !valid_item_bytes(value_bytes))
    return (int)hipErrorInvalidValue;
  return with_item_bytes(thrust_amd_dtype_size(key_dtype), [&](auto kt) {
    using K = typename decltype(kt)::type;
    return with_item_bytes(value_bytes, [&](auto vt) {
      using V = typename decltype(vt)::type;
      return sort_impl<K, V, true>(temp, temp_bytes, keys, values, n, key_dtype, descending,
                                   begin_bit, end_bit, (hipStream_t)stream);
    });
  });
}
