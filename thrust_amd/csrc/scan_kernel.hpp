// Single-pass prefix scan with decoupled look-back: the kernel and its launcher, shared by
// the plain scans (scan.hip) and the scans of a transformed input (transform_scan.hip).
// `Pre` is applied to every element as it is loaded; everything after that is the same.
//
// Tile order is a dynamic ticket (one atomic per workgroup), so a tile only ever waits
// for tiles that have already started: correct under any workgroup scheduling order.
// Data layout inside a tile ("wave-striped vectors"): wave w owns a contiguous span of
// 64*CHUNKS 16-byte vectors; its lane l holds vectors l, 64+l, 128+l, ... of that span.
// Every global load/store instruction of a wave therefore covers 1 KiB of consecutive
// addresses, and no LDS transpose is needed: the scan runs as CHUNKS wave scans (DPP)
// chained by the wave total, then one cross-wave step through LDS.
//
// HBM traffic: n*sizeof(T) read + n*sizeof(T) written; tile descriptors add
// 8*W bytes per tile (W = 32-bit words of T).  Short arrays take one or two launches without
// look-back instead (below); what they read twice comes from the caches the second time.
#pragma once
#include "common.hpp"
#include "dispatch.hpp"
#include "launch.hpp"

namespace ta {

// Tile shapes (threads x 16-byte vectors per lane) of the single-pass kernel.  The per-tile cost of
// the ticket (a same-address atomic retires every ~12 ns on MI355X) and of the look-back makes
// large tiles win; the small ones are left to short arrays in storage that is kept clean.
struct ScanShapeLarge { static constexpr int BLOCK = 1024, CHUNKS = 12; };
struct ScanShapeSmall { static constexpr int BLOCK = 256, CHUNKS = 4; };
constexpr uint64_t SCAN_LARGE_MIN_BYTES = (uint64_t)32 << 20;

// Arrays of up to SCAN_TWO_MAX_BYTES are scanned by two launches that wait for nothing (scan_partials_kernel,
// scan_apply_kernel): their second read of the input meets the caches, and no tile queues at the ticket.
// Whole call back to back in us, single pass with the shape it takes at that size / two launches: 4 MiB of int32 11.2 / 7.2,
// 17 MiB 28.6 / 10.9, 31 MiB 45 / 17, 44 MiB 32.0 / 24.0, 60 MiB 45 / 31.7; int64 4 MiB 11.7 / 7.1, 31 MiB 47 / 17.4;
// int8 60 MiB 325 / 50; int16 60 MiB 70 / 37.  Tiles of 64 KiB instead of 16: 64 MB 32.5, the others alike.
// The single pass is the faster one where its large tiles all run at once, if the last, ragged one, which is loaded
// element by element, is short: int32 34, 37, 40, 43 and 46 MiB (that tile a third full) 19.1 / 18.7, 19.7 / 21.5, 20.1 / 23.0,
// 20.6 / 24.6, 21.6 / 25.9, but two thirds full 38 MiB 24.7 / 22.0, 44 MiB 25.3 / 24.9, 47 MiB 26.2 / 26.5; a third full 49 MiB
// 30.2 / 27.3, 58 MiB 30.7 / 30.6, 64 MiB 32.9 / 33.6.  With 8-byte elements the ragged tile matters less: 33 MiB 19.5 / 18.4,
// 34 MiB 18.4 / 19.0, 35 MiB 18.8 / 20.2, 47 MiB 22.1 / 26.7, 50 MiB 29.8 / 28.1, 61 MiB 31.5 / 32.6.
// Only where the input is memory of this device: elsewhere both reads go over the link (4 MiB of pinned or managed host
// memory 91 us by the single pass, 192 by two launches, 64 MiB 1260 and 2500), and the single pass does it.
struct ScanShapeTwo { static constexpr int BLOCK = 256, CHUNKS = 4; };
constexpr uint64_t SCAN_TWO_MAX_BYTES = (uint64_t)64 << 20;
constexpr uint64_t SCAN_TWO_MAX_BYTES_8 = (uint64_t)33 << 20;        // 8-byte elements
constexpr uint64_t SCAN_TWO_MAX_BYTES_4_SHORT = (uint64_t)36 << 20;  // 4-byte elements, last tile at most half full

template <typename T>
inline bool scan_takes_two(uint64_t n) {
  if (n > SCAN_TWO_MAX_BYTES / sizeof(T)) return false;
  const uint64_t bytes = n * sizeof(T);
  if (sizeof(T) == 8) return bytes <= SCAN_TWO_MAX_BYTES_8;
  constexpr uint64_t LARGE_TILE = (uint64_t)ScanShapeLarge::BLOCK * ScanShapeLarge::CHUNKS * 16;
  if (sizeof(T) == 4 && bytes % LARGE_TILE <= LARGE_TILE / 2) return bytes <= SCAN_TWO_MAX_BYTES_4_SHORT;
  return true;
}

// An array that fits one workgroup takes the second launch alone: up to 16 KiB one of the shape above, elements of 4 and
// 8 bytes up to 64 KiB one of this shape.  Whole call back to back in us, single pass / here: 4093 int32 7.2 / 4.3, 8445
// 7.3 / 4.7, 16381 7.2 / 6.8 (two launches 7.1), 8189 float64 7.5 / 4.8; int8 8189 7.9 / 6.3, uint8 minimum 4093 7.7 / 5.7.
// Eight vectors per lane, and arrays of up to 128 KiB: 16381 int32 7.1, 32509 11.7 (two launches 7.2); smaller elements, as
// many more of them, spill, 102397 int8 36 (two launches 7.9).
struct ScanShapeOne { static constexpr int BLOCK = 1024, CHUNKS = 4; };

static __global__ void tile_state_init_kernel(uint64_t* __restrict__ words, uint64_t count,
                                       uint32_t* __restrict__ counters, uint32_t num_counters) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) words[i] = 0;
  if (i < num_counters) counters[i] = 0;
}

// Previous lane's value (lane 0 receives `id`).
template <typename T>
TA_DEVICE T wave_shift_up(T v, T id) {
  return dpp_move<0x138 /* wave_shr:1 */>(id, v);
}

// `finished`, when given, makes the kernel leave its descriptors the way it found them: every tile
// counts itself in once its look-back is over, and the tile that completes the count clears the
// descriptors, the ticket and the counter again.  Storage that is only ever used that way (the
// library's own, all zero when the module is loaded) needs no clearing launch in front of the kernel.
template <typename T, typename Op, typename Pre, bool EXCLUSIVE, bool ALIGNED, typename Shape>
__global__ __launch_bounds__(Shape::BLOCK) void scan_kernel(const T* in, T* out, uint64_t n, T init,
                                                          uint64_t* __restrict__ status,
                                                          uint32_t* __restrict__ ticket,
                                                          uint32_t* __restrict__ finished) {
  constexpr int SCAN_BLOCK = Shape::BLOCK;
  constexpr int SCAN_CHUNKS = Shape::CHUNKS;
  constexpr int VEC = Vec16<T>::N;
  constexpr int WAVES = SCAN_BLOCK / WAVE;
  constexpr uint32_t WAVE_SPAN = WAVE * SCAN_CHUNKS * VEC;  // elements per wave
  constexpr uint32_t TILE = WAVES * WAVE_SPAN;
  constexpr int W = TileWords<T>::W;
  const Op op;
  const Pre pre;
  const T id = Op::template identity<T>();

  __shared__ uint32_t s_tile;
  __shared__ T s_wave_agg[WAVES];
  __shared__ T s_prefix;
  __shared__ uint32_t s_last;

  if (threadIdx.x == 0) {
    s_tile = atomicAdd(ticket, 1u);
    s_last = 0;
  }
  __syncthreads();
  const uint32_t tile = s_tile;
  const uint64_t tile_base = (uint64_t)tile * TILE;
  const uint32_t valid = (uint32_t)((n - tile_base < TILE) ? (n - tile_base) : TILE);
  const int wave = threadIdx.x / WAVE;
  const int lane = threadIdx.x % WAVE;
  const uint32_t lane_off = wave * WAVE_SPAN + lane * VEC;  // + j*64*VEC per chunk

  // ---- load
  Vec16<T> x[SCAN_CHUNKS];
  if (valid == TILE) {
#pragma unroll
    for (int j = 0; j < SCAN_CHUNKS; ++j)
      x[j] = load_vec<ALIGNED>(in + tile_base + lane_off + j * (WAVE * VEC));
#pragma unroll
    for (int j = 0; j < SCAN_CHUNKS; ++j) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) x[j].v[i] = pre(x[j].v[i]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < SCAN_CHUNKS; ++j) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        const uint32_t e = lane_off + j * (WAVE * VEC) + i;
        x[j].v[i] = (e < valid) ? pre(in[tile_base + e]) : id;
      }
    }
  }

  // ---- the tile's aggregate first, and published at once: a later tile's look-back can pass
  // this tile as soon as the sum is known, it does not have to wait for the scan below
  // (plus, minimum and maximum commute, so the lanes may fold their own elements first)
  {
    T lane_total = id;
#pragma unroll
    for (int j = 0; j < SCAN_CHUNKS; ++j) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) lane_total = op(lane_total, x[j].v[i]);
    }
    const T wave_total = wave_reduce(lane_total, op);
    if (lane == 0) s_wave_agg[wave] = wave_total;
  }
  __syncthreads();
  T wave_prefix = id;
  T block_agg = id;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    if (w == wave) wave_prefix = block_agg;
    block_agg = op(block_agg, s_wave_agg[w]);
  }
  uint64_t* my_slot = status + (size_t)tile * W;
  if (threadIdx.x == 0) tile_publish<T>(my_slot, tile == 0 ? TS_INCLUSIVE : TS_PARTIAL, block_agg);

  // ---- wave-local scan in place: every element becomes the fold of the wave's span up to
  // it (inclusive), or up to but excluding it (exclusive); CHUNKS DPP wave scans chained by
  // the wave total.  Nothing but x[] and the carry stays live.
  T carry = id;  // fold of this wave's chunks before chunk j
#pragma unroll
  for (int j = 0; j < SCAN_CHUNKS; ++j) {
    T s = x[j].v[0];
#pragma unroll
    for (int i = 1; i < VEC; ++i) s = op(s, x[j].v[i]);
    const T incl = wave_inclusive_scan(s, op, id);
    T run = op(carry, wave_shift_up(incl, id));
    carry = op(carry, readlane(incl, WAVE - 1));
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      if constexpr (EXCLUSIVE) {
        const T next = op(run, x[j].v[i]);
        x[j].v[i] = run;
        run = next;
      } else {
        run = op(run, x[j].v[i]);
        x[j].v[i] = run;
      }
    }
  }

  // ---- cross-tile prefix
  if (wave == 0) {
    T tile_excl = id;
    if (tile != 0) {
      tile_excl = tile_lookback<T>(status, tile, op, id);
      if (lane == 0) tile_publish<T>(my_slot, TS_INCLUSIVE, op(tile_excl, block_agg));
    }
    if (lane == 0) {
      s_prefix = tile_excl;
      // Counted in only after this tile's last descriptor store has been acknowledged (the wait
      // below; descriptor stores and this counter are agent-scope accesses that bypass the
      // non-coherent caches, so no cache write-back is involved -- a release fence here would
      // write back the L2 with the kernel's output in it, once per tile).  Whoever completes the
      // count knows that no descriptor will be read or written again.
      if (finished != nullptr) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        s_last = __hip_atomic_fetch_add(finished, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
      }
    }
  }
  __syncthreads();
  T prefix = s_prefix;
  if constexpr (EXCLUSIVE) prefix = (tile == 0) ? init : op(init, prefix);
  prefix = op(prefix, wave_prefix);

  // ---- apply the prefix of everything before this wave and store
#pragma unroll
  for (int j = 0; j < SCAN_CHUNKS; ++j) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) x[j].v[i] = op(prefix, x[j].v[i]);
  }
  if (valid == TILE) {
#pragma unroll
    for (int j = 0; j < SCAN_CHUNKS; ++j)
      store_vec<ALIGNED>(out + tile_base + lane_off + j * (WAVE * VEC), x[j]);
  } else {
#pragma unroll
    for (int j = 0; j < SCAN_CHUNKS; ++j) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        const uint32_t e = lane_off + j * (WAVE * VEC) + i;
        if (e < valid) out[tile_base + e] = x[j].v[i];
      }
    }
  }
  if (s_last) {
    const uint64_t words = (uint64_t)gridDim.x * W;
    for (uint64_t i = threadIdx.x; i < words; i += SCAN_BLOCK) status[i] = 0;
    if (threadIdx.x == 0) {
      *ticket = 0;
      *finished = 0;
    }
  }
}

// ------------------------------------------------------------------ two launches
// Vector j of a lane in a tile of which `valid` elements exist (its last tile): a whole vector where the
// wave's vectors j exist altogether, else elements, none past the last one; what does not exist becomes id.
template <bool ALIGNED, typename T, typename Pre>
TA_DEVICE Vec16<T> scan_load_ragged(const T* tile, uint32_t first, uint32_t wave_first, uint32_t valid, T id, Pre pre) {
  constexpr int VEC = Vec16<T>::N;
  Vec16<T> x;
  if (wave_first + WAVE * VEC <= valid) {
    x = load_vec<ALIGNED>(tile + first);
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) x.v[i] = tile[first + i < valid ? first + i : valid - 1];
  }
#pragma unroll
  for (int i = 0; i < VEC; ++i) x.v[i] = (first + i < valid) ? pre(x.v[i]) : id;
  return x;
}

// First launch: the fold of every tile but the last one.
template <typename T, typename Op, typename Pre, bool ALIGNED, typename Shape>
__global__ __launch_bounds__(Shape::BLOCK) void scan_partials_kernel(const T* __restrict__ in, T* __restrict__ partials) {
  constexpr int VEC = Vec16<T>::N;
  const Op op;
  const Pre pre;
  const T* tile = in + (uint64_t)blockIdx.x * (Shape::BLOCK * Shape::CHUNKS * VEC);
  Vec16<T> x[Shape::CHUNKS];
#pragma unroll
  for (int j = 0; j < Shape::CHUNKS; ++j) x[j] = load_vec<ALIGNED>(tile + (j * Shape::BLOCK + threadIdx.x) * VEC);
  T acc[VEC];
#pragma unroll
  for (int i = 0; i < VEC; ++i) acc[i] = pre(x[0].v[i]);
#pragma unroll
  for (int j = 1; j < Shape::CHUNKS; ++j) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = op(acc[i], pre(x[j].v[i]));
  }
#pragma unroll
  for (int i = 1; i < VEC; ++i) acc[0] = op(acc[0], acc[i]);
  __shared__ T s_wave[Shape::BLOCK / WAVE];
  const T wave_total = wave_reduce(acc[0], op);
  if (threadIdx.x % WAVE == 0) s_wave[threadIdx.x / WAVE] = wave_total;
  __syncthreads();
  if (threadIdx.x == 0) {
    T total = s_wave[0];
#pragma unroll
    for (int w = 1; w < Shape::BLOCK / WAVE; ++w) total = op(total, s_wave[w]);
    partials[blockIdx.x] = total;
  }
}

// Second launch: every tile folds the partials of the tiles before it (they fit the caches, and arrive
// while its own elements do) and scans its elements.  A call of one tile needs nothing but this launch.
template <typename T, typename Op, typename Pre, bool EXCLUSIVE, bool ALIGNED, typename Shape>
__global__ __launch_bounds__(Shape::BLOCK) void scan_apply_kernel(const T* in, T* out, uint64_t n, T init,
                                                                  const T* __restrict__ partials) {
  constexpr int SCAN_BLOCK = Shape::BLOCK;
  constexpr int SCAN_CHUNKS = Shape::CHUNKS;
  constexpr int VEC = Vec16<T>::N;
  constexpr int WAVES = SCAN_BLOCK / WAVE;
  constexpr uint32_t WAVE_SPAN = WAVE * SCAN_CHUNKS * VEC;
  constexpr uint32_t TILE = WAVES * WAVE_SPAN;
  const Op op;
  const Pre pre;
  const T id = Op::template identity<T>();
  __shared__ T s_wave_agg[WAVES];
  __shared__ T s_before[WAVES];

  const uint32_t tile = blockIdx.x;
  const uint64_t tile_base = (uint64_t)tile * TILE;
  const uint32_t valid = (uint32_t)((n - tile_base < TILE) ? (n - tile_base) : TILE);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
  const int lane = threadIdx.x % WAVE;
  const uint32_t lane_off = wave * WAVE_SPAN + lane * VEC;

  Vec16<T> x[SCAN_CHUNKS];
  if (valid == TILE) {
#pragma unroll
    for (int j = 0; j < SCAN_CHUNKS; ++j) x[j] = load_vec<ALIGNED>(in + tile_base + lane_off + j * (WAVE * VEC));
  } else {
#pragma unroll
    for (int j = 0; j < SCAN_CHUNKS; ++j) {
      const uint32_t wave_first = wave * WAVE_SPAN + j * (WAVE * VEC);
      if (wave_first < valid) {
        x[j] = scan_load_ragged<ALIGNED>(in + tile_base, lane_off + j * (WAVE * VEC), wave_first, valid, id, pre);
      } else {
#pragma unroll
        for (int i = 0; i < VEC; ++i) x[j].v[i] = id;
      }
    }
  }
  T before = id;
  for (uint32_t t = threadIdx.x; t < tile; t += SCAN_BLOCK) before = op(before, partials[t]);
  if (valid == TILE) {
#pragma unroll
    for (int j = 0; j < SCAN_CHUNKS; ++j) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) x[j].v[i] = pre(x[j].v[i]);
    }
  }

  // ---- wave-local scan in place, as in scan_kernel
  T carry = id;
#pragma unroll
  for (int j = 0; j < SCAN_CHUNKS; ++j) {
    T s = x[j].v[0];
#pragma unroll
    for (int i = 1; i < VEC; ++i) s = op(s, x[j].v[i]);
    const T incl = wave_inclusive_scan(s, op, id);
    T run = op(carry, wave_shift_up(incl, id));
    carry = op(carry, readlane(incl, WAVE - 1));
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      const T next = op(run, x[j].v[i]);
      x[j].v[i] = EXCLUSIVE ? run : next;
      run = next;
    }
  }
  before = wave_reduce(before, op);
  if (lane == 0) {
    s_wave_agg[wave] = carry;
    s_before[wave] = before;
  }
  __syncthreads();
  T wave_prefix = id;
  T prefix = id;
  if constexpr (WAVES > 4) {
    // the totals of many waves by a scan of their own: fewer terms in a row, in time and in rounding
    const T totals = wave_inclusive_scan(lane < WAVES ? s_wave_agg[lane] : id, op, id);
    if (wave > 0) wave_prefix = readlane(totals, wave - 1);
  } else {
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      if (w < wave) wave_prefix = op(wave_prefix, s_wave_agg[w]);
    }
  }
#pragma unroll
  for (int w = 0; w < WAVES; ++w) prefix = op(prefix, s_before[w]);
  if constexpr (EXCLUSIVE) prefix = (tile == 0) ? init : op(init, prefix);
  prefix = op(prefix, wave_prefix);
#pragma unroll
  for (int j = 0; j < SCAN_CHUNKS; ++j) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) x[j].v[i] = op(prefix, x[j].v[i]);
    const uint32_t wave_first = wave * WAVE_SPAN + j * (WAVE * VEC);
    T* dst = out + tile_base + lane_off + j * (WAVE * VEC);
    if (wave_first + WAVE * VEC <= valid) {
      store_vec<ALIGNED>(dst, x[j]);
    } else {
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        if (lane_off + j * (WAVE * VEC) + i < valid) dst[i] = x[j].v[i];
      }
    }
  }
}

template <bool EXCLUSIVE, typename Pre>
struct ScanLaunch {
  template <typename Shape, typename T>
  static constexpr uint64_t tile_of() { return (uint64_t)Shape::BLOCK * Shape::CHUNKS * Vec16<T>::N; }

  // The single-pass kernel's temporary storage for n elements: shape, tiles, and where what begins.
  struct SinglePass {
    bool large;
    uint64_t tiles;
    size_t off_ticket, off_status, bytes;
  };
  template <typename T>
  static SinglePass single_pass(uint64_t n) {
    SinglePass p;
    p.large = n >= SCAN_LARGE_MIN_BYTES / sizeof(T);
    const uint64_t tile = p.large ? tile_of<ScanShapeLarge, T>() : tile_of<ScanShapeSmall, T>();
    p.tiles = n / tile + (n % tile != 0);
    TempLayout lay;
    p.off_ticket = lay.add(2 * sizeof(uint32_t));  // the ticket and the count of finished tiles
    p.off_status = lay.add((size_t)p.tiles * TileWords<T>::W * sizeof(uint64_t));
    p.bytes = lay.total;
    return p;
  }

  // KEPT_CLEAN: `temp` is storage of the library's own that only this function uses and that was all zero to begin
  // with; the kernel then clears up after itself and no clearing launch precedes it.
  template <typename T, typename Op, typename Shape, bool KEPT_CLEAN>
  static int launch_single_pass(void* temp, const SinglePass& p, const T* in, T* out, uint64_t n, T init, hipStream_t stream) {
    uint32_t* ticket = reinterpret_cast<uint32_t*>(static_cast<char*>(temp) + p.off_ticket);
    uint64_t* status = reinterpret_cast<uint64_t*>(static_cast<char*>(temp) + p.off_status);
    const uint64_t words = p.tiles * TileWords<T>::W;
    uint32_t* finished = KEPT_CLEAN ? ticket + 1 : nullptr;
    if (!KEPT_CLEAN) {
      TA_LAUNCH("tile_state_init", stream, tile_state_init_kernel, dim3((uint32_t)((words + 255) / 256)), dim3(256), status, words, ticket, 2u);
      TA_CHECK_LAUNCH();
    }
    if (is_aligned16(in) && is_aligned16(out))
      TA_LAUNCH("scan", stream, (scan_kernel<T, Op, Pre, EXCLUSIVE, true, Shape>), dim3((uint32_t)p.tiles), dim3(Shape::BLOCK), in, out, n, init, status, ticket, finished);
    else
      TA_LAUNCH("scan", stream, (scan_kernel<T, Op, Pre, EXCLUSIVE, false, Shape>), dim3((uint32_t)p.tiles), dim3(Shape::BLOCK), in, out, n, init, status, ticket, finished);
    TA_CHECK_LAUNCH();
    return 0;
  }

  // Two launches; `temp` holds the partials of the tiles.
  template <typename T>
  static size_t partials_bytes(uint64_t n) {
    return align_up((size_t)(n / tile_of<ScanShapeTwo, T>() + 1) * sizeof(T), 256);
  }

  template <typename T, typename Op>
  static int launch_two(void* temp, const T* in, T* out, uint64_t n, T init, hipStream_t stream) {
    using Shape = ScanShapeTwo;
    const uint32_t tiles = (uint32_t)((n + tile_of<Shape, T>() - 1) / tile_of<Shape, T>());
    T* partials = static_cast<T*>(temp);
    if (is_aligned16(in))
      TA_LAUNCH("scan_partials", stream, (scan_partials_kernel<T, Op, Pre, true, Shape>), dim3(tiles - 1), dim3(Shape::BLOCK), in, partials);
    else
      TA_LAUNCH("scan_partials", stream, (scan_partials_kernel<T, Op, Pre, false, Shape>), dim3(tiles - 1), dim3(Shape::BLOCK), in, partials);
    TA_CHECK_LAUNCH();
    return launch_apply<T, Op, Shape>(tiles, in, out, n, init, partials, stream);
  }

  template <typename T, typename Op, typename Shape>
  static int launch_apply(uint32_t tiles, const T* in, T* out, uint64_t n, T init, const T* partials, hipStream_t stream) {
    if (is_aligned16(in) && is_aligned16(out))
      TA_LAUNCH("scan", stream, (scan_apply_kernel<T, Op, Pre, EXCLUSIVE, true, Shape>), dim3(tiles), dim3(Shape::BLOCK), in, out, n, init, partials);
    else
      TA_LAUNCH("scan", stream, (scan_apply_kernel<T, Op, Pre, EXCLUSIVE, false, Shape>), dim3(tiles), dim3(Shape::BLOCK), in, out, n, init, partials);
    TA_CHECK_LAUNCH();
    return 0;
  }

  // Checks the arguments of a call; reads the initial value where there is one.
  template <typename T, typename Op>
  static int check_args(size_t held, size_t need, const T* in, T* out, uint64_t n, const void* init, T& init_v) {
    init_v = Op::template identity<T>();
    if (held < need) return (int)hipErrorInvalidValue;
    if (n == 0) return 0;
    if (!in || !out || (EXCLUSIVE && !init)) return (int)hipErrorInvalidValue;
    if (EXCLUSIVE) __builtin_memcpy(&init_v, init, sizeof(T));
    return 0;
  }

  template <typename T, typename Op>
  static int run(void* temp, size_t* temp_bytes, const void* in_, void* out_, uint64_t n, const void* init, hipStream_t stream) {
    const T* in = static_cast<const T*>(in_);
    T* out = static_cast<T*>(out_);
    const SinglePass single = single_pass<T>(n);
    if (single.tiles > 0xffffffffull) return (int)hipErrorInvalidValue;
    const bool two = scan_takes_two<T>(n);
    const size_t partials = two ? partials_bytes<T>(n) : 0;
    if (temp == nullptr) {
      *temp_bytes = single.bytes > partials ? single.bytes : partials;
      return 0;
    }
    T init_v;
    const int rc = check_args<T, Op>(*temp_bytes, single.bytes, in, out, n, init, init_v);
    if (rc != 0 || n == 0) return rc;
    if (n <= tile_of<ScanShapeTwo, T>()) return launch_apply<T, Op, ScanShapeTwo>(1, in, out, n, init_v, nullptr, stream);
    if constexpr (sizeof(T) >= 4) {
      if (n <= tile_of<ScanShapeOne, T>()) return launch_apply<T, Op, ScanShapeOne>(1, in, out, n, init_v, nullptr, stream);
    }
    // (storage that was asked for with a longer array may hold the single pass's descriptors and not the partials)
    if (two && *temp_bytes >= partials && is_memory_of_this_device(in)) return launch_two<T, Op>(temp, in, out, n, init_v, stream);
    return single.large ? launch_single_pass<T, Op, ScanShapeLarge, false>(temp, single, in, out, n, init_v, stream)
                        : launch_single_pass<T, Op, ScanShapeSmall, false>(temp, single, in, out, n, init_v, stream);
  }

  // In storage that is kept clean (temp null: the size query).
  template <typename T, typename Op>
  static int run_kept_clean(void* temp, size_t* temp_bytes, const void* in_, void* out_, uint64_t n, hipStream_t stream) {
    const T* in = static_cast<const T*>(in_);
    T* out = static_cast<T*>(out_);
    const SinglePass single = single_pass<T>(n);
    if (single.tiles > 0xffffffffull) return (int)hipErrorInvalidValue;
    if (temp == nullptr) {
      *temp_bytes = single.bytes;
      return 0;
    }
    T init_v;
    const int rc = check_args<T, Op>(*temp_bytes, single.bytes, in, out, n, nullptr, init_v);
    if (rc != 0 || n == 0) return rc;
    return single.large ? launch_single_pass<T, Op, ScanShapeLarge, true>(temp, single, in, out, n, init_v, stream)
                        : launch_single_pass<T, Op, ScanShapeSmall, true>(temp, single, in, out, n, init_v, stream);
  }
};

}  // namespace ta
