// thrust_amd_reduce: tree reduction in two launches, or one.
//
//   kernel 1  grid-stride over tiles of BLOCK*VEC*UNROLL elements; every lane issues
//             UNROLL independent 16-byte loads per tile, folds them into one register
//             accumulator, then wave64 DPP reduction -> LDS across the waves -> one
//             partial per workgroup.
//   kernel 2  one workgroup folds init and the partials and writes *d_out.
//
// Short arrays one workgroup folds in one launch (reduce_takes_one).
//
// HBM traffic: n*sizeof(T) read, (grid+1)*sizeof(T) written -- the kernel is bound by
// the read stream alone.  Replaces the ReduceAgent pair of the reference
// (thrust/system/cuda/detail/reduce.h:151-665) and cub::DispatchReduce (:946-954).
#include "common.hpp"
#include "dispatch.hpp"
#include "launch.hpp"
#include "reduce_common.hpp"

namespace ta {

// Short arrays: one workgroup, one launch.  One CU draws some 110 GB/s, so its time grows by 4.7 us with every
// 512 KiB, while the second launch costs 3 us, most of it the host's: whole call back to back, two launches
// against one, 400 KB 10.2 -> 7.0 us, 800 KB 10.4 -> 7.8, 1 MiB 10.0 -> 8.5, 1.6 MB 10.1 -> 12.9.  The line is drawn
// at half of where they meet, for a call that is waited for pays its launches but once.
// The order of addition: the 8 vectors of a step by a tree, up to four steps in a row, the places of a vector, the lanes
// and the waves by trees again, so that short sums of floats are no less exact than by two launches, where a lane adds
// up to 32 terms in a row.  Restated on the CPU, 200 arrays of uniform [0, 1) each, rms relative error two launches / here
// (/ each place of the vectors in a row, then the waves in a row): float32 5003 4.5e-8 / 4.2e-8 (7.9e-8), 100003 4.5e-8 /
// 3.5e-8 (6.8e-8), 131072 4.4e-8 / 4.5e-8 (6.5e-8); float64 20011 9.2e-17 / 7.7e-17 (1.4e-16), 65536 8.1e-17 / 7.9e-17 (1.1e-16).
constexpr int REDUCE_ONE_BLOCK = 1024;
constexpr uint64_t REDUCE_ONE_MAX_BYTES = (uint64_t)512 << 10;
// Single bytes: unpacking them is what takes the time (int8 minimum back to back, two launches / one, 300 KiB 7.3 / 6.9 us,
// 511 KiB 7.3 / 9.5).
constexpr uint64_t REDUCE_ONE_MAX_BYTES_1 = (uint64_t)256 << 10;
// Memory behind a link, pinned host memory for one: a workgroup alone draws some 25 GB/s from it (100 KiB of int32 8.4 / 6.2
// us, 300 KiB 11.1 / 15.2, 511 KiB 15.6 / 22.0).
constexpr uint64_t REDUCE_ONE_MAX_BYTES_FAR = (uint64_t)128 << 10;

// Whether one workgroup folds an array of so many bytes (at least one element).
template <typename T>
inline bool reduce_takes_one(const T* in, uint64_t n) {
  constexpr uint64_t most = sizeof(T) == 1 ? REDUCE_ONE_MAX_BYTES_1 : REDUCE_ONE_MAX_BYTES;
  if (n > most / sizeof(T)) return false;
  return n <= REDUCE_ONE_MAX_BYTES_FAR / sizeof(T) || is_memory_of_this_device(in);
}

template <typename T, typename Op, bool ALIGNED>
__global__ __launch_bounds__(REDUCE_BLOCK) void reduce_partials_kernel(const T* __restrict__ in,
                                                                       uint64_t n,
                                                                       T* __restrict__ partials) {
  constexpr int VEC = Vec16<T>::N;
  constexpr uint64_t TILE = (uint64_t)REDUCE_BLOCK * VEC * REDUCE_UNROLL;
  const Op op;
  T acc = Op::template identity<T>();

  const uint64_t full_tiles = n / TILE;
  for (uint64_t tile = blockIdx.x; tile < full_tiles; tile += gridDim.x) {
    const T* base = in + tile * TILE + (uint64_t)threadIdx.x * VEC;
    Vec16<T> x[REDUCE_UNROLL];
#pragma unroll
    for (int u = 0; u < REDUCE_UNROLL; ++u)
      x[u] = load_vec<ALIGNED>(base + (uint64_t)u * REDUCE_BLOCK * VEC);
#pragma unroll
    for (int u = 0; u < REDUCE_UNROLL; ++u) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc = op(acc, x[u].v[i]);
    }
  }
  // Ragged tail (< TILE elements): element-wise, spread over the first workgroups.
  const uint64_t tail_begin = full_tiles * TILE;
  for (uint64_t i = tail_begin + (uint64_t)blockIdx.x * REDUCE_BLOCK + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * REDUCE_BLOCK)
    acc = op(acc, in[i]);

  __shared__ T lds[REDUCE_BLOCK / WAVE];
  const T r = block_reduce<REDUCE_BLOCK>(acc, op, lds);
  if (threadIdx.x == 0) partials[blockIdx.x] = r;
}

template <typename T, typename Op, bool ALIGNED>
__global__ __launch_bounds__(REDUCE_ONE_BLOCK) void reduce_one_kernel(const T* __restrict__ in, uint32_t n, T init, T* __restrict__ out) {
  constexpr int VEC = Vec16<T>::N;
  constexpr int WAVES = REDUCE_ONE_BLOCK / WAVE;
  constexpr int UNROLL = sizeof(T) == 1 ? 4 : REDUCE_UNROLL;  // (8 vectors of single bytes, unpacked, do not fit the registers)
  constexpr uint32_t STEP = REDUCE_ONE_BLOCK * UNROLL;
  static_assert((UNROLL & (UNROLL - 1)) == 0 && WAVES <= WAVE, "trees");
  const Op op;
  const T id = Op::template identity<T>();
  T acc[VEC];
#pragma unroll
  for (int i = 0; i < VEC; ++i) acc[i] = id;
  const uint32_t vecs = n / VEC;
  auto fold = [&](Vec16<T> (&x)[UNROLL]) {
#pragma unroll
    for (int half = UNROLL / 2; half > 0; half /= 2) {
#pragma unroll
      for (int u = 0; u < half; ++u) {
#pragma unroll
        for (int i = 0; i < VEC; ++i) x[u].v[i] = op(x[u].v[i], x[u + half].v[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = op(acc[i], x[0].v[i]);
  };
  // the elements behind the last whole vector
  const bool has_rest = threadIdx.x < n - vecs * VEC;
  T rest = id;
  if (has_rest) rest = in[vecs * VEC + threadIdx.x];
  uint32_t v = threadIdx.x;
  for (; v - threadIdx.x + STEP <= vecs; v += STEP) {
    Vec16<T> x[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) x[u] = load_vec<ALIGNED>(in + (uint64_t)(v + u * REDUCE_ONE_BLOCK) * VEC);
    fold(x);
  }
  if (v - threadIdx.x < vecs) {
    // the last step, not whole: loads without predicates (a predicated one is waited for before the next
    // is issued), of the last vector where there is none
    Vec16<T> x[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const uint32_t at = v + u * REDUCE_ONE_BLOCK;
      x[u] = load_vec<ALIGNED>(in + (uint64_t)(at < vecs ? at : vecs - 1) * VEC);
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
#pragma unroll
      for (int i = 0; i < VEC; ++i) x[u].v[i] = v + u * REDUCE_ONE_BLOCK < vecs ? x[u].v[i] : id;
    }
    fold(x);
  }
#pragma unroll
  for (int half = VEC / 2; half > 0; half /= 2) {
#pragma unroll
    for (int i = 0; i < half; ++i) acc[i] = op(acc[i], acc[i + half]);
  }
  __shared__ T lds[WAVES];
  const T total = wave_reduce(op(acc[0], rest), op);
  if (threadIdx.x % WAVE == 0) lds[threadIdx.x / WAVE] = total;
  __syncthreads();
  if (threadIdx.x < WAVE) {
    const T r = wave_reduce(threadIdx.x < WAVES ? lds[threadIdx.x] : id, op);
    if (threadIdx.x == 0) *out = op(init, r);
  }
}

struct ReduceLaunch {
  template <typename T, typename Op>
  static int run(void* temp, const void* in, uint64_t n, const void* init, void* d_out,
                 hipStream_t stream) {
    T init_v;
    __builtin_memcpy(&init_v, init, sizeof(T));
    T* partials = static_cast<T*>(temp);
    const uint32_t grid = reduce_grid(n, sizeof(T));
    const T* src = static_cast<const T*>(in);
    if (n == 0) {
      TA_LAUNCH("reduce_final", stream, (reduce_final_kernel<T, Op>), dim3(1), dim3(REDUCE_BLOCK), partials, 0u, init_v, static_cast<T*>(d_out));
      TA_CHECK_LAUNCH();
      return 0;
    }
    if (reduce_takes_one(src, n)) {
      if (is_aligned16(in))
        TA_LAUNCH("reduce_one", stream, (reduce_one_kernel<T, Op, true>), dim3(1), dim3(REDUCE_ONE_BLOCK), src, (uint32_t)n, init_v, static_cast<T*>(d_out));
      else
        TA_LAUNCH("reduce_one", stream, (reduce_one_kernel<T, Op, false>), dim3(1), dim3(REDUCE_ONE_BLOCK), src, (uint32_t)n, init_v, static_cast<T*>(d_out));
      TA_CHECK_LAUNCH();
      return 0;
    }
    if (is_aligned16(in))
      TA_LAUNCH("reduce_partials", stream, (reduce_partials_kernel<T, Op, true>), dim3(grid), dim3(REDUCE_BLOCK), src, n, partials);
    else
      TA_LAUNCH("reduce_partials", stream, (reduce_partials_kernel<T, Op, false>), dim3(grid), dim3(REDUCE_BLOCK), src, n, partials);
    TA_CHECK_LAUNCH();
    TA_LAUNCH("reduce_final", stream, (reduce_final_kernel<T, Op>), dim3(1), dim3(REDUCE_BLOCK), partials, grid, init_v, static_cast<T*>(d_out));
    TA_CHECK_LAUNCH();
    return 0;
  }
};

}  // namespace ta

TA_EXPORT int thrust_amd_reduce(void* temp, size_t* temp_bytes, const void* in, uint64_t n,
                                 int dtype, int op, const void* init, void* d_out, void* stream) {
  using namespace ta;
  if (!temp_bytes || !valid_dtype(dtype) || !valid_binop(op)) return (int)hipErrorInvalidValue;
  const size_t elem = thrust_amd_dtype_size(dtype);
  const size_t need = align_up((size_t)NUM_CU * REDUCE_BLOCKS_PER_CU * elem, 256);
  if (temp == nullptr) {
    *temp_bytes = need;
    return 0;
  }
  if (*temp_bytes < need || !init || !d_out || (n && !in)) return (int)hipErrorInvalidValue;
  return dispatch_dtype_op<ReduceLaunch>(dtype, op, temp, in, n, init, d_out, (hipStream_t)stream);
}
