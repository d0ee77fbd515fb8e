// thrust_amd_reduce: tree reduction in two launches, or one.
//
//   kernel 1  grid-stride over tiles of BLOCK*VEC*UNROLL elements; every lane issues
//             UNROLL independent 16-byte loads per tile, folds them into one register
//             accumulator, then wave64 DPP reduction -> LDS across the waves -> one
//             partial per workgroup.
//   kernel 2  one workgroup folds init and the partials and writes *d_out.
//
// Up to REDUCE_ONE_MAX_BYTES one workgroup does it all in one launch.
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
// A lane folds each place of its vectors by itself: no sum has more terms in a row than before.
constexpr int REDUCE_ONE_BLOCK = 1024;
constexpr uint64_t REDUCE_ONE_MAX_BYTES = (uint64_t)512 << 10;

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
  constexpr uint32_t STEP = REDUCE_ONE_BLOCK * REDUCE_UNROLL;
  const Op op;
  T acc[VEC];
#pragma unroll
  for (int i = 0; i < VEC; ++i) acc[i] = Op::template identity<T>();
  const uint32_t vecs = n / VEC;
  auto fold = [&](const Vec16<T>& x) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = op(acc[i], x.v[i]);
  };
  // the elements behind the last whole vector
  const bool has_rest = threadIdx.x < n - vecs * VEC;
  T rest = Op::template identity<T>();
  if (has_rest) rest = in[vecs * VEC + threadIdx.x];
  uint32_t v = threadIdx.x;
  for (; v - threadIdx.x + STEP <= vecs; v += STEP) {
    Vec16<T> x[REDUCE_UNROLL];
#pragma unroll
    for (int u = 0; u < REDUCE_UNROLL; ++u) x[u] = load_vec<ALIGNED>(in + (uint64_t)(v + u * REDUCE_ONE_BLOCK) * VEC);
#pragma unroll
    for (int u = 0; u < REDUCE_UNROLL; ++u) fold(x[u]);
  }
  if (v - threadIdx.x < vecs) {
    // the last step, not whole: loads without predicates (a predicated one is waited for before the next
    // is issued), of the last vector where there is none
    Vec16<T> x[REDUCE_UNROLL];
#pragma unroll
    for (int u = 0; u < REDUCE_UNROLL; ++u) {
      const uint32_t at = v + u * REDUCE_ONE_BLOCK;
      x[u] = load_vec<ALIGNED>(in + (uint64_t)(at < vecs ? at : vecs - 1) * VEC);
    }
#pragma unroll
    for (int u = 0; u < REDUCE_UNROLL; ++u) {
      if (v + u * REDUCE_ONE_BLOCK < vecs) fold(x[u]);
    }
  }
  acc[0] = op(acc[0], rest);
#pragma unroll
  for (int i = 1; i < VEC; ++i) acc[0] = op(acc[0], acc[i]);
  __shared__ T lds[REDUCE_ONE_BLOCK / WAVE];
  const T r = block_reduce<REDUCE_ONE_BLOCK>(acc[0], op, lds);
  if (threadIdx.x == 0) *out = op(init, r);
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
    if (n <= REDUCE_ONE_MAX_BYTES / sizeof(T)) {
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
