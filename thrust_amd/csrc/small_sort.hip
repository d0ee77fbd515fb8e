// Instantiations and launcher of the one-workgroup sort (small_sort.hpp).
#include "common.hpp"
#include "dispatch.hpp"
#include "launch.hpp"
#include "small_sort.hpp"

namespace ta {

// Four waves have fewer barriers to wait at, sixteen rank faster (copy and sort of 2048 uint32: 12.9 us with
// 256 threads, 10.9 with 1024; of 1000: 10 us with either).  Kernels for no more keys per thread than a size needs: with
// code and loads for eight, copy and sort of 1025 (uint64, uint64) took 13.8 us (12.8 with each load behind its own
// predicate), now 11.5; 3001 uint32 13.0 -> 12.3, with uint32 values 14.1 -> 13.0, 1000 (uint64, uint64) 11.3 -> 10.7.
constexpr uint32_t SMALL_SORT_NARROW_MAX = 1024;

template <typename K, typename V, bool HAS_VALUES>
static int run_small_sort(K* keys, V* values, uint32_t n, const KeyCodec<K>& codec, int begin_bit, int end_bit, hipStream_t stream) {
  auto launch = [&](auto kernel, uint32_t block) {
    TA_LAUNCH("small_sort", stream, kernel, dim3(1), dim3(block), keys, values, n, codec, begin_bit, end_bit);
  };
  if (n <= SMALL_SORT_NARROW_MAX) launch(small_sort_kernel<K, V, HAS_VALUES, 256, 4>, 256);
  else if (n <= 2 * 1024) launch(small_sort_kernel<K, V, HAS_VALUES, 1024, 2>, 1024);
  else if (n <= 4 * 1024) launch(small_sort_kernel<K, V, HAS_VALUES, 1024, 4>, 1024);
  else launch(small_sort_kernel<K, V, HAS_VALUES, 1024, SMALL_ITEMS>, 1024);
  TA_CHECK_LAUNCH();
  return 0;
}

int small_sort(void* keys, void* values, uint32_t n, int key_dtype, size_t value_bytes, int descending, int begin_bit,
               int end_bit, hipStream_t stream) {
  return with_item_bytes(thrust_amd_dtype_size(key_dtype), [&](auto kt) {
    using K = typename decltype(kt)::type;
    const KeyCodec<K> codec = make_codec<K>(key_dtype, descending);
    if (value_bytes == 0)
      return run_small_sort<K, uint32_t, false>(static_cast<K*>(keys), nullptr, n, codec, begin_bit, end_bit, stream);
    return with_item_bytes(value_bytes, [&](auto vt) {
      using V = typename decltype(vt)::type;
      return run_small_sort<K, V, true>(static_cast<K*>(keys), static_cast<V*>(values), n, codec, begin_bit, end_bit, stream);
    });
  });
}

}  // namespace ta
