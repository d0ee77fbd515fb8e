// Host-side check of the rule by which device-to-device copies go to the library's copy kernel
// (thrust_amd/csrc/copy_rule.hpp, the functions runtime.hip calls): every copy it takes is a legal launch
// whose threads cover all its vectors, the larger ones are left to the runtime, and so are ranges that
// reach beyond the allocation they begin in.
#include <cstdint>
#include <cstdio>

#include "../../thrust_amd/csrc/copy_rule.hpp"

using namespace ta;

int main() {
  int failures = 0;
  auto expect = [&](bool ok, const char* what) {
    if (!ok) {
      std::printf("FAILED: %s\n", what);
      ++failures;
    }
  };
  const uint64_t GIB = (uint64_t)1 << 30, A = 0x7f0000000000;
  for (uint64_t bytes = 1; bytes <= 512 * GIB; bytes += bytes / 3 + 1) {
    for (int64_t d = -4097; d <= 4097; d += 4097) {
      const uint64_t b = bytes + (uint64_t)d;
      if ((int64_t)b <= 0 || !copy_kernel_takes(A, 2 * A, b)) continue;
      expect(copy_blocks(b) * COPY_BLOCK <= 0xffffffffull, "a launch has fewer than 2^32 threads");
      expect(copy_blocks(b) * COPY_BLOCK >= b / 16, "every vector has a thread");
    }
  }
  expect(copy_kernel_takes(A, 2 * A, 64 * GIB - 8192), "just below 64 GiB");
  expect(!copy_kernel_takes(A, 2 * A, 64 * GIB), "64 GiB is left to the runtime");
  expect(!copy_kernel_takes(A, 2 * A, 128 * GIB), "128 GiB is left to the runtime");
  expect(copy_kernel_takes(A + 5, 2 * A + 21, GIB), "equally misaligned buffers");
  expect(!copy_kernel_takes(A, 2 * A + 1, GIB), "differently misaligned buffers");
  expect(!copy_kernel_takes(A, 2 * A, COPY_KERNEL_MIN_BYTES - 1), "small copies");
  expect(copy_range_known(A, GIB, A, GIB), "a whole allocation");
  expect(copy_range_known(A + 16, GIB - 16, A, GIB), "the end of an allocation");
  expect(!copy_range_known(A, GIB + 1, A, GIB), "a byte past the end");
  expect(!copy_range_known(A + 16, GIB, A, GIB), "past the end from inside");
  expect(!copy_range_known(A + GIB + 1, 1, A, GIB), "behind the allocation");
  expect(!copy_range_known(A - 1, 1, A, GIB), "in front of the allocation");
  expect(!copy_range_known(A + 16, ~(uint64_t)0, A, GIB), "a size that wraps round");
  if (failures == 0) std::printf("PASSED\n");
  return failures != 0;
}
