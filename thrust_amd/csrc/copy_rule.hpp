// Which device-to-device copies the copy kernel of runtime.hip takes; the others go to the runtime's own copy.
// Plain C++ (also compiled for the host by tests/cpp/test_copy_rule.cpp, which checks the limits).
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace ta {

constexpr uint32_t COPY_BLOCK = 256;  // threads of a workgroup, one 16-byte vector each

// Below this the copy lives in the caches and the runtime's kernel is as fast (64 MiB: 19.7 us with the kernel,
// 19.5 us with the runtime; 256 MiB: 88.8 against 98.9 us), without the pointer lookups.
constexpr uint64_t COPY_KERNEL_MIN_BYTES = (uint64_t)128 << 20;

// A launch may have at most 2^32 - 1 threads in a dimension (hipModuleLaunchKernel): copies from 64 GiB on go
// to the runtime.
constexpr uint64_t COPY_BLOCKS_MAX = 0xffffffffull / COPY_BLOCK;

inline uint64_t copy_blocks(uint64_t bytes) { return bytes / 16 / COPY_BLOCK + 1; }

// [p, p + bytes) lies inside the allocation [base, base + size).  The runtime's copy refuses a range that does not
// (the caller's mistake, which the kernel would carry out); it also knows buffers mapped from several allocations.
inline bool copy_range_known(uintptr_t p, uint64_t bytes, uintptr_t base, uint64_t size) {
  return p >= base && p - base <= size && bytes <= size - (p - base);
}

inline bool copy_kernel_takes(uintptr_t dst, uintptr_t src, uint64_t bytes) {
  return bytes >= COPY_KERNEL_MIN_BYTES && ((dst ^ src) & 15) == 0 && copy_blocks(bytes) <= COPY_BLOCKS_MAX;
}

}  // namespace ta
