// Ranking the keys of one wave by digit: shared by the kernels of the radix sort.
#pragma once
#include "common.hpp"

namespace ta {

constexpr int RADIX_BITS = 8;
constexpr int RADIX_SIZE = 1 << RADIX_BITS;

// f(a, b, c) = a & ~(b ^ c): truth table index = a*4 + b*2 + c.
constexpr int BITOP_AND_XNOR = 0x90;

// Lanes with the same 8-bit d as this one: narrows the 64-bit mask (peers_lo, peers_hi) to them.
// Per digit bit: v_bfe_i32 (the lane's bit as 0 / -1), one ballot, and two v_bitop3 folding "same bit
// as mine" into the mask.
TA_DEVICE void wave_match_digit(uint32_t d, uint32_t& peers_lo, uint32_t& peers_hi) {
#pragma unroll
  for (int b = 0; b < RADIX_BITS; ++b) {
    int sb;
    // opaque to the optimiser so that the compare below is made on sb itself
    asm volatile("v_bfe_i32 %0, %1, %2, 1" : "=v"(sb) : "v"(d), "n"(b));
    const uint64_t m = __builtin_amdgcn_ballot_w64(sb != 0);
    peers_lo = __builtin_amdgcn_bitop3_b32(peers_lo, (uint32_t)m, (uint32_t)sb, BITOP_AND_XNOR);
    peers_hi = __builtin_amdgcn_bitop3_b32(peers_hi, (uint32_t)(m >> 32), (uint32_t)sb, BITOP_AND_XNOR);
  }
}

// Rank of this lane's key among the keys the wave has ranked so far and the ones of this round, lanes in
// order: my_cnt[d] (a counter in LDS private to the wave) plus the number of lower lanes with digit d.
// Raises the counter by the number of lanes with digit d; LDS executes a wave's instructions in
// order, so the next round reads the raised count.
TA_DEVICE uint32_t wave_rank_round(uint32_t d, uint32_t* my_cnt) {
  const uint32_t old = my_cnt[d];
  uint32_t peers_lo = ~0u, peers_hi = ~0u;
  wave_match_digit(d, peers_lo, peers_hi);
  // the count of peers in lower lanes is accumulated onto the counter's value
  const uint32_t rank = __builtin_amdgcn_mbcnt_hi(peers_hi, __builtin_amdgcn_mbcnt_lo(peers_lo, old));
  // The lowest lane of every group of peers bumps the counter for all of them: one LDS
  // write per distinct digit instead of an atomic per key, which an LDS bank serialises
  // when many lanes hold the same digit (float exponents, skewed keys).
  if (rank == old) my_cnt[d] = old + (uint32_t)__builtin_popcount(peers_lo) + (uint32_t)__builtin_popcount(peers_hi);
  return rank;
}

}  // namespace ta
