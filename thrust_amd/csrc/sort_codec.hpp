// Order-preserving map between keys and unsigned radix codes.
#pragma once
#include "common.hpp"

namespace ta {

// Key <-> radix encoding, decided at run time (uniform across the grid).
//   sign:   sign bit for signed integers and floats, else 0
//   fmask:  all ones for floating point, else 0
//   dmask:  all ones for descending order, else 0
template <typename K>
struct KeyCodec {
  K sign, fmask, dmask;
  uint32_t plain;  // all three masks are zero: encode/decode are the identity
  TA_DEVICE K encode(K k) const {
    using SK = typename std::make_signed<K>::type;
    const K neg = (K)((SK)k >> (sizeof(K) * 8 - 1));
    return k ^ ((neg & fmask) | sign) ^ dmask;
  }
  TA_DEVICE K decode(K e) const {
    using SK = typename std::make_signed<K>::type;
    e ^= dmask;
    const K pos = (K)((SK)e >> (sizeof(K) * 8 - 1));
    return e ^ ((~pos & fmask) | sign);
  }
};

template <typename K>
static KeyCodec<K> make_codec(int dtype, int descending) {
  KeyCodec<K> c;
  const bool is_float = dtype == THRUST_AMD_F32 || dtype == THRUST_AMD_F64;
  const bool is_signed = is_float || dtype == THRUST_AMD_I8 || dtype == THRUST_AMD_I16 ||
                         dtype == THRUST_AMD_I32 || dtype == THRUST_AMD_I64;
  c.sign = is_signed ? (K)((K)1 << (sizeof(K) * 8 - 1)) : (K)0;
  c.fmask = is_float ? (K)~(K)0 : (K)0;
  c.dmask = descending ? (K)~(K)0 : (K)0;
  c.plain = (!is_signed && !descending) ? 1u : 0u;
  return c;
}

}  // namespace ta
