// Rotary embedding of 16-bit channels, two a word, with the roundings of the
// eager expression x * cos + rotate_half(x) * sin: each product and the sum
// are rounded to the storage type.
#pragma once

#include "page_chunk.h"

namespace tw {

// Two floats rounded to nearest even, in one word (a conversion instruction).
__device__ __forceinline__ uint32_t narrow_pair(float a, float b, F16) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  const h2 w = {static_cast<_Float16>(a), static_cast<_Float16>(b)};
  return __builtin_bit_cast(uint32_t, w);
}
__device__ __forceinline__ uint32_t narrow_pair(float a, float b, BF16) {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  const b2 w = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  return __builtin_bit_cast(uint32_t, w);
}

// x * c + rot * s of two channels; rot holds rotate_half(x) at these channels.
template <typename DT>
__device__ __forceinline__ uint32_t rope_word(uint32_t x, uint32_t rot, uint32_t c, uint32_t s) {
  float xa, xb, ra, rb, ca, cb, sa, sb;
  unpack_pair<DT>(x, xa, xb);
  unpack_pair<DT>(rot, ra, rb);
  unpack_pair<DT>(c, ca, cb);
  unpack_pair<DT>(s, sa, sb);
  unpack_pair<DT>(narrow_pair(xa * ca, xb * cb, DT{}), xa, xb);
  unpack_pair<DT>(narrow_pair(ra * sa, rb * sb, DT{}), ra, rb);
  return narrow_pair(xa + ra, xb + rb, DT{});
}

}  // namespace tw
