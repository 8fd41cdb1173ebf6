// One wavefront's view of 16 consecutive rows of 128 16-bit keys (a page, or
// 16 rows outside the pages), held in registers: the page min/max and the
// affine INT4 code of every row, bit for bit what the row-at-a-time routine
// of metadata.hip gives.
//
// Lane l holds channels 8 (l % 16) .. + 7 of rows 4 j + l / 16, j = 0 .. 3: a
// load is four whole rows, 1 KB.  Values are compared as signed 16-bit
// integers in the IEEE total order, two channels an instruction: the page
// reduces over j in the lane and over the four 16-lane groups by row swaps, a
// row over the 16 lanes of its group by DPP, its minimum and the complement of
// its maximum side by side in one register.
#pragma once

#include <type_traits>

#include "tw_common.h"

namespace tw {

typedef short i16x2 __attribute__((ext_vector_type(2)));

constexpr int kChunkRows = 16;

template <typename DT>
struct Order16;  // the total order's infinities and the canonical NaN, both halves; the least scale of the fast quotient
template <>
struct Order16<F16> {
  static constexpr uint32_t inf = 0x7c007c00u, ninf = 0x83ff83ffu, nan = 0x7e007e00u;
  static constexpr float plain_scale = 0x1p-14f;
};
template <>
struct Order16<BF16> {
  static constexpr uint32_t inf = 0x7f807f80u, ninf = 0x807f807fu, nan = 0x7fc07fc0u;
  static constexpr float plain_scale = 0x1p-60f;
};

__device__ __forceinline__ i16x2 as_pair(uint32_t x) { return __builtin_bit_cast(i16x2, x); }
__device__ __forceinline__ uint32_t as_word(i16x2 x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ uint32_t pair_min(uint32_t a, uint32_t b) {
  return as_word(__builtin_elementwise_min(as_pair(a), as_pair(b)));
}
__device__ __forceinline__ uint32_t pair_max(uint32_t a, uint32_t b) {
  return as_word(__builtin_elementwise_max(as_pair(a), as_pair(b)));
}
// Sign-magnitude bits to two's complement order and back (an involution).
__device__ __forceinline__ uint32_t pair_order(uint32_t x) {
  return x ^ (as_word(as_pair(x) >> static_cast<short>(15)) & 0x7fff7fffu);
}
__device__ __forceinline__ uint32_t swap_halves(uint32_t x) { return __builtin_amdgcn_alignbit(x, x, 16); }

// Ordered min/max pair to storage bits, NaN (outside the infinities) canonical.
template <typename DT>
__device__ __forceinline__ void pair_finish(uint32_t& mn, uint32_t& mx) {
  const i16x2 over = as_pair(pair_max(mx, Order16<DT>::inf)) - as_pair(Order16<DT>::inf);
  const i16x2 under = as_pair(Order16<DT>::ninf) - as_pair(pair_min(mn, Order16<DT>::ninf));
  const i16x2 zero = {0, 0};
  const uint32_t nan = as_word((zero - (over | under)) >> static_cast<short>(15));
  mn = (pair_order(mn) & ~nan) | (Order16<DT>::nan & nan);
  mx = (pair_order(mx) & ~nan) | (Order16<DT>::nan & nan);
}

template <typename DT>
__device__ __forceinline__ void unpack_pair(uint32_t w, float& a, float& b) {
  a = to_f32(DT{}, static_cast<uint16_t>(w & 0xffffu));
  b = to_f32(DT{}, static_cast<uint16_t>(w >> 16));
}

// The value that lane J of this lane's 16-lane group holds.
template <int J>
__device__ __forceinline__ float row_value(float x) {
  constexpr int kDppRowNewBcast = 0x150;
  return __uint_as_float(dpp_u32<kDppRowNewBcast + J>(__float_as_uint(x)));
}

// Page min/max of the chunk's 16 rows: mn/mx_row point at the page's rows of
// page_min / page_max (the first 16 lanes store the one, the next the other).
template <typename DT>
__device__ __forceinline__ void chunk_page_minmax(const u32x4 (&x)[4], int lane, uint16_t* __restrict__ mn_row,
                                                  uint16_t* __restrict__ mx_row) {
  u32x4 out;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    uint32_t mn = pair_order(x[0][c]), mx = mn;
#pragma unroll
    for (int j = 1; j < 4; ++j) {
      const uint32_t s = pair_order(x[j][c]);
      mn = pair_min(mn, s);
      mx = pair_max(mx, s);
    }
    auto a = __builtin_amdgcn_permlane16_swap(mn, mn, false, false);
    mn = pair_min(a[0], a[1]);
    a = __builtin_amdgcn_permlane32_swap(mn, mn, false, false);
    mn = pair_min(a[0], a[1]);
    a = __builtin_amdgcn_permlane16_swap(mx, mx, false, false);
    mx = pair_max(a[0], a[1]);
    a = __builtin_amdgcn_permlane32_swap(mx, mx, false, false);
    mx = pair_max(a[0], a[1]);
    pair_finish<DT>(mn, mx);
    out[c] = lane < 16 ? mn : mx;
  }
  if (lane < 32) *reinterpret_cast<u32x4*>((lane < 16 ? mn_row : mx_row) + 8 * (lane % 16)) = out;
}

// INT4 codes, scale and minimum of the chunk's first `rows` rows, to row 0 of
// the given arrays (packed rows are 64 bytes).
//
// code = rint((k - min) / scale) takes the correctly rounded quotient.  With
// y = 1 / scale correctly rounded, q = x y and the exact remainder
// e = x - q scale (one fma), q + e y is that quotient: scale has at most 11
// significant bits, so x / scale is never a midpoint of two floats and stays
// 2^-12 ulp away from every one, and e y is within 2^-23 ulp of e / scale
// (the division refinement of Markstein, IBM J. Res. Dev. 34, 1990).  A normal
// scale is within 2^-8 of range / 15, so no quotient passes 15.2 and the clamp
// has nothing to do.  Scales below the normal range or outside 2^+-60, where a
// step could leave it, and rows with an infinity or a NaN take the division
// and the clamp.
template <typename DT>
__device__ __forceinline__ void chunk_int4(const u32x4 (&x)[4], int rows, int lane, uint8_t* __restrict__ packed,
                                           uint16_t* __restrict__ scale, uint16_t* __restrict__ minimum) {
  const int unit = lane % 16, quad = lane / 16;
  // lane `unit` of a group forms the scale of its row unit % 4 (all 16 rows of
  // the chunk at once), which the group's lanes then read from it
  uint32_t mine = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t s0 = pair_order(x[j][0]), s1 = pair_order(x[j][1]), s2 = pair_order(x[j][2]),
                   s3 = pair_order(x[j][3]);
    uint32_t lo = pair_min(pair_min(s0, s1), pair_min(s2, s3));
    uint32_t hi = ~pair_max(pair_max(s0, s1), pair_max(s2, s3));
    lo = pair_min(lo, swap_halves(lo));
    hi = pair_min(hi, swap_halves(hi));
    uint32_t both = (lo & 0xffffu) | (hi & 0xffff0000u);  // the minimum, and the complement of the maximum
    both = pair_min(both, dpp_u32<kDppQuadXor1>(both));
    both = pair_min(both, dpp_u32<kDppQuadXor2>(both));
    both = pair_min(both, dpp_u32<kDppRowHalfMirror>(both));
    both = pair_min(both, dpp_u32<kDppRowMirror>(both));
    mine = unit % 4 == j ? both : mine;
  }
  uint32_t mnb = mine & 0xffffu, mxb = ~mine >> 16;
  pair_finish<DT>(mnb, mxb);
  const float mnf = to_f32(DT{}, static_cast<uint16_t>(mnb));
  const uint16_t sc = from_f32(DT{}, int4_scale<DT>(mnf, to_f32(DT{}, static_cast<uint16_t>(mxb))));
  const float sf = to_f32(DT{}, sc);
  const int row_mine = 4 * unit + quad;  // lanes 0 .. 3 of each group hold the 16 rows between them
  if (unit < 4 && row_mine < rows) {
    scale[row_mine] = sc;
    minimum[row_mine] = static_cast<uint16_t>(mnb);
  }
  u32x4 code;
  if (__all(sf >= Order16<DT>::plain_scale && sf <= 0x1p60f)) {  // false for NaN
    const float y = 1.0f / sf;
    auto quotients = [&](auto jc) {
      constexpr int j = decltype(jc)::value;
      const float mn_j = row_value<j>(mnf), sf_j = row_value<j>(sf), y_j = row_value<j>(y);
      float c[8];
#pragma unroll
      for (int p = 0; p < 4; ++p) unpack_pair<DT>(x[j][p], c[2 * p], c[2 * p + 1]);
#pragma unroll
      for (int p = 0; p < 8; ++p) {
        const float d = c[p] - mn_j;
        const float q = d * y_j;
        c[p] = rintf(__builtin_fmaf(__builtin_fmaf(-q, sf_j, d), y_j, q));
      }
      // four codes a float, exact below 2^16
      const float w0 = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(c[3], 16.0f, c[2]), 16.0f, c[1]), 16.0f, c[0]);
      const float w1 = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(c[7], 16.0f, c[6]), 16.0f, c[5]), 16.0f, c[4]);
      code[j] = static_cast<uint32_t>(w0) | (static_cast<uint32_t>(w1) << 16);
    };
    quotients(std::integral_constant<int, 0>{});
    quotients(std::integral_constant<int, 1>{});
    quotients(std::integral_constant<int, 2>{});
    quotients(std::integral_constant<int, 3>{});
  } else {
    const float mn_rows[4] = {row_value<0>(mnf), row_value<1>(mnf), row_value<2>(mnf), row_value<3>(mnf)};
    const float sf_rows[4] = {row_value<0>(sf), row_value<1>(sf), row_value<2>(sf), row_value<3>(sf)};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t w = 0;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        float a, b;
        unpack_pair<DT>(x[j][p], a, b);
        w |= (int4_code(a, mn_rows[j], sf_rows[j]) | (int4_code(b, mn_rows[j], sf_rows[j]) << 4)) << (8 * p);
      }
      code[j] = w;
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (4 * j + quad < rows) reinterpret_cast<uint32_t*>(packed)[(4 * j + quad) * 16 + unit] = code[j];
}

}  // namespace tw
