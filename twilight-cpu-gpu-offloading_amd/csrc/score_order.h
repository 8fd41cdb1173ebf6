// The Quest score's per-channel operand: for query channel value q_d the
// page's max (q_d > 0) or min, widened exactly to fp32
// (quest_offload_cache.py:371-372, twilight_fused_quest.py:17-31).  Shared by
// the score kernels of quest.hip and the fused score + INT4 QK kernel of
// twilight.hip, so both form every product from the same operands.
#pragma once

#include "tw_common.h"

namespace tw {
namespace {

// x[i] = q[i] > 0 ? max[i] : min[i] for 8 consecutive channels of one page
// (16-byte aligned LDS rows).
__device__ __forceinline__ void select8(const uint8_t* mn, const uint8_t* mx, const float (&q)[8], float (&x)[8],
                                        F16) {
  const uint4 a = *reinterpret_cast<const uint4*>(mn);
  const uint4 b = *reinterpret_cast<const uint4*>(mx);
  const uint32_t lo[4] = {a.x, a.y, a.z, a.w}, hi[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t w = q[i] > 0.0f ? hi[i / 2] : lo[i / 2];
    x[i] = to_f32(F16{}, static_cast<uint16_t>((i & 1) ? (w >> 16) : (w & 0xffffu)));
  }
}
__device__ __forceinline__ void select8(const uint8_t* mn, const uint8_t* mx, const float (&q)[8], float (&x)[8],
                                        BF16) {
  const uint4 a = *reinterpret_cast<const uint4*>(mn);
  const uint4 b = *reinterpret_cast<const uint4*>(mx);
  const uint32_t lo[4] = {a.x, a.y, a.z, a.w}, hi[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t w = q[i] > 0.0f ? hi[i / 2] : lo[i / 2];
    x[i] = to_f32(BF16{}, static_cast<uint16_t>((i & 1) ? (w >> 16) : (w & 0xffffu)));
  }
}
__device__ __forceinline__ void select8(const uint8_t* mn, const uint8_t* mx, const float (&q)[8], float (&x)[8],
                                        F32) {
  float lo[8], hi[8];
  *reinterpret_cast<float4*>(lo) = reinterpret_cast<const float4*>(mn)[0];
  *reinterpret_cast<float4*>(lo + 4) = reinterpret_cast<const float4*>(mn)[1];
  *reinterpret_cast<float4*>(hi) = reinterpret_cast<const float4*>(mx)[0];
  *reinterpret_cast<float4*>(hi + 4) = reinterpret_cast<const float4*>(mx)[1];
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = q[i] > 0.0f ? hi[i] : lo[i];
}

// ---- the tile score of D = 128, all heads of a group in one pass (quest.hip)
//
// A block of 8 wavefronts scores a tile of 64 pages staged in LDS, lane = page.
// Wavefront w owns accumulators 4 w .. 4 w + 3 of the 32 (channels d with
// d mod 32 in that range) for every head: it reads and widens each of its
// channels' min and max once, whatever the number of heads, where a wavefront
// per head read both rows again for each.  The queries are wave-uniform and
// live in scalar registers (constant address space), so the q > 0 choice is a
// scalar mask and a head costs three vector instructions a channel (select,
// multiply, add).  At 8 heads they are more than the registers beside the rest:
// 22 scalars (25 of fp32 metadata, 10 there at 7 heads) wait in vector lanes, a
// lane read each; 8 heads, 32K, still 31.0 -> 29.3 us a layer against the
// wavefront a head.  The accumulators and their adjacent-pair tree are those of
// the 32-accumulator order: the in-lane tree covers 4, the combine the other 8.
constexpr int kScoreWaves = 8;

__device__ __forceinline__ void load4(const uint8_t* p, float (&x)[4], F16) {
  const uint2 w = *reinterpret_cast<const uint2*>(p);
  x[0] = to_f32(F16{}, static_cast<uint16_t>(w.x & 0xffffu));
  x[1] = to_f32(F16{}, static_cast<uint16_t>(w.x >> 16));
  x[2] = to_f32(F16{}, static_cast<uint16_t>(w.y & 0xffffu));
  x[3] = to_f32(F16{}, static_cast<uint16_t>(w.y >> 16));
}
__device__ __forceinline__ void load4(const uint8_t* p, float (&x)[4], BF16) {
  const uint2 w = *reinterpret_cast<const uint2*>(p);
  x[0] = to_f32(BF16{}, static_cast<uint16_t>(w.x & 0xffffu));
  x[1] = to_f32(BF16{}, static_cast<uint16_t>(w.x >> 16));
  x[2] = to_f32(BF16{}, static_cast<uint16_t>(w.y & 0xffffu));
  x[3] = to_f32(BF16{}, static_cast<uint16_t>(w.y >> 16));
}
__device__ __forceinline__ void load4(const uint8_t* p, float (&x)[4], F32) {
  *reinterpret_cast<float4*>(x) = *reinterpret_cast<const float4*>(p);
}

// The queries of two 32-channel chunks from C0 on, at the wavefront's
// residues, into scalar registers.  qg: the group's q, [R][128].  All loads go
// out together and ahead of what the wavefront waits for next: one by one at
// their uses, each is a round trip of its own (scalar loads return out of order,
// so every use waits for all of them).
template <int R>
struct ScoreQ {
  u32x4 w[2][R];
  __device__ __forceinline__ void load(const float* qg, int wave, int C0) {
    typedef uint32_t WordQuad __attribute__((ext_vector_type(4), aligned(4)));  // queries start on any word
    typedef const __attribute__((address_space(4))) WordQuad* ConstQuads;
    const ConstQuads q = (ConstQuads)(reinterpret_cast<uintptr_t>(qg));
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int r = 0; r < R; ++r) w[c][r] = q[r * 32 + 8 * (C0 + c) + wave];
    __builtin_amdgcn_sched_barrier(0);
  }
};

// Adds 32-channel chunks C0 and C0 + 1 of the wavefront's residues to acc for R
// heads.
template <typename DT, int R, int C0>
__device__ __forceinline__ void score_chunks(const uint8_t* min_row, const uint8_t* max_row, int wave,
                                             const ScoreQ<R>& q, float (&acc)[R][4]) {
  constexpr int es = static_cast<int>(sizeof(typename DT::storage));
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int d0 = 32 * (C0 + c) + 4 * wave;
    float lo[4], hi[4];
    load4(min_row + d0 * es, lo, DT{});
    load4(max_row + d0 * es, hi, DT{});
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t qb = q.w[c][r][i];
        const bool up = static_cast<int32_t>(qb) > 0;  // q > 0 on its bits (a NaN's product is a NaN either way)
        acc[r][i] = acc[r][i] + (up ? hi[i] : lo[i]) * __uint_as_float(qb);
      }
    }
  }
}

// The wavefronts' four-accumulator trees to part[(w * NR + r) * 64 + lane].
template <int NR>
__device__ __forceinline__ void score_store_parts(float* part, int wave, int lane, const float (&acc)[NR][4]) {
#pragma unroll
  for (int r = 0; r < NR; ++r)
    part[(wave * NR + r) * kWave + lane] = (acc[r][0] + acc[r][1]) + (acc[r][2] + acc[r][3]);
}
// Head r's score of page `lane` (after a barrier).
template <int NR>
__device__ __forceinline__ float score_combine(const float* part, int r, int lane) {
  float p[kScoreWaves];
#pragma unroll
  for (int w = 0; w < kScoreWaves; ++w) p[w] = part[(w * NR + r) * kWave + lane];
  return ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
}

}  // namespace
}  // namespace tw
