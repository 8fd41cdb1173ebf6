// Dense causal attention of a prompt on the matrix cores (head_dim 128,
// fp16 / bf16): every query row attends to the key rows at or before it, the
// attention the reference's prefill runs (mp.py:475-482).
//
// A wavefront owns 32 query rows of one query head; its block walks the key rows
// in tiles of 64, the next tile's loads in flight (registers, then the other LDS
// buffer) while the current one is computed.  The products are taken transposed,
// so that a query stays in one lane column from the scores to the output:
//
//   S^T = K Q^T    v_mfma_f32_32x32x16: A = 32 key rows, B = 32 query rows
//   O^T += V^T P^T the same shape: A = 32 channels, B = the 32 query columns
//
// In the 32 x 32 result lane l holds query l % 32, registers the keys
// (i % 4) + 8 (i / 4) + 4 (l / 32): a query's maximum and sum are in-lane
// reductions plus one exchange of the two lane halves, its rescaling factor
// is a per-lane scalar, and registers 8 t .. 8 t + 7, rounded to 16 bits,
// are the B fragment of the second product over keys 16 t .. 16 t + 15 --
// the contraction takes that key order on both sides, the V^T fragment being
// two transposing LDS reads of 4 keys each.
//
// Bound: the matrix cores and, beside them, the vector unit (a score costs a
// multiply-add, an exponential, a sum, half a conversion and half a maximum: as
// many issue cycles as its share of the products).  8 KV heads of 4 query heads,
// bf16: 32768 rows 8.1 ms, 1090 TFLOP/s of the causal half (library products of
// 8192^3 and 16384^3 reach 1317 and 1587 here), against 137 ms for the score tiles
// through batched products, mask and softmax; 2048 rows 62 us against 1.0 ms.  The
// matrix cores are busy 53% of that time, at 1.9 GHz under this load.  Two 32-row
// query tiles a wavefront (half the LDS reads a product, one wavefront a SIMD)
// took 10.5 ms; wavefronts 4 .. 7 a product phase behind 0 .. 3, with a barrier
// a phase, 8.7 ms.
//
// The running maximum moves only when a score passes it by more than 2^8 of
// weight, the condition that FlashAttention-4 rescales under.  What that, the fp32
// shift of the exponents and the division at the end could get wrong at the ends of
// the operands' range is taken care of at its place below, for 0 to 1% of the time
// (2048 rows 61.6 -> 60.6 us in bf16, 62.5 -> 63.5 in fp16; 32768 rows 8.20 -> 8.18 ms).
#pragma clang fp contract(off)

#include <limits>
#include <type_traits>

#include "rope.h"
#include "tw_common.h"

namespace tw {
namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kHead = 128;                 // channels
constexpr int kKeys = 64;                  // key rows of a tile
constexpr int kQ = 32;                     // query rows of a wavefront
constexpr int kRowUnits = kHead / 8;       // 16-byte units of a row

struct PrefillArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* out;
  int64_t q_row, q_head, k_row, k_head, v_row, v_head, out_row;  // in elements
  const uint16_t* cos;  // nullable: q is rotated by row s of cos / sin as it is loaded
  const uint16_t* sin;
  int64_t cos_row, sin_row;
  int S, G, R, tiles;
  float scale_log2;
  // Raw scores past the running maximum by less than this (8 / scale_log2) are
  // taken without moving it: their weights stay below 2^8, and the accumulators
  // are not rescaled on every tile.  Finite for any scale, so that a first maximum,
  // up from -inf, is always taken.
  float slack;
};

template <typename DT>
struct Frag;
template <>
struct Frag<F16> {
  typedef f16x8 type;
  typedef _Float16 quad __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ f32x16 mfma(type a, type b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ auto narrow(float x) { return static_cast<_Float16>(x); }
};
template <>
struct Frag<BF16> {
  typedef bf16x8 type;
  typedef __bf16 quad __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ f32x16 mfma(type a, type b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ auto narrow(float x) { return static_cast<__bf16>(x); }
};

// LDS slot (in 16-byte units) of unit u of tile row r.  A row is 256 bytes, one
// turn of the 64 banks: the units of 16 consecutive rows go to 16 different
// slots (a fragment read of K: 16 rows, one unit), and the four units of 4
// consecutive rows to different slot quadruples (the transposing reads of V).
__device__ __forceinline__ int slot(int r, int u) {
  return r * kRowUnits + (u ^ (((r & 3) << 2) | ((r >> 2) & 3)));
}

// (v_max3_f32; fmaxf would first quiet every operand, an instruction each)
__device__ __forceinline__ float max3(float a, float b, float c) {
  const float inf = __builtin_inff();
  return __builtin_amdgcn_fmed3f(__builtin_amdgcn_fmed3f(a, b, inf), c, inf);
}
__device__ __forceinline__ float both_halves_max(float x) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
}
__device__ __forceinline__ float both_halves_sum(float x) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(h[0]) + __uint_as_float(h[1]);
}

// A weight is 2^(x unit - shift) of a score x: unit = scale_log2 and shift =
// m scale_log2 against the row's maximum m, one multiply-add a score.  The shift
// is rounded, by up to half a unit in its last place for every key of the row
// alike: 2^-11 at kNearShift, no more than the scores themselves, but in the end
// hundreds of powers of two.  Past it the scores become (x - m) scale_log2 first,
// 0 for the maximum; the bound leaves the largest scores that fp16 holds (65504 /
// sqrt(128), a shift of 8353) to the multiply-add.  8192 rows of 32 heads, bf16: 521
// us with shifts up to the bound, 600 past it.
//
// A row whose keys so far all score -inf has no maximum yet: against 0 those keys
// weigh 0 (-inf against -inf is a NaN that would stay in the row's sums).
constexpr float kNearShift = 16384.0f;
struct Exponents {
  float unit, shift;
  __device__ __forceinline__ Exponents(f32x16 (&sc)[2], float m, float scale_log2, float drop)
      : unit(scale_log2), shift(m * scale_log2 + drop) {
    if (__any(!(fabsf(shift) <= kNearShift))) {  // hardly ever taken
      const float against = m == -__builtin_inff() ? 0.0f : m;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[kb][i] = (sc[kb][i] - against) * scale_log2;
      unit = 1.0f;
      shift = drop;
    }
  }
};

// The powers of two by which a block's second pass lowers its weights.  A weight is
// below 2^8 and their sum below 2^8 S, so V past the largest float over that may
// leave the accumulators' range though the row, their quotient, is in it; lowered,
// |o| stays below half the largest |v|.  (Lowered in every pass, the smallest V
// would fall below the range instead.  fp16 values have no such size.)
__device__ __forceinline__ float second_pass_drop(int S) { return static_cast<float>(9 + 32 - __clz(S)); }
// Whether some wavefront of the block has `over`; flag: a word of LDS, 0 since the block's start.
__device__ __forceinline__ bool block_any(bool over, int* flag) {
  if (__any(over) && lane_id() == 0) *flag = 1;
  __syncthreads();
  return *flag != 0;
}

// Q^T fragments of query row `row`, rotated if the tables are given.
template <typename DT>
__device__ __forceinline__ void load_queries(const PrefillArgs& a, int head, int row, int half,
                                             typename Frag<DT>::type (&qf)[8]) {
  typedef typename Frag<DT>::type frag;
  const int S = a.S;
  const uint16_t* qp = a.q + head * a.q_head + static_cast<int64_t>(row < S ? row : S - 1) * a.q_row + 8 * half;
#pragma unroll
  for (int s = 0; s < 8; ++s) qf[s] = __builtin_bit_cast(frag, *reinterpret_cast<const u32x4*>(qp + 16 * s));
  if (a.cos != nullptr) {
    // a rotation pair is 64 channels apart: fragments s and s + 4 of the lane
    const int64_t at = row < S ? row : S - 1;
    const uint16_t* cp = a.cos + at * a.cos_row + 8 * half;
    const uint16_t* sp = a.sin + at * a.sin_row + 8 * half;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const u32x4 x = __builtin_bit_cast(u32x4, qf[s]), y = __builtin_bit_cast(u32x4, qf[s + 4]);
      const u32x4 cx = *reinterpret_cast<const u32x4*>(cp + 16 * s);
      const u32x4 cy = *reinterpret_cast<const u32x4*>(cp + 16 * s + 64);
      const u32x4 sx = *reinterpret_cast<const u32x4*>(sp + 16 * s);
      const u32x4 sy = *reinterpret_cast<const u32x4*>(sp + 16 * s + 64);
      u32x4 rx, ry;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        rx[p] = rope_word<DT>(x[p], y[p] ^ 0x80008000u, cx[p], sx[p]);
        ry[p] = rope_word<DT>(y[p], x[p], cy[p], sy[p]);
      }
      qf[s] = __builtin_bit_cast(frag, rx);
      qf[s + 4] = __builtin_bit_cast(frag, ry);
    }
  }
}

// Stores the lane's half of its row, o / l, if `store`; whether it held an infinity or a NaN (bf16 only).
template <typename DT>
__device__ __forceinline__ bool store_output(const PrefillArgs& a, int row, int head, int half, bool store,
                                             const f32x16 (&o)[4], float l) {
  const float inv = 1.0f / both_halves_sum(l);
  if (!store) return false;
  float bad[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // four chains of sums of 0 x
  uint16_t* p = a.out + static_cast<int64_t>(row) * a.out_row + head * kHead + 4 * half;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      typename Frag<DT>::quad w;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float x = o[c][4 * i + j] * inv;
        if constexpr (std::is_same_v<DT, BF16>) bad[j] = __builtin_fmaf(x, 0.0f, bad[j]);
        w[j] = Frag<DT>::narrow(x);
      }
      *reinterpret_cast<typename Frag<DT>::quad*>(p + 32 * c + 8 * i) = w;
    }
  return (bad[0] + bad[1]) + (bad[2] + bad[3]) != 0.0f;  // a NaN
}

// Query rows q_block .. + 32 NW - 1 of a head by a block of NW wavefronts, each
// taking a tile's scores, weights and values in turn.  Stores the lanes' rows with
// `store`, weights lowered by 2^drop; whether the lane's held an infinity or a NaN.
template <typename DT, int NW, bool AGAIN>
__device__ __forceinline__ bool attend(const PrefillArgs& a, u32x4* s_tiles, int g, int head, int q_block, bool store,
                                       float drop) {
  typedef typename Frag<DT>::type frag;
  constexpr int kLoads = kKeys * kRowUnits / (NW * kWave);  // 16-byte units a thread stages, for K and for V
  u32x4* const s_k = s_tiles;  // tiles of even and odd index
  u32x4* const s_v = s_tiles + 2 * kKeys * kRowUnits;

  int tid = threadIdx.x;
  if constexpr (AGAIN) asm volatile("" : "+v"(tid));  // a second pass forms its addresses anew: kept over the first, they spill
  const int lane = tid % kWave, wave = wave_uniform(tid / kWave);
  const int col = lane % 32, half = lane / 32;
  const int q0 = q_block + wave * kQ;
  const int S = a.S;

  const uint16_t* kg = a.k + g * a.k_head;
  const uint16_t* vg = a.v + g * a.v_head;

  const int row = q0 + col;
  frag qf[8];
  load_queries<DT>(a, head, row, half, qf);

  const int last_row = q_block + NW * kQ - 1;
  const int n_keys = (last_row < S ? last_row : S - 1) + 1;
  const int n_tiles = (n_keys + kKeys - 1) / kKeys;

  const int st_row = tid / kRowUnits, st_unit = tid % kRowUnits;
  u32x4 rk[kLoads], rv[kLoads];
#define LOAD_TILE(t)                                                                                       \
  _Pragma("unroll") for (int i = 0; i < kLoads; ++i) {                                                     \
    int r = (t) * kKeys + st_row + i * (kKeys / kLoads);                                                   \
    r = r < S ? r : S - 1; /* past the prompt: a real row, whose keys are masked */                        \
    rk[i] = *reinterpret_cast<const u32x4*>(kg + static_cast<int64_t>(r) * a.k_row + 8 * st_unit);         \
    rv[i] = *reinterpret_cast<const u32x4*>(vg + static_cast<int64_t>(r) * a.v_row + 8 * st_unit);         \
  }
#define STORE_TILE(b)                                                                                      \
  _Pragma("unroll") for (int i = 0; i < kLoads; ++i) {                                                     \
    const int at = slot(st_row + i * (kKeys / kLoads), st_unit);                                           \
    s_k[(b) * kKeys * kRowUnits + at] = rk[i];                                                             \
    s_v[(b) * kKeys * kRowUnits + at] = rv[i];                                                             \
  }

  f32x16 o[4];
  float m = -__builtin_inff(), l = 0.0f;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[c][i] = 0.0f;

  LOAD_TILE(0)
  STORE_TILE(0)
  for (int t = 0; t < n_tiles; ++t) {
    const int b = t & 1;
    __syncthreads();
    LOAD_TILE(t + 1)                       // past the last tile: clamped rows that no tile reads
    const int k0 = t * kKeys;
    if (k0 <= q0 + kQ - 1) {               // the wavefront has rows that see this tile
      f32x16 sc[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[kb][i] = 0.0f;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          const frag kf = __builtin_bit_cast(frag, s_k[b * kKeys * kRowUnits + slot(32 * kb + col, 2 * s + half)]);
          sc[kb] = Frag<DT>::mfma(kf, qf[s], sc[kb]);
        }
      }
      if (k0 + kKeys - 1 > q0) {           // keys past the limit are in the row's future
        const int limit = row - k0 - 4 * half;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (32 * kb + (i % 4) + 8 * (i / 4) > limit) sc[kb][i] = -__builtin_inff();
      }
      float mx = max3(sc[0][0], sc[1][0], sc[0][1]), mx1 = max3(sc[1][1], sc[0][2], sc[1][2]);
#pragma unroll
      for (int i = 3; i < 15; i += 2) {
        mx = max3(mx, sc[0][i], sc[1][i]);
        mx1 = max3(mx1, sc[0][i + 1], sc[1][i + 1]);
      }
      mx = fmaxf(max3(mx, sc[0][15], sc[1][15]), mx1);
      mx = both_halves_max(mx);
      if (__any(mx - m > a.slack)) {
        const float mn = fmaxf(m, mx);
        // an unmoved maximum keeps its sums (-inf - -inf is not a factor)
        const float f = m == mn ? 1.0f : __builtin_amdgcn_exp2f((m - mn) * a.scale_log2);
        m = mn;
        l *= f;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[c][i] *= f;
      }
      const Exponents ex(sc, m, a.scale_log2, drop);
      float sum = 0.0f;
      frag pf[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        frag w;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float p =
              __builtin_amdgcn_exp2f(__builtin_fmaf(sc[ks / 2][8 * (ks % 2) + i], ex.unit, -ex.shift));
          sum += p;
          w[i] = Frag<DT>::narrow(p);
        }
        pf[ks] = w;
      }
      l += sum;
      // V^T fragments: lane i of a 16-lane group names key row i / 4 and channels 4 (i % 4) .. + 3
      const int vrow = 4 * half + (lane % 16) / 4;
      const int vch = 16 * ((lane / 16) % 2) + 4 * (lane % 4);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          s16x8 vf;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int r = 16 * ks + 8 * h + vrow, ch = 32 * c + vch;
            const uint2* p = reinterpret_cast<const uint2*>(&s_v[b * kKeys * kRowUnits + slot(r, ch / 8)]) + (ch % 8) / 4;
            const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) s16x4*)(reinterpret_cast<uintptr_t>(p)));
#pragma unroll
            for (int j = 0; j < 4; ++j) vf[4 * h + j] = x[j];
          }
          o[c] = Frag<DT>::mfma(__builtin_bit_cast(frag, vf), pf[ks], o[c]);
        }
      }
    }
    STORE_TILE(b ^ 1)
  }

#undef LOAD_TILE
#undef STORE_TILE

  return store_output<DT>(a, row, head, half, store, o, l);
}

// Blocks of 4 wavefronts; two blocks share a CU and drift apart.
template <typename DT>
__global__ __launch_bounds__(4 * kWave, 2) void prefill_attn_kernel(PrefillArgs a) {
  constexpr int NW = 4;
  __shared__ u32x4 s_tiles[4 * kKeys * kRowUnits];
  __shared__ int s_over;
  if (threadIdx.x == 0) s_over = 0;  // (ahead of the first of many barriers)
  // group-minor, the longest query tiles first
  const int g = blockIdx.x % a.G;
  const int rest = blockIdx.x / a.G;
  const int head = g * a.R + rest % a.R;
  const int q_block = (a.tiles - 1 - rest / a.R) * NW * kQ;
  const int row = q_block + static_cast<int>(threadIdx.x) / kWave * kQ + static_cast<int>(threadIdx.x) % kQ;
  const bool over = attend<DT, NW, false>(a, s_tiles, g, head, q_block, row < a.S, 0.0f);
  if constexpr (std::is_same_v<DT, BF16>)
    if (block_any(over, &s_over)) attend<DT, NW, true>(a, s_tiles, g, head, q_block, over, second_pass_drop(a.S));
}

// Blocks of 8 wavefronts, with the three streams of neighbouring tiles
// interleaved in each wavefront.  Against attend() with blocks of 8 (32768 rows of
// 32 heads): 17.5 M cycles and 8.4 ms, 15.9 M and 8.1 ms.  Of the 256 registers a
// wavefront can have, 74 spill (184 bytes a lane), none of them inside the loop over
// the tiles: a wavefront with an odd number of tiles stores and reloads them around
// its last.
constexpr int kWideWaves = 8;
constexpr int kWideThreads = kWideWaves * kWave;
constexpr int kWideRows = kWideWaves * kQ;                      // query rows of a block
template <typename DT>
__global__ __launch_bounds__(kWideThreads, 2) void prefill_attn_wide(PrefillArgs a) {
  typedef typename Frag<DT>::type frag;
  __shared__ u32x4 s_tiles[4 * kKeys * kRowUnits];  // K tiles of even and odd index, then V's
  __shared__ int s_over;
  if (threadIdx.x == 0) s_over = 0;  // (ahead of the first of many barriers)

  const int tid = threadIdx.x, lane = tid % kWave, wave = wave_uniform(tid / kWave);
  const int col = lane % 32, half = lane / 32;
  // group-minor, the longest query tiles first
  const int g = blockIdx.x % a.G;
  const int rest = blockIdx.x / a.G;
  const int head = g * a.R + rest % a.R;
  const int qt = a.tiles - 1 - rest / a.R;
  const int q_block = qt * kWideRows;
  const int q0 = q_block + wave * kQ;
  const int S = a.S;

  const uint16_t* kg = a.k + g * a.k_head;
  const uint16_t* vg = a.v + g * a.v_head;

  const int row = q0 + col;
  frag qf[8];
  load_queries<DT>(a, head, row, half, qf);

  const int last_row = q_block + kWideRows - 1;
  const int n_keys = (last_row < S ? last_row : S - 1) + 1;
  const int n_tiles = (n_keys + kKeys - 1) / kKeys;

  // tiles that some row of the wavefront sees
  const int w_tiles = (q0 + kQ - 1) / kKeys + 1 < n_tiles ? (q0 + kQ - 1) / kKeys + 1 : n_tiles;

  // staging: the tile's base is wave-uniform, a thread's rows are 32-bit byte offsets from it
  const int st_row = tid / kRowUnits, st_unit = tid % kRowUnits;
  const int all_tiles = (S + kKeys - 1) / kKeys;
  constexpr int kLoads = kKeys * kRowUnits / kWideThreads;  // 16-byte units a thread stages, for K and for V
  u32x4 rk[kLoads], rv[kLoads];
  auto load_rows = [&](const uint16_t* base, int64_t stride, int t, u32x4 (&x)[kLoads]) {
    // past the prompt: real rows, whose keys are masked or whose tile is not read
    const int tile = t < all_tiles ? t : all_tiles - 1;
    const char* p = reinterpret_cast<const char*>(base + static_cast<int64_t>(tile) * kKeys * stride);
    const int last = S - 1 - tile * kKeys;
    const uint32_t bytes = static_cast<uint32_t>(stride) * 2, end = (last < kKeys ? last : kKeys) * bytes;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      uint32_t at = static_cast<uint32_t>(st_row + i * (kKeys / kLoads)) * bytes;
      at = at < end ? at : end;
      x[i] = *reinterpret_cast<const u32x4*>(p + (at + 16u * st_unit));
    }
  };
  const int st_at = slot(st_row, st_unit);  // rows kKeys / kLoads apart share the swizzle
  static_assert((kKeys / kLoads) % 16 == 0, "the swizzle repeats every 16 rows");
  auto store_rows = [&](int tile, const u32x4 (&x)[kLoads]) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) s_tiles[st_at + (tile * kKeys + i * (kKeys / kLoads)) * kRowUnits] = x[i];
  };

  f32x16 o[4], sc[2];
  frag p_even[4], p_odd[4];
  const f32x16 zero = {0.0f};  // the first product of every chain adds to it (as an operand, in no register)
  float m = -__builtin_inff(), l = 0.0f;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[c][i] = 0.0f;

  // fragment addresses in the first tile; the tile and the rest of the row index are immediates
  typedef __attribute__((address_space(3))) char* lds_ptr;
  const lds_ptr lds = (lds_ptr)(reinterpret_cast<uintptr_t>(s_tiles));
  lds_ptr k_at[8], v_at[4][2];
#pragma unroll
  for (int s = 0; s < 8; ++s) k_at[s] = lds + 16 * slot(col, 2 * s + half);
  // V^T fragments: lane i of a 16-lane group names key row i / 4 and channels 4 (i % 4) .. + 3
  const int vrow = 4 * half + (lane % 16) / 4;
  const int vch = 16 * ((lane / 16) % 2) + 4 * (lane % 4);
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int h = 0; h < 2; ++h) v_at[c][h] = lds + 16 * slot(8 * h + vrow, (32 * c + vch) / 8) + 8 * ((vch % 8) / 4);
  constexpr int kTileBytes = kKeys * 256;
  auto key_frag = [&](int tile, int j) {  // K fragment j of 16: 32 keys x 16 channels
    return *(__attribute__((address_space(3))) frag*)(k_at[j % 8] + tile * kTileBytes + (j / 8) * 32 * 256);
  };
  auto value_frag = [&](int tile, int j) {  // V^T fragment j of 16: 16 keys x 32 channels
    s16x8 x;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const s16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(
          v_at[j % 4][h] + tile * kTileBytes + (j / 4) * 16 * 256));
#pragma unroll
      for (int i = 0; i < 4; ++i) x[4 * h + i] = y[i];
    }
    return __builtin_bit_cast(frag, x);
  };
  auto stage = [&](int t, int parity) {  // iteration t's share of the tiles to come
    store_rows(parity, rk);
    store_rows(2 + parity, rv);
    load_rows(kg, a.k_row, t + 3, rk);
    load_rows(vg, a.v_row, t + 1, rv);
  };

  // Iteration t takes the weights of tile t on the vector unit while the
  // matrix cores form the scores of tile t + 1 and then the values of tile
  // t - 1.  The three streams are independent and interleaved by hand, a
  // matrix instruction and a few vector instructions a step (a wavefront's
  // products and exponentials one after the other leave either unit idle half
  // the time, with two wavefronts on the SIMD too).  It stores K tile t + 2 and
  // V tile t over K t and V t - 2, which iteration t - 1 read last.  LAST: the
  // tile holds keys in the future of some row -- the last of the wavefront's
  // tiles, and no other.
  auto iteration = [&](int t, auto parity, auto first, auto last, const frag (&pf)[4], frag (&pn)[4]) __attribute__((always_inline)) {
    constexpr int PAR = decltype(parity)::value;  // of t
    constexpr bool FIRST = decltype(first)::value, LAST = decltype(last)::value;
    constexpr int kAhead = 3;  // steps between a fragment's LDS read and its use
    constexpr int kMaxSteps = 4;
    // first weight of step j: scores 0 .. 15 before step 16, from which their registers take the next tile's, the
    // others before step 24
    auto exp_begin = [](int j) { return j <= 16 ? (j - kMaxSteps - 1) * 16 / (15 - kMaxSteps) : j < 24 ? 2 * j - 16 : 32; };
    frag ring[kAhead + 1];
    auto fetch = [&](int j) {
      if (j < 16) {
        if constexpr (!FIRST) ring[j % (kAhead + 1)] = value_frag(2 + (PAR ^ 1), j);
      } else if (j < 32) {
        if constexpr (!LAST) ring[j % (kAhead + 1)] = key_frag(PAR ^ 1, j - 16);
      }
    };
#pragma unroll
    for (int j = 0; j < kAhead; ++j) fetch(j);
    if constexpr (LAST) {
      const int limit = row - t * kKeys - 4 * half;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (32 * kb + (i % 4) + 8 * (i / 4) > limit) sc[kb][i] = -__builtin_inff();
    }
    float mx = -__builtin_inff(), f = 1.0f, unit = 0.0f, shift = 0.0f, sum = 0.0f, p0 = 0.0f;
    bool moved = false;
    uint32_t pw[16];
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      __builtin_amdgcn_sched_barrier(0);
      fetch(j + kAhead);
      if (j < 16) {
        if constexpr (!FIRST) o[j % 4] = Frag<DT>::mfma(ring[j % (kAhead + 1)], pf[j / 4], o[j % 4]);
      } else {
        if constexpr (!LAST)
          sc[j / 8 - 2] = Frag<DT>::mfma(ring[j % (kAhead + 1)], qf[j % 8], j % 8 == 0 ? zero : sc[j / 8 - 2]);
      }
      if (j < kMaxSteps) {
#pragma unroll
        for (int i = 4 * j; i < 4 * j + 4; ++i) mx = max3(mx, sc[0][i], sc[1][i]);
      } else if (j == kMaxSteps) {
        mx = both_halves_max(mx);
        moved = __any(mx - m > a.slack);
        const float mn = moved ? fmaxf(m, mx) : m;
        // an unmoved maximum keeps its sums (-inf - -inf is not a factor)
        f = m == mn ? 1.0f : __builtin_amdgcn_exp2f((m - mn) * a.scale_log2);
        m = mn;
        const Exponents ex(sc, m, a.scale_log2, 0.0f);
        unit = ex.unit, shift = ex.shift;
      } else {
#pragma unroll
        for (int i = exp_begin(j); i < exp_begin(j + 1); ++i) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i / 16][i % 16], unit, -shift));
          sum += p;
          if (i % 2 == 0)
            p0 = p;
          else
            pw[i / 2] = narrow_pair(p0, p, DT{});
          // (formed here, not where they are used after the branch below)
          if (i % 2 == 1) asm volatile("" : "+v"(pw[i / 2]), "+v"(sum));
        }
      }
      if (j == 1) stage(t, PAR);
    }
    __builtin_amdgcn_sched_barrier(0);
    l = l * f + sum;
    if (moved) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[c][i] *= f;
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const u32x4 w = {pw[4 * ks], pw[4 * ks + 1], pw[4 * ks + 2], pw[4 * ks + 3]};
      pn[ks] = __builtin_bit_cast(frag, w);
    }
  };

  load_rows(kg, a.k_row, 0, rk);
  store_rows(0, rk);
  load_rows(kg, a.k_row, 1, rk);
  store_rows(1, rk);
  load_rows(kg, a.k_row, 2, rk);
  load_rows(vg, a.v_row, 0, rv);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 16; ++j)
    sc[j / 8] = Frag<DT>::mfma(key_frag(0, j), qf[j % 8], j % 8 == 0 ? zero : sc[j / 8]);
  __syncthreads();  // iteration 0 stores over K tile 0
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  // an even iteration reads p_odd and leaves p_even
  if (w_tiles == 1)
    iteration(0, even, yes, yes, p_odd, p_even);
  else
    iteration(0, even, yes, no, p_odd, p_even);
  __syncthreads();
  int t = 1;
  for (; t + 1 < w_tiles - 1; t += 2) {
    iteration(t, odd, no, no, p_even, p_odd);
    __syncthreads();
    iteration(t + 1, even, no, no, p_odd, p_even);
    __syncthreads();
  }
  if (t < w_tiles - 1) {
    iteration(t, odd, no, no, p_even, p_odd);
    __syncthreads();
    ++t;
  }
  auto finish = [&](int tile, const frag (&pf)[4]) {
#pragma unroll
    for (int j = 0; j < 16; ++j) o[j % 4] = Frag<DT>::mfma(value_frag(tile, j), pf[j / 4], o[j % 4]);
  };
  if (w_tiles % 2 != 0) {  // the last tile's index is even
    if (w_tiles > 1) {
      iteration(t, even, no, yes, p_odd, p_even);
      __syncthreads();
    }
    finish(2, p_even);
  } else {
    iteration(t, odd, no, yes, p_even, p_odd);
    __syncthreads();
    finish(3, p_odd);
  }
  for (t = w_tiles; t < n_tiles; ++t) {  // the block's later wavefronts go on
    stage(t, t & 1);
    __syncthreads();
  }

  const bool over = store_output<DT>(a, row, head, half, row < S, o, l);
  if constexpr (std::is_same_v<DT, BF16>)
    if (block_any(over, &s_over)) attend<DT, kWideWaves, true>(a, s_tiles, g, head, q_block, over, second_pass_drop(S));
}

constexpr int kWideBlocks = 512;

// The wide kernel from two blocks a CU on; with fewer, blocks of half the rows
// balance better, and two of them on a CU overlap by themselves.  The attention
// alone, blocks of 128 rows against wide ones, bf16: 2048 rows of 32 heads (256
// wide blocks) 62 against 73 us, 3072 (384) 100 and 104, 3584 (448) 136 and 126,
// 4096 (512) 171 and 156, 5120 (640) 242 and 246, 8192 (1024) 587 and 546, 32768
// 9.04 and 8.06 ms; 6000 of 16 (384) 172 and 177, 8192 of 28 (896) 521 and 491.  (At
// 448 the wide ones are already ahead.)
template <typename DT>
int launch(PrefillArgs a, hipStream_t s) {
  const int heads = a.G * a.R;
  const int wide = (a.S + kWideRows - 1) / kWideRows;
  const int64_t far = 1 << 24;  // the wide kernel's offsets inside a tile are 32-bit
  if (static_cast<int64_t>(wide) * heads >= kWideBlocks && a.k_row <= far && a.v_row <= far) {
    a.tiles = wide;
    hipLaunchKernelGGL(prefill_attn_wide<DT>, dim3(wide * heads), dim3(kWideThreads), 0, s, a);
  } else {
    a.tiles = (a.S + 4 * kQ - 1) / (4 * kQ);
    hipLaunchKernelGGL(prefill_attn_kernel<DT>, dim3(a.tiles * heads), dim3(4 * kWave), 0, s, a);
  }
  return tw_host::check_launch();
}

}  // namespace
}  // namespace tw

extern "C" int tw_prefill_attention(const void* q, const void* k, const void* v, int dtype, int S, int G, int R, int D,
                                    int64_t q_row, int64_t q_head, int64_t k_row, int64_t k_head, int64_t v_row,
                                    int64_t v_head, const void* cos, const void* sin, int64_t cos_row, int64_t sin_row,
                                    float softmax_scale, void* out, void* stream) {
  using namespace tw;
  if (S < 0 || G <= 0 || R <= 0) return TW_EINVAL;
  if (S == 0) return TW_OK;
  if (q == nullptr || k == nullptr || v == nullptr || out == nullptr) return TW_EINVAL;
  if (D != kHead || (dtype != TW_DTYPE_F16 && dtype != TW_DTYPE_BF16) || !(softmax_scale > 0.0f))
    return TW_EUNSUPPORTED;
  if (static_cast<int64_t>((S + 127) / 128) * G * R > 0x7fffffff || S > (1 << 24)) return TW_EUNSUPPORTED;
  if ((cos == nullptr) != (sin == nullptr)) return TW_EINVAL;
  const int64_t strides[] = {q_row, q_head, k_row, k_head, v_row, v_head, cos_row, sin_row};
  for (const int64_t s : strides)
    if (s < 0 || s % 8 != 0) return TW_EINVAL;  // every row starts on 16 bytes
  if (((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
        reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(cos) | reinterpret_cast<uintptr_t>(sin)) & 15) != 0)
    return TW_EINVAL;
  PrefillArgs a;
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.out = static_cast<uint16_t*>(out);
  a.q_row = q_row, a.q_head = q_head, a.k_row = k_row, a.k_head = k_head, a.v_row = v_row, a.v_head = v_head;
  a.cos = static_cast<const uint16_t*>(cos), a.sin = static_cast<const uint16_t*>(sin);
  a.cos_row = cos_row, a.sin_row = sin_row;
  a.out_row = static_cast<int64_t>(G) * R * D;
  a.S = S, a.G = G, a.R = R;
  a.scale_log2 = softmax_scale * 1.4426950408889634f;
  a.slack = fminf(8.0f / a.scale_log2, std::numeric_limits<float>::max());
  const hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == TW_DTYPE_F16 ? launch<F16>(a, s) : launch<BF16>(a, s);
}
