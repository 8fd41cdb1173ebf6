// Dense causal attention of a prompt on the matrix cores (head_dim 128,
// fp16 / bf16): every query row attends to the key rows at or before it, the
// attention the reference's prefill runs (mp.py:475-482).
//
// One block owns NW wavefronts x 32 query rows of one query head and walks the
// key rows in tiles of 64, the next tile's loads in flight (registers, then
// the other LDS buffer) while the current one is computed.  The products are
// taken transposed, so that a query stays in one lane column from the scores
// to the output:
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
// Bound: the matrix cores and, beside them, the exponentials (32 a lane and
// tile, as many issue cycles as half the tile's MFMAs).  8 KV heads of 4 query
// heads, bf16, 32768 rows: 9.0 ms, 975 TFLOP/s of the causal half (a library
// product of 8192^3 reaches 1186 here), against 137 ms for the score tiles in
// fp32 through batched products, mask and softmax; 2048 rows: 60 us against
// 1.0 ms.  Two 32-row query tiles a wavefront (half the LDS reads a product,
// one wavefront a SIMD) took 10.5 ms and 91 us: the second wavefront of a
// SIMD, whose products run under the first one's exponentials, is worth more.
#pragma clang fp contract(off)

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

// LDS slot (in 16-byte units) of unit u of tile row r: a row is 256 bytes, one
// turn of the 64 banks, so unit u of 8 consecutive rows goes to 8 different
// slots (the fragment reads of K: 8 rows, one unit), and the unit pairs of 4
// consecutive rows to 4 different slot pairs (the transposing reads of V).
__device__ __forceinline__ int slot(int r, int u) { return r * kRowUnits + (u ^ (2 * (r & 7))); }

__device__ __forceinline__ float both_halves_max(float x) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
}
__device__ __forceinline__ float both_halves_sum(float x) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(h[0]) + __uint_as_float(h[1]);
}

template <typename DT, int NW>
__global__ __launch_bounds__(NW * kWave, 2) void prefill_attn_kernel(PrefillArgs a) {
  typedef typename Frag<DT>::type frag;
  constexpr int kLoads = kKeys * kRowUnits / (NW * kWave);  // 16-byte units a thread stages, for K and for V
  __shared__ u32x4 s_k[2][kKeys * kRowUnits];
  __shared__ u32x4 s_v[2][kKeys * kRowUnits];

  const int tid = threadIdx.x, lane = tid % kWave, wave = wave_uniform(tid / kWave);
  const int col = lane % 32, half = lane / 32;
  // group-minor, the longest query tiles first
  const int g = blockIdx.x % a.G;
  const int rest = blockIdx.x / a.G;
  const int head = g * a.R + rest % a.R;
  const int qt = a.tiles - 1 - rest / a.R;
  const int q_block = qt * NW * kQ;
  const int q0 = q_block + wave * kQ;
  const int S = a.S;

  const uint16_t* kg = a.k + g * a.k_head;
  const uint16_t* vg = a.v + g * a.v_head;

  // Q^T fragments, kept in registers
  frag qf[8];
  const int row = q0 + col;
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
    s_k[b][at] = rk[i];                                                                                    \
    s_v[b][at] = rv[i];                                                                                    \
  }

  f32x16 o[4];
  float m = -__builtin_inff(), l = 0.0f;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[c][i] = 0.0f;
  // raw scores past the running maximum by less than this are taken without
  // moving it: their weights stay below 2^8, and the accumulators are not
  // rescaled on every tile
  const float slack = 8.0f / a.scale_log2;

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
          const frag kf = __builtin_bit_cast(frag, s_k[b][slot(32 * kb + col, 2 * s + half)]);
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
      float mx = fmaxf(sc[0][0], sc[1][0]);
#pragma unroll
      for (int i = 1; i < 16; ++i) mx = fmaxf(mx, fmaxf(sc[0][i], sc[1][i]));
      mx = both_halves_max(mx);
      if (__any(mx > m + slack)) {
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
      const float ms = m * a.scale_log2;
      float sum = 0.0f;
      frag pf[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        frag w;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float p =
              __builtin_amdgcn_exp2f(__builtin_fmaf(sc[ks / 2][8 * (ks % 2) + i], a.scale_log2, -ms));
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
            const uint2* p = reinterpret_cast<const uint2*>(&s_v[b][slot(r, ch / 8)]) + (ch % 8) / 4;
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

  const float inv = 1.0f / both_halves_sum(l);
  if (row < S) {
    uint16_t* p = a.out + static_cast<int64_t>(row) * a.out_row + head * kHead + 4 * half;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        typename Frag<DT>::quad w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = Frag<DT>::narrow(o[c][4 * i + j] * inv);
        *reinterpret_cast<typename Frag<DT>::quad*>(p + 32 * c + 8 * i) = w;
      }
  }
}

template <typename DT, int NW>
int launch(PrefillArgs a, hipStream_t s) {
  a.tiles = (a.S + NW * kQ - 1) / (NW * kQ);
  hipLaunchKernelGGL((prefill_attn_kernel<DT, NW>), dim3(a.tiles * a.G * a.R), dim3(NW * kWave), 0, s, a);
  return tw_host::check_launch();
}

// 8 wavefronts share each staged tile where there are enough blocks to keep
// every CU in work to the end (8 a CU); with fewer, smaller blocks balance
// better.  32 heads: 32768 rows (4096 blocks) 9.0 ms against 9.4 with 4
// wavefronts, 8192 rows (1024 blocks) 0.63 ms both, 2048 rows 69 us against 60.
template <typename DT>
int launch_any(const PrefillArgs& a, hipStream_t s) {
  const int64_t wide = static_cast<int64_t>((a.S + 8 * kQ - 1) / (8 * kQ)) * a.G * a.R;
  return wide >= 2048 ? launch<DT, 8>(a, s) : launch<DT, 4>(a, s);
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
  const hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == TW_DTYPE_F16 ? launch_any<F16>(a, s) : launch_any<BF16>(a, s);
}
