// Prompt metadata: per-page key min/max (Quest) fused with per-token affine
// INT4 packing (Twilight), one wavefront per page.
//
// Reference: QuestTopKOffloadedCache._build_metadata (quest_offload_cache.py:
// 276-289) and affine_int4_pack (twilight_offload_cache.py:25-37), called
// together from the Twilight override (twilight_offload_cache.py:925-936).
//
// The general layout (build_metadata_kernel; 16-row pages of 128 16-bit
// channels have build_metadata_chunks): a wavefront owns one page of bs rows (or, for rows outside complete
// pages, a chunk of 16 rows).  Lane l owns the channel pairs
// (2l + 128c, 2l + 1 + 128c), so a row of 128 16-bit keys is one coalesced
// 256-byte load and the packed INT4 row is one coalesced 64-byte store
// (lane l writes byte l, whose low nibble is channel 2l).  The row min/max
// needed by INT4 is a wave reduction; the page min/max is a per-lane running
// reduction over the page's rows, so the keys are read exactly once.
#pragma clang fp contract(off)

#include "page_chunk.h"
#include "rope.h"
#include "tw_common.h"

namespace tw {
namespace {

constexpr int kMaxPairChunks = 8;  // D <= 1024

__device__ __forceinline__ void load_pair(const uint16_t* p, uint16_t& a, uint16_t& b) {
  const uint32_t w = *reinterpret_cast<const uint32_t*>(p);
  a = static_cast<uint16_t>(w & 0xffffu);
  b = static_cast<uint16_t>(w >> 16);
}
__device__ __forceinline__ void load_pair(const float* p, float& a, float& b) {
  const float2 w = *reinterpret_cast<const float2*>(p);
  a = w.x;
  b = w.y;
}


template <typename DT>
__device__ __forceinline__ void process_row(const typename DT::storage* __restrict__ row, int D, int nchunk,
                                            int lane, bool want_pages, uint32_t (&pmin)[2 * kMaxPairChunks],
                                            uint32_t (&pmax)[2 * kMaxPairChunks], uint32_t& pnan,
                                            uint8_t* __restrict__ packed_row,
                                            typename DT::storage* __restrict__ scale_out,
                                            typename DT::storage* __restrict__ min_out) {
  using S = typename DT::storage;
  S v[2 * kMaxPairChunks];
  uint32_t kmin = 0xffffffffu, kmax = 0u;
  bool any_nan = false;
#pragma unroll
  for (int c = 0; c < kMaxPairChunks; ++c) {
    if (c >= nchunk) break;
    const int d = 2 * lane + 128 * c;
    if (d < D) {
      load_pair(row + d, v[2 * c], v[2 * c + 1]);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const S x = v[2 * c + h];
        const bool nan = is_nan(DT{}, x);
        const uint32_t k = order_key(DT{}, x);
        any_nan |= nan;
        kmin = k < kmin ? k : kmin;
        kmax = k > kmax ? k : kmax;
        if (want_pages) {
          pnan |= nan ? (1u << (2 * c + h)) : 0u;
          pmin[2 * c + h] = k < pmin[2 * c + h] ? k : pmin[2 * c + h];
          pmax[2 * c + h] = k > pmax[2 * c + h] ? k : pmax[2 * c + h];
        }
      }
    }
  }
  if (packed_row == nullptr) return;
  kmin = wave_min_u32(kmin);
  kmax = wave_max_u32(kmax);
  any_nan = __ballot(any_nan) != 0ull;
  S mn = any_nan ? canonical_nan(DT{}) : from_order_key(DT{}, kmin);
  S mx = any_nan ? canonical_nan(DT{}) : from_order_key(DT{}, kmax);
  const float mnf = to_f32(DT{}, mn);
  const float mxf = to_f32(DT{}, mx);
  const S sc = from_f32(DT{}, int4_scale<DT>(mnf, mxf));
  const float sf = to_f32(DT{}, sc);
#pragma unroll
  for (int c = 0; c < kMaxPairChunks; ++c) {
    if (c >= nchunk) break;
    const int d = 2 * lane + 128 * c;
    if (d < D) {
      const uint32_t lo = int4_code(to_f32(DT{}, v[2 * c]), mnf, sf);
      const uint32_t hi = int4_code(to_f32(DT{}, v[2 * c + 1]), mnf, sf);
      packed_row[d / 2] = static_cast<uint8_t>(lo | (hi << 4));
    }
  }
  if (lane == 0) {
    *scale_out = sc;
    *min_out = mn;
  }
}

template <typename DT>
__global__ __launch_bounds__(256) void build_metadata_kernel(
    const typename DT::storage* __restrict__ keys, int64_t key_entry_stride, int T, int D, int sink,
    int bs, int pages, int other_rows, typename DT::storage* __restrict__ page_min,
    typename DT::storage* __restrict__ page_max, int64_t page_entry_stride,
    uint8_t* __restrict__ packed, typename DT::storage* __restrict__ scale,
    typename DT::storage* __restrict__ minimum, int64_t quant_entry_stride) {
  using S = typename DT::storage;
  const int e = blockIdx.y;
  const int wave = blockIdx.x * (blockDim.x / kWave) + static_cast<int>(threadIdx.x) / kWave;
  const int lane = lane_id();
  const int other_chunks = (other_rows + 15) / 16;
  if (wave >= pages + other_chunks) return;
  const int nchunk = (D + 127) / 128;
  const S* kb = keys + static_cast<int64_t>(e) * key_entry_stride;
  const bool quant = packed != nullptr;

  uint32_t pmin[2 * kMaxPairChunks], pmax[2 * kMaxPairChunks], pnan = 0;
#pragma unroll
  for (int i = 0; i < 2 * kMaxPairChunks; ++i) {
    pmin[i] = 0xffffffffu;
    pmax[i] = 0u;
  }

  if (wave < pages) {
    const int t0 = sink + wave * bs;
    for (int i = 0; i < bs; ++i) {
      const int t = t0 + i;
      const int64_t qrow = static_cast<int64_t>(e) * quant_entry_stride + t;
      process_row<DT>(kb + static_cast<int64_t>(t) * D, D, nchunk, lane, page_min != nullptr, pmin, pmax,
                      pnan, quant ? packed + qrow * (D / 2) : nullptr, quant ? scale + qrow : nullptr,
                      quant ? minimum + qrow : nullptr);
    }
    if (page_min != nullptr) {
      S* mn_row = page_min + static_cast<int64_t>(e) * page_entry_stride + static_cast<int64_t>(wave) * D;
      S* mx_row = page_max + static_cast<int64_t>(e) * page_entry_stride + static_cast<int64_t>(wave) * D;
#pragma unroll
      for (int c = 0; c < kMaxPairChunks; ++c) {
        if (c >= nchunk) break;
        const int d = 2 * lane + 128 * c;
        if (d < D) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const bool nan = (pnan >> (2 * c + h)) & 1u;
            mn_row[d + h] = nan ? canonical_nan(DT{}) : from_order_key(DT{}, pmin[2 * c + h]);
            mx_row[d + h] = nan ? canonical_nan(DT{}) : from_order_key(DT{}, pmax[2 * c + h]);
          }
        }
      }
    }
    return;
  }
  // Rows outside complete pages (sink rows and the partial tail): INT4 only.
  if (!quant) return;
  const int head_rows = sink < T ? sink : T;
  const int base = (wave - pages) * 16;
  for (int i = 0; i < 16; ++i) {
    const int j = base + i;
    if (j >= other_rows) break;
    const int t = j < head_rows ? j : sink + pages * bs + (j - head_rows);
    const int64_t qrow = static_cast<int64_t>(e) * quant_entry_stride + t;
    process_row<DT>(kb + static_cast<int64_t>(t) * D, D, nchunk, lane, false, pmin, pmax, pnan,
                    packed + qrow * (D / 2), scale + qrow, minimum + qrow);
  }
}

// The same outputs for 16-row pages of 128 16-bit channels, a wavefront a page
// (or 16 rows outside the pages) with the page's 4 KB loaded at once.  Bound:
// HBM; a row at a time the loads went out one by one and every row's wave
// reductions and eight IEEE divisions stood in series behind them.
// 32768 rows x 8 KV heads, bf16, with INT4: 22.4 us (4.2 TB/s) against 80, the
// vector unit's share about as long as the memory's; without INT4 15.5 us (4.9
// TB/s) against 49.
template <typename DT, bool QUANT>
__global__ __launch_bounds__(256) void build_metadata_chunks(
    const uint16_t* __restrict__ keys, int64_t key_entry_stride, int T, int sink, int pages, int head_chunks,
    int chunks, uint16_t* __restrict__ page_min, uint16_t* __restrict__ page_max, int64_t page_entry_stride,
    uint8_t* __restrict__ packed, uint16_t* __restrict__ scale, uint16_t* __restrict__ minimum,
    int64_t quant_entry_stride) {
  const int e = blockIdx.y;
  const int chunk = wave_uniform(blockIdx.x * (blockDim.x / kWave) + static_cast<int>(threadIdx.x) / kWave);
  if (chunk >= chunks) return;
  const int lane = lane_id();
  // pages first, then the rows before them, then the rows after them
  int t0 = sink + chunk * kChunkRows, end = T;
  if (chunk >= pages) {
    const int c = chunk - pages;
    const bool head = c < head_chunks;
    t0 = head ? c * kChunkRows : sink + pages * kChunkRows + (c - head_chunks) * kChunkRows;
    end = head && sink < T ? sink : T;
  }
  const uint16_t* kb = keys + static_cast<int64_t>(e) * key_entry_stride + 8 * (lane % 16);
  u32x4 x[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    int t = t0 + 4 * j + lane / 16;
    t = t < end ? t : end - 1;
    x[j] = *reinterpret_cast<const u32x4*>(kb + static_cast<int64_t>(t) * 128);
  }
  if (chunk < pages) {
    const int64_t at = static_cast<int64_t>(e) * page_entry_stride + static_cast<int64_t>(chunk) * 128;
    chunk_page_minmax<DT>(x, lane, page_min + at, page_max + at);
  }
  if constexpr (QUANT) {
    const int64_t at = static_cast<int64_t>(e) * quant_entry_stride + t0;
    chunk_int4<DT>(x, end - t0, lane, packed + at * 64, scale + at, minimum + at);
  }
}

// The prompt's K and V of one layer into the cache in one pass: K rotated, both
// rows stored, the page min/max and (QUANT) the INT4 keys formed from the
// rotated rows while they are in registers.  A wavefront takes 16 rows of a KV
// head like build_metadata_chunks, K, V, cos and sin loaded at once; the other
// half of a rotation pair is 8 lanes away in the 16 that hold a row.
//
// Bound: HBM, 2 x 2 x 256 bytes a row and head.  8 heads, bf16: 32768 rows with
// INT4 69 us (4.2 TB/s), 2048 rows without 7.5 us.  As separate passes (rotation
// in five elementwise launches with q's, two copies, the slab copies and the
// metadata of each head) 1.2 ms and 0.22 ms.
struct PromptKvArgs {
  const uint16_t* k;
  const uint16_t* v;
  int64_t k_row, k_head, v_row, v_head;  // in elements
  const uint16_t* cos;
  const uint16_t* sin;
  int64_t cos_row, sin_row;
  int T, G, sink, pages, head_chunks, chunks;
  uint16_t* out_k;
  uint16_t* out_v;
  int64_t out_entry;
  uint16_t* page_min;
  uint16_t* page_max;
  int64_t page_entry;
  uint8_t* packed;
  uint16_t* scale;
  uint16_t* minimum;
  int64_t quant_entry;
};

template <typename DT, bool QUANT>
__global__ __launch_bounds__(256) void prompt_kv_kernel(PromptKvArgs a) {
  // head-minor: the heads' pieces of a projection row are read together
  const int e = static_cast<int>(blockIdx.x) % a.G;
  const int chunk = wave_uniform(static_cast<int>(blockIdx.x) / a.G * (256 / kWave) +
                                 static_cast<int>(threadIdx.x) / kWave);
  if (chunk >= a.chunks) return;
  const int lane = lane_id();
  const int unit = lane % 16, quad = lane / 16;
  // pages first, then the rows before them, then the rows after them
  int t0 = a.sink + chunk * kChunkRows, end = a.T;
  if (chunk >= a.pages) {
    const int c = chunk - a.pages;
    const bool head = c < a.head_chunks;
    t0 = head ? c * kChunkRows : a.sink + a.pages * kChunkRows + (c - a.head_chunks) * kChunkRows;
    end = head && a.sink < a.T ? a.sink : a.T;
  }
  u32x4 x[4], y[4], c[4], s[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    int64_t t = t0 + 4 * j + quad;
    t = t < end ? t : end - 1;
    x[j] = *reinterpret_cast<const u32x4*>(a.k + e * a.k_head + t * a.k_row + 8 * unit);
    c[j] = *reinterpret_cast<const u32x4*>(a.cos + t * a.cos_row + 8 * unit);
    s[j] = *reinterpret_cast<const u32x4*>(a.sin + t * a.sin_row + 8 * unit);
    y[j] = *reinterpret_cast<const u32x4*>(a.v + e * a.v_head + t * a.v_row + 8 * unit);
  }
  constexpr int kDppRowRor8 = 0x128;  // lane u of a 16-lane row reads lane u ^ 8: channels 64 away
  const uint32_t negate = unit < 8 ? 0x80008000u : 0u;
  const int64_t out = e * a.out_entry + static_cast<int64_t>(t0) * 128 + 8 * unit;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    u32x4 r;
#pragma unroll
    for (int p = 0; p < 4; ++p)
      r[p] = rope_word<DT>(x[j][p], dpp_u32<kDppRowRor8>(x[j][p]) ^ negate, c[j][p], s[j][p]);
    x[j] = r;
    const int row = 4 * j + quad;
    if (t0 + row < end) {
      *reinterpret_cast<u32x4*>(a.out_k + out + row * 128) = r;
      *reinterpret_cast<u32x4*>(a.out_v + out + row * 128) = y[j];
    }
  }
  if (chunk < a.pages) {
    const int64_t at = e * a.page_entry + static_cast<int64_t>(chunk) * 128;
    chunk_page_minmax<DT>(x, lane, a.page_min + at, a.page_max + at);
  }
  if constexpr (QUANT) {
    const int64_t at = e * a.quant_entry + t0;
    chunk_int4<DT>(x, end - t0, lane, a.packed + at * 64, a.scale + at, a.minimum + at);
  }
}

// Decode-time update after row `position` of each entry was written: the
// row's INT4 code and, when the row completes page p = (position - sink) / bs
// (position - sink + 1 a multiple of bs), that page's min/max over its bs
// rows.  One wavefront per entry, the same row routine as the prompt build,
// so the result equals a rebuild over position + 1 rows bit for bit.
template <typename DT>
__global__ __launch_bounds__(256) void update_metadata_kernel(
    const typename DT::storage* __restrict__ keys, int64_t key_entry_stride, int n_entries, int position_all,
    const int32_t* __restrict__ positions, int max_position, int max_pages, int D,
    int sink, int bs, typename DT::storage* __restrict__ page_min, typename DT::storage* __restrict__ page_max,
    int64_t page_entry_stride, uint8_t* __restrict__ packed, typename DT::storage* __restrict__ scale,
    typename DT::storage* __restrict__ minimum, int64_t quant_entry_stride) {
  using S = typename DT::storage;
  const int e = blockIdx.x * (blockDim.x / kWave) + static_cast<int>(threadIdx.x) / kWave;
  if (e >= n_entries) return;
  // ragged entries: each its own row; rows beyond the buffers are skipped
  const int position = positions != nullptr ? positions[e] : position_all;
  if (position < 0 || position > max_position) return;
  if (page_min != nullptr && position >= sink && (position - sink + 1) % bs == 0 &&
      (position - sink) / bs >= max_pages)
    return;
  const int lane = lane_id();
  const int nchunk = (D + 127) / 128;
  const S* kb = keys + static_cast<int64_t>(e) * key_entry_stride;
  const bool quant = packed != nullptr;
  const int64_t qrow = static_cast<int64_t>(e) * quant_entry_stride + position;
  uint8_t* prow = quant ? packed + qrow * (D / 2) : nullptr;
  S* srow = quant ? scale + qrow : nullptr;
  S* mrow = quant ? minimum + qrow : nullptr;
  uint32_t pmin[2 * kMaxPairChunks], pmax[2 * kMaxPairChunks], pnan = 0;
#pragma unroll
  for (int i = 0; i < 2 * kMaxPairChunks; ++i) {
    pmin[i] = 0xffffffffu;
    pmax[i] = 0u;
  }
  const bool completes = page_min != nullptr && position >= sink && (position - sink + 1) % bs == 0;
  if (!completes) {
    if (quant)
      process_row<DT>(kb + static_cast<int64_t>(position) * D, D, nchunk, lane, false, pmin, pmax, pnan, prow,
                      srow, mrow);
    return;
  }
  const int page = (position - sink) / bs;
  const int t0 = sink + page * bs;
  for (int i = 0; i < bs; ++i) {
    const int t = t0 + i;
    const bool last = t == position;
    process_row<DT>(kb + static_cast<int64_t>(t) * D, D, nchunk, lane, true, pmin, pmax, pnan,
                    last ? prow : nullptr, last ? srow : nullptr, last ? mrow : nullptr);
  }
  S* mn_row = page_min + static_cast<int64_t>(e) * page_entry_stride + static_cast<int64_t>(page) * D;
  S* mx_row = page_max + static_cast<int64_t>(e) * page_entry_stride + static_cast<int64_t>(page) * D;
#pragma unroll
  for (int c = 0; c < kMaxPairChunks; ++c) {
    if (c >= nchunk) break;
    const int d = 2 * lane + 128 * c;
    if (d < D) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bool nan = (pnan >> (2 * c + h)) & 1u;
        mn_row[d + h] = nan ? canonical_nan(DT{}) : from_order_key(DT{}, pmin[2 * c + h]);
        mx_row[d + h] = nan ? canonical_nan(DT{}) : from_order_key(DT{}, pmax[2 * c + h]);
      }
    }
  }
}

template <typename DT>
int launch_update(const void* keys, int64_t key_entry_stride, int n_entries, int position,
                  const int32_t* positions, int max_position, int max_pages, int D, int sink, int bs,
                  void* page_min, void* page_max, int64_t page_entry_stride, void* packed, void* scale,
                  void* minimum, int64_t quant_entry_stride, hipStream_t stream) {
  using S = typename DT::storage;
  hipLaunchKernelGGL(update_metadata_kernel<DT>, dim3((n_entries + 3) / 4), dim3(256), 0, stream,
                     static_cast<const S*>(keys), key_entry_stride, n_entries, position, positions, max_position,
                     max_pages, D, sink, bs,
                     static_cast<S*>(page_min), static_cast<S*>(page_max), page_entry_stride,
                     static_cast<uint8_t*>(packed), static_cast<S*>(scale), static_cast<S*>(minimum),
                     quant_entry_stride);
  return tw_host::check_launch();
}

int dispatch_update(int dtype, const void* keys, int64_t key_entry_stride, int n_entries, int position,
                    const int32_t* positions, int max_position, int max_pages, int D, int sink, int bs,
                    void* page_min, void* page_max, int64_t page_entry_stride, void* packed, void* scale,
                    void* minimum, int64_t quant_entry_stride, hipStream_t s) {
  switch (dtype) {
    case TW_DTYPE_F16:
      return launch_update<F16>(keys, key_entry_stride, n_entries, position, positions, max_position, max_pages, D,
                                sink, bs, page_min, page_max, page_entry_stride, packed, scale, minimum,
                                quant_entry_stride, s);
    case TW_DTYPE_BF16:
      return launch_update<BF16>(keys, key_entry_stride, n_entries, position, positions, max_position, max_pages, D,
                                 sink, bs, page_min, page_max, page_entry_stride, packed, scale, minimum,
                                 quant_entry_stride, s);
    case TW_DTYPE_F32:
      return launch_update<F32>(keys, key_entry_stride, n_entries, position, positions, max_position, max_pages, D,
                                sink, bs, page_min, page_max, page_entry_stride, packed, scale, minimum,
                                quant_entry_stride, s);
    default:
      return TW_EINVAL;
  }
}

template <typename DT>
__global__ __launch_bounds__(256) void int4_dequant_kernel(const uint8_t* __restrict__ packed,
                                                           const typename DT::storage* __restrict__ scale,
                                                           const typename DT::storage* __restrict__ minimum,
                                                           int64_t N, int D, float* __restrict__ out) {
  const int64_t total = N * D;
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t n = i / D;
    const int d = static_cast<int>(i - n * D);
    const uint32_t byte = packed[n * (D / 2) + d / 2];
    const uint32_t code = (d & 1) ? (byte >> 4) & 15u : byte & 15u;
    const float s = to_f32(DT{}, scale[n]);
    const float m = to_f32(DT{}, minimum[n]);
    out[i] = static_cast<float>(code) * s + m;
  }
}

template <typename DT>
int launch_build(const void* keys, int64_t key_entry_stride, int n_entries, int T, int D, int sink, int bs,
                 void* page_min, void* page_max, int64_t page_entry_stride, void* packed, void* scale,
                 void* minimum, int64_t quant_entry_stride, hipStream_t stream) {
  using S = typename DT::storage;
  const int pages = (page_min != nullptr && T > sink) ? (T - sink) / bs : 0;
  // Rows not covered by a page wave still need INT4 codes.
  int other_rows = 0;
  if (packed != nullptr) {
    const int head_rows = sink < T ? sink : T;
    const int covered = (page_min != nullptr) ? pages * bs : 0;
    other_rows = T - covered;
    (void)head_rows;
  }
  int pages_eff = pages;
  if (page_min == nullptr) pages_eff = 0;
  // Without page waves the "other" rows are simply all rows: treat sink as T
  // so the index mapping (j < head_rows -> j) covers everything.
  const int sink_eff = (page_min == nullptr) ? T : sink;
  const int waves = pages_eff + (other_rows + 15) / 16;
  if (waves == 0) return TW_OK;
  if constexpr (sizeof(S) == 2) {
    // whole 16-byte units of keys and page rows, whole words of packed rows
    const uintptr_t wide = reinterpret_cast<uintptr_t>(keys) | reinterpret_cast<uintptr_t>(page_min) |
                           reinterpret_cast<uintptr_t>(page_max);
    if (D == 128 && bs == kChunkRows && (wide & 15) == 0 && (reinterpret_cast<uintptr_t>(packed) & 3) == 0 &&
        key_entry_stride % 8 == 0 && page_entry_stride % 8 == 0) {
      const int head_rows = packed == nullptr ? 0 : (sink_eff < T ? sink_eff : T);
      const int head_chunks = (head_rows + kChunkRows - 1) / kChunkRows;
      const int tail_rows = packed == nullptr ? 0 : other_rows - head_rows;
      const int chunks = pages_eff + head_chunks + (tail_rows + kChunkRows - 1) / kChunkRows;
      const auto kernel = packed != nullptr ? build_metadata_chunks<DT, true> : build_metadata_chunks<DT, false>;
      hipLaunchKernelGGL(kernel, dim3((chunks + 3) / 4, n_entries), dim3(256), 0, stream,
                         static_cast<const uint16_t*>(keys), key_entry_stride, T, sink_eff, pages_eff, head_chunks,
                         chunks, static_cast<uint16_t*>(page_min), static_cast<uint16_t*>(page_max),
                         page_entry_stride, static_cast<uint8_t*>(packed), static_cast<uint16_t*>(scale),
                         static_cast<uint16_t*>(minimum), quant_entry_stride);
      return tw_host::check_launch();
    }
  }
  dim3 grid((waves + 3) / 4, n_entries);
  hipLaunchKernelGGL(build_metadata_kernel<DT>, grid, dim3(256), 0, stream, static_cast<const S*>(keys),
                     key_entry_stride, T, D, sink_eff, bs, pages_eff, other_rows, static_cast<S*>(page_min),
                     static_cast<S*>(page_max), page_entry_stride, static_cast<uint8_t*>(packed),
                     static_cast<S*>(scale), static_cast<S*>(minimum), quant_entry_stride);
  return tw_host::check_launch();
}

}  // namespace
}  // namespace tw

extern "C" int tw_prompt_kv(const void* k, const void* v, int64_t k_row, int64_t k_head, int64_t v_row, int64_t v_head,
                            const void* cos, const void* sin, int64_t cos_row, int64_t sin_row, int dtype, int T, int G,
                            int D, int sink, int block_size, void* out_k, void* out_v, int64_t out_entry_stride,
                            void* page_min, void* page_max, int64_t page_entry_stride, void* packed, void* scale,
                            void* minimum, int64_t quant_entry_stride, void* stream) {
  using namespace tw;
  if (k == nullptr || v == nullptr || cos == nullptr || sin == nullptr || out_k == nullptr || out_v == nullptr)
    return TW_EINVAL;
  if (T < 0 || G <= 0 || sink < 0) return TW_EINVAL;
  if (D != 128 || block_size != kChunkRows || (dtype != TW_DTYPE_F16 && dtype != TW_DTYPE_BF16) || T > (1 << 24))
    return TW_EUNSUPPORTED;
  if ((packed == nullptr) != (scale == nullptr) || (packed == nullptr) != (minimum == nullptr)) return TW_EINVAL;
  const int pages = T > sink ? (T - sink) / kChunkRows : 0;
  if (pages > 0 && (page_min == nullptr || page_max == nullptr)) return TW_EINVAL;
  const int64_t strides[] = {k_row, k_head, v_row, v_head, cos_row, sin_row, out_entry_stride, page_entry_stride};
  for (const int64_t x : strides)
    if (x < 0 || x % 8 != 0) return TW_EINVAL;  // every row starts on 16 bytes
  const void* wide[] = {k, v, cos, sin, out_k, out_v, page_min, page_max};
  for (const void* x : wide)
    if ((reinterpret_cast<uintptr_t>(x) & 15) != 0) return TW_EINVAL;
  if ((reinterpret_cast<uintptr_t>(packed) & 3) != 0) return TW_EINVAL;
  if (G > 1 && (out_entry_stride < static_cast<int64_t>(T) * D || (packed != nullptr && quant_entry_stride < T) ||
                page_entry_stride < static_cast<int64_t>(pages) * D))
    return TW_EINVAL;
  if (T == 0) return TW_OK;
  PromptKvArgs a;
  a.k = static_cast<const uint16_t*>(k), a.v = static_cast<const uint16_t*>(v);
  a.k_row = k_row, a.k_head = k_head, a.v_row = v_row, a.v_head = v_head;
  a.cos = static_cast<const uint16_t*>(cos), a.sin = static_cast<const uint16_t*>(sin);
  a.cos_row = cos_row, a.sin_row = sin_row;
  a.T = T, a.G = G, a.sink = sink, a.pages = pages;
  const int head_rows = sink < T ? sink : T;
  const int tail_rows = T - head_rows - pages * kChunkRows;
  a.head_chunks = (head_rows + kChunkRows - 1) / kChunkRows;
  a.chunks = pages + a.head_chunks + (tail_rows + kChunkRows - 1) / kChunkRows;
  const int64_t blocks = static_cast<int64_t>((a.chunks + 3) / 4) * G;
  if (blocks > 0x7fffffff) return TW_EUNSUPPORTED;
  a.out_k = static_cast<uint16_t*>(out_k), a.out_v = static_cast<uint16_t*>(out_v), a.out_entry = out_entry_stride;
  a.page_min = static_cast<uint16_t*>(page_min), a.page_max = static_cast<uint16_t*>(page_max);
  a.page_entry = page_entry_stride;
  a.packed = static_cast<uint8_t*>(packed), a.scale = static_cast<uint16_t*>(scale);
  a.minimum = static_cast<uint16_t*>(minimum), a.quant_entry = quant_entry_stride;
  void (*kern)(PromptKvArgs);
  if (dtype == TW_DTYPE_F16)
    kern = packed != nullptr ? prompt_kv_kernel<F16, true> : prompt_kv_kernel<F16, false>;
  else
    kern = packed != nullptr ? prompt_kv_kernel<BF16, true> : prompt_kv_kernel<BF16, false>;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, static_cast<hipStream_t>(stream), a);
  return tw_host::check_launch();
}

extern "C" int tw_build_page_metadata(const void* keys, int64_t key_entry_stride, int n_entries, int T,
                                      int D, int dtype, int sink, int block_size, void* page_min,
                                      void* page_max, int64_t page_entry_stride, void* packed, void* scale,
                                      void* minimum, int64_t quant_entry_stride, void* stream) {
  if (keys == nullptr || n_entries <= 0 || T < 0 || D <= 0 || (D % 2) != 0 || D > 1024) return TW_EINVAL;
  if (sink < 0 || block_size <= 0) return TW_EINVAL;
  if ((page_min == nullptr) != (page_max == nullptr)) return TW_EINVAL;
  if (!((packed == nullptr) == (scale == nullptr) && (scale == nullptr) == (minimum == nullptr)))
    return TW_EINVAL;
  if (key_entry_stride < static_cast<int64_t>(T) * D && n_entries > 1) return TW_EINVAL;
  if (packed != nullptr && n_entries > 1 && quant_entry_stride < T) return TW_EINVAL;
  if (T == 0) return TW_OK;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case TW_DTYPE_F16:
      return tw::launch_build<tw::F16>(keys, key_entry_stride, n_entries, T, D, sink, block_size, page_min,
                                       page_max, page_entry_stride, packed, scale, minimum,
                                       quant_entry_stride, s);
    case TW_DTYPE_BF16:
      return tw::launch_build<tw::BF16>(keys, key_entry_stride, n_entries, T, D, sink, block_size, page_min,
                                        page_max, page_entry_stride, packed, scale, minimum,
                                        quant_entry_stride, s);
    case TW_DTYPE_F32:
      return tw::launch_build<tw::F32>(keys, key_entry_stride, n_entries, T, D, sink, block_size, page_min,
                                       page_max, page_entry_stride, packed, scale, minimum,
                                       quant_entry_stride, s);
    default:
      return TW_EINVAL;
  }
}

extern "C" int tw_update_page_metadata(const void* keys, int64_t key_entry_stride, int n_entries, int position,
                                       int D, int dtype, int sink, int block_size, void* page_min, void* page_max,
                                       int64_t page_entry_stride, void* packed, void* scale, void* minimum,
                                       int64_t quant_entry_stride, void* stream) {
  if (keys == nullptr || n_entries <= 0 || position < 0 || D <= 0 || (D % 2) != 0 || D > 1024) return TW_EINVAL;
  if (sink < 0 || block_size <= 0) return TW_EINVAL;
  if ((page_min == nullptr) != (page_max == nullptr)) return TW_EINVAL;
  if (!((packed == nullptr) == (scale == nullptr) && (scale == nullptr) == (minimum == nullptr)))
    return TW_EINVAL;
  if (n_entries > 1 && key_entry_stride < static_cast<int64_t>(position + 1) * D) return TW_EINVAL;
  if (packed != nullptr && n_entries > 1 && quant_entry_stride <= position) return TW_EINVAL;
  if (page_min != nullptr && n_entries > 1 && position >= sink && (position - sink + 1) % block_size == 0 &&
      page_entry_stride < static_cast<int64_t>((position - sink) / block_size + 1) * D)
    return TW_EINVAL;
  if (page_min == nullptr && packed == nullptr) return TW_OK;
  const int big = 0x7fffffff;
  return tw::dispatch_update(dtype, keys, key_entry_stride, n_entries, position, nullptr, big, big, D, sink,
                             block_size, page_min, page_max, page_entry_stride, packed, scale, minimum,
                             quant_entry_stride, static_cast<hipStream_t>(stream));
}

extern "C" int tw_update_page_metadata_ragged(const void* keys, int64_t key_entry_stride, int n_entries,
                                              const int32_t* positions, int max_position, int D, int dtype, int sink,
                                              int block_size, void* page_min, void* page_max, int max_pages,
                                              int64_t page_entry_stride, void* packed, void* scale, void* minimum,
                                              int64_t quant_entry_stride, void* stream) {
  if (keys == nullptr || positions == nullptr || n_entries <= 0 || max_position < 0 || D <= 0 || (D % 2) != 0 ||
      D > 1024)
    return TW_EINVAL;
  if (sink < 0 || block_size <= 0) return TW_EINVAL;
  if ((page_min == nullptr) != (page_max == nullptr)) return TW_EINVAL;
  if (!((packed == nullptr) == (scale == nullptr) && (scale == nullptr) == (minimum == nullptr)))
    return TW_EINVAL;
  if (n_entries > 1 && key_entry_stride < static_cast<int64_t>(max_position + 1) * D) return TW_EINVAL;
  if (packed != nullptr && n_entries > 1 && quant_entry_stride <= max_position) return TW_EINVAL;
  if (page_min != nullptr && (max_pages < 0 || (n_entries > 1 && page_entry_stride < static_cast<int64_t>(max_pages) * D)))
    return TW_EINVAL;
  if (page_min == nullptr && packed == nullptr) return TW_OK;
  return tw::dispatch_update(dtype, keys, key_entry_stride, n_entries, 0, positions, max_position, max_pages, D,
                             sink, block_size, page_min, page_max, page_entry_stride, packed, scale, minimum,
                             quant_entry_stride, static_cast<hipStream_t>(stream));
}

extern "C" int tw_int4_dequantize(const void* packed, const void* scale, const void* minimum, int dtype,
                                  int64_t N, int D, float* out, void* stream) {
  if (N < 0 || D <= 0 || (D % 2) != 0) return TW_EINVAL;
  if (N == 0) return TW_OK;
  if (packed == nullptr || scale == nullptr || minimum == nullptr || out == nullptr) return TW_EINVAL;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t total = N * D;
  const int blocks = static_cast<int>((total + 255) / 256 < 65536 ? (total + 255) / 256 : 65536);
  switch (dtype) {
    case TW_DTYPE_F16:
      hipLaunchKernelGGL(tw::int4_dequant_kernel<tw::F16>, dim3(blocks), dim3(256), 0, s,
                         static_cast<const uint8_t*>(packed), static_cast<const uint16_t*>(scale),
                         static_cast<const uint16_t*>(minimum), N, D, out);
      break;
    case TW_DTYPE_BF16:
      hipLaunchKernelGGL(tw::int4_dequant_kernel<tw::BF16>, dim3(blocks), dim3(256), 0, s,
                         static_cast<const uint8_t*>(packed), static_cast<const uint16_t*>(scale),
                         static_cast<const uint16_t*>(minimum), N, D, out);
      break;
    case TW_DTYPE_F32:
      hipLaunchKernelGGL(tw::int4_dequant_kernel<tw::F32>, dim3(blocks), dim3(256), 0, s,
                         static_cast<const uint8_t*>(packed), static_cast<const float*>(scale),
                         static_cast<const float*>(minimum), N, D, out);
      break;
    default:
      return TW_EINVAL;
  }
  return tw_host::check_launch();
}
