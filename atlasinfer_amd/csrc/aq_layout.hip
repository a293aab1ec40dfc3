// aq_layout.hip -- outlier index bookkeeping, the reference's compacted code
// stream, and dequantization.
//
// Reference: atlasinfer_core/quant/adaptive_quantizer.py
//   compacted stream of non-outlier codes     :110,125-126,136 (written)
//                                             :209-212         (read back)
//   dequantize_tensor per-block loop          :185-245
// The reference finds the outliers of each block by comparing against all
// outlier indices (O(blocks * nnz)) and syncs to the host once per block
// (:194-195,234).  Here a workgroup owns a span of 8192 elements, finds its
// slice of the ascending index list with two wave-wide searches and turns it
// into a bitmap in LDS with a running count, so that a thread knows the
// outliers of its 8 elements and those before them without a search.
#include "aq_common.h"
#include "aq_tiles.h"

namespace {

// A workgroup of 256 threads takes a span of consecutive elements, each
// thread kRuns runs of 8 consecutive elements: 8 codes are one 8-byte access
// and 8 fp16 one 16-byte access, and a wave's accesses are contiguous.
constexpr int kRuns = 4;
constexpr int kSpan = 256 * 8 * kRuns;

__device__ __forceinline__ int64_t lower_bound_i64(const int64_t* a, int64_t n, int64_t key) {
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    int64_t mid = (lo + hi) >> 1;
    if (a[mid] < key)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

__global__ __launch_bounds__(256) void segment_offsets_kernel(const int64_t* idx, int64_t nnz, int64_t nseg,
                                                              int64_t seg_len, int32_t* seg_ptr) {
  const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (s > nseg) return;
  seg_ptr[s] = (int32_t)lower_bound_i64(idx, nnz, s * seg_len);
}

__global__ __launch_bounds__(256) void outlier_cols_kernel(const int64_t* idx, int64_t nnz, int64_t K,
                                                           int32_t* cols) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p < nnz) cols[p] = (int32_t)(idx[p] % K);
}

// First position in ascending a[0, n) whose value is >= key, found by one
// wave: 64 probes a step, so a list of 2^18 takes three dependent loads
// instead of 18.  The same in every lane.
__device__ __forceinline__ int64_t wave_lower_bound_i64(const int64_t* a, int64_t n, int64_t key) {
  const int lane = threadIdx.x & 63;
  int64_t lo = 0;
  while (n > 0) {
    const int64_t step = (n + 63) >> 6;
    const int64_t p = lane * step;
    const bool below = p < n && a[lo + p] < key;
    const int c = __builtin_popcountll(__ballot(below));  // the first c probes lie below key
    if (c == 0) break;
    const int64_t from = (c - 1) * step + 1;
    n = min(step - 1, n - from);
    lo += from;
  }
  return lo;
}

// The outliers of a workgroup's span [t0, t1) as a bitmap in LDS with the
// number before each 32-element word, so that a thread knows where its run's
// codes sit in the compacted stream without a search.
struct SpanOutliers {
  uint32_t bits[kSpan / 32];
  int before[kSpan / 32];
  int64_t lb[2];
  int scan[4];

  // Every thread of the workgroup calls it.
  __device__ __forceinline__ int64_t build(const int64_t* idx, int64_t nnz, int64_t t0, int64_t t1) {
    const int t = threadIdx.x;
    bits[t] = 0;
    if (t < 128) {
      const int64_t p = wave_lower_bound_i64(idx, nnz, t < 64 ? t0 : t1);
      if ((t & 63) == 0) lb[t >> 6] = p;
    }
    __syncthreads();
    const int64_t lb0 = lb[0];
    const int cnt = (int)(lb[1] - lb0);
    for (int i = t; i < cnt; i += 256) {
      const int64_t e = idx[lb0 + i] - t0;
      // always so in an ascending list; one that is not writes nothing past
      // bits (and may put a run's codes outside the stream: the callers look)
      if ((uint64_t)e < (uint64_t)kSpan) atomicOr(&bits[e >> 5], 1u << (e & 31));
    }
    __syncthreads();
    int total;
    before[t] = team_excl_scan_i32<256>(__builtin_popcount(bits[t]), scan, &total);
    __syncthreads();
    return lb0;
  }
  // outlier flags of the 8 elements at `off` in the span; *pre: outliers of the span before them
  __device__ __forceinline__ uint32_t run(int off, int* pre) const {
    const uint32_t w = bits[off >> 5];
    const int sh = off & 31;
    *pre = before[off >> 5] + __builtin_popcount(w & ((1u << sh) - 1u));
    return (w >> sh) & 255u;
  }
};
static_assert(kSpan / 32 == 256, "one bitmap word per thread");

// 8 bytes at any address (gfx950 loads and stores them unaligned).
__device__ __forceinline__ uint64_t load8(const uint8_t* p) {
  uint64_t w;
  __builtin_memcpy(&w, p, 8);
  return w;
}
__device__ __forceinline__ uint64_t low_bytes(int n) { return ((uint64_t)1 << (8 * n)) - 1; }  // n < 8

// Whether positions c0 .. c0 + 7 lie in a stream of `len` codes (one comparison).
__device__ __forceinline__ bool in_stream8(int64_t c0, int64_t len) {
  return (uint64_t)c0 < (uint64_t)max(len - 7, (int64_t)0);
}

// The codes of a run from a compacted stream of `len` codes: n - popcount(bits)
// of them from position c0 on, a 0 code put in at each flagged element.
// Nothing outside the stream is read: c0 is negative after repeated indices.
__device__ __forceinline__ uint64_t stream_codes(const uint8_t* stream, int64_t len, int64_t c0, uint32_t bits,
                                                 int n) {
  uint64_t w = 0;
  if (in_stream8(c0, len)) {
    w = load8(stream + c0);
  } else if (c0 >= 0) {
    const int need = n - __builtin_popcount(bits);
    for (int b = 0; b < need && c0 + b < len; b++) w |= (uint64_t)stream[c0 + b] << (8 * b);
  }
  while (bits) {
    const int e = __builtin_ctz(bits);
    bits &= bits - 1;
    const uint64_t lo = low_bytes(e);
    w = (w & lo) | ((w & ~lo) << 8);
  }
  return w;
}

// MODE 0: compact (dense -> stream); MODE 1: expand (stream -> dense).
// Memory-bound: each code read and written once.  Moving a byte per thread
// and instruction and searching the list per 16 elements took 46 us to
// compact the 16.8 M codes of a 2048 x 8192 weight and 36 us to expand them.
template <int MODE>
__global__ __launch_bounds__(256) void reorder_codes_kernel(const uint8_t* src, int64_t padded, const int64_t* idx,
                                                            int64_t nnz, uint8_t* dst) {
  __shared__ SpanOutliers so;
  const int64_t t0 = (int64_t)blockIdx.x * kSpan;
  const int64_t t1 = min(padded, t0 + kSpan);
  const int64_t lb0 = so.build(idx, nnz, t0, t1);
#pragma unroll
  for (int r = 0; r < kRuns; r++) {
    const int off = (r * 256 + threadIdx.x) * 8;
    const int64_t j0 = t0 + off;
    if (j0 >= t1) break;
    const int n = (int)min((int64_t)8, t1 - j0);
    int pre;
    uint32_t bits = so.run(off, &pre);
    const int64_t c0 = j0 - lb0 - pre;  // the run's first code in the stream
    if (MODE == 1) {
      uint64_t w = stream_codes(src, padded - nnz, c0, bits, n);
      if (n == 8) {
        __builtin_memcpy(dst + j0, &w, 8);
      } else {
        for (int b = 0; b < n; b++) dst[j0 + b] = (uint8_t)(w >> (8 * b));
      }
    } else {
      uint64_t w = 0;
      if (n == 8) {
        w = load8(src + j0);
      } else {
        for (int b = 0; b < n; b++) w |= (uint64_t)src[j0 + b] << (8 * b);
        bits &= (1u << n) - 1u;
      }
      const int left = n - __builtin_popcount(bits);
      // outside the stream only after indices that do not ascend
      if (!in_stream8(c0, padded - nnz) && (c0 < 0 || c0 + left > padded - nnz)) continue;
      while (bits) {  // from the last flagged element down
        const int e = 31 - __builtin_clz(bits);
        bits &= ~(1u << e);
        const uint64_t lo = low_bytes(e);
        w = (w & lo) | ((w >> 8) & ~lo);
      }
      uint8_t* d = dst + c0;
      if (left == 8) {
        __builtin_memcpy(d, &w, 8);
      } else {
        if (left & 4) {
          const uint32_t v = (uint32_t)w;
          __builtin_memcpy(d, &v, 4);
          d += 4;
          w >>= 32;
        }
        if (left & 2) {
          const uint16_t v = (uint16_t)w;
          __builtin_memcpy(d, &v, 2);
          d += 2;
          w >>= 16;
        }
        if (left & 1) *d = (uint8_t)w;
      }
    }
  }
}

// Flat <-> tiled: one thread moves one 16-byte piece (16 consecutive codes of
// a row occupy 16 consecutive bytes in both layouts).
template <int TO_TILED>
__global__ __launch_bounds__(256) void retile_kernel(const uint8_t* src, int64_t N, int64_t K, uint8_t* dst) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p * 16 >= N * K) return;
  const int64_t j = p * 16;
  const int64_t t = tiled_offset(j / K, j % K, K / 128);
  if (TO_TILED)
    *reinterpret_cast<uint4*>(dst + t) = *reinterpret_cast<const uint4*>(src + j);
  else
    *reinterpret_cast<uint4*>(dst + j) = *reinterpret_cast<const uint4*>(src + t);
}

// fp16(value(code) * s) of 8 codes.  Code value and scale are exact fp16
// values: one native fp16 multiply is the single rounding of the exact
// product (and keeps the sign of 0, which a widened multiply fused with a +0
// addend would not).
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
template <int FMT>
__device__ __forceinline__ uint4 dequant8(uint64_t w, uint16_t sbits) {
  const half2v s2 = {bits_to_h(sbits), bits_to_h(sbits)};
  uint32_t r[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t d = (uint32_t)(w >> (32 * (i >> 1)));
    half2v v;
    if (FMT == AQ_FMT_INT8) {
      // 0x6400 | (c ^ 0x80) is the fp16 1024 + (c + 128); subtract 1152
      const uint32_t p = __builtin_amdgcn_perm(0u, d, (i & 1) ? 0x0C030C02u : 0x0C010C00u);
      v = __builtin_bit_cast(half2v, (p ^ 0x00800080u) | 0x64006400u) - (half2v){(f16)1152.0f, (f16)1152.0f};
    } else {
      // codes in the high bytes: sign stays, exponent and mantissa one down, then 2^8 (e4m3_to_h, two at a time)
      const uint32_t p = __builtin_amdgcn_perm(0u, d, (i & 1) ? 0x030C020Cu : 0x010C000Cu);
      v = __builtin_bit_cast(half2v, ((p >> 1) & 0x3F803F80u) | (p & 0x80008000u)) * (half2v){(f16)256.0f, (f16)256.0f};
    }
    r[i] = __builtin_bit_cast(uint32_t, v * s2);
  }
  return make_uint4(r[0], r[1], r[2], r[3]);
}

// The same for a run of n codes that starts `in` elements into block b of G
// and may reach into the blocks behind it.
template <int FMT>
__device__ __forceinline__ uint4 dequant_run(uint64_t w, const uint16_t* scales, int64_t b, int64_t in, int n,
                                             int64_t G) {
  const uint4 v = dequant8<FMT>(w, scales[b]);
  if (in + n <= G) return v;
  uint32_t o[4] = {v.x, v.y, v.z, v.w};
  for (int e = 1; e < n; e++) {
    const int64_t be = (in + e) / G;
    if (be == 0) continue;
    const uint4 u = dequant8<FMT>(w, scales[b + be]);
    const uint32_t uw[4] = {u.x, u.y, u.z, u.w};
    const uint32_t m = 0xFFFFu << (16 * (e & 1));
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (i == e >> 1) o[i] = (o[i] & ~m) | (uw[i] & m);
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// 8 fp16 to out + j: one 16-byte store when whole and aligned.
__device__ __forceinline__ void store_run(uint16_t* out, int64_t j, int n, bool aligned, uint4 v) {
  if (n == 8 && aligned) {
    *reinterpret_cast<uint4*>(out + j) = v;
    return;
  }
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int e = 0; e < 8; e++)
    if (e < n) out[j + e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
}

// Flat codes: dense (STREAM = 0; the outliers are scattered by a second
// kernel) or the compacted int8 stream (STREAM = 1), whose outliers the
// thread that owns their run stores behind it.  Memory-bound: one pass over
// codes and output.  The 16.8 M codes of an int8 8192 x 2048 weight from its
// stream: 12.5 us a call, 4.0 TB/s; 49.7 us as an expansion into dense codes,
// a dequantize kernel of 16 elements and 32 scattered bytes a thread, and a
// scatter.
template <int FMT, int STREAM>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* codes, const uint16_t* scales, int64_t numel,
                                                      int64_t padded, int64_t G, int gshift, uint16_t* out,
                                                      int aligned, const int64_t* idx, const uint16_t* vals,
                                                      int64_t nnz) {
  __shared__ SpanOutliers so;
  const int64_t t0 = (int64_t)blockIdx.x * kSpan;
  const int64_t t1 = min(padded, t0 + kSpan);
  int64_t lb0 = 0;
  if (STREAM) lb0 = so.build(idx, nnz, t0, t1);
  const int64_t b0 = gshift >= 0 ? t0 >> gshift : t0 / G;  // the span's first block
  const int64_t rem0 = t0 - b0 * G;
  const bool g32 = G < ((int64_t)1 << 31);  // block numbers inside the span by 32-bit division
#pragma unroll
  for (int r = 0; r < kRuns; r++) {
    const int off = (r * 256 + threadIdx.x) * 8;
    const int64_t j0 = t0 + off;
    if (j0 >= numel) break;
    const int n = (int)min((int64_t)8, numel - j0);
    uint64_t w = 0;
    uint32_t bits = 0;
    int pre = 0;
    if (STREAM) {
      bits = so.run(off, &pre);
      const int64_t c0 = j0 - lb0 - pre;
      w = stream_codes(codes, padded - nnz, c0, bits, (int)min((int64_t)8, padded - j0));
    } else if (n == 8) {
      w = load8(codes + j0);
    } else {
      for (int b = 0; b < n; b++) w |= (uint64_t)codes[j0 + b] << (8 * b);
    }
    const int64_t rel = rem0 + off;
    const int64_t q = gshift >= 0 ? rel >> gshift : g32 ? (int64_t)((uint32_t)rel / (uint32_t)G) : rel / G;
    const int64_t in = rel - q * G;  // the run's place in its block
    store_run(out, j0, n, aligned, dequant_run<FMT>(w, scales, b0 + q, in, n, G));
    if (STREAM) {
      int64_t p = lb0 + pre;
      for (; bits; bits &= bits - 1, p++) {
        const int e = __builtin_ctz(bits);
        if (e < n) out[j0 + e] = vals[p];
      }
    }
  }
}

// Tiled codes: a wave takes whole tiles of 16 rows x 128 columns.  16 lanes
// cover a row's 128 columns in runs of 8, so that a store instruction writes
// 256 contiguous bytes of four rows and reads 64-byte pieces of the tile's
// eight 256-byte groups; kTilesPerWave tiles have their loads in flight
// together.  Neighbouring waves take neighbouring tiles of the tile row.
// Memory-bound: 14336 x 4096 in blocks of 128 29.3 us, 6.1 TB/s of codes and
// output (81.7 us with 16 consecutive elements a thread, whose 16-byte loads
// each touch a line of their own, and two 64-bit divisions per 16).
// ROWS: blocks of a multiple of 8 divide the rows (every weight quantized
// into this layout), so a run has one scale, at kg per row; otherwise the
// blocks go on over the flat elements.
constexpr int kTilesPerWave = 2;
template <int FMT, int ROWS>
__global__ __launch_bounds__(256) void dequant_tiled_kernel(const uint8_t* codes, const uint16_t* scales, int64_t K,
                                                            int nchunks, int bands, int64_t G, int gshift, int64_t kg,
                                                            uint16_t* out, int aligned) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t rb = blockIdx.x / (unsigned)bands;
  const int c0 = (int)(blockIdx.x % (unsigned)bands) * 4 * kTilesPerWave + wave;
  const int col = 8 * (lane & 15);
  const int rl = lane >> 4;  // row 4 i + rl of the tile in step i
  const int at = ((col >> 6) << 10) + (((col >> 4) & 3) << 8) + (col & 8);  // the run's place in a tile, for row 0
  uint64_t w[kTilesPerWave][4];
  uint16_t sc[kTilesPerWave][4];
#pragma unroll
  for (int j = 0; j < kTilesPerWave; j++) {
    const int c = min(c0 + 4 * j, nchunks - 1);
    const uint8_t* tile = codes + ((rb * nchunks + c) << 11) + at;
    const unsigned k = (unsigned)c * 128 + col;
    const unsigned kb = !ROWS ? 0 : gshift >= 0 ? k >> gshift : k / (unsigned)G;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int row = 4 * i + rl;
      w[j][i] = *reinterpret_cast<const uint64_t*>(tile + row * 16);
      sc[j][i] = ROWS ? scales[(rb * 16 + row) * kg + kb] : (uint16_t)0;
    }
  }
#pragma unroll
  for (int j = 0; j < kTilesPerWave; j++) {
    const int c = c0 + 4 * j;
    if (c >= nchunks) break;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int64_t e = (rb * 16 + 4 * i + rl) * K + (int64_t)c * 128 + col;
      store_run(out, e, 8, aligned,
                ROWS ? dequant8<FMT>(w[j][i], sc[j][i]) : dequant_run<FMT>(w[j][i], scales, e / G, e % G, 8, G));
    }
  }
}

__global__ __launch_bounds__(256) void scatter_outliers_kernel(const int64_t* idx, const uint16_t* vals, int64_t nnz,
                                                               int64_t numel, uint16_t* out) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= nnz) return;
  const int64_t j = idx[p];
  if (j >= 0 && j < numel) out[j] = vals[p];
}

using aq::block_position;
using aq::lower_bound_i32;
using aq::raise_to;

// One workgroup per tile row (aq_tiles.h); workgroup nrb writes the list's
// end and the 64 padding entries.  LDS: 33 * nch ints.
__global__ __launch_bounds__(256) void outlier_tile_rows_kernel(const int32_t* row_ptr, int64_t rstride,
                                                                const int32_t* cols, const uint16_t* vals, int nrb,
                                                                int nch, int32_t* tile_ptr, uint32_t* tile_ent,
                                                                int32_t* tile_max) {
  extern __shared__ int sm[];
  __shared__ int part[4];
  const int rb = blockIdx.x, t = threadIdx.x;
  if (rb == nrb) {
    const int end = row_ptr[(int64_t)nrb * 16 * rstride];
    if (t == 0) tile_ptr[(int64_t)nrb * nch] = end;
    if (t < 64) tile_ent[end + t] = 0u;
    return;
  }
  aq::CsrTileSrc src;
#pragma unroll
  for (int r = 0; r <= 16; r++) src.rs[r] = row_ptr[(int64_t)(rb * 16 + r) * rstride];
  src.cols = cols;
  src.vals = vals;
  aq::tile_row_sort<256, 4>(src, rb, nch, src.rs[0], src.rs[16], sm, part, tile_ptr, tile_ent, tile_max);
}

constexpr int kTileMaxWG = 32;  // workgroups a list
__global__ __launch_bounds__(256) void tile_max_kernel(aq::TileMaxGroup g) {
  __shared__ int part[4];
  const int m = blockIdx.x / kTileMaxWG;
  const int32_t* p = nullptr;
  int32_t* out = nullptr;
  int64_t n = 0;
#pragma unroll
  for (int j = 0; j < aq::kMaxTileMax; j++)
    if (j == m) {
      p = g.tile_ptr[j];
      n = g.n[j];
      out = g.tile_max[j];
    }
  if (!out) return;
  int mx = 0;
  // eight blocks a thread and round, their loads in flight together
  for (int64_t i0 = (int64_t)(blockIdx.x % kTileMaxWG) * 2048 + threadIdx.x; i0 < n; i0 += 2048 * kTileMaxWG) {
    int lo[8], hi[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int64_t i = min(i0 + 256 * k, n - 1);
      lo[k] = p[i];
      hi[k] = p[i + 1];
    }
#pragma unroll
    for (int k = 0; k < 8; k++) mx = max(mx, hi[k] - lo[k]);
  }
  for (int d = 32; d >= 1; d >>= 1) mx = max(mx, __shfl_xor(mx, d));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    mx = max(max(part[0], part[1]), max(part[2], part[3]));
    if (mx > 0) raise_to(out, mx);
  }
}

// One thread per block of 16 rows x 64 columns (tile row rb, chunk c), for
// rows wider than outlier_tile_rows_kernel takes.  Entries are ordered by
// block, then row, then column, so a block starts after every outlier of
// the rows above it plus, in each of its own rows, the outliers left of
// column 64c.
__global__ __launch_bounds__(256) void outlier_tiles_kernel(const int32_t* row_ptr, int64_t rstride,
                                                            const int32_t* cols, const uint16_t* vals, int nrb,
                                                            int nch, int32_t* tile_ptr, uint32_t* tile_ent,
                                                            int32_t* tile_max) {
  const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t nblk = (int64_t)nrb * nch;
  if (b > nblk) return;
  if (b == nblk) {
    const int end = row_ptr[(int64_t)nrb * 16 * rstride];
    tile_ptr[b] = end;
    for (int k = 0; k < 64; k++) tile_ent[end + k] = 0u;
    return;
  }
  const int rb = (int)(b / nch), c = (int)(b % nch);
  if (c == 0 && tile_max) {
    int mx = 0;
    for (int cc = 0; cc < nch; cc++) {
      int n = 0;
      for (int r = 0; r < 16; r++) {
        const int p0 = row_ptr[(int64_t)(rb * 16 + r) * rstride], p1 = row_ptr[(int64_t)(rb * 16 + r + 1) * rstride];
        n += lower_bound_i32(cols, p0, p1, cc * 64 + 64) - lower_bound_i32(cols, p0, p1, cc * 64);
      }
      mx = max(mx, n);
    }
    if (mx > 0) raise_to(tile_max, mx);
  }
  int lo[16], hi[16];
  int pos = row_ptr[(int64_t)rb * 16 * rstride];
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int p0 = row_ptr[(int64_t)(rb * 16 + r) * rstride], p1 = row_ptr[(int64_t)(rb * 16 + r + 1) * rstride];
    lo[r] = lower_bound_i32(cols, p0, p1, c * 64);
    hi[r] = lower_bound_i32(cols, lo[r], p1, c * 64 + 64);
    pos += lo[r] - p0;
  }
  tile_ptr[b] = pos;
#pragma unroll
  for (int r = 0; r < 16; r++)
    for (int p = lo[r]; p < hi[r]; p++)
      tile_ent[pos++] = ((uint32_t)vals[p] << 16) | block_position(r, cols[p] - c * 64);
}

}  // namespace

extern "C" int aq_segment_offsets(const int64_t* flat_idx, int64_t nnz, int64_t nseg, int64_t seg_len,
                                  int32_t* seg_ptr, void* stream) {
  AQ_CHECK_ARG(nnz >= 0 && nseg >= 0 && seg_len >= 1, "aq_segment_offsets: bad sizes");
  AQ_CHECK_ARG(seg_ptr && (nnz == 0 || flat_idx), "aq_segment_offsets: null pointer argument");
  AQ_CHECK_ARG(nnz < ((int64_t)1 << 31), "aq_segment_offsets: nnz exceeds int32");
  const int64_t grid = aq::ceil_div(nseg + 1, 256);
  hipLaunchKernelGGL(segment_offsets_kernel, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, flat_idx, nnz,
                     nseg, seg_len, seg_ptr);
  AQ_LAUNCH_CHECK("aq_segment_offsets: launch");
  return AQ_OK;
}

extern "C" int aq_outlier_cols(const int64_t* flat_idx, int64_t nnz, int64_t K, int32_t* cols, void* stream) {
  AQ_CHECK_ARG(nnz >= 0 && K >= 1, "aq_outlier_cols: bad sizes");
  if (nnz == 0) return AQ_OK;
  AQ_CHECK_ARG(flat_idx && cols, "aq_outlier_cols: null pointer argument");
  hipLaunchKernelGGL(outlier_cols_kernel, dim3((unsigned)aq::ceil_div(nnz, 256)), dim3(256), 0, (hipStream_t)stream,
                     flat_idx, nnz, K, cols);
  AQ_LAUNCH_CHECK("aq_outlier_cols: launch");
  return AQ_OK;
}

static int reorder(int mode, const void* src, int64_t padded, const int64_t* idx, int64_t nnz, void* dst,
                   void* stream, const char* name) {
  AQ_CHECK_ARG(padded >= 0 && nnz >= 0 && nnz <= padded, "%s: bad sizes", name);
  if (padded == 0) return AQ_OK;
  AQ_CHECK_ARG(dst && (nnz == padded || src) && (nnz == 0 || idx), "%s: null pointer argument", name);
  const int64_t grid = aq::ceil_div(padded, kSpan);
  if (mode == 0)
    hipLaunchKernelGGL((reorder_codes_kernel<0>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream,
                       (const uint8_t*)src, padded, idx, nnz, (uint8_t*)dst);
  else
    hipLaunchKernelGGL((reorder_codes_kernel<1>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream,
                       (const uint8_t*)src, padded, idx, nnz, (uint8_t*)dst);
  AQ_LAUNCH_CHECK(name);
  return AQ_OK;
}

extern "C" int aq_compact_codes(const void* dense, int64_t padded, const int64_t* flat_idx, int64_t nnz,
                                void* compact, void* stream) {
  if (padded == nnz) return AQ_OK;  // every element is an outlier: empty stream
  return reorder(0, dense, padded, flat_idx, nnz, compact, stream, "aq_compact_codes");
}

extern "C" int aq_expand_codes(const void* compact, int64_t padded, const int64_t* flat_idx, int64_t nnz,
                               void* dense, void* stream) {
  return reorder(1, compact, padded, flat_idx, nnz, dense, stream, "aq_expand_codes");
}

static int retile(int to_tiled, const void* src, int64_t N, int64_t K, void* dst, void* stream, const char* name) {
  AQ_CHECK_ARG(N >= 0 && K >= 128 && N % 16 == 0 && K % 128 == 0,
               "%s: needs N %% 16 == 0 and K %% 128 == 0 (N=%lld, K=%lld)", name, (long long)N, (long long)K);
  if (N == 0) return AQ_OK;
  AQ_CHECK_ARG(src && dst && (uintptr_t)src % 16 == 0 && (uintptr_t)dst % 16 == 0,
               "%s: null or unaligned pointer", name);
  const int64_t grid = aq::ceil_div(N * K / 16, 256);
  if (to_tiled)
    hipLaunchKernelGGL((retile_kernel<1>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream,
                       (const uint8_t*)src, N, K, (uint8_t*)dst);
  else
    hipLaunchKernelGGL((retile_kernel<0>), dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream,
                       (const uint8_t*)src, N, K, (uint8_t*)dst);
  AQ_LAUNCH_CHECK(name);
  return AQ_OK;
}

extern "C" int aq_tile_codes(const void* flat, int64_t N, int64_t K, void* tiled, void* stream) {
  return retile(1, flat, N, K, tiled, stream, "aq_tile_codes");
}

extern "C" int aq_untile_codes(const void* tiled, int64_t N, int64_t K, void* flat, void* stream) {
  return retile(0, tiled, N, K, flat, stream, "aq_untile_codes");
}

static int log2_of(int64_t g) {
  if (g <= 0 || (g & (g - 1))) return -1;
  return __builtin_ctzll((uint64_t)g);
}

template <int FMT>
static void launch_dequant(const void* codes, const void* scales, int64_t numel, int64_t G, int64_t K, int tiled,
                           void* out, hipStream_t s) {
  const int aligned = (uintptr_t)out % 16 == 0;
  const uint8_t* c = (const uint8_t*)codes;
  const uint16_t* sc = (const uint16_t*)scales;
  if (tiled) {
    const int64_t nch = K / 128, bands = aq::ceil_div(nch, 4 * kTilesPerWave);
    const dim3 grid((unsigned)(numel / (16 * K) * bands));
    if (G % 8 == 0 && K % G == 0 && K < ((int64_t)1 << 31))
      hipLaunchKernelGGL((dequant_tiled_kernel<FMT, 1>), grid, dim3(256), 0, s, c, sc, K, (int)nch, (int)bands, G,
                         log2_of(G), K / G, (uint16_t*)out, aligned);
    else
      hipLaunchKernelGGL((dequant_tiled_kernel<FMT, 0>), grid, dim3(256), 0, s, c, sc, K, (int)nch, (int)bands, G,
                         log2_of(G), (int64_t)0, (uint16_t*)out, aligned);
  } else {
    const int64_t padded = aq::ceil_div(numel, G) * G;
    hipLaunchKernelGGL((dequant_kernel<FMT, 0>), dim3((unsigned)aq::ceil_div(numel, kSpan)), dim3(256), 0, s, c, sc,
                       numel, padded, G, log2_of(G), (uint16_t*)out, aligned, (const int64_t*)nullptr,
                       (const uint16_t*)nullptr, (int64_t)0);
  }
}

extern "C" int aq_dequantize(const void* codes, const void* scales, int64_t numel, int64_t G, int fmt, int64_t K,
                             int layout, const int64_t* flat_idx, const void* vals, int64_t nnz, void* out,
                             void* stream) {
  AQ_CHECK_ARG(numel >= 0 && G >= 1 && nnz >= 0, "aq_dequantize: bad sizes");
  AQ_CHECK_ARG(fmt == AQ_FMT_INT8 || fmt == AQ_FMT_E4M3, "aq_dequantize: unknown code format %d", fmt);
  AQ_CHECK_ARG(layout == AQ_LAYOUT_FLAT || layout == AQ_LAYOUT_TILED, "aq_dequantize: unknown layout %d", layout);
  if (numel == 0) return AQ_OK;
  AQ_CHECK_ARG(codes && scales && out && (nnz == 0 || (flat_idx && vals)), "aq_dequantize: null pointer argument");
  const int tiled = layout == AQ_LAYOUT_TILED;
  if (tiled)
    AQ_CHECK_ARG(K >= 128 && K % 128 == 0 && numel % (16 * K) == 0 && (uintptr_t)codes % 16 == 0,
                 "aq_dequantize: tiled codes need K %% 128 == 0 and rows %% 16 == 0");
  hipStream_t s = (hipStream_t)stream;
  if (fmt == AQ_FMT_INT8)
    launch_dequant<AQ_FMT_INT8>(codes, scales, numel, G, K, tiled, out, s);
  else
    launch_dequant<AQ_FMT_E4M3>(codes, scales, numel, G, K, tiled, out, s);
  AQ_LAUNCH_CHECK("aq_dequantize: launch");
  if (nnz > 0) {
    hipLaunchKernelGGL(scatter_outliers_kernel, dim3((unsigned)aq::ceil_div(nnz, 256)), dim3(256), 0, s, flat_idx,
                       (const uint16_t*)vals, nnz, numel, (uint16_t*)out);
    AQ_LAUNCH_CHECK("aq_dequantize: scatter launch");
  }
  return AQ_OK;
}

extern "C" int aq_dequantize_stream(const void* stream_codes, const void* scales, int64_t numel, int64_t G,
                                    const int64_t* flat_idx, const void* vals, int64_t nnz, void* out, void* stream) {
  AQ_CHECK_ARG(numel >= 0 && G >= 1 && nnz >= 0, "aq_dequantize_stream: bad sizes");
  if (numel == 0) return AQ_OK;
  const int64_t padded = aq::ceil_div(numel, G) * G;
  AQ_CHECK_ARG(nnz <= padded, "aq_dequantize_stream: %lld outliers of %lld elements", (long long)nnz,
               (long long)padded);
  AQ_CHECK_ARG((stream_codes || nnz == padded) && scales && out && (nnz == 0 || (flat_idx && vals)),
               "aq_dequantize_stream: null pointer argument");
  hipLaunchKernelGGL((dequant_kernel<AQ_FMT_INT8, 1>), dim3((unsigned)aq::ceil_div(numel, kSpan)), dim3(256), 0,
                     (hipStream_t)stream, (const uint8_t*)stream_codes, (const uint16_t*)scales, numel, padded, G,
                     log2_of(G), (uint16_t*)out, (int)((uintptr_t)out % 16 == 0), flat_idx, (const uint16_t*)vals,
                     nnz);
  AQ_LAUNCH_CHECK("aq_dequantize_stream: launch");
  return AQ_OK;
}

hipError_t aq::launch_tile_max(const TileMaxGroup& g, int count, hipStream_t stream) {
  hipLaunchKernelGGL(tile_max_kernel, dim3((unsigned)(count * kTileMaxWG)), dim3(256), 0, stream, g);
  return hipGetLastError();
}

hipError_t aq::launch_outlier_tiles(const int32_t* row_ptr, int64_t rstride, const int32_t* cols, const uint16_t* vals,
                                    int64_t N, int64_t K, int32_t* tile_ptr, uint32_t* tile_ent, int32_t* tile_max,
                                    hipStream_t stream) {
  const int64_t nblk = (N / 16) * (K / 64);
  if (K / 64 <= aq::kTileRowsMaxChunks) {
    const bool raise = N / 16 <= aq::kRaiseTileRows;
    hipLaunchKernelGGL(outlier_tile_rows_kernel, dim3((unsigned)(N / 16 + 1)), dim3(256),
                       (size_t)33 * (K / 64) * sizeof(int), stream, row_ptr, rstride, cols, vals, (int)(N / 16),
                       (int)(K / 64), tile_ptr, tile_ent, raise ? tile_max : nullptr);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || !tile_max || raise) return e;
    TileMaxGroup g{};
    g.tile_ptr[0] = tile_ptr;
    g.n[0] = nblk;
    g.tile_max[0] = tile_max;
    return launch_tile_max(g, 1, stream);
  }
  hipLaunchKernelGGL(outlier_tiles_kernel, dim3((unsigned)aq::ceil_div(nblk + 1, 256)), dim3(256), 0, stream, row_ptr,
                     rstride, cols, vals, (int)(N / 16), (int)(K / 64), tile_ptr, tile_ent, tile_max);
  return hipGetLastError();
}

extern "C" int aq_outlier_tiles(const int32_t* row_ptr, const int32_t* cols, const void* vals, int64_t N, int64_t K,
                                int32_t* tile_ptr, uint32_t* tile_ent, int32_t* tile_max, void* stream) {
  AQ_CHECK_ARG(N >= 16 && N % 16 == 0 && K >= 64 && K % 64 == 0 && N < (1 << 30) && K < (1 << 30) &&
                   (N / 16) * (K / 64) < ((int64_t)1 << 31),
               "aq_outlier_tiles: N must be a multiple of 16 and K of 64 (N=%lld K=%lld)", (long long)N,
               (long long)K);
  AQ_CHECK_ARG(row_ptr && tile_ptr, "aq_outlier_tiles: null pointer argument");
  const hipError_t e = aq::launch_outlier_tiles(row_ptr, 1, cols, (const uint16_t*)vals, N, K, tile_ptr, tile_ent,
                                                tile_max, (hipStream_t)stream);
  if (e != hipSuccess) return aq::check_hip(e, "aq_outlier_tiles: launch");
  return AQ_OK;
}
