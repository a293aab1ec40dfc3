// aq_qlinear_mid.hip -- the quantized linear for a large decode batch (33 to
// 64 rows of x) on short and on tall grids.  The weights are still what costs
// (1 byte a weight against 2 M flops), but x no longer fits beside every wave
// as in the GEMVs (aq_qlinear.hip): staged through registers for 8 waves it
// left room for 4 waves per tile row only, which on N = 4096 occupied half
// the CUs.
//
// A workgroup of 4 waves takes 128 output columns, each wave two 16-row tile
// rows of W, over a part of K.  Codes go from HBM straight to registers in
// MFMA operand order (the tiled layout), kMidAhead chunks of 128 columns
// ahead, and are decoded there; x goes to LDS by direct loads (no registers,
// no LDS write instructions), a chunk shared by the four waves, its 16-byte
// pieces placed so that the 16 rows of a fragment read fall on 16 different
// bank groups; each fragment feeds both tile rows.  Outliers come from the
// block lists, multiplied by one more MFMA per chunk and row group (x columns
// gathered from LDS against the values).  One barrier a chunk, which waits
// only for the x of the next chunk.
//
// K is split over workgroups until they fill the CUs (mid_split); the parts (or
// the one part) leave fp32 partial sums in the caller's workspace and
// mid_reduce_kernel adds them in order, with the bias and the decode epilogue,
// and puts right what an infinite x does to this kernel's sums.
//
// Bound by instruction issue, not bytes: gate+up [28672, 4096] at M = 64 takes
// 39 us for 119 MB.  A wave's step is 259 vector instructions (1061 cycles;
// decoding and the outliers' addresses and selects the most of them), 40 MFMAs
// (644) and 32 LDS reads; a third of its time it waits to issue, a third for
// memory or the barrier (profiles/qlinear_mid_llama3_8b_m64_counters.txt).
#include <algorithm>

#include "aq_common.h"
#include "aq_qlinear_internal.h"
#include "aq_tiles.h"

namespace {

using namespace aqk;

constexpr int kMidWaves = 4;
constexpr int kMidAhead = 2;  // chunks whose codes are in flight per wave
constexpr int kMidSlots = 2;  // outlier slots a lane whose entries travel with the codes (8 entries a chunk)
typedef _Float16 half4 __attribute__((ext_vector_type(4)));

// fp16 output o of row m, column n: ReLU, then the residual added in fp16.
__device__ __forceinline__ uint16_t mid_epilogue(f16 o, int act, uint16_t res, bool has_res) {
  if (act == 1 && (float)o < 0.0f) o = (f16)0.0f;
  if (has_res) o = rn_h((float)bits_to_h(res) + (float)o);
  return h_to_bits(o);
}

// A wave's share of one chunk of x straight into LDS: mg loads of 1 KiB, lane
// l's 16 bytes from xo[i] + at to dst + i KiB + 16 l.
struct MidX {
  __amdgpu_buffer_rsrc_t xr;
  uint32_t xo[8];
};
__device__ __forceinline__ void mid_load_x(const MidX& X, uint8_t* dst, uint32_t at, int mg) {
#pragma unroll
  for (int i = 0; i < 8; i++)
    if (i < mg)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(X.xr, (void*)(dst + i * 1024), 16,
                                               at == kOutOfRange ? at : X.xo[i] + at, 0, 0, 0);
}

// MG: groups of 16 rows of x.  PAIR: matrices 0 and 1 are gate and up; a
// wave's two tile rows are the same rows of each, and the output is
// fp16(fp16(silu(g)) u).
template <int FMT, int PC, int MG, int PAIR>
__global__ __launch_bounds__(64 * kMidWaves, 2) void qlinear_mid_kernel(QLArgs a) {
  constexpr int ST = 3;              // stages of x
  constexpr int XB = MG * 16 * 256;    // bytes of a stage: rows of 128 fp16
  __shared__ __attribute__((aligned(16))) uint8_t xs[ST * XB];

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int grp = lane >> 4, li = lane & 15;
  const int M = a.M, K = a.K;
  const int nch = K >> 7, nb64 = K >> 6;
  // units of all matrices in one list, the parts of K outermost
  const int nunits = a.first[a.count];
  const int part = (int)blockIdx.x / nunits, unit = (int)blockIdx.x % nunits;
  int mi = 0;
#pragma unroll
  for (int j = 1; j < kMaxGroup; j++)
    if (j < a.count && unit >= a.first[j]) mi = j;
  const QLMat W = pick(a, PAIR ? 0 : mi);
  const QLMat W1 = PAIR ? a.mat[1] : W;
  const int nrb = W.N / 16;
  const int u = unit - a.first[PAIR ? 0 : mi];
  const int rb0 = PAIR ? u * kMidWaves + wave : (u * kMidWaves + wave) * 2;
  const int rb1 = PAIR ? rb0 : rb0 + 1;
  const int c_first = (int)((int64_t)nch * part / a.split), c_end = (int)((int64_t)nch * (part + 1) / a.split);

  // Tile rows past the matrix: empty ranges, every load reads zero.
  const QLMat* const Ws[2] = {&W, &W1};
  const int rbs[2] = {rb0, rb1};
  __amdgpu_buffer_rsrc_t cr[2], sr[2], tr[2], er[2];
  uint16_t sb_row[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const bool in = rbs[i] < nrb;
    const int rb = in ? rbs[i] : 0;
    cr[i] = __builtin_amdgcn_make_buffer_rsrc((void*)(Ws[i]->codes + ((size_t)rb * nch << 11)), (short)0,
                                              in ? nch * 2048 : 0, kBufferDword3);
    sr[i] = __builtin_amdgcn_make_buffer_rsrc((void*)(Ws[i]->scales + (size_t)rb * 16 * Ws[i]->kg), (short)0,
                                              in ? 16 * Ws[i]->kg * 2 : 0, kBufferDword3);
    tr[i] = __builtin_amdgcn_make_buffer_rsrc((void*)(Ws[i]->tptr + (size_t)rb * nb64), (short)0,
                                              in ? (nb64 + 1) * 4 : 0, kBufferDword3);
    er[i] = __builtin_amdgcn_make_buffer_rsrc((void*)Ws[i]->tent, (short)0, in ? 0x7FFFFFFF : 0, kBufferDword3);
    sb_row[i] = PC == 1 ? (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(sr[i], li * 2, 0, 0) : (uint16_t)0;
  }
  // x rows past M lie past the end of this range: zeros
  MidX X;
  X.xr = __builtin_amdgcn_make_buffer_rsrc((void*)a.x, (short)0, M * K * 2, kBufferDword3);
  // direct load i of wave w fills stage bytes (MG w + i) KiB + 16 l: row
  // 4 (MG w + i) + l / 16, stored piece l % 16, which holds logical piece
  // (l % 16) ^ (row & 15)
#pragma unroll
  for (int i = 0; i < MG; i++) {
    const int row = 4 * (MG * wave + i) + grp;
    X.xo[i] = (uint32_t)(row * K + 8 * (li ^ (row & 15))) * 2;
  }
  // The part's chunks in order from a start of the workgroup's own (step j
  // takes chunk_of(j); c_end past the last): rows of x lie a multiple of 4 KiB
  // apart for most K, so the same columns of all rows share few L2 channels,
  // and workgroups walking the columns in step would all read from those
  // (gate+up at M = 32 37.9 -> 35.4 us).  The start goes by the tile rows' 128
  // columns, so that a pair sums as its members alone do.
  const int nsteps = c_end - c_first;
  const int rot = ((PAIR ? u >> 1 : u) >> 3) % nsteps;
  auto chunk_of = [&](int j) {
    const int r = j + rot;
    return j < nsteps ? c_first + (r < nsteps ? r : r - nsteps) : c_end;
  };
  // past the part: out of range, the stage is filled with zeros
  auto load_x = [&](int j, int stage) {
    const int c = chunk_of(j);
    mid_load_x(X, xs + stage * XB + MG * wave * 1024, c < c_end ? (uint32_t)c * 256 : kOutOfRange, MG);
  };

  // lane i: first entry, first entry of the second block and end of step
  // g0 + i's chunk of each tile row
  uint32_t rg[2][3];
  auto load_ranges = [&](int g0) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int c = chunk_of(g0 + lane);
      const uint32_t off = c < c_end ? (uint32_t)c * 8 : kOutOfRange;
#pragma unroll
      for (int j = 0; j < 3; j++) rg[i][j] = __builtin_amdgcn_raw_buffer_load_b32(tr[i], off + 4 * j, 0, 0);
    }
  };
  struct Slot {
    u32x4 q[2][2];
    uint32_t s[2][2];
    uint32_t ent[2][kMidSlots];          // entry 4 b + grp of each tile row's chunk (0 past its end)
    int e_start[2], e_mid[2], e_cnt[2];  // wave-uniform
  };
  auto load = [&](Slot& sl, int j) {
    const int c = chunk_of(j);
    const uint32_t co = c < c_end ? (uint32_t)(c * 2048 + lane * 16) : kOutOfRange;
    const int gl = j & 63;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      // codes are read once per call: non-temporal
      sl.q[i][0] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(cr[i], co, 0, 2));
      sl.q[i][1] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(cr[i], co + 1024, 0, 2));
      if (PC != 1) {
        const uint32_t k = (uint32_t)(c < c_end ? c : c_first) * 128 + (PC == 2 ? 0 : 16 * grp);
        const int gs = Ws[i]->gshift, G = Ws[i]->G;
        const uint32_t k0 = gs >= 0 ? k >> gs : k / G;
        sl.s[i][0] = __builtin_amdgcn_raw_buffer_load_b16(sr[i], ((uint32_t)li * Ws[i]->kg + k0) * 2, 0, 0);
        if (PC == 0) {
          const uint32_t k1 = gs >= 0 ? (k + 64) >> gs : (k + 64) / G;
          sl.s[i][1] = __builtin_amdgcn_raw_buffer_load_b16(sr[i], ((uint32_t)li * Ws[i]->kg + k1) * 2, 0, 0);
        }
      }
      const int e0 = __builtin_amdgcn_readlane((int)rg[i][0], gl);
      sl.e_start[i] = e0;
      sl.e_mid[i] = __builtin_amdgcn_readlane((int)rg[i][1], gl) - e0;
      sl.e_cnt[i] = __builtin_amdgcn_readlane((int)rg[i][2], gl) - e0;
#pragma unroll
      for (int b = 0; b < kMidSlots; b++) {
        const int e = 4 * b + grp;
        sl.ent[i][b] =
            __builtin_amdgcn_raw_buffer_load_b32(er[i], e < sl.e_cnt[i] ? (uint32_t)(e0 + e) * 4 : kOutOfRange, 0, 0);
      }
    }
  };

  float4v acc[2][MG];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int gi = 0; gi < MG; gi++) acc[i][gi] = (float4v){0.f, 0.f, 0.f, 0.f};

  // Outliers of one tile row's chunk, 4 kMidSlots entries at a time as k slots
  // of one MFMA per row group: slot (grp, b) holds entry base + 4 b + grp, its
  // A operand the entry's x column, its B operand the value in the column of
  // its row and zero elsewhere.
  struct Outl {
    half4 bv;
    half4 av[MG];
  };
  auto gather = [&](Outl& o, const uint32_t (&ent)[kMidSlots], int base, int e_mid, int e_cnt, const uint8_t* xb) {
    o.bv = (half4){};
#pragma unroll
    for (int gi = 0; gi < MG; gi++) o.av[gi] = (half4){};
#pragma unroll
    for (int b = 0; b < kMidSlots; b++) {
      const int e = base + 4 * b + grp;
      const bool valid = e < e_cnt;
      const int k = (int)(ent[b] & 63u) + (e >= e_mid ? 64 : 0);
      o.bv[b] = valid && (int)((ent[b] >> 6) & 15u) == li ? bits_to_h((uint16_t)(ent[b] >> 16)) : (f16)0.0f;
      // row 16 gi + li, column k
      const uint8_t* xp = xb + li * 256 + ((((k >> 3) ^ li) << 4) | ((k & 7) << 1));
#pragma unroll
      for (int gi = 0; gi < MG; gi++) {
        const f16 xv = bits_to_h(*reinterpret_cast<const uint16_t*>(xp + gi * 16 * 256));
        o.av[gi][b] = valid ? xv : (f16)0.0f;
      }
    }
  };
  auto add = [&](int i, const Outl& o) {
#pragma unroll
    for (int gi = 0; gi < MG; gi++)
      acc[i][gi] = __builtin_amdgcn_mfma_f32_16x16x16f16(o.av[gi], o.bv, acc[i][gi], 0, 0, 0);
  };
  // entries past the ones that came with the codes
  auto add_rest = [&](int i, int e_start, int e_mid, int e_cnt, const uint8_t* xb) {
    for (int base = 4 * kMidSlots; base < e_cnt; base += 4 * kMidSlots) {
      uint32_t ent[kMidSlots];
#pragma unroll
      for (int b = 0; b < kMidSlots; b++) {
        const int e = base + 4 * b + grp;
        ent[b] = __builtin_amdgcn_raw_buffer_load_b32(er[i], e < e_cnt ? (uint32_t)(e_start + e) * 4 : kOutOfRange, 0, 0);
      }
      Outl o;
      gather(o, ent, base, e_mid, e_cnt, xb);
      add(i, o);
    }
    // its loads are done: left pending, every step would carry their wait
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  };

  // the pieces of a fragment read: row li of a group, columns 16 grp + {0, 8, 64, 72}
  uint32_t fo[4];
#pragma unroll
  for (int q = 0; q < 4; q++) fo[q] = li * 256 + (((2 * grp + (q & 1) + 8 * (q >> 1)) ^ li) << 4);

  auto step = [&](Slot& sl, int j, const uint8_t* xb) {
    half8 w[2][4];
    uint32_t ent[2][kMidSlots];
    int es[2], em[2], ec[2];
    half8 xf[2][MG];
    auto frags = [&](half8 (&f)[MG], int q) {
#pragma unroll
      for (int gi = 0; gi < MG; gi++) f[gi] = *reinterpret_cast<const half8*>(xb + gi * 16 * 256 + fo[q]);
    };
    frags(xf[0], 0);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const half2v s0 = scale2(PC == 1 ? sb_row[i] : (uint16_t)sl.s[i][0]);
      const half2v s1 = PC == 0 ? scale2((uint16_t)sl.s[i][1]) : s0;
      w[i][0] = deq8<FMT>(sl.q[i][0].x, sl.q[i][0].y, s0);
      w[i][1] = deq8<FMT>(sl.q[i][0].z, sl.q[i][0].w, s0);
      w[i][2] = deq8<FMT>(sl.q[i][1].x, sl.q[i][1].y, s1);
      w[i][3] = deq8<FMT>(sl.q[i][1].z, sl.q[i][1].w, s1);
#pragma unroll
      for (int b = 0; b < kMidSlots; b++) ent[i][b] = sl.ent[i][b];
      es[i] = sl.e_start[i];
      em[i] = sl.e_mid[i];
      ec[i] = sl.e_cnt[i];
    }
    __builtin_amdgcn_sched_barrier(0);
    load(sl, j + kMidAhead);
    __builtin_amdgcn_sched_barrier(0);
    // fragments one k-step ahead of their MFMAs, the outliers' x behind the
    // last (left alone, the compiler reads each next to its use)
    Outl o[2];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if (q < 3) {
        frags(xf[(q + 1) & 1], q + 1);
      } else {
#pragma unroll
        for (int i = 0; i < 2; i++) gather(o[i], ent[i], 0, em[i], ec[i], xb);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int gi = 0; gi < MG; gi++) {
        acc[0][gi] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[q & 1][gi], w[0][q], acc[0][gi], 0, 0, 0);
        acc[1][gi] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[q & 1][gi], w[1][q], acc[1][gi], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
      add(i, o[i]);
      if (ec[i] > 4 * kMidSlots) add_rest(i, es[i], em[i], ec[i], xb);
    }
  };

  Slot slots[kMidAhead];
  load_ranges(0);
#pragma unroll
  for (int s = 0; s < ST - 1; s++) load_x(s, s);
#pragma unroll
  for (int s = 0; s < kMidAhead; s++) load(slots[s], s);
  // the newest loads of one step: the next x (if its stage is filled this
  // step) and one slot's codes, scales and entries
  constexpr int kSlotLoads = 2 * (2 + (PC == 1 ? 0 : PC == 2 ? 1 : 2) + kMidSlots);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  int cur = 0;  // stage of step j
  for (int j0 = 0; j0 < nsteps; j0 += kMidAhead) {
#pragma unroll
    for (int s = 0; s < kMidAhead; s++) {
      const int j = j0 + s;
      // the stage of step j - 1, which every wave is done with
      const int nxt = cur == 0 ? ST - 1 : cur - 1;
      load_x(j + ST - 1, nxt);
      if (((j + kMidAhead) & 63) == 0) {
        load_ranges(j + kMidAhead);
        // waited for here: left pending, the loop's other path would carry a
        // full wait in every step, behind which no load stays in flight
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      }
      step(slots[s], j, xs + cur * XB);
      // x of step j + 1 done: it was issued a step ago, before that step's
      // slot and this step's x and slot
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"n"(
                       2 * kSlotLoads + MG)
                   : "memory");
      cur = cur == ST - 1 ? 0 : cur + 1;
    }
  }

  // C layout: lane l, element i -> row 16 gi + 4 (l / 16) + i, column l % 16
#pragma unroll
  for (int i = 0; i < 2; i++) {
    if (rbs[i] >= nrb) continue;
    float* p = Ws[i]->part + (size_t)part * M * Ws[i]->N + rbs[i] * 16 + li;
#pragma unroll
    for (int gi = 0; gi < MG; gi++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int m = 16 * gi + 4 * grp + e;
        if (m < M) p[(size_t)m * Ws[i]->N] = acc[i][gi][e];
      }
  }
}

// The launch's arguments read again from where they lie, so that a rare path's
// share of them is not loaded, or picked out of the group, before it is taken.
typedef const __attribute__((address_space(4))) QLArgs* KernelArgs;
__device__ __forceinline__ KernelArgs kernel_args() {
  uint64_t p = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();  // QLArgs is the only argument
  asm volatile("" : "+s"(p));
  return (KernelArgs)p;
}

// What mid_infinite reads of a matrix.
struct MidWeight {
  const uint8_t* codes;
  const uint16_t* scales;
  const int32_t* row_ptr;
  const int32_t* cols;
  const uint16_t* vals;
  int G, kg, gshift;
};

// The dequantized weight at (n, k): an outlier's value where the code is 0 and
// the row's list has the column.
template <int FMT>
__device__ __forceinline__ float weight_at(const MidWeight& w, int K, int n, int k) {
  const uint32_t code = w.codes[tiled_offset(n, k, K >> 7)];
  if (code == 0) {
    const int end = w.row_ptr[n + 1];
    const int p = aq::lower_bound_i32(w.cols, w.row_ptr[n], end, k);
    if (p < end && w.cols[p] == k) return (float)bits_to_h(w.vals[p]);
  }
  const uint16_t s = w.scales[(size_t)n * w.kg + (w.gshift >= 0 ? k >> w.gshift : k / w.G)];
  return (float)deq8<FMT>(code, 0u, scale2(s))[0];
}

__device__ __forceinline__ bool not_finite(uint32_t h) { return (h & 0x7C00u) == 0x7C00u; }

// qlinear_mid_kernel multiplies x by zeros that stand for other values: an
// outlier's decoded zero, the zeros beside an outlier's value in its B operand.
// Where x is infinite they make NaN of sums that F.linear on the dequantized
// weight leaves infinite (and the GEMM, which has each outlier's value in its
// place).  A wave takes such sums v[c] of row m, columns n + c, again: a sum
// with an infinite x is what its non-finite terms add up to, whatever the rest.
// (Weights that are not finite themselves: all terms.)  Rows of x with a NaN,
// or that are finite, keep theirs.  Every lane of the wave calls it.
template <int FMT>
__device__ __forceinline__ void mid_infinite(int mat, int m, int n, bool live, float (&v)[4]) {
  const KernelArgs a = kernel_args();
  const MidWeight w = {a->mat[mat].codes, a->mat[mat].scales, a->mat[mat].row_ptr, a->mat[mat].cols,
                       a->mat[mat].vals,  a->mat[mat].G,      a->mat[mat].kg,      a->mat[mat].gshift};
  const int lane = threadIdx.x & 63, K = a->K;
  const uint16_t* x = a->x;
  const bool nan = live && (v[0] != v[0] || v[1] != v[1] || v[2] != v[2] || v[3] != v[3]);
  uint64_t todo = __ballot(nan);
  while (todo) {
    const int mr = __builtin_amdgcn_readlane(m, __builtin_ctzll(todo));
    const bool mine = nan && m == mr;
    todo &= ~__ballot(mine);
    bool odd = false;
    if (mine) {
      for (int b = 0; b < 4 * w.kg; b++) odd = odd || not_finite(w.scales[(size_t)n * w.kg + b]);
      for (int p = w.row_ptr[n]; p < w.row_ptr[n + 4]; p++) odd = odd || not_finite(w.vals[p]);
    }
    const bool all = __ballot(odd) != 0;
    float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    bool again = all, stop = false;
    for (int k0 = 0; k0 < K && !stop; k0 += 512) {
      const int k = k0 + 8 * lane;
      u32x4 xv = (u32x4){0, 0, 0, 0};
      if (k < K) xv = *reinterpret_cast<const u32x4*>(x + (size_t)mr * K + k);
      uint32_t take = 0, nans = 0;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const uint32_t h = (xv[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
        take |= not_finite(h) ? 1u << j : 0u;
        nans |= not_finite(h) && (h & 0x3FFu) ? 1u : 0u;
      }
      again = again || __ballot(take != 0) != 0;
      if (__ballot(nans != 0)) {
        again = false;
        break;
      }
      if (all) take = k < K ? 0xFFu : 0u;
      for (uint64_t from = __ballot(take != 0); from; from &= from - 1) {
        const int s = __builtin_ctzll(from);
        for (uint32_t q = (uint32_t)__builtin_amdgcn_readlane((int)take, s); q; q &= q - 1) {
          const int j = __builtin_ctz(q);
          const uint32_t word = j < 2 ? xv[0] : j < 4 ? xv[1] : j < 6 ? xv[2] : xv[3];
          const float xk =
              (float)bits_to_h((uint16_t)((uint32_t)__builtin_amdgcn_readlane((int)word, s) >> (16 * (j & 1))));
          if (mine)
#pragma unroll
            for (int c = 0; c < 4; c++) t[c] = fmaf(xk, weight_at<FMT>(w, K, n + c, k0 + 8 * s + j), t[c]);
        }
      }
      // NaN whatever else comes
      stop = !__ballot(mine && (t[0] == t[0] || t[1] == t[1] || t[2] == t[2] || t[3] == t[3]));
    }
    if (mine && again)
#pragma unroll
      for (int c = 0; c < 4; c++)
        if (v[c] != v[c]) v[c] = t[c];
  }
}

// The parts' sums in order, the bias, one rounding, the epilogue: 4 columns a
// thread; grid row y is matrix y (the pair's gate).
template <int FMT, int PAIR>
__global__ __launch_bounds__(256) void mid_reduce_kernel(QLArgs a) {
  const QLMat W = PAIR ? a.mat[0] : pick(a, (int)blockIdx.y);
  const int N = W.N;
  const int64_t mn = (int64_t)a.M * N;
  const int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const bool live = i0 < mn;
  const int64_t i = live ? i0 : 0;
  const int m = (int)(i / N), n = (int)(i - (int64_t)m * N);  // N is a multiple of 16: the 4 columns are of one row
  // every load goes out before the sums are looked at
  auto sum = [&](const QLMat& w, float (&v)[4], float (&bias)[4]) {
    float4v s = *reinterpret_cast<const float4v*>(w.part + i);
    for (int p = 1; p < a.split; p++) s += *reinterpret_cast<const float4v*>(w.part + (size_t)p * mn + i);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      v[j] = s[j];
      bias[j] = w.bias ? (float)bits_to_h(w.bias[n + j]) : 0.0f;
    }
  };
  float v[4], u[4], bv[4], bu[4];
  uint16_t res[4] = {0, 0, 0, 0};
  sum(W, v, bv);
  if (PAIR) sum(a.mat[1], u, bu);
  if (!PAIR && W.res)
#pragma unroll
    for (int j = 0; j < 4; j++) res[j] = W.res[i + j];
  bool nan = false;
#pragma unroll
  for (int j = 0; j < 4; j++) nan = nan || v[j] != v[j] || (PAIR && u[j] != u[j]);
  if (__builtin_expect(__ballot(live && nan) != 0, 0)) {
    mid_infinite<FMT>((int)blockIdx.y, m, n, live, v);
    if (PAIR) mid_infinite<FMT>(1, m, n, live, u);
  }
  if (!live) return;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    v[j] += bv[j];
    if (PAIR) u[j] += bu[j];
  }
  uint16_t o[4];
#pragma unroll
  for (int j = 0; j < 4; j++)
    o[j] = PAIR ? h_to_bits(silu_mul_h((float)rn_h(v[j]), (float)rn_h(u[j])))
                : mid_epilogue(rn_h(v[j]), W.act, res[j], W.res != nullptr);
  if ((uintptr_t)W.y % 8 == 0) {
    *reinterpret_cast<uint2*>(W.y + i) = make_uint2(o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16));
  } else {
#pragma unroll
    for (int j = 0; j < 4; j++) W.y[i + j] = o[j];
  }
}

template <int FMT, int PC, int MG, int PAIR>
hipError_t launch_mid(const QLArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)(a.first[a.count] * a.split));
  hipLaunchKernelGGL((qlinear_mid_kernel<FMT, PC, MG, PAIR>), grid, dim3(64 * kMidWaves), 0, s, a);
  return hipGetLastError();
}

template <int FMT, int PC, int MG>
hipError_t launch_mid(const QLArgs& a, bool pair, hipStream_t s) {
  return pair ? launch_mid<FMT, PC, MG, 1>(a, s) : launch_mid<FMT, PC, MG, 0>(a, s);
}

template <int FMT, int PC>
hipError_t launch_mid(const QLArgs& a, int mg, bool pair, hipStream_t s) {
  return mg == 3 ? launch_mid<FMT, PC, 3>(a, pair, s) : launch_mid<FMT, PC, 4>(a, pair, s);
}

template <int FMT>
hipError_t launch_mid(const QLArgs& a, int pc, int mg, bool pair, hipStream_t s) {
  return pc == 1 ? launch_mid<FMT, 1>(a, mg, pair, s)
         : pc == 2 ? launch_mid<FMT, 2>(a, mg, pair, s) : launch_mid<FMT, 0>(a, mg, pair, s);
}

template <int FMT>
hipError_t launch_reduce(const QLArgs& a, int64_t nmax, bool pair, hipStream_t s) {
  const dim3 grid((unsigned)aq::ceil_div((int64_t)a.M * nmax, 1024), (unsigned)(pair ? 1 : a.count));
  if (pair)
    hipLaunchKernelGGL((mid_reduce_kernel<FMT, 1>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((mid_reduce_kernel<FMT, 0>), grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace

namespace aqk {

// Workgroups of an unsplit launch.
static int64_t mid_units(const int64_t* Ns, int64_t count, bool pair) {
  if (pair) return aq::ceil_div(Ns[0], 16 * kMidWaves);
  int64_t n = 0;
  for (int64_t i = 0; i < count; i++) n += aq::ceil_div(Ns[i], 32 * kMidWaves);
  return n;
}

// One workgroup per CU, in parts of at least 4 chunks: down_proj [4096,
// 14336] at M = 64, 32 units, takes 70 us in 2 parts, 42 in 4, 31 in 8 and
// 34 in 16; gate+up [28672, 4096], 224 units, 54 in one, 47 in 2 parts and 49
// in 4.
int mid_split(const int64_t* Ns, int64_t count, int64_t K) {
  const int64_t units = mid_units(Ns, count, false);  // a pair splits as its members alone do
  const int64_t want = aq::ceil_div(aq::cu_count(), units);
  return (int)std::max<int64_t>(1, std::min({want, K / 128 / 4, (int64_t)16}));
}

hipError_t launch_qlinear_mid(QLArgs a, int fmt, int pc, bool pair, hipStream_t s) {
  int64_t Ns[kMaxGroup], first = 0, nmax = 0;
  for (int i = 0; i < a.count; i++) {
    Ns[i] = a.mat[i].N;
    nmax = std::max<int64_t>(nmax, Ns[i]);
    a.first[i] = (int)first;
    first += mid_units(Ns + i, 1, pair);
    if (pair) break;  // gate's units hold up's
  }
  for (int i = pair ? 1 : a.count; i <= kMaxGroup; i++) a.first[i] = (int)first;
  const int mg = (int)aq::ceil_div(a.M, 16);
  const hipError_t e = fmt == AQ_FMT_E4M3 ? launch_mid<AQ_FMT_E4M3>(a, pc, mg, pair, s)
                                          : launch_mid<AQ_FMT_INT8>(a, pc, mg, pair, s);
  if (e != hipSuccess) return e;
  return fmt == AQ_FMT_E4M3 ? launch_reduce<AQ_FMT_E4M3>(a, nmax, pair, s)
                            : launch_reduce<AQ_FMT_INT8>(a, nmax, pair, s);
}

}  // namespace aqk
