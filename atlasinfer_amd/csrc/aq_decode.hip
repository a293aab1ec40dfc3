// aq_decode.hip -- the work of one decode step around the quantized linears:
// attention over a static key/value cache (the position read from device
// memory, so that a HIP graph replays it), the residual add + RMSNorm /
// LayerNorm of a row, and the SwiGLU product.
#include "aq_common.h"

namespace {

__device__ __forceinline__ float h2f(uint16_t b) { return (float)bits_to_h(b); }

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));

// s + the dot product of eight fp16 pairs (v_dot2_f32_f16: the products are
// exact in f32, each pair's sum added to s in f32).
__device__ __forceinline__ float dot8(uint4 a, uint4 b, float s) {
  s = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, a.x), __builtin_bit_cast(h2_t, b.x), s, false);
  s = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, a.y), __builtin_bit_cast(h2_t, b.y), s, false);
  s = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, a.z), __builtin_bit_cast(h2_t, b.z), s, false);
  s = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, a.w), __builtin_bit_cast(h2_t, b.w), s, false);
  return s;
}

// w * v + c with v the low / high fp16 of a pair, entering exactly.
__device__ __forceinline__ float fma_lo(float w, uint32_t v, float c) {
  asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel:[0,0,0] op_sel_hi:[0,1,0]" : "+v"(c) : "v"(w), "v"(v));
  return c;
}
__device__ __forceinline__ float fma_hi(float w, uint32_t v, float c) {
  asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "+v"(c) : "v"(w), "v"(v));
  return c;
}

// The maximum over a row group's four rows (reduce4's result lanes), in all
// its lanes.
template <int KV>
__device__ __forceinline__ float max4(float x) {
  if (KV == 16) {
    x = xlane_level_max_f32<4>(x);
    return xlane_level_max_f32<3>(x);
  }
  x = xlane_level_max_f32<3>(x);
  return xlane_level_max_f32<2>(x);
}

// The value of lane 4 n of each row of 16 lanes, in the whole row.
__device__ __forceinline__ float row_bcast(float x, int n) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  return __builtin_bit_cast(float, n == 0   ? __builtin_amdgcn_mov_dpp(u, 0x150, 0xF, 0xF, false)  // row_newbcast
                                   : n == 1 ? __builtin_amdgcn_mov_dpp(u, 0x154, 0xF, 0xF, false)
                                   : n == 2 ? __builtin_amdgcn_mov_dpp(u, 0x158, 0xF, 0xF, false)
                                            : __builtin_amdgcn_mov_dpp(u, 0x15C, 0xF, 0xF, false));
}

// The sum over the lanes of equal index in the wave's aligned groups of KV
// lanes (8 or 16), in all of them.
template <int KV>
__device__ __forceinline__ float row_groups_sum(float x) {
  if (KV == 8) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(u, 0x128, 0xF, 0xF, false));  // row_ror:8, lane i ^ 8
  }
  return xlane_level_sum_f32<6>(xlane_level_sum_f32<5>(x));
}

// x * f rounded to fp16 (fp16 tensor times a Python float); f = 1 is exact.
__device__ __forceinline__ f16 scale_h(f16 x, float f) { return f == 1.0f ? x : rn_h((float)x * f); }

// Sums over aligned groups of KV lanes (8 or 16) of four values each lane
// holds, the sum of value n left in the lanes whose first two group bits are
// n: a butterfly of DPP mirrors and quad permutations, each level's partners
// agreeing in the bits already used, that halves the values twice.
template <int KV>
__device__ __forceinline__ float reduce4(const float (&v)[4], int ln) {
  constexpr int B = KV / 2;  // the first bit
  auto partner = [](float x, int level) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    return __builtin_bit_cast(float, level == 4   ? xlane_partner_u32<4>(u)    // lane 15 - i
                                     : level == 3 ? xlane_partner_u32<3>(u)    // 7 - i of 8
                                     : level == 2 ? xlane_partner_u32<2>(u)    // i ^ 2
                                                  : xlane_partner_u32<1>(u));  // i ^ 1
  };
  const bool hi = ln & B, hi2 = ln & (B / 2);
  constexpr int L0 = KV == 16 ? 4 : 3;
  const float a = (hi ? v[2] : v[0]) + partner(hi ? v[0] : v[2], L0);
  const float b = (hi ? v[3] : v[1]) + partner(hi ? v[1] : v[3], L0);
  float r = (hi2 ? b : a) + partner(hi2 ? a : b, L0 - 1);
  if (KV == 16) r += partner(r, 2);
  r += partner(r, 1);
  return r;
}

// One rotate-half element: partner is x[d + D/2] (negated, lo = true) or
// x[d - D/2]; fp16(fp16(x c) + fp16(r s)).
__device__ __forceinline__ f16 rope_h(f16 x, f16 partner, bool lo, uint16_t c, uint16_t s) {
  const float r = lo ? -(float)partner : (float)partner;
  const f16 a = rn_h((float)x * (float)bits_to_h(c));
  const f16 b2 = rn_h(r * (float)bits_to_h(s));
  return rn_h((float)a + (float)b2);
}

// Splitting of the cache among workgroups.  A cache of at most 16 chunks of
// 64 positions is one span per head, its steps dealt to nw = 4 (or fewer)
// waves of one workgroup that merge their results in LDS (no second kernel),
// when a wave's serial share is short -- at most 8 steps, and at most 8
// chunk-units, a chunk costing G D / 64 units -- or when B Hkv >= 128
// workgroups share the CUs.
// (G = 4, D = 128, 30 positions of 3 chunks: one span 7.5 us, split and
// merged 9.4; 16 sequences x 8 heads at 300 of 7 chunks 13.3 against 18.1;
// one sequence at 700 of 13 chunks 18.5 against 11.5, and 16 heads of G = 1,
// 13 steps a wave, 9.9 against 8.1, so split.)  Otherwise
// the cache is split into spans of nt chunks, up to 4 waves each, nt the
// smallest power of two that leaves ns = ceil(L / (64 nt)) <= 64 spans per
// head and B Hkv ns <= 384 workgroups (or one span for the whole cache);
// decode_combine_kernel merges the spans.  A workgroup's start and merge cost
// as much as 100 positions: 4 sequences x 8 heads at 1500 of 26 chunks 15.9 us
// in 7 spans a head, 16.7 in 13, 19.8 in 26; 8 sequences x 8 heads at 4000
// 30.0 in 5 spans, 31.7 in 9.
// For the same reason spans of D = 64 that hold a whole short cache take one
// wave instead of four once the workgroups fill the CUs without (2048 heads
// at 130 positions 15.1 against 19.9 us, at 700 both 63.8).
constexpr int kChunk = 64;
constexpr int kOneSpanChunks = 16;
constexpr int kMaxWaves = 4;  // one per SIMD: 8 would halve the registers a wave may hold (D = 128 then spills)
constexpr int64_t kMaxGroups = 384;
constexpr int64_t kMaxSpans = 64;

struct Split {
  int64_t nt, ns, nw, part_floats, bytes;
};

// G query heads share a key/value head; a span's partial result is its
// running maximum and denominator per query head and its G x D weighted sum.
inline Split split_of(int64_t B, int64_t Hkv, int64_t G, int64_t D, int64_t L) {
  Split sp;
  const int64_t chunks = (L + kChunk - 1) / kChunk;
  sp.part_floats = G * D + 2 * G;
  const int64_t step = 4 * 64 / (D / 8);  // positions a wave takes at a time
  const int64_t nw1 = std::min<int64_t>(kMaxWaves, chunks * kChunk / step);
  const int64_t serial_units = (chunks + nw1 - 1) / nw1 * G * D / 64;
  const int64_t serial_steps = (chunks * kChunk / step + nw1 - 1) / nw1;
  if (chunks <= kOneSpanChunks && ((serial_units <= 8 && serial_steps <= 8) || B * Hkv >= 128)) {
    sp.nt = chunks;
    sp.ns = 1;
    sp.nw = nw1;
  } else {
    sp.nt = 1;
    auto spans = [&](int64_t nt) { return (L + kChunk * nt - 1) / (kChunk * nt); };
    while (kChunk * sp.nt < L && (spans(sp.nt) > kMaxSpans || B * Hkv * spans(sp.nt) > kMaxGroups)) sp.nt *= 2;
    sp.ns = spans(sp.nt);
    sp.nw = std::min<int64_t>(kMaxWaves, sp.nt * kChunk / step);
  }
  if (D == 64 && sp.ns == 1 && (B * Hkv >= 1024 || (B * Hkv >= 512 && chunks <= 5))) sp.nw = 1;
  sp.bytes = B * Hkv * sp.ns * sp.part_floats * 4;
  return sp;
}

// LDS of one workgroup of nw waves, in floats: per wave the softmax numerators
// of a step (D = 64: [G][32]; D = 128 passes them between lanes) and its merged
// result [G D + 2 G].
__host__ __device__ constexpr int numerators(int G, int D) { return D == 64 ? G * 32 : 0; }
inline size_t attention_lds(int G, int D, int64_t nw) { return (size_t)nw * (numerators(G, D) + G * D + 2 * G) * 4; }

// Workgroup (j, b, z) takes key/value head j of batch row b (query heads
// j G .. j G + G - 1) and cache positions z span .. z span + span - 1
// (span = 64 nt); q [B, H, D], k_new / v_new [B, Hkv, D], k_cache and
// v_cache [B, Hkv, L, D], out [B, H, D], all fp16.  The span holding pos
// writes k_new / v_new there.  For each query head g: scores s_p = fp16(q .
// k_p) * scale for p <= pos (the product accumulated in f32 and rounded to
// fp16, as a half-precision matrix product returns it), softmax over them in
// f32 and o = sum_p softmax_p v_p accumulated in f32, rounded to fp16 once.
//
// Wave w of the workgroup takes steps w, w + nw, ... of the span, a step being
// four loads of keys and of values (16 positions of D = 128, 32 of 64), each row
// group rs with a running maximum of its own (when one grows, the sums so far
// are rescaled by exp(m_old - m_new)); the next step's loads are in flight
// meanwhile:
//   loads   lane ln takes the 16-byte chunk ch = ln % (D / 8) of rows
//           rs + RPW n, rs = ln / (D / 8), of keys and values alike, so that a
//           load instruction reads RPW = 64 / (D / 8) whole rows, 1 KiB;
//   scores  each lane's part of the rows' dot products against its chunk of
//           the queries (in registers), summed over the lanes of a row
//           (reduce4): lane ln holds the score of row rs + RPW n_of(ch);
//   values  weighted by their rows' numerators, broadcast to the row's lanes;
//   sums    each lane keeps its share of the denominator.
// Bound by HBM for long caches, by its chain of loads for short ones.  With
// the merge of the spans, 8 sequences of 4000 positions (8 key/value heads of
// 4 queries, 131 MB) take 30.0 us and one of 700 11.5; a wave per 64 positions,
// a key row per lane and no loads ahead took 39.8 and 13.3.
// Position pos's key and value come from k_new / v_new (the cache's copy is
// this kernel's own store); positions past pos read as zero and weigh zero.  Before use the queries are multiplied by q_scale (rounded to fp16;
// skipped for 1) and, given rcos / rsin (fp16 [L, D] tables), the queries
// and the new key are rotated at position pos in the rotate-half form:
// x' = fp16(fp16(x c) + fp16(r s)), r = (-x[D/2:], x[:D/2]) -- the order
// and roundings of fp16 tensor arithmetic.
//
// The waves' results meet in LDS (maximum M over the waves, each wave's
// sums scaled by exp(m_w - M), waves in order).  With one span holding
// positions the workgroup writes out itself; otherwise every span with
// positions writes (M, l, sum) to its slot of part and
// decode_combine_kernel, launched next on the same stream, merges them.  (A
// merge inside this kernel by the last span to arrive would need an
// agent-scope release per span, which writes back the whole L2 of the
// span's XCD; the kernel boundary orders the slots for free.)
// (Registers: up to 128, four waves a SIMD, for G <= 2; one more and 1024
// workgroups, G = 2, D = 64, come in two rounds.)
template <int D, int G>
__global__ __launch_bounds__(64 * kMaxWaves, G <= 2 ? 4 : 2) void decode_attention_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_new, const uint16_t* __restrict__ v_new,
    uint16_t* __restrict__ k_cache, uint16_t* __restrict__ v_cache, const int64_t* __restrict__ pos_p, int H, int Hkv,
    int L, float scale, float q_scale, const uint16_t* __restrict__ rcos, const uint16_t* __restrict__ rsin, int nt,
    int ns, float* __restrict__ part, uint16_t* __restrict__ out) {
  constexpr int KV = D / 8;     // 16-byte chunks of a row
  constexpr int RPW = 64 / KV;  // rows one wave-wide load covers
  constexpr int NS = 4;         // loads of keys, and of values, a step
  constexpr int PS = RPW * NS;  // positions a step
  constexpr int PF = G * D + 2 * G;
  static_assert(KV == 16 || numerators(G, D) == G * PS, "a step's numerators");
  const int j = blockIdx.x, b = blockIdx.y, z = blockIdx.z, t = threadIdx.x;
  const int nw = blockDim.x >> 6, ln = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t pos = *pos_p;
  if (pos < 0 || pos >= L) return;  // the caller guards this; no access outside the cache
  const int64_t span = (int64_t)kChunk * nt, z0 = (int64_t)z * span;
  if (z0 > pos) return;  // no cached position in this span yet
  const int nact = (int)(pos / span) + 1;
  const int64_t kv = (int64_t)b * Hkv + j;
  uint16_t* Kc = k_cache + kv * L * D;
  uint16_t* Vc = v_cache + kv * L * D;
  const uint4* kn = reinterpret_cast<const uint4*>(k_new + kv * D);
  const uint4* vn = reinterpret_cast<const uint4*>(v_new + kv * D);
  uint16_t* o = out + ((int64_t)b * H + (int64_t)j * G) * D;

  const int ch = ln % KV, rs = ln / KV;
  const int nsteps = nt * (kChunk / PS);
  // the span's rows below pos: the rest read as zero without touching memory,
  // so no load has a condition, and waiting for one step's rows leaves the
  // next step's in flight
  const int bytes = (int)((min(pos, z0 + span) - z0) * D * 2);
  const __amdgpu_buffer_rsrc_t kbuf = __builtin_amdgcn_make_buffer_rsrc(Kc + z0 * D, (short)0, bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t vbuf = __builtin_amdgcn_make_buffer_rsrc(Vc + z0 * D, (short)0, bytes, 0x00020000);
  struct Rows {
    uint4 k[NS], v[NS];
  };
  auto load = [&](Rows& r, int64_t t0) {
    const uint32_t off = (uint32_t)((int)(t0 - z0) + rs) * (D * 2) + ch * 16;
#pragma unroll
    for (int n = 0; n < NS; n++)
      r.k[n] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(kbuf, off + n * RPW * D * 2, 0, 0));
#pragma unroll
    for (int n = 0; n < NS; n++)
      r.v[n] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(vbuf, off + n * RPW * D * 2, 0, 0));
  };
  // the first rows are on their way while the queries are staged
  Rows ra, rb;
  const int64_t hop = (int64_t)nw * PS;
  int64_t t0 = z0 + (int64_t)wave * PS;
  load(ra, t0);
  __shared__ uint4 qs[G][KV];    // the group's queries, fp16
  __shared__ uint4 krot[KV];     // position pos's key as cached (last span only)
  extern __shared__ float dyn[];
  float* w = dyn + wave * numerators(G, D);  // this wave's numerators [G][PS] (D = 64)
  float* res = dyn + nw * numerators(G, D);  // the waves' results [nw][PF]

  const uint16_t* cs = rcos ? rcos + pos * D : nullptr;
  const uint16_t* sn = rsin ? rsin + pos * D : nullptr;
  const uint16_t* qb = q + ((int64_t)b * H + (int64_t)j * G) * D;
  for (int i = t; i < G * D; i += 64 * nw) {
    const int d = i % D;
    f16 v = scale_h(bits_to_h(qb[i]), q_scale);
    if (cs) v = rope_h(v, scale_h(bits_to_h(qb[i - d + (d + D / 2) % D]), q_scale), d < D / 2, cs[d], sn[d]);
    reinterpret_cast<uint16_t*>(&qs[0][0])[i] = h_to_bits(v);
  }
  const bool last = z == nact - 1;  // the span holding pos
  if (last) {
    const uint16_t* kb = k_new + kv * D;
    for (int d = t; d < D; d += 64 * nw) {
      f16 v = bits_to_h(kb[d]);
      if (cs) v = rope_h(v, bits_to_h(kb[(d + D / 2) % D]), d < D / 2, cs[d], sn[d]);
      reinterpret_cast<uint16_t*>(krot)[d] = h_to_bits(v);
    }
  }
  __syncthreads();
  if (last && t < KV) {
    reinterpret_cast<uint4*>(Kc + pos * D)[t] = krot[t];
    reinterpret_cast<uint4*>(Vc + pos * D)[t] = vn[t];
  }

  uint4 qv[G];  // this lane's chunk of the queries
#pragma unroll
  for (int g = 0; g < G; g++) qv[g] = qs[g][ch];
  float acc[G][8], m[G], lt[G];
#pragma unroll
  for (int g = 0; g < G; g++) {
    m[g] = -INFINITY;
    lt[g] = 0.0f;
#pragma unroll
    for (int h = 0; h < 8; h++) acc[g][h] = 0.0f;
  }

  const int nrow = ch >> (KV == 16 ? 2 : 1);  // the row (of four per rs) whose score this lane holds
  const bool first = (ch & (KV == 16 ? 3 : 1)) == 0;  // one of the lanes holding it
  auto step = [&](Rows& r, int64_t t0) {
    const bool valid = t0 + RPW * nrow + rs <= pos;
    if (last) {  // position pos: its key as cached and its value
#pragma unroll
      for (int n = 0; n < NS; n++)
        if (t0 + RPW * n + rs == pos) {
          r.k[n] = krot[ch];
          r.v[n] = vn[ch];
        }
    }
    float e[G], mn[G];
    bool grows = false;
#pragma unroll
    for (int g = 0; g < G; g++) {
      float v[NS];
#pragma unroll
      for (int n = 0; n < NS; n++) v[n] = dot8(r.k[n], qv[g], 0.0f);
      const float dot = reduce4<KV>(v, ln);  // every lane takes part, whether its own row is valid or not
      const float sg = valid ? (float)rn_h(dot) * scale : -INFINITY;
      mn[g] = fmaxf(m[g], max4<KV>(sg));  // the same in every lane of a row group
      grows = grows || mn[g] != m[g];
      // a score of -inf (an fp16 overflow) weighs nothing, also while its row
      // group has met no other
      e[g] = sg == -INFINITY ? 0.0f : __expf(sg - mn[g]);
    }
    if (__ballot(grows)) {
#pragma unroll
      for (int g = 0; g < G; g++) {
        const float c = m[g] == -INFINITY ? 0.0f : __expf(m[g] - mn[g]);  // 1 where it stays
        lt[g] *= c;
#pragma unroll
        for (int h = 0; h < 8; h++) acc[g][h] *= c;
        m[g] = mn[g];
      }
    }
#pragma unroll
    for (int g = 0; g < G; g++) lt[g] += first ? e[g] : 0.0f;
    if (KV == 8) {
      // w is this wave's own: its LDS writes complete before its reads, in
      // order; the compiler keeps the reads after the writes
#pragma unroll
      for (int g = 0; g < G; g++)
        if (first) w[g * PS + RPW * nrow + rs] = e[g];
      __builtin_amdgcn_wave_barrier();
      asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int n = 0; n < NS; n++) {
      const uint32_t wd[4] = {r.v[n].x, r.v[n].y, r.v[n].z, r.v[n].w};
#pragma unroll
      for (int g = 0; g < G; g++) {
        const float wg = KV == 16 ? row_bcast(e[g], n) : w[g * PS + RPW * n + rs];
#pragma unroll
        for (int h = 0; h < 4; h++) {
          acc[g][2 * h] = fma_lo(wg, wd[h], acc[g][2 * h]);
          acc[g][2 * h + 1] = fma_hi(wg, wd[h], acc[g][2 * h + 1]);
        }
      }
    }
    if (KV == 8) {
      __builtin_amdgcn_wave_barrier();  // this step's reads of w before the next step's writes
      asm volatile("" ::: "memory");
    }
  };
  for (int i = wave; i < nsteps && t0 <= pos; i += 2 * nw) {
    load(rb, t0 + hop);
    __builtin_amdgcn_sched_barrier(0);
    step(ra, t0);
    load(ra, t0 + 2 * hop);
    __builtin_amdgcn_sched_barrier(0);
    if (i + nw < nsteps && t0 + hop <= pos) step(rb, t0 + hop);
    t0 += 2 * hop;
  }

  // waves whose first step lies past pos have nothing to add
  const int na = (int)min((int64_t)nw, (pos - z0) / PS + 1);
  if (wave < na) {
    // the wave's sums: the row groups' maxima meet, then the lanes' denominators
    // and the RPW row groups' outputs
#pragma unroll
    for (int g = 0; g < G; g++) {
      const float mw = wave_group_max_f32<64>(m[g]);
      const float c = m[g] == -INFINITY ? 0.0f : __expf(m[g] - mw);
      m[g] = mw;
      lt[g] *= c;
#pragma unroll
      for (int h = 0; h < 8; h++) acc[g][h] *= c;
      lt[g] = wave_group_sum_f32<64>(lt[g]);
#pragma unroll
      for (int h = 0; h < 8; h++) acc[g][h] = row_groups_sum<KV>(acc[g][h]);
    }
    if (nw == 1 && nact == 1) {
      if (rs == 0) {
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
          for (int h = 0; h < 8; h++) o[g * D + 8 * ch + h] = h_to_bits(rn_h(acc[g][h] / lt[g]));
      }
      return;
    }
    float* pp = nw == 1 ? part + (kv * ns + z) * PF : res + wave * PF;
    if (rs == 0) {
#pragma unroll
      for (int g = 0; g < G; g++)
#pragma unroll
        for (int h = 0; h < 8; h++) pp[g * D + 8 * ch + h] = acc[g][h];
    }
    if (ln == 0) {
#pragma unroll
      for (int g = 0; g < G; g++) {
        pp[G * D + g] = m[g];
        pp[G * D + G + g] = lt[g];
      }
    }
  }
  if (nw == 1) return;  // the span's partial is in part; decode_combine_kernel merges
  __syncthreads();
  // the waves' results, merged in wave order: out when one span holds every
  // position, else the span's partial (M, l, sum) into part
  float* sp = part + (kv * ns + z) * PF;
  for (int i = t; i < G * D + G; i += 64 * nw) {
    const int g = i < G * D ? i / D : i - G * D;
    float mx = -INFINITY;
    for (int v = 0; v < na; v++) mx = fmaxf(mx, res[v * PF + G * D + g]);
    float num = 0.0f, den = 0.0f;
    for (int v = 0; v < na; v++) {
      const float mv = res[v * PF + G * D + g];
      const float f = mv == -INFINITY ? 0.0f : __expf(mv - mx);
      den = fmaf(res[v * PF + G * D + G + g], f, den);
      if (i < G * D) num = fmaf(res[v * PF + i], f, num);
    }
    if (i < G * D) {
      if (nact == 1)
        o[i] = h_to_bits(rn_h(num / den));
      else
        sp[i] = num;
    } else if (nact > 1) {
      sp[G * D + g] = mx;
      sp[G * D + G + g] = den;
    }
  }
}

// Merges the spans' partial results of decode_attention_kernel for query head
// h of batch row b: M = max_z m_z, f_z = exp(m_z - M), out = fp16(sum_z f_z
// sum_z / sum_z f_z l_z).  256 / D groups of D threads take every
// (256 / D)-th span each, in order, and their sums are added in order.  A
// workgroup per query head (one per key/value head, its spans' weights
// summed by one thread each, took 9.1 us for 33 spans of 64 heads).  Does
// nothing when one span held every position (that span wrote out).
template <int D, int G>
__global__ __launch_bounds__(256) void decode_combine_kernel(const int64_t* __restrict__ pos_p, int H, int Hkv, int L,
                                                             int nt, int ns, const float* __restrict__ part,
                                                             uint16_t* __restrict__ out) {
  constexpr int PF = G * D + 2 * G;
  constexpr int NG = 256 / D;
  const int h = blockIdx.x, b = blockIdx.y, t = threadIdx.x;
  const int j = h / G, g = h % G;
  const int64_t pos = *pos_p;
  if (pos < 0 || pos >= L) return;
  const int nact = (int)(pos / ((int64_t)kChunk * nt)) + 1;
  if (nact == 1) return;
  const float* pk = part + ((int64_t)b * Hkv + j) * ns * PF;
  const int grp = t / D, d = t % D;
  // eight spans' loads in flight, then their products in span order
  auto load = [&](float (&v)[8], int z0) {
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int z = z0 + NG * k + grp;
      v[k] = z < nact ? pk[z * PF + g * D + d] : 0.0f;
    }
  };
  float v[8];
  load(v, 0);
  __shared__ float f[kMaxSpans];
  __shared__ float sum[NG][D];
  // every wave has all spans' (m, l), one a lane (at most 64 spans)
  const int z = t & 63;
  const float m = z < nact ? pk[z * PF + G * D + g] : -INFINITY;
  const float l = z < nact ? pk[z * PF + G * D + G + g] : 0.0f;
  const float mx = wave_group_max_f32<64>(m);
  const float e = z < nact ? __expf(m - mx) : 0.0f;
  const float den = wave_group_sum_f32<64>(l * e);
  if (t < 64) f[z] = e;
  __syncthreads();
  float num = 0.0f;
  for (int z0 = 0; z0 < nact; z0 += 8 * NG) {
    float nx[8];
    load(nx, z0 + 8 * NG);
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int zz = z0 + NG * k + grp;
      if (zz < nact) num = fmaf(v[k], f[zz], num);
      v[k] = nx[k];
    }
  }
  sum[grp][d] = num;
  __syncthreads();
  if (grp == 0) {
#pragma unroll
    for (int k = 1; k < NG; k++) num += sum[k][d];
    out[((int64_t)b * H + h) * D + d] = h_to_bits(rn_h(num / den));
  }
}

}  // namespace

extern "C" int64_t aq_decode_attention_workspace(int64_t B, int64_t H, int64_t Hkv, int64_t D, int64_t L) {
  if (B <= 0 || Hkv <= 0 || H <= 0 || H % Hkv != 0 || D <= 0 || L <= 0) return -1;
  return split_of(B, Hkv, H / Hkv, D, L).bytes;
}

extern "C" int aq_decode_attention(const void* q, const void* k_new, const void* v_new, void* k_cache, void* v_cache,
                                   const int64_t* pos, int64_t B, int64_t H, int64_t Hkv, int64_t D, int64_t L,
                                   float scale, float q_scale, const void* rope_cos, const void* rope_sin,
                                   void* workspace, int64_t ws_bytes, void* out, void* stream) {
  AQ_CHECK_ARG(q && k_new && v_new && k_cache && v_cache && pos && out && workspace,
               "aq_decode_attention: null pointer");
  AQ_CHECK_ARG((rope_cos == nullptr) == (rope_sin == nullptr),
               "aq_decode_attention: rope_cos and rope_sin come together");
  AQ_CHECK_ARG(B > 0 && Hkv > 0 && H > 0 && H % Hkv == 0 &&
                   (H / Hkv == 1 || H / Hkv == 2 || H / Hkv == 4 || H / Hkv == 8),
               "aq_decode_attention: H (%lld) must be 1, 2, 4 or 8 times Hkv (%lld)", (long long)H, (long long)Hkv);
  AQ_CHECK_ARG(D == 64 || D == 128, "aq_decode_attention: head dim %lld (64 or 128 supported)", (long long)D);
  AQ_CHECK_ARG((uintptr_t)k_cache % 16 == 0 && (uintptr_t)v_cache % 16 == 0 && (uintptr_t)k_new % 16 == 0 &&
                   (uintptr_t)v_new % 16 == 0 && (uintptr_t)workspace % 16 == 0,
               "aq_decode_attention: k_new, v_new, the caches and the workspace must be 16-byte aligned");
  AQ_CHECK_ARG(L > 0 && L <= (1 << 24) && B <= 65535 && Hkv <= 65535, "aq_decode_attention: sizes out of range");
  const Split sp = split_of(B, Hkv, H / Hkv, D, L);
  AQ_CHECK_ARG(ws_bytes >= sp.bytes, "aq_decode_attention: workspace of %lld bytes, %lld needed", (long long)ws_bytes,
               (long long)sp.bytes);
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)Hkv, (unsigned)B, (unsigned)sp.ns);  // spans past pos exit at once
  const int G = (int)(H / Hkv);
  float* part = (float*)workspace;
#define AQ_DECODE_LAUNCH(DD, GG)                                                                                     \
  do {                                                                                                               \
    hipLaunchKernelGGL((decode_attention_kernel<DD, GG>), grid, dim3(64 * (unsigned)sp.nw),                       \
                       attention_lds(GG, DD, sp.nw), s, (const uint16_t*)q,                                          \
                       (const uint16_t*)k_new, (const uint16_t*)v_new, (uint16_t*)k_cache, (uint16_t*)v_cache, pos, \
                       (int)H, (int)Hkv, (int)L, scale, q_scale, (const uint16_t*)rope_cos,                        \
                       (const uint16_t*)rope_sin, (int)sp.nt, (int)sp.ns, part, (uint16_t*)out);                    \
    if (sp.ns > 1)                                                                                                   \
      hipLaunchKernelGGL((decode_combine_kernel<DD, GG>), dim3((unsigned)H, (unsigned)B), dim3(256), 0, s, pos,     \
                         (int)H, (int)Hkv, (int)L, (int)sp.nt, (int)sp.ns, part, (uint16_t*)out);                  \
  } while (0)
  if (D == 64) {
    if (G == 1) AQ_DECODE_LAUNCH(64, 1);
    else if (G == 2) AQ_DECODE_LAUNCH(64, 2);
    else if (G == 4) AQ_DECODE_LAUNCH(64, 4);
    else AQ_DECODE_LAUNCH(64, 8);
  } else {
    if (G == 1) AQ_DECODE_LAUNCH(128, 1);
    else if (G == 2) AQ_DECODE_LAUNCH(128, 2);
    else if (G == 4) AQ_DECODE_LAUNCH(128, 4);
    else AQ_DECODE_LAUNCH(128, 8);
  }
#undef AQ_DECODE_LAUNCH
  AQ_LAUNCH_CHECK("aq_decode_attention");
  return AQ_OK;
}

// ------------------------------------------------------------ decode glue

namespace {

constexpr int kNormThreads = 256;
constexpr int kNormChunks = 8;  // 8 fp16 each: rows of up to 256 * 8 * 8 = 16384

__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_group_sum_f32<64>(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// One workgroup per row of n fp16.  With delta: x = fp16(x + delta), stored
// back (a residual add).  Then y = norm(x):
//   MODE 0 (RMSNorm): r = 1 / sqrt(mean_f32(x^2) + eps), y = fp16(w fp16(x r))
//   MODE 1 (LayerNorm): mean and variance in f32, y = fp16((x - mean) rstd w + b)
// (the operation order of HF's Llama/Mistral RMSNorm and torch's layer_norm
// on fp16 inputs).
template <int MODE>
__global__ __launch_bounds__(kNormThreads) void decode_norm_kernel(uint16_t* __restrict__ x,
                                                                  const uint16_t* __restrict__ delta,
                                                                  const uint16_t* __restrict__ w,
                                                                  const uint16_t* __restrict__ bias, float eps, int n,
                                                                  uint16_t* __restrict__ y) {
  __shared__ float red[4];
  const int t = threadIdx.x;
  uint16_t* xr = x + (int64_t)blockIdx.x * n;
  const uint16_t* dr = delta ? delta + (int64_t)blockIdx.x * n : nullptr;
  uint16_t* yr = y + (int64_t)blockIdx.x * n;
  float v[kNormChunks][8];
  float s = 0.0f;
  // the weights (and bias) go out with x, ahead of the reduction
  uint4 wv[kNormChunks], bv[kNormChunks];
#pragma unroll
  for (int c = 0; c < kNormChunks; c++) {
    const int i = (c * kNormThreads + t) * 8;
    if (i < n) {
      wv[c] = *reinterpret_cast<const uint4*>(w + i);
      bv[c] = MODE == 1 ? *reinterpret_cast<const uint4*>(bias + i) : make_uint4(0, 0, 0, 0);
    }
  }
#pragma unroll
  for (int c = 0; c < kNormChunks; c++) {
    const int i = (c * kNormThreads + t) * 8;
    if (i < n) {
      uint4 a = *reinterpret_cast<const uint4*>(xr + i);
      if (dr) {
        const uint4 d = *reinterpret_cast<const uint4*>(dr + i);
        const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, dw[4] = {d.x, d.y, d.z, d.w};
        uint32_t ow[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const f16 lo = rn_h((float)bits_to_h((uint16_t)aw[k]) + (float)bits_to_h((uint16_t)dw[k]));
          const f16 hi = rn_h((float)bits_to_h((uint16_t)(aw[k] >> 16)) + (float)bits_to_h((uint16_t)(dw[k] >> 16)));
          ow[k] = (uint32_t)h_to_bits(lo) | ((uint32_t)h_to_bits(hi) << 16);
        }
        a = make_uint4(ow[0], ow[1], ow[2], ow[3]);
        *reinterpret_cast<uint4*>(xr + i) = a;
      }
      const uint32_t aw[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
      for (int k = 0; k < 8; k++) {
        v[c][k] = (float)bits_to_h((uint16_t)(aw[k >> 1] >> (16 * (k & 1))));
        s += MODE == 0 ? v[c][k] * v[c][k] : v[c][k];
      }
    }
  }
  const float tot = block_sum(s, red);
  float mean = 0.0f, r;
  if (MODE == 0) {
    r = 1.0f / sqrtf(tot / (float)n + eps);
  } else {
    mean = tot / (float)n;
    float q = 0.0f;
#pragma unroll
    for (int c = 0; c < kNormChunks; c++)
      if ((c * kNormThreads + t) * 8 < n)
#pragma unroll
        for (int k = 0; k < 8; k++) q += (v[c][k] - mean) * (v[c][k] - mean);
    r = 1.0f / sqrtf(block_sum(q, red) / (float)n + eps);
  }
#pragma unroll
  for (int c = 0; c < kNormChunks; c++) {
    const int i = (c * kNormThreads + t) * 8;
    if (i < n) {
      const uint32_t ww[4] = {wv[c].x, wv[c].y, wv[c].z, wv[c].w}, bw[4] = {bv[c].x, bv[c].y, bv[c].z, bv[c].w};
      uint32_t ow[4] = {0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const float wk = (float)bits_to_h((uint16_t)(ww[k >> 1] >> (16 * (k & 1))));
        f16 o;
        if (MODE == 0) {
          o = bits_to_h((uint16_t)(ww[k >> 1] >> (16 * (k & 1)))) * rn_h(v[c][k] * r);  // fp16 multiply: same rounding
        } else {
          const float bk = (float)bits_to_h((uint16_t)(bw[k >> 1] >> (16 * (k & 1))));
          o = rn_h((v[c][k] - mean) * r * wk + bk);
        }
        ow[k >> 1] |= (uint32_t)h_to_bits(o) << (16 * (k & 1));
      }
      *reinterpret_cast<uint4*>(yr + i) = make_uint4(ow[0], ow[1], ow[2], ow[3]);
    }
  }
}

// out = fp16(fp16(silu(g)) u), silu(g) = g / (1 + exp(-g)) in f32: the
// gate activation and product of a SwiGLU MLP.  Eight elements a thread.
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ g, const uint16_t* __restrict__ u,
                                                       uint16_t* __restrict__ out, int64_t n8) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const uint4 gv = reinterpret_cast<const uint4*>(g)[i];
  const uint4 uv = reinterpret_cast<const uint4*>(u)[i];
  const uint32_t gw[4] = {gv.x, gv.y, gv.z, gv.w}, uw[4] = {uv.x, uv.y, uv.z, uv.w};
  uint32_t ow[4] = {0, 0, 0, 0};
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const float gk = (float)bits_to_h((uint16_t)(gw[k >> 1] >> (16 * (k & 1))));
    const float uk = (float)bits_to_h((uint16_t)(uw[k >> 1] >> (16 * (k & 1))));
    ow[k >> 1] |= (uint32_t)h_to_bits(silu_mul_h(gk, uk)) << (16 * (k & 1));
  }
  reinterpret_cast<uint4*>(out)[i] = make_uint4(ow[0], ow[1], ow[2], ow[3]);
}

}  // namespace

extern "C" int aq_decode_norm(void* x, const void* delta, const void* weight, const void* bias, float eps, int64_t rows,
                              int64_t n, int mode, void* y, void* stream) {
  AQ_CHECK_ARG(x && weight && y, "aq_decode_norm: null pointer");
  AQ_CHECK_ARG(mode == 0 || (mode == 1 && bias), "aq_decode_norm: mode %d (0 RMSNorm, 1 LayerNorm with bias)", mode);
  AQ_CHECK_ARG(rows > 0 && rows <= (1 << 20) && n > 0 && n % 8 == 0 && n <= kNormThreads * kNormChunks * 8,
               "aq_decode_norm: %lld rows of %lld (a multiple of 8, at most %d)", (long long)rows, (long long)n,
               kNormThreads * kNormChunks * 8);
  AQ_CHECK_ARG((uintptr_t)x % 16 == 0 && (uintptr_t)delta % 16 == 0 && (uintptr_t)weight % 16 == 0 &&
                   (uintptr_t)bias % 16 == 0 && (uintptr_t)y % 16 == 0,
               "aq_decode_norm: buffers must be 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  if (mode == 0)
    hipLaunchKernelGGL(decode_norm_kernel<0>, dim3((unsigned)rows), dim3(kNormThreads), 0, s, (uint16_t*)x,
                       (const uint16_t*)delta, (const uint16_t*)weight, (const uint16_t*)bias, eps, (int)n,
                       (uint16_t*)y);
  else
    hipLaunchKernelGGL(decode_norm_kernel<1>, dim3((unsigned)rows), dim3(kNormThreads), 0, s, (uint16_t*)x,
                       (const uint16_t*)delta, (const uint16_t*)weight, (const uint16_t*)bias, eps, (int)n,
                       (uint16_t*)y);
  AQ_LAUNCH_CHECK("aq_decode_norm");
  return AQ_OK;
}

extern "C" int aq_silu_mul(const void* g, const void* u, void* out, int64_t n, void* stream) {
  AQ_CHECK_ARG(g && u && out, "aq_silu_mul: null pointer");
  AQ_CHECK_ARG(n > 0 && n % 8 == 0, "aq_silu_mul: %lld elements (a positive multiple of 8)", (long long)n);
  AQ_CHECK_ARG((uintptr_t)g % 16 == 0 && (uintptr_t)u % 16 == 0 && (uintptr_t)out % 16 == 0,
               "aq_silu_mul: buffers must be 16-byte aligned");
  const int64_t n8 = n / 8;
  hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     (const uint16_t*)g, (const uint16_t*)u, (uint16_t*)out, n8);
  AQ_LAUNCH_CHECK("aq_silu_mul");
  return AQ_OK;
}
