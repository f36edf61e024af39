// Chunked-prefill paged attention over the INT8 arena (gfx950): the sequences of
// a step that carry more than one query token (a prompt chunk in
// PagedAttentionRunner.forward_batch, paged_attention.py:168-215), with the
// visibility rules of online_attention_statistics (online_attention.py:178-188):
// query token i of a sequence with n query tokens and context ctx (the chunk
// already appended) sits at position p = ctx - n + i and sees key k iff
//   k <= p (causal; else k < ctx)  and  k > p - window (window > 0).
//
// Work unit: (kv head, sequence, tile of TQ query tokens), TQ * G = 128 (token, head)
// columns of one kv head, 32 per wave (64 columns and half of each key step per wave where a
// head-dim 256 call leaves CUs idle, PrefillShape). The unit's visible key range is streamed in steps
// of four 16-token blocks; each wave loads one block of the step into registers and
// converts it once, one step ahead, into f16 operands in LDS that all four waves read:
//   S^T[t][c]  = K[t][:] . Q[c][:]     v_mfma_f32_32x32x16_f16: the K codes (exact in f16)
//                                        against the query, 16-bit queries exact, fp32
//                                        queries as two f16 terms
//   O^T[d][c] += V^T[d][t] . P^T[t][c]  v_mfma_f32_32x32x16_f16 (V times its f16 scale)
// so every K/V byte of the unit's range is read once per query tile and shared by
// the G heads and TQ tokens of the tile. Softmax statistics are per column, in
// base 2, with the lazy rescale of the decode kernels. Converting per workgroup instead
// of per wave and per score took a 512-token chunk on 16000 keys (bf16, int8, 32/8 heads
// of 128) from 583 to 486 us, cutting its units into key ranges (below) to 195 us.
//
// Units of one (kv head, sequence) are consecutive, longest (latest) tile first,
// and the linear workgroup id is remapped so that each XCD (workgroups are dealt
// to the 8 XCDs round robin) runs one contiguous range of units: the tiles
// sharing a sequence's K/V then share that XCD's L2.
#include <algorithm>
#include <climits>
#include <cstddef>
#include <type_traits>

#include "attention_common.h"

namespace astr {
namespace attn {
namespace {

#ifndef ASTR_KF
#define ASTR_KF 0
#endif
constexpr int KF = ASTR_KF;  // this translation unit's code format

constexpr int kXcds = 8;

// Per-wave timeline of the prefix-tile kernel (trace builds only, -DASTR_TRACE=1, built
// apart from the product library by `python -m aster_amd.build --trace`): wall-clock
// marks (100 MHz s_memrealtime) of each wave of the last launch, read back with
// astr_trace_read_tiles. Marks: 0 entry, 1 tile and members checked, 2 query columns
// quantized (the first steps' loads in flight), 3 first key step done, 4 key steps done,
// 5 partials stored. Info: key steps, XCC id, kv head, key range.
#ifndef ASTR_TRACE
#define ASTR_TRACE 0
#endif
constexpr bool kTrace = ASTR_TRACE != 0;
#if ASTR_TRACE
constexpr int kTileTraceWaves = 8192;
static __device__ long long g_ttrace[kTileTraceWaves][8];
static __device__ int g_ttrace_info[kTileTraceWaves][4];
#endif

// KS = 2: the waves are two column groups and two halves of every key step (32 of its 64
// keys), whose states merge at the unit's end: half the columns, and half the chain of MFMAs
// and operand reads per step, for grids that leave CUs idle (launch()).
template <int D, int KS = 1>
struct PrefillShape {
  static constexpr int NT = 1;                         // 32-column MFMA tiles per wave
  static constexpr int kGroups = kWaves / KS;          // column groups (waves that store)
  static constexpr int kCols = kGroups * 32 * NT;      // (token, head) columns per workgroup
};

// Workgroups per CU: the LDS holds one at head dim 256 (130 KB), the registers two at 128
// and, with 16-bit queries, three at 64 (four, 128 registers each, spill: 91.3 against
// 76.8 us for ragged FP8 prompts with their append).
template <typename QT, int D>
constexpr int prefill_occupancy() {
  return D == 256 ? 1 : D == 64 && sizeof(QT) == 2 ? 3 : 2;
}

// Keys visible to query tile `tile` (tokens [t0, t1) of the sequence's n query tokens,
// context ctx): positions [lo, hi], blocks [b_lo, b_hi).
struct TileSpan {
  int pos0, t0, t1, lo, hi, b_lo, b_hi;
};

__device__ __forceinline__ TileSpan tile_span(const AttnArgs& a, int ctx, int n, int tile, int tq) {
  TileSpan t;
  t.pos0 = ctx - n;  // position of the sequence's first query token
  t.t0 = tile * tq;
  t.t1 = min(n, t.t0 + tq);
  t.lo = a.window > 0 ? max(0, t.pos0 + t.t0 - a.window + 1) : 0;
  t.hi = a.causal ? min(t.pos0 + t.t1 - 1, ctx - 1) : ctx - 1;
  t.b_lo = t.lo / kBlockTokens;
  t.b_hi = t.hi >= t.lo ? t.hi / kBlockTokens + 1 : t.b_lo;  // exclusive
  return t;
}

constexpr int kOrderMax = 256;  // chunk rows ordered longest first; beyond this, index order

__device__ __forceinline__ int query_tiles(const ChunkArgs& a, int s, int tq) {
  int begin;
  const int n = seq_queries(a, s, begin);
  return n >= a.pf_min_rows ? (n + tq - 1) / tq : 0;
}

// The dispatch plan, from one round of loads of the offsets and context lengths, in
// the LDS table `tab` (PlanTab::kInts ints): the chunk rows (sequences with at least
// pf_min_rows query tokens) with their sequence, query offset, query count and context length
// as loaded, and the rows in dispatch order, longest first (key: key blocks of the
// row's last tile, which sees the most keys; ties by index), with the inclusive prefix
// of their tile counts in that order. Returns the number of rows and the total tile
// count, or -1 when there are more than kOrderMax rows (then every sequence is taken
// in index order by scan_tiles). Every thread calls it.
struct PlanTab {
  enum { kSeq, kTiles, kKey, kQ0, kN, kCtx, kOrder, kIncl, kArrays };
  static constexpr int kInts = kArrays * kOrderMax;
  __device__ static int* at(int* tab, int array) { return tab + array * kOrderMax; }
};

__device__ int plan_rows(const ChunkArgs& a, int tq, int* tab, int* s_wsum, int& total) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  int* const r_tiles = PlanTab::at(tab, PlanTab::kTiles);
  int* const r_key = PlanTab::at(tab, PlanTab::kKey);
  int* const o_row = PlanTab::at(tab, PlanTab::kOrder);
  int* const o_incl = PlanTab::at(tab, PlanTab::kIncl);
  int count = 0;
  for (int c0 = 0; c0 < a.num_seqs; c0 += kWaves * kWave) {
    const int s = c0 + (int)threadIdx.x;
    int key = -1, tiles = 0, q0 = 0, n = 0, ctx_raw = 0;
    if (s < a.num_seqs) {
      n = seq_queries(a, s, q0);
      if (n >= a.pf_min_rows) {
        ctx_raw = a.context_lens[s];
        const TileSpan sp = tile_span(a, clamp_ctx(a, ctx_raw, false), n, (n - 1) / tq, tq);
        key = sp.b_hi - sp.b_lo;
        tiles = (n + tq - 1) / tq;
      }
    }
    const uint64_t rows = __ballot(key >= 0);
    const int before = __builtin_popcountll(rows & ((1ull << lane) - 1));
    if (lane == 0) s_wsum[wave] = __builtin_popcountll(rows);
    __syncthreads();
    int idx = count + before;
    for (int w = 0; w < wave; ++w) idx += s_wsum[w];
    if (key >= 0 && idx < kOrderMax) {
      PlanTab::at(tab, PlanTab::kSeq)[idx] = s;
      PlanTab::at(tab, PlanTab::kQ0)[idx] = q0;
      PlanTab::at(tab, PlanTab::kN)[idx] = n;
      PlanTab::at(tab, PlanTab::kCtx)[idx] = ctx_raw;
      r_tiles[idx] = tiles;
      r_key[idx] = key;
    }
    count += s_wsum[0] + s_wsum[1] + s_wsum[2] + s_wsum[3];
    __syncthreads();
  }
  if (count > kOrderMax) return -1;
  static_assert(kOrderMax == kWaves * kWave, "one row per thread below");
  const int i = threadIdx.x;
  int tiles = 0;
  if (i < count) {
    const int k = r_key[i];
    int rank = 0;
    for (int j = 0; j < count; ++j) {
      const int kj = r_key[j];
      rank += (kj > k) | ((kj == k) & (j < i));
    }
    o_row[rank] = i;
    o_incl[rank] = r_tiles[i];
  }
  __syncthreads();
  if (i < count) tiles = o_incl[i];
  int incl = tiles;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int v = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += v;
  }
  if (lane == kWave - 1) s_wsum[wave] = incl;
  __syncthreads();
  for (int w = 0; w < wave; ++w) incl += s_wsum[w];
  if (i < count) o_incl[i] = incl;
  total = s_wsum[0] + s_wsum[1] + s_wsum[2] + s_wsum[3];
  __syncthreads();
  return count;
}

// Workgroup-wide scan of the query-tile counts of all sequences in index order. Returns
// the total; when `unit` >= 0, the sequence holding that unit and the unit's index
// within the sequence land in found[0], found[1]. Every thread calls it.
__device__ int scan_tiles(const ChunkArgs& a, int tq, int unit, int* s_wsum, int* found) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  int base = 0;
  for (int c0 = 0; c0 < a.num_seqs; c0 += kWaves * kWave) {
    const int s = c0 + (int)threadIdx.x;
    const int t = s < a.num_seqs ? query_tiles(a, s, tq) : 0;
    int incl = t;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int v = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += v;
    }
    if (lane == kWave - 1) s_wsum[wave] = incl;
    __syncthreads();
    int wb = base;
    for (int w = 0; w < wave; ++w) wb += s_wsum[w];
    incl += wb;
    if (unit >= incl - t && unit < incl) {
      found[0] = s;
      found[1] = unit - (incl - t);
    }
    base += s_wsum[0] + s_wsum[1] + s_wsum[2] + s_wsum[3];
    __syncthreads();
  }
  return base;
}

// |s| <= D 2^15 max|code as f16| for a column whose largest |q| is below 2^15; a key
// factor below this keeps every score finite (max code 127; 448 2^-8 for E4M3FN; 57344).
constexpr float safe_factor() { return KF == kInt8 ? 1.0e29f : KF == kE4M3 ? 1.0e31f : 5.0e26f; }

constexpr uint32_t kScaledBit = 4, kLargeBit = 8;  // beside a half step's block bits

// A scaled column's factor 2^ex in [kBackLeast, 1] keeps its scores (before the key factor)
// in range on either side; any other takes the edge path.
constexpr float kBackLeast = 0x1p-64f;

// A running maximum (base 2) at or below this is none yet to the key steps: they take the
// scores as they are and then the maximum of these. Reduced by it, a later score far above
// keeps only the digits that the maximum leaves it (down to kFarMax a step of 2^-13, near
// -FLT_MAX none, and the difference overflows), however ordinary the score itself is. A column
// whose scores all lie there takes the rescale on every step.
constexpr float kFarMax = -2048.f;

typedef float float16v_t __attribute__((ext_vector_type(16)));
typedef float float2_t __attribute__((ext_vector_type(2)));

// Maximum and sum over a lane and the one 32 away (v_permlane32_swap_b32: the pair of
// results holds the low half's and the high half's value in every lane).
__device__ __forceinline__ float max32(float x) {
  const uint32_t b = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}
__device__ __forceinline__ float sum32(float x) {
  const uint32_t b = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}

// The lane's index, from the lane mask: no register holds it through the key steps.
// (as an asm, so that the compiler does not work it out ahead and keep it after all)
__device__ __forceinline__ int lane_id() {
  int lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
  return lane;
}

// Query operands of one 32-column tile: B operands of the 16-wide d chunks (lane (c, h):
// column c, d = 16 cc + 8 h + [0, 8)). A 16-bit query is exact in f16 and takes one term;
// an fp32 query takes hi = f16(q) and lo = f16(q - hi), 22 bits.
template <typename QT, int D>
struct QOp {
  static constexpr int kTerms = sizeof(QT) == 4 ? 2 : 1;
  // whether the registers hold key-step operands ahead of their use beside the query's (two
  // terms at head dim 128 and 256 leave none; at head dim 64 a third wave per SIMD is worth
  // more, ragged FP8 prompts 83.9 -> 76.8 us)
  static constexpr bool kAhead = kTerms == 1 && D >= 128;
  // else how many operands are read ahead of their use (one wave per SIMD at head dim 256 has
  // no other to cover a read: 1500 tokens, 16/4 heads, 119 -> 101 us)
  static constexpr int kDepth = !kAhead && D == 256 ? 4 : 0;
  // whether a block's padding bytes are loaded with it (at head dim 256 their register spills,
  // and the spill waits for every load of the block right after its issue: 1500 tokens in bf16,
  // 16/4 heads, 98.2 us instead of 86.5)
  static constexpr bool kPad = kAhead && D < 256;
  half8_t op[kTerms][D / 16];
};

// The lane's elements of one query column as loaded.
template <typename QT, int D>
struct QueryTile {
  static constexpr int kWords = 8 * (int)sizeof(QT) / 16;  // 16-byte words per chunk
  uint4 w[D / 16][kWords];
};
template <typename QT, int D>
__device__ __forceinline__ void load_query_tile(const QT* qp, QueryTile<QT, D>& raw) {
#pragma unroll
  for (int cc = 0; cc < D / 16; ++cc)
#pragma unroll
    for (int i = 0; i < QueryTile<QT, D>::kWords; ++i)
      raw.w[cc][i] = reinterpret_cast<const uint4*>(qp + 16 * cc)[i];
}

// The column's f16 operands. A column whose largest |q| is below 2^15, and at least 2^-3
// unless q is f16 already, or 0, enters as it is: f16's own step of 2^-24 then rounds an
// element (a bf16 one below 2^-17, an fp32 one's second term) by 2^-22 of that maximum at
// most. Any other column is scaled by the exact 2^-ex that brings its maximum into [2^14,
// 2^15); the return value 2^ex (1 when unscaled, NaN for a non-finite column, which makes
// each of its scores non-finite as in fp32 arithmetic) goes back onto its scores.
// Cross-lane: uniform control flow.
template <typename QT, int D>
__device__ __forceinline__ float query_operand(const QueryTile<QT, D>& raw, bool valid,
                                               QOp<QT, D>& q) {
  float x[D / 16][8];
  float mx = 0.f;
#pragma unroll
  for (int cc = 0; cc < D / 16; ++cc) {
    const QT* e = reinterpret_cast<const QT*>(raw.w[cc]);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[cc][i] = valid ? to_float<QT>(e[i]) : 0.f;
      mx = vmax(mx, fabsf(x[cc][i]));  // NaN-propagating
    }
  }
  mx = vmax(mx, shfl_xor(mx, 32));
  constexpr float kLeast = __is_same(QT, _Float16) ? 0.f : 0x1p-3f;
  float back = 1.f;
  const bool plain = mx == 0.f || (mx >= kLeast && mx < 32768.f);
  if (__ballot(!plain) != 0) {
    int ex = 0;
    const bool finite = __builtin_isfinite(mx);
    if (!plain && finite) {
      frexpf(mx, &ex);
      ex = max(ex - 15, -126);
    }
#pragma unroll
    for (int cc = 0; cc < D / 16; ++cc)
#pragma unroll
      for (int i = 0; i < 8; ++i) x[cc][i] = ldexpf(x[cc][i], -ex);
    back = finite ? ldexpf(1.f, ex) : __builtin_nanf("");
  }
#pragma unroll
  for (int cc = 0; cc < D / 16; ++cc)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const _Float16 hi = (_Float16)x[cc][i];
      q.op[0][cc][i] = hi;
      if constexpr (QOp<QT, D>::kTerms == 2) q.op[1][cc][i] = (_Float16)(x[cc][i] - (float)hi);
    }
  return back;
}

// The LDS of one workgroup: the f16 operands of two key steps (the one computed and the
// one being converted), each of four 16-token blocks in two 32-key tiles.
//   k  A operands of S^T = K Q^T: entry (tile, chunk cc, lane (key, h)) holds
//      K[key][16 cc + 8 h + [0, 8)], the codes as f16 (exact)
//   v  A operands of O^T += V^T P^T: entry (block, n, lane (r, h)) holds, of dimension
//      d = (D / 32) r + n, the block's tokens 4 h + [0, 4) and 8 + 4 h + [0, 4), the rows
//      of S^T that lane half h holds, times the token's V scale and 2^-e of the block
//   ks the keys' score factors k_scale * qk_scale_log2 (* code_scale)
//   pad the blocks' padding bytes; flags: the block's V exponent e, plus kLargeFlag where
//   a key factor exceeds safe_factor()
constexpr int kLargeFlag = 1 << 16;
template <int D>
struct PrefillLds {
  static constexpr int kChunks = D / 16, kRowsN = D / 32;
  uint4 k[2][2 * kChunks * kWave];
  uint4 v[2][kWaves * kRowsN * kWave];
  __attribute__((aligned(16))) float ks[2][kWaves * kBlockTokens];
  __attribute__((aligned(16))) uint32_t pad[2][kWaves * 4];
  __attribute__((aligned(16))) int flags[2][kWaves];
};

// One block of the wave's own as loaded from the arena, on its way to the operands. K:
// lane (key = lane % 16, lane / 16) takes 16 consecutive d per 64. V: 16 lanes take a token
// row, D / 16 bytes each, and lane group g = lane / 16 the tokens 4 g + [0, 4): four loads
// of D / 16 bytes a lane (dwords of whole rows took eight at head dim 128, and the loads
// were 14 % of the kernel).
template <int D>
struct RawBlock {
  static constexpr int kWords = D / 64;  // dwords of a token row per lane
  uint4 k[D / 64];
  uint32_t v[4][kWords];
  float4_t vs;
  float ks;
  uint32_t pad;
  int id;
};

template <int D>
__device__ __forceinline__ uint32_t load_pad(const AttnArgs& a, int id, int lane) {
  return *reinterpret_cast<const uint32_t*>(a.cache.key_valid + (int64_t)id * kBlockTokens +
                                            4 * (lane & 3));
}

// kPad: the padding bytes too (else convert_raw reads them). Every address is a uniform
// base and a 32-bit lane offset.
template <int D, bool kPad>
__device__ __forceinline__ void load_raw(const AttnArgs& a, int id, int kvh, int lane, bool masks,
                                         RawBlock<D>& b) {
  const int64_t code = id * a.cache.code_block_stride + kvh * a.cache.code_head_stride;
  const int64_t scale = id * a.cache.scale_block_stride + kvh * a.cache.scale_head_stride;
  const int8_t* const kp = a.cache.k_codes + code;
  const int8_t* const vp = a.cache.v_codes + code;
  const float* const ksp = a.cache.k_scales + scale;
  const float* const vsp = a.cache.v_scales + scale;
  const uint32_t r = lane & 15, g = lane >> 4;
  const uint32_t koff = r * D + g * 16;
#pragma unroll
  for (int i = 0; i < D / 64; ++i) b.k[i] = *reinterpret_cast<const uint4*>(kp + (koff + 64 * i));
  struct alignas(D / 16) Row {
    uint32_t w[RawBlock<D>::kWords];
  };
  const uint32_t voff = 4 * g * D + r * (D / 16);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const Row row = *reinterpret_cast<const Row*>(vp + (voff + t * D));
#pragma unroll
    for (int i = 0; i < RawBlock<D>::kWords; ++i) b.v[t][i] = row.w[i];
  }
  b.vs = *reinterpret_cast<const float4_t*>(vsp + 4 * g);
  b.ks = ksp[r];
  b.id = id;
  if constexpr (kPad) b.pad = masks ? load_pad<D>(a, id, lane) : 0x01010101u;
}

// The wave's block into the operands of buffer `buf`, as block `w` of its step. The V
// exponent e is the unit's current `ve`, or more where a scale exceeds `vlim` = 2^(15 + ve)
// / format_max, so that every f16 product stays below 2^15.
template <int D, bool kPad>
__device__ __forceinline__ void convert_raw(const AttnArgs& a, const RawBlock<D>& b,
                                            PrefillLds<D>& L, int buf, int w, int lane, bool masks,
                                            int ve, float vlim) {
  using Lds = PrefillLds<D>;
  // K: 16 codes -> the two lane halves' entries of one chunk
  uint4* kd = L.k[buf] + (w / 2) * Lds::kChunks * kWave + 16 * (w % 2) + (lane & 15);
#pragma unroll
  for (int i = 0; i < D / 64; ++i) {
    uint4* e = kd + (4 * i + (lane >> 4)) * kWave;
    half2_t p[8];
    codes_to_f16<KF>(b.k[i].x, p[0], p[1]);
    codes_to_f16<KF>(b.k[i].y, p[2], p[3]);
    codes_to_f16<KF>(b.k[i].z, p[4], p[5]);
    codes_to_f16<KF>(b.k[i].w, p[6], p[7]);
    auto word = [&](int j) { return __builtin_bit_cast(uint32_t, p[j]); };
    e[0] = uint4{word(0), word(1), word(2), word(3)};
    e[32] = uint4{word(4), word(5), word(6), word(7)};
  }
  // V
  const float vsm = fmaxf(fmaxf(b.vs[0], b.vs[1]), fmaxf(b.vs[2], b.vs[3]));
  constexpr float cs = v_weight_scale<KF>();
  int e = ve;
  float c = cs;
  if (__ballot(vsm > vlim) != 0 || ve != 0) {
    if (__ballot(vsm > vlim) != 0) {
      float wm = 0.f;  // each group of 16 lanes holds the same scales
#pragma unroll
      for (int i = 0; i < kWave; i += 16)
        wm = fmaxf(wm, __builtin_bit_cast(float, __builtin_amdgcn_readlane(
                                                     __builtin_bit_cast(int, vsm), i)));
      int x;
      frexpf(wm * (format_max<KF>() / 32768.f), &x);  // wm * M / 2^15 in [2^(x-1), 2^x)
      e = max(ve, __builtin_amdgcn_readfirstlane(x));
    }
    c = ldexpf(cs, -e);
  }
  // dimension d = (D / 16) (lane % 16) + i is row r = d / (D / 32) of operand n =
  // d % (D / 32); the lane's quad of tokens, 2 a' + h, is half a' of lane half h's entry
  const int g = lane >> 4;
  const half4_t vsh = {(_Float16)(b.vs[0] * c), (_Float16)(b.vs[1] * c), (_Float16)(b.vs[2] * c),
                       (_Float16)(b.vs[3] * c)};
  uint2* vd = reinterpret_cast<uint2*>(L.v[buf] + w * Lds::kRowsN * kWave + 32 * (g & 1) +
                                       2 * (lane & 15)) + (g >> 1);
#pragma unroll
  for (int i = 0; i < D / 16; ++i) {
    const uint32_t col[4] = {b.v[0][i / 4], b.v[1][i / 4], b.v[2][i / 4], b.v[3][i / 4]};
    half4_t v;
    switch (i % 4) {
      case 0: v = v_operand<0, KF>(col); break;
      case 1: v = v_operand<1, KF>(col); break;
      case 2: v = v_operand<2, KF>(col); break;
      default: v = v_operand<3, KF>(col); break;
    }
    if constexpr (KF == kE5M2) {
      constexpr _Float16 down = (_Float16)(1.f / 256.f);
      v = v * half4_t{down, down, down, down};  // exact: E5M2 values times 2^-8 fit f16
    }
    vd[2 * (i % Lds::kRowsN * kWave + i / Lds::kRowsN)] = __builtin_bit_cast(uint2, v * vsh);
  }
  // key factors: a NaN scale counts as infinite, which the steps' edge path reports where a
  // key of it is seen
  float ksf = b.ks * (a.qk_scale_log2 * code_scale<KF>());
  ksf = b.ks == b.ks ? ksf : INFINITY;
  const bool large = __ballot(!(fabsf(ksf) <= safe_factor())) != 0;
  if (lane < 16) L.ks[buf][16 * w + lane] = ksf;
  if (masks && lane < 4) L.pad[buf][4 * w + lane] = kPad ? b.pad : load_pad<D>(a, b.id, lane);
  if (lane == 0) L.flags[buf][w] = e | (large ? kLargeFlag : 0);
}

// A workgroup's columns: flat column f = (wave * NT + t) * 32 + c. The unit's columns
// read query token rows q0 + tok (an invalid column reads row q0 + t0 and is zeroed)
// and see keys [lo, hi]; per wave, the bounds of its columns' key ranges (lo_min ..
// hi_max: keys some column sees; lo_max .. hi_min: keys every valid column sees) and
// whether it has a valid column.
struct ColumnInfo {
  int tok, head, lo, hi;
  bool valid;
};
struct WaveBounds {
  int lo_min, lo_max, hi_min, hi_max;
  bool any;
};

// Half a key step: the 32 keys from position kb0 on (blocks w = 0, 1 of tile kt of the
// step's operands) through the MFMAs for the wave's NT column tiles:
//   S^T = K Q^T       v_mfma_f32_32x32x16_f16 over the 16-wide d chunks
//   O^T += V^T P^T    v_mfma_f32_32x32x16_f16 over each block's 16 keys
// Lane (c, h) holds column c's scores of keys 8 a + 4 h + b (element 4 a + b), which is
// the layout that P^T enters the second product in. t = s * ks - m is the base-2 score
// over the running maximum, p = exp2(t). Bit w of `use` (wave-uniform): block w holds keys
// some column of the wave sees; of `bounded`: the column bounds [lo, hi] cut into block w.
// Further bits of `use`: kScaledBit, a column is scaled; kLargeBit, a key factor is large (and
// kScaledBit). Keys that are all used, not bounded, not padded and not large take no per-score
// condition (no score can overflow) unless a column is scaled beyond kBackLeast, only the
// scaled columns' factors; otherwise scores are masked to -inf outside the bounds, for padding
// keys and for unused blocks (which repeat the range's last one) and checked for non-finite
// values. vf: the blocks' exponent factors 2^(e_w - ve) on the weights of the numerator only,
// where `vmix`.
//
// The operands come from LDS well ahead of their MFMAs (a read takes over 100 cycles, and a
// wave that waits for each pair of them spends more time there than on the arithmetic): the
// caller passes this half's K operands, and the V operands go out before the scores.
// `between` runs ahead of the output MFMAs (it loads the next half's K operands).
template <int D>
__device__ __forceinline__ void load_k_operands(const PrefillLds<D>& L, int buf, int kt, int lane,
                                                half8_t (&kop)[D / 16]) {
  const uint4* kp = L.k[buf] + kt * PrefillLds<D>::kChunks * kWave + lane;
#pragma unroll
  for (int cc = 0; cc < D / 16; ++cc) kop[cc] = __builtin_bit_cast(half8_t, kp[cc * kWave]);
}

template <typename QT, int D, int NT, typename Between>
__device__ __forceinline__ void prefill_half(const PrefillLds<D>& L, int buf, int kt, uint32_t use,
                                             uint32_t bounded, bool masks, int kb0,
                                             half8_t (&kop)[D / 16], Between between,
                                             const QOp<QT, D> (&qop)[NT], const float (&back)[NT],
                                             const int (&lo)[NT], const int (&hi)[NT], int lane,
                                             bool vmix, half2_t vf,
                                             float16v_t (&acc)[NT][D / 32], float (&m)[NT],
                                             float (&l)[NT], bool& bad_score) {
  using Lds = PrefillLds<D>;
  const int h = lane >> 5;
  bool padded = false;
  if (masks) {
    const uint4 pw = *reinterpret_cast<const uint4*>(&L.pad[buf][8 * kt + 4 * (lane & 1)]);
    padded = __ballot(pw.x != 0x01010101u || pw.y != 0x01010101u || pw.z != 0x01010101u ||
                      pw.w != 0x01010101u) != 0;
  }
  constexpr int kAhead = QOp<QT, D>::kAhead ? 2 * Lds::kRowsN : 0;
  half8_t vop[2 * Lds::kRowsN];
  auto load_v = [&](int n0, int n1) __attribute__((always_inline)) {
#pragma unroll
    for (int n = n0; n < n1; ++n)
      vop[n] = __builtin_bit_cast(half8_t, L.v[buf][(2 * kt * Lds::kRowsN + n) * kWave + lane]);
  };
  if constexpr (QOp<QT, D>::kAhead) {
    load_v(0, kAhead);
    __builtin_amdgcn_sched_barrier(0);
  }
  constexpr int kDepth = QOp<QT, D>::kDepth;
  auto load_k = [&](int cc) __attribute__((always_inline)) {
    kop[cc] = __builtin_bit_cast(half8_t, L.k[buf][(kt * Lds::kChunks + cc) * kWave + lane]);
  };
#pragma unroll
  for (int cc = 0; cc < kDepth; ++cc) load_k(cc);
  float16v_t s[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) s[t][j] = 0.f;
#pragma unroll
  for (int cc = 0; cc < Lds::kChunks; ++cc) {
    if constexpr (kDepth > 0) {
      __builtin_amdgcn_sched_barrier(0);
      if (cc + kDepth < Lds::kChunks) load_k(cc + kDepth);
    } else if constexpr (!QOp<QT, D>::kAhead) {
      load_k(cc);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int x = 0; x < QOp<QT, D>::kTerms; ++x)
        s[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kop[cc], qop[t].op[x][cc], s[t], 0, 0, 0);
  }
  float4_t ks[4];  // factors of keys 8 x + 4 h + [0, 4)
#pragma unroll
  for (int x = 0; x < 4; ++x)
    ks[x] = *reinterpret_cast<const float4_t*>(&L.ks[buf][32 * kt + 8 * x + 4 * h]);
  if constexpr (QOp<QT, D>::kAhead) __builtin_amdgcn_sched_barrier(0);
  if (use != 3u || bounded != 0 || padded) {
    asm volatile("");  // keeps this a branch: if-converted, the interior steps would pay for it
    bool factors = use == (3u | kScaledBit) && bounded == 0 && !padded;  // those alone?
    if (factors) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
        factors = factors && __ballot(!(back[t] <= 1.f && back[t] >= kBackLeast)) == 0;
    }
    if (factors) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) s[t][j] *= back[t];
    } else {
      // Per-score masks as all-ones/zero words in VGPRs (sign bits of differences, bit
      // selects): lane masks of unrolled compares would stay live in SGPRs and spill.
      uint32_t nonfinite = 0;
      uint32_t pads[4] = {0x01010101u, 0x01010101u, 0x01010101u, 0x01010101u};
      if (masks) {
#pragma unroll
        for (int x = 0; x < 4; ++x) pads[x] = L.pad[buf][8 * kt + 2 * x + h];
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int w = x / 2;
        const uint32_t pad = pads[x];
        const bool used = (use >> w) & 1u, bnd = (bounded >> w) & 1u;  // wave-uniform
#pragma unroll
        for (int y = 0; y < 4; ++y) {
          const int j = 4 * x + y;
          const int key = kb0 + 8 * x + 4 * h + y;
          const int32_t padding = (int32_t)(((pad >> (8 * y)) & 0xffu) - 1u) >> 31;  // -1: padding
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            // -1 when key < lo or key > hi (either difference negative), else 0
            const int32_t outside = bnd ? ((key - lo[t]) | (hi[t] - key)) >> 31 : 0;
            const uint32_t hide = used ? (uint32_t)(outside | padding) : 0xffffffffu;
            // (the factors first: a large query's beside a small key's stays in range)
            const uint32_t xb = __builtin_bit_cast(uint32_t, s[t][j] * (back[t] * ks[x][y]));
            // exponent field all ones (inf or NaN) -> bit 31 after the carry
            nonfinite |= ((xb & 0x7f800000u) + 0x00800000u) & ~hide;
            s[t][j] = __builtin_bit_cast(float, (xb & ~hide) | (0xff800000u & hide));  // -inf
          }
          static_assert(NT == 1, "the scores hold the one column tile's factors from here on");
          ks[x][y] = 1.f;
        }
      }
      if (__ballot((nonfinite >> 31) != 0) != 0) bad_score = true;
    }
  }
  bool need = false;
  float me[NT], tmax[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    me[t] = m[t] > kFarMax ? m[t] : 0.f;  // (and in a column without a key so far)
    float mu = -INFINITY;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      s[t][j] = __builtin_fmaf(s[t][j], ks[j / 4][j % 4], -me[t]);
      mu = vmax(mu, s[t][j]);  // NaN-propagating
    }
    tmax[t] = mu;
    need |= !(mu <= kRescaleSlack) || m[t] <= kFarMax;
  }
  if (__ballot(need) != 0) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float x = max32(tmax[t]) + me[t];
      const float mn = fmaxf(m[t], x);
      const float alpha = __builtin_amdgcn_exp2f(m[t] - mn);
      const float shift = (mn > -FLT_MAX ? mn : 0.f) - me[t];
#pragma unroll
      for (int n = 0; n < Lds::kRowsN; ++n) acc[t][n] *= alpha;
      l[t] *= alpha;
      m[t] = mn;
#pragma unroll
      for (int j = 0; j < 16; ++j) s[t][j] -= shift;
    }
  }
  // weights rounded to f16; the sums take the same rounded weights as the numerator
  typedef uint32_t word4_t __attribute__((ext_vector_type(4)));
  word4_t pop[NT][2];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i0 = 8 * w + 2 * j;
        const uint32_t pair = pack2<_Float16>(__builtin_amdgcn_exp2f(s[t][i0]),
                                              __builtin_amdgcn_exp2f(s[t][i0 + 1]));
        l[t] = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, pair),
                                      half2_t{(_Float16)1.f, (_Float16)1.f}, l[t], false);
        pop[t][w][j] = pair;
      }
  if constexpr (QOp<QT, D>::kAhead) {
    load_v(kAhead, 2 * Lds::kRowsN);
    between();
    __builtin_amdgcn_sched_barrier(0);
  }
  load_v(0, kDepth);
  // (the sums are done here: sunk past the branch, they would keep a second copy of the weights)
#pragma unroll
  for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(l[t]));
  if (__builtin_expect(vmix, 0)) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const _Float16 f = vf[w];
        pop[t][w] = __builtin_bit_cast(word4_t, __builtin_bit_cast(half8_t, pop[t][w]) *
                                                    half8_t{f, f, f, f, f, f, f, f});
      }
  }
#pragma unroll
  for (int w = 0; w < 2; ++w)
#pragma unroll
    for (int n = 0; n < Lds::kRowsN; ++n) {
      const int x = w * Lds::kRowsN + n;
      if constexpr (kDepth > 0) {
        __builtin_amdgcn_sched_barrier(0);
        if (x + kDepth < 2 * Lds::kRowsN) load_v(x + kDepth, x + kDepth + 1);
      } else if constexpr (!QOp<QT, D>::kAhead) {
        load_v(x, x + 1);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[t][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
            vop[x], __builtin_bit_cast(half8_t, pop[t][w]), acc[t][n], 0, 0, 0);
    }
}

// N consecutive outputs from fp32, with 16-byte stores.
template <typename QT, int N>
__device__ __forceinline__ void store_run(QT* dst, const float (&v)[N]) {
  constexpr int kVec = 16 / (int)sizeof(QT);
  static_assert(N % kVec == 0, "whole 16-byte stores");
#pragma unroll
  for (int c = 0; c < N / kVec; ++c) {
    uint4 w;
    if constexpr (sizeof(QT) == 2) {
      w = uint4{pack2<QT>(v[8 * c], v[8 * c + 1]), pack2<QT>(v[8 * c + 2], v[8 * c + 3]),
                pack2<QT>(v[8 * c + 4], v[8 * c + 5]), pack2<QT>(v[8 * c + 6], v[8 * c + 7])};
    } else {
      QT* e = reinterpret_cast<QT*>(&w);
#pragma unroll
      for (int i = 0; i < kVec; ++i) e[i] = from_float<QT>(v[c * kVec + i]);
    }
    reinterpret_cast<uint4*>(dst)[c] = w;
  }
}

// The D / 8 consecutive outputs that lane half h holds of its column in accumulator rows
// 8 x + 4 h + [0, 4): elements D / 4 x + D / 8 h + [0, D / 8).
template <int D>
__device__ __forceinline__ void acc_run(const float16v_t (&acc)[D / 32], int x, float scale,
                                        float (&v)[D / 8]) {
#pragma unroll
  for (int y = 0; y < 4; ++y)
#pragma unroll
    for (int n = 0; n < D / 32; ++n) v[y * (D / 32) + n] = acc[n][4 * x + y] * scale;
}

// One unit of the chunked-prefill kernels: the key blocks [b_lo, b_hi) of kv head kvh
// (physical id of block b: blocks[b], a window of the arena's ids) against the
// workgroup's query columns (column_of(f), bounds_of(wave)), through the key steps
// described at the top of this file; store(t, acc, m, l, ve, col) then takes column
// tile t of each wave (acc in units of 2^-ve, l the sums of the column's weights).
// prologue() runs (in uniform control flow) once the first block id is on its way,
// before any column is read: it returns false (uniformly) to end the unit there, with
// nothing stored. mark(k) is called at the unit's timeline marks 2-5 (the tile kernel's
// trace builds).
template <typename QT, int D, int KS, typename ColumnOf, typename BoundsOf, typename Store,
          typename Prologue, typename Mark>
__device__ __forceinline__ void prefill_unit(const AttnArgs& a, PrefillLds<D>& L, int kvh,
                                             int b_lo, int b_hi, const int32_t* blocks, int q0,
                                             int t0, ColumnOf column_of, BoundsOf bounds_of,
                                             Store store, Prologue prologue, Mark mark) {
  using Shape = PrefillShape<D, KS>;
  constexpr int NT = Shape::NT;
  constexpr int kRowsN = D / 32;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lane = threadIdx.x % kWave;
  const int group = KS == 1 ? wave : wave % Shape::kGroups;
  const int half = KS == 1 ? 0 : wave / Shape::kGroups;
  const int nsteps = (b_hi - b_lo + kWaves - 1) / kWaves;

  // Block b_lo + 4 * step + w is wave w's; its id is read (a scalar load) one step before
  // its block. A block past the range repeats the last one (its keys are not used).
  typedef const __attribute__((address_space(4))) int32_t* scalar_ids_t;
  const scalar_ids_t sids = (scalar_ids_t)blocks;
  auto id_of = [&](int step) __attribute__((always_inline)) -> int {
    return sids[min(b_lo + step * kWaves + wave, b_hi - 1)];
  };
  int next_id = nsteps > 0 ? id_of(0) : 0;
  __syncthreads();  // what the stage memory held before (the dispatch plan) has been read
  if (!prologue()) return;

  int lo[NT], hi[NT];
  QueryTile<QT, D> qraw[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const ColumnInfo c = column_of((group * NT + t) * 32 + (lane & 31));
    lo[t] = c.valid ? c.lo : INT_MAX;
    hi[t] = c.valid ? c.hi : -1;
    // an invalid column reads token t0's row (in range) and is zeroed
    load_query_tile<QT, D>(static_cast<const QT*>(a.q) + (int64_t)(q0 + (c.valid ? c.tok : t0)) * a.q_tok +
                               (int64_t)c.head * a.q_head + 8 * (lane >> 5), qraw[t]);
  }

  bool bad_index = false, bad_score = false;
  const bool masks = a.cache.key_valid != nullptr;  // the arena has key padding bytes
  RawBlock<D> raw;
  auto load_step = [&](int step) __attribute__((always_inline)) {
    int id = next_id;
    if (step + 1 < nsteps) next_id = id_of(step + 1);
    if ((unsigned)id >= (unsigned)a.cache.num_blocks) {
      bad_index = true;
      id = 0;
    }
    load_raw<D, QOp<QT, D>::kPad>(a, id, kvh, lane, masks, raw);
  };
  if (QOp<QT, D>::kAhead && nsteps > 0) load_step(0);

  QOp<QT, D> qop[NT];
  float back[NT];
  bool scaled = false;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    back[t] = query_operand<QT, D>(qraw[t], hi[t] >= 0, qop[t]);
    scaled |= __ballot(back[t] != 1.f) != 0;
  }
  const WaveBounds wb = bounds_of(group);
  mark(2);

  float16v_t acc[NT][kRowsN];
  float m[NT], l[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
#pragma unroll
    for (int n = 0; n < kRowsN; ++n)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[t][n][j] = 0.f;
    m[t] = -FLT_MAX;
    l[t] = 0.f;
  }
  // The PV accumulators are in units of 2^-ve: ve is the largest block exponent so far
  // (0 unless a block's V scales need more, see convert_raw); vlim is its scale limit.
  int ve = 0;
  float vlim = 32768.f / format_max<KF>();

  // steps [inner_lo, inner_hi) see every key of theirs with every valid column
  const int keys0 = b_lo * kBlockTokens;
  constexpr int kStepKeys = kWaves * kBlockTokens;
  const int inner_lo = max(0, (wb.lo_max - keys0 + kStepKeys - 1) / kStepKeys);
  const int inner_end = min(wb.hi_min, b_hi * kBlockTokens - 1) + 1 - keys0;
  const int inner_hi = wb.any && inner_end > 0 ? inner_end / kStepKeys : 0;
  if (nsteps > 0) {
    if constexpr (!QOp<QT, D>::kAhead) load_step(0);
    convert_raw<D, QOp<QT, D>::kPad>(a, raw, L, 0, wave, lane, masks, ve, vlim);
    if (nsteps > 1) load_step(1);
    __syncthreads();
  }
  for (int i = 0; i < nsteps; ++i) {
    const int buf = i & 1;
    half8_t kop[D / 16];
    if constexpr (QOp<QT, D>::kAhead) load_k_operands<D>(L, buf, KS == 2 ? half : 0, lane, kop);
    // the step's block exponents (each at least ve at its conversion): a larger one
    // becomes the new ve (the accumulators scale by the exact 2^(ve_old - ve)); blocks
    // converted below it weigh their products by 2^(e_w - ve)
    const int4_t fv = *reinterpret_cast<const int4_t*>(L.flags[buf]);
    const int f0 = __builtin_amdgcn_readfirstlane(fv[0]), f1 = __builtin_amdgcn_readfirstlane(fv[1]);
    const int f2 = __builtin_amdgcn_readfirstlane(fv[2]), f3 = __builtin_amdgcn_readfirstlane(fv[3]);
    bool vmix = false;
    uint32_t slow = scaled ? kScaledBit : 0u;
    half4_t vf = {(_Float16)1.f, (_Float16)1.f, (_Float16)1.f, (_Float16)1.f};
    if (__builtin_expect((f0 | f1 | f2 | f3 | ve) != 0, 0)) {
      if (((f0 | f1 | f2 | f3) & kLargeFlag) != 0) slow = kScaledBit | kLargeBit;
      const int e4[kWaves] = {f0 & (kLargeFlag - 1), f1 & (kLargeFlag - 1), f2 & (kLargeFlag - 1),
                              f3 & (kLargeFlag - 1)};
      const int emax = max(max(e4[0], e4[1]), max(e4[2], e4[3]));
      if (emax > ve) {
        const float down = ldexpf(1.f, ve - emax);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int n = 0; n < kRowsN; ++n) acc[t][n] *= down;
        ve = emax;
        vlim = ldexpf(32768.f / format_max<KF>(), ve);
      }
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        vmix |= e4[w] != ve;
        vf[w] = (_Float16)ldexpf(1.f, e4[w] - ve);
      }
    }
    const int kb0 = (b_lo + i * kWaves) * kBlockTokens;
    uint32_t use = 15, bounded = 0;
    if (i < inner_lo || i >= inner_hi) {
      const int kend = b_hi * kBlockTokens;
      use = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const int kb = kb0 + w * kBlockTokens;
        if (wb.any && kb < kend && kb <= wb.hi_max && kb + kBlockTokens - 1 >= wb.lo_min)
          use |= 1u << w;
        if (!(kb >= wb.lo_max && kb + kBlockTokens - 1 <= wb.hi_min)) bounded |= 1u << w;
      }
      bounded &= use;
    }
    if constexpr (KS == 2) {
      const uint32_t mine = use >> (2 * half) & 3u;
      if (mine != 0)
        prefill_half<QT, D, NT>(L, buf, half, mine | slow, bounded >> (2 * half) & 3u, masks,
                                kb0 + 32 * half, kop, []() {}, qop, back, lo, hi, lane, vmix,
                                half != 0 ? half2_t{vf[2], vf[3]} : half2_t{vf[0], vf[1]}, acc, m,
                                l, bad_score);
    } else if (use != 0) {
      prefill_half<QT, D, NT>(L, buf, 0, (use & 3u) | slow, bounded & 3u, masks, kb0, kop,
                              [&]() __attribute__((always_inline)) {
                                load_k_operands<D>(L, buf, 1, lane, kop);
                              },
                              qop, back, lo, hi, lane, vmix, half2_t{vf[0], vf[1]}, acc, m, l,
                              bad_score);
      prefill_half<QT, D, NT>(L, buf, 1, use >> 2 | slow, bounded >> 2, masks, kb0 + 32, kop,
                              []() {}, qop, back, lo, hi, lane, vmix, half2_t{vf[2], vf[3]}, acc,
                              m, l, bad_score);
    }
    if (i + 1 < nsteps) {
      // the other buffer was last read in step i - 1, before the barrier that ended it
      convert_raw<D, QOp<QT, D>::kPad>(a, raw, L, buf ^ 1, wave, lane, masks, ve, vlim);
      if (i + 2 < nsteps) load_step(i + 2);
    }
    __syncthreads();
    if (i == 0) mark(3);
  }
  mark(4);
  if (bad_index && lane == 0) atomicOr(a.err_flag, ASTR_FLAG_BAD_INDEX);
  if (bad_score && lane == 0) atomicOr(a.err_flag, ASTR_FLAG_NONFINITE_SCORE);
  if constexpr (KS == 2) {
    // the second half's state through the operand buffers (last read before the barrier that
    // ended the last step), in the merge_softmax rule (online_attention.py:42-63)
    static_assert(Shape::kGroups * kRowsN * 4 * kWave * sizeof(float4_t) <= sizeof(L.k) &&
                      Shape::kGroups * kWave * sizeof(float2_t) <= sizeof(L.v),
                  "the groups' states fit the buffers");
    float4_t* const o = reinterpret_cast<float4_t*>(L.k) + group * kRowsN * 4 * kWave + lane;
    float2_t* const ml = reinterpret_cast<float2_t*>(L.v) + group * kWave + lane;
    if (half != 0) {
#pragma unroll
      for (int n = 0; n < kRowsN; ++n)
#pragma unroll
        for (int x = 0; x < 4; ++x)
          o[(n * 4 + x) * kWave] = float4_t{acc[0][n][4 * x], acc[0][n][4 * x + 1],
                                            acc[0][n][4 * x + 2], acc[0][n][4 * x + 3]};
      *ml = float2_t{m[0], l[0]};
    }
    __syncthreads();
    if (half != 0) return;
    const float2_t other = *ml;
    const float mn = fmaxf(m[0], other[0]);
    const float w0 = __builtin_amdgcn_exp2f(m[0] - mn), w1 = __builtin_amdgcn_exp2f(other[0] - mn);
    m[0] = mn;
    l[0] = l[0] * w0 + other[1] * w1;
#pragma unroll
    for (int n = 0; n < kRowsN; ++n)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float4_t v = o[(n * 4 + x) * kWave];
#pragma unroll
        for (int y = 0; y < 4; ++y)
          acc[0][n][4 * x + y] = fmaf(v[y], w1, acc[0][n][4 * x + y] * w0);
      }
  }

#pragma unroll
  for (int t = 0; t < NT; ++t) {
    // worked out again: kept through the steps it would cost registers (the empty asm hides
    // that it is the same value)
    int f = (group * NT + t) * 32 + (lane_id() & 31);
    asm volatile("" : "+v"(f));
    store(t, acc[t], m[t], sum32(l[t]), ve, column_of(f));
  }
  mark(5);
}

// A unit of the prefill launch: query tile `tile` of sequence `seq`.
struct UnitRef {
  int seq, tile, q0, n, ctx_raw;
  bool last;  // the sequence's last tile
};

// Units of one kv head, from the dispatch plan (in `tab` when rows >= 0) or the scan in
// index order beyond kOrderMax rows. Every thread calls both.
__device__ __forceinline__ int count_units(const ChunkArgs& a, int tq, int* tab, int* s_wsum,
                                           int* s_found, int& rows) {
  int per_kv = 0;
  rows = plan_rows(a, tq, tab, s_wsum, per_kv);
  if (rows < 0) per_kv = scan_tiles(a, tq, -1, s_wsum, s_found);
  return per_kv;
}
__device__ __forceinline__ bool unit_ref(const ChunkArgs& a, int tq, int* tab, int* s_wsum,
                                         int* s_found, int rows, int unit, UnitRef& u) {
  int within;
  if (rows >= 0) {
    // the first row whose inclusive prefix exceeds the unit (prefixes strictly grow)
    const int* const o_incl = PlanTab::at(tab, PlanTab::kIncl);
    int lo_r = 0, hi_r = rows - 1;
    while (lo_r < hi_r) {
      const int mid = (lo_r + hi_r) / 2;
      if (o_incl[mid] > unit) hi_r = mid;
      else lo_r = mid + 1;
    }
    // uniform values read from LDS: readfirstlane keeps them (and all they derive) scalar
    const int row = __builtin_amdgcn_readfirstlane(PlanTab::at(tab, PlanTab::kOrder)[lo_r]);
    within = __builtin_amdgcn_readfirstlane(unit - (lo_r > 0 ? o_incl[lo_r - 1] : 0));
    u.seq = __builtin_amdgcn_readfirstlane(PlanTab::at(tab, PlanTab::kSeq)[row]);
    u.q0 = __builtin_amdgcn_readfirstlane(PlanTab::at(tab, PlanTab::kQ0)[row]);
    u.n = __builtin_amdgcn_readfirstlane(PlanTab::at(tab, PlanTab::kN)[row]);
    u.ctx_raw = __builtin_amdgcn_readfirstlane(PlanTab::at(tab, PlanTab::kCtx)[row]);
  } else {
    if (threadIdx.x == 0) s_found[0] = -1;  // ordered before the scan's writes by its barriers
    scan_tiles(a, tq, unit, s_wsum, s_found);
    u.seq = __builtin_amdgcn_readfirstlane(s_found[0]);
    within = __builtin_amdgcn_readfirstlane(s_found[1]);
    if (u.seq < 0) return false;  // unreachable for unit < per_kv; keeps every index in range
    u.n = seq_queries(a, u.seq, u.q0);
    u.ctx_raw = a.context_lens[u.seq];
  }
  const int tiles = (u.n + tq - 1) / tq;
  u.tile = tiles - 1 - within;  // latest (longest) tiles first
  u.last = within == 0;
  return true;
}

// The partial of one piece of a split unit: the accumulators as the lanes hold them
// (float4 x of operand n of wave w at ((w * D / 32 + n) * 4 + x) * 64 + lane), then (m, l)
// per column.
template <int D, int KS>
struct PiecePartial {
  static constexpr int kAcc = PrefillShape<D, KS>::kGroups * (D / 32) * 4 * kWave * 4;  // floats
  static constexpr int kFloats = kAcc + PrefillShape<D, KS>::kCols * 2;
  static_assert(PrefillShape<D, KS>::NT == 1, "one column tile per wave");
  __device__ static float4_t* acc(float* base, int wave, int n, int x, int lane) {
    return reinterpret_cast<float4_t*>(base) + ((wave * (D / 32) + n) * 4 + x) * kWave + lane;
  }
};

// The outputs of one column of each lane pair, normalised (fully masked columns: l = 0,
// acc = 0 -> 0).
template <typename QT, int D>
__device__ __forceinline__ void store_column(const AttnArgs& a, const float16v_t (&acc)[D / 32],
                                             float inv, int token, int head, int lane) {
  QT* op = static_cast<QT*>(a.out) + (int64_t)token * a.o_tok + (int64_t)head * a.o_head +
           D / 8 * (lane >> 5);
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    float v[D / 8];
    acc_run<D>(acc, x, inv, v);
    store_run<QT, D / 8>(op + D / 4 * x, v);
  }
}

template <typename QT, int D, int G, int KS>
__global__ __launch_bounds__(256, (prefill_occupancy<QT, D>())) void prefill_mfma_kernel(ChunkArgs a) {
  static_assert(D == 64 || D == 128 || D == 256, "head_dim");
  constexpr int NT = PrefillShape<D, KS>::NT;
  constexpr int TQ = PrefillShape<D, KS>::kCols / G;
  static_assert(PrefillShape<D, KS>::kCols % G == 0, "GQA group must divide the column tile");

  // one struct, the operand buffers at its start: every LDS address of the key steps then
  // has a constant offset
  __shared__ struct {
    PrefillLds<D> unit;
    int wsum[kWaves], found[2];
  } lds;
  PrefillLds<D>& L = lds.unit;

  const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int hkv = a.cache.num_kv_heads;

  // ---- 1. this workgroup's unit (uniform over the workgroup). The plan lives in the
  // operand buffers until the first conversion.
  static_assert(PlanTab::kInts * sizeof(int) <= sizeof(L.k), "the dispatch plan fits the buffers");
  int* const tab = reinterpret_cast<int*>(L.k);
  int rows;
  const int per_kv = count_units(a, TQ, tab, lds.wsum, lds.found, rows);
  const int64_t units = (int64_t)per_kv * hkv * a.pf_pieces;
  const int64_t per_xcd = (units + kXcds - 1) / kXcds;
  int64_t slot = blockIdx.x / kXcds;
  if (slot >= per_xcd) return;
  // Where every unit is resident at once, an XCD's CUs take its units in rows of one per
  // CU, longest first: every second row is reversed, so that the CU with the longest unit
  // of one gets the shortest of the next (a causal prompt's tiles grow linearly).
  if (per_xcd <= (int64_t)prefill_occupancy<QT, D>() * a.pf_cus) {
    const int64_t r = slot / a.pf_cus, c = slot % a.pf_cus;
    const int64_t len = min((int64_t)a.pf_cus, per_xcd - r * a.pf_cus);
    if (r & 1) slot = r * a.pf_cus + len - 1 - c;
  }
  const int64_t logical = (int64_t)(blockIdx.x % kXcds) * per_xcd + slot;
  if (logical >= units) return;
  const int piece = (int)(logical % a.pf_pieces);
  const int head_unit = (int)(logical / a.pf_pieces);
  const int kvh = head_unit / per_kv;
  UnitRef u;
  if (!unit_ref(a, TQ, tab, lds.wsum, lds.found, rows, head_unit % per_kv, u)) return;
  const int seq = u.seq, q0 = u.q0, n = u.n;
  const bool reporter = kvh == 0 && u.last && threadIdx.x == 0;
  const int ctx = clamp_ctx(a, u.ctx_raw, reporter);
  // chunk longer than the context (a one-token row may be empty, as in a decode launch)
  if (ctx < n && n > 1 && reporter) atomicOr(a.err_flag, ASTR_FLAG_BAD_INDEX);

  TileSpan span = tile_span(a, ctx, n, u.tile, TQ);
  const int pos0 = span.pos0, t0 = span.t0, t1 = span.t1;
  // the piece's key steps; a unit within pf_steps is its first piece alone
  float* part = nullptr;
  if (a.pf_pieces > 1) {
    const int steps = (span.b_hi - span.b_lo + kWaves - 1) / kWaves;
    if (piece > 0 && piece * a.pf_steps >= steps) return;
    if (steps > a.pf_steps) {
      if ((uint64_t)(logical + 1) * PiecePartial<D, KS>::kFloats * sizeof(float) > a.pf_bytes) {
        if (threadIdx.x == 0) atomicOr(a.err_flag, ASTR_FLAG_BAD_INDEX);  // offsets past the bound
        return;
      }
      part = a.pf_ws + logical * PiecePartial<D, KS>::kFloats;
      span.b_lo += piece * a.pf_steps * kWaves;
      // (the last piece takes whatever a context past the host's bound adds)
      if (piece < a.pf_pieces - 1) span.b_hi = min(span.b_hi, span.b_lo + a.pf_steps * kWaves);
    }
  }

  // flat column f -> token t0 + f / G, head kvh * G + f % G, keys by its position
  auto column_of = [&](int f) __attribute__((always_inline)) -> ColumnInfo {
    const int tok = t0 + f / G;
    const int p = pos0 + tok;
    return ColumnInfo{tok, kvh * G + f % G, a.window > 0 ? max(0, p - a.window + 1) : 0,
                      a.causal ? p : ctx - 1, tok < t1};
  };
  // key bounds over the wave's valid columns (positions grow with f)
  auto bounds_of = [&](int wave) __attribute__((always_inline)) -> WaveBounds {
    const int tk_lo = t0 + (wave * NT * 32) / G;
    const int tk_hi = min(t1 - 1, t0 + ((wave + 1) * NT * 32 - 1) / G);
    return WaveBounds{a.window > 0 ? max(0, pos0 + tk_lo - a.window + 1) : 0,
                      a.window > 0 ? max(0, pos0 + tk_hi - a.window + 1) : 0,
                      a.causal ? pos0 + tk_lo : ctx - 1, a.causal ? pos0 + tk_hi : ctx - 1,
                      tk_lo < t1};
  };
  auto store = [&](int, const float16v_t (&acc)[D / 32], float m, float l, int ve,
                   const ColumnInfo& c) __attribute__((always_inline)) {
    const float up = ldexpf(1.f, ve);  // the PV tiles carry 2^-ve
    const int lane = lane_id();
    if (part != nullptr) {
#pragma unroll
      for (int k = 0; k < D / 32; ++k)
#pragma unroll
        for (int x = 0; x < 4; ++x)
          *PiecePartial<D, KS>::acc(part, wave_id, k, x, lane) =
              float4_t{acc[k][4 * x] * up, acc[k][4 * x + 1] * up, acc[k][4 * x + 2] * up,
                       acc[k][4 * x + 3] * up};
      if (lane < 32) {
        float* ml = part + PiecePartial<D, KS>::kAcc + (wave_id * 32 + lane) * 2;
        ml[0] = m;
        ml[1] = l;
      }
    } else if (c.valid) {
      store_column<QT, D>(a, acc, up / fmaxf(l, FLT_MIN), q0 + c.tok, c.head, lane);
    }
  };
  prefill_unit<QT, D, KS>(a, L, kvh, span.b_lo, span.b_hi,
                      a.block_tables + (int64_t)seq * a.bt_stride, q0, t0, column_of,
                      bounds_of, store, []() { return true; }, [](int) {});
}

constexpr int kMostPieces = 16;

// Merges the pieces of split units with the merge_softmax rule (online_attention.py:42-63). A
// lane takes one of the four parts of its column as it held it in the pieces: a workgroup one
// part of a unit's 128 columns, or two of 64 (KS = 2). Bound by the chain of its loads: the statistics
// and the first pieces' rows, whose place the unit's index alone gives, are on their way while
// the dispatch plan is worked out (a place past the unit's own pieces is read, inside the
// workspace, and not used). 512 tokens on 16000 (32/8 heads of 128: 34 MB of
// partials) 14.1 -> 10.1 us against a workgroup per unit that read the plan, the statistics and
// the rows of one piece after another; 256 tokens on 8000 (16/4 heads, 16 pieces a unit) 71.0 ->
// 47.1 us a call.
template <int D>
struct MergeShape {
  static constexpr int kParts = 4;         // parts of a lane's column
  static constexpr int kRows = D / 32;     // float4 rows of one in a piece
  static constexpr int kAtOnce = 512 / D;  // pieces whose rows are in flight together
};

template <typename QT, int D, int G, int KS>
__global__ __launch_bounds__(256) void prefill_merge_kernel(ChunkArgs a) {
  using Shape = PrefillShape<D, KS>;
  using Partial = PiecePartial<D, KS>;
  using M = MergeShape<D>;
  constexpr int TQ = Shape::kCols / G;
  constexpr int kGrid = M::kParts / KS;  // workgroups per unit
  __shared__ int tab[PlanTab::kInts];
  __shared__ int s_wsum[kWaves], s_found[2];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int group = wave % Shape::kGroups;
  const int part = (int)(blockIdx.x % kGrid) * KS + wave / Shape::kGroups;
  const int unit = blockIdx.x / kGrid;
  const int64_t first = (int64_t)unit * a.pf_pieces;
  if ((uint64_t)(first + a.pf_pieces) * Partial::kFloats * sizeof(float) > a.pf_bytes) return;
  float* const base = a.pf_ws + first * Partial::kFloats;

  const int col = Partial::kAcc + (group * 32 + (lane & 31)) * 2;
  float2_t ml[kMostPieces];
#pragma unroll
  for (int j = 0; j < kMostPieces; ++j)
    if (j < a.pf_pieces)
      ml[j] = *reinterpret_cast<const float2_t*>(base + j * (int64_t)Partial::kFloats + col);
  float4_t v[M::kAtOnce][M::kRows];
  auto load_rows = [&](int j0, int pieces) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < M::kAtOnce; ++j)
      if (j0 + j < pieces)
#pragma unroll
        for (int n = 0; n < M::kRows; ++n)
          v[j][n] = *Partial::acc(base + (j0 + j) * (int64_t)Partial::kFloats, group, n, part, lane);
  };
  load_rows(0, a.pf_pieces);

  int rows;
  const int per_kv = count_units(a, TQ, tab, s_wsum, s_found, rows);
  if ((int64_t)unit >= (int64_t)per_kv * a.cache.num_kv_heads) return;
  const int kvh = unit / per_kv;
  UnitRef u;
  if (!unit_ref(a, TQ, tab, s_wsum, s_found, rows, unit % per_kv, u)) return;
  const TileSpan span = tile_span(a, clamp_ctx(a, u.ctx_raw, false), u.n, u.tile, TQ);
  const int steps = (span.b_hi - span.b_lo + kWaves - 1) / kWaves;
  const int pieces = min((steps + a.pf_steps - 1) / a.pf_steps, a.pf_pieces);
  if (pieces <= 1) return;
  float mx = -FLT_MAX;
#pragma unroll
  for (int j = 0; j < kMostPieces; ++j)
    if (j < pieces) mx = fmaxf(mx, ml[j][0]);
  float4_t acc[M::kRows];
#pragma unroll
  for (int n = 0; n < M::kRows; ++n) acc[n] = float4_t{};
  float l = 0.f;
#pragma unroll
  for (int j0 = 0; j0 < kMostPieces; j0 += M::kAtOnce) {
    if (j0 > 0) load_rows(j0, pieces);
#pragma unroll
    for (int j = 0; j < M::kAtOnce; ++j)
      if (j0 + j < pieces) {
        const float w = __builtin_amdgcn_exp2f(ml[j0 + j][0] - mx);
        l = fmaf(ml[j0 + j][1], w, l);
#pragma unroll
        for (int n = 0; n < M::kRows; ++n)
#pragma unroll
          for (int y = 0; y < 4; ++y) acc[n][y] = fmaf(v[j][n][y], w, acc[n][y]);
      }
  }
  const int f = group * 32 + (lane & 31);
  const int token = span.t0 + f / G;
  if (token >= span.t1) return;
  const float inv = 1.f / fmaxf(l, FLT_MIN);
  float o[D / 8];
#pragma unroll
  for (int y = 0; y < 4; ++y)
#pragma unroll
    for (int n = 0; n < M::kRows; ++n) o[y * M::kRows + n] = acc[n][y] * inv;
  store_run<QT, D / 8>(static_cast<QT*>(a.out) + (int64_t)(u.q0 + token) * a.o_tok +
                           (int64_t)(kvh * G + f % G) * a.o_head + D / 4 * part +
                           D / 8 * (lane >> 5), o);
}

// Prefix tiles of a decode plan (decode_plan.cpp): the shared blocks of sequences whose
// block tables begin with the same blocks, every key visible to each, read once per
// tile of up to TQ member sequences (TQ * G columns: member j's head g is column
// j G + g) and key range, as the chunked-prefill kernel reads a chunk's keys against
// its query tokens, with no mask: each column's partial (m, l, acc) of the range goes to
// the member row's chunk slot, for the chunk-merge kernel (decode_planned.hip) to merge
// with the row's other ranges and its own blocks. Tiles reading the same blocks (one kv
// head and range) are consecutive and run on one XCD, whose L2 then serves their keys.
constexpr int kTileWords = 8, kMemberWords = 3;

template <typename QT, int D, int G>
__global__ __launch_bounds__(256, (prefill_occupancy<QT, D>())) void prefix_tiles_kernel(PlanArgs p) {
  static_assert(D == 64 || D == 128 || D == 256, "head_dim");
  constexpr int TQ = PrefillShape<D>::kCols / G;
  static_assert(PrefillShape<D>::kCols % G == 0, "GQA group must divide the column tile");
  const AttnArgs& a = p.a;

  // one struct, the operand buffers at its start: every LDS address of the key steps then
  // has a constant offset
  __shared__ struct {
    PrefillLds<D> unit;
    int row[TQ];   // member j's query token row
    int slot[TQ];  // its chunk slot for this tile's kv head and range
    int ctx[QOp<QT, D>::kAhead ? 1 : TQ];  // its length (fp32 queries leave no register for it)
    int bad;
  } lds;
  PrefillLds<D>& L = lds.unit;

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int hkv = a.cache.num_kv_heads;
  long long tm[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // trace marks (kTrace)
  if constexpr (kTrace) tm[0] = wall_clock64();
  const int64_t units = p.info.num_tiles;
  const int64_t per_xcd = (units + kXcds - 1) / kXcds;
  const int64_t slot = blockIdx.x / kXcds;
  const int64_t unit = (int64_t)(blockIdx.x % kXcds) * per_xcd + slot;
  if (slot >= per_xcd || unit >= units) return;

  // ---- the tile, every index checked (the plan is untrusted); its members are read and
  // checked in the unit's prologue, while the first block ids load
  const int32_t* rec = p.plan + p.info.off_tiles + unit * kTileWords;
  const int m0 = rec[0], n = rec[1], kvh = rec[2], range = rec[3];
  const int blk0 = rec[4], nblk = rec[5], ids_off = rec[6], lead = rec[7];
  if (!(m0 >= 0 && n >= 1 && n <= TQ && n <= p.info.num_tile_members - m0 && kvh >= 0 &&
        kvh < hkv && range >= 0 && range < p.info.tile_ranges && blk0 >= 0 && nblk >= 0 &&
        ids_off >= 0 && nblk <= p.info.num_ids - ids_off && lead >= 0 && lead < a.num_seqs)) {
    if (threadIdx.x == 0) atomicOr(a.err_flag, ASTR_FLAG_BAD_INDEX);
    return;  // the whole workgroup (every thread read the same record)
  }
  if (threadIdx.x == 0) lds.bad = 0;  // ordered before the prologue by the unit's barriers
  int mctx = 0;  // thread j < n: member j's context length, checked after the unit
  auto prologue = [&]() __attribute__((always_inline)) -> bool {
    if ((int)threadIdx.x < n) {
      const int32_t* mem = p.plan + p.info.off_tile_members + (int64_t)(m0 + threadIdx.x) * kMemberWords;
      const int seq = mem[0], c0 = mem[1], span = mem[2];
      if (!(seq >= 0 && seq < a.num_seqs && c0 >= 0 && span > range &&
            (int64_t)c0 + (int64_t)hkv * span <= p.info.num_chunks)) {
        lds.bad = 1;
      } else {
        lds.row[threadIdx.x] = seq;  // decode rows: sequence s's query token is row s
        lds.slot[threadIdx.x] = c0 + kvh * span + range;
        mctx = a.context_lens[seq];  // its wait falls after the key steps
        if constexpr (!QOp<QT, D>::kAhead) lds.ctx[threadIdx.x] = mctx;
      }
    }
    __syncthreads();
    if constexpr (kTrace) tm[1] = wall_clock64();
    return __builtin_amdgcn_readfirstlane(lds.bad) == 0;
  };

  // an invalid column reads member 0's query row (and is zeroed when quantized)
  auto column_of = [&](int f) __attribute__((always_inline)) -> ColumnInfo {
    const int j = f / G;
    return ColumnInfo{lds.row[j < n ? j : 0], kvh * G + f % G, 0, INT_MAX, j < n};
  };
  // every key of the range is visible to every column: no step is bounded
  auto bounds_of = [&](int wave) __attribute__((always_inline)) -> WaveBounds {
    return WaveBounds{0, 0, INT_MAX, INT_MAX, (wave * PrefillShape<D>::NT * 32) / G < n};
  };
  // the partial of column (member j, head g): m, l and acc into the member's chunk
  // slot, head g, with acc and l in the decode kernels' units (both times norm_scale,
  // as the decode partials they merge with). A lane holds 64-byte runs of its column: the
  // columns go through the wave's share of the operand buffers (free after the last key
  // step's barrier), 16 at a time, and each store instruction then writes 1 KB of whole
  // columns.
  constexpr int kRow = D + 4;  // floats per staged column (padded against bank conflicts)
  static_assert(kWaves * 16 * kRow * sizeof(float) <= sizeof(L.k) + sizeof(L.v) &&
                    offsetof(PrefillLds<D>, v) == sizeof(L.k),
                "a wave's half tile fits its share of the buffers");
  auto store = [&](int t, const float16v_t (&acc)[D / 32], float m, float l, int ve,
                   const ColumnInfo& c) __attribute__((always_inline)) {
    const int f0 = (wave * PrefillShape<D>::NT + t) * 32;  // the tile's first column
    float* const tile = reinterpret_cast<float*>(&L) + wave * 16 * kRow;
    const float up = ldexpf(norm_scale<KF>(), ve);  // the PV tiles carry 2^-ve
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      __builtin_amdgcn_wave_barrier();  // after the previous half's reads of this share
      if (((lane >> 4) & 1) == half) {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          float v[D / 8];
          acc_run<D>(acc, x, up, v);
#pragma unroll
          for (int k = 0; k < D / 32; ++k)
            *reinterpret_cast<float4_t*>(tile + (lane & 15) * kRow + D / 4 * x + D / 8 * (lane >> 5) +
                                         4 * k) =
                float4_t{v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]};
        }
      }
      __builtin_amdgcn_wave_barrier();  // a wave's LDS accesses complete in issue order
#pragma unroll
      for (int i = 0; i < D / 16; ++i) {
        const int e = i * kWave + lane;  // float4 e of the half tile: column e / (D/4)
        const int cc = e / (D / 4), q = e % (D / 4);
        const int f = f0 + 16 * half + cc;
        const float4_t v = *reinterpret_cast<const float4_t*>(tile + cc * kRow + 4 * q);
        if (f / G < n) {
          // non-temporal: the decode kernel reads the partials only after streaming the
          // rows' own blocks, long after they would have left the cache, and dirty lines
          // left in the cache are written back at this kernel's end (measured: config 4's
          // call 69.2 -> 68.6 us)
          const int64_t col = plan_chunk_slot(p, lds.slot[f / G], G) + f % G;
          __builtin_nontemporal_store(v, reinterpret_cast<float4_t*>(a.ws_o + col * D + 4 * q));
        }
      }
    }
    if (c.valid && lane < 32) {
      const int f = f0 + lane;
      const int64_t col = plan_chunk_slot(p, lds.slot[f / G], G) + f % G;
      a.ws_ml[col * 2] = m;
      a.ws_ml[col * 2 + 1] = l * norm_scale<KF>();
    }
  };
  const int32_t* ids = p.plan + p.info.off_ids + ids_off - blk0;  // id of block b at ids[b]
  auto mark = [&](int k) __attribute__((always_inline)) {
    if constexpr (kTrace) tm[k] = wall_clock64();
  };
  prefill_unit<QT, D, 1>(a, L, kvh, blk0, blk0 + nblk, ids, 0, 0, column_of, bounds_of, store,
                         prologue, mark);
  const int tid = wave * kWave + lane_id();
  if (lds.bad) {  // a member failed its checks: nothing was stored
    if (tid == 0) atomicOr(a.err_flag, ASTR_FLAG_BAD_INDEX);
    return;
  }
  // every key of the range must be visible to each member (its length as planned)
  if (tid < n) {
    if constexpr (!QOp<QT, D>::kAhead) mctx = lds.ctx[tid];
    const RowSpan sp = row_span(a, mctx);
    if (sp.kv_begin > blk0 * kBlockTokens || (int64_t)sp.ctx < (int64_t)(blk0 + nblk) * kBlockTokens)
      atomicOr(a.err_flag, ASTR_FLAG_BAD_INDEX);
  }
#if ASTR_TRACE
  const int64_t tw = unit * kWaves + wave;
  if (lane == 0 && tw < kTileTraceWaves) {
    for (int k = 0; k < 8; ++k) g_ttrace[tw][k] = tm[k];
    g_ttrace_info[tw][0] = (nblk + kWaves - 1) / kWaves;
    g_ttrace_info[tw][1] = (int)__builtin_amdgcn_s_getreg((20 << 0) | (0 << 6) | (3 << 11));  // XCC_ID
    g_ttrace_info[tw][2] = kvh;
    g_ttrace_info[tw][3] = range;
  }
#endif
}

// Compute units of the current device (256 where that cannot be read).
int prefill_cus() {
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) == hipSuccess &&
      hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
    return v;
  return 256;
}

// Key steps below which a unit is not split: a piece costs its start (~2 steps) and its
// partial, written and read again; at head dim 256, where a step takes twice as long, less.
template <int D>
constexpr int least_piece_steps() { return D == 256 ? 4 : 8; }

// Head dim 256, in thirds of a key step of KS = 2 (1.8 us): a step by KS, and what a split
// costs beside its steps (starts, partials and the merge launch, 10 us).
constexpr int kSplitTime = 17;
template <int KS>
constexpr int step_time() { return KS == 2 ? 3 : 4; }

// Units of a call: the sum over sequences of ceil(n / tq) for n >= pf_min_rows, at most (each
// adds at most tq - 1 to the token count, and there are at most tokens / pf_min_rows of them).
int64_t unit_bound(const ChunkArgs& a, int tq) {
  const int64_t seqs = std::min<int64_t>(a.num_seqs, a.num_q_tokens / a.pf_min_rows);
  return ((int64_t)a.num_q_tokens + seqs * (tq - 1)) / tq * a.cache.num_kv_heads;
}

// The call's units and their key split. Units that leave half the resident workgroups or more
// without work are cut into equal key ranges, as many as there are idle workgroups per unit
// and the workspace holds (512 tokens on 16000: 128 units of 258 steps on 512 workgroups,
// 477 -> 186 us in 4 pieces).
struct Split {
  int64_t units;
  int32_t pieces, steps;  // as pf_pieces, pf_steps
  int64_t time;           // of the longest unit (step_time, kSplitTime)
};
template <typename QT, int D, int G, int KS>
Split key_split(const ChunkArgs& a, int cus) {
  constexpr int TQ = PrefillShape<D, KS>::kCols / G;
  int64_t keys = a.max_context;
  if (a.window > 0) keys = std::min<int64_t>(keys, (int64_t)a.window + TQ + kBlockTokens);
  const int64_t steps = (keys + kWaves * kBlockTokens - 1) / (kWaves * kBlockTokens) + 1;
  const int64_t room = (int64_t)(a.pf_bytes / (PiecePartial<D, KS>::kFloats * sizeof(float)));
  const int64_t resident = (int64_t)cus * prefill_occupancy<QT, D>();
  Split s{unit_bound(a, TQ), 1, INT32_MAX / kWaves, steps * step_time<KS>()};
  if (s.units == 0) return s;
  const int64_t pieces = std::min<int64_t>(std::min(resident, room) / s.units, kMostPieces);
  if (pieces < 2 || steps < 2 * least_piece_steps<D>()) return s;
  const int64_t longest = std::max<int64_t>((steps + pieces - 1) / pieces, least_piece_steps<D>());
  const int64_t time = longest * step_time<KS>() + kSplitTime;
  if (D == 256 && time >= s.time) return s;
  return Split{s.units, (int32_t)((steps + longest - 1) / longest), (int32_t)longest, time};
}

template <typename QT, int D, int G, int KS>
int launch_shape(ChunkArgs a, const Split& split, int cus, hipStream_t stream) {
  a.pf_cus = cus >= kXcds ? cus / kXcds : 1;
  a.pf_pieces = split.pieces;
  a.pf_steps = split.steps;
  const int64_t grid = (split.units * a.pf_pieces + kXcds - 1) / kXcds * kXcds;
  if (grid > INT32_MAX) return fail(ASTR_EUNSUPPORTED, "prefill grid too large");
  hipLaunchKernelGGL((prefill_mfma_kernel<QT, D, G, KS>), dim3((uint32_t)grid),
                     dim3(kWaves * kWave), 0, stream, a);
  if (a.pf_pieces > 1)
    hipLaunchKernelGGL((prefill_merge_kernel<QT, D, G, KS>),
                       dim3((uint32_t)split.units * (MergeShape<D>::kParts / KS)),
                       dim3(kWaves * kWave), 0, stream, a);
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? 0 : hip_fail(err, "paged_attention (prefill) launch");
}

// At head dim 256, where one workgroup holds a CU, KS = 2 takes what fits the GPU and is done
// sooner: 500 tokens (16 query / 2 KV heads, bf16) 37.7 us with KS = 1, 31.6 with KS = 2, split
// 34.4; 16 tokens on 900, 3 sequences (32/8 heads) 54.0, 47.4 and, split, 36.0; 256 on 8000 (16/4
// heads) stay with KS = 1 and 8 pieces, 75.8 us. Past the GPU's CUs its units queue: 1500 tokens
// (16/4 heads) 86.5 us with KS = 1, 96.8 with KS = 2.
template <typename QT, int D, int G>
int launch(const ChunkArgs& a, hipStream_t stream) {
  const int cus = prefill_cus();
  const Split whole = key_split<QT, D, G, 1>(a, cus);
  if (whole.units == 0) return 0;
  if constexpr (D == 256) {
    const Split halves = key_split<QT, D, G, 2>(a, cus);
    if (halves.units <= cus && halves.time < whole.time)
      return launch_shape<QT, D, G, 2>(a, halves, cus, stream);
  }
  return launch_shape<QT, D, G, 1>(a, whole, cus, stream);
}

template <typename QT, int D>
int dispatch_group(const ChunkArgs& a, int G, hipStream_t s) {
  switch (G) {
    case 1: return launch<QT, D, 1>(a, s);
    case 2: return launch<QT, D, 2>(a, s);
    case 4: return launch<QT, D, 4>(a, s);
    case 8: return launch<QT, D, 8>(a, s);
    case 16: return launch<QT, D, 16>(a, s);
    default: return fail(ASTR_EUNSUPPORTED, "GQA group size %d not supported", G);
  }
}

template <typename QT>
int dispatch_dim(const ChunkArgs& a, int G, hipStream_t s) {
  switch (a.cache.head_dim) {
    case 64: return dispatch_group<QT, 64>(a, G, s);
    case 128: return dispatch_group<QT, 128>(a, G, s);
    case 256: return dispatch_group<QT, 256>(a, G, s);
    default: return fail(ASTR_EUNSUPPORTED, "head_dim %d not in {64,128,256}", a.cache.head_dim);
  }
}

template <typename QT, int D, int G>
int launch_tiles(const PlanArgs& p, hipStream_t stream) {
  const int64_t grid = ((int64_t)p.info.num_tiles + kXcds - 1) / kXcds * kXcds;
  if (grid == 0) return 0;
  if (grid > INT32_MAX) return fail(ASTR_EUNSUPPORTED, "prefix tile grid too large");
  hipLaunchKernelGGL((prefix_tiles_kernel<QT, D, G>), dim3((uint32_t)grid), dim3(kWaves * kWave),
                     0, stream, p);
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? 0 : hip_fail(err, "paged_attention (prefix tiles) launch");
}

template <typename QT, int D>
int tiles_group(const PlanArgs& p, int G, hipStream_t s) {
  switch (G) {
    case 1: return launch_tiles<QT, D, 1>(p, s);
    case 2: return launch_tiles<QT, D, 2>(p, s);
    case 4: return launch_tiles<QT, D, 4>(p, s);
    case 8: return launch_tiles<QT, D, 8>(p, s);
    case 16: return launch_tiles<QT, D, 16>(p, s);
    default: return fail(ASTR_EUNSUPPORTED, "GQA group size %d not supported", G);
  }
}

template <typename QT>
int tiles_dim(const PlanArgs& p, int G, hipStream_t s) {
  switch (p.a.cache.head_dim) {
    case 64: return tiles_group<QT, 64>(p, G, s);
    case 128: return tiles_group<QT, 128>(p, G, s);
    case 256: return tiles_group<QT, 256>(p, G, s);
    default: return fail(ASTR_EUNSUPPORTED, "head_dim %d not in {64,128,256}", p.a.cache.head_dim);
  }
}

}  // namespace

#if ASTR_TRACE && ASTR_KF == 0
// Trace builds: copies the marks and info of the first `waves` waves of the last
// prefix-tile launch of the int8 format (8 int64 + 4 int32 per wave; wave w of tile
// unit u at u * 4 + w) to host memory.
extern "C" int astr_trace_read_tiles(void* marks, void* info, int waves) {
  if (waves < 0 || waves > kTileTraceWaves) return ASTR_EINVAL;
  hipError_t e = hipMemcpyFromSymbol(marks, HIP_SYMBOL(g_ttrace), (size_t)waves * 64);
  if (e == hipSuccess) e = hipMemcpyFromSymbol(info, HIP_SYMBOL(g_ttrace_info), (size_t)waves * 16);
  return e == hipSuccess ? 0 : (int)e;
}
#endif

template <>
int launch_prefix_tiles_kf<KF>(const PlanArgs& p, int32_t q_dtype, hipStream_t stream) {
  const int G = p.a.num_q_heads / p.a.cache.num_kv_heads;
  switch (q_dtype) {
    case ASTR_F32: return tiles_dim<float>(p, G, stream);
    case ASTR_F16: return tiles_dim<_Float16>(p, G, stream);
    default: return tiles_dim<bf16_t>(p, G, stream);
  }
}

template <>
int launch_prefill_kf<KF>(const ChunkArgs& a, int32_t q_dtype, hipStream_t stream) {
  const int G = a.num_q_heads / a.cache.num_kv_heads;
  switch (q_dtype) {
    case ASTR_F32: return dispatch_dim<float>(a, G, stream);
    case ASTR_F16: return dispatch_dim<_Float16>(a, G, stream);
    default: return dispatch_dim<bf16_t>(a, G, stream);
  }
}

}  // namespace attn
}  // namespace astr
