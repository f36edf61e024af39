// Fused quantize-and-append of new K/V token rows into the paged arena (INT8, FP8
// E4M3FN or FP8 E5M2 codes).
//
// Arithmetic follows quantize_kv (src/aster/optimization/kv_quantization.py:82-94)
// bit for bit: fp32 source, amax over the row, scale = amax==0 ? 1 :
// max(amax/M, FLT_MIN) with an IEEE-correct division (M = 127, 448 or 57344),
// c = clamp(x/scale, -M, M) again with IEEE division (never x*(1/scale)); int8
// codes are rint(c) (half to even, v_rndne), FP8 codes c rounded to nearest even
// in the format (the float32 -> float8 conversion of .to(dtype), :94). The library
// is built with -fhip-fp32-correctly-rounded-divide-sqrt and without denormal
// flushing.
//
// Two launches per call: a finiteness scan that sets ASTR_FLAG_NONFINITE_INPUT,
// then the quantize/scatter kernel that does nothing when that bit is set, so a
// bad suffix mutates no slot (kv_quantization.py:77-81, state.py:292 runs the
// check before any copy). For slots the caller has reserved and rolls back when
// the flag is raised (the runner's step), one launch: the quantize/scatter kernel
// checks its own row and leaves a non-finite row unwritten.
//
// Head dims 64, 128, 256 and 512 run the wide kernels, bound by memory for prompts and
// by latency for a decode step's few rows. D / 8 lanes hold one row (8 elements each: a
// 16-byte load of 16-bit input, an 8-byte store of codes), and a workgroup takes 2048 / D
// consecutive tokens of one head, K and V together, so that all of its loads are in
// flight at once and a block's codes and scales are written by one workgroup where its
// tokens are consecutive. The division is one reciprocal per row and two fused steps per
// element (quant_unit), FP8 codes come from the conversion instructions. 4096 tokens x 8
// heads x 128 in bf16: 22.9 -> 9.1 us (25.5 MB), the scan 9.2 -> 4.4 us, against one wave per
// row, 4 bytes a lane and a full IEEE division sequence per element. Any other head dim
// takes the generic kernels, one wave per row.
#include <cfloat>
#include <type_traits>

#include "common.h"

namespace astr {
namespace {

constexpr int kRowsPerBlock = 4;  // one wave per (token, head, K|V) row

constexpr int kMaxPerLane = 8;    // head_dim <= 512

struct AppendArgs {
  const void* key;
  const void* value;
  int64_t key_token_stride, key_head_stride, value_token_stride, value_head_stride;
  int64_t num_tokens;
  const int64_t* slot_mapping;
  astr_paged_kv cache;
  int32_t* err_flag;
  int32_t block_shift;  // log2 of the block size, -1 when it is no power of two
  bool wide;            // rows and codes aligned for the wide kernels' vector accesses
};

// Row (token t, head h, K or V) handled by this wave; false past the last row.
struct RowRef {
  int t, h;
  bool is_v;
};

__device__ __forceinline__ bool row_of(const AppendArgs& a, RowRef& rr) {
  const int heads = a.cache.num_kv_heads;
  const int rows = (int)a.num_tokens * heads;  // host checks rows * 2 < 2^31
  const int row = blockIdx.x * kRowsPerBlock + (int)(threadIdx.x >> 6);
  if (row >= (a.value ? 2 : 1) * rows) return false;
  rr.is_v = row >= rows;
  const int r = rr.is_v ? row - rows : row;
  rr.t = r / heads;
  rr.h = r - rr.t * heads;
  return true;
}

template <typename T>
__device__ __forceinline__ const T* row_src(const AppendArgs& a, const RowRef& rr) {
  return static_cast<const T*>(rr.is_v ? a.value : a.key) +
         rr.t * (rr.is_v ? a.value_token_stride : a.key_token_stride) +
         rr.h * (rr.is_v ? a.value_head_stride : a.key_head_stride);
}

// The row's elements lane, lane + 64, ...: loads clamped in bounds, so that they all
// issue before the first use.
template <typename T>
__device__ __forceinline__ void load_row(const T* src, int D, int lane, float (&x)[kMaxPerLane]) {
#pragma unroll
  for (int i = 0; i < kMaxPerLane; ++i) {
    const int d = lane + i * kWave;
    const float v = to_float<T>(src[d < D ? d : D - 1]);
    x[i] = d < D ? v : 0.f;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void finite_scan_kernel(AppendArgs a) {
  RowRef rr;
  if (!row_of(a, rr)) return;
  const int lane = threadIdx.x & 63;
  float x[kMaxPerLane];
  load_row<T>(row_src<T>(a, rr), a.cache.head_dim, lane, x);
  bool bad = false;
#pragma unroll
  for (int i = 0; i < kMaxPerLane; ++i) bad |= !__builtin_isfinite(x[i]);
  if (__ballot(bad) != 0 && lane == 0) atomicOr(a.err_flag, ASTR_FLAG_NONFINITE_INPUT);
}

// The block and offset of a slot; false (flagged) past the arena.
__device__ __forceinline__ bool slot_of(const AppendArgs& a, int64_t slot, bool report,
                                        int64_t& block, int64_t& offset) {
  block = a.block_shift >= 0 ? slot >> a.block_shift : slot / a.cache.block_size;
  offset = slot - block * a.cache.block_size;
  if (block < a.cache.num_blocks) return true;
  if (report) atomicOr(a.err_flag, ASTR_FLAG_BAD_INDEX);
  return false;
}

template <typename T, int KF, bool kOwnCheck>
__global__ __launch_bounds__(256) void quantize_append_kernel(AppendArgs a) {
  // All-or-nothing: the finite scan of this call (or an unacknowledged earlier
  // one) flagged the input, so leave every slot untouched. The flag, slot and
  // row loads are independent and issue together. kOwnCheck (reserved slots, no
  // scan launch): the row's own check keeps a non-finite row out of its slot.
  RowRef rr;
  if (!row_of(a, rr)) return;
  const int lane = threadIdx.x & 63;
  const int flag = __atomic_load_n(a.err_flag, __ATOMIC_RELAXED);
  const int64_t slot = a.slot_mapping[rr.t];
  const int D = a.cache.head_dim;
  float x[kMaxPerLane];
  load_row<T>(row_src<T>(a, rr), D, lane, x);
  if constexpr (kOwnCheck) {
    bool bad = false;
#pragma unroll
    for (int i = 0; i < kMaxPerLane; ++i) bad |= !__builtin_isfinite(x[i]);
    if (__ballot(bad) != 0) {
      if (lane == 0) atomicOr(a.err_flag, ASTR_FLAG_NONFINITE_INPUT);
      return;
    }
  }
  if (flag & ASTR_FLAG_NONFINITE_INPUT) return;
  if (slot < 0) return;  // padding token: no slot
  int64_t block, offset;
  if (!slot_of(a, slot, lane == 0, block, offset)) return;
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < kMaxPerLane; ++i) amax = fmaxf(amax, fabsf(x[i]));
  amax = wave_max(amax);
  const float scale = quant_scale<KF>(amax);
  int8_t* codes = (rr.is_v ? a.cache.v_codes : a.cache.k_codes) +
                  block * a.cache.code_block_stride + rr.h * a.cache.code_head_stride + offset * D;
#pragma unroll
  for (int i = 0; i < kMaxPerLane; ++i) {
    const int d = lane + i * kWave;
    if (d < D) codes[d] = quant_code<KF>(x[i], scale);
  }
  if (lane == 0) {
    float* scales = (rr.is_v ? a.cache.v_scales : a.cache.k_scales) +
                    block * a.cache.scale_block_stride + rr.h * a.cache.scale_head_stride + offset;
    *scales = scale;
  }
}

// ---- wide kernels -------------------------------------------------------------------

constexpr int kVec = 8;  // elements of a row per lane
constexpr int kWideThreads = 256;

template <int D>
struct WideShape {
  static constexpr int kLanes = D / kVec;                    // lanes per row
  static constexpr int kTokens = kWideThreads / kLanes;      // tokens per workgroup
  static_assert(kLanes >= 8 && kLanes <= kWave && (kLanes & (kLanes - 1)) == 0, "rows fit a wave");
};

// The lane's 8 elements: 16-byte loads where every row is 16-byte aligned (a.wide).
template <typename T>
struct RowVec {
  uint4 w[kVec * sizeof(T) / 16];
};
template <typename T>
__device__ __forceinline__ void load_vec(const AppendArgs& a, const T* src, RowVec<T>& v) {
  constexpr int kWords = kVec * (int)sizeof(T) / 16;
  if (a.wide) {
#pragma unroll
    for (int i = 0; i < kWords; ++i) v.w[i] = reinterpret_cast<const uint4*>(src)[i];
  } else {
    T* e = reinterpret_cast<T*>(v.w);
#pragma unroll
    for (int i = 0; i < kVec; ++i) e[i] = src[i];
  }
}

// Whether any of the lane's elements is inf or NaN: an exponent field of all ones carries
// into the bit above it, two 16-bit elements per word.
template <typename T>
__device__ __forceinline__ bool any_nonfinite(const RowVec<T>& v) {
  constexpr uint32_t kExp = sizeof(T) == 4 ? 0x7f800000u
                            : __is_same(T, bf16_t) ? 0x7f807f80u : 0x7c007c00u;
  constexpr uint32_t kLow = sizeof(T) == 4 ? 0x00800000u
                            : __is_same(T, bf16_t) ? 0x00800080u : 0x04000400u;
  uint32_t carry = 0;
  const uint32_t* w = reinterpret_cast<const uint32_t*>(v.w);
#pragma unroll
  for (int i = 0; i < (int)sizeof(v.w) / 4; ++i) carry |= (w[i] & kExp) + kLow;
  return (carry & (sizeof(T) == 4 ? 0x80000000u : 0x80008000u)) != 0;
}

// This thread's token and its rows: workgroup (tile, head), head fastest.
template <int D>
struct WideRow {
  int64_t t;
  int h, e0;  // head, the lane's first element
  bool live;
  __device__ explicit WideRow(const AppendArgs& a) {
    const int heads = a.cache.num_kv_heads;
    h = blockIdx.x % heads;
    t = (int64_t)(blockIdx.x / heads) * WideShape<D>::kTokens + threadIdx.x / WideShape<D>::kLanes;
    e0 = threadIdx.x % WideShape<D>::kLanes * kVec;
    live = t < a.num_tokens;
    if (!live) t = a.num_tokens - 1;  // loads stay in range, nothing is stored
  }
};

template <typename T, int D>
__device__ __forceinline__ void load_rows(const AppendArgs& a, const WideRow<D>& r,
                                          RowVec<T>& k, RowVec<T>& v) {
  load_vec<T>(a, static_cast<const T*>(a.key) + r.t * a.key_token_stride +
                     r.h * a.key_head_stride + r.e0, k);
  if (a.value != nullptr)
    load_vec<T>(a, static_cast<const T*>(a.value) + r.t * a.value_token_stride +
                       r.h * a.value_head_stride + r.e0, v);
}

template <typename T, int D>
__global__ __launch_bounds__(kWideThreads) void finite_scan_wide_kernel(AppendArgs a) {
  const WideRow<D> r(a);
  RowVec<T> k{}, v{};
  load_rows<T, D>(a, r, k, v);
  if (__ballot(any_nonfinite<T>(k) || any_nonfinite<T>(v)) != 0 && threadIdx.x % kWave == 0)
    atomicOr(a.err_flag, ASTR_FLAG_NONFINITE_INPUT);
}

// One row (this lane's 8 elements of it) quantized and stored.
template <typename T, int D, int KF>
__device__ __forceinline__ void quantize_row(const AppendArgs& a, const RowVec<T>& raw,
                                             const WideRow<D>& r, bool store, int64_t block,
                                             int64_t offset, int8_t* codes_base,
                                             float* scales_base) {
  const T* e = reinterpret_cast<const T*>(raw.w);
  float x[kVec];
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < kVec; ++i) {
    x[i] = to_float<T>(e[i]);
    amax = fmaxf(amax, fabsf(x[i]));
  }
  const float scale = quant_scale<KF>(group_max<WideShape<D>::kLanes>(amax));
  uint32_t w[2];
  if (__builtin_expect(__ballot(scale < kMinFastScale) != 0, 0)) {
    uint8_t c[kVec];
#pragma unroll
    for (int i = 0; i < kVec; ++i) c[i] = (uint8_t)quant_code<KF>(x[i], scale);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      w[i] = c[4 * i] | c[4 * i + 1] << 8 | c[4 * i + 2] << 16 | (uint32_t)c[4 * i + 3] << 24;
  } else {
    const float inv = 1.f / scale;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float n[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) n[j] = quant_unit<KF>(x[4 * i + j], scale, inv);
      w[i] = quant_pack<KF>(n);
    }
  }
  if (!store) return;
  int8_t* dst = codes_base + block * a.cache.code_block_stride + r.h * a.cache.code_head_stride +
                offset * D + r.e0;
  if (a.wide) {
    *reinterpret_cast<uint2*>(dst) = uint2{w[0], w[1]};
  } else {
#pragma unroll
    for (int i = 0; i < kVec; ++i) dst[i] = (int8_t)(w[i / 4] >> (8 * (i % 4)));
  }
  if (r.e0 == 0)
    scales_base[block * a.cache.scale_block_stride + r.h * a.cache.scale_head_stride + offset] = scale;
}

template <typename T, int D, int KF, bool kOwnCheck>
__global__ __launch_bounds__(kWideThreads) void quantize_append_wide_kernel(AppendArgs a) {
  constexpr int kLanes = WideShape<D>::kLanes;
  const WideRow<D> r(a);
  const int flag = __atomic_load_n(a.err_flag, __ATOMIC_RELAXED);
  const int64_t slot = a.slot_mapping[r.t];
  RowVec<T> k{}, v{};
  load_rows<T, D>(a, r, k, v);
  bool keep_k = true, keep_v = a.value != nullptr;
  if constexpr (kOwnCheck) {  // rows of reserved slots check themselves, each on its own
    const int lane = threadIdx.x % kWave;
    const uint64_t row = (kLanes == kWave ? ~0ull : (1ull << kLanes) - 1) << (lane / kLanes * kLanes);
    const uint64_t bad_k = __ballot(any_nonfinite<T>(k)), bad_v = __ballot(any_nonfinite<T>(v));
    if ((bad_k | bad_v) != 0 && lane == 0) atomicOr(a.err_flag, ASTR_FLAG_NONFINITE_INPUT);
    keep_k = (bad_k & row) == 0;
    keep_v = keep_v && (bad_v & row) == 0;
  }
  if (flag & ASTR_FLAG_NONFINITE_INPUT) return;
  int64_t block = 0, offset = 0;
  const bool store = r.live && slot >= 0 && slot_of(a, slot, r.e0 == 0, block, offset);
  quantize_row<T, D, KF>(a, k, r, store && keep_k, block, offset, a.cache.k_codes, a.cache.k_scales);
  if (a.value != nullptr)
    quantize_row<T, D, KF>(a, v, r, store && keep_v, block, offset, a.cache.v_codes,
                           a.cache.v_scales);
}

template <typename T, int D, bool kOwnCheck>
void launch_quantize(const AppendArgs& a, uint32_t blocks, hipStream_t stream) {
  auto go = [&](auto format) {
    constexpr int KF = decltype(format)::value;
    if constexpr (D > 0)
      hipLaunchKernelGGL((quantize_append_wide_kernel<T, D, KF, kOwnCheck>), dim3(blocks),
                         dim3(kWideThreads), 0, stream, a);
    else
      hipLaunchKernelGGL((quantize_append_kernel<T, KF, kOwnCheck>), dim3(blocks), dim3(256), 0,
                         stream, a);
  };
  switch (a.cache.code_format) {
    case kInt8: go(std::integral_constant<int, kInt8>{}); break;
    case kE4M3: go(std::integral_constant<int, kE4M3>{}); break;
    default: go(std::integral_constant<int, kE5M2>{}); break;
  }
}

// D: the head dim of the wide kernels, 0 for the generic ones. reserved: the caller rolls
// the slots back on a flagged call, so no scan launch
template <typename T, int D>
int launch_append(const AppendArgs& a, bool reserved, hipStream_t stream) {
  uint32_t blocks;
  if constexpr (D > 0) {
    constexpr int kTokens = WideShape<D>::kTokens;
    blocks = (uint32_t)((a.num_tokens + kTokens - 1) / kTokens * a.cache.num_kv_heads);
  } else {
    const int64_t rows = (a.value ? 2 : 1) * a.num_tokens * a.cache.num_kv_heads;
    blocks = (uint32_t)((rows + kRowsPerBlock - 1) / kRowsPerBlock);
  }
  if (reserved) {
    launch_quantize<T, D, true>(a, blocks, stream);
  } else {
    if constexpr (D > 0)
      hipLaunchKernelGGL((finite_scan_wide_kernel<T, D>), dim3(blocks), dim3(kWideThreads), 0,
                         stream, a);
    else
      hipLaunchKernelGGL((finite_scan_kernel<T>), dim3(blocks), dim3(256), 0, stream, a);
    launch_quantize<T, D, false>(a, blocks, stream);
  }
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? 0 : hip_fail(err, "quantize_append launch");
}

template <typename T>
int launch_append_dim(AppendArgs a, bool reserved, hipStream_t stream) {
  // 16-byte loads and 8-byte stores where every row starts on them, else by elements
  auto rows16 = [&](const void* p, int64_t tok, int64_t head) {
    return p == nullptr || (reinterpret_cast<uintptr_t>(p) % 16 == 0 &&
                            tok * sizeof(T) % 16 == 0 && head * sizeof(T) % 16 == 0);
  };
  a.wide = rows16(a.key, a.key_token_stride, a.key_head_stride) &&
           rows16(a.value, a.value_token_stride, a.value_head_stride) &&
           a.cache.code_block_stride % 8 == 0 && a.cache.code_head_stride % 8 == 0 &&
           reinterpret_cast<uintptr_t>(a.cache.k_codes) % 8 == 0 &&
           (a.value == nullptr || reinterpret_cast<uintptr_t>(a.cache.v_codes) % 8 == 0);
  switch (a.cache.head_dim) {
    case 64: return launch_append<T, 64>(a, reserved, stream);
    case 128: return launch_append<T, 128>(a, reserved, stream);
    case 256: return launch_append<T, 256>(a, reserved, stream);
    case 512: return launch_append<T, 512>(a, reserved, stream);
    default: return launch_append<T, 0>(a, reserved, stream);
  }
}

// One thread per token: the slot's key-padding byte (state.py:339-344 copies the
// padding leaf into the page like every other leaf).
__global__ __launch_bounds__(256) void write_key_valid_kernel(uint8_t* key_valid, int64_t slots,
                                                              const int64_t* slot_mapping,
                                                              const uint8_t* token_valid,
                                                              int64_t num_tokens, int32_t* err_flag) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= num_tokens) return;
  const int64_t slot = slot_mapping[i];
  if (slot < 0) return;
  if (slot >= slots) {
    atomicOr(err_flag, ASTR_FLAG_BAD_INDEX);
    return;
  }
  key_valid[slot] = token_valid == nullptr || token_valid[i] != 0 ? 1 : 0;
}

}  // namespace
}  // namespace astr

extern "C" int astr_kv_write_key_valid(const astr_paged_kv* cache, const int64_t* slot_mapping,
                                       const uint8_t* token_valid, int64_t num_tokens,
                                       int32_t* err_flag, void* stream) {
  astr::CallRange range("astr_kv_write_key_valid");
  using namespace astr;
  if (cache == nullptr || err_flag == nullptr)
    return fail(ASTR_EINVAL, "cache descriptor and err_flag are required");
  if (cache->key_valid == nullptr) return fail(ASTR_EINVAL, "cache key_valid pointer is required");
  if (num_tokens < 0) return fail(ASTR_EINVAL, "num_tokens must be >= 0");
  if (num_tokens == 0) return 0;
  if (slot_mapping == nullptr) return fail(ASTR_EINVAL, "slot_mapping is required");
  if (cache->num_blocks < 1 || cache->block_size < 1)
    return fail(ASTR_EINVAL, "cache sizes must be positive");
  const int64_t blocks = (num_tokens + 255) / 256;
  if (blocks > INT32_MAX) return fail(ASTR_EINVAL, "too many tokens for one launch");
  hipLaunchKernelGGL(write_key_valid_kernel, dim3((uint32_t)blocks), dim3(256), 0,
                     static_cast<hipStream_t>(stream), cache->key_valid,
                     (int64_t)cache->num_blocks * cache->block_size, slot_mapping, token_valid,
                     num_tokens, err_flag);
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? 0 : hip_fail(err, "write_key_valid launch");
}

namespace {

int quantize_append(const astr_paged_kv* cache, const void* key, const void* value,
                    int32_t in_dtype, int64_t num_tokens, int64_t key_token_stride,
                    int64_t key_head_stride, int64_t value_token_stride,
                    int64_t value_head_stride, const int64_t* slot_mapping, int32_t* err_flag,
                    void* stream, bool reserved) {
  using namespace astr;
  if (cache == nullptr || err_flag == nullptr)
    return fail(ASTR_EINVAL, "cache descriptor and err_flag are required");
  if (num_tokens < 0) return fail(ASTR_EINVAL, "num_tokens must be >= 0");
  if (num_tokens == 0) return 0;
  if (key == nullptr || slot_mapping == nullptr)
    return fail(ASTR_EINVAL, "key and slot_mapping are required");
  if (cache->k_codes == nullptr || cache->k_scales == nullptr ||
      (value != nullptr && (cache->v_codes == nullptr || cache->v_scales == nullptr)))
    return fail(ASTR_EINVAL, "cache code/scale pointers are required");
  if (cache->head_dim < 1 || cache->head_dim > kWave * kMaxPerLane)
    return fail(ASTR_EUNSUPPORTED, "head_dim %d outside 1..%d", cache->head_dim,
                kWave * kMaxPerLane);
  if (cache->num_kv_heads < 1 || cache->block_size < 1 || cache->num_blocks < 1)
    return fail(ASTR_EINVAL, "cache sizes must be positive");
  if (cache->code_format != ASTR_KV_INT8 && cache->code_format != ASTR_KV_FP8_E4M3FN &&
      cache->code_format != ASTR_KV_FP8_E5M2)
    return fail(ASTR_EUNSUPPORTED, "code format %d is not int8 / fp8 e4m3fn / fp8 e5m2",
                cache->code_format);
  if ((value ? 2 : 1) * num_tokens * (int64_t)cache->num_kv_heads >= INT32_MAX)
    return fail(ASTR_EINVAL, "too many rows for one append launch");
  AppendArgs a{key, value, key_token_stride, key_head_stride, value_token_stride,
               value_head_stride, num_tokens, slot_mapping, *cache, err_flag,
               (cache->block_size & (cache->block_size - 1)) == 0
                   ? __builtin_ctz(cache->block_size) : -1,
               false};
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (in_dtype) {
    case ASTR_F32: return launch_append_dim<float>(a, reserved, s);
    case ASTR_F16: return launch_append_dim<_Float16>(a, reserved, s);
    case ASTR_BF16: return launch_append_dim<bf16_t>(a, reserved, s);
    default: return fail(ASTR_EUNSUPPORTED, "input dtype %d is not f32/f16/bf16", in_dtype);
  }
}

}  // namespace

extern "C" int astr_kv_quantize_append_i8(const astr_paged_kv* cache, const void* key,
                                          const void* value, int32_t in_dtype, int64_t num_tokens,
                                          int64_t key_token_stride, int64_t key_head_stride,
                                          int64_t value_token_stride, int64_t value_head_stride,
                                          const int64_t* slot_mapping, int32_t* err_flag,
                                          void* stream) {
  astr::CallRange range("astr_kv_quantize_append_i8");
  return quantize_append(cache, key, value, in_dtype, num_tokens, key_token_stride,
                         key_head_stride, value_token_stride, value_head_stride, slot_mapping,
                         err_flag, stream, false);
}

extern "C" int astr_kv_quantize_append_i8_reserved(
    const astr_paged_kv* cache, const void* key, const void* value, int32_t in_dtype,
    int64_t num_tokens, int64_t key_token_stride, int64_t key_head_stride,
    int64_t value_token_stride, int64_t value_head_stride, const int64_t* slot_mapping,
    int32_t* err_flag, void* stream) {
  astr::CallRange range("astr_kv_quantize_append_i8_reserved");
  return quantize_append(cache, key, value, in_dtype, num_tokens, key_token_stride,
                         key_head_stride, value_token_stride, value_head_stride, slot_mapping,
                         err_flag, stream, true);
}
