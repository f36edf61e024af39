// Shared device helpers for the gfx950 INT8 paged-KV kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <cfloat>
#include <stdint.h>

#include "aster_kv.h"

namespace astr {

constexpr int kWave = 64;
constexpr float kLog2e = 1.4426950408889634f;

// Record a message for astr_last_error() and return `code`.
int fail(int code, const char* fmt, ...);
int hip_fail(hipError_t err, const char* what);

// A roctx range over one C-ABI call on the host (argument checks and launches), named
// after the entry point: `rocprofv3 --marker-trace` shows each call beside the
// kernels it enqueued. Without a profiler attached the push and pop are no-ops.
struct CallRange {
  explicit CallRange(const char* name);
  ~CallRange();
  CallRange(const CallRange&) = delete;
  CallRange& operator=(const CallRange&) = delete;
};

// ---- element conversion -----------------------------------------------------

struct bf16_t {
  uint16_t bits;
};

template <typename T>
__device__ __forceinline__ float to_float(T v);
template <>
__device__ __forceinline__ float to_float<float>(float v) { return v; }
template <>
__device__ __forceinline__ float to_float<_Float16>(_Float16 v) { return (float)v; }
template <>
__device__ __forceinline__ float to_float<bf16_t>(bf16_t v) {
  return __builtin_bit_cast(float, (uint32_t)v.bits << 16);
}

template <typename T>
__device__ __forceinline__ T from_float(float v);
template <>
__device__ __forceinline__ float from_float<float>(float v) { return v; }
template <>
__device__ __forceinline__ _Float16 from_float<_Float16>(float v) { return (_Float16)v; }
template <>
__device__ __forceinline__ bf16_t from_float<bf16_t>(float v) {
  // round-to-nearest-even fp32 -> bf16, NaN stays NaN (v_cvt_pk_bf16_f32)
  return bf16_t{__builtin_bit_cast(uint16_t, (__bf16)v)};
}

// Two values rounded to nearest even and packed in one word, a in the low half
// (one v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32).
typedef float f32x2_t __attribute__((ext_vector_type(2)));
template <typename T>
__device__ __forceinline__ uint32_t pack2(float a, float b);
template <>
__device__ __forceinline__ uint32_t pack2<bf16_t>(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t));
}
template <>
__device__ __forceinline__ uint32_t pack2<_Float16>(float a, float b) {
  typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, f16x2_t));
}

// ---- cross-lane reductions ----------------------------------------------------
// DPP control words (GCN/CDNA encoding).
constexpr int kDppXor1 = 0xB1;         // quad_perm [1,0,3,2]
constexpr int kDppXor2 = 0x4E;         // quad_perm [2,3,0,1]
constexpr int kDppHalfMirror = 0x141;  // lane i <-> 7-i inside each 8-lane half row
constexpr int kDppMirror = 0x140;      // lane i <-> 15-i inside each 16-lane row
constexpr int kDppRor8 = 0x128;        // lane i <- (i+8)%16 inside each row

template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}

// Sum over aligned groups of N consecutive lanes (N in 1,2,4,8,16); every lane
// of the group receives the group total.
template <int N>
__device__ __forceinline__ float group_sum(float x) {
  if constexpr (N >= 2) x += dpp<kDppXor1>(x);
  if constexpr (N >= 4) x += dpp<kDppXor2>(x);
  if constexpr (N >= 8) x += dpp<kDppHalfMirror>(x);
  if constexpr (N >= 16) x += dpp<kDppMirror>(x);
  return x;
}

__device__ __forceinline__ float shfl_xor(float x, int mask) { return __shfl_xor(x, mask, kWave); }

// Reduce over lanes whose index differs only in bits >= log2(STRIDE): every
// lane receives the total over its residue class (lane % STRIDE).
template <int STRIDE>
__device__ __forceinline__ float strided_sum(float x) {
  if constexpr (STRIDE <= 8) x += dpp<kDppRor8>(x);
  if constexpr (STRIDE <= 16) x += shfl_xor(x, 16);
  x += shfl_xor(x, 32);
  if constexpr (STRIDE <= 4) x += shfl_xor(x, 4);
  return x;
}

template <int STRIDE>
__device__ __forceinline__ float strided_max(float x) {
  if constexpr (STRIDE <= 8) x = fmaxf(x, dpp<kDppRor8>(x));
  if constexpr (STRIDE <= 16) x = fmaxf(x, shfl_xor(x, 16));
  x = fmaxf(x, shfl_xor(x, 32));
  if constexpr (STRIDE <= 4) x = fmaxf(x, shfl_xor(x, 4));
  return x;
}

// Maximum over aligned groups of N consecutive lanes (N in 8,16,32,64), in every lane.
template <int N>
__device__ __forceinline__ float group_max(float x) {
  x = fmaxf(x, dpp<kDppXor1>(x));
  x = fmaxf(x, dpp<kDppXor2>(x));
  x = fmaxf(x, dpp<kDppHalfMirror>(x));
  if constexpr (N >= 16) x = fmaxf(x, dpp<kDppMirror>(x));
  if constexpr (N >= 32) x = fmaxf(x, shfl_xor(x, 16));
  if constexpr (N >= 64) x = fmaxf(x, shfl_xor(x, 32));
  return x;
}
__device__ __forceinline__ float wave_max(float x) { return group_max<kWave>(x); }

// Sum over the 64 lanes (every lane gets it): after the xor-1/xor-2 butterflies a
// lane holds its quad's sum, and each mirror step adds the mirrored (disjoint)
// group of the same size.
__device__ __forceinline__ float wave_sum(float x) {
  x += dpp<kDppXor1>(x);
  x += dpp<kDppXor2>(x);
  x += dpp<kDppHalfMirror>(x);
  x += dpp<kDppMirror>(x);
  x += shfl_xor(x, 16);
  x += shfl_xor(x, 32);
  return x;
}

// Code formats (astr_kv_format) as template arguments.
constexpr int kInt8 = ASTR_KV_INT8;
constexpr int kE4M3 = ASTR_KV_FP8_E4M3FN;
constexpr int kE5M2 = ASTR_KV_FP8_E5M2;

// Largest code magnitude of a format (KVQuantization.maximum, kv_quantization.py:23-25).
template <int KF>
__device__ __forceinline__ constexpr float format_max() {
  return KF == kInt8 ? 127.f : KF == kE4M3 ? 448.f : 57344.f;
}

// Finite c with |c| <= format_max -> FP8 bits, round to nearest even with subnormals and
// the sign of zero kept: the OCP conversions of gfx950, equal to the float32 -> float8
// conversion for every such float.
template <int KF>
__device__ __forceinline__ uint32_t fp8_pair(float lo, float hi) {
  if constexpr (KF == kE4M3) return __builtin_amdgcn_cvt_pk_fp8_f32(lo, hi, 0, false);
  else return __builtin_amdgcn_cvt_pk_bf8_f32(lo, hi, 0, false);
}

// The row's scale from its largest magnitude (kv_quantization.py:86-90): true
// division, then the FLT_MIN clamp; an all-zero row gets scale 1.
template <int KF>
__device__ __forceinline__ float quant_scale(float amax) {
  return amax == 0.f ? 1.f : fmaxf(amax / format_max<KF>(), FLT_MIN);
}

// One code (kv_quantization.py:91-94): divide by the scale, clamp to the format's
// range, round half to even (int8) or to the nearest-even FP8 value; as a byte.
template <int KF>
__device__ __forceinline__ int8_t quant_code(float x, float scale) {
  constexpr float kMax = format_max<KF>();
  const float n = fminf(fmaxf(x / scale, -kMax), kMax);
  if constexpr (KF == kInt8) return (int8_t)__builtin_rintf(n);
  else return (int8_t)fp8_pair<KF>(n, 0.f);
}

// x / scale clamped to the format's range, with the code of the correctly rounded quotient,
// from inv = 1 / scale (correctly rounded): the product's residual, in one fma, corrects it
// (Markstein's division step). The product is within 1.5 steps of the quotient, its residual
// and inv within 2^-24 of themselves, so that the corrected one is rounded from within 3 2^-24
// of a step: it can differ from the division only where the quotient lies that near a rounding
// boundary, and its code only where this boundary is beside a tie of two codes. All float32
// pairs there (up to scaling by powers of two) give the division's result, and so does every
// pair of f16 significands (the tests list them). scale >= kMinFastScale keeps the residual of
// every quotient that can round to a code above the denormals.
constexpr float kMinFastScale = 0x1p-64f;
template <int KF>
__device__ __forceinline__ float quant_unit(float x, float scale, float inv) {
  constexpr float kMax = format_max<KF>();
  const float q = x * inv;
  float n = __builtin_fmaf(__builtin_fmaf(-q, scale, x), inv, q);
  if constexpr (KF != kInt8) n = __builtin_copysignf(n, x);  // x = -0 gives +0 above
  return fminf(fmaxf(n, -kMax), kMax);
}

// Four quotients of quant_unit as a word of codes. int8: adding 1.5 2^23 rounds half to
// even and leaves the integer in the low byte.
template <int KF>
__device__ __forceinline__ uint32_t quant_pack(const float (&n)[4]) {
  if constexpr (KF == kInt8) {
    uint32_t b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = __builtin_bit_cast(uint32_t, n[i] + 12582912.f);
    return __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u) |
           __builtin_amdgcn_perm(b[3], b[2], 0x04000c0cu);
  } else {
    return (fp8_pair<KF>(n[0], n[1]) & 0xffffu) | fp8_pair<KF>(n[2], n[3]) << 16;
  }
}

// The f16 conversions below give a code's value times 2^-8 for E4M3FN (its bits
// land one exponent step of 8 apart from f16's) and the value itself otherwise;
// code_scale undoes that (exactly: a power of two) where the scales are applied.
template <int KF>
__device__ __forceinline__ constexpr float code_scale() {
  return KF == kE4M3 ? 256.f : 1.f;
}

// PV weights and V operands are rounded to f16 after the V scale is applied, so the
// scale enters times v_weight_scale: for E4M3FN that undoes its codes' 2^-8; E5M2's
// scales (amax / 57344) lie below f16's normal range for |V| up to ~3.5, and 2^8
// lifts them into it. Where the E5M2 codes enter at their own value (the decode
// kernels) the softmax normaliser carries the same 2^8 (norm_scale), which cancels
// in acc / l; the prefill kernel takes E5M2 codes times 2^-8 instead (exact in f16).
template <int KF>
__device__ __forceinline__ constexpr float v_weight_scale() {
  return KF == kInt8 ? 1.f : 256.f;
}
template <int KF>
__device__ __forceinline__ constexpr float norm_scale() {
  return KF == kE5M2 ? 256.f : 1.f;
}

// FP8 codes placed in the high byte of each f16 half (low bytes zero) -> the f16
// pair: E5M2 is the top byte of the f16 with the same value; E4M3FN keeps its
// sign and shifts |code| right by one bit into f16's exponent/mantissa fields,
// which is its value times 2^-8 (subnormals included).
template <int KF>
__device__ __forceinline__ uint32_t fp8_hi_bytes_to_f16(uint32_t h) {
  if constexpr (KF == kE5M2) return h;
  else return ((h >> 1) & 0x3f803f80u) | (h & 0x80008000u);
}

// Code byte `b` of a packed dword, as float (exact; times 2^-8 for E4M3FN).
template <int KF>
__device__ __forceinline__ float code_to_f(uint32_t w, int b) {
  if constexpr (KF == kInt8) {
    return (float)(int8_t)(w >> (8 * b));
  } else {
    const uint32_t h = fp8_hi_bytes_to_f16<KF>(((w >> (8 * b)) & 0xffu) << 8);
    return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
  }
}

// int8 byte `b` of a packed dword, as float (exact).
__device__ __forceinline__ float i8_to_f(uint32_t w, int b) { return code_to_f<kInt8>(w, b); }

}  // namespace astr
