// The per-(token, kv head) scaled quantiser, shared by the store kernels and
// the decode kernel that stores its step's rows itself.
#pragma once

#include <type_traits>

#include "common.h"

namespace prism {

constexpr float kFp8Max = 448.0f;
constexpr float kScaleFloor = 1.0e-6f;  // the Python float 1e-6 rounded to fp32

template <int IN_DTYPE>
struct InVec8;  // 8 input elements -> 8 floats

template <>
struct InVec8<PRISM_DTYPE_BF16> {
  __device__ static void load(const void* p, float (&x)[8]) {
    u32x4 w = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = __uint_as_float(w[i] << 16);
      x[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
    }
  }
};

template <>
struct InVec8<PRISM_DTYPE_F16> {
  __device__ static void load(const void* p, float (&x)[8]) {
    u32x4 w = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = f16_bits_to_f32(w[i] & 0xFFFFu);
      x[2 * i + 1] = f16_bits_to_f32(w[i] >> 16);
    }
  }
};

template <>
struct InVec8<PRISM_DTYPE_F32> {
  __device__ static void load(const void* p, float (&x)[8]) {
    const floatx4* f = reinterpret_cast<const floatx4*>(p);
    floatx4 a = f[0], b = f[1];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i] = a[i];
      x[4 + i] = b[i];
    }
  }
};

// Four finite values of magnitude at most 448 (1 + 2^-22) -> E4M3FN bytes
// (the native RNE conversion, which saturates: values above 448 and below
// 464 give 448 either way; fp8_encode4's NaN and overflow handling cannot
// apply).
__device__ __forceinline__ uint32_t fp8_cvt4_in_range(float a, float b, float c, float d) {
  const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(c, d, lo, true));
}

// Eight elements of one (token, head) row -> E4M3FN bytes of
// clamp(x / s, -448, 448), where x / s is the correctly rounded fp32
// quotient, as IEEE division gives it.
//
// One division per row gives y = RN(1 / s).  Per element, q0 = RN(x * y) is
// within one ulp of x / s, so the residual e' = q0 * s - x is exact in fp32
// and one fused step q = RN(q0 - e' * y) is the correctly rounded quotient
// (Markstein's theorem on division by a correctly rounded reciprocal).  The
// quotients here are at most 448 (1 + 2^-22) in magnitude and s >= 1e-6, so
// nothing overflows; a quotient below 2^-126 may lose the theorem's
// guarantee but keeps its sign and is far below 2^-10, so its fp8 byte (a
// signed zero) is unaffected.  Signs of zeros: x = -0 gives q0 = -0,
// e' = -0 * s + 0 = +0 and q = -0 - (+0 * y) = -0; x = +0 gives +0 (with the
// residual of the other sign, x - q0 * s, the sum of opposite zeros would
// round -0 up to +0).  No clamp: s is amax / 448 rounded (or the 1e-6 floor
// above it), so |x / s| <= 448 (1 + 2^-22), which the native conversion
// rounds to 448 like the clamped value.  Rows whose scale is infinite or
// NaN (an infinite or NaN element) take the division itself.
__device__ __forceinline__ u32x2 quantize8(const float (&x)[8], float s) {
  float q[8];
  if (s < 0x1p125f) {
    const float y = 1.0f / s;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float q0 = x[i] * y;
      const float en = __builtin_fmaf(q0, s, -x[i]);
      q[i] = __builtin_fmaf(-en, y, q0);
    }
    u32x2 out;
    out[0] = fp8_cvt4_in_range(q[0], q[1], q[2], q[3]);
    out[1] = fp8_cvt4_in_range(q[4], q[5], q[6], q[7]);
    return out;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = nan_min(nan_max(x[i] / s, -kFp8Max), kFp8Max);
  u32x2 out;
  out[0] = fp8_encode4(q[0], q[1], q[2], q[3]);
  out[1] = fp8_encode4(q[4], q[5], q[6], q[7]);
  return out;
}

// Max over each aligned group of LANES lanes (LANES <= 16 by DPP row
// operations inside a 16-lane row; wider groups finish with shuffles).
// NaN-propagating like nan_max.
template <int LANES>
__device__ __forceinline__ float group_max(float v) {
  auto dpp = [](float x, auto ctrl) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xF, 0xF, false));
  };
  if constexpr (LANES >= 2) v = nan_max(v, dpp(v, std::integral_constant<int, 0xB1>{}));   // quad_perm [1,0,3,2]
  if constexpr (LANES >= 4) v = nan_max(v, dpp(v, std::integral_constant<int, 0x4E>{}));   // quad_perm [2,3,0,1]
  if constexpr (LANES >= 8) v = nan_max(v, dpp(v, std::integral_constant<int, 0x141>{}));  // row_half_mirror
  if constexpr (LANES >= 16) v = nan_max(v, dpp(v, std::integral_constant<int, 0x140>{})); // row_mirror
#pragma unroll
  for (int off = 16; off < LANES; off <<= 1) v = nan_max(v, __shfl_xor(v, off, LANES));
  return v;
}

// One row of D = 8 * LANES elements, eight per lane -> E4M3FN bytes and the
// row's scale s = max(amax|x| / 448, 1e-6).
template <int LANES>
__device__ __forceinline__ u32x2 quantize_row(const float (&x)[8], float& s) {
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) amax = nan_max(amax, fabsf(x[i]));
  amax = group_max<LANES>(amax);
  s = amax / kFp8Max;
  s = (s < kScaleFloor) ? kScaleFloor : s;  // clamp(min=) keeping NaN
  return quantize8(x, s);
}

}  // namespace prism
