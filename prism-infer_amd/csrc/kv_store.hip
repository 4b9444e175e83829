// KV store: bf16/fp16/fp32 K and V -> paged cache slots.
//
// Scaled FP8 (the hot path) restates the per-(token, kv head) quantiser of
// prism_infer/ops/kv_cache_store.py:81-167 (Triton) / :205-227 (eager):
//     s = max(amax|x| / 448, 1e-6)      fp32, IEEE division
//     q = e4m3fn(clamp(x / s, -448, 448))
// bit-exactly against the eager path (correctly rounded division, native RNE
// conversion, NaN propagation as torch's amax/clamp/cast do).
//
// The division is evaluated as one reciprocal per row plus two fused steps
// per element (quantize8), which gives the same correctly rounded quotient.
//
// Work layout.  A "unit" is one (token, K|V, head) row of D elements, handled
// by D/8 lanes that each load 8 consecutive elements (16 bytes for bf16/fp16),
// reduce |x| max across the unit, and write 8 FP8 bytes.
// * Token path (a token's heads fill whole waves, e.g. 8 heads x 128): one
//   wave per token issues all of the token's K and V loads at once and
//   writes through buffer resources that drop the stores of skipped slots.
// * Vector path (other power-of-two D): one thread group per unit.
// * Row path (16- and 32-bit caches): a plain or converting copy of a token's
//   K and V rows, one wave per token.
// * Scalar path: anything else (any D, alignment or stride).
#include "common.h"
#include "kv_quant.h"

#include <type_traits>

namespace prism {
namespace {

__device__ __forceinline__ float load_scalar(const void* base, int dtype, int64_t idx) {
  if (dtype == PRISM_DTYPE_F32) return static_cast<const float*>(base)[idx];
  uint32_t bits = static_cast<const uint16_t*>(base)[idx];
  return dtype == PRISM_DTYPE_BF16 ? bf16_bits_to_f32(bits) : f16_bits_to_f32(bits);
}

// Vector path: LANES = D / 8 lanes per unit, power of two <= 64.
template <int IN_DTYPE, int LANES, bool SCALED>
__global__ void __launch_bounds__(256)
kv_store_vec_kernel(const char* __restrict__ key, const char* __restrict__ value,
                    int64_t key_tok_stride_bytes, int64_t value_tok_stride_bytes,
                    uint8_t* __restrict__ k_cache, uint8_t* __restrict__ v_cache,
                    float* __restrict__ k_scale, float* __restrict__ v_scale,
                    const int32_t* __restrict__ slot_mapping, int64_t num_units, int num_heads,
                    int64_t num_slots) {
  constexpr int IN_BYTES = (IN_DTYPE == PRISM_DTYPE_F32) ? 4 : 2;
  constexpr int D = LANES * 8;
  const int64_t unit = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / LANES;
  const int sub = threadIdx.x % LANES;
  if (unit >= num_units) return;  // whole units leave together
  const int two_h = 2 * num_heads;
  const int64_t token = unit / two_h;
  const int rem = static_cast<int>(unit - token * two_h);
  const int which = rem >= num_heads;  // 0 = K, 1 = V
  const int head = rem - which * num_heads;
  const int32_t slot = slot_mapping[token];
  if (slot < 0 || slot >= num_slots) return;

  const char* src = which ? value : key;
  const int64_t tok_stride = which ? value_tok_stride_bytes : key_tok_stride_bytes;
  const char* row = src + token * tok_stride + static_cast<int64_t>(head) * D * IN_BYTES;
  float x[8];
  InVec8<IN_DTYPE>::load(row + sub * 8 * IN_BYTES, x);

  uint8_t* cache = which ? v_cache : k_cache;
  uint8_t* dst = cache + (static_cast<int64_t>(slot) * num_heads + head) * D + sub * 8;
  u32x2 packed;
  if constexpr (SCALED) {
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = nan_max(amax, fabsf(x[i]));
#pragma unroll
    for (int off = 1; off < LANES; off <<= 1) amax = nan_max(amax, __shfl_xor(amax, off, LANES));
    float s = amax / kFp8Max;
    s = (s < kScaleFloor) ? kScaleFloor : s;  // clamp(min=) keeping NaN
    packed = quantize8(x, s);
    if (sub == 0) {
      float* scales = which ? v_scale : k_scale;
      scales[static_cast<int64_t>(slot) * num_heads + head] = s;
    }
  } else {
    packed[0] = fp8_encode4(x[0], x[1], x[2], x[3]);
    packed[1] = fp8_encode4(x[4], x[5], x[6], x[7]);
  }
  *reinterpret_cast<u32x2*>(dst) = packed;
}

// A raw buffer resource over [base, base + bytes); accesses at or past
// `bytes` are dropped by the hardware (stores) or read as zero (loads).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_over(void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(base, 0, static_cast<int>(bytes), 0x00020000);
}

// Cache-policy operand of the token path's buffer stores: non-temporal.  The
// cache rows are written once here and read back by a later decode, so
// they need not occupy the caches on the way (the input rows are read with
// non-temporal loads for the same reason).
constexpr int kNtPolicy = 2;

// Token path: one wave per token, no branches on the slot.  Every lane
// issues all of its 2 * PASSES 16-byte input loads (K passes, then V passes)
// together with the slot load, so a wave has the token's whole K and V rows
// in flight at once.  The slot selects the destination rows through buffer
// resources whose extent is zero when the slot is -1 or out of range, so
// those stores are dropped by the hardware.  Pass p of a tensor covers heads
// [p * 64 / LANES, (p + 1) * 64 / LANES): consecutive lanes read consecutive
// 16-byte chunks of the token row and write consecutive 8-byte chunks of the
// slot row.  Quantisation is quantize8, as on the vector path.
template <int IN_DTYPE, int LANES, int PASSES, bool SCALED>
__global__ void __launch_bounds__(256)
kv_store_token_kernel(const char* __restrict__ key, const char* __restrict__ value,
                      int64_t key_tok_stride_bytes, int64_t value_tok_stride_bytes,
                      uint8_t* __restrict__ k_cache, uint8_t* __restrict__ v_cache,
                      float* __restrict__ k_scale, float* __restrict__ v_scale,
                      const int32_t* __restrict__ slot_mapping, int64_t num_tokens, int64_t num_slots) {
  constexpr int IN_BYTES = (IN_DTYPE == PRISM_DTYPE_F32) ? 4 : 2;
  constexpr int D = LANES * 8;
  constexpr int HEADS_PER_PASS = 64 / LANES;
  constexpr int H = HEADS_PER_PASS * PASSES;
  constexpr uint32_t kRowBytes = H * D;          // one token's payload row
  constexpr uint32_t kScaleBytes = H * 4;         // one token's scale row
  const int64_t token = static_cast<int64_t>(blockIdx.x) * (blockDim.x / 64) + threadIdx.x / 64;
  if (token >= num_tokens) return;  // wave-uniform
  const int lane = threadIdx.x % 64;
  const int sub = lane % LANES;

  using Raw = typename std::conditional<IN_BYTES == 4, u32x4[2], u32x4[1]>::type;
  Raw raw[2][PASSES];
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    const char* row = (which ? value + token * value_tok_stride_bytes : key + token * key_tok_stride_bytes) +
                      static_cast<int64_t>(lane) * 8 * IN_BYTES;
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const u32x4* src = reinterpret_cast<const u32x4*>(row + p * 64 * 8 * IN_BYTES);
#pragma unroll
      for (int c = 0; c < IN_BYTES / 2; ++c) raw[which][p][c] = __builtin_nontemporal_load(src + c);
    }
  }
  const int32_t slot = __builtin_amdgcn_readfirstlane(slot_mapping[token]);
  const bool valid = slot >= 0 && slot < num_slots;
  const int64_t row_slot = valid ? slot : 0;

#pragma unroll
  for (int which = 0; which < 2; ++which) {
    const __amdgpu_buffer_rsrc_t out_row =
        buffer_over((which ? v_cache : k_cache) + row_slot * kRowBytes, valid ? kRowBytes : 0u);
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      float x[8];
      InVec8<IN_DTYPE>::load(&raw[which][p][0], x);
      const int head = p * HEADS_PER_PASS + lane / LANES;
      u32x2 packed;
      if constexpr (SCALED) {
        float s;
        packed = quantize_row<LANES>(x, s);
        if (sub == 0) {
          const __amdgpu_buffer_rsrc_t scale_row =
              buffer_over((which ? v_scale : k_scale) + row_slot * H, valid ? kScaleBytes : 0u);
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(s), scale_row, head * 4, 0, kNtPolicy);
        }
      } else {
        packed[0] = fp8_encode4(x[0], x[1], x[2], x[3]);
        packed[1] = fp8_encode4(x[4], x[5], x[6], x[7]);
      }
      __builtin_amdgcn_raw_buffer_store_b64(packed, out_row, (p * 64 + lane) * 8, 0, kNtPolicy);
    }
  }
}

// Eight elements of a dense row, converted to the cache's dtype (through fp32,
// as the scalar path does; elements of the cache's own dtype move bit for bit).
template <int IN_DTYPE, int OUT_DTYPE>
__device__ __forceinline__ void convert8(const u32x4* in, u32x4* out) {
  if constexpr (IN_DTYPE == OUT_DTYPE) {
    out[0] = in[0];
    if constexpr (IN_DTYPE == PRISM_DTYPE_F32) out[1] = in[1];
  } else {
    float x[8];
    InVec8<IN_DTYPE>::load(in, x);
    if constexpr (OUT_DTYPE == PRISM_DTYPE_F32) {
#pragma unroll
      for (int i = 0; i < 8; ++i) out[i / 4][i % 4] = __float_as_uint(x[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t lo = OUT_DTYPE == PRISM_DTYPE_BF16 ? f32_to_bf16_bits(x[2 * i]) : f32_to_f16_bits(x[2 * i]);
        const uint32_t hi =
            OUT_DTYPE == PRISM_DTYPE_BF16 ? f32_to_bf16_bits(x[2 * i + 1]) : f32_to_f16_bits(x[2 * i + 1]);
        out[0][i] = lo | (hi << 16);
      }
    }
  }
}

// Row path: a token's heads are one dense row of `chunks` 8-element chunks, in
// the input and in the cache, so the store is a copy (with a conversion where
// the dtypes differ) bound by HBM.  One wave per token, kRowUnroll chunks of K
// and of V per lane in flight (the whole of an 8 x 128 row), each byte touched
// once: non-temporal both ways.  The scalar path walks a row per thread, two
// bytes at a time, lanes 2 D bytes apart.
// 3001 tokens of 8 x 128 bf16: 89 us on the scalar path, 5.9 us (4.2 TB/s) here;
// 32 tokens: 73 us and 4.1 us.
constexpr int kRowUnroll = 2;

template <int IN_DTYPE, int OUT_DTYPE>
__global__ void __launch_bounds__(256)
kv_store_row_kernel(const char* __restrict__ key, const char* __restrict__ value, int64_t key_tok_stride_bytes,
                    int64_t value_tok_stride_bytes, char* __restrict__ k_cache, char* __restrict__ v_cache,
                    const int32_t* __restrict__ slot_mapping, int64_t num_tokens, int chunks, int64_t num_slots) {
  constexpr int kIn = IN_DTYPE == PRISM_DTYPE_F32 ? 2 : 1;    // 16-byte words of an input chunk
  constexpr int kOut = OUT_DTYPE == PRISM_DTYPE_F32 ? 2 : 1;  // and of a cache chunk
  const int64_t token = static_cast<int64_t>(blockIdx.x) * (blockDim.x / 64) + threadIdx.x / 64;
  if (token >= num_tokens) return;  // wave-uniform
  const int lane = threadIdx.x % 64;
  const int32_t slot = __builtin_amdgcn_readfirstlane(slot_mapping[token]);
  const bool valid = slot >= 0 && slot < num_slots;
  const u32x4* src[2] = {reinterpret_cast<const u32x4*>(key + token * key_tok_stride_bytes),
                         reinterpret_cast<const u32x4*>(value + token * value_tok_stride_bytes)};
  const int64_t row = static_cast<int64_t>(valid ? slot : 0) * chunks * kOut;
  u32x4* dst[2] = {reinterpret_cast<u32x4*>(k_cache) + row, reinterpret_cast<u32x4*>(v_cache) + row};
  for (int c0 = lane; c0 < chunks; c0 += 64 * kRowUnroll) {
    u32x4 raw[2][kRowUnroll][kIn];
#pragma unroll
    for (int which = 0; which < 2; ++which) {
#pragma unroll
      for (int u = 0; u < kRowUnroll; ++u) {
        const int c = c0 + 64 * u;
#pragma unroll
        for (int w = 0; w < kIn; ++w)
          if (c < chunks) raw[which][u][w] = __builtin_nontemporal_load(src[which] + c * kIn + w);
      }
    }
    if (!valid) return;  // the loads above do not wait for the slot
#pragma unroll
    for (int which = 0; which < 2; ++which) {
#pragma unroll
      for (int u = 0; u < kRowUnroll; ++u) {
        const int c = c0 + 64 * u;
        if (c >= chunks) continue;
        u32x4 out[kOut];
        convert8<IN_DTYPE, OUT_DTYPE>(raw[which][u], out);
#pragma unroll
        for (int w = 0; w < kOut; ++w) __builtin_nontemporal_store(out[w], dst[which] + c * kOut + w);
      }
    }
  }
}

// Scalar path: one thread per unit (any head_dim, any alignment, any cache
// dtype).  Used for shapes the other paths do not cover.
__global__ void __launch_bounds__(256)
kv_store_scalar_kernel(const void* __restrict__ key, const void* __restrict__ value, int in_dtype,
                       int64_t k_st, int64_t k_sh, int64_t k_sd, int64_t v_st, int64_t v_sh,
                       int64_t v_sd, void* __restrict__ k_cache, void* __restrict__ v_cache,
                       int cache_dtype, float* __restrict__ k_scale, float* __restrict__ v_scale,
                       const int32_t* __restrict__ slot_mapping, int64_t num_units, int num_heads,
                       int head_dim, int64_t num_slots) {
  const int64_t unit = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (unit >= num_units) return;
  const int two_h = 2 * num_heads;
  const int64_t token = unit / two_h;
  const int rem = static_cast<int>(unit - token * two_h);
  const int which = rem >= num_heads;
  const int head = rem - which * num_heads;
  const int32_t slot = slot_mapping[token];
  if (slot < 0 || slot >= num_slots) return;
  const void* src = which ? value : key;
  const int64_t base = which ? (token * v_st + head * v_sh) : (token * k_st + head * k_sh);
  const int64_t sd = which ? v_sd : k_sd;
  void* cache = which ? v_cache : k_cache;
  const int64_t out_base = (static_cast<int64_t>(slot) * num_heads + head) * head_dim;
  const bool scaled = k_scale != nullptr;
  float s = 1.0f;
  if (scaled) {
    float amax = 0.0f;
    for (int d = 0; d < head_dim; ++d) amax = nan_max(amax, fabsf(load_scalar(src, in_dtype, base + d * sd)));
    s = amax / kFp8Max;
    s = (s < kScaleFloor) ? kScaleFloor : s;
    float* scales = which ? v_scale : k_scale;
    scales[static_cast<int64_t>(slot) * num_heads + head] = s;
  }
  for (int d = 0; d < head_dim; ++d) {
    float x = load_scalar(src, in_dtype, base + d * sd);
    if (cache_dtype == PRISM_DTYPE_FP8_E4M3FN) {
      if (scaled) x = nan_min(nan_max(x / s, -kFp8Max), kFp8Max);
      static_cast<uint8_t*>(cache)[out_base + d] = static_cast<uint8_t>(fp8_encode4(x, 0.f, 0.f, 0.f) & 0xFFu);
    } else if (cache_dtype == PRISM_DTYPE_F32) {
      static_cast<float*>(cache)[out_base + d] = x;
    } else if (cache_dtype == PRISM_DTYPE_BF16) {
      // Inputs of the cache's own dtype are copied bit for bit.
      uint16_t bits = (in_dtype == PRISM_DTYPE_BF16)
                          ? static_cast<const uint16_t*>(src)[base + d * sd]
                          : f32_to_bf16_bits(x);
      static_cast<uint16_t*>(cache)[out_base + d] = bits;
    } else {
      uint16_t bits = (in_dtype == PRISM_DTYPE_F16)
                          ? static_cast<const uint16_t*>(src)[base + d * sd]
                          : f32_to_f16_bits(x);
      static_cast<uint16_t*>(cache)[out_base + d] = bits;
    }
  }
}

template <int IN_DTYPE, int LANES, int PASSES>
int launch_token(const void* key, const void* value, int64_t k_tok_bytes, int64_t v_tok_bytes,
                 void* k_cache, void* v_cache, float* k_scale, float* v_scale, const int32_t* slots,
                 int64_t num_tokens, int64_t num_slots, hipStream_t stream) {
  const int64_t blocks = ceil_div(num_tokens, 4);  // four waves (tokens) per block
  if (blocks > INT32_MAX) {
    set_error("prism_kv_store: too many tokens for one launch");
    return PRISM_ERR_INVALID;
  }
  const char* k = static_cast<const char*>(key);
  const char* v = static_cast<const char*>(value);
  uint8_t* kc = static_cast<uint8_t*>(k_cache);
  uint8_t* vc = static_cast<uint8_t*>(v_cache);
  if (k_scale) {
    hipLaunchKernelGGL((kv_store_token_kernel<IN_DTYPE, LANES, PASSES, true>), dim3(blocks), dim3(256), 0, stream,
                       k, v, k_tok_bytes, v_tok_bytes, kc, vc, k_scale, v_scale, slots, num_tokens, num_slots);
  } else {
    hipLaunchKernelGGL((kv_store_token_kernel<IN_DTYPE, LANES, PASSES, false>), dim3(blocks), dim3(256), 0, stream,
                       k, v, k_tok_bytes, v_tok_bytes, kc, vc, nullptr, nullptr, slots, num_tokens, num_slots);
  }
  return check_launch("kv_store_token_kernel launch");
}

template <int IN_DTYPE, int LANES>
int launch_vec(const void* key, const void* value, int64_t k_tok_bytes, int64_t v_tok_bytes,
               void* k_cache, void* v_cache, float* k_scale, float* v_scale, const int32_t* slots,
               int64_t num_units, int num_heads, int64_t num_slots, hipStream_t stream) {
  // A token's heads fill whole waves: one wave per token.
  if constexpr (LANES >= 4) {
    if (num_heads * LANES % 64 == 0) {
      const int64_t tokens = num_units / (2 * num_heads);
      switch (num_heads * LANES / 64) {
        case 1: return launch_token<IN_DTYPE, LANES, 1>(key, value, k_tok_bytes, v_tok_bytes, k_cache, v_cache,
                                                        k_scale, v_scale, slots, tokens, num_slots, stream);
        case 2: return launch_token<IN_DTYPE, LANES, 2>(key, value, k_tok_bytes, v_tok_bytes, k_cache, v_cache,
                                                        k_scale, v_scale, slots, tokens, num_slots, stream);
        case 4: return launch_token<IN_DTYPE, LANES, 4>(key, value, k_tok_bytes, v_tok_bytes, k_cache, v_cache,
                                                        k_scale, v_scale, slots, tokens, num_slots, stream);
        default: break;
      }
    }
  }
  const int64_t threads = num_units * LANES;
  const int64_t blocks = ceil_div(threads, 256);
  if (blocks > INT32_MAX) {
    set_error("prism_kv_store: too many tokens for one launch");
    return PRISM_ERR_INVALID;
  }
  if (k_scale) {
    hipLaunchKernelGGL((kv_store_vec_kernel<IN_DTYPE, LANES, true>), dim3(blocks), dim3(256), 0, stream,
                       static_cast<const char*>(key), static_cast<const char*>(value), k_tok_bytes,
                       v_tok_bytes, static_cast<uint8_t*>(k_cache), static_cast<uint8_t*>(v_cache),
                       k_scale, v_scale, slots, num_units, num_heads, num_slots);
  } else {
    hipLaunchKernelGGL((kv_store_vec_kernel<IN_DTYPE, LANES, false>), dim3(blocks), dim3(256), 0, stream,
                       static_cast<const char*>(key), static_cast<const char*>(value), k_tok_bytes,
                       v_tok_bytes, static_cast<uint8_t*>(k_cache), static_cast<uint8_t*>(v_cache),
                       nullptr, nullptr, slots, num_units, num_heads, num_slots);
  }
  return check_launch("kv_store_vec_kernel launch");
}

template <int IN_DTYPE>
int dispatch_lanes(int lanes, const void* key, const void* value, int64_t kb, int64_t vb, void* kc,
                   void* vc, float* ks, float* vs, const int32_t* slots, int64_t units, int heads,
                   int64_t num_slots, hipStream_t stream) {
  switch (lanes) {
    case 1: return launch_vec<IN_DTYPE, 1>(key, value, kb, vb, kc, vc, ks, vs, slots, units, heads, num_slots, stream);
    case 2: return launch_vec<IN_DTYPE, 2>(key, value, kb, vb, kc, vc, ks, vs, slots, units, heads, num_slots, stream);
    case 4: return launch_vec<IN_DTYPE, 4>(key, value, kb, vb, kc, vc, ks, vs, slots, units, heads, num_slots, stream);
    case 8: return launch_vec<IN_DTYPE, 8>(key, value, kb, vb, kc, vc, ks, vs, slots, units, heads, num_slots, stream);
    case 16: return launch_vec<IN_DTYPE, 16>(key, value, kb, vb, kc, vc, ks, vs, slots, units, heads, num_slots, stream);
    case 32: return launch_vec<IN_DTYPE, 32>(key, value, kb, vb, kc, vc, ks, vs, slots, units, heads, num_slots, stream);
    case 64: return launch_vec<IN_DTYPE, 64>(key, value, kb, vb, kc, vc, ks, vs, slots, units, heads, num_slots, stream);
    default: return PRISM_ERR_LAYOUT;
  }
}

template <int IN_DTYPE, int OUT_DTYPE>
int launch_rows(const void* key, const void* value, int64_t k_tok_bytes, int64_t v_tok_bytes, void* k_cache,
                void* v_cache, const int32_t* slots, int64_t num_tokens, int chunks, int64_t num_slots,
                hipStream_t stream) {
  // Four tokens per block; one where the tokens alone would leave most CUs
  // without a block.  One and four: 8 x 128 float32, 256 tokens 3.1 and 3.8 us,
  // 1023 5.2 and 5.4, 2048 8.8 and 8.7; bf16, up to 1023 tokens within 0.2 us,
  // 2048 5.2 and 4.6, 3001 6.3 and 5.6; 1 x 128, 8192 tokens 5.0 and 4.1.
  const int waves = num_tokens >= 1024 ? 4 : 1;
  const int64_t blocks = ceil_div(num_tokens, waves);
  if (blocks > INT32_MAX) {
    set_error("prism_kv_store: too many tokens for one launch");
    return PRISM_ERR_INVALID;
  }
  hipLaunchKernelGGL((kv_store_row_kernel<IN_DTYPE, OUT_DTYPE>), dim3(blocks), dim3(64 * waves), 0, stream,
                     static_cast<const char*>(key), static_cast<const char*>(value), k_tok_bytes, v_tok_bytes,
                     static_cast<char*>(k_cache), static_cast<char*>(v_cache), slots, num_tokens, chunks, num_slots);
  return check_launch("kv_store_row_kernel launch");
}

template <int IN_DTYPE>
int dispatch_rows(int cache_dtype, const void* key, const void* value, int64_t kb, int64_t vb, void* kc, void* vc,
                  const int32_t* slots, int64_t tokens, int chunks, int64_t num_slots, hipStream_t stream) {
  switch (cache_dtype) {
    case PRISM_DTYPE_F32:
      return launch_rows<IN_DTYPE, PRISM_DTYPE_F32>(key, value, kb, vb, kc, vc, slots, tokens, chunks, num_slots, stream);
    case PRISM_DTYPE_BF16:
      return launch_rows<IN_DTYPE, PRISM_DTYPE_BF16>(key, value, kb, vb, kc, vc, slots, tokens, chunks, num_slots, stream);
    default:
      return launch_rows<IN_DTYPE, PRISM_DTYPE_F16>(key, value, kb, vb, kc, vc, slots, tokens, chunks, num_slots, stream);
  }
}

}  // namespace

// Loads this file's code object now rather than at its first kernel launch.
int preload_kv_store() {
  hipFuncAttributes attr;
  return check_hip(hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(&kv_store_scalar_kernel)), "preload_kv_store");
}

}  // namespace prism

extern "C" int prism_kv_store(const void* key, const void* value, int in_dtype,
                              const int64_t key_strides[3], const int64_t value_strides[3],
                              void* k_cache, void* v_cache, int cache_dtype, float* k_scale,
                              float* v_scale, const int32_t* slot_mapping, int64_t num_tokens,
                              int num_heads, int head_dim, int64_t num_slots, void* stream_ptr) {
  using namespace prism;
  clear_error();
  if (num_tokens < 0 || num_heads <= 0 || head_dim <= 0 || num_slots < 0) {
    set_error("prism_kv_store: invalid geometry tokens=%lld heads=%d head_dim=%d slots=%lld",
              static_cast<long long>(num_tokens), num_heads, head_dim, static_cast<long long>(num_slots));
    return PRISM_ERR_INVALID;
  }
  if (in_dtype != PRISM_DTYPE_F32 && in_dtype != PRISM_DTYPE_BF16 && in_dtype != PRISM_DTYPE_F16) {
    set_error("prism_kv_store: unsupported input dtype code %d", in_dtype);
    return PRISM_ERR_INVALID;
  }
  if (dtype_size(cache_dtype) == 0) {
    set_error("prism_kv_store: unsupported cache dtype code %d", cache_dtype);
    return PRISM_ERR_INVALID;
  }
  if ((k_scale == nullptr) != (v_scale == nullptr)) {
    set_error("prism_kv_store: K/V scale caches must be provided together");
    return PRISM_ERR_INVALID;
  }
  if (k_scale && cache_dtype != PRISM_DTYPE_FP8_E4M3FN) {
    set_error("prism_kv_store: token-head scales require FP8 K/V payload caches");
    return PRISM_ERR_INVALID;
  }
  if (!key || !value || !k_cache || !v_cache || !slot_mapping || !key_strides || !value_strides) {
    if (num_tokens == 0) return PRISM_OK;
    set_error("prism_kv_store: null pointer argument");
    return PRISM_ERR_INVALID;
  }
  if (num_tokens == 0) return PRISM_OK;
  hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
  const int64_t units = num_tokens * 2 * num_heads;
  const int in_bytes = dtype_size(in_dtype);
  const int lanes = head_dim / 8;
  const bool dense_rows = key_strides[2] == 1 && value_strides[2] == 1 && key_strides[1] == head_dim &&
                          value_strides[1] == head_dim;
  const bool pow2_lanes = head_dim % 8 == 0 && lanes >= 1 && lanes <= 64 && (lanes & (lanes - 1)) == 0;
  const int64_t kb = key_strides[0] * in_bytes;
  const int64_t vb = value_strides[0] * in_bytes;
  const bool vec_aligned = aligned(key, 16) && aligned(value, 16) && kb % 16 == 0 && vb % 16 == 0 &&
                           aligned(k_cache, 8) && aligned(v_cache, 8);
  if (cache_dtype == PRISM_DTYPE_FP8_E4M3FN && dense_rows && pow2_lanes && vec_aligned) {
    switch (in_dtype) {
      case PRISM_DTYPE_BF16:
        return dispatch_lanes<PRISM_DTYPE_BF16>(lanes, key, value, kb, vb, k_cache, v_cache, k_scale, v_scale,
                                                slot_mapping, units, num_heads, num_slots, stream);
      case PRISM_DTYPE_F16:
        return dispatch_lanes<PRISM_DTYPE_F16>(lanes, key, value, kb, vb, k_cache, v_cache, k_scale, v_scale,
                                               slot_mapping, units, num_heads, num_slots, stream);
      default:
        return dispatch_lanes<PRISM_DTYPE_F32>(lanes, key, value, kb, vb, k_cache, v_cache, k_scale, v_scale,
                                               slot_mapping, units, num_heads, num_slots, stream);
    }
  }
  // Row path: dense rows of whole 16-byte chunks on both sides (8 elements; the
  // cache's rows follow from its base, which 16-byte aligned rows keep aligned).
  const int64_t row_elems = static_cast<int64_t>(num_heads) * head_dim;
  if (cache_dtype != PRISM_DTYPE_FP8_E4M3FN && dense_rows && row_elems % 8 == 0 && row_elems <= INT32_MAX &&
      aligned(key, 16) && aligned(value, 16) && kb % 16 == 0 && vb % 16 == 0 && aligned(k_cache, 16) &&
      aligned(v_cache, 16)) {
    const int chunks = static_cast<int>(row_elems / 8);
    switch (in_dtype) {
      case PRISM_DTYPE_BF16:
        return dispatch_rows<PRISM_DTYPE_BF16>(cache_dtype, key, value, kb, vb, k_cache, v_cache, slot_mapping,
                                               num_tokens, chunks, num_slots, stream);
      case PRISM_DTYPE_F16:
        return dispatch_rows<PRISM_DTYPE_F16>(cache_dtype, key, value, kb, vb, k_cache, v_cache, slot_mapping,
                                              num_tokens, chunks, num_slots, stream);
      default:
        return dispatch_rows<PRISM_DTYPE_F32>(cache_dtype, key, value, kb, vb, k_cache, v_cache, slot_mapping,
                                              num_tokens, chunks, num_slots, stream);
    }
  }
  const int64_t blocks = ceil_div(units, 256);
  hipLaunchKernelGGL(kv_store_scalar_kernel, dim3(blocks), dim3(256), 0, stream, key, value, in_dtype,
                     key_strides[0], key_strides[1], key_strides[2], value_strides[0], value_strides[1],
                     value_strides[2], k_cache, v_cache, cache_dtype, k_scale, v_scale, slot_mapping, units,
                     num_heads, head_dim, num_slots);
  return check_launch("kv_store_scalar_kernel launch");
}
