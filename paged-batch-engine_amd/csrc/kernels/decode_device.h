// Device helpers of the two decode readers (decode_kernels.hip,
// decode_split_kernels.hip).
#pragma once
#include "decode_kernels.h"
#include "fp8_device.h"

namespace pbe {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

template <typename T>
using gptr = __attribute__((address_space(1))) T*;  // global memory

constexpr int kBlockTokens = 16;
template <int kCtrl>
__device__ __forceinline__ float dpp(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xf, 0xf, false));
}

// Max / sum over the four lanes j, j+16, j+32, j+48 with the gfx950 row
// swaps (VALU only, no LDS round trip). Every lane ends with the same value,
// combined in the same order.
__device__ __forceinline__ float group_max4(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

__device__ __forceinline__ float group_sum4(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Orders this wave's LDS writes before its other lanes' reads.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// fp32 -> bf16, round to nearest even; NaN stays NaN (quiet).
__device__ __forceinline__ uint16_t to_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

__device__ __forceinline__ uint32_t fast_div(uint32_t n, const FastDiv& f) {
  return (__umulhi(n, f.mul) + n) >> f.shift;
}

// Four E4M3 bytes -> four BF16 with the gfx950 scaled converter (scale 1: exact).
__device__ __forceinline__ u32x2 e4m3x4_to_bf16x4_cvt(uint32_t w) {
  return u32x2{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w, 1.0f, false)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w, 1.0f, true))};
}

// Per-lane registers of one block of 16 tokens of one KV head: the lane's
// part of key row j, its whole-row-mapped part of the value tile and one scale.
template <int D, bool kFp8>
struct Geo {
  static constexpr int E = kFp8 ? 1 : 2;
  static constexpr int WORDS = D * E / 16;   // key words = value words per lane
  static constexpr int PITCH = D * E + 16;   // LDS row pitch of the value tile
};

template <int W, bool kFp8>
struct BlockRegs {
  uint32_t k[W];
  uint32_t v[W];
  // FP8: lane (g, n): log2(e)/sqrt(D) * key scale (n%8 < 4) or value scale
  // (otherwise) of token 4g + n%4
  float scale;
};

template <int kCtrl>
__device__ __forceinline__ int max_step(int x) {
  return max(x, __builtin_amdgcn_update_dpp(x, x, kCtrl, 0xf, 0xf, false));
}
__device__ __forceinline__ int wave_max_int(int x) {
  x = max_step<0xb1>(x);
  x = max_step<0x4e>(x);
  x = max_step<0x141>(x);
  x = max_step<0x140>(x);
  return max(max(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 16)),
             max(__builtin_amdgcn_readlane(x, 32), __builtin_amdgcn_readlane(x, 48)));
}

// Blocks of a length; a bad one (negative, or beyond the table) has none.
__device__ __forceinline__ int blocks_of(int seq, int max_blocks) {
  const int n = seq > 0 ? (int)(((uint32_t)seq + kBlockTokens - 1) / kBlockTokens) : 0;
  return n <= max_blocks ? n : 0;
}

// Whether the batch's sequences are of about equal length (the shortest at
// least 7/8 of the longest). Every wave finds the same.
__device__ __forceinline__ bool alike(const int32_t* __restrict__ lens, int batch, int max_blocks, int lane) {
  int most = 0, least = 0x7fffffff;
  for (int i = lane; i < batch; i += 64) {
    const int n = blocks_of(lens[i], max_blocks);
    most = max(most, n);
    least = min(least, n);
  }
  return (int64_t)-wave_max_int(-least) * 8 >= (int64_t)wave_max_int(most) * 7;
}

}  // namespace
}  // namespace pbe
