// gfx950 writer of new tokens' K/V into their page slots: the device side of
// scatter_kv_batch_to_pages_cu / scatter_kv_batch_to_pages_fp8_e4m3_cu
// (scatter_kv_kernel.cu:99-216).
//
// Work unit: one lane moves one 16-byte vector of a token's K row and the same
// of its V row. Units run token-major ([token][vector]), so a wave reads a
// contiguous stretch of the token-major K and V inputs and writes whole rows
// of the pages. A token's rows share one slot, so every lane of a row takes
// the same skip-or-write decision; for FP8 a (token, head) group of lanes
// shares one amax through DPP, and the group's first lane writes the scale.
//
// Memory: each input vector is read once (non-temporal load); the pages are
// read by this layer's attention next, so stores keep the default policy.
//
// What bounds it: the index arithmetic and the divisions per vector in large
// calls (hence K and V in one lane, which share the former and interleave the
// latter), the launch and one chain of arguments, slot and input in small
// ones. MI355X, launches in a graph, one unit per vector of K or V before:
// 8,192 tokens of 4 x 128 BF16 to FP8 9.2 to 7.4 us (3.4 TB/s), FP32 kept 16.0
// to 14.1 (4.8 TB/s); 5,040 tokens of 2 x 128 FP32 to FP8 6.0 to 5.2, BF16 to
// FP8 4.4 to 4.3; 700 tokens 2.9 both; 1 token 1.9 to 2.1.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fp8_device.h"
#include "scatter_kernels.h"

namespace pbe {
namespace {

__device__ __forceinline__ uint32_t div_by(uint32_t n, const FastDiv& f) {
  return (__umulhi(n, f.mul) + n) >> f.shift;
}

template <bool kF32, bool kFp8, int kLanesPerHead>
__global__ __launch_bounds__(kThreadsPerBlock) void scatter_kv_kernel(const ScatterParams p) {
  // One field of each cache line of the arguments, so that their first reads
  // overlap instead of each waiting where it is used.
  asm volatile("" ::"s"(p.keys), "s"(p.key_pool), "s"(p.key_pool_bytes), "s"(p.value_scales), "s"(p.slots),
               "s"(p.row_out_bytes), "s"(p.block_out_bytes), "s"(p.by_block_size.mul), "s"(p.by_row.mul), "s"(p.units));
  const uint32_t u = blockIdx.x * kThreadsPerBlock + threadIdx.x;
  if (u >= p.units) return;
  const uint32_t token = div_by(u, p.by_row);
  const uint32_t vec = u - token * p.vecs_per_row;
  // The input vectors do not depend on the slot: all loads go out together,
  // so a wave waits for one memory round trip before its stores, not two.
  const uint64_t in = (uint64_t)token * p.row_in_bytes + (uint64_t)vec * 16u;
  const u32x4 k = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.keys + in));
  const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.values + in));
  const int32_t slot = p.slots ? p.slots[token] : p.fixed_slot;
  if (slot < 0) return;  // scatter_kv_kernel.cu:147-149
  const uint32_t block = div_by((uint32_t)slot, p.by_block_size);
  const uint32_t offset = (uint32_t)slot - block * p.block_size;
  const uint64_t out_row = (uint64_t)block * p.block_out_bytes + (uint64_t)offset * p.row_out_bytes;
  bool k_fits = out_row + p.row_out_bytes <= p.key_pool_bytes, v_fits = out_row + p.row_out_bytes <= p.value_pool_bytes;
  uint8_t* const k_out = p.key_pool + out_row;
  uint8_t* const v_out = p.value_pool + out_row;
  if constexpr (!kFp8) {  // plain: the pools hold the input type
    if (k_fits) *reinterpret_cast<u32x4*>(k_out + (uint64_t)vec * 16u) = k;
    if (v_fits) *reinterpret_cast<u32x4*>(v_out + (uint64_t)vec * 16u) = v;
  } else {
    // Both rows' chains (amax, divisions, codes) are independent and run
    // interleaved; only the stores are conditional.
    const uint64_t scale_idx = ((uint64_t)block * p.block_size + offset) * p.kv_heads + vec / kLanesPerHead;
    k_fits = k_fits && scale_idx < p.key_scale_count;
    v_fits = v_fits && scale_idx < p.value_scale_count;
    const float km = group_max<kLanesPerHead>(kF32 ? amax4(k) : amax8(k)), vm = group_max<kLanesPerHead>(kF32 ? amax4(v) : amax8(v));
    const float kinv = km > 0.f ? 448.f / km : 0.f, vinv = vm > 0.f ? 448.f / vm : 0.f;
    const float ks = km > 0.f ? km / 448.f : 1.f, vs = vm > 0.f ? vm / 448.f : 1.f;
    const bool first = vec % kLanesPerHead == 0;
    if constexpr (kF32) {
      const uint32_t kc = quantise4(k, kinv), vc = quantise4(v, vinv);
      if (k_fits) *reinterpret_cast<uint32_t*>(k_out + (uint64_t)vec * 4u) = kc;
      if (v_fits) *reinterpret_cast<uint32_t*>(v_out + (uint64_t)vec * 4u) = vc;
    } else {
      const u32x2 kc = quantise8(k, kinv), vc = quantise8(v, vinv);
      if (k_fits) *reinterpret_cast<u32x2*>(k_out + (uint64_t)vec * 8u) = kc;
      if (v_fits) *reinterpret_cast<u32x2*>(v_out + (uint64_t)vec * 8u) = vc;
    }
    if (first && k_fits) p.key_scales[scale_idx] = ks;
    if (first && v_fits) p.value_scales[scale_idx] = vs;
  }
}

template <bool kF32, bool kFp8>
hipError_t launch_lanes(const ScatterParams& p, uint32_t lanes_per_head, hipStream_t stream) {
  const dim3 grid((p.units + kThreadsPerBlock - 1) / kThreadsPerBlock), block(kThreadsPerBlock);
  if constexpr (!kFp8) {  // plain rows need no per-head grouping
    hipLaunchKernelGGL((scatter_kv_kernel<kF32, false, 1>), grid, block, 0, stream, p);
    return hipGetLastError();
  }
  switch (lanes_per_head) {
    case 1: hipLaunchKernelGGL((scatter_kv_kernel<kF32, kFp8, 1>), grid, block, 0, stream, p); break;
    case 2: hipLaunchKernelGGL((scatter_kv_kernel<kF32, kFp8, 2>), grid, block, 0, stream, p); break;
    case 4: hipLaunchKernelGGL((scatter_kv_kernel<kF32, kFp8, 4>), grid, block, 0, stream, p); break;
    case 8: hipLaunchKernelGGL((scatter_kv_kernel<kF32, kFp8, 8>), grid, block, 0, stream, p); break;
    case 16: hipLaunchKernelGGL((scatter_kv_kernel<kF32, kFp8, 16>), grid, block, 0, stream, p); break;
    case 32: hipLaunchKernelGGL((scatter_kv_kernel<kF32, kFp8, 32>), grid, block, 0, stream, p); break;
    case 64: hipLaunchKernelGGL((scatter_kv_kernel<kF32, kFp8, 64>), grid, block, 0, stream, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_scatter_kv(const ScatterParams& p, bool f32_input, bool fp8, uint32_t lanes_per_head,
                             hipStream_t stream) {
  if (p.units == 0) return hipSuccess;
  if (!fp8) return f32_input ? launch_lanes<true, false>(p, 1, stream) : launch_lanes<false, false>(p, 1, stream);
  return f32_input ? launch_lanes<true, true>(p, lanes_per_head, stream)
                   : launch_lanes<false, true>(p, lanes_per_head, stream);
}

}  // namespace pbe
