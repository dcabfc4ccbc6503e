// gfx950 writer of new tokens' K/V into their page slots: the device side of
// scatter_kv_batch_to_pages_cu / scatter_kv_batch_to_pages_fp8_e4m3_cu
// (scatter_kv_kernel.cu:99-216).
//
// Work unit: one lane moves one 16-byte vector of a token's K row and the same
// of its V row, or (scatter_kv_vector_kernel) one vector of either. Units run
// token-major ([token][vector], [token][K|V][vector]), so a wave reads
// contiguous stretches of the token-major K and V inputs and writes whole rows
// of the pages. A token's rows share one slot, so every lane of a row takes
// the same skip-or-write decision; for FP8 a (token, K|V, head) group of lanes
// shares one amax through DPP, and the group's first lane writes the scale.
//
// Memory: each input vector is read once (non-temporal load); the pages are
// read by this layer's attention next, so stores keep the default policy.
//
// What bounds it: the index arithmetic and the divisions per vector in large
// calls (hence K and V in one lane, which share the former and interleave the
// latter), the launch and one chain of arguments, slot and input in small
// ones, where a pair's chain is the longer one. us on MI355X, launches in a
// graph, a vector against a pair per lane: 8,192 tokens of 4 x 128 BF16 to FP8
// 8.3 and 7.2 (3.4 TB/s), FP32 kept 15.3 and 12.7 (5.2 TB/s); 5,040 tokens of
// 2 x 128 FP32 to FP8 5.7 and 4.8, BF16 to FP8 4.1 and 4.0; 1 token to FP8 1.9
// and 2.1, 700 tokens 2.45 and 2.53. The line: pairs in more than two
// workgroups per compute unit, or, where nothing is converted, in at most one;
// in between the pairs' workgroups load some compute units twice and others
// once (1,500 tokens of 4 x 128 BF16 kept 2.57 and 2.68, to FP8 3.03 and 3.21;
// of 2 x 128 FP32 kept 2.50 and 2.72; 16 tokens BF16 kept 2.00 and 1.87).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

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

template <bool kF32, bool kFp8, int kLanesPerHead>
__global__ __launch_bounds__(kThreadsPerBlock) void scatter_kv_vector_kernel(const ScatterParams p) {
  const uint32_t u = blockIdx.x * kThreadsPerBlock + threadIdx.x;
  if (u >= p.units) return;
  const uint32_t token = div_by(u, p.by_row);           // 2 rows (K, V) per token
  const uint32_t in_pair = u - token * 2u * p.vecs_per_row;
  const uint32_t kv = in_pair >= p.vecs_per_row ? 1u : 0u;
  const uint32_t vec = in_pair - kv * p.vecs_per_row;
  // The input vector does not depend on the slot: both loads go out together,
  // so a wave waits for one memory round trip before its store, not two.
  const uint8_t* in = (kv ? p.values : p.keys) + (uint64_t)token * p.row_in_bytes;
  const u32x4 x = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(in + (uint64_t)vec * 16u));
  const int32_t slot = p.slots ? p.slots[token] : p.fixed_slot;
  if (slot < 0) return;  // scatter_kv_kernel.cu:147-149
  const uint32_t block = div_by((uint32_t)slot, p.by_block_size);
  const uint32_t offset = (uint32_t)slot - block * p.block_size;
  const uint64_t out_row = (uint64_t)block * p.block_out_bytes + (uint64_t)offset * p.row_out_bytes;
  if (out_row + p.row_out_bytes > (kv ? p.value_pool_bytes : p.key_pool_bytes)) return;
  uint8_t* out = (kv ? p.value_pool : p.key_pool) + out_row;
  if constexpr (!kFp8) {
    *reinterpret_cast<u32x4*>(out + (uint64_t)vec * 16u) = x;  // plain: the pool holds the input type
  } else {
    const uint32_t head = vec / kLanesPerHead;
    const uint64_t scale_idx = ((uint64_t)block * p.block_size + offset) * p.kv_heads + head;
    if (scale_idx >= (kv ? p.value_scale_count : p.key_scale_count)) return;
    const float m = group_max<kLanesPerHead>(kF32 ? amax4(x) : amax8(x));
    const float inv = m > 0.f ? 448.f / m : 0.f;
    if (vec % kLanesPerHead == 0) (kv ? p.value_scales : p.key_scales)[scale_idx] = m > 0.f ? m / 448.f : 1.f;
    if constexpr (kF32)
      *reinterpret_cast<uint32_t*>(out + (uint64_t)vec * 4u) = quantise4(x, inv);
    else
      *reinterpret_cast<u32x2*>(out + (uint64_t)vec * 8u) = quantise8(x, inv);
  }
}

template <bool kF32, bool kFp8>
hipError_t launch_lanes(const ScatterParams& p, uint32_t lanes_per_head, hipStream_t stream) {
  const dim3 grid((p.units + kThreadsPerBlock - 1) / kThreadsPerBlock), block(kThreadsPerBlock);
  auto run = [&](auto lanes) {
    constexpr int L = decltype(lanes)::value;
    if (p.pairs) hipLaunchKernelGGL((scatter_kv_kernel<kF32, kFp8, L>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((scatter_kv_vector_kernel<kF32, kFp8, L>), grid, block, 0, stream, p);
    return hipGetLastError();
  };
  if constexpr (!kFp8) {  // plain rows need no per-head grouping
    return run(std::integral_constant<int, 1>{});
  } else {
    switch (lanes_per_head) {
      case 1: return run(std::integral_constant<int, 1>{});
      case 2: return run(std::integral_constant<int, 2>{});
      case 4: return run(std::integral_constant<int, 4>{});
      case 8: return run(std::integral_constant<int, 8>{});
      case 16: return run(std::integral_constant<int, 16>{});
      case 32: return run(std::integral_constant<int, 32>{});
      case 64: return run(std::integral_constant<int, 64>{});
      default: return hipErrorInvalidValue;
    }
  }
}

}  // namespace

bool scatter_pairs(uint64_t pairs, bool fp8, int64_t compute_units) {
  const int64_t workgroups = (int64_t)((pairs + kThreadsPerBlock - 1) / kThreadsPerBlock);
  return workgroups > 2 * compute_units || (!fp8 && workgroups <= compute_units);
}

hipError_t launch_scatter_kv(const ScatterParams& p, bool f32_input, bool fp8, uint32_t lanes_per_head,
                             hipStream_t stream) {
  if (p.units == 0) return hipSuccess;
  if (!fp8) return f32_input ? launch_lanes<true, false>(p, 1, stream) : launch_lanes<false, false>(p, 1, stream);
  return f32_input ? launch_lanes<true, true>(p, lanes_per_head, stream)
                   : launch_lanes<false, true>(p, lanes_per_head, stream);
}

}  // namespace pbe
