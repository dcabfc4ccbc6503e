// Prints how the decode reader would read each batch given on standard input:
//   batch kv_heads q_heads head_dim fp8 max_blocks splits compute_units atomics address
// as
//   mode slots hshift one_round used_bytes given_bytes
// (mode 0: slots, 1: splits, 2: either; used_bytes: what the plan may write of
// the workspace, from its start). Host code only.
#include <algorithm>
#include <cstdint>
#include <cstdio>

#include "kernels/decode_kernels.h"

int main() {
  long long batch, kv, q, dim, fp8, blocks, splits, cus, atomics, address;
  while (std::scanf("%lld %lld %lld %lld %lld %lld %lld %lld %lld %lld", &batch, &kv, &q, &dim, &fp8, &blocks, &splits, &cus, &atomics, &address) == 10) {
    pbe::DecodeParams p{};
    p.batch = (int32_t)batch, p.kv_heads = (int32_t)kv, p.q_heads = (int32_t)q, p.head_dim = (int32_t)dim;
    p.max_blocks = (int32_t)blocks, p.workgroups = (int32_t)cus;
    const uint64_t bytes = pbe::decode_workspace_bytes(p.batch, p.q_heads, p.head_dim, (int32_t)splits);
    pbe::plan_decode_slots(&p, fp8 != 0, (int32_t)splits, reinterpret_cast<void*>(address), bytes, atomics != 0);
    uint64_t end = 0;
    const int64_t rows = (int64_t)p.batch * p.q_heads;
    if (p.mode != pbe::DecodeMode::kSplits && p.slots > p.batch)
      end = reinterpret_cast<uint64_t>(p.tickets + (int64_t)p.slots * (p.kv_heads >> p.hshift)) - address;
    if (p.mode != pbe::DecodeMode::kSlots) end = std::max(end, (uint64_t)(reinterpret_cast<uint64_t>(p.split_l + rows * p.splits) - address));
    std::printf("%d %d %d %d %llu %llu\n", (int)p.mode, (int)p.slots, (int)p.hshift, (int)p.one_round, (unsigned long long)end, (unsigned long long)bytes);
  }
}
