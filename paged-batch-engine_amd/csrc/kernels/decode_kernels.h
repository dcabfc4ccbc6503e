// Internal interface of the decode-side paged-attention reader (one query
// token per sequence) over the page-major arena layout the handoff writes.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pbe {

constexpr int kDecodeMaxSegments = 16;
constexpr int kDecodeMaxKvMul = 8;    // query heads per KV head held in registers
constexpr int kDecodeMaxSplits = 1024;  // slots of one sequence

// Of one launch: 2^32 threads less one, in workgroups of 512.
constexpr int64_t kDecodeMaxWorkgroups = 0xffffffffll / 512;

struct DecodeView {
  const char* base[kDecodeMaxSegments];
  uint64_t segment_bytes;
  uint64_t bytes;
};

// Division by a fixed divisor d >= 1 for numerators below 2^31:
// q = (mulhi(n, mul) + n) >> shift (round-up reciprocal method).
struct FastDiv {
  uint32_t d = 1, mul = 1, shift = 0;
};
FastDiv make_fast_div(uint32_t d);

// How a batch is read: in slots by one launch (decode_kernels.hip), in equal
// splits by two (decode_split_kernels.hip), or in splits if its sequences are
// of about equal length and in slots otherwise. Lengths are device memory, so
// for the last all three kernels are launched and look at them.
enum class DecodeMode : int32_t { kSlots, kSplits, kEither };

struct DecodeParams {
  DecodeView kv;           // payload arena (FP8: int8 E4M3 planes; BF16: bf16 planes)
  const float* scales;     // FP8 only: page-major [layer][K|V][token][kv_head] fp32
  uint64_t scale_bytes;
  const uint16_t* q;       // bf16 [batch][q_heads][head_dim]
  uint16_t* out;           // bf16 [batch][q_heads][head_dim]
  const int32_t* tables;   // [batch][max_blocks] page-major block ids
  const int32_t* seq_lens; // [batch]
  // Partial results of the slots (see decode_kernels.hip) of sequences that
  // take more than one, and their arrival tickets.
  float* part_acc;         // [slots][q_heads][head_dim]
  float* part_ml;          // [slots][q_heads][2]: maximum, sum
  uint64_t* tickets;       // [slots][kv_heads >> hshift]
  uint64_t tag;            // of this launch (decode_tag())
  int32_t workgroups;      // that fill the GPU: one per compute unit
  int32_t one_round;       // slots that are one workgroup per compute unit
  DecodeMode mode;
  // Splits: partial results of one per (sequence, query head, split).
  int32_t splits;
  float* split_acc;        // [batch][q_heads][splits][head_dim]
  float* split_m;          // [batch][q_heads][splits]
  float* split_l;          // [batch][q_heads][splits]
  int32_t slots;           // >= batch; == batch: one slot per sequence, no partials
  int32_t hshift;          // log2 of the KV heads read by one workgroup
  int32_t batch, q_heads, kv_heads, head_dim, layers, layer, max_blocks;
  uint64_t half;           // bytes of one K or V plane of one block
  int64_t v_delta;         // V rows of a block relative to its K rows (bytes): half page-major
  int64_t vscale_delta;    // V scales relative to K scales (floats): one plane page-major
  float scale;             // log2(e) / sqrt(head_dim): scores in base 2
  int32_t id_max;          // largest valid block id (rows and scales inside the pools)
  FastDiv by_stride;       // block ids per page: 2 * layers page-major, 1 for per-layer pools
  FastDiv by_seg_pages;    // divides page indices by pages per segment
  // Append form (both set or both null): bf16 [batch][kv_heads][head_dim] K and V
  // of each sequence's new token, written at its last position before it is
  // read; the payload and scale pools above are then written as well.
  const uint16_t* new_k;
  const uint16_t* new_v;
  // Append form only: writable views of the payload bases and of the scale
  // pool (the same memory as kv.base and scales).
  char* wbase[kDecodeMaxSegments];
  float* wscales;
};

// Bytes of a workspace that holds the partials of `splits` slots per sequence.
uint64_t decode_workspace_bytes(int32_t batch, int32_t q_heads, int32_t head_dim, int32_t splits);

// Lays slots and splits out in `bytes` bytes at `workspace` (at least
// decode_workspace_bytes(.., splits) of them) and sets p.one_round .. p.hshift.
// `atomics`: whether the workspace takes device atomics, which the slots need.
void plan_decode_slots(DecodeParams* p, bool fp8, int32_t splits, void* workspace, uint64_t bytes, bool atomics);

hipError_t launch_paged_decode(const DecodeParams& p, bool fp8, hipStream_t stream);
hipError_t launch_paged_decode_splits(const DecodeParams& p, bool fp8, hipStream_t stream);

}  // namespace pbe
