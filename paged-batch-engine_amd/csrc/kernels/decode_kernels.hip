// Decode-side reader of handed-off KV pages: split-K paged attention for one
// query token per sequence, over the page-major arena (FP8 E4M3 planes with
// per-(token, head) scales, or BF16 planes). Same arithmetic as the
// reference's splitkv_paged_mha_fp8_stage1_kernel / _fast_stage1_kernel and
// splitkv_paged_mha_fast_stage2_kernel (paged_mha_fast_kernel.cu:391-800):
// score = (q . k) * (log2(e)/sqrt(D) * k_scale), online softmax in base 2,
// acc += v * (p * v_scale), output = acc / sum as BF16 (round to nearest even).
//
// gfx950 mapping. The batch's blocks of 16 tokens are cut into slots of about
// equal length, however long each sequence is (find_slot). A workgroup of 8
// waves takes one slot for one or two KV heads; the waves of a KV head take
// the slot's blocks in turn, and the KV heads of a block are read by
// neighbouring waves:
//  - loads: a key load instruction covers 64 contiguous bytes of each of the
//    16 rows (the MFMA wants one row per lane). A value load instruction
//    covers whole rows, i.e. full 128-byte lines, since the value tile is
//    rearranged in LDS anyway; requesting half lines instead costs 10% of
//    the BF16 step. Two register sets take turns: the next block is in flight
//    while one is computed. The queries lie in LDS, which keeps the wave at
//    128 registers or fewer, so that two workgroups share a compute unit.
//  - scores, transposed: one v_mfma_f32_16x16x32_bf16 per 32 head dims,
//    A = the block's 16 keys (rows), B = the query heads sharing the KV head
//    (columns, padded to 16). FP8 keys become BF16 exactly (an E4M3 value has
//    at most 3 mantissa bits). The contraction order over head dims follows
//    the load order, in A and B alike. Lane (g, j) ends with tokens 4g..4g+3
//    of query head j.
//  - softmax: per head in-lane, across the four lane groups with the gfx950
//    row swaps (v_permlane32_swap / v_permlane16_swap).
//  - values: the value tile goes through LDS once and comes back transposed
//    with ds_read_b64_tr_b8 / _b16, four tokens of one head dim per lane, as
//    the A operand of O^T += V^T P^T (P^T as held, split into a BF16 high and
//    low part, K = 32).
//  - results: the waves of a KV head are combined through LDS, and the slots
//    of a sequence by the workgroup that finishes last (tickets below), in
//    slot order, so the result does not depend on which one that is.
//
// What bounds it: large batches the HBM rate (64 sequences of 5,040 tokens,
// 2 KV heads x 128: FP8 36.3 us, 4.7 TB/s over the call), small ones the chain
// of dependent reads (arguments, lengths, block table, rows, partials, ticket,
// partials: 4 x 5,040 tokens, 2 x 64 BF16, 11.4 us). Two launches with an equal
// split count for every sequence take, in the same order, 37.5 and 11.1; 64
// sequences of mixed lengths up to 7,040 BF16 62.0 (here 40.2); a layer of 8
// mixed up to 16,384, 4 x 128 FP8, 29.0 (21.2). They remain in
// decode_split_kernels.hip for the calls they are the faster at: see
// decode_mode().
//
// Append variant (kAppend): the step's new token of every sequence, at its
// last position, is written into its page slot by the one wave that reads
// that block (per KV head only one wave reads a given row), with the page
// writer's arithmetic (scatter_kv_kernel.cu:128-216). The wave takes the row
// from its registers rather than from memory, so no ordering between the
// store and any load is needed, and the result equals writing the row first
// and reading the pages afterwards, byte for byte.
#include <algorithm>
#include <atomic>
#include <chrono>

#include "decode_device.h"

namespace pbe {
namespace {

constexpr int kStream = 0x02;  // buffer load policy: non-temporal

constexpr int kWavesLog = 3, kWaves = 1 << kWavesLog, kThreads = 64 * kWaves;  // of a workgroup
static_assert(kThreads * kDecodeMaxWorkgroups < (1ll << 32), "a launch has fewer than 2^32 threads");
// Slots of one sequence that one workgroup combines in one go; more of them
// are combined in two levels, groups of about the square root first.
constexpr int kCombineDirect = 64;
// A sequence of at most kWhole blocks stays whole; a longer one is cut into
// slots of at least min_chunk blocks (a row: one token of one KV head). us:
// 64 mixed up to 19 blocks, BF16 x 128, 9.8 whole against 11.0; 10 x 47 blocks
// of 256-byte rows 11.8 in slots of 8 against 13.1 of 16, 1 x 315 of 128-byte
// rows 12.0 against 11.3.
constexpr int kWhole = 24;
constexpr int min_chunk(int row_bytes) { return row_bytes >= 256 ? 8 : 16; }

// ---- which blocks a workgroup reads ---------------------------------------
template <int kCtrl, int kRows>
__device__ __forceinline__ int scan_step(int x) {
  return x + __builtin_amdgcn_update_dpp(0, x, kCtrl, kRows, 0xf, false);
}
// Inclusive prefix sum over the wave's lanes.
__device__ __forceinline__ int wave_scan(int x) {
  x = scan_step<0x111, 0xf>(x);  // row_shr 1, 2, 4, 8: within rows of 16
  x = scan_step<0x112, 0xf>(x);
  x = scan_step<0x114, 0xf>(x);
  x = scan_step<0x118, 0xf>(x);
  x = scan_step<0x142, 0xa>(x);     // row_bcast 15 into rows 1 and 3
  return scan_step<0x143, 0xc>(x);  // row_bcast 31 into rows 2 and 3
}
__device__ __forceinline__ int wave_total(int x) { return __builtin_amdgcn_readlane(wave_scan(x), 63); }
// Slots of a sequence of n blocks at c blocks per slot.
__device__ __forceinline__ int slots_of(int n, uint32_t c) {
  return n <= kWhole ? 1 : (int)(((uint32_t)n + c - 1) / c);
}

// One slot: a chunk of one sequence's blocks. The chunk length c is the same
// for the whole batch, so a batch of mixed lengths keeps every workgroup
// equally busy: a sequence of n blocks takes ceil(n / c) slots (one if n is at
// most kWhole), c being about the shortest (at least min_chunk) whose slots fit the slots of
// the launch. The lengths are device memory, so each workgroup works this out
// for itself: its waves try one c each, then find their slot with a prefix
// scan over the batch. (A binary search in every wave took 3.6 us of a batch
// of 160, 10 us with two workgroups per compute unit; this takes 1.6 and 3.)
//
// How many slots (W = the GPU's compute units / workgroups per slot; us on
// MI355X, 256 of them, 2 KV heads x 128 unless said otherwise):
//  - batch < W: W slots. Twice as many (two workgroups per compute unit) read
//    64 x 5,040 tokens in 65.0 against 57.7 (BF16), 39.2 against 37.8 (FP8):
//    the second set's slots start and end at the same time as the first's.
//    But for FP8, where W slots would leave a quarter of the chip idle (160
//    equal sequences: 160 slots), 2W: 160 x 2,000 tokens 41.4 against 45.7,
//    130 x 2,307 44.2 against 50.9. BF16 gains nothing: 130 x 2,307 80.5
//    against 79.8, 130 x 4,615 of 2 x 64 92.1 against 76.2. Equal lengths that
//    leave W slots idle are read in splits instead (decode_mode()); mixed ones
//    of that number take 34 against 49 and 56 here.
//  - batch >= W: a sequence is split only where it is longer than 5/4 of the
//    mean. FP8 256 x 1,000 equal lengths 30.5 against 36.6 with two slots
//    each, BF16 256 mixed up to 1,000 42.4 against 51.1 with W/2 more slots
//    than sequences. With the automatic split count BF16 has the slots for it
//    up to batch = W with two KV heads per workgroup, FP8 up to 2W; beyond, that
//    count is 1 and every sequence stays whole (mixed up to 7,000, 2 x 128 BF16:
//    256 86, 257 191; two launches 202 and 293) unless the caller asks for 2.
struct Slot {
  int b = -1;  // sequence; -1: no work for this workgroup
  int seq = 0;
  int k = 1, s = 0;  // the sequence's slots, and which of them this is
  int per = 1;       // blocks per slot
};

// `z`: this workgroup's slot; `slots` of the launch; `fit`: LDS.
template <int kMin>
__device__ __forceinline__ Slot find_slot(uint32_t (*fit)[kWaves], const int32_t* __restrict__ lens, int batch,
                                          int max_blocks, int slots, int one_round, int z, int w, int lane) {
  Slot r;
  if (slots == batch) {
    r.b = z;
    r.seq = lens[z];
    r.per = max(1, blocks_of(r.seq, max_blocks));
    return r;
  }
  // A lane's sequences are lane, lane + 64, ...; the first few stay in registers.
  constexpr int kKept = 4;
  int seqs[kKept], kept[kKept], sum = 0, most = 0;
#pragma unroll
  for (int i = 0; i < kKept; ++i) seqs[i] = lane + 64 * i < batch ? lens[lane + 64 * i] : 0;
#pragma unroll
  for (int i = 0; i < kKept; ++i) {
    kept[i] = blocks_of(seqs[i], max_blocks);
    sum += kept[i];
    most = max(most, kept[i]);
  }
  for (int i = lane + 64 * kKept; i < batch; i += 64) {
    const int n = blocks_of(lens[i], max_blocks);
    sum += n;
    most = max(most, n);
  }
  const uint32_t total = (uint32_t)wave_total(sum), longest = (uint32_t)wave_max_int(most);
  auto count = [&](uint32_t c) {
    int x = 0;
#pragma unroll
    for (int i = 0; i < kKept; ++i)
      if (64 * i < batch) x += lane + 64 * i < batch ? slots_of(kept[i], c) : 0;
    for (int i = lane + 64 * kKept; i < batch; i += 64) x += slots_of(blocks_of(lens[i], max_blocks), c);
    return wave_total(x);
  };
  const bool many = batch >= one_round;
  const uint32_t mean = many ? total / (uint32_t)batch : 0u;
  auto chunk = [&](uint32_t T, int round) {
    // sum of ceil(n/c) <= total/c + batch, so c >= total/(T - batch) fits
    const uint32_t extra = T - (uint32_t)batch;
    if (!many && (uint64_t)total <= (uint64_t)extra * kMin && longest <= (uint32_t)(kDecodeMaxSplits * kMin)) return (uint32_t)kMin;
    const uint32_t lo = max(max((total + T - 1) / T, (longest + kDecodeMaxSplits - 1) / kDecodeMaxSplits),
                            max(mean + mean / 4, (uint32_t)kMin));
    const uint32_t hi = max(lo, min(max(1u, longest), (total + extra - 1) / extra));
    if (lo == hi) return lo;
    const uint32_t c = lo + (uint32_t)((uint64_t)w * (hi - lo) / kWaves);
    const bool fits = count(c) <= (int)T;
    if (lane == 0) fit[round][w] = fits ? c : hi;
    __syncthreads();
    uint32_t best = hi;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) best = min(best, fit[round][i]);
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)best);
  };
  uint32_t c = 0;
  for (int round = 0; round < 2; ++round) {
    c = chunk((uint32_t)(many || round ? slots : min(slots, one_round)), round);
    const bool idle = !many && slots > one_round && c > (uint32_t)kMin &&
                      (uint64_t)total * 4 < (uint64_t)c * (uint32_t)one_round * 3;
    if (!idle) break;
  }
  // the sequence whose slots hold z; the other workgroups have nothing to do
  int before = 0;
  for (int i = 0; i < batch; i += 64) {
    int seq = seqs[0];
#pragma unroll
    for (int e = 1; e < kKept; ++e) seq = i == 64 * e ? seqs[e] : seq;
    if (i >= 64 * kKept) seq = i + lane < batch ? lens[i + lane] : 0;
    const int n = blocks_of(seq, max_blocks);
    const int k = i + lane < batch ? slots_of(n, c) : 0;
    const int upto = wave_scan(k) + before;
    const uint64_t past = __ballot(upto > z);
    if (past) {
      const int at = __builtin_ctzll(past);
      r.b = i + at;
      r.seq = __builtin_amdgcn_readlane(seq, at);
      r.k = __builtin_amdgcn_readlane(k, at);
      r.s = z - (__builtin_amdgcn_readlane(upto, at) - r.k);
      const int nb = __builtin_amdgcn_readlane(n, at);
      r.per = max(1, (nb + r.k - 1) / r.k);        // even slots ...
      r.k = slots_of(nb, (uint32_t)r.per);         // ... which may need fewer of them
      if (r.s >= r.k) r.b = -1;
      return r;
    }
    before = __builtin_amdgcn_readlane(upto, 63);
  }
  return r;
}

// ---- partial results between workgroups -----------------------------------
// A slot's partial (fp32 output, maximum and sum) is written and read at
// agent scope (relaxed atomics: written through, read past the XCD's own L2),
// so no L2 write-back or invalidate is needed: the writer waits for its
// stores to complete, then takes a ticket; whoever takes the last one reads.
constexpr int kAgent = 0x10;  // buffer access policy: agent scope

// Arrival tickets. A word holds tag << kTicketBits | arrivals of launch `tag`;
// anything else in it (a workspace may hold anything) counts as none. The last
// arrival leaves 0, so a replayed launch, which has the same tag, starts anew.
constexpr int kTicketBits = 11;
static_assert(kDecodeMaxSplits < (1 << kTicketBits), "arrivals fit the ticket");
// Makes a word that is 0 ready for arrivals; nothing waits for it.
__device__ __forceinline__ void open_ticket(gptr<uint64_t> word, uint64_t tag) {
  uint64_t none = 0;
  (void)__hip_atomic_compare_exchange_strong(word, &none, tag << kTicketBits, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
}
// Whether this is the last of `members` arrivals: one round trip where the
// word was opened; a word that held something else is claimed by exchange.
__device__ __forceinline__ bool last_arrival(gptr<uint64_t> word, uint64_t tag, uint32_t members) {
  uint64_t now = __hip_atomic_fetch_add(word, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
  if ((now >> kTicketBits) != tag) {
    uint64_t seen = now;
    do {
      now = (seen >> kTicketBits) == tag ? seen + 1 : (tag << kTicketBits) | 1u;
    } while (!__hip_atomic_compare_exchange_strong(word, &seen, now, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT));
  }
  if ((now & ((1u << kTicketBits) - 1)) != members) return false;
  __hip_atomic_store(word, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// One head's running combination of partials: maximum, sum and output, the
// latter two weighted by 2^(m_i - m) (paged_mha_fast_kernel.cu:730-799). A NaN
// sum stays NaN; a partial of weight 0 is left out whatever its output holds.
struct Combined {
  float m = -INFINITY, l = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  __device__ __forceinline__ void raise(float top) {  // to a maximum top >= m
    const float scale = l > 0.f ? __builtin_amdgcn_exp2f(m - top) : 0.f;
    l = l != l ? l : l * scale;
    acc = scale > 0.f ? acc * scale : f32x4{0.f, 0.f, 0.f, 0.f};
    m = top;
  }
  __device__ __forceinline__ void weigh(float m_i, float l_i, const f32x4& acc_i) {  // m_i <= m
    const float wt = l_i > 0.f ? __builtin_amdgcn_exp2f(m_i - m) : 0.f;
    l += l_i != l_i ? l_i : l_i * wt;
    if (wt > 0.f) acc += acc_i * wt;
  }
};

// ---- the kernel -------------------------------------------------------------
template <int D, bool kFp8, int KVM, bool kAppend>
__global__ __launch_bounds__(kThreads, 4) void paged_decode_kernel(
    const int32_t* __restrict__ lens, const int32_t* __restrict__ tables, const int batch, const int max_blocks, const int slots,
    const int hshift_mode, const uint32_t groups_d, const uint32_t groups_mul, const uint32_t groups_shift,
    const DecodeParams p) {
  using G = Geo<D, kFp8>;
  constexpr int E = G::E;
  constexpr int NK = D / 32;  // score MFMAs per block
  constexpr int NT = D / 16;  // value MFMAs (16 head dims each) per block
  constexpr int W = G::WORDS, PITCH = G::PITCH;
  constexpr int OUT_PITCH = D + 4;  // floats; the pad spreads the heads over the banks
  constexpr int kTile = kBlockTokens * PITCH, kOut = KVM * OUT_PITCH * 4;
  constexpr int kTeams = 64 * 24;  // what a wave's threads exchange when they share slots
  constexpr int kWaveLds = kTile > kOut ? (kTile > kTeams ? kTile : kTeams) : (kOut > kTeams ? kOut : kTeams);
  // value tiles while blocks are read, then the waves' outputs
  __shared__ __attribute__((aligned(16))) unsigned char lds[kWaves][kWaveLds];
  __shared__ float lds_m[kWaves][16], lds_l[kWaves][16];
  __shared__ int lds_last[2];
  __shared__ uint32_t fit[2][kWaves];
  __shared__ __attribute__((aligned(16))) unsigned char lds_new[kAppend ? kWaves : 1][kAppend ? 2 * D * E : 16];
  __shared__ bf16x8 lds_q[kWaves][NK][64];

  const int hshift = hshift_mode & 0xff;
  // The arguments that follow the first ones, read in one go: left to
  // itself the compiler reads each where it is used, one scalar round trip
  // after another.
  gptr<const char> kv0 = (gptr<const char>)p.kv.base[0];
  gptr<const float> scales = (gptr<const float>)p.scales;
  gptr<const uint16_t> q_rows = (gptr<const uint16_t>)p.q;
  gptr<uint16_t> out = (gptr<uint16_t>)p.out;
  gptr<float> part_acc = (gptr<float>)p.part_acc, part_ml = (gptr<float>)p.part_ml;
  gptr<uint64_t> tickets = (gptr<uint64_t>)p.tickets;
  uint64_t tag = p.tag, half = p.half;
  int64_t v_delta = p.v_delta, vscale_delta = p.vscale_delta;
  int q_heads = p.q_heads, layer = p.layer, id_max = p.id_max;
  float score_scale = p.scale;
  FastDiv by_stride = p.by_stride, by_seg_pages = p.by_seg_pages;
  asm volatile("" : "+s"(kv0), "+s"(q_rows), "+s"(out), "+s"(part_acc), "+s"(part_ml), "+s"(tickets), "+s"(tag), "+s"(half),
               "+s"(v_delta), "+s"(q_heads), "+s"(layer), "+s"(id_max), "+s"(score_scale), "+s"(by_stride.d),
               "+s"(by_stride.mul), "+s"(by_stride.shift), "+s"(by_seg_pages.d), "+s"(by_seg_pages.mul), "+s"(by_seg_pages.shift));
  if constexpr (kFp8) asm volatile("" : "+s"(scales), "+s"(vscale_delta));
  gptr<const uint16_t> new_k = nullptr, new_v = nullptr;
  gptr<char> kv0_w = nullptr;
  gptr<float> wscales = nullptr;
  if constexpr (kAppend) {
    new_k = (gptr<const uint16_t>)p.new_k, new_v = (gptr<const uint16_t>)p.new_v;
    kv0_w = (gptr<char>)p.wbase[0], wscales = (gptr<float>)p.wscales;
    asm volatile("" : "+s"(new_k), "+s"(new_v), "+s"(kv0_w), "+s"(wscales));
  }
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if ((hshift_mode >> 8) == (int)DecodeMode::kEither && alike(lens, batch, max_blocks, lane)) return;
  const int head_groups = (int)groups_d, kv_heads = head_groups << hshift;
  const int z = (int)fast_div(blockIdx.x, FastDiv{groups_d, groups_mul, groups_shift});
  const int hg = (int)blockIdx.x - z * head_groups;
  const Slot slot = find_slot<min_chunk(D * E)>(fit, lens, batch, max_blocks, slots, p.one_round, z, w, lane);
  if (slot.b < 0) return;
  const int b = slot.b, seq = slot.seq;
  // Of the workgroup's waves, every (1 << hshift)th reads the same KV head:
  // the KV heads of a token row are read together, by neighbouring waves.
  const int hw = 1 << hshift, sub_shift = kWavesLog - hshift, subs = 1 << sub_shift;
  const int hloc = w & (hw - 1), sub = w >> hshift;
  const int kvh = (hg << hshift) + hloc;
  const int g = lane >> 4, j = lane & 15;
  const int nblk = seq > 0 ? (int)(((uint32_t)seq + kBlockTokens - 1) / kBlockTokens) : 0;
  bool bad = seq < 0 || nblk > max_blocks;
  // The slot's blocks, dealt to the waves of a KV head in turn.
  const int chunk0 = slot.s * slot.per;
  const int blk0 = chunk0 + sub;
  int blk1 = bad ? chunk0 : min(chunk0 + slot.per, nblk);

  const uint64_t H = (uint64_t)kv_heads;
  const uint32_t token_stride = (uint32_t)(H * D * E);
  const uint64_t stride = by_stride.d;
  // The wave's next 64 block ids, one per lane (a vector load every 64 blocks
  // instead of a scalar round trip before each).
  gptr<const int32_t> table = (gptr<const int32_t>)tables + (int64_t)b * max_blocks;
  int32_t window = table[min(blk0 + (lane << sub_shift), max_blocks - 1)];
  const uint64_t head_off = 2ull * layer * half + (uint64_t)kvh * D * E;
  // Key load v of lane (g, j) reads bytes 64v + 16g.. of key row j: 64
  // contiguous bytes of every row per instruction. The key's head dims are
  // consumed in that order; the queries are read in the same order.
  const uint32_t key_off = (uint32_t)j * token_stride + (uint32_t)(16 * g);
  // Value load v of lane l reads the 16 bytes at column vcol of row
  // v * RPI + vrow0: each instruction covers RPI whole rows.
  constexpr int LPR = D * E / 16, RPI = 64 / LPR;  // lanes per row, rows per load
  constexpr int RL = D / 8;  // append: 16-byte BF16 input vectors per head row
  const int vrow0 = lane / LPR, vcol = 16 * (lane % LPR);
  const uint32_t val_off = (uint32_t)vrow0 * token_stride + (uint32_t)vcol;
  // lane (g, j): scale of token 4g + j%4 from the key (j%8 < 4) or value plane
  const int64_t scale_off =
      (int64_t)((2u * layer * kBlockTokens + 4u * g + (j & 3)) * H + kvh) + ((j >> 2) & 1 ? vscale_delta : 0);
  const uint32_t row_span = (uint32_t)(half - (uint64_t)kvh * D * E);  // this head's rows, to the plane's end
  // Loads block `blk` into `r`. Every call issues the same loads (an
  // unconditional count keeps the compiler's in-flight accounting exact), but
  // a block past the split's end, or whose id is not a page id inside the
  // arena and scale pool, is an empty buffer: its row loads return zeros and
  // read no memory (the scale load reads a row of block 0). Reports false
  // when such a bad block was wanted.
  auto load = [&](int blk, BlockRegs<W, kFp8>& r) -> bool {
    const bool want = blk < blk1;
    const int at = (blk - blk0) >> sub_shift;
    if (at && (at & 63) == 0) window = table[min(blk + (lane << sub_shift), max_blocks - 1)];
    int32_t id = want ? __builtin_amdgcn_readlane(window, at & 63) : 0;
    uint32_t page = fast_div((uint32_t)max(id, 0), by_stride);
    const bool ok = id >= 0 && id <= id_max && page * by_stride.d == (uint32_t)id;
    if (!ok) id = 0, page = 0;
    const uint32_t seg = fast_div(page, by_seg_pages);
    gptr<const char> kplane =
        (seg ? (gptr<const char>)p.kv.base[seg] : kv0) + (uint64_t)(page - seg * by_seg_pages.d) * stride * half + head_off;
    const uint32_t span = want && ok ? row_span : 0u;
    const __amdgpu_buffer_rsrc_t rk =
        __builtin_amdgcn_make_buffer_rsrc((void*)kplane, (short)0, span, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv =
        __builtin_amdgcn_make_buffer_rsrc((void*)(kplane + v_delta), (short)0, span, 0x00020000);
    uint32_t val_step = RPI * token_stride;
    asm volatile("" : "+s"(val_step));  // added per block: the offsets would take W/4 registers
#pragma unroll
    for (int v = 0; v < W / 4; ++v) {
      const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(rk, key_off + 64 * v, 0, kStream);
      const u32x4 y = __builtin_amdgcn_raw_buffer_load_b128(rv, val_off + (uint32_t)v * val_step, 0, kStream);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        r.k[4 * v + e] = x[e];
        r.v[4 * v + e] = y[e];
      }
    }
    if constexpr (kFp8) {  // key scales carry the score scale: score_scale * k_scale
      // Non-temporal like the page rows: plain loads cost 8% of the FP8 step.
      const float sc = __builtin_nontemporal_load(scales + (uint64_t)id * kBlockTokens * H + scale_off);
      r.scale = (j & 4) ? sc : score_scale * sc;
    }
    return ok || !want;
  };

  // Slots of one sequence are combined in groups, and the groups after them.
  int group = slot.k, groups = 1, gi = 0;
  if (slot.k > kCombineDirect) {
    group = 8;
    while (group * group < slot.k) group += 4;
    groups = (slot.k + group - 1) / group;
    gi = slot.s / group;
  }
  const int z0 = z - slot.s;  // the sequence's first slot
  const int zg = z0 + gi * group, in_group = min(group, slot.k - gi * group);
  float m = -INFINITY, l = 0.f;  // of head j
  f32x4 acc[NT];                 // O^T: lane (g, j) = head j, dims 16nt + 4g + 0..3
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Append: the new token's row of this KV head lies in lds_new (keys, then
  // values); its scales, and the block it lands in (-1: nothing to write here).
  float nks = 0.f, nvs = 0.f;
  int patch_blk = -1, slot_row = 0;

  unsigned char* vt_w = &lds[w][0];
  auto compute = [&](int blk, const BlockRegs<W, kFp8>& r) {
    const int valid = blk == nblk - 1 ? seq - kBlockTokens * (nblk - 1) : kBlockTokens;
    const bool patch = kAppend && blk == patch_blk;
    // Value tile -> LDS rows (tail rows zeroed: tail slots may hold anything, even NaN).
    {
      unsigned char* dst = vt_w + vrow0 * PITCH + vcol;
#pragma unroll
      for (int v = 0; v < W / 4; ++v) {
        const u32x4 x = vrow0 < valid - v * RPI
                            ? u32x4{r.v[4 * v], r.v[4 * v + 1], r.v[4 * v + 2], r.v[4 * v + 3]}
                            : u32x4{0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4*>(dst + v * RPI * PITCH) = x;
      }
      // The new row replaces what was read (LDS writes of one wave land in
      // issue order).
      if constexpr (kAppend) {
        if (patch && lane >= 32 && (lane & 31) < RL) {
          const int at = (kFp8 ? 8 : 16) * (lane & 31);
          unsigned char* row = vt_w + slot_row * PITCH + at;
          const unsigned char* from = lds_new[w] + D * E + at;
          if constexpr (kFp8) *reinterpret_cast<u32x2*>(row) = *reinterpret_cast<const u32x2*>(from);
          else *reinterpret_cast<u32x4*>(row) = *reinterpret_cast<const u32x4*>(from);
        }
      }
    }
    // Scores, transposed: lane (g, j) gets tokens 4g..4g+3 of head j.
    uint32_t kw[W];
#pragma unroll
    for (int i = 0; i < W; ++i) kw[i] = r.k[i];
    float rscale = kFp8 ? r.scale : 0.f;
    if constexpr (kAppend) {
      if (patch) {
        if (j == slot_row) {
#pragma unroll
          for (int v = 0; v < W / 4; ++v) {
            const u32x4 x = *reinterpret_cast<const u32x4*>(lds_new[w] + 64 * v + 16 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) kw[4 * v + e] = x[e];
          }
        }
        if (4 * g + (j & 3) == slot_row) rscale = (j & 4) ? nvs : score_scale * nks;
      }
    }
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      bf16x8 kb;
      if constexpr (kFp8) {
        const u32x2 lo = e4m3x4_to_bf16x4_cvt(kw[2 * kk]);
        const u32x2 hi = e4m3x4_to_bf16x4_cvt(kw[2 * kk + 1]);
        kb = __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
      } else {
        kb = __builtin_bit_cast(bf16x8, u32x4{kw[4 * kk], kw[4 * kk + 1], kw[4 * kk + 2], kw[4 * kk + 3]});
      }
      s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb, lds_q[w][kk][lane], s, 0, 0, 0);
    }
    wave_sync();
    float ks[4] = {score_scale, score_scale, score_scale, score_scale}, vs[4] = {1.f, 1.f, 1.f, 1.f};
    if constexpr (kFp8) {  // broadcast within each 16-lane row
      ks[0] = dpp<0x150>(rscale);
      ks[1] = dpp<0x151>(rscale);
      ks[2] = dpp<0x152>(rscale);
      ks[3] = dpp<0x153>(rscale);
      vs[0] = dpp<0x154>(rscale);
      vs[1] = dpp<0x155>(rscale);
      vs[2] = dpp<0x156>(rscale);
      vs[3] = dpp<0x157>(rscale);
    }
    // Online softmax of head j over the block's 16 tokens.
    float sv[4], tmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sv[i] = 4 * g < valid - i ? s[i] * ks[i] : -INFINITY;
      tmax = fmaxf(tmax, sv[i]);
    }
    tmax = group_max4(tmax);
    const float mn = fmaxf(m, tmax);
    const float alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mn);
    float psum = 0.f;
    uint32_t phi[2], plo[2];
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      const bool ok0 = 4 * g < valid - i, ok1 = 4 * g < valid - i - 1;
      const float p0 = ok0 ? __builtin_amdgcn_exp2f(sv[i] - mn) : 0.f;
      const float p1 = ok1 ? __builtin_amdgcn_exp2f(sv[i + 1] - mn) : 0.f;
      psum += p0 + p1;
      // p * v_scale as a bf16 hi + bf16 lo pair by truncation: hi keeps the
      // top 8 significant bits, lo the next 8 of the exact remainder, so the
      // pair is within 2^-15 of the fp32 product.
      const float a0 = ok0 ? p0 * vs[i] : 0.f, a1 = ok1 ? p1 * vs[i + 1] : 0.f;
      const uint32_t h0 = __float_as_uint(a0) & 0xffff0000u, h1 = __float_as_uint(a1) & 0xffff0000u;
      const uint32_t l0 = __float_as_uint(a0 - __uint_as_float(h0)) & 0xffff0000u;
      const uint32_t l1 = __float_as_uint(a1 - __uint_as_float(h1)) & 0xffff0000u;
      phi[i / 2] = (h0 >> 16) | h1;
      plo[i / 2] = (l0 >> 16) | l1;
    }
    psum = group_sum4(psum);
    l = l * alpha + psum;
    m = mn;
    const bf16x8 pb = __builtin_bit_cast(bf16x8, u32x4{phi[0], phi[1], plo[0], plo[1]});
    // Rescale: the accumulators hold O^T, lane (g, j) = head j, so alpha is
    // in-lane; skipped when no head's maximum moved (the common case).
    if (__ballot(alpha != 1.f) != 0) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[nt][i] *= alpha;
    }
    // O^T += V^T P^T: A = value rows 4g..4g+3 at head dim 16nt + j, B = P^T as held.
    // Transposing LDS reads: lane (g, j) gets tokens 4g..4g+3 of head dim
    // 16nt + j. ds_read_b64_tr_b8 hands lane i of a 16-lane group byte e of
    // the row addressed by lane 2e + i/8 (at byte i%8); tr_b16 hands it
    // element e of the row addressed by lane 4e + i/4 (at element i%4).
    const unsigned char* vt;
    if constexpr (kFp8) vt = vt_w + (4 * g + ((j >> 1) & 3)) * PITCH + 8 * (j & 1);
    else vt = vt_w + (4 * g + (j >> 2)) * PITCH + 8 * (j & 3);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      u32x2 vw;
      if constexpr (kFp8) {
        typedef int i32x2 __attribute__((ext_vector_type(2)));
        const i32x2 t = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
            (__attribute__((address_space(3))) i32x2*)(vt + 16 * nt));
        vw = e4m3x4_to_bf16x4_cvt((uint32_t)t[0]);
      } else {
        const s16x4 t = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(vt + 32 * nt));
        vw = __builtin_bit_cast(u32x2, t);
      }
      // K = 32: the four tokens twice, against p_hi then p_lo.
      acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, u32x4{vw[0], vw[1], vw[0], vw[1]}),
                                                         pb, acc[nt], 0, 0, 0);
    }
    wave_sync();  // the next block rewrites the tile
  };

  // Append: the wave that reads the sequence's last block takes the new token's
  // row, lanes 0..RL-1 of the keys and lanes 32..32+RL-1 of the values.
  const int last = nblk - 1;
  const bool writer = kAppend && !bad && seq > 0 && last >= chunk0 && last < chunk0 + slot.per && ((last - chunk0) & (subs - 1)) == sub;
  const bool is_v = lane >= 32, act = (lane & 31) < RL;
  u32x4 row_in = {0u, 0u, 0u, 0u};
  if constexpr (kAppend) {
    if (writer && act)
      row_in = __builtin_nontemporal_load((gptr<const u32x4>)((is_v ? new_v : new_k) + ((int64_t)b * kv_heads + kvh) * D + 8 * (lane & 31)));
  }
  // Query rows as the B operand of the scores: lane (g, j) holds head j's
  // dims matching the key bytes MFMA kk consumes (rows past the group's
  // heads are zero).
  u32x4 q_in[NK];
  {
    const bool has = j < KVM;
    gptr<const uint16_t> qrow = q_rows + ((int64_t)b * q_heads + (int64_t)kvh * KVM + (has ? j : 0)) * D;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      // the head dims of the key bytes this MFMA consumes (see key_off)
      const int cb = kk * 8 * E;
      const int dim0 = (64 / E) * (cb / 16) + (16 / E) * g + (cb % 16) / E;
      q_in[kk] = *(gptr<const u32x4>)(qrow + dim0);
    }
  }
  // Two register sets in turn: while one block is computed, the next is in flight.
  BlockRegs<W, kFp8> r[2];
  auto fetch = [&](int blk, BlockRegs<W, kFp8>& rr) {
    if (!load(blk, rr)) bad = true, blk1 = min(blk1, blk);
  };
  fetch(blk0, r[0]);
  fetch(blk0 + subs, r[1]);
#pragma unroll
  for (int kk = 0; kk < NK; ++kk) lds_q[w][kk][lane] = __builtin_bit_cast(bf16x8, j < KVM ? q_in[kk] : u32x4{0u, 0u, 0u, 0u});
  if (slot.k > 1 && threadIdx.x == 0) {
    open_ticket(tickets + (int64_t)zg * head_groups + hg, tag);
    if (groups > 1) open_ticket(tickets + (int64_t)(z0 + 1) * head_groups + hg, tag);
  }
  if constexpr (kAppend) {
    // It writes the row (while its first blocks are in flight) as the page
    // writer does with D/8 lanes per head.
    if (writer) {
      const int at = (last - blk0) >> sub_shift;
      const int32_t id = at < 64 ? __builtin_amdgcn_readlane(window, at) : table[last];
      const uint32_t page = fast_div((uint32_t)max(id, 0), by_stride);
      if (id >= 0 && id <= id_max && page * by_stride.d == (uint32_t)id) {
        const int row = seq - 1 - kBlockTokens * last;
        const uint32_t seg = fast_div(page, by_seg_pages);
        gptr<char> krow = (seg ? (gptr<char>)p.wbase[seg] : kv0_w) + (uint64_t)(page - seg * by_seg_pages.d) * stride * half +
                          head_off + (uint64_t)row * token_stride;
        const int li = lane & 31;
        const u32x4 x = row_in;
        gptr<char> dst = krow + (is_v ? v_delta : 0);
        if constexpr (kFp8) {
          const float mx = group_max<RL>(amax8(x));
          const float inv = mx > 0.f ? 448.f / mx : 0.f;
          const float sc = mx > 0.f ? mx / 448.f : 1.f;
          const u32x2 c = quantise8(x, inv);
          if (act) *(gptr<u32x2>)(dst + 8 * li) = c;
          if (act && li == 0)
            wscales[(uint64_t)id * kBlockTokens * H +
                                         (2u * layer * kBlockTokens + row) * H + kvh + (is_v ? vscale_delta : 0)] = sc;
          nks = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sc), 0));
          nvs = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sc), 32));
          if (act) *reinterpret_cast<u32x2*>(lds_new[w] + (is_v ? D * E : 0) + 8 * li) = c;
        } else {
          if (act) *(gptr<u32x4>)(dst + 16 * li) = x;
          if (act) *reinterpret_cast<u32x4*>(lds_new[w] + (is_v ? D * E : 0) + 16 * li) = x;
        }
        patch_blk = last;
        slot_row = row;
        wave_sync();
      }
    }
  }
  for (int blk = blk0; blk < blk1; blk += 2 * subs) {
    compute(blk, r[0]);
    fetch(blk + 2 * subs, r[0]);
    if (blk + subs < blk1) compute(blk + subs, r[1]);
    fetch(blk + 3 * subs, r[1]);
  }

  // ---- the waves of a KV head into one partial (lane (g, j): head j, dims 16nt + 4g + i)
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));  // lane numbers anew: kept over the loop they cost registers
  const int tg = (t & 63) >> 4, tj = t & 15;
  if (tg == 0) {
    lds_m[w][tj] = m;
    lds_l[w][tj] = bad ? __builtin_nanf("") : l;
  }
  if (tj < KVM) {
    float* dst = reinterpret_cast<float*>(&lds[w][0]) + tj * OUT_PITCH + 4 * tg;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) *reinterpret_cast<f32x4*>(dst + 16 * nt) = acc[nt];
  }
  __syncthreads();
  // From here on a thread holds four dims of one head; where the workgroup has
  // threads to spare, `teams` of them share the slots that are read back.
  constexpr int COLS = D / 4, kUnits = KVM * COLS;  // of one KV head
  static_assert(2 * kUnits <= kThreads, "one unit per thread");
  const int units = hshift ? 2 * kUnits : kUnits;
  const int teams = hshift ? kThreads / (2 * kUnits) : kThreads / kUnits;
  const int team = hshift ? t / (2 * kUnits) : t / kUnits, unit = t - team * units;
  const int rh = unit / kUnits, rj = unit / COLS - rh * KVM, col = unit % COLS;  // KV head, query head of it, float4 column
  const int64_t head = ((int64_t)(hg << hshift) + rh) * KVM + rj;
  Combined c;
  if (team == 0) {
    // the waves of KV head rh: rh, rh + hw, ...
    constexpr int kHalf = kWaves / 2;
    float mi[kWaves], li[kWaves];
    f32x4 x[kWaves];
    auto read = [&](int n) {
      const int i = rh + (n << hshift);
      mi[n] = lds_m[i][rj];
      li[n] = lds_l[i][rj];
      x[n] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(&lds[i][0]) + rj * OUT_PITCH + 4 * col);
    };
    auto fold = [&](int first) {
      float top = c.m;
#pragma unroll
      for (int n = 0; n < kHalf; ++n) top = fmaxf(top, mi[first + n]);
      c.raise(top);
#pragma unroll
      for (int n = 0; n < kHalf; ++n) c.weigh(mi[first + n], li[first + n], x[first + n]);
    };
#pragma unroll
    for (int n = 0; n < kHalf; ++n) read(n);
    if (!hshift) {
#pragma unroll
      for (int n = kHalf; n < kWaves; ++n) read(n);
      fold(kHalf);
    }
    fold(0);
  }
  if (slot.k > 1) {
    // The sequence's partials; offsets from its first slot fit 31 bits.
    const uint32_t acc_pitch = (uint32_t)q_heads * D * 4, ml_pitch = (uint32_t)q_heads * 8;
    const __amdgpu_buffer_rsrc_t r_acc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(part_acc + (int64_t)z0 * q_heads * D), (short)0, (uint32_t)slot.k * acc_pitch, 0x00020000);
    const __amdgpu_buffer_rsrc_t r_ml = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(part_ml + (int64_t)z0 * q_heads * 2), (short)0, (uint32_t)slot.k * ml_pitch, 0x00020000);
    const uint32_t acc_at = (uint32_t)head * (D * 4) + 16 * col, ml_at = (uint32_t)head * 8;
    auto put = [&](int s) {
      if (team != 0) return;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, c.acc), r_acc, acc_at + s * acc_pitch, 0, kAgent);
      if (col == 0) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f32x2{c.m, c.l}), r_ml, ml_at + s * ml_pitch, 0, kAgent);
    };
    // Publishes this workgroup's partial; true in the last of `members`.
    auto arrive = [&](int z, int members, int level) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's partial stores have completed
      __syncthreads();
      if (t == 0) lds_last[level] = last_arrival(tickets + (int64_t)z * head_groups + hg, tag, (uint32_t)members);
      __syncthreads();
      return __builtin_amdgcn_readfirstlane(lds_last[level]) != 0;
    };
    // c = slots s, s + step, ... (`members` of them) combined, eight in flight per thread.
    auto take = [&](int s, int step, int members) {
      c = Combined{};
      if (team < teams) {
        for (int i0 = team; i0 < members; i0 += 8 * teams) {
          f32x2 q[8];
          f32x4 x[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {  // past the end: nothing read, weight 0
            const int at = i0 + i * teams;
            const uint32_t from = at < members ? (uint32_t)(s + at * step) : (uint32_t)slot.k;
            q[i] = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r_ml, ml_at + from * ml_pitch, 0, kAgent));
            x[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r_acc, acc_at + from * acc_pitch, 0, kAgent));
          }
          float top = c.m;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            if (i0 + i * teams >= members) q[i][0] = -INFINITY;
            top = fmaxf(top, q[i][0]);
          }
          c.raise(top);
#pragma unroll
          for (int i = 0; i < 8; ++i) c.weigh(q[i][0], q[i][1], x[i]);
        }
      }
      if (teams > 1) {
        f32x4* team_acc = reinterpret_cast<f32x4*>(&lds[0][0]);
        f32x2* team_ml = reinterpret_cast<f32x2*>(team_acc + kThreads);
        team_acc[t] = c.acc;
        team_ml[t] = f32x2{c.m, c.l};
        __syncthreads();
        if (team == 0) {
          float top = c.m;
          for (int i = 1; i < teams; ++i) top = fmaxf(top, team_ml[t + i * units][0]);
          c.raise(top);
          for (int i = 1; i < teams; ++i) {
            const f32x2 q = team_ml[t + i * units];
            c.weigh(q[0], q[1], team_acc[t + i * units]);
          }
        }
      }
    };
    put(slot.s);
    if (!arrive(zg, in_group, 0)) return;
    take(gi * group, 1, in_group);
    if (groups > 1) {
      put(gi * group);
      if (!arrive(z0 + 1, groups, 1)) return;
      take(0, group, groups);
    }
  }
  if (team != 0) return;
  uint16_t o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = to_bf16(c.l != c.l ? __builtin_nanf("") : (c.l > 0.f ? c.acc[e] / c.l : 0.f));
  *(gptr<u32x2>)(out + ((int64_t)b * q_heads + head) * D + 4 * col) = u32x2{o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16};
}

template <int D, bool kFp8, int KVM>
void launch(const DecodeParams& p, hipStream_t stream) {
  const FastDiv by_groups = make_fast_div((uint32_t)(p.kv_heads >> p.hshift));
  const dim3 grid((unsigned)(p.slots * (p.kv_heads >> p.hshift))), block(kThreads);
  if (p.new_k)
    hipLaunchKernelGGL((paged_decode_kernel<D, kFp8, KVM, true>), grid, block, 0, stream, p.seq_lens, p.tables, p.batch, p.max_blocks, p.slots, p.hshift | (int)p.mode << 8, by_groups.d, by_groups.mul, by_groups.shift, p);
  else
    hipLaunchKernelGGL((paged_decode_kernel<D, kFp8, KVM, false>), grid, block, 0, stream, p.seq_lens, p.tables, p.batch, p.max_blocks, p.slots, p.hshift | (int)p.mode << 8, by_groups.d, by_groups.mul, by_groups.shift, p);
}

template <int D, bool kFp8>
bool launch_kvm(const DecodeParams& p, hipStream_t stream) {
  switch (p.q_heads / p.kv_heads) {
    case 1: launch<D, kFp8, 1>(p, stream); return true;
    case 2: launch<D, kFp8, 2>(p, stream); return true;
    case 3: launch<D, kFp8, 3>(p, stream); return true;
    case 4: launch<D, kFp8, 4>(p, stream); return true;
    case 5: launch<D, kFp8, 5>(p, stream); return true;
    case 6: launch<D, kFp8, 6>(p, stream); return true;
    case 7: launch<D, kFp8, 7>(p, stream); return true;
    case 8: launch<D, kFp8, 8>(p, stream); return true;
    default: return false;
  }
}

}  // namespace

FastDiv make_fast_div(uint32_t d) {
  FastDiv f;
  f.d = d ? d : 1;
  uint32_t s = 0;
  while ((1ull << s) < f.d) ++s;
  f.shift = s;
  f.mul = (uint32_t)(((1ull << 32) * ((1ull << s) - f.d)) / f.d + 1);
  return f;
}

uint64_t decode_workspace_bytes(int32_t batch, int32_t q_heads, int32_t head_dim, int32_t splits) {
  const uint64_t rows = (uint64_t)batch * q_heads * splits;
  return rows * head_dim * 4ull + 2ull * rows * 4ull;
}

namespace {
// A launch's tag in the arrival tickets: never the same twice in a process,
// and a word no float, code or id pattern makes (all twelve top bits set). The
// clock keeps processes apart, and unlike a random device it cannot throw.
uint64_t decode_tag() {
  static std::atomic<uint64_t> next{(uint64_t)std::chrono::steady_clock::now().time_since_epoch().count() * 0x9e3779b97f4a7c15ull};
  return 0xfffull << 41 | (next.fetch_add(1, std::memory_order_relaxed) & ((1ull << 41) - 1));
}
}  // namespace

namespace {
// How the batch is read; `slots` of one_round are one workgroup per compute
// unit. us on MI355X, the whole call, two launches against one:
//  - Few sequences: one launch combines a sequence's slots in one workgroup per
//    KV head, the second launch in up to 32. 1 x 16,384 tokens 2 x 128 BF16
//    14.2 and 17.2, 1 x 9,000 12.9 and 15.7, 2 x 5,040 12.9 and 13.9, 4 x 2,000
//    of 8 x 128 FP8 12.7 and 14.0; up to 160 blocks of less than 8 x 128 the
//    other way round, 2 x 2,000 12.4 and 11.7.
//  - Small batches of 64-dim heads, where finding the slot counts: 16 x 1,000
//    tokens 2 x 64 10.7 and 11.3, 8 x 2,000 10.9 and 11.3; 4 x 5,040 11.1 and
//    11.4, mixed 11.0 and 10.8.
//  - 64-byte rows that head_pairs() cannot or does not join: 32 x 4,000 of 5 x
//    64 32.3 and 41.6 (mixed 25.7 and 27.9), of 3 x 64 23.9 and 30.9 (20.1 and
//    20.0), 16 x 4,000 of 16 x 64 47.3 and 57.8 (42.8 and 48.0).
//  - Equal lengths whose whole slots leave compute units idle: 130 x 2,000 2 x
//    128 BF16 55 and 70, 153 x 2,000 62 and 80, 65 x 4,500 of 4 x 128 117 and
//    167, FP8 66 and 80; or of many or an odd number of KV heads, whose rows
//    the two launches read whole: 48 x 4,000 of 8 x 128 FP8 92 and 106, 64 x
//    3,000 of 5 x 128 57 and 75. Mixed lengths are the reverse (130 mixed up to
//    7,000 131 and 36), so there the kernels look at them; the launches that
//    find nothing to do cost about 3 us.
DecodeMode decode_mode(const DecodeParams& p, bool fp8, int32_t splits, int64_t one_round, bool atomics) {
  if (splits <= 1) return DecodeMode::kSlots;
  if (!atomics) return DecodeMode::kSplits;
  if (p.max_blocks <= kWhole) return DecodeMode::kSlots;
  const int64_t batch = p.batch, blocks = batch * p.max_blocks, rows = blocks * p.kv_heads;
  const bool odd = p.kv_heads % 2 && p.kv_heads >= 3;
  const bool few = batch <= 2 || batch * p.kv_heads <= 3;
  if (p.kv_heads >= 8 ? few || rows <= 4096 : p.head_dim == 64 ? few || blocks <= 1100 : few && p.max_blocks > 160) return DecodeMode::kSplits;
  const int64_t out_rows = batch * p.q_heads;  // each costs the combining launch a workgroup
  if (fp8 && p.head_dim == 64 && (odd || p.kv_heads >= 16) && out_rows * splits <= 1 << 26) return DecodeMode::kSplits;
  if (odd && rows >= 100ll * p.workgroups && batch < 2 * one_round && out_rows <= 2048) return DecodeMode::kEither;
  if (batch >= one_round || out_rows > 3072) return DecodeMode::kSlots;
  if (rows >= 64ll * p.workgroups) {
    // Of the launch's slots those that equal lengths would use, in percent. The
    // line, at 2,000 tokens each, two launches, one, and both as they look at
    // the lengths: BF16 2 x 128 87 (two slots each, 67%) 38.4, 42.2, 41.5; 66
    // (three, 77%) 30.6, 32.4, 33.5; 179 (one, 70%, and no more than two splits)
    // 82, 79; 2 x 64 130 (51%) 36.3, 41.4, 39.4, 168 (66%) 37.1, 38.6. FP8 4 x
    // 128 65 (three, 76%) 36.4, 42.6, 39.6; 89 (two, 70%) 47, 56, 50.7; 96 (75%)
    // 48.5, 49.2, 52.3.
    const int64_t used = fp8 ? 2 * one_round : one_round, each = used / batch, full = 100 * each * batch / used;
    const bool idle = p.head_dim == 64 ? !fp8 && each == 1 && full < 66
                      : fp8            ? full < (each == 3 ? 78 : 72) && each <= 3
                                       : full < 79 && each <= 2 && splits >= each + 2;
    if (idle) return DecodeMode::kEither;
  }
  return p.kv_heads >= 8 && rows >= 180ll * p.workgroups ? DecodeMode::kEither : DecodeMode::kSlots;
}

// Two KV heads per workgroup read whole 256-byte (FP8) or 512-byte pieces of
// a token's row; one per workgroup gives twice the workgroups, which is
// better where one per slot would leave the chip idle. MI355X, us: 8 x 5,040
// BF16 14.5 against 19.9, 64 mixed up to 300 tokens 11.1 against 12.6; 64
// mixed up to 7,040 51.1 (one head) against 41.9. In small batches it needs
// more blocks per workgroup the fewer of a token's bytes lie beside the
// head's: 4 x 128 BF16 16 x 9,000 55.9 against 61.8 (mixed 33.0 against 35.4),
// 8 x 4,000 mixed 17.1 against 15.3; FP8 16 x 9,000 36.7 against 40.1, 8 x
// 16,000 mixed 24.3 against 23.2; 8 x 128 8 x 4,000 FP8 24.3 against 28.2; 2 x
// 64 FP8 16 x 9,000 18.7 against 22.5.
bool head_pairs(const DecodeParams& p, bool fp8, int64_t most) {
  if (p.kv_heads % 2 || most * p.kv_heads <= p.workgroups) return false;
  if (p.batch > 16) return true;
  const int64_t each = (int64_t)p.batch * p.max_blocks * p.kv_heads / p.workgroups;  // blocks of one head per workgroup
  if (p.head_dim * (fp8 ? 1 : 2) == 64 && p.kv_heads < 8) return p.batch >= 4 && each >= 64;
  if (p.kv_heads >= 8) return each >= (fp8 ? 20 : p.batch <= 8 ? 16 : 36);
  if (p.kv_heads >= 4) return each >= (p.batch >= 12 ? (fp8 ? 48 : 32) : p.batch >= 6 ? (fp8 ? 192 : 64) : fp8 ? INT32_MAX : 120);
  return p.head_dim == 128 && !fp8 && p.batch >= 12 && each >= 110;
}
}  // namespace

void plan_decode_slots(DecodeParams* p, bool fp8, int32_t splits, void* workspace, uint64_t bytes, bool atomics) {
  const int64_t batch = p->batch;
  const int row_bytes = p->head_dim * (fp8 ? 1 : 2), chunk = min_chunk(row_bytes);
  const int64_t most = p->max_blocks <= kWhole ? batch : batch * ((p->max_blocks + chunk - 1) / chunk);  // slots that could hold work
  p->hshift = head_pairs(*p, fp8, most) ? 1 : 0;
  const int64_t groups = p->kv_heads >> p->hshift;
  const uintptr_t base = (reinterpret_cast<uintptr_t>(workspace) + 15) & ~(uintptr_t)15;
  const uint64_t pad = base - reinterpret_cast<uintptr_t>(workspace);
  const uint64_t slot_bytes = (uint64_t)p->q_heads * (p->head_dim + 2) * 4 + (uint64_t)groups * 8;
  int64_t slots = (int64_t)((bytes - std::min(bytes, pad)) / slot_bytes);
  // see find_slot
  const int64_t one_round = std::max<int64_t>(1, p->workgroups / groups);
  p->one_round = (int32_t)one_round;
  p->mode = decode_mode(*p, fp8, splits, one_round, atomics);
  const bool twice = batch >= one_round || (fp8 && batch * 8 > one_round);
  slots = std::min(slots, twice ? 2 * std::max(batch, one_round) : one_round);
  slots = std::min(slots, most);
  // One slot per sequence: nothing to combine. Block totals are 32-bit sums,
  // and a sequence's partials are addressed with 31 bits.
  if (splits <= 1 || slots <= batch || batch * p->max_blocks > 0x7fffffff ||
      (int64_t)p->q_heads * p->head_dim * 4 * kDecodeMaxSplits > 0x7fffffff)
    slots = batch;
  p->slots = (int32_t)slots;
  p->tag = decode_tag();
  p->part_acc = reinterpret_cast<float*>(base);
  p->part_ml = p->part_acc + (uint64_t)slots * p->q_heads * p->head_dim;
  p->tickets = reinterpret_cast<uint64_t*>(p->part_ml + (uint64_t)slots * p->q_heads * 2);
  p->splits = splits;
  p->split_acc = static_cast<float*>(workspace);
  p->split_m = p->split_acc + (uint64_t)batch * p->q_heads * splits * p->head_dim;
  p->split_l = p->split_m + (uint64_t)batch * p->q_heads * splits;
}

hipError_t launch_paged_decode(const DecodeParams& p, bool fp8, hipStream_t stream) {
  if (p.mode != DecodeMode::kSlots) {
    const hipError_t e = launch_paged_decode_splits(p, fp8, stream);
    if (e != hipSuccess || p.mode == DecodeMode::kSplits) return e;
  }
  bool ok = false;
  if (p.head_dim == 128) ok = fp8 ? launch_kvm<128, true>(p, stream) : launch_kvm<128, false>(p, stream);
  else if (p.head_dim == 64) ok = fp8 ? launch_kvm<64, true>(p, stream) : launch_kvm<64, false>(p, stream);
  if (!ok) return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace pbe
