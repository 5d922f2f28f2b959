// Launch interface of the fused decode-attention kernels (attn_decode.hip).
#pragma once

#include "nv_common.cuh"

namespace nv {

constexpr uint32_t kKvBlockTokens = 16;   // tokens per paged KV block (types.cuh:64)
constexpr uint32_t kAttnMaxSplits = 64;   // split-KV partials per kv head

// KV cache layout (library-owned): [layer][physical block][kv_head][tile of 16 tokens x head_dim]
// 16-bit, K and V in separate arrays. One (block, kv_head) tile is contiguous
// (4 KiB at head_dim 128), so a wave streams it with four 1 KiB load instructions.
// Inside a tile, head_dim 64 and 128 are stored in matrix-core operand order (kv_k_elem, kv_v_elem);
// every other head_dim is row-major [token][dim].
__host__ __device__ __forceinline__ uint64_t kv_tile_offset(uint32_t block_count, uint32_t kv_heads,
                                                            uint32_t head_dim, uint32_t layer,
                                                            uint32_t physical_block, uint32_t kv_head) {
  return ((static_cast<uint64_t>(layer) * block_count + physical_block) * kv_heads + kv_head) *
         kKvBlockTokens * head_dim;
}

__host__ __device__ __forceinline__ bool kv_operand_order(uint32_t head_dim) { return head_dim == 128 || head_dim == 64; }
// Element offset of (token row, dim d) inside a K tile. In operand order load j of lane
// l = (d%32/8)*16 + row holds dims 32j + 8*(l/16) .. +7 of token l%16, the A operand of a
// 16x16x32 matrix-core product over dims.
__host__ __device__ __forceinline__ uint32_t kv_k_elem(uint32_t head_dim, uint32_t row, uint32_t d) {
  if (!kv_operand_order(head_dim)) return row * head_dim + d;
  return (d / 32) * 512 + (((d % 32) / 8) * 16 + row) * 8 + d % 8;
}
// Same for a V tile: load j of lane l = (row/4)*16 + d%16 holds tokens
// 4*(l/16) .. +3 of dim 32j + l%16, then of dim 32j + 16 + l%16: the A operands of two
// 16x16x16 products over tokens (V transposed).
__host__ __device__ __forceinline__ uint32_t kv_v_elem(uint32_t head_dim, uint32_t row, uint32_t d) {
  if (!kv_operand_order(head_dim)) return row * head_dim + d;
  const uint32_t slab = d / 16, n = d % 16;
  return (slab / 2) * 512 + ((row / 4) * 16 + n) * 8 + (slab % 2) * 4 + row % 4;
}

// One sequence of a batch launch: the cache a token row belongs to and its position there.
struct AttnSeq {
  uint16_t *k_cache, *v_cache;
  const uint32_t *table;
  uint32_t block_count, position;
};

struct AttnParams {
  const float *qkv;            // [heads*hd | kv_heads*hd | kv_heads*hd] raw f32 projections
  const uint16_t *q_norm, *k_norm;           // optional [hd]
  const uint16_t *q_bias, *k_bias, *v_bias;  // optional
  uint16_t *k_cache, *v_cache;
  const uint32_t *table;       // [block_count]
  const float *rope_freq;      // [hd/2]: powf(theta, 2i/hd), or null = no RoPE
  const float *rope_cs;        // optional [hd]: cos | sin of pos / rope_freq[i], precomputed for this step
  float *part_acc;             // [heads][splits][hd]  un-normalised partial outputs
  float *part_m, *part_l;      // [heads][splits]
  uint32_t *counters;          // [kv_heads] arrival counters, zero between launches
  // Decode step kernel: the splits' partials as (f32 value, tag) 8-byte words, [heads][splits][head_dim + 2]
  // (accumulators, then m and l), all tags zero between launches (attn_step_workspace_bytes)
  uint64_t *part_tagged;
  float *out_f32;              // optional [heads*hd]
  uint16_t *out16;             // [heads*hd]
  uint32_t heads, kv_heads, head_dim, layer, block_count, splits;
  float eps;
  const uint32_t *cursor;      // device position, or null -> `position`
  uint32_t position, max_steps, append;
  uint64_t *trace;             // tuning aid: [32] device timestamps of selected workgroups' stages, or null
  // A block of `tokens` consecutive positions in one launch (grid z; 0 or 1 = a single token).
  // Token z works at position + z (the cursor is not used then) with its own q/k/v, output, rotation
  // table and split workspace: the strides below are added z times.
  uint32_t tokens;
  uint32_t qkv_token_stride;   // f32 elements between tokens' q|k|v
  // Batches of sequences only: qkv_slices = 2..4 says that `qkv` holds that many partial sums of every value,
  // qkv_slice_stride f32 elements apart (the K slices of the projection, as its kernel leaves them), and the launch
  // adds them in slice order as it reads them - what the projection's own slice-adding launch would have written.
  uint32_t qkv_slices, qkv_slice_stride;
  uint32_t out_token_stride;   // elements between tokens' outputs (out16 and out_f32)
  uint32_t rope_token_stride;  // f32 elements between tokens' cos|sin tables
  uint64_t ws_token_stride;    // bytes between tokens' split workspaces (attn_workspace_bytes)
  // A batch of sequences instead of consecutive positions of one: token z belongs to seqs[z] (device
  // memory, `tokens` entries), which replaces k_cache, v_cache, table, block_count and the position.
  // Applies to z = 0 as well, and to a block of one token. With append = 1 every sequence's new row
  // is written to its cache by the launch itself.
  const AttnSeq *seqs;
  uint32_t seq_blocks;         // with seqs: cache blocks of the longest of them (0: not known), which the kernel is chosen by
  // Block launches only: != 0 writes out16 in the multi-row GEMM's operand order (gemm_x_packed_index)
  // with this many token tiles, instead of [token][heads * head_dim] rows.
  uint32_t out_packed_tiles;
  // Decode step only, optional: this step's split plan (attn_plan_fill), written once per step for
  // all layers - position, split geometry and every wave's first physical blocks - so that a launch
  // reaches its tile requests through one scalar read instead of position -> block table -> tiles.
  // Valid for launches with `splits` = the plan's split factor and 8 waves per workgroup.
  const uint32_t *plan;
  // Decode step only: up to this many blocks in use, one split takes them all (attn_split_geometry). 0: never.
  uint32_t single_split_blocks;
  // Decode step only, the splits' merge. A partial is valid for the launch whose tag it carries: the tag is made
  // of the launch's sequence number on this workspace - the plan's step number, or `launches` without a plan -
  // and the layer, so a word that a late or earlier launch left behind can never be taken for this launch's.
  // `launches`, a word for each kv head: kAttnLaunchQuantum for every launch on this workspace whose splits merged, added up
  // by the workgroups themselves: a host's number would come back with every replay of a captured launch, and with it the
  // words of the replay before. A workgroup adds its share behind its own look, so all of a kv head see the same number of
  // whole quanta. (28 heads on 4, 900 keys: 8.8 -> 8.9 us; with one word for all
  // kv heads and a look of its own 10.2.)
  uint64_t *launches;
  // A merge gives up after this many polls of the words it waits for (0 = kAttnMergeSpinLimit), sets *fault
  // (optional device word, never cleared by a kernel) and leaves NaN in the outputs it feeds.
  uint32_t merge_spin_limit;
  uint32_t *fault;
  // Test hook: 1 + the index of a split that keeps its partial to itself (0 = none), so that the bounded wait of
  // the merges that need it can be seen to end; every kernel still exits normally.
  uint32_t withhold_split;
};
constexpr uint32_t kAttnMergeSpinLimit = 1u << 20;
constexpr uint64_t kAttnLaunchQuantum = 65536;   // more than a kv head has splits
constexpr uint32_t kAttnLaunchStride = 8;        // 64-bit words between kv heads': a cache line's part each
// Tag of the partials of launch `seq` (never 0, the cleared state): distinct for 2^23 consecutive steps of up
// to 256 layers; a session's words are cleared when a sequence starts as well.
__host__ __device__ __forceinline__ uint32_t attn_launch_tag(uint32_t seq, uint32_t layer) {
  return ((seq * 256u + (layer & 255u)) << 1) | 1u;
}
// The step kernel's merges need every active split of a kv head on the machine at once (a merging workgroup
// holds its CU while it polls), one 8-wave workgroup per CU: the largest split factor a launch may use there.
uint32_t attn_resident_splits(uint32_t kv_heads);

// Heads of 64, and 3, 5, 6 or 7 query heads a kv head: the shapes whose queries and probabilities were f32 in the general
// kernel before the matrix cores took them, and whose launches waited for nobody. (Heads of 128 with 1, 2, 4 or 8 query heads
// always had two 16-bit parts of them and a merge by every split.)
constexpr bool attn_f32_shape(uint32_t head_dim, uint32_t group) { return head_dim != 128 || (group & (group - 1)) != 0; }
// At those shapes no more than this many workgroups of a launch merge, and wait: sessions on streams of their own run
// their launches side by side, a workgroup has a CU to itself, and 28 heads on 4 (or 40 on 8) were 112 (160) that poll on
// 256 CUs - two launches could hold each other's CUs until the waits gave up. Consecutive workgroups go round the eight
// XCDs, so that is seven of an XCD's 32 CUs: four launches at once, one a hardware queue, leave it four that nobody waits on. A merging workgroup then
// has up to four parts at a time (28 heads on 4 at 900 / 8000 keys: 7.9 / 8.8 -> 8.8 / 10.0 us a launch, one part after the other
// 9.2 / 10.0; 40 on 8 at 4000: 8.7 -> 10.1, 11.1; 32 heads of 64 on 8 at 8000: 8.4 -> 8.6, 9.2).
constexpr uint32_t kAttnWaitingWorkgroups = 56;

// ---- per-step split plan of the decode attention ---------------------------------------------
// words [0..7]: position, blocks, blocks per split, active splits, step number (the caller's), 3 spare;
// then one 8-word entry per (split, wave): tiles of the wave, its first block, the physical blocks
// of its first four tiles (clamped), 2 spare.
constexpr uint32_t kAttnPlanHeader = 8, kAttnPlanEntry = 8, kAttnPlanWaves = 8;
__host__ __device__ __forceinline__ uint64_t attn_plan_bytes(uint32_t splits) {
  return (kAttnPlanHeader + static_cast<uint64_t>(splits) * kAttnPlanWaves * kAttnPlanEntry) * sizeof(uint32_t);
}
// The shapes of the matrix-core kernels: up to eight query heads a kv head (a wave's sixteen columns hold the hi and the
// lo half of each), heads of 64 or 128. Everything else takes the general kernel, one token a launch.
__host__ __device__ __forceinline__ bool attn_matrix_cores(uint32_t heads, uint32_t kv_heads, uint32_t head_dim) {
  return kv_operand_order(head_dim) && kv_heads != 0 && heads % kv_heads == 0 && heads / kv_heads >= 1 && heads / kv_heads <= 8;
}
// Split geometry shared by the kernel and the plan: a split takes ceil(blocks / splits) blocks - or all of
// them while the context is short (single_blocks, 0 = never): the exchange between splits costs about 3 us
// whatever the context, and up to some 300 keys one workgroup per kv head has read its keys before that
// (measured on the Qwen3-8B head shape: 64 keys 4.8 us against 12.7, 256 keys 6.5 against 8.2, 512 keys 10.0
// against 8.0).
constexpr uint32_t kAttnSingleSplitBlocks = 20;
// The same for a batch step, whose splits merge behind a ticket. us in a running session, 6 sequences, 16 heads on 8, 158 / 338 / 548 / 753 keys: in
// six splits 12.6 / 14.4 / 14.9 / 15.6, in one 6.4 / 8.9 / 12.4 / 13.8; 8 heads of 64 on 2, 9 sequences: 9.8 / 10.2 / 10.1 / 10.4 and 5.2 / 6.8 /
// 8.3 / 9.6. With up to three query heads of 128 a key head the merge is so short that few workgroups lose by one split before that: 4
// sequences, 16 on 8, 548 / 628 / 708 / 753 keys 12.7 / 12.8 / 13.1 / 12.9 in eight splits, 11.8 / 13.0 / 13.4 / 13.6 in one; 2 sequences
// 12.2 / 12.1 / 12.1 / 12.4 and 11.4 / 12.9 / 13.2 / 13.8.
constexpr uint32_t kAttnBatchSingleSplitBlocks = 48, kAttnBatchSingleSplitFew = 36;
// Cache blocks up to which the longest of a batch step's sequences gets one split.
uint32_t attn_batch_single_split(uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t sequences);
// Whether a batch step's launch takes the step kernel (attn_decode.hip), the longest sequence in `longest_blocks` cache blocks.
constexpr uint32_t kAttnBatchStepBlocks = 128;
bool attn_batch_in_step(uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t sequences, uint32_t splits, uint32_t longest_blocks);
__host__ __device__ __forceinline__ void attn_split_geometry(uint32_t pos, uint32_t splits, uint32_t single_blocks,
                                                             uint32_t &nblk, uint32_t &bps, uint32_t &active) {
  nblk = (pos + 1 + kKvBlockTokens - 1) / kKvBlockTokens;
  bps = nblk <= single_blocks ? nblk : (nblk + splits - 1) / splits;
  active = (nblk + bps - 1) / bps;
}
// One thread per (split, wave) entry (`entry` < splits * 8); entry 0 also writes the header.
__device__ __forceinline__ void attn_plan_fill(uint32_t *plan, const uint32_t *table, uint32_t pos, uint32_t splits,
                                               uint32_t single_blocks, uint32_t entry, uint32_t step_number) {
  uint32_t nblk, bps, active;
  attn_split_geometry(pos, splits, single_blocks, nblk, bps, active);
  if (entry == 0) {
    plan[0] = pos;
    plan[1] = nblk;
    plan[2] = bps;
    plan[3] = active;
    plan[4] = step_number;
  }
  const uint32_t split = entry / kAttnPlanWaves, wave = entry % kAttnPlanWaves;
  const uint32_t b0 = split * bps, b1 = min(nblk, b0 + bps), first = b0 + wave;
  uint32_t *e = plan + kAttnPlanHeader + entry * kAttnPlanEntry;
  e[0] = first < b1 ? (b1 - first + kAttnPlanWaves - 1) / kAttnPlanWaves : 0u;
  e[1] = first;
  for (uint32_t f = 0; f < 4; ++f) e[2 + f] = table[min(first + f * kAttnPlanWaves, nblk - 1)];
}

// Index of output element e (= head * head_dim + dim) behind a token's out16 base.
__host__ __device__ __forceinline__ uint32_t attn_out_elem(const AttnParams &p, uint32_t e) {
  return p.out_packed_tiles != 0 ? (e / 32u) * p.out_packed_tiles * 512u + ((e % 32u) / 8u) * 128u + e % 8u : e;
}
// Offset of token z's out16 base.
__host__ __device__ __forceinline__ uint64_t attn_out_token(const AttnParams &p, uint32_t z) {
  return p.out_packed_tiles != 0 ? static_cast<uint64_t>(z / 16u) * 512u + (z % 16u) * 8u
                                 : static_cast<uint64_t>(z) * p.out_token_stride;
}

// Split-KV factor. The matrix-core kernel keeps one 8-wave workgroup per CU, so kv_heads x splits
// stays within the 256 CUs (a second round of workgroups costs more than the shorter tile loops
// save); within that, more splits mean fewer 16-token tiles per wave in a row.
inline uint32_t attn_default_splits(uint32_t kv_heads, uint32_t block_count) {
  uint32_t splits = attn_resident_splits(kv_heads);
  if (splits > kAttnMaxSplits) splits = kAttnMaxSplits;
  if (splits > block_count) splits = block_count;
  return splits == 0 ? 1 : splits;
}
// The same for the step kernel of a model: one split where a workgroup a kv head would be more than may wait.
inline uint32_t attn_step_splits(uint32_t heads, uint32_t kv_heads, uint32_t head_dim) {
  const bool few_wait = attn_f32_shape(head_dim, heads / kv_heads);
  return few_wait && kv_heads > kAttnWaitingWorkgroups ? 1u : attn_resident_splits(kv_heads);
}
uint64_t attn_workspace_bytes(uint32_t heads, uint32_t head_dim);
// Bytes of AttnParams::part_tagged (head_dim up to 128), zero-initialised once.
uint64_t attn_step_workspace_bytes(uint32_t heads);
// Carves part_acc/part_m/part_l/counters out of a workspace of attn_workspace_bytes().
void attn_bind_workspace(AttnParams &p, void *workspace);
hipError_t launch_attn_decode(uint32_t dtype, const AttnParams &p, hipStream_t stream);

// Prompt block: rounds and writes the K and V rows of `tokens` consecutive positions
// (position .. position + tokens - 1) into the cache - bias, per-head RMSNorm (k_norm) and RoPE
// as in the decode kernel - so that a following launch_attn_decode with append = 0 and the same
// token block finds every row of the block in place. attn_matrix_cores shapes only. Uses qkv, k_norm, k_bias,
// v_bias, the caches and table, rope_freq / rope_cs and the token strides of `p`.
hipError_t launch_kv_publish_rows(uint32_t dtype, const AttnParams &p, hipStream_t stream);

// Attention of a prompt block with the K/V tiles of the prefix shared by the block's tokens
// (attn_prompt.hip): same inputs and outputs as launch_attn_decode for a block (tokens consecutive
// positions from `position`, rows already in the cache, append = 0, per-token strides, per-token split
// workspaces, rotation tables per token row), attn_matrix_cores shapes only.
// p.splits = 0 lets the launcher choose.
hipError_t launch_attn_prompt(uint32_t dtype, const AttnParams &p, hipStream_t stream);
// Tokens a launch should take of a pass of `tokens` from `position` on: a block (of at most `block` tokens, which is what the
// splits' workspace is for), or all of them, without splits.
uint32_t attn_prompt_launch_tokens(uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t position, uint32_t tokens, uint32_t block);

}  // namespace nv
