// A decode step's layers in one launch: of narrow models (step_chain.hip) and of wider ones (step_wide.hip).
#pragma once

#include "nv_common.cuh"
#include "nerva_hip_api.h"

namespace nv {

// One decoder layer's weights in device memory.
struct LayerDev {
  const uint16_t *rms_attn, *rms_mlp, *wqkv, *q_norm, *k_norm, *q_bias, *k_bias, *v_bias, *wo, *o_bias,
      *wgu, *wdown;
};

// One projection of one layer, as a launch's workgroups walk it: one read through the scalar path.
struct alignas(64) ChainStage {
  const uint16_t *w;
  const uint16_t *vec;         // the norm's weights in front of it, or the o projection's bias, or null
  uint32_t cols, chunks, groups, units;
  uint32_t unit_bytes, row_bytes, up_bytes;   // from unit to unit, from a unit's first row to its second, from its first two to its last two
  uint32_t in_at, in_words, out_at;           // 8-byte words of ChainModel::words
  uint32_t whole, spare;                      // every request of a row is a whole one, and every group has four
};
// The same as a wide model's workgroups walk it (pairs of rows of gate and up).
struct alignas(64) WideStage {
  const uint16_t *w;
  const uint16_t *vec;
  uint32_t cols, row_bytes, rows, up_bytes;   // up_bytes: from a gate row to its up row
  uint32_t log_parts, per_part;               // parts a row is cut into, requests a part
  uint32_t in_at, in_words, out_at, spare;
};
// What a model's chain works on, in device memory (a session's, written once).
struct ChainModel {
  const LayerDev *layer;       // device memory, [layers]
  const ChainStage *stage;     // ..., [layers][4]; a wide model's are `wide`
  const WideStage *wide;
  const uint16_t *emb;
  const uint32_t *prompt;
  const NervaHipSyntheticTokenSlot *slots;
  const uint32_t *state;       // position, prompt tokens, step number (the words' tags derive from it), -, -, steps that gave up in a row
  uint32_t *gave_up;           // set by a launch whose waits ran out
  uint16_t *k_cache, *v_cache;
  const uint32_t *table;
  const float *rope_freq;      // null: no rotation
  float *x;                    // [hidden]: the last layer's output
  uint64_t *words;             // what the workgroups hand to each other, cleared when a sequence starts
  uint32_t layers, hidden, heads, kv_heads, ff, vocab, max_steps, block_count, pair_gap;
  uint32_t at_x, at_qkv, at_attn, at_part, at_r, at_ff;   // places in `words` (chain_place)
  float eps, inv_hidden;
};

// Cache blocks up to which a key head's attention stays with one workgroup: 61 / 101 / 151 keys in one 65.5 / 66 / 68 us a step, in several
// 67.9 / 68.3 / 68.6; 201 keys 73 and 68.6.
constexpr uint32_t kChainSingleBlocks = 8;
constexpr uint32_t kChainMaxHidden = 1024, kChainMaxIn = 4096, kChainMaxQkv = 8192, kChainMaxSplits = 16;
// Tokens of context up to which any model's steps run as a chain (chain_context: less for some)
constexpr uint32_t kChainContext = 4096;
// ... and those of a wide model, by its key heads: the fewer, the fewer workgroups have a part of the context (sixteen splits of
// each at the most, where a step's attention launch makes as many as there are CUs), and the sooner its attention outlasts what
// the ring holds. 43 shapes of 1 to 32 key heads, one to four layers, 768 to 8192 wide, 22 to 1380 MB a layer, at 700 to 32000
// keys, time over that of the step in launches. Less than eight key heads, 8000 keys: .87 to .996 and one 1.003 (4096 x 12288,
// one key head of eight query heads, two layers); at 12000 .89 to 1.03, at 32000 .99 to 1.24. Eight and more, 32000 keys: .88 to
// .987 and one 1.005 (768 x 4096, nine heads of 64).
constexpr uint32_t wide_context(uint32_t kv_heads) { return kv_heads >= 8 ? 32768u : 8192u; }
// Polls after which a wait gives up: 3.1 ms (a step whose workgroup 0 stays away), where the longest wait of a healthy launch is
// some 20 us.
constexpr uint32_t kChainSpinLimit = 1u << 14;
// Whether a model's steps can run as a chain.
bool chain_takes(uint32_t layers, uint32_t hidden, uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t ff);
// Tokens of context up to which they do.
uint32_t chain_context(uint32_t hidden, uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t ff);
uint32_t chain_workgroups(uint32_t hidden, uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t ff);
// ... and whether the device holds all of them at once.
bool chain_resident(uint32_t dtype, uint32_t hidden, uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t ff);
// 8-byte words of ChainModel::words, whose places it fills in.
uint64_t chain_place(ChainModel &model, uint32_t head_dim);
// The walks of a layer's four projections.
void chain_stages(const ChainModel &model, uint32_t head_dim, const LayerDev &layer, ChainStage (&stage)[4]);
struct ChainLaunch {
  const ChainModel *model;     // device memory
  char *trace;                 // test hook: every link's vector, 256 bytes apart (step_trace_bytes), or null
  uint32_t spin_limit;         // polls after which a wait gives up
  uint32_t withhold;           // test hook: so often in a row a workgroup is missing
  uint32_t row_at, ring_at, rounds;   // wide models: places in LDS (launch_step_wide)
};
// `model`: the same on the host.
hipError_t launch_step_chain(uint32_t dtype, uint32_t head_dim, const ChainModel &model, const ChainLaunch &p, hipStream_t stream);

// Whether a wider model's steps run as one launch, and whether the device holds all of it.
bool wide_takes(uint32_t dtype, uint32_t layers, uint32_t hidden, uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t ff);
bool wide_resident(uint32_t dtype, uint32_t heads, uint32_t kv_heads, uint32_t head_dim);
void wide_stages(const ChainModel &model, uint32_t head_dim, const LayerDev &layer, WideStage (&stage)[4]);
hipError_t launch_step_wide(uint32_t dtype, uint32_t head_dim, const ChainModel &model, const ChainLaunch &p, hipStream_t stream);

}  // namespace nv
