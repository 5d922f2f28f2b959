// A decode session's object and what the translation units that implement its steps share of it.
#pragma once

#include <algorithm>
#include <atomic>
#include <memory>
#include <mutex>
#include <vector>

#include "argmax.cuh"
#include "attn_decode.cuh"
#include "gemm_rows.cuh"
#include "gemv_stream.cuh"
#include "runtime_state.hpp"
#include "sampler.cuh"
#include "step_chain.cuh"

namespace nv {

using Slot = NervaHipSyntheticTokenSlot;

enum StepMode { kDecodeStep = 0, kPromptStep = 1, kPromptHeadStep = 2 };
enum LaunchKind { kLEmbed = 0, kLQkv, kLAttn, kLO, kLGateUp, kLDown, kLHead, kLAdvance, kLKinds };

// Token rows of a prompt block or a batch step between the launches of the layers. Uniform decoder layers (16-bit rows by
// type) and mixed stacks (untyped rows of the session's precision) each use their part.
struct RowScratch {
  float *px = nullptr, *pr = nullptr, *pqkv = nullptr, *prope = nullptr;
  uint16_t *pxn16 = nullptr, *pattn16 = nullptr, *pff16 = nullptr;
  char *pgemm_ws = nullptr;        // partial sums of the K-sliced projections
  uint64_t pgemm_ws_bytes = 0;
  float *py = nullptr;               // output of the sublayer under way, before its norm
  void *pxn = nullptr, *pmix = nullptr, *pff = nullptr;   // 16-bit or f32 token rows (the session's precision)
  // layers whose sublayers read the same row: the feed-forward's normalised rows and output
  void *pxn2 = nullptr;
  float *pz = nullptr;
  void *pql = nullptr;               // latent attention: normalised query latents, queries
  float *pq = nullptr;
  void *stack_attn_ws = nullptr;     // split partials of the attention kernels
  uint32_t prefill_pass_tokens = kGemmMaxTokens;   // token rows there is room for: what a pass of the layers takes
};

// The weight arena of a session and of every session forked from it (one stream of the weights can
// then serve a token row of each of them); freed by the last of them to go.
struct SharedWeights {
  // Rows for passes of more than a block of a prompt, of the creating session and all its forks: at 4096 x 12288 another
  // 435 MB, which 32 forks would hold once each and hardly use at the same time. Sessions take turns (PassTurn), in
  // the order in which they enqueue: the event says when the turn before has left the device.
  RowScratch pass;
  std::mutex pass_turn;
  hipEvent_t pass_done = nullptr;
  // Prompts under way of the creating session and all its forks, each behind an event: one that begins comes behind the last but
  // kPromptsAhead (PromptTurn), so that no more than those (and one for each thread that is enqueuing its own) are on the device
  // at once, however many a caller begins. As many as there are hardware queues: 32 prompts of 65 to 195 tokens 4096 wide take
  // 27.8 ms with four or with eight, 29.5 with two; six of 37 to 112 tokens 1024 wide 2.6 and 3.7.
  static constexpr uint32_t kPromptsAhead = 4;
  hipEvent_t prompt_done[kPromptsAhead] = {};
  uint64_t prompts = 0;              // recorded so far
  std::mutex prompt_turn;
  char *origin = nullptr;  // what the allocator returned (and takes back)
  char *base = nullptr;    // the first kMatrixAlign boundary in it: offsets of the weight layout count from here
  uint64_t bytes = 0;
  std::atomic<uint32_t> refs{1};
};

// What a batch step needs to know of each of its sequences, in device memory: the cache and position
// for the attention launches, the token slots for the embedding.
struct BatchTable {
  AttnSeq seq[kGemmMaxTokens];
  const Slot *slots[kGemmMaxTokens];
  SamplerParams sample[kGemmMaxTokens];
};

// Launches whose workgroups wait for each other find a place for all of them or wait in vain, and two at once may each hold what
// the other one needs. Of a device's sessions: who has such launches that may still be under way (InOrder).
struct LaunchOrder {
  std::mutex mutex;
  NervaHipHfDecodeSequenceSession *alone = nullptr;             // the last one that needs the device to itself,
  std::vector<NervaHipHfDecodeSequenceSession *> beside;        // and those behind it that fit beside each other
  std::atomic<uint32_t> sessions{0}, calls{0};   // calls of theirs that are taking steps
};

struct StackModel;   // layer_stack.hpp

}  // namespace nv

struct NervaHipHfDecodeSequenceSession : nv::RowScratch {
  uint32_t dtype = 0, hidden = 0, heads = 0, kv_heads = 0, head_dim = 0, intermediate = 0, vocab = 0,
           layers = 0, max_ctx = 0;
  float eps = 0.0f, theta = 0.0f;
  hipStream_t stream = nullptr;
  nv::SharedWeights *weights = nullptr;  // shared with forks
  char *arena = nullptr;             // everything but the weights: KV cache, sequence state, activations, workspaces
  uint32_t pair_gap = 0;             // elements between a layer's gate rows and its up rows (see kPairGapElems)
  bool arena_in_weights = false;     // `arena` lies behind the weights in their allocation (the creating session)
  uint64_t state_bytes = 0;          // size of `arena`
  uint64_t arena_bytes = 0;          // weights + state, as reported to the caller
  char *pinned = nullptr;
  uint64_t pinned_bytes = 0;
  std::vector<nv::LayerDev> layer;
  const uint16_t *emb = nullptr, *final_norm = nullptr, *lm_head = nullptr;
  uint16_t *kc = nullptr, *vc = nullptr;
  uint32_t block_count = 0;
  uint32_t *table = nullptr, *prompt = nullptr;
  uint32_t *state = nullptr;  // state[0] cursor, state[1] prompt count, state[2] step number: another one for every step's tags (embed counts it up, a
                              // narrow model's sampler too, so that its longer contexts count by two),
                              // state[3] fault word (set by a kernel whose bounded wait gave up; cleared by start),
                              // state[4] the step's chain gave up, state[5] how many in a row have (step_given_up)
  nv::Slot *slots = nullptr;
  float *x = nullptr, *r = nullptr, *qkv = nullptr, *logits = nullptr, *rope_freq = nullptr, *rope_cs = nullptr;
  uint16_t *attn16 = nullptr, *ff16 = nullptr;
  void *attn_ws = nullptr, *sample_ws = nullptr;
  uint32_t attn_splits = 1;
  uint32_t attn_single_blocks = 0;   // contexts of up to this many blocks go to one split (0 with a forced split factor)
  uint64_t *attn_tagged = nullptr;   // tagged split partials of the decode step kernel
  uint32_t *attn_plan = nullptr;     // this step's split plan of the decode attention (attn_plan_fill), or null
  uint64_t *attn_trace = nullptr;  // NERVA_HIP_ATTN_TRACE=1: per-layer stage timestamps of selected attention workgroups
  nv::Slot *host_slots = nullptr;
  uint32_t *host_prompt = nullptr;
  uint32_t *host_state = nullptr;    // 64 words
  // captured steps: 0 decode step with the greedy finish, 1 prompt step, 2 decode step with the
  // temperature / top-k / top-p sampler (its parameters live in device memory, so one capture
  // serves every such configuration), 3 and 4 the two decode steps with their layers in one launch
  static constexpr int kGraphs = 5;
  hipGraph_t graph[kGraphs] = {};
  hipGraphExec_t exec[kGraphs] = {};
  uint64_t graph_nodes[kGraphs] = {};
  // Of graphs 3 and 4, kStepsTogether steps of them in one graph (ensure_together) (each graph saves all but one of its steps' 4
  // us; what a call has left over goes out singly: six save 3.3 us a step and leave five at the most, twelve 3.7 and eleven)
  static constexpr uint32_t kStepsTogether = 6;
  hipGraph_t together_graph[2] = {};
  hipGraphExec_t together[2] = {};
  uint64_t chain_steps = 0;          // steps that went out as chains
  // positions below chain_context step with their layers in one launch (step_chain.cuh); 0: never
  uint32_t chain_context = 0;
  nv::ChainModel chain_model{};      // ... what that launch works on, and its copy on the device
  nv::ChainModel *chain_model_dev = nullptr;
  uint64_t chain_word_bytes = 0;
  bool chain_wide = false;           // ... of the kind that has the whole device to itself (step_wide.hip)
  nv::LaunchOrder *order = nullptr;  // the device's, where this session is counted
  hipEvent_t launched = nullptr;     // recorded by whoever has to come behind this session's launches
  uint32_t steps_ahead = 0;          // steps that a call sends ahead of those it has seen the end of, where others may be waiting (RunAhead)
  hipEvent_t mark = nullptr;         // ... and the event that it looks at
  uint32_t *given_up = nullptr;      // host_state[0]: steps that gave up since the host looked (step_given_up writes it)
  uint32_t chain_sent = 0, chain_missed = 0;   // such steps sent since then; those that gave up with none between them that did not, as far as looks tell
  uint32_t chain_avoid = 0;          // steps that are still taken launch by launch instead (take_given_up)
  // prompt blocks: up to prefill_pass_tokens prompt tokens per pass through the layers (weights streamed
  // once per pass on the matrix cores), in a long prompt prefill_long_tokens; false = one prompt step per token
  bool block_prefill = false;
  // the multi-row kernels take this model's shapes (prompt blocks and batch steps need it)
  bool rows_ready = false;
  bool rows_plain = false;           // ... also for rows as they come, without matrix-operand order
  bool batch_ready = false;          // batch steps stream the weights once for all sequences
  float *blogits = nullptr;          // [NERVA_HIP_BATCH_MAX_BLOCK_TOKENS][vocab] logits of a batch step, or of rows of a prompt block
  uint32_t head_run = 0;             // rows of the last of the latter
  nv::BatchTable *btable = nullptr, *host_btable = nullptr;
  nv::Slot *host_bslots = nullptr;   // a batch step's published slots, side by side in pinned memory
  char *pattn_ws = nullptr;
  uint64_t pattn_ws_stride = 0;
  uint32_t prefill_long_tokens = 0;   // tokens a pass of a prompt of more than prefill_pass_tokens takes, with the rows of all sessions on these weights (0: no such passes)
  uint32_t prefill_block_tokens = nv::kGemmMaxTokens;   // tokens per prompt block: 512 or 256 where every projection has the kernel for it
  nv::SamplerDev sampler{};            // normalised configuration of the active sequence
  nv::SamplerDev *sampler_dev = nullptr;
  uint64_t *sampler_keys = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  char *stage = nullptr;          // two halves of pinned memory that results leave through (copy_out), and their events
  uint64_t stage_half = 0;
  hipEvent_t staged[2] = {nullptr, nullptr};
  // test hook: the next decode step is launched kernel by kernel and every intermediate vector is
  // copied behind the previous one into this caller-owned device buffer (step_trace_bytes)
  char *trace_buf = nullptr;
  uint64_t trace_used = 0;
  // echo of the caller's weight plan
  uint32_t planned_weight_blocks = 0, planned_gpu_resident_blocks = 0, planned_gpu_staged_blocks = 0,
           planned_weight_descriptor_count = 0;
  uint64_t planned_weight_bytes = 0, planned_gpu_resident_weight_bytes = 0,
           planned_gpu_staged_weight_bytes = 0, planned_weight_descriptor_hash = 0;
  uint64_t resident_weight_bytes = 0, kv_bytes = 0;
  // A mixed layer stack (layer_stack.hpp) instead of the uniform decoder layers above: its layers and weights, shared
  // with forks, and this sequence's part of it. The members above that describe one uniform layer are then unused or
  // hold the largest sizes; hidden, vocab, max_ctx, the prompt, the slots, the cursor words, the sampler, the graphs
  // and the lifecycle are the same.
  std::shared_ptr<const nv::StackModel> stack;
  char *stack_cache = nullptr;       // keys and values of the layers that have any, each layer in its own block ring
  uint32_t *stack_tables = nullptr;  // logical block -> block of the layer's ring, per caching layer
  float *stack_state = nullptr;      // recurrent state, f32, all recurrent layers
  uint64_t stack_state_bytes = 0;
  float *y = nullptr;                // output of the sublayer under way, before its norm: decode row
  uint64_t stack_launches = 0;       // kernel launches of the step enqueued last (where the layers do not tell)
  float *prouter = nullptr, *pslots = nullptr;   // experts: router logits, one output row per (token, choice)
  void *pplan = nullptr;             // ... and the block's routing (MoePlan)
  void *pwant = nullptr;             // normalised rows whose logits are asked for, with their row numbers and logits
  uint32_t *pwant_rows = nullptr;
  float *pwant_logits = nullptr;
  // active sequence
  bool started = false, finished = false;
  uint32_t prompt_count = 0, observed = 0, cursor = 0, seed_token = 0, has_eos = 0, eos = 0;
};

namespace nv {

using Session = NervaHipHfDecodeSequenceSession;

struct Carver {
  uint64_t offset = 0;
  uint64_t take(uint64_t bytes, uint64_t align = 256) {
    const uint64_t at = (offset + align - 1) & ~(align - 1);
    offset = at + ((bytes + 255u) & ~uint64_t{255});
    return at;
  }
};
// Weight matrices start on 8 MiB boundaries of device memory (the arena's first such boundary is its origin for
// the weight layout). What the gate/up launch costs depends on its matrix's address modulo 8 MiB - the up rows lie
// a fixed 96 MiB behind the gate rows, and the memory channels are chosen by a hash that reaches up to those bits:
// with the rotated walk 31.0 us at 0 modulo 8 MiB, 31.4 at 2 and 6 MiB, 31.8 at 4 MiB, 32.1 at an odd KiB (the
// plain walk: 33.0 / 31.7 / 31.3 / 31.8 / 31.7). At most 8 MiB a matrix is left unused: under 1.2 GB for 36 layers.
constexpr uint64_t kMatrixAlign = 8u << 20;

// A prompt of `tokens` tokens: while this lives its session works on the shared rows of its weights, if it has more tokens
// than the session's own rows take. Everything that reads rows has to be enqueued before it ends.
class PassTurn {
 public:
  PassTurn(Session *session, uint32_t tokens) : s(session) {
    if (tokens <= s->prefill_pass_tokens || s->prefill_long_tokens <= s->prefill_pass_tokens) return;
    turn = std::unique_lock<std::mutex>(s->weights->pass_turn);
    own = *s;
    static_cast<RowScratch &>(*s) = s->weights->pass;
    s->prefill_pass_tokens = s->prefill_long_tokens;
    error = hipStreamWaitEvent(s->stream, s->weights->pass_done, 0);   // (nothing to wait for before its first record)
  }
  ~PassTurn() {
    if (!turn.owns_lock()) return;
    static_cast<RowScratch &>(*s) = own;
    // whoever comes next waits on the device; where that cannot be arranged, here
    if (hipEventRecord(s->weights->pass_done, s->stream) != hipSuccess) (void)hipStreamSynchronize(s->stream);
  }
  PassTurn(const PassTurn &) = delete;
  PassTurn &operator=(const PassTurn &) = delete;
  hipError_t error = hipSuccess;

 private:
  Session *s;
  RowScratch own;
  std::unique_lock<std::mutex> turn;
};

// While this lives the session enqueues a launch whose workgroups wait for each other, behind those of other sessions that it
// must not meet - of calls in other threads, and of starts that have returned while a prompt that is walked, or whose last token
// takes a step, is under way. The streams keep that order: nobody waits on the host or on the device in front of what is to be
// waited for, and a session that has no other's launches under way beside it enqueues no more than the launch. (Turns that a
// launch of one wave took by polling a word stood in front of what would have given the word back where two sessions share a
// hardware queue; and they took two launches more a step beside any other session, idle or not: 69.4 -> 72.3 us at 512 wide, 845
// -> 848 at 4096.)
enum class Place { kBeside, kAlone };   // meets its like (narrow models' steps); nobody
class InOrder {
 public:
  InOrder(Session *session, Place place) {
    LaunchOrder *const order = session->order;
    if (order == nullptr) return;
    turn = std::unique_lock<std::mutex>(order->mutex);
    std::vector<Session *> &beside = order->beside;
    const auto at = std::find(beside.begin(), beside.end(), session);
    if (place == Place::kBeside && at != beside.end()) return;   // (behind `alone` already)
    if (order->alone != nullptr && order->alone != session) error = follow(session, order->alone);
    if (place == Place::kBeside) {
      if (error == hipSuccess) beside.push_back(session);
      return;
    }
    for (Session *other : beside)
      if (error == hipSuccess && other != session) error = follow(session, other);
    if (error != hipSuccess) return;
    beside.clear();
    order->alone = session;
  }
  InOrder(const InOrder &) = delete;
  InOrder &operator=(const InOrder &) = delete;
  hipError_t error = hipSuccess;

 private:
  static hipError_t follow(Session *session, Session *other) {
    hipError_t err = hipEventRecord(other->launched, other->stream);
    if (err == hipSuccess) err = hipStreamWaitEvent(session->stream, other->launched, 0);
    if (err == hipSuccess) return err;
    (void)hipGetLastError();
    return hipStreamSynchronize(other->stream);
  }
  std::unique_lock<std::mutex> turn;
};
// A session's stream is idle: there is nothing left of it to come behind, nor of what it came behind.
inline void out_of_order(Session *session) {
  LaunchOrder *const order = session->order;
  if (order == nullptr) return;
  const std::lock_guard<std::mutex> lock(order->mutex);
  std::vector<Session *> &beside = order->beside;
  const auto at = std::find(beside.begin(), beside.end(), session);
  if (order->alone == session || at != beside.end()) order->alone = nullptr;
  if (at != beside.end()) beside.erase(at);
}
// The steps that a call enqueues without looking at them: where a device has other sessions, no more than twice steps_ahead (some
// 2 ms each, or a graph of several) before the call waits for the older ones, so that whoever else steps comes in between; of
// steps in one launch never more than twice kUnseen, so that the host hears of those that give up before so many have in a row
// that the device ends the sequence.
class RunAhead {
  static constexpr uint32_t kUnseen = 96;
  static_assert(2 * kUnseen + Session::kStepsTogether < kMostGivenUp, "");

 public:
  explicit RunAhead(Session *session) : s(session) {
    if (s->order != nullptr) s->order->calls += 1;
  }
  ~RunAhead() {
    if (s->order != nullptr) s->order->calls -= 1;
  }
  RunAhead(const RunAhead &) = delete;
  RunAhead &operator=(const RunAhead &) = delete;
  // Whether it is one step at a time: long ones, while others are calling.
  bool singly() const { return s->order != nullptr && s->steps_ahead < Session::kStepsTogether && s->order->calls.load(std::memory_order_relaxed) > 1; }
  // Ahead of the next steps; `sent`: with those that went out since it was last asked.
  hipError_t room(uint32_t sent) {
    unseen += sent;
    const bool others = s->order != nullptr && s->order->sessions.load(std::memory_order_relaxed) > 1;
    if (unseen < (others ? s->steps_ahead : kUnseen) || (!others && s->given_up == nullptr)) return hipSuccess;
    hipError_t err = marked ? hipEventSynchronize(s->mark) : hipSuccess;
    if (err == hipSuccess) err = hipEventRecord(s->mark, s->stream);
    marked = true;
    unseen = 0;
    return err;
  }

 private:
  Session *s;
  uint32_t unseen = 0;
  bool marked = false;
};

// A prompt's place among those under way: as long as its launches are enqueued this lives. The stream waits, not the host (five
// starts of 8000 tokens, 12 layers 4096 wide: 47.9 -> 3.3 ms of the caller, done after 262 either way; 20 steps of another
// session behind them 22.8 ms and 25.4), so it is made behind whatever the host itself waits for.
class PromptTurn {
 public:
  explicit PromptTurn(Session *session) : s(session) {
    SharedWeights &w = *s->weights;
    const std::lock_guard<std::mutex> lock(w.prompt_turn);
    const hipEvent_t oldest = w.prompt_done[w.prompts % SharedWeights::kPromptsAhead];
    if (hipStreamWaitEvent(s->stream, oldest, 0) == hipSuccess) return;   // (nothing to wait for before its first record)
    (void)hipGetLastError();
    if (hipEventSynchronize(oldest) != hipSuccess) (void)hipGetLastError();
  }
  ~PromptTurn() {
    SharedWeights &w = *s->weights;
    const std::lock_guard<std::mutex> lock(w.prompt_turn);
    (void)hipEventRecord(w.prompt_done[w.prompts++ % SharedWeights::kPromptsAhead], s->stream);
  }
  PromptTurn(const PromptTurn &) = delete;
  PromptTurn &operator=(const PromptTurn &) = delete;

 private:
  Session *s;
};

// Moves the sequence's device-side position words (decode_session.hip).
hipError_t set_device_position(Session *s, uint32_t cursor, uint32_t prompt_count, uint32_t clear_fault);
void destroy_session(Session *s);
void fill_create_result(const Session *s, NervaHipHfDecodeSequenceSessionCreateResult *out);
// `bytes` from device memory to the caller's memory, behind what the session's stream holds; there when the call returns, for which it
// waits (one more in *waits) - or, where it enqueues a copy by the runtime and `now` is not asked for, when the stream gets there.
hipError_t copy_out(Session *s, void *dst, const void *src, uint64_t bytes, uint64_t *waits, bool now);
// Stream, the arena of s->weights->bytes (with_weights) + s->state_bytes, the pinned mirrors and the events.
hipError_t allocate_session(Session *s, int32_t *failure_stage, bool with_weights);

}  // namespace nv
