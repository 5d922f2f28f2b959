// Device side of a parallel layer's decode projections (gemv_layer.cuh): the walks over weight rows, which a launch of their own takes or
// workgroups beside those of another launch (riders, attn_latent_wide.hip).
#pragma once

#include "activations.cuh"
#include "gemv_layer.cuh"
#include "gemv_stream.cuh"

namespace nv {
namespace layer {

constexpr uint32_t kChunk = kWave * 8;       // columns of a load instruction
constexpr size_t kMaxLds = 56 * 1024;
__host__ __device__ __forceinline__ uint32_t padded(uint32_t cols) { return (cols + kChunk - 1) / kChunk * kChunk; }
__host__ __device__ __forceinline__ uint32_t back_columns(uint32_t mix_cols, uint32_t top, uint32_t ff, uint32_t shared_ff) {
  return padded(mix_cols) + top * padded(ff) + padded(shared_ff);
}

// A 16-bit vector into LDS, with zeros behind it up to a whole chunk (the weights there are taken as zero as well). cols % 8 == 0.
template <int THREADS>
__device__ __forceinline__ void clear_tail(uint16_t *xs, uint32_t cols) {
  for (uint32_t c = cols + threadIdx.x; c < padded(cols); c += THREADS) xs[c] = 0;
}
template <int THREADS>
__device__ __forceinline__ void stage_vector(uint16_t *xs, const uint16_t *src, uint32_t cols) {
  for (uint32_t c = threadIdx.x * 8u; c < cols; c += THREADS * 8u) *reinterpret_cast<uint4 *>(xs + c) = *reinterpret_cast<const uint4 *>(src + c);
  clear_tail<THREADS>(xs, cols);
}

// Two rows of weights that a wave walks together, and what becomes of their sums.
struct Unit {
  const uint16_t *w0, *w1;
  uint32_t at;             // the staged input's place in LDS
  uint32_t cols;
  float *out0, *out1;      // plain rows (out1 null: there is no second one)
  uint16_t *act;           // gate and up row: one activation
  float limit;
};

constexpr int kBatch = 4;   // chunks of a request batch: 4 KiB of each row

// A wave's walk over its units first, first + stride, .. < units; unit_at(i) -> Unit (i is wave-uniform). The first two
// batches of weights are requested by start(), which does not need the staged inputs.
template <uint32_t DT, typename At>
struct PairWalk {
  At unit_at;
  uint32_t units, stride, lane;
  uint4 b0[2][kBatch], b1[2][kBatch];
  uint32_t iu, ic;      // next batch to request: unit, first column
  Unit in;
  uint32_t cu, cc;      // next batch to multiply
  Unit cur;
  float acc0, acc1;

  __device__ __forceinline__ PairWalk(At at, uint32_t n, uint32_t first, uint32_t step)
      : unit_at(at), units(n), stride(step), lane(threadIdx.x & (kWave - 1)), iu(first), ic(0), in{}, cu(first), cc(0), cur{}, acc0(0.0f), acc1(0.0f) {}
  __device__ __forceinline__ void issue(uint4 (&to)[2][kBatch]) {
    if (iu >= units) return;
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const uint32_t c = ic + u * kChunk + lane * 8u;
      const bool on = c < in.cols;
      to[0][u] = on ? load_stream(in.w0 + c) : make_uint4(0u, 0u, 0u, 0u);
      to[1][u] = on ? load_stream(in.w1 + c) : make_uint4(0u, 0u, 0u, 0u);
    }
    ic += kBatch * kChunk;
    if (ic >= in.cols) {
      ic = 0;
      iu += stride;
      if (iu < units) in = unit_at(iu);
    }
  }
  __device__ __forceinline__ void consume(const uint4 (&from)[2][kBatch], const uint16_t *xs) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      if (cc + u * kChunk < cur.cols) {
        const uint4 x = *reinterpret_cast<const uint4 *>(xs + cur.at + cc + u * kChunk + lane * 8u);
        acc0 = dot8<DT, true>(from[0][u], x, acc0);
        acc1 = dot8<DT, true>(from[1][u], x, acc1);
      }
    }
    cc += kBatch * kChunk;
    if (cc < cur.cols) return;
    acc0 = wave_sum(acc0);
    acc1 = wave_sum(acc1);
    if (lane == 0) {
      if (cur.act != nullptr) {
        *cur.act = enc16<DT>(clamped_glu(acc0, acc1, cur.limit));
      } else {
        *cur.out0 = acc0;
        if (cur.out1 != nullptr) *cur.out1 = acc1;
      }
    }
    acc0 = acc1 = 0.0f;
    cc = 0;
    cu += stride;
    if (cu < units) cur = unit_at(cu);
  }
  __device__ __forceinline__ void start() {
    if (iu < units) in = cur = unit_at(iu);
    issue(b0);
    issue(b1);
  }
  __device__ __forceinline__ void run(const uint16_t *xs) {
    while (cu < units) {
      consume(b0, xs);
      issue(b0);
      if (cu >= units) break;
      consume(b1, xs);
      issue(b1);
    }
  }
};

__device__ __forceinline__ Unit two_rows(const uint16_t *w, uint32_t cols, uint32_t rows, uint32_t i, uint32_t at, float *out) {
  const uint32_t r0 = 2u * i, r1 = min(r0 + 1u, rows - 1u);
  return Unit{w + static_cast<uint64_t>(r0) * cols, w + static_cast<uint64_t>(r1) * cols, at, cols, out + r0, r0 + 1u < rows ? out + r1 : nullptr,
              nullptr, 0.0f};
}
__device__ __forceinline__ Unit gate_and_up(const uint16_t *w, uint32_t cols, uint32_t ff, uint32_t i, uint32_t at, uint16_t *act, float limit) {
  return Unit{w + static_cast<uint64_t>(i) * cols, w + static_cast<uint64_t>(ff + i) * cols, at, cols, nullptr, nullptr, act + i, limit};
}

// The expert chosen in a place. A step past the end of the context leaves none there: what earlier launches had in this memory, and weights are asked for
// before the step's guard is known, so the number is kept among those there are.
__device__ __forceinline__ uint32_t expert_of(const uint32_t *ids, uint32_t k, uint32_t experts) {
  return __builtin_amdgcn_readfirstlane(min(ids[k], experts - 1u));
}

// Gate/up pairs begin .. end-1 of the chosen experts (or of one matrix) beside another launch's workgroups: workgroup `block` of `blocks`,
// `xs` LDS for the row.
template <uint32_t DT, int WAVES>
__device__ __forceinline__ void ride_pairs(const RiderPairs &p, const uint32_t *cursor, uint32_t max_steps, uint16_t *xs, uint32_t block, uint32_t blocks) {
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const auto unit_at = [&](uint32_t i) {
    i += p.begin;
    const uint32_t k = i / p.ff, e = p.ids != nullptr ? expert_of(p.ids, k, p.experts) : 0u;
    return gate_and_up(p.w + static_cast<uint64_t>(e) * 2u * p.ff * p.hidden, p.hidden, p.ff, i - k * p.ff, 0u, p.act + k * p.ff, p.limit);
  };
  PairWalk<DT, decltype(unit_at)> walk(unit_at, p.end - p.begin, wave * blocks + block, blocks * WAVES);
  walk.start();
  if (*cursor < max_steps) {   // (after the requests, which read matrices that exist whatever it says)
    stage_vector<WAVES * kWave>(xs, p.h16, p.hidden);
    __syncthreads();
    walk.run(xs);
  }
}

// A row's columns are the pieces' columns one after the other, each piece padded to whole chunks, as their inputs lie in
// LDS. A chunk: where it starts in row 0, bytes from row to row, lanes that have columns, what its products are worth.
struct Chunk {
  uint64_t base;
  uint16_t stride, lanes;
  float factor;
};
static_assert(sizeof(Chunk) == 16, "one LDS read");
constexpr uint32_t kMaxChunks = kMaxLds / (2 * kChunk);
constexpr int kBackBatch = 8;   // chunks of a request batch

// Workgroup `block` of `blocks`; LDS: `xs` the pieces' inputs, `table` their chunks.
template <uint32_t DT, int WAVES>
__device__ __forceinline__ void walk_back(const LayerBack &p, uint16_t *xs, Chunk *table, uint32_t block, uint32_t blocks) {
  constexpr int kThreads = WAVES * kWave;
  const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const uint32_t expert_at = padded(p.mix_cols), shared_at = expert_at + p.top * padded(p.ff);
  const uint32_t chunks = (shared_at + padded(p.shared_ff)) / kChunk, batches = (chunks + kBackBatch - 1) / kBackBatch;
  for (uint32_t i = tid; i < batches * kBackBatch; i += kThreads) {
    const uint32_t at = i * kChunk;
    const uint16_t *base = p.w_o;
    uint32_t cols = p.mix_cols, c = at;
    float factor = 1.0f;
    if (at >= shared_at) {
      base = p.shared_out;
      cols = p.shared_ff;
      c = at - shared_at;
    } else if (at >= expert_at) {
      const uint32_t k = (at - expert_at) / padded(p.ff);
      base = p.e_out + static_cast<uint64_t>(min(p.ids[k], p.experts - 1u)) * p.hidden * p.ff;
      cols = p.ff;
      c = at - expert_at - k * padded(p.ff);
      factor = p.weights[k];
    }
    const uint32_t lanes = i < chunks ? min((cols - c) / 8u, static_cast<uint32_t>(kWave)) : 0u;   // (the last batch's chunks past the end)
    table[i] = Chunk{reinterpret_cast<uint64_t>(base) + 2u * (lanes != 0 ? c : 0u), static_cast<uint16_t>(2u * cols), static_cast<uint16_t>(lanes), factor};
  }
  __syncthreads();
  const uint32_t stride = blocks * WAVES;
  uint4 b0[kBackBatch], b1[kBackBatch];
  uint32_t irow = wave * blocks + block, ib = 0, crow = irow, cb = 0;
  float total = 0.0f;
  const auto issue = [&](uint4 (&to)[kBackBatch]) {
    if (irow >= p.hidden) return;
#pragma unroll
    for (int u = 0; u < kBackBatch; ++u) {
      const Chunk k = table[ib * kBackBatch + u];
      to[u] = make_uint4(0u, 0u, 0u, 0u);
      if (lane < k.lanes) to[u] = load_stream(reinterpret_cast<const char *>(k.base) + static_cast<uint64_t>(irow) * k.stride + lane * 16u);
    }
    if (++ib == batches) {
      ib = 0;
      irow += stride;
    }
  };
  const auto consume = [&](const uint4 (&from)[kBackBatch]) {
#pragma unroll
    for (int u = 0; u < kBackBatch; ++u) {
      const uint32_t i = cb * kBackBatch + u;
      if (i < chunks) total = fmaf(table[i].factor, dot8<DT, true>(from[u], *reinterpret_cast<const uint4 *>(xs + i * kChunk + lane * 8u), 0.0f), total);
    }
    if (++cb < batches) return;
    total = wave_sum(total);
    if (lane == 0) {
      if (p.y != nullptr) p.y[crow] = total;
      else p.x[crow] += p.add != nullptr ? total + p.add[crow] : total;
    }
    total = 0.0f;
    cb = 0;
    crow += stride;
  };
  issue(b0);
  issue(b1);
  if (*p.cursor >= p.max_steps) return;   // (after the requests, which read matrices that exist whatever it says)
  // the inputs, under the first requests
  if (p.mix_cols != 0) stage_vector<kThreads>(xs, p.mixed, p.mix_cols);
  for (uint32_t k = 0; k < p.top; ++k) stage_vector<kThreads>(xs + expert_at + k * padded(p.ff), p.act + k * p.ff, p.ff);
  if (p.shared_ff != 0) stage_vector<kThreads>(xs + shared_at, p.shared_act, p.shared_ff);
  __syncthreads();
  while (crow < p.hidden) {
    consume(b0);
    issue(b0);
    if (crow >= p.hidden) break;
    consume(b1);
    issue(b1);
  }
}

}  // namespace layer
}  // namespace nv
