// A decode step's layers in one launch, for narrow models.
//
// What bounds a step of a narrow model is neither its bytes (5.8 MB a layer at 512 x 1376: a microsecond) nor its arithmetic but the
// five launches a layer, 3.4 to 4.2 us each, of which a boundary and the first accesses behind it are most. Here the workgroups stay for the
// whole step and hand vectors to each other as words of (value, tag), which a reader polls until the tag is its own, and the
// weights of the next projection are requested before the wait for its input begins: 12 us a layer instead of 19. us a step of a call of 24, 12 / 100 /
// 260 / 1000 / 3950 keys, launches and chain, head and sampler (10 us) and the call's own share included:
//   4 layers  512 x 1376,  8 heads of  64 on 4:   86 /  87 /  93 /  93 /  94     65 /  68 /  68 /  72 /  80
//   8 layers  512 x 1792,  4 heads of 128 on 2:  161 / 168 / 176 / 174 / 176    127 / 132 / 133 / 141 / 160
//   6 layers  640 x 1600,  5 heads of 128 on 5:  133 / 139 / 142 / 143 / 148    120 / 124 / 125 / 131 / 144
//   8 layers  768 x 2304, 12 heads of  64 on 4:  171 / 174 / 184 / 185 / 188    165 / 167 / 168 / 175 / 191     (not taken: chain_takes)
// (in a stack of 13.8 MB a layer the requests, which a launch of 128 workgroups has too few of in flight, cost most of what the boundaries did).
//
// A layer is five hand-overs: x -> qkv -> attention -> r = x + o -> activation -> x = r + down. Every workgroup reads the whole of x, of
// the attention's output, of r and of the activation (the residual rows and the norms come with them); a key head's q, k
// and v go to the workgroups of its attention alone. Contexts of more than kChainSingleBlocks blocks are split over workgroups, whose partial
// sums others merge: a sixth hand-over. What a layer costs beyond them is instructions, one wave's at a time - requests 0.4 to 0.8 us a
// projection, its products 0.6 to 1.0, a norm 0.4, the attention 2.8 -, so everything about a projection that can be known before is in
// one table entry (ChainStage).
//
// The workgroups wait for each other, so all of a launch have to be resident: 128 of four waves at most, with registers and LDS for two or three
// a CU. A device that does not hold them never runs a chain (chain_resident). One that does may still be shared, with other sessions' chains on more
// hardware queues than there is room for, with an attention launch that wants every CU for itself and waits too, with another process: launches that
// are each partly resident would then hold each other's places. So a chain's waits are short (kChainSpinLimit): when one runs out the launch says so, waits for
// nothing any more and leaves the chip, and the step is void - its token is not handed out, the cursor stays (step_given_up), whatever it wrote is written
// again - and taken once more. Only kMostGivenUp of them in a row are the step fault that a wait of the decode attention's is.
//
// No word is written before all its readers have read what it held. Every workgroup has rows of o, of gate and up and of down, and writes
// them behind its own reads of what came before; so when x is whole, everyone has read the activation and the r of that layer, and the
// attention's output and the x before it.
#include <float.h>

#include "step_parts.cuh"

namespace nv {

namespace {

using namespace chain;

constexpr int kThreads = 256, kWaves = 4;
constexpr uint32_t kMaxWorkgroups = 128;
constexpr int kRing = 4, kGroup = 4;          // request groups in flight a wave, 16-byte requests of a lane in each

struct Meet {
  __device__ __forceinline__ void operator()() { __syncthreads(); }
};
// The wave's share of n words that lie together, i * 256 + thread.
template <int N>
__device__ __forceinline__ void poll_words(const uint64_t *src, uint32_t n, uint32_t tag, Waiter &wait, uint64_t (&v)[N]) {
  uint32_t spins = 0;
  bool ok;
  const uint32_t thread = fresh_thread();
  do {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = load_tagged(at_bytes(src, min(thread + i * kThreads, n - 1) * 8u));
    ok = true;
#pragma unroll
    for (int i = 0; i < N; ++i) ok = ok && tag_is(v[i], tag);
  } while (wait.again(ok, spins));
}
// Packed 16-bit pairs into LDS.
template <int N>
__device__ __forceinline__ void take_pairs_n(const uint64_t *src, uint32_t n, uint32_t tag, Waiter &wait, uint16_t *dst) {
  uint64_t v[N];
  poll_words<N>(src, n, tag, wait, v);
  const uint32_t thread = fresh_thread();
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (thread + i * kThreads < n) reinterpret_cast<uint32_t *>(dst)[thread + i * kThreads] = static_cast<uint32_t>(v[i]);
}
__device__ __forceinline__ void take_pairs(const uint64_t *src, uint32_t n, uint32_t tag, Waiter &wait, uint16_t *dst) {
  if (n <= 3u * kThreads) take_pairs_n<3>(src, n, tag, wait, dst);
  else take_pairs_n<kChainMaxIn / 2 / kThreads>(src, n, tag, wait, dst);
}

// A projection as a wave walks it. A workgroup's units lie together - every workgroup has some - and go round its waves. A unit is four
// rows, sixteen lanes each (128 columns a request) - of a gate/up pair of matrices two gate rows and their two up rows -, or one row
// (512 columns a request) where rows are few. It takes `groups` request groups; four are in flight. One walk, and one piece of code, for all
// four projections: a kernel with a copy for each (60 KB, a layer's loop through nearly all of it) spent most of its time on fetching instructions.
enum : uint32_t { kQkv = 0, kO = 1, kGateUp = 2, kDown = 3, kStages = 4 };
typedef const __attribute__((address_space(4))) ChainStage *StageAt;
__device__ __forceinline__ ChainStage read_stage(Model m, uint32_t at) {
  const StageAt s = (StageAt)(reinterpret_cast<uint64_t>(m->stage)) + at;
  return ChainStage{s->w,          s->vec,       s->cols,     s->chunks, s->groups,   s->units,  s->unit_bytes,
                    s->row_bytes, s->up_bytes, s->in_at, s->in_words, s->out_at, s->whole,  0u};
}
struct Walk {
  uint32_t total;
  uint32_t first;         // the wave's first unit; the others are kWaves apart
  uint32_t unit, group;   // requested next: unit, place in it
  uint32_t row;           // of the lane: bytes from the unit's first row
  uint32_t col, last;     // ... of its piece of a request, in bytes, and of a row's last piece
  // The request that the lane's row begins with: rows begin at different ones and wrap, so that what the chip asks for at any one time
  // lies on all memory channels (rows are a multiple of their interleave apart: without it 1024 wide requests took 2.5 times as long).
  uint32_t turn;
  uint32_t shift;         // log2 of a request's bytes of a row
};
__device__ __forceinline__ void request_group(Walk &k, const ChainStage &d, uint4 (&dst)[kGroup]) {
  const char *const base = reinterpret_cast<const char *>(d.w) + static_cast<uint64_t>(k.unit) * d.unit_bytes;
  uint32_t c = k.turn + k.group * kGroup;
#pragma unroll
  for (int u = 0; u < kGroup; ++u) {   // (requests that the row does not have: its last pieces once more)
    c = min(c, c - d.chunks);
    // (kept in the caches: a small model's weights are still there when the next step asks for them, 62.5 -> 60.8 us at 512 x 1376)
    dst[u] = *reinterpret_cast<const uint4 *>(base + (k.row + min((c << k.shift) + k.col, k.last)));
    ++c;
  }
  if (++k.group == d.groups) {
    k.group = 0;
    k.unit += kWaves;
  }
}
__device__ __forceinline__ void walk_begin(Walk &k, const ChainStage &d, bool rows, uint32_t log_grid, uint4 (&ring)[kRing][kGroup]) {
  const uint32_t lane = fresh_thread() & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t begin = blockIdx.x * d.units >> log_grid, end = (blockIdx.x + 1) * d.units >> log_grid;
  k.first = k.unit = begin + wave;
  k.total = k.first < end ? (end - k.first + kWaves - 1) / kWaves * d.groups : 0u;
  k.group = 0;
  k.row = rows ? 0u : (lane / 16 & 1u) * d.row_bytes + (lane / 32) * d.up_bytes;
  k.col = (rows ? lane : lane % 16) * 16;
  k.last = d.cols * 2 - 16;
  k.shift = rows ? 10 : 8;
  k.turn = wave + (rows ? 0u : lane / 16 * (d.chunks / 4));
  k.turn = min(k.turn, k.turn - d.chunks);
  k.turn = min(k.turn, k.turn - d.chunks);
  k.turn = min(k.turn, k.turn - d.chunks);
  k.turn = min(k.turn, k.turn - d.chunks);
  // (what the ring held is over: without this, requests under a condition would keep it alive from one walk to the next, through the attention)
#pragma unroll
  for (int f = 0; f < kRing; ++f)
#pragma unroll
    for (int u = 0; u < kGroup; ++u) asm volatile("" : "=v"(ring[f][u].x), "=v"(ring[f][u].y), "=v"(ring[f][u].z), "=v"(ring[f][u].w));
#pragma unroll
  for (int f = 0; f < kRing; ++f)
    if (static_cast<uint32_t>(f) < k.total) request_group(k, d, ring[f]);
}
// done(unit, sum): the sum of a lane's row, in every lane of its sixteen (of the wave, where a unit is a row).
template <uint32_t DT, typename Done>
__device__ __forceinline__ void walk(Walk &k, const ChainStage &d, bool rows, const uint16_t *x, uint4 (&ring)[kRing][kGroup], Done done) {
  const uint32_t lane = fresh_thread() & (kWave - 1);
  const char *const in = reinterpret_cast<const char *>(x);
  uint32_t unit = k.first, group = 0, c = k.turn;
  float open = 0.0f;   // of the unit under way
#pragma unroll 1
  for (uint32_t t = 0; t < k.total; t += kRing) {
    float ends[kRing];
    uint32_t ended = 0;
#pragma unroll
    for (int f = 0; f < kRing; ++f) {
      ends[f] = 0.0f;
      if (t + f < k.total) {
        uint4 xv[kGroup];
        uint32_t at[kGroup];
        float acc[kGroup];
#pragma unroll
        for (int u = 0; u < kGroup; ++u) {
          at[u] = (c << k.shift) + k.col;
          xv[u] = *reinterpret_cast<const uint4 *>(in + min(at[u], k.last));
          ++c;
          c = min(c, c - d.chunks);
        }
#pragma unroll
        for (int u = 0; u < kGroup; ++u) acc[u] = dot8<DT, true>(ring[f][u], xv[u], 0.0f);
        if (!d.whole) {
#pragma unroll
          for (int u = 0; u < kGroup; ++u) acc[u] = at[u] <= k.last && group * kGroup + u < d.chunks ? acc[u] : 0.0f;
        }
        if (t + f + kRing < k.total) request_group(k, d, ring[f]);
        float sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
        sum += dpp_move<kDppQuadSwap1>(sum);
        sum += dpp_move<kDppQuadSwap2>(sum);
        sum += dpp_move<kDppRowHalfMirror>(sum);
        sum += dpp_move<kDppRowMirror>(sum);
        ends[f] = open = open + sum;
        if (++group == d.groups) {
          ended |= 1u << f;
          group = 0;
          c = k.turn;
          open = 0.0f;
        }
      }
    }
#pragma unroll 1
    for (int f = 0; f < kRing && ended >> f != 0; ++f) {
      if ((ended >> f & 1u) == 0) continue;
      float sum = f == 0 ? ends[0] : f == 1 ? ends[1] : f == 2 ? ends[2] : ends[3];
      if (rows) sum = (lane_value(sum, 0) + lane_value(sum, 16)) + (lane_value(sum, 32) + lane_value(sum, 48));
      done(unit, sum, lane);
      unit += kWaves;
    }
  }
}

template <int HD, int G, bool PARTS>
struct ChainShared {
  alignas(16) float xf[kChainMaxHidden];
  alignas(16) float rf[kChainMaxHidden];
  alignas(16) uint16_t x16[kChainMaxHidden];
  float red[2][kWaves];
  float cs[HD];
  union {
    alignas(16) uint16_t in16[kChainMaxIn];
    ChainAttnShared<HD, G, PARTS, kWaves> attn;
    ChainMergeShared<kWaves> merge;
  };
};

template <uint32_t DT, int HD, int G, bool PARTS>
__global__ __launch_bounds__(kThreads, 2) void step_chain_kernel(ChainLaunch p) {
  __shared__ ChainShared<HD, G, PARTS> sh;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  Model m = (Model)(reinterpret_cast<uint64_t>(p.model));
  const uint32_t pos = scalar_load(m->state), step = scalar_load(m->state + 2);
  if (pos >= m->max_steps) return;
  if (p.withhold != 0 && blockIdx.x == 0 && scalar_load(m->state + 5) < p.withhold) return;
  constexpr int kX = kChainMaxHidden / kThreads;
  uint4 ring[kRing][kGroup];
  Walk k;
  const uint32_t log_grid = 31 - __builtin_clz(gridDim.x);   // (chain_workgroups: a power of two)
  ChainStage d = read_stage(m, 0);
  walk_begin(k, d, false, log_grid, ring);

  uint32_t nblk, bps, active;
  chain_splits<kWaves>(m->kv_heads, pos, gridDim.x, nblk, bps, active);
  const bool attends = blockIdx.x < m->kv_heads * active;
  const uint32_t kvh = blockIdx.x % m->kv_heads, split = blockIdx.x / m->kv_heads;
  if (attends && m->rope_freq != nullptr) {
    for (int i = threadIdx.x; i < HD / 2; i += kThreads) {
      float sn, cs;
      sincosf(static_cast<float>(pos) / m->rope_freq[i], &sn, &cs);
      sh.cs[i] = cs;
      sh.cs[HD / 2 + i] = sn;
    }
  }
  Waiter wait{p.spin_limit, m->gave_up};
  Meet meet;
  // test hook: where a layer's vectors go. Workgroup 0 reads all of them but the raw heads, which their producers write
  const auto slot = [](uint32_t bytes) { return (bytes + 255u) & ~255u; };
  const bool traces = p.trace != nullptr;
  const auto trace_at = [&](uint32_t layer, int link) {
    const uint32_t H = m->hidden, h16 = slot(H * 2), h32 = slot(H * 4), qkv = slot((m->heads + 2 * m->kv_heads) * HD * 4), a16 = slot(m->heads * HD * 2), f16 = slot(m->ff * 2);
    uint64_t at = h32 + static_cast<uint64_t>(layer) * (2 * h16 + qkv + a16 + 2 * h32 + f16);
    if (link > 0) at += h16;
    if (link > 1) at += qkv;
    if (link > 2) at += a16;
    if (link > 3) at += h32;
    if (link > 4) at += h16;
    if (link > 5) at += f16;
    return p.trace + at;
  };
  const auto dump16 = [&](uint32_t layer, int link, const uint16_t *from, uint32_t n) {
    if (traces && blockIdx.x == 0)
      for (uint32_t i = fresh_thread(); i < n; i += kThreads) reinterpret_cast<uint16_t *>(trace_at(layer, link))[i] = from[i];
  };

  // A row of x or r: its elements as they come, in f32 and normalised.
  uint32_t turn = 0;
  const auto take_row = [&](float (&v)[kX], const uint16_t (&g)[kX], float *raw) {
    const uint32_t H = m->hidden, thread = fresh_thread();
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < kX; ++i) {
      const uint32_t c = thread + i * kThreads;
      if (c < H) ss = fmaf(v[i], v[i], ss);
    }
    ss = wave_sum(ss);
    if (thread % kWave == 0) sh.red[turn][wave] = ss;
    __syncthreads();
    // 1 / sqrt by the hardware's (an ulp) and a step of Newton's: what a square root and a division leave of it, in a tenth of the time. Neither where
    // the hardware takes the mean for zero (a denormal), nor where the step multiplies zero and infinity (a sum that overflowed, whose row is zero).
    const float mean = fmaf((sh.red[turn][0] + sh.red[turn][1]) + (sh.red[turn][2] + sh.red[turn][3]), m->inv_hidden, m->eps);
    const float rough = __builtin_amdgcn_rsqf(mean);
    float scale = fmaf(rough * 0.5f, fmaf(-mean * rough, rough, 1.0f), rough);
    if (__builtin_expect(!(scale <= FLT_MAX), 0)) scale = 1.0f / sqrtf(mean);
    turn ^= 1u;
#pragma unroll
    for (int i = 0; i < kX; ++i) {
      const uint32_t c = thread + i * kThreads;
      if (c < H) {
        raw[c] = v[i];
        sh.x16[c] = enc16<DT>(v[i] * scale * dec16<DT>(g[i]));
      }
    }
    __syncthreads();
  };
  const auto poll_row = [&](const uint64_t *src, uint32_t tag, float (&v)[kX]) {
    const uint32_t H = m->hidden;
    uint64_t words[kX];
    if (H <= 2u * kThreads) {
      uint64_t few[2];
      poll_words<2>(src, H, tag, wait, few);
      words[0] = few[0];
      words[1] = few[1];
#pragma unroll
      for (int i = 2; i < kX; ++i) words[i] = 0;
    } else {
      poll_words<kX>(src, H, tag, wait, words);
    }
#pragma unroll
    for (int i = 0; i < kX; ++i) v[i] = tag_value(words[i]);
  };

  const uint32_t stages = m->layers * kStages;
#pragma unroll 1
  for (uint32_t at = 0; at < stages; ++at) {
    const uint32_t layer = at / kStages, stage = at % kStages;
    const bool rows = (stage & 1u) != 0;
    const uint32_t tag = step * 256u + layer + 1u;   // (never that of another step until 2^24 of them)
    fresh(m);
    const ChainStage next = read_stage(m, min(at + 1, stages - 1));
    uint64_t *const words = m->words;
    if (!rows) {
      float v[kX];
      uint16_t g[kX];
      const uint32_t thread = fresh_thread();
#pragma unroll
      for (int i = 0; i < kX; ++i) g[i] = *at_bytes(d.vec, min(thread + i * kThreads, m->hidden - 1) * 2u);   // (requested before the wait for the row)
      if (at == 0) {
        uint32_t token = pos < scalar_load(m->state + 1) ? m->prompt[pos] : m->slots[pos - 1].token;
        if (token >= m->vocab) token = 0;   // prompts are validated on the host; sampled ids are < vocab
        const uint16_t *row = m->emb + static_cast<uint64_t>(token) * m->hidden;
#pragma unroll
        for (int i = 0; i < kX; ++i) v[i] = dec16<DT>(row[min(thread + i * kThreads, m->hidden - 1)]);
        if (traces && blockIdx.x == 0)
          for (int i = 0; i < kX; ++i)
            if (thread + i * kThreads < m->hidden) reinterpret_cast<float *>(p.trace)[thread + i * kThreads] = v[i];
      } else {
        poll_row(words + d.in_at, tag, v);
      }
      float *raw = stage == kQkv ? sh.xf : sh.rf;
      take_row(v, g, raw);
      if (traces && stage == kGateUp && blockIdx.x == 0)
        for (uint32_t i = fresh_thread(); i < m->hidden; i += kThreads) reinterpret_cast<float *>(trace_at(layer, 3))[i] = raw[i];
    } else {
      take_pairs(words + d.in_at, d.in_words, tag, wait, sh.in16);
      __syncthreads();
    }
    const uint16_t *const in = rows ? sh.in16 : sh.x16;
    if (traces) dump16(layer, stage == kQkv ? 0 : stage == kO ? 2 : stage == kGateUp ? 4 : 5, in, d.cols);
    uint64_t *const out = words + d.out_at;
    const bool last = at + 1 == stages;
    walk<DT>(k, d, rows, in, ring, [&](uint32_t unit, float sum, uint32_t lane) {
      if (stage == kQkv) {
        if (lane % 16 == 0) {
          store_tagged(at_bytes(out, unit * 32 + lane / 2), sum, tag);
          if (traces) reinterpret_cast<float *>(trace_at(layer, 1))[unit * 4 + lane / 16] = sum;
        }
      } else if (stage == kGateUp) {
        const float other = lane_value(sum, 32), own = lane_value(sum, 48);
        const float g = sum, u = lane < 16 ? other : own;   // (lanes 0 to 31: the two gate rows)
        const uint32_t half = enc16<DT>(gated(g, 1.0f) * u);
        const uint32_t pair = half | (static_cast<uint32_t>(__builtin_amdgcn_readlane(half, 16)) << 16);
        if (lane == 0) store_word(at_bytes(out, unit * 8), pair, tag);
      } else if (lane == 0) {
        float y = sum;
        if (d.vec != nullptr) y += dec16<DT>(d.vec[unit]);
        y += stage == kO ? sh.xf[unit] : sh.rf[unit];
        if (last) m->x[unit] = y;
        else store_tagged(at_bytes(out, unit * 8), y, stage == kO ? tag : tag + 1u);
        if (traces && stage == kDown) reinterpret_cast<float *>(trace_at(layer, 6))[unit] = y;
      }
    });
    if (stage == kQkv) {
      fresh(m);
      if (attends) chain_attention<DT, HD, G, PARTS, kWaves>(m, layer, pos, kvh, split, nblk, bps, active, tag, wait, sh.cs, sh.attn, meet);
      if (active > 1) {   // (heads from the other end of the grid)
        for (uint32_t h = gridDim.x - 1 - blockIdx.x; h < m->heads; h += gridDim.x) chain_merge<DT, HD, kWaves>(m, h, active, tag, wait, sh.merge, meet);
      }
    }
    d = next;
    if (!last) walk_begin(k, d, !rows, log_grid, ring);
  }
}

}  // namespace

bool chain_takes(uint32_t layers, uint32_t hidden, uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t ff) {
  if (!attn_matrix_cores(heads, kv_heads, head_dim) || heads > 512 || hidden > kChainMaxHidden || ff > kChainMaxIn || heads * head_dim > kChainMaxIn) return false;
  // At least as many units of o, of gate and up and of down as workgroups, whole 16-byte pieces, and a table of layers that the tags can tell
  // apart. Stacks of one to three layers would gain what taller ones do (512 x 1376, 700 keys: 38.2 us in launches and 30.0, 56.4 and 42.4, 75.1 and 54.8);
  // they keep their launches: the smallest models are what a step is inspected on, launch by launch.
  if (layers < 4 || layers >= 255 || hidden < kMaxWorkgroups || hidden % 8 != 0 || ff < 2 * kMaxWorkgroups || ff % 8 != 0 || kv_heads > 32) return false;
  // More rows of qkv than that are most of a layer, and their words most of its hand-overs (256 x 768, 32 heads of 128 on 32, 12 / 150 / 400 / 1000
  // keys: 20.4 / 22.0 / 23.3 / 24.0 us a layer in launches, 21.3 / 22.0 / 23.2 / 26.1; 128 x 1024: 20.4 / 22.2 / 23.7 / 24.4, 19.6 / 20.4 / 21.6 / 24.4).
  if ((heads + 2 * kv_heads) * head_dim > kChainMaxQkv) return false;
  // Up to 10 MB of weights a layer. That is no line between faster and slower, but as far as all that was measured is faster: 1.00 to 1.32 times
  // as fast at 40 keys and 1.04 to 1.42 at 700 below it (5 to 10 MB); above it eleven stacks of 10.1 to 14.2 MB 1.04 to 1.17 and 1.07 to 1.25.
  return hidden * (2 * heads + 2 * kv_heads) * head_dim + 3 * hidden * ff <= 5000000u;
}

// A unit or two for a wave (512 x 1376: 64 / 128 / 256 workgroups 76 / 65 / 74 us a step), a power of two.
uint32_t chain_workgroups(uint32_t hidden, uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t ff) {
  const uint32_t units = std::max(ff / 2, (heads + 2 * kv_heads) * head_dim / 4) * ((hidden + 511) / 512);
  const uint32_t want = std::max({(units + 2 * kWaves - 1) / (2 * kWaves), 32u, kv_heads});
  uint32_t grid = 32;
  while (grid < want && grid < kMaxWorkgroups) grid *= 2;
  return grid;
}

// A wave's cache blocks follow one another, so that a chain's attention grows with the blocks that a wave has where the launches' attention, on more
// workgroups, hardly does: by 1.0 to 1.2 us a layer for each, of a gain of 0.4 to 6. With up to two - 2048 keys in sixteen splits - no stack is
// slower by more than 2.4 % (1024 x 768, 8 heads of 128 on one, 1600 keys: 21.0 us a layer in launches, 21.5 here), most are 5 to 40 % faster. With three and four
// those stay faster whose projections are at most seven request groups a wave, one after the other (512 x 1376, 8 heads of 64 on 4, 3950 keys: 21.5 and 18.0; of
// seventeen one is slower, by 2.4 %), but for eight heads of 128 on one; of twenty with more groups nine are slower at 3000 keys (1024 x 768, 8 of 128 on 2: 20.5 and
// 22.2; 432 x 872, 6 on 3, would not be: 21.9 and 20.5). Where there are fewer than sixteen splits there are more key heads, whose blocks the launches'
// attention feels too: up to four all are faster (768 x 768, 16 of 64 on 16, 1600 keys: 22.6 and 22.2), with eight not (3950 keys: 23.8 and 25.8). 48 stacks
// of eight layers, eight contexts each; of forty others, drawn, the slowest step is so by 3.6 %.
uint32_t chain_context(uint32_t hidden, uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t ff) {
  const uint32_t grid = chain_workgroups(hidden, heads, kv_heads, head_dim, ff), waves = grid * kWaves, splits = std::min(kChainMaxSplits, grid / kv_heads);
  const auto up = [](uint32_t n, uint32_t d) { return (n + d - 1) / d; };
  const uint32_t wide = up(hidden, 128 * kGroup);   // request groups of a row of qkv or of gate and up; of o and of down below
  const uint32_t walks = up((heads + 2 * kv_heads) * head_dim / 4, waves) * wide + up(ff / 2, waves) * wide +
                         up(hidden, waves) * (up(heads * head_dim, 512 * kGroup) + up(ff, 512 * kGroup));
  const bool long_contexts = splits < kChainMaxSplits || (walks <= 7 && !(head_dim == 128 && heads / kv_heads == 8));
  return std::min(kChainContext, (long_contexts ? 4 : 2) * kWaves * splits * kKvBlockTokens);
}

uint64_t chain_place(ChainModel &m, uint32_t head_dim) {
  uint64_t end = 0;
  const auto take = [&](uint32_t &at, uint64_t words) {   // on cache lines
    at = static_cast<uint32_t>(end);
    end += (words + 15u) & ~uint64_t{15};
  };
  take(m.at_x, m.hidden);
  take(m.at_qkv, static_cast<uint64_t>(m.heads + 2 * m.kv_heads) * head_dim);
  take(m.at_attn, static_cast<uint64_t>(m.heads) * head_dim / 2);
  take(m.at_part, static_cast<uint64_t>(m.heads) * kChainMaxSplits * (head_dim + 2));
  take(m.at_r, m.hidden);
  take(m.at_ff, m.ff / 2);
  return end;
}

void chain_stages(const ChainModel &m, uint32_t head_dim, const LayerDev &w, ChainStage (&stage)[4]) {
  const uint32_t A = m.heads * head_dim;
  const uint16_t *const matrix[4] = {w.wqkv, w.wo, w.wgu, w.wdown}, *const vec[4] = {w.rms_attn, w.o_bias, w.rms_mlp, nullptr};
  const uint32_t cols[4] = {m.hidden, A, m.hidden, m.ff}, units[4] = {(m.heads + 2 * m.kv_heads) * head_dim / 4, m.hidden, m.ff / 2, m.hidden};
  const uint32_t in_at[4] = {m.at_x, m.at_attn, m.at_r, m.at_ff}, out_at[4] = {m.at_qkv, m.at_r, m.at_ff, m.at_x};
  for (uint32_t i = 0; i < 4; ++i) {
    const bool rows = i % 2 != 0;
    ChainStage &s = stage[i];
    s = ChainStage{};
    s.w = matrix[i];
    s.vec = vec[i];
    s.cols = cols[i];
    s.chunks = (cols[i] + (rows ? 511 : 127)) / (rows ? 512 : 128);
    s.groups = (s.chunks + kGroup - 1) / kGroup;
    s.units = units[i];
    s.row_bytes = cols[i] * 2;
    s.unit_bytes = s.row_bytes * (rows ? 1 : i == kQkv ? 4 : 2);
    s.up_bytes = i == kGateUp ? m.ff * s.row_bytes + m.pair_gap * 2 : s.row_bytes * 2;
    s.in_at = in_at[i];
    s.in_words = rows ? cols[i] / 2 : cols[i];
    s.out_at = out_at[i];
    s.whole = cols[i] % (rows ? 512 : 128) == 0 && s.chunks % kGroup == 0;
  }
}

namespace {
using Kernel = void (*)(ChainLaunch);
template <uint32_t DT>
Kernel kernel_of(uint32_t head_dim, uint32_t group) {
  if (head_dim == 64) {
    if (group == 1) return step_chain_kernel<DT, 64, 1, true>;
    if (group == 2) return step_chain_kernel<DT, 64, 2, true>;
    if (group <= 4) return step_chain_kernel<DT, 64, 4, true>;
    return step_chain_kernel<DT, 64, 8, true>;
  }
  if (group == 1) return step_chain_kernel<DT, 128, 1, false>;
  if (group == 2) return step_chain_kernel<DT, 128, 2, false>;
  if (group == 3) return step_chain_kernel<DT, 128, 4, true>;
  if (group == 4) return step_chain_kernel<DT, 128, 4, false>;
  if (group < 8) return step_chain_kernel<DT, 128, 8, true>;
  return step_chain_kernel<DT, 128, 8, false>;
}
Kernel kernel_of(uint32_t dtype, uint32_t head_dim, uint32_t group) {
  return dtype == kBF16 ? kernel_of<kBF16>(head_dim, group) : dtype == kF16 ? kernel_of<kF16>(head_dim, group) : nullptr;
}
}  // namespace

bool chain_resident(uint32_t dtype, uint32_t hidden, uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t ff) {
  const Kernel kernel = kernel_of(dtype, head_dim, heads / kv_heads);
  int device = 0, cus = 0, each = 0;
  if (kernel == nullptr || hipGetDevice(&device) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&each, reinterpret_cast<const void *>(kernel), kThreads, 0) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return static_cast<uint64_t>(cus) * static_cast<uint64_t>(each) >= chain_workgroups(hidden, heads, kv_heads, head_dim, ff);
}

hipError_t launch_step_chain(uint32_t dtype, uint32_t head_dim, const ChainModel &m, const ChainLaunch &p, hipStream_t stream) {
  if (!chain_takes(m.layers, m.hidden, m.heads, m.kv_heads, head_dim, m.ff) || p.model == nullptr || m.words == nullptr || p.spin_limit == 0)
    return hipErrorInvalidValue;
  const Kernel kernel = kernel_of(dtype, head_dim, m.heads / m.kv_heads);
  if (kernel == nullptr) return hipErrorInvalidValue;
  hipLaunchKernelGGL(kernel, dim3(chain_workgroups(m.hidden, m.heads, m.kv_heads, head_dim, m.ff)), dim3(kThreads), 0, stream, p);
  return hipGetLastError();
}

}  // namespace nv
