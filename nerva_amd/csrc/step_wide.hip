// A decode step's layers in one launch, for models whose layers are too large for step_chain.hip.
//
// What a step of these models costs beyond its bytes is the five launches a layer: behind each boundary memory stands idle until
// the next launch's first requests are served (2.5 to 3 us, a layer of 101 MB 30 us for 15 us of reads). Here a workgroup a CU
// stays for the whole step and hands vectors on as words of (value, tag), as in step_chain.hip, and the weights run ahead of
// that: two waves of a workgroup do nothing but ask for them, in the order in which they will be used, whole layers long,
// straight into a ring in LDS (what the vectors leave of it, 64 to 140 KiB) that the other eight read. So while those wait for a
// vector, memory goes on until the ring is full - 16 to 35 MB over the chip, 2.5 to 5 us of it. us a layer, launches and here, 40
// / 700 / 8000 keys of context:
//    1024 x  3072, 16 heads of 128 on 8:  20.9 / 23.4 / 26.9    18.1 / 20.3 / 25.0     (31 MB)
//    2048 x  6144, 16 heads of 128 on 8:  30.2 / 32.7 / 36.2    25.0 / 27.4 / 32.1     (101 MB)
//    2048 x  8192, 32 heads of  64 on 8:  33.6 / 36.3 / 38.3    29.2 / 30.3 / 33.7     (122 MB)
//    2560 x  9728, 32 heads of 128 on 8:  47.2 / 49.7 / 53.7    41.3 / 44.1 / 48.6     (202 MB)
//    4096 x 12288, 32 heads of 128 on 8:  70.6 / 73.1 / 77.0    68.0 / 69.8 / 74.7     (386 MB)
//    5120 x 13824, 40 heads of 128 on 8: 106.0 / 109 / 114      97.0 / 98.8 / 103      (551 MB)
// What bounds it now: the hand-overs (1.2 us each and more under load, for the words travel through the memory that the weights
// come from), and the slowest of 256 shares of a projection.
//
// Three things that cost more than they look:
//   * how much is on its way. The more weights a CU has asked for, the longer a word waits behind them: with 16 KiB a loader 2048
//     x 6144 took 25.2 us a layer, with 40 KiB 28, with 52 KiB 32; with 4 KiB, too few, 27.
//   * polling too early. A workgroup that looks for words while their writers still write them takes those lines from them: words
//     of 256 writers, eight to a line, are there after 0.9 us if everyone waits half of that before the first look, after 2 us
//     otherwise. So a wait begins with a pause (kPause: none / 14 / 22 / 30: 28.3 / 27.2 / 25.0 / 24.9 us a layer at 2048 x 6144,
//     16.9 / 15.3 / 14.3 / 15.0 at 512 x 1376).
//   * where the rows begin. Consecutive rows start their walk a request further on, and wrap: rows are a multiple of the memory
//     channels' interleave apart.
//
// The ring: a round is a request of 1 KiB (512 columns of a row) for each of the eight waves; a loader asks for four waves' and
// says how many rounds have arrived, a wave says how many it has used. A projection's rows lie together in a workgroup. Where
// they do not go round the waves evenly a row is cut into two to eight parts (ten rows of nineteen requests: five rounds of five
// in four parts, not two of nineteen); parts meet in LDS.
//
// The loaders take part in no barrier, so the others' is a counter in LDS (Meet). Everything else - the places of words, who
// overwrites what when, waits that run out, steps that are void and taken again - is as in step_chain.hip. A workgroup has a CU
// to itself here, all 256 wait for each other: two such launches that started at once could each hold half of the chip until both
// give up. So a step comes behind what other sessions of the device have under way of that sort (InOrder in session.hpp).
#include <float.h>

#include "step_parts.cuh"

namespace nv {

namespace {

using namespace chain;

constexpr int kWaves = 8, kThreads = kWaves * kWave, kLoaders = 2, kPer = kWaves / kLoaders;
constexpr uint32_t kWorkgroups = 256, kLogWorkgroups = 8;
constexpr uint32_t kRequest = 1024, kRound = kWaves * kRequest;
constexpr uint32_t kOnTheWay = 3;      // rounds that a loader has asked for and not seen, at most one more
constexpr int kPause = 22;             // x 64 cycles
constexpr uint32_t kLdsBytes = 160 * 1024, kLeastRounds = 8, kMostSums = 512, kMostOwn = 32;

enum : uint32_t { kQkv = 0, kO = 1, kGateUp = 2, kDown = 3, kStages = 4 };
typedef const __attribute__((address_space(4))) WideStage *StageAt;
__device__ __forceinline__ WideStage read_stage(Model m, uint32_t at) {
  const StageAt s = (StageAt)(reinterpret_cast<uint64_t>(m->wide)) + at;
  return WideStage{s->w, s->vec, s->cols, s->row_bytes, s->rows, s->up_bytes, s->log_parts, s->per_part, s->in_at, s->in_words, s->out_at, 0u};
}

struct alignas(16) Flags {
  uint32_t met, spare[3];
  uint32_t arrived[4];                     // rounds in LDS, of each loader
  alignas(16) uint32_t used[kWaves];       // rounds a wave has read
};
template <int HD, int G, bool PARTS>
struct WideShared {
  Flags flags;
  float own[2][kMostOwn];                  // the workgroup's own elements of x and of r
  alignas(16) float sums[kMostSums];
  alignas(16) float red[2][kWaves];
  float cs[HD];
  union {                                  // the last: in front of the attention's place lies nothing that the input's may not run over
    ChainAttnShared<HD, G, PARTS, kWaves> attn;
    ChainMergeShared<kWaves> merge;
  };
};

__device__ __forceinline__ uint32_t lds_at(const void *p) {
  return static_cast<uint32_t>(reinterpret_cast<uint64_t>((__attribute__((address_space(3))) const void *)p));
}
// Flags by hand: with requests into LDS under way the compiler waits for all of them ahead of an access of its own.
__device__ __forceinline__ uint32_t read_flag(uint32_t at) {
  uint32_t v;
  asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(at) : "memory");
  return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ void write_flag(uint32_t at, uint32_t v) { asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(v) : "memory"); }

// The barrier of the eight waves: what they wrote to LDS before it is there behind it.
struct Meet {
  uint32_t at, target;
  __device__ __forceinline__ void operator()() {
    target += kWaves;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if ((threadIdx.x & (kWave - 1)) == 0) asm volatile("ds_add_u32 %0, %1" ::"v"(at), "v"(1u) : "memory");
    while (static_cast<int32_t>(read_flag(at) - target) < 0) {
    }
    asm volatile("" ::: "memory");
  }
};

// Rows of a projection (pairs of rows of gate and up) that a workgroup has; of the pairs a whole number of two, which make a word.
struct Share {
  uint32_t first, n;
};
__device__ __forceinline__ Share share_of(const WideStage &d, uint32_t stage) {
  const uint32_t twos = stage == kGateUp ? 1u : 0u, units = d.rows >> twos;
  const uint32_t b = blockIdx.x * units >> kLogWorkgroups, e = (blockIdx.x + 1) * units >> kLogWorkgroups;
  return Share{b << twos, (e - b) << twos};
}
// A wave's part of a row, as its requests go: bytes from the row's first, where the part begins and ends, where its walk does.
struct Part {
  uint32_t low, end, at;
  __device__ __forceinline__ void next() {
    at += kRequest;
    if (at >= end) at = low;
  }
};
__device__ __forceinline__ Part part_of(const WideStage &d, const Share &s, uint32_t q, uint32_t lane_bytes) {
  const uint32_t low = (q & ((1u << d.log_parts) - 1)) * d.per_part * kRequest + lane_bytes;
  return Part{low, low + d.per_part * kRequest, low + (s.first + (q >> d.log_parts)) % d.per_part * kRequest};
}

template <int N>
__device__ __forceinline__ void wait_requests() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// All but the newest n rounds of this loader have arrived.
__device__ __forceinline__ void wait_rounds(uint32_t n) {
  static_assert(kOnTheWay == 3, "a case for each");
  if (n == 0) wait_requests<0>();
  else if (n == 1) wait_requests<kPer>();
  else if (n == 2) wait_requests<2 * kPer>();
  else wait_requests<3 * kPer>();
}

// A loader wave: every request of the step, in order, as far ahead as the ring has room.
__device__ __forceinline__ void load_ahead(Model m, uint32_t stages, uint32_t rounds, char *ring, uint32_t flags) {
  const uint32_t lane = threadIdx.x & (kWave - 1), j = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) - kWaves;
  const uint32_t arrived_at = flags + offsetof(Flags, arrived) + j * 4, used_at = flags + offsetof(Flags, used) + j * kPer * 4;
  uint32_t asked = 0, seen = 0, used = 0, slot = 0;
  const auto see = [&](uint32_t behind) {   // the oldest round that is under way
    wait_rounds(behind);
    ++seen;
    write_flag(arrived_at, seen);
  };
#pragma unroll 1
  for (uint32_t at = 0; at < stages; ++at) {
    const WideStage d = read_stage(m, at);
    const uint32_t stage = at % kStages, last = d.row_bytes - 16, both = stage == kGateUp ? 2 : 1;
    const Share s = share_of(d, stage);
    const uint32_t parts = s.n << d.log_parts;
#pragma unroll 1
    for (uint32_t g = 0; g < parts; g += kWaves) {
      const char *row[kPer];
      Part part[kPer];
#pragma unroll
      for (int k = 0; k < kPer; ++k) {   // (a wave without a part: one line of the last part's again)
        const uint32_t q = g + j * kPer + k, have = min(q, parts - 1);
        row[k] = reinterpret_cast<const char *>(d.w) + static_cast<uint64_t>(s.first + (have >> d.log_parts)) * d.row_bytes;
        part[k] = part_of(d, s, have, q < parts ? lane * 16 : 0u);
      }
#pragma unroll 1
      for (uint32_t c = 0; c < d.per_part; ++c) {
#pragma unroll 1
        for (uint32_t h = 0; h < both; ++h) {
          while (static_cast<int32_t>(asked - used) >= static_cast<int32_t>(rounds)) {
            uint4 v;
            asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(used_at) : "memory");
            const uint32_t least = __builtin_amdgcn_readfirstlane(min(min(v.x, v.y), min(v.z, v.w)));
            if (least != used) used = least;
            else if (seen != asked) see(asked - seen - 1);
          }
#pragma unroll
          for (int k = 0; k < kPer; ++k)   // (once used, never again in this step: past the caches)
            __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint32_t *>(row[k] + h * d.up_bytes + min(part[k].at, last)),
                                             (__attribute__((address_space(3))) uint32_t *)(ring + slot * kRound + (j * kPer + k) * kRequest), 16, 0, 2);
          ++asked;
          if (++slot == rounds) slot = 0;
          if (asked - seen > kOnTheWay) see(kOnTheWay);
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k) part[k].next();
      }
    }
  }
  while (seen != asked) see(asked - seen - 1);
}

// A wave's place in the ring.
struct Reader {
  uint32_t round, arrived, slot, rounds;
  const char *mine;   // the wave's and the lane's piece of the ring's first round
  uint32_t arrived_at, used_at;
  __device__ __forceinline__ void need(uint32_t n) {
    while (static_cast<int32_t>(arrived - (round + n)) < 0) arrived = read_flag(arrived_at);
  }
  __device__ __forceinline__ uint4 take() {
    const uint4 v = *reinterpret_cast<const uint4 *>(mine + slot * kRound);
    ++round;
    if (++slot == rounds) slot = 0;
    return v;
  }
  __device__ __forceinline__ void skip(uint32_t n) {
    round += n;
    slot = (slot + n) % rounds;
  }
  __device__ __forceinline__ void done() { write_flag(used_at, round); }   // (LDS serves a wave's accesses in their order)
};
// The wave's parts of a projection: sums[part], of a pair of rows sums[2 * part] and the next.
template <uint32_t DT>
__device__ __forceinline__ void walk(Reader &r, const WideStage &d, uint32_t stage, const Share &s, const uint16_t *x, float *sums) {
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t parts = s.n << d.log_parts, last = d.row_bytes - 16;
  const char *const in = reinterpret_cast<const char *>(x);
#pragma unroll 1
  for (uint32_t q = wave; q < parts + wave; q += kWaves) {   // (as many turns for every wave)
    if (q >= parts) {
      r.skip(stage == kGateUp ? 2 * d.per_part : d.per_part);
      r.done();
      continue;
    }
    Part part = part_of(d, s, q, lane * 16);
    float a = 0.0f, b = 0.0f;
    uint32_t c = 0;
    if (stage != kGateUp) {
      for (; c + 4 <= d.per_part; c += 4) {
        r.need(4);
        uint4 w[4], v[4];
        bool live[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          w[u] = r.take();
          v[u] = *reinterpret_cast<const uint4 *>(in + min(part.at, last));
          live[u] = part.at <= last;
          part.next();
        }
        r.done();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float p = dot8<DT, true>(w[u], v[u], 0.0f);
          float &sum = u & 1 ? b : a;
          sum += live[u] ? p : 0.0f;
        }
      }
      for (; c < d.per_part; ++c) {
        r.need(1);
        const uint4 w = r.take(), v = *reinterpret_cast<const uint4 *>(in + min(part.at, last));
        r.done();
        const float p = dot8<DT, true>(w, v, 0.0f);
        a += part.at <= last ? p : 0.0f;
        part.next();
      }
      a = wave_sum(a + b);
      if (lane == 0) sums[q] = a;
    } else {
      for (; c + 2 <= d.per_part; c += 2) {
        r.need(4);
        uint4 w[4], v[2];
        bool live[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          w[2 * u] = r.take();
          w[2 * u + 1] = r.take();
          v[u] = *reinterpret_cast<const uint4 *>(in + min(part.at, last));
          live[u] = part.at <= last;
          part.next();
        }
        r.done();
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const float p = dot8<DT, true>(w[2 * u], v[u], 0.0f), t = dot8<DT, true>(w[2 * u + 1], v[u], 0.0f);
          a += live[u] ? p : 0.0f;
          b += live[u] ? t : 0.0f;
        }
      }
      if (c < d.per_part) {
        r.need(2);
        const uint4 w = r.take(), t = r.take(), v = *reinterpret_cast<const uint4 *>(in + min(part.at, last));
        r.done();
        const float p = dot8<DT, true>(w, v, 0.0f), o = dot8<DT, true>(t, v, 0.0f);
        a += part.at <= last ? p : 0.0f;
        b += part.at <= last ? o : 0.0f;
      }
      a = wave_sum(a);
      b = wave_sum(b);
      if (lane == 0) {
        sums[2 * q] = a;
        sums[2 * q + 1] = b;
      }
    }
  }
}

// N loads of two words each, past the L1, and their wait. (A word's value and tag arrive together; two words need not.)
template <int N>
__device__ __forceinline__ void load_words(const uint64_t *base, const uint32_t (&at)[N], u32x4_t (&v)[N]) {
  static_assert(N >= 1 && N <= 5, "");
  if constexpr (N == 1)
    asm volatile("global_load_dwordx4 %0, %1, %2 sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(v[0]) : "v"(at[0]), "s"(base) : "memory");
  else if constexpr (N == 2)
    asm volatile("global_load_dwordx4 %0, %2, %4 sc1\n\tglobal_load_dwordx4 %1, %3, %4 sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1])
                 : "v"(at[0]), "v"(at[1]), "s"(base)
                 : "memory");
  else if constexpr (N == 3)
    asm volatile("global_load_dwordx4 %0, %3, %6 sc1\n\tglobal_load_dwordx4 %1, %4, %6 sc1\n\tglobal_load_dwordx4 %2, %5, %6 sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2])
                 : "v"(at[0]), "v"(at[1]), "v"(at[2]), "s"(base)
                 : "memory");
  else if constexpr (N == 4)
    asm volatile("global_load_dwordx4 %0, %4, %8 sc1\n\tglobal_load_dwordx4 %1, %5, %8 sc1\n\tglobal_load_dwordx4 %2, %6, %8 sc1\n\t"
                 "global_load_dwordx4 %3, %7, %8 sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
                 : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "s"(base)
                 : "memory");
  else
    asm volatile("global_load_dwordx4 %0, %5, %10 sc1\n\tglobal_load_dwordx4 %1, %6, %10 sc1\n\tglobal_load_dwordx4 %2, %7, %10 sc1\n\t"
                 "global_load_dwordx4 %3, %8, %10 sc1\n\tglobal_load_dwordx4 %4, %9, %10 sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4])
                 : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "v"(at[4]), "s"(base)
                 : "memory");
}
// Of `pairs` pairs of words those at thread + i * 512.
template <int N>
__device__ __forceinline__ void poll_pairs(const uint64_t *src, uint32_t pairs, uint32_t tag, Waiter &wait, u32x4_t (&v)[N]) {
  uint32_t spins = 0;
  bool ok;
  const uint32_t thread = fresh_thread();
  uint32_t at[N];
#pragma unroll
  for (int i = 0; i < N; ++i) at[i] = min(thread + i * kThreads, pairs - 1) * 16u;
  do {
    load_words<N>(src, at, v);
    ok = true;
#pragma unroll
    for (int i = 0; i < N; ++i) ok = ok && v[i].y == tag && v[i].w == tag;
  } while (wait.again(ok, spins));
}
// Packed 16-bit pairs into LDS.
template <int N>
__device__ __forceinline__ void take_pairs_n(const uint64_t *src, uint32_t pairs, uint32_t tag, Waiter &wait, uint16_t *dst) {
  u32x4_t v[N];
  poll_pairs<N>(src, pairs, tag, wait, v);
  const uint32_t thread = fresh_thread();
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (thread + i * kThreads < pairs) reinterpret_cast<uint2 *>(dst)[thread + i * kThreads] = make_uint2(v[i].x, v[i].z);
}
__device__ __forceinline__ void take_pairs(const uint64_t *src, uint32_t words, uint32_t tag, Waiter &wait, uint16_t *dst) {
  uint32_t pairs = words / 2;
  for (;;) {
    if (pairs <= 1u * kThreads) return take_pairs_n<1>(src, pairs, tag, wait, dst);
    if (pairs <= 2u * kThreads) return take_pairs_n<2>(src, pairs, tag, wait, dst);
    if (pairs <= 3u * kThreads) return take_pairs_n<3>(src, pairs, tag, wait, dst);
    take_pairs_n<5>(src, min(pairs, 5u * kThreads), tag, wait, dst);
    if (pairs <= 5u * kThreads) return;
    pairs -= 5u * kThreads;
    src += 2 * 5 * kThreads;
    dst += 4 * 5 * kThreads;
  }
}

template <uint32_t DT, int HD, int G, bool PARTS>
__global__ __launch_bounds__(kThreads + kLoaders *kWave, 1) void step_wide_kernel(ChainLaunch p) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  auto &sh = *reinterpret_cast<WideShared<HD, G, PARTS> *>(smem);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  Model m = (Model)(reinterpret_cast<uint64_t>(p.model));
  const uint32_t pos = scalar_load(m->state), step = scalar_load(m->state + 2);
  if (pos >= m->max_steps) return;
  if (p.withhold != 0 && blockIdx.x == 0 && scalar_load(m->state + 5) < p.withhold) return;
  const uint32_t stages = m->layers * kStages;
  if (threadIdx.x < sizeof(Flags) / 4) reinterpret_cast<uint32_t *>(&sh.flags)[threadIdx.x] = 0;
  __syncthreads();
  const uint32_t flags = lds_at(&sh.flags);
  if (wave >= kWaves) {
    load_ahead(m, stages, p.rounds, smem + p.ring_at, flags);
    return;
  }
  Meet meet{flags, 0};
  Reader reader{0, 0, 0, p.rounds, smem + p.ring_at + wave * kRequest + (fresh_thread() & (kWave - 1)) * 16, flags + static_cast<uint32_t>(offsetof(Flags, arrived)) + wave / kPer * 4,
                flags + static_cast<uint32_t>(offsetof(Flags, used)) + wave * 4};
  uint16_t *const x16 = reinterpret_cast<uint16_t *>(smem + p.row_at), *const in16 = reinterpret_cast<uint16_t *>(&sh.attn);
  WideStage d = read_stage(m, 0);
  const uint32_t own0 = blockIdx.x * m->hidden >> kLogWorkgroups, own1 = (blockIdx.x + 1) * m->hidden >> kLogWorkgroups;

  uint32_t nblk, bps, active;
  chain_splits<kWaves>(m->kv_heads, pos, kWorkgroups, nblk, bps, active);
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
  // test hook: where a layer's vectors go (as in step_chain.hip)
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

  // A row of x or r as it comes (`first`: the token's embedding), pairs of elements thread + i * 512: normalised into x16, the
  // workgroup's own elements kept.
  uint32_t turn = 0;
  const auto take_row = [&](auto n_, const uint64_t *src, const uint16_t *gamma, uint32_t tag, float *own, bool first, char *raw) {
    constexpr int N = decltype(n_)::value, kAtOnce = N <= 5 ? N : N / 2;
    const uint32_t pairs = m->hidden / 2, thread = fresh_thread();
    uint32_t g[N];
#pragma unroll
    for (int i = 0; i < N; ++i) g[i] = *at_bytes(reinterpret_cast<const uint32_t *>(gamma), min(thread + i * kThreads, pairs - 1) * 4u);   // (asked for before the wait)
    float v[2 * N];
    if (first) {
      uint32_t token = pos < scalar_load(m->state + 1) ? m->prompt[pos] : m->slots[pos - 1].token;
      if (token >= m->vocab) token = 0;   // prompts are validated on the host; sampled ids are < vocab
      const uint32_t *row = reinterpret_cast<const uint32_t *>(m->emb + static_cast<uint64_t>(token) * m->hidden);
#pragma unroll
      for (int i = 0; i < N; ++i) unpack2<DT>(row[min(thread + i * kThreads, pairs - 1)], v[2 * i], v[2 * i + 1]);
    } else {
#pragma unroll
      for (int from = 0; from < N; from += kAtOnce) {
        u32x4_t w[kAtOnce];
        const uint32_t skip = from * kThreads;
        // (a row that ends within the first half asks for its last words again)
        const uint32_t at = min(skip, pairs - 1);
        poll_pairs<kAtOnce>(src + 2 * at, pairs - at, tag, wait, w);
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i) {
          v[2 * (from + i)] = __uint_as_float(w[i].x);
          v[2 * (from + i) + 1] = __uint_as_float(w[i].z);
        }
      }
    }
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (thread + i * kThreads < pairs) ss = fmaf(v[2 * i], v[2 * i], fmaf(v[2 * i + 1], v[2 * i + 1], ss));
    ss = wave_sum(ss);
    if (thread % kWave == 0) sh.red[turn][wave] = ss;
    meet();
    // (as in step_chain.hip: 1 / sqrt by the hardware's and a step of Newton's, but for means that it takes for zero and sums
    // that overflowed)
    const float4 r0 = *reinterpret_cast<const float4 *>(&sh.red[turn][0]), r1 = *reinterpret_cast<const float4 *>(&sh.red[turn][4]);
    const float mean = fmaf(((r0.x + r0.y) + (r0.z + r0.w)) + ((r1.x + r1.y) + (r1.z + r1.w)), m->inv_hidden, m->eps);
    const float rough = __builtin_amdgcn_rsqf(mean);
    float scale = fmaf(rough * 0.5f, fmaf(-mean * rough, rough, 1.0f), rough);
    if (__builtin_expect(!(scale <= FLT_MAX), 0)) scale = 1.0f / sqrtf(mean);
    turn ^= 1u;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const uint32_t c = thread + i * kThreads;
      if (c < pairs) {
        float g0, g1;
        unpack2<DT>(g[i], g0, g1);
        reinterpret_cast<uint32_t *>(x16)[c] = enc16<DT>(v[2 * i] * scale * g0) | (static_cast<uint32_t>(enc16<DT>(v[2 * i + 1] * scale * g1)) << 16);
        if (2 * c >= own0 && 2 * c < own1) own[2 * c - own0] = v[2 * i];
        if (2 * c + 1 >= own0 && 2 * c + 1 < own1) own[2 * c + 1 - own0] = v[2 * i + 1];
        if (raw != nullptr) reinterpret_cast<float2 *>(raw)[c] = make_float2(v[2 * i], v[2 * i + 1]);
      }
    }
    meet();
  };

#pragma unroll 1
  for (uint32_t at = 0; at < stages; ++at) {
    const uint32_t layer = at / kStages, stage = at % kStages;
    const uint32_t tag = step * 256u + layer + 1u;   // (never that of another step until 2^24 of them)
    fresh(m);
    const WideStage next = read_stage(m, min(at + 1, stages - 1));
    uint64_t *const words = m->words;
    if (at != 0) __builtin_amdgcn_s_sleep(kPause);
    if (stage == kQkv || stage == kGateUp) {
      const uint32_t per = (m->hidden / 2 + kThreads - 1) / kThreads;
      float *const own = sh.own[stage == kQkv ? 0 : 1];
      char *const raw = traces && blockIdx.x == 0 ? (at == 0 ? p.trace : stage == kGateUp ? trace_at(layer, 3) : nullptr) : nullptr;
#define NV_WIDE_ROW(N) take_row(std::integral_constant<int, N>{}, words + d.in_at, d.vec, tag, own, at == 0, raw)
      if (per <= 1) NV_WIDE_ROW(1);
      else if (per <= 2) NV_WIDE_ROW(2);
      else if (per <= 4) NV_WIDE_ROW(4);
      else if (per <= 5) NV_WIDE_ROW(5);
      else NV_WIDE_ROW(8);
#undef NV_WIDE_ROW
    } else {
      take_pairs(words + d.in_at, d.in_words, tag, wait, in16);
      meet();
    }
    const uint16_t *const in = stage == kO || stage == kDown ? in16 : x16;
    if (traces && blockIdx.x == 0)
      for (uint32_t i = fresh_thread(); i < d.cols; i += kThreads)
        reinterpret_cast<uint16_t *>(trace_at(layer, stage == kQkv ? 0 : stage == kO ? 2 : stage == kGateUp ? 4 : 5))[i] = in[i];
    uint64_t *const out = words + d.out_at;
    const bool final_ = at + 1 == stages;
    const Share s = share_of(d, stage);
    walk<DT>(reader, d, stage, s, in, sh.sums);
    meet();
    if (wave == 0) {
      const uint32_t parts = 1u << d.log_parts, lane = fresh_thread() & (kWave - 1);
      if (stage == kGateUp) {
        for (uint32_t t = lane; t < s.n / 2; t += kWave) {
          const float4 *sums = reinterpret_cast<const float4 *>(sh.sums) + t * parts;
          float4 y = sums[0];
          if (parts > 1) {   // (two parts of one pair of rows each)
            float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            for (uint32_t i = 0; i < parts / 2; ++i) {
              const float4 u = sums[i], v = sums[parts / 2 + i];
              a.x += u.x + u.z;
              a.y += u.y + u.w;
              a.z += v.x + v.z;
              a.w += v.y + v.w;
            }
            y = a;
          }
          const uint32_t low = enc16<DT>(gated(y.x, 1.0f) * y.y), high = enc16<DT>(gated(y.z, 1.0f) * y.w);
          store_word(out + s.first / 2 + t, low | (high << 16), tag);
        }
      } else {
        for (uint32_t t = lane; t < s.n; t += kWave) {
          const uint32_t row = s.first + t;
          float y = sh.sums[t * parts];
          for (uint32_t i = 1; i < parts; ++i) y += sh.sums[t * parts + i];
          if (stage == kQkv) {
            if (traces) reinterpret_cast<float *>(trace_at(layer, 1))[row] = y;
          } else {
            if (d.vec != nullptr) y += dec16<DT>(d.vec[row]);
            y += sh.own[stage == kO ? 0 : 1][t];
            if (traces && stage == kDown) reinterpret_cast<float *>(trace_at(layer, 6))[row] = y;
          }
          if (final_) m->x[row] = y;
          else store_tagged(out + row, y, stage == kDown ? tag + 1u : tag);
        }
      }
    }
    if (stage == kQkv) {
      fresh(m);
      if (attends) chain_attention<DT, HD, G, PARTS, kWaves>(m, layer, pos, kvh, split, nblk, bps, active, tag, wait, sh.cs, sh.attn, meet);
      if (active > 1) {   // (heads from the other end of the grid)
        for (uint32_t h = kWorkgroups - 1 - blockIdx.x; h < m->heads; h += kWorkgroups) chain_merge<DT, HD, kWaves>(m, h, active, tag, wait, sh.merge, meet);
      }
    }
    d = next;
  }
}

using Kernel = void (*)(ChainLaunch);
struct Variant {
  Kernel kernel;
  uint32_t shared, scratch;   // bytes of LDS in front of the row, and of those the attention's, where inputs lie as well
};
template <uint32_t DT, int HD, int G, bool PARTS>
Variant variant() {
  using S = WideShared<HD, G, PARTS>;
  return {step_wide_kernel<DT, HD, G, PARTS>, sizeof(S), static_cast<uint32_t>(sizeof(S) - offsetof(S, attn))};
}
template <uint32_t DT>
Variant variant_of(uint32_t head_dim, uint32_t group) {
  if (head_dim == 64) {
    if (group == 1) return variant<DT, 64, 1, true>();
    if (group == 2) return variant<DT, 64, 2, true>();
    if (group <= 4) return variant<DT, 64, 4, true>();
    return variant<DT, 64, 8, true>();
  }
  if (group == 1) return variant<DT, 128, 1, false>();
  if (group == 2) return variant<DT, 128, 2, false>();
  if (group == 3) return variant<DT, 128, 4, true>();
  if (group == 4) return variant<DT, 128, 4, false>();
  if (group < 8) return variant<DT, 128, 8, true>();
  return variant<DT, 128, 8, false>();
}
Variant variant_of(uint32_t dtype, uint32_t head_dim, uint32_t group) {
  return dtype == kBF16 ? variant_of<kBF16>(head_dim, group) : dtype == kF16 ? variant_of<kF16>(head_dim, group) : Variant{};
}
// Where the row and the ring lie in LDS, and the rounds there are.
struct Places {
  uint32_t row_at, ring_at, rounds;
};
Places places(const Variant &v, uint32_t hidden, uint32_t inputs) {
  Places p;
  p.row_at = (v.shared - v.scratch + std::max(v.scratch, 2 * inputs) + 15u) / 16u * 16u;
  p.ring_at = (p.row_at + 2 * hidden + kRequest - 1) / kRequest * kRequest;
  p.rounds = p.ring_at < kLdsBytes ? (kLdsBytes - p.ring_at) / kRound : 0u;
  return p;
}

}  // namespace

bool wide_takes(uint32_t dtype, uint32_t layers, uint32_t hidden, uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t ff) {
  if (!attn_matrix_cores(heads, kv_heads, head_dim) || heads > 512 || kv_heads > 32) return false;
  // Every workgroup has rows of o and down and pairs of gate and up, whole 16-byte pieces of them, no more of x than it keeps.
  if (layers == 0 || layers >= 255 || hidden < kWorkgroups || hidden > kWorkgroups * kMostOwn || hidden % 8 != 0 || ff < 2 * kWorkgroups || ff % 8 != 0) return false;
  // From 12 MB of weights a layer on (chain_takes ends at 10). 27 stacks drawn between 14 and 501 MB, widths of 768 to 3520, 40 /
  // 700 / 3000 keys: 0.85 of the launches' time on average, 0.71 the least; one is no faster (3520 x 8096, 27 heads of 128 on 27,
  // whose q, k and v are as long as its attention: 59.5 / 61.3 / 66.3 us a layer in launches, 59.7 / 62.1 / 66.1). Two and three
  // layers: from 64 MB each on, where 21 models, those of one layer among them, take 0.77 to 0.97 of the launches' time a step,
  // at 40 to 3000 keys (2 layers of 2048 x 6144 82.6 -> 67.0 us at 700 keys, 3 of 4096 x 12288 238 -> 223); smaller ones would
  // gain as well, and keep the launches. One layer: from 256 MB on, what the memory-side cache holds (4096 x 12288 96.6 -> 87.6,
  // 5120 x 13824 136 -> 116); of a smaller one the launches read the weights there, and past 2000 keys some are the faster steps
  // (1536 x 7000 51.6, 61.3 in one launch; 2560 x 7000 65.0, 66.2).
  const uint64_t weights = static_cast<uint64_t>(hidden) * (2 * heads + 2 * kv_heads) * head_dim + 3ull * hidden * ff;
  if (weights <= (layers >= 4 ? 6000000u : layers >= 2 ? 32000000u : 128000000u)) return false;
  const uint32_t rows = std::max((heads + 2 * kv_heads) * head_dim, 2 * ff + 2 * kWorkgroups);
  if ((rows + kWorkgroups - 1) / kWorkgroups > kMostSums) return false;
  const Variant v = variant_of(dtype, head_dim, heads / kv_heads);
  return v.kernel != nullptr && places(v, hidden, std::max(ff, heads * head_dim)).rounds >= kLeastRounds;
}

bool wide_resident(uint32_t dtype, uint32_t heads, uint32_t kv_heads, uint32_t head_dim) {
  const Variant v = variant_of(dtype, head_dim, heads / kv_heads);
  int device = 0, cus = 0, each = 0;
  if (v.kernel == nullptr || hipGetDevice(&device) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
      hipFuncSetAttribute(reinterpret_cast<const void *>(v.kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&each, reinterpret_cast<const void *>(v.kernel), kThreads + kLoaders * kWave, kLdsBytes) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return static_cast<uint64_t>(cus) * static_cast<uint64_t>(each) >= kWorkgroups;
}

void wide_stages(const ChainModel &m, uint32_t head_dim, const LayerDev &w, WideStage (&stage)[4]) {
  const uint32_t A = m.heads * head_dim;
  const uint16_t *const matrix[4] = {w.wqkv, w.wo, w.wgu, w.wdown}, *const vec[4] = {w.rms_attn, w.o_bias, w.rms_mlp, nullptr};
  const uint32_t cols[4] = {m.hidden, A, m.hidden, m.ff}, rows[4] = {(m.heads + 2 * m.kv_heads) * head_dim, m.hidden, m.ff, m.hidden};
  const uint32_t in_at[4] = {m.at_x, m.at_attn, m.at_r, m.at_ff}, out_at[4] = {m.at_qkv, m.at_r, m.at_ff, m.at_x};
  for (uint32_t i = 0; i < 4; ++i) {
    WideStage &s = stage[i];
    s = WideStage{};
    s.w = matrix[i];
    s.vec = vec[i];
    s.cols = cols[i];
    s.row_bytes = cols[i] * 2;
    s.rows = rows[i];
    s.up_bytes = i == kGateUp ? m.ff * s.row_bytes + m.pair_gap * 2 : 0u;
    s.in_at = in_at[i];
    s.in_words = i % 2 != 0 ? cols[i] / 2 : cols[i];
    s.out_at = out_at[i];
    // As many parts a row as make the fewest rounds of the largest share; fewer where that is the same.
    const uint32_t requests = (s.row_bytes + kRequest - 1) / kRequest, both = i == kGateUp ? 2 : 1;
    const uint32_t most = both * ((s.rows / both + kWorkgroups - 1) / kWorkgroups);
    uint32_t least = ~0u;
    for (uint32_t log = 0; log <= 3 && (most * both << log) <= kMostSums; ++log) {
      const uint32_t per = (requests + (1u << log) - 1) >> log, takes = ((most << log) + kWaves - 1) / kWaves * per;
      if (takes < least) {
        least = takes;
        s.log_parts = log;
        s.per_part = per;
      }
    }
  }
}

hipError_t launch_step_wide(uint32_t dtype, uint32_t head_dim, const ChainModel &m, const ChainLaunch &p, hipStream_t stream) {
  if (!wide_takes(dtype, m.layers, m.hidden, m.heads, m.kv_heads, head_dim, m.ff) || p.model == nullptr || m.words == nullptr || p.spin_limit == 0)
    return hipErrorInvalidValue;
  const Variant v = variant_of(dtype, head_dim, m.heads / m.kv_heads);
  const Places at = places(v, m.hidden, std::max(m.ff, m.heads * head_dim));
  ChainLaunch q = p;
  q.row_at = at.row_at;
  q.ring_at = at.ring_at;
  q.rounds = at.rounds;
  hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void *>(v.kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(v.kernel, dim3(kWorkgroups), dim3(kThreads + kLoaders * kWave), kLdsBytes, stream, q);
  return hipGetLastError();
}

}  // namespace nv
