// What the launches that hold a whole step's layers share (step_chain.hip, step_wide.hip): the model through the scalar path,
// bounded waits for tagged words, and the attention of one layer as its q, k and v arrive. W: waves of a workgroup that take
// part; Meet: their barrier.
#pragma once

#include <algorithm>
#include <type_traits>

#include "attn_tile.cuh"
#include "gemv_stream.cuh"
#include "step_chain.cuh"

namespace nv {

namespace chain {

using namespace attn;

// The model through the scalar path. `fresh` forgets what has been read of it, so that a stage holds what it uses and no more:
// held over the whole loop, the model's and the layer's words and the addresses made of them take more registers than there are.
typedef const __attribute__((address_space(4))) ChainModel *Model;
__device__ __forceinline__ void fresh(Model &m) { asm volatile("" : "+s"(m)); }
__device__ __forceinline__ uint32_t fresh_thread() {
  uint32_t t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}
// Member number `which` of a layer's weights.
enum : int { kRmsAttn = 0, kRmsMlp, kWqkv, kQNorm, kKNorm, kQBias, kKBias, kVBias, kWo, kOBias, kWgu, kWdown };
static_assert(sizeof(LayerDev) == 12 * sizeof(void *), "twelve pointers");
__device__ __forceinline__ const uint16_t *weight(Model m, uint32_t layer, int which) {
  typedef const uint16_t *Pointer;
  typedef const __attribute__((address_space(4))) Pointer *Constant;
  return ((Constant)(reinterpret_cast<uint64_t>(m->layer)))[layer * 12 + which];
}

// Elements through a uniform base and a 32-bit offset in bytes: one address instruction each.
template <typename T>
__device__ __forceinline__ T *at_bytes(T *base, uint32_t bytes) {
  typedef typename std::conditional<std::is_const<T>::value, const char, char>::type Byte;
  return reinterpret_cast<T *>(reinterpret_cast<Byte *>(base) + bytes);
}
__device__ __forceinline__ void store_word(uint64_t *at, uint32_t payload, uint32_t tag) {
  __hip_atomic_store(at, (static_cast<uint64_t>(tag) << 32) | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A wait for words: until every lane's tags are this launch's, or the limit is reached.
struct Waiter {
  uint32_t limit;     // 0: a wait has run out, nothing is waited for any more
  uint32_t *gave_up;
  __device__ __forceinline__ bool again(bool ok, uint32_t &spins) {
    if (__all(ok) || limit == 0) return false;
    if (++spins <= limit) return true;
    limit = 0;
    if ((threadIdx.x & (kWave - 1)) == 0) __hip_atomic_store(gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return false;
  }
};
template <int HD, int G, bool PARTS, int W>
struct ChainAttnShared {
  static constexpr int kRow = HD + 8;
  alignas(16) uint16_t qhl[(PARTS ? 3 : 2) * G][kRow];   // as in the step kernel (StepShared)
  float qdown[G];
  alignas(16) uint16_t knew[HD];
  alignas(16) uint16_t vnew[HD];
  float wm[W][G], wl[W][G];
  alignas(16) float wacc[W][G][HD];
};
template <int W>
struct ChainMergeShared {   // [thread sets][dim]: of 64 threads at the least
  alignas(16) float o[W][128];
  float m[W], l[W];
};
// Split geometry of a step: blocks a split, splits.
// (as many cache blocks as a split has waves in each: with twice as many 600 keys 72 us a step instead of 69 at 512 x 1376, four waves)
template <int W>
__device__ __forceinline__ void chain_splits(uint32_t kv_heads, uint32_t pos, uint32_t workgroups, uint32_t &nblk, uint32_t &bps, uint32_t &active) {
  nblk = pos / kKvBlockTokens + 1;
  uint32_t splits = 1;
  if (nblk > kChainSingleBlocks) splits = max(1u, min(min(kChainMaxSplits, workgroups / kv_heads), (nblk + W - 1) / W));
  bps = (nblk + splits - 1) / splits;
  active = (nblk + bps - 1) / bps;
}

// The attention of one (key head, split): its q, k and v as they arrive, the cache's tiles through the matrix cores (attn_tile),
// and the 16-bit output or, of several splits, the partial sums.
template <uint32_t DT, int HD, int G, bool PARTS, int W, typename Meet>
__device__ __forceinline__ void chain_attention(Model m_, uint32_t layer, uint32_t pos, uint32_t kvh, uint32_t split, uint32_t nblk, uint32_t bps,
                                                uint32_t active, uint32_t tag, Waiter &wait, const float *rotation, ChainAttnShared<HD, G, PARTS, W> &sh, Meet &meet) {
  constexpr uint32_t kThreads = W * kWave;
  Model p = m_;
  fresh(p);
  const int lane = fresh_thread() & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t A = p->heads * HD, KV = p->kv_heads * HD, n_keys = pos + 1, group = p->heads / p->kv_heads;
  const uint16_t *const q_norm = weight(p, layer, kQNorm), *const k_norm = weight(p, layer, kKNorm);
  const uint16_t *const q_bias = weight(p, layer, kQBias), *const k_bias = weight(p, layer, kKBias), *const v_bias = weight(p, layer, kVBias);
  const bool rotates = p->rope_freq != nullptr;
  const float eps = p->eps;
  const uint32_t b0 = split * bps, b1 = min(nblk, b0 + bps);
  const uint32_t new_block = pos / kKvBlockTokens, new_row = pos % kKvBlockTokens;
  const bool owns_new = new_block >= b0 && new_block < b1;
  const int pl = pair_of<HD>(lane);

  // the wave's first tile is on its way before anything is waited for
  uint4 kreg[HD / 32], vreg[HD / 32];
  const auto load_tile = [&](uint32_t block) {
    const uint64_t tile = kv_tile_offset(p->block_count, p->kv_heads, HD, layer, scalar_load(p->table + block), kvh);
#pragma unroll
    for (int i = 0; i < HD / 32; ++i) {
      kreg[i] = load_stream(p->k_cache + tile + i * 512 + lane * 8);
      vreg[i] = load_stream(p->v_cache + tile + i * 512 + lane * 8);
    }
  };
  uint32_t b = b0 + wave;
  if (b < b1) load_tile(b);

  // heads of this wave, of the group's queries, the key and the value
  constexpr int kMine = (G + 2 + W - 1) / W;
  uint32_t head[kMine];
  float b_0[kMine], b_1[kMine], g_0[kMine], g_1[kMine];
  const uint64_t *src[kMine];
#pragma unroll
  for (int i = 0; i < kMine; ++i) {
    head[i] = wave + i * W;
    const uint32_t h = min(head[i], group + 1);
    const uint32_t off = h < group ? (kvh * group + h) * HD : (h == group ? A : A + KV) + kvh * HD;
    src[i] = p->words + p->at_qkv + off + pl;
    const uint16_t *bias = h < group ? q_bias : h == group ? k_bias : v_bias;
    const uint16_t *gamma = h < group ? q_norm : h == group ? k_norm : nullptr;
    const uint32_t boff = (h < group ? kvh * group + h : kvh) * HD + pl;
    b_0[i] = bias != nullptr ? dec16<DT>(bias[boff]) : 0.0f;
    b_1[i] = bias != nullptr ? dec16<DT>(bias[boff + HD / 2]) : 0.0f;
    g_0[i] = gamma != nullptr ? dec16<DT>(gamma[pl]) : 1.0f;
    g_1[i] = gamma != nullptr ? dec16<DT>(gamma[pl + HD / 2]) : 1.0f;
  }
  const float rc = rotation[pl], rs = rotation[HD / 2 + pl];
  uint64_t v0[kMine], v1[kMine];
  {
    uint32_t spins = 0;
    bool ok;
    do {
#pragma unroll
      for (int i = 0; i < kMine; ++i) {
        v0[i] = load_tagged(src[i]);
        v1[i] = load_tagged(src[i] + HD / 2);
      }
      ok = true;
#pragma unroll
      for (int i = 0; i < kMine; ++i) ok = ok && tag_is(v0[i], tag) && tag_is(v1[i], tag);
    } while (wait.again(ok, spins));
  }
#pragma unroll
  for (int i = 0; i < kMine; ++i) {
    float x0 = tag_value(v0[i]), x1 = tag_value(v1[i]);
    const bool query = head[i] < group, key = head[i] == group;
    const bool norm = query ? q_norm != nullptr : key && k_norm != nullptr;
    const bool bias = query ? q_bias != nullptr : key ? k_bias != nullptr : v_bias != nullptr;
    if (head[i] < group + 2) {
      head_values<DT, HD>(x0, x1, bias, b_0[i], b_1[i], norm, g_0[i], g_1[i], rotates && (query || key), rc, rs, eps);
      if (query) {
        const float scale = kLog2e / sqrtf(static_cast<float>(HD));
        const uint32_t g = head[i];
        uint16_t h0, l0, h1, l1;
        x0 *= scale;
        x1 *= scale;
        if constexpr (PARTS) {
          uint16_t t0, t1;
          if constexpr (DT == kF16) {
            const int up = attn_query_exponent(wave_max(fmaxf(fabsf(x0), fabsf(x1))));
            x0 = ldexpf(x0, up);
            x1 = ldexpf(x1, up);
            if (lane == 0) sh.qdown[g] = ldexpf(1.0f, -up);
          }
          split16<DT>(x0, h0, l0, t0);
          split16<DT>(x1, h1, l1, t1);
          sh.qhl[2 * G + g][pl] = t0;
          sh.qhl[2 * G + g][pl + HD / 2] = t1;
        } else {
          split16<DT>(x0, h0, l0);
          split16<DT>(x1, h1, l1);
        }
        sh.qhl[g][pl] = h0;
        sh.qhl[g][pl + HD / 2] = h1;
        sh.qhl[G + g][pl] = l0;
        sh.qhl[G + g][pl + HD / 2] = l1;
      } else {
        uint16_t *row = key ? sh.knew : sh.vnew;
        row[pl] = enc16<DT>(x0);
        row[pl + HD / 2] = enc16<DT>(x1);
      }
    }
  }
  meet();
  if (owns_new && wave == W - 1) {   // the new row, in operand order
    const uint64_t tile = kv_tile_offset(p->block_count, p->kv_heads, HD, layer, scalar_load(p->table + new_block), kvh);
    if (lane < HD / 8)
      *reinterpret_cast<uint4 *>(p->k_cache + tile + kv_k_elem(HD, new_row, lane * 8)) = *reinterpret_cast<const uint4 *>(sh.knew + lane * 8);
#pragma unroll
    for (int i = 0; i < HD / kWave; ++i) {
      const uint32_t d = lane + i * kWave;
      p->v_cache[tile + kv_v_elem(HD, new_row, d)] = sh.vnew[d];
    }
  }
  // columns of heads that the group does not have are zero
  const int col = lane & 15, grp = lane >> 4;
  const bool has = col < G ? static_cast<uint32_t>(col) < group : col < 2 * G && static_cast<uint32_t>(col - G) < group;
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  uint4 qx[HD / 32], third[PARTS ? HD / 32 : 1];
  float down = 1.0f;
#pragma unroll
  for (int j = 0; j < HD / 32; ++j) {
    const uint4 q = *reinterpret_cast<const uint4 *>(&sh.qhl[has ? col : 0][j * 32 + grp * 8]);
    qx[j] = has ? q : zero;
    if constexpr (PARTS) {
      const bool own = has && col < G;
      const uint4 t = *reinterpret_cast<const uint4 *>(&sh.qhl[2 * G + (own ? col : 0)][j * 32 + grp * 8]);
      third[j] = own ? t : zero;
    }
  }
  if constexpr (PARTS && DT == kF16) down = has ? sh.qdown[col < G ? col : col - G] : 1.0f;

  float m = -INFINITY, l = 0.0f;
  f32x4_t acc[HD / 16];
#pragma unroll
  for (int s = 0; s < HD / 16; ++s) acc[s] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  for (; b < b1; b += W) {
    attn_tile<DT, HD, G, false, PARTS, PARTS && DT == kF16>(kreg, vreg, qx, nullptr, b, n_keys, col, grp, owns_new && b == new_block, new_row, sh.knew, sh.vnew, m, l, acc,
                                       down, third);
    if (b + W < b1) load_tile(b + W);
  }
  l += __shfl_xor(l, 16, kWave);
  l += __shfl_xor(l, 32, kWave);
#pragma unroll
  for (int s = 0; s < HD / 16; ++s) {
    float4 o;
    o.x = acc[s][0] + row_shl<G>(acc[s][0]);
    o.y = acc[s][1] + row_shl<G>(acc[s][1]);
    o.z = acc[s][2] + row_shl<G>(acc[s][2]);
    o.w = acc[s][3] + row_shl<G>(acc[s][3]);
    if (col < G) *reinterpret_cast<float4 *>(&sh.wacc[wave][col][s * 16 + grp * 4]) = o;
  }
  if (lane < G) {
    sh.wm[wave][lane] = m;
    sh.wl[wave][lane] = l;
  }
  meet();
  for (uint32_t e = threadIdx.x; e < group * (HD / 2); e += kThreads) {
    const uint32_t g = e / (HD / 2), d = e % (HD / 2) * 2;
    float M = -INFINITY;
#pragma unroll
    for (int i = 0; i < W; ++i) M = fmaxf(M, sh.wm[i][g]);
    float L = 0.0f, o0 = 0.0f, o1 = 0.0f;
#pragma unroll
    for (int i = 0; i < W; ++i) {
      const float mw = sh.wm[i][g], f = mw > -INFINITY ? attn_exp2(mw - M) : 0.0f;   // a wave without a tile
      L = fmaf(sh.wl[i][g], f, L);
      o0 = fmaf(sh.wacc[i][g][d], f, o0);
      o1 = fmaf(sh.wacc[i][g][d + 1], f, o1);
    }
    const uint32_t h = kvh * group + g;
    if (active == 1) {
      if (L > 0.0f && isfinite(L)) {
        o0 /= L;
        o1 /= L;
      }
      store_word(p->words + p->at_attn + (h * HD + d) / 2, enc16<DT>(o0) | (static_cast<uint32_t>(enc16<DT>(o1)) << 16), tag);
    } else {
      uint64_t *rec = p->words + p->at_part + (static_cast<uint64_t>(h) * kChainMaxSplits + split) * (HD + 2);
      store_tagged(rec + d, o0, tag);
      store_tagged(rec + d + 1, o1, tag);
      if (d == 0) {
        store_tagged(rec + HD, M, tag);
        store_tagged(rec + HD + 1, L, tag);
      }
    }
  }
  meet();   // (the scratch is the next input's place)
}

// One head's splits: the threads of a dimension take every (256 / HD)-th of them, in order, and meet in LDS.
template <uint32_t DT, int HD, int W, typename Meet>
__device__ __forceinline__ void chain_merge(Model m_, uint32_t h, uint32_t active, uint32_t tag, Waiter &wait, ChainMergeShared<W> &sh, Meet &meet) {
  constexpr uint32_t kThreads = W * kWave;
  Model p = m_;
  fresh(p);
  constexpr uint32_t kSets = kThreads / HD, kPer = kChainMaxSplits / kSets;
  const uint32_t thread = fresh_thread(), d = thread % HD, q = thread / HD;
  const uint64_t *rec = p->words + p->at_part + static_cast<uint64_t>(h) * kChainMaxSplits * (HD + 2);
  uint64_t av[kPer], mv[kPer], lv[kPer];
  uint32_t spins = 0;
  bool ok;
  do {
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
      const uint32_t r = min(q + i * kSets, active - 1) * ((HD + 2) * 8u);
      av[i] = load_tagged(at_bytes(rec, r + d * 8u));
      mv[i] = load_tagged(at_bytes(rec, r + HD * 8u));
      lv[i] = load_tagged(at_bytes(rec, r + HD * 8u + 8u));
    }
    ok = true;
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i)
      if (q + i * kSets < active) ok = ok && tag_is(av[i], tag) && tag_is(mv[i], tag) && tag_is(lv[i], tag);
  } while (wait.again(ok, spins));
  float M = -INFINITY, L = 0.0f, o = 0.0f;
#pragma unroll
  for (uint32_t i = 0; i < kPer; ++i)
    if (q + i * kSets < active) M = fmaxf(M, tag_value(mv[i]));
#pragma unroll
  for (uint32_t i = 0; i < kPer; ++i) {
    if (q + i * kSets < active) {
      const float f = attn_exp2(tag_value(mv[i]) - M);
      L = fmaf(tag_value(lv[i]), f, L);
      o = fmaf(tag_value(av[i]), f, o);
    }
  }
  sh.o[q][d] = o;
  if (d == 0) {
    sh.m[q] = M;
    sh.l[q] = L;
  }
  meet();
  if (threadIdx.x < HD / 2) {
    float Mt = -INFINITY, Lt = 0.0f, o0 = 0.0f, o1 = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < kSets; ++i) Mt = fmaxf(Mt, sh.m[i]);
#pragma unroll
    for (uint32_t i = 0; i < kSets; ++i) {
      const float f = sh.m[i] > -INFINITY ? attn_exp2(sh.m[i] - Mt) : 0.0f;
      Lt = fmaf(sh.l[i], f, Lt);
      o0 = fmaf(sh.o[i][2 * threadIdx.x], f, o0);
      o1 = fmaf(sh.o[i][2 * threadIdx.x + 1], f, o1);
    }
    if (Lt > 0.0f && isfinite(Lt)) {
      o0 /= Lt;
      o1 /= Lt;
    }
    store_word(p->words + p->at_attn + (h * HD) / 2 + threadIdx.x, enc16<DT>(o0) | (static_cast<uint32_t>(enc16<DT>(o1)) << 16), tag);
  }
  meet();
}

}  // namespace chain

}  // namespace nv
