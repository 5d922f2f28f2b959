// Attention of a prompt block: consecutive positions of one sequence (up to 512, or a pass of up to 4096) in one launch, every
// K/V tile of the prefix fetched once per workgroup and used by all its tokens.
// Reference: the chunked prefill's attention (session_decode_prefill.inc.cu:1879-2243) over the
// arithmetic of exact_blockwise_attention_into (attention/exact/run.rs:13-127) per token; the rows
// of the block itself are in the cache already (launch_kv_publish_rows), so token t simply attends to
// keys 0 .. position + t.
//
// gfx950 mapping (head_dim 64 or 128, G = heads / kv_heads up to 8): a wave fills two 16-column matrix-core tiles with
// (token, head) pairs - 32 / G tokens of the kv head's G query heads - and the hi and lo halves of a query (and of a
// step's probabilities) are two products into the same accumulators, with the causal limit n_keys chosen per column.
// The 8 waves of a (wide) workgroup take 8 * 32 / G consecutive tokens and walk the SAME keys, 64 a step: the step's four K and
// four V tiles (one each per wave) go from the cache straight into a ring of four LDS stages, two steps ahead.
// What bounds it is the matrix cores and the exponentials beside them, so a step is laid out for both: 64 keys share one
// running maximum, one rescale and one look at the mask (only steps that reach the diagonal have one), every K or V piece
// read from LDS meets 32 columns, the product with V contracts over two tiles at once with the full-rate 32-deep
// instruction - the operand order of the cache keeps a lane's four tokens of a tile side by side, so the pair's operand is
// a choice of registers - and the two waves of a SIMD take turns: one multiplies while the other works on its
// probabilities, kept half a step apart by two barriers a step. Against 16 keys a step, 16 columns a wave
// and the 16-deep product, blocks of 512 tokens of 32 heads over contexts 512 to 8192: 111.8 -> 82.7 us a launch on
// average (85.8 without the turns), 0.94 PFLOP/s with the hi and lo halves counted, where the products of the same block
// reach 1.1.
// Prompts of less than some 3000 tokens do not fill the chip with such workgroups, and each of them is long: queries of 256
// pairs prepared by four SIMDs (half of a short launch), then 3.3 to 4 us a step. The narrow workgroup has four waves of one
// column tile: a quarter of the work for each SIMD, two workgroups a CU with two LDS stages each, and no
// turns - the other workgroup's wave fills in. The same sums in the same order (32 heads on 8, 146 tokens 20.8 -> 11.4 us, 512 tokens in four splits 38 ->
// 18.7 in one, 1024 tokens 64.7 -> 34.2; prompt_shape has the line between the two).
// Grid (kv head, split of the prefix, token group, the last one first); split partials go to the per-token workspaces the decode kernel uses
// and a small second launch merges them.
#include <algorithm>
#include <mutex>

#include "attn_decode.cuh"
#include "attn_tile.cuh"

namespace nv {

namespace {

using namespace attn;

// A workgroup's waves and the 16-column tiles of (token, head) pairs each of them has.
constexpr int kWideWaves = 8, kWideTiles = 2;
constexpr int kNarrowWaves = 4, kNarrowTiles = 1;
constexpr uint32_t kStepBlocks = 4;   // cache blocks (16 keys) of a step
constexpr int stages_of(int waves) { return waves == kWideWaves ? 4 : 2; }
constexpr uint32_t group_tokens_of(bool wide, uint32_t group) {
  return wide ? kWideWaves * (kWideTiles * 16u / group) : kNarrowWaves * (kNarrowTiles * 16u / group);
}

// Split geometry of a token group, the same on both launches: blocks per split (whole steps), active splits.
__device__ __forceinline__ void prompt_splits(uint32_t last_pos, uint32_t S, uint32_t &bps, uint32_t &active, uint32_t &nblk) {
  nblk = last_pos / kKvBlockTokens + 1;
  bps = ((nblk + S - 1) / S + kStepBlocks - 1) / kStepBlocks * kStepBlocks;
  active = (nblk + bps - 1) / bps;
}

constexpr uint32_t prompt_tile_bytes(int hd) { return kKvBlockTokens * hd * 2u; }
constexpr uint32_t prompt_stage_bytes(int hd) { return 2u * kStepBlocks * prompt_tile_bytes(hd); }

#define NV_PR_LDS(P) ((__attribute__((address_space(3))) void *)(P))

// Operand reads, issued one group ahead of the products that use them and awaited by count: the awaited registers are
// in/out operands of the wait, so that nothing that uses them can come before it.
#define NV_PR_READ(DST, AT, OFF) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(DST) : "v"(AT), "n"(OFF) : "memory")
#define NV_PR_AWAIT2(N_, A_, B_) asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(A_), "+v"(B_) : "n"(N_) : "memory")

template <uint32_t DT>
__device__ __forceinline__ bool finite16(uint16_t bits) { return (bits & 0x7fffu) < (DT == kBF16 ? 0x7f80u : 0x7c00u); }

template <uint32_t DT, int HD, int G, int PW, int NC>
__global__ __launch_bounds__(PW *kWave, 2) void attn_prompt_kernel(AttnParams p) {
  constexpr int kCols = 16 * NC, kStages = stages_of(PW);
  constexpr int kTokensPerWave = kCols / G, kPairs = kTokensPerWave * G;   // (columns kPairs .. kCols - 1 repeat the last pair, unused)
  constexpr uint32_t kGroupTokens = PW * kTokensPerWave;
  constexpr int kWaveTiles = 2 * kStepBlocks / PW;   // K/V tiles of a step that a wave fetches
  constexpr int kPieces = HD / 32;               // 1 KiB pieces of a tile
  constexpr uint32_t kTile = prompt_tile_bytes(HD), kStage = prompt_stage_bytes(HD);
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t kvh = blockIdx.x, split = blockIdx.y, S = gridDim.y, T = p.tokens;
  const uint32_t group_first = (gridDim.z - 1 - blockIdx.z) * kGroupTokens;   // the longest prefix first
  const uint32_t group_last = min(T, group_first + kGroupTokens) - 1;
  uint32_t bps, active, nblk;
  prompt_splits(p.position + group_last, S, bps, active, nblk);
  if (split >= active) return;
  const uint32_t b0 = split * bps, steps = (min(nblk, b0 + bps) - b0 + kStepBlocks - 1) / kStepBlocks;

  // this wave's tiles of a step, wave, wave + PW, ...: K (even ones) or V of block tile / 2; blocks past the last are that one
  // again, masked
  const uint16_t *cache = (wave & 1) == 0 ? p.k_cache : p.v_cache;
  auto request = [&](uint32_t step) {
#pragma unroll
    for (int n = 0; n < kWaveTiles; ++n) {
      const uint32_t tile = wave + n * PW;
      const uint32_t block = min(b0 + step * kStepBlocks + (tile >> 1), nblk - 1);
      const uint16_t *src = cache + kv_tile_offset(p.block_count, p.kv_heads, HD, p.layer, scalar_load(p.table + block), kvh) + lane * 8;
      unsigned char *at = smem + (step % kStages) * kStage + tile * kTile;
#pragma unroll
      for (int i = 0; i < kPieces; ++i)
        __builtin_amdgcn_global_load_lds(reinterpret_cast<const u32x4_t *>(src + i * 512), NV_PR_LDS(at + i * 1024), 16, 0, 0);
    }
  };

  // ---- this wave's (token, head) pairs: bias, norm, rotation -> hi and lo operands. A lane fetches what it will hold of
  // its column's pair, eight dims of every 32: both ends of each rotation are among them, the sum of squares takes two
  // exchanges, and every input of the wave's pairs is requested at once.
  const uint32_t wave_first = group_first + wave * kTokensPerWave;   // may lie past the block: clamped, never stored
  const int col = lane & 15, grp = lane >> 4;
  u32x4_t qhi[NC][kPieces], qlo[NC][kPieces];
  uint32_t n_keys[NC];
  constexpr bool kScaled = attn_scaled<DT, HD, G>();
  float down[NC];   // undoes the scale of the column's query
  {
    constexpr int kHalf = kPieces / 2;   // pieces of a rotation's first ends
    const bool has_bias = p.q_bias != nullptr, has_gamma = p.q_norm != nullptr, has_rope = p.rope_freq != nullptr;
    const uint16_t *bias_base = has_bias ? p.q_bias : p.k_cache;    // any readable address when unused
    const float *rope_base = has_rope ? p.rope_cs : p.qkv;
    const uint32_t rope_stride = has_rope ? p.rope_token_stride : 0u;
    const uint16_t *gamma_base = has_gamma ? p.q_norm : p.k_cache;
    f32x4_t x[NC][kPieces][2], rc[NC][kHalf][2], rs[NC][kHalf][2];
    u32x4_t bias[NC][kPieces], gamma[kPieces];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int vh = min(c * 16 + col, kPairs - 1);
      const uint32_t tok = min(wave_first + vh / G, T - 1);
      const uint32_t h = kvh * G + vh % G;
      const float *src = p.qkv + static_cast<uint64_t>(tok) * p.qkv_token_stride + h * HD + grp * 8;
      const float *rope = rope_base + static_cast<uint64_t>(tok) * rope_stride + grp * 8;
#pragma unroll
      for (int j = 0; j < kPieces; ++j) {
#pragma unroll
        for (int i = 0; i < 2; ++i) x[c][j][i] = *reinterpret_cast<const f32x4_t *>(src + j * 32 + i * 4);
        bias[c][j] = *reinterpret_cast<const u32x4_t *>(bias_base + h * HD + j * 32 + grp * 8);
      }
#pragma unroll
      for (int j = 0; j < kHalf; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          rc[c][j][i] = *reinterpret_cast<const f32x4_t *>(rope + j * 32 + i * 4);
          rs[c][j][i] = *reinterpret_cast<const f32x4_t *>(rope + HD / 2 + j * 32 + i * 4);
        }
      n_keys[c] = p.position + tok + 1;   // causal limit of the column
    }
#pragma unroll
    for (int j = 0; j < kPieces; ++j) gamma[j] = *reinterpret_cast<const u32x4_t *>(gamma_base + j * 32 + grp * 8);
    __builtin_amdgcn_sched_barrier(0);
    request(0);   // the first tiles behind the inputs, on their way while the queries are prepared
    if (steps > 1) request(1);
    __builtin_amdgcn_sched_barrier(0);
    const auto elem16 = [](const u32x4_t &v, int e) { return dec16<DT>(static_cast<uint16_t>(v[e / 2] >> (16 * (e % 2)))); };
    const float scale = kLog2e / sqrtf(static_cast<float>(HD));
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float y[kPieces][8], ss = 0.0f;
#pragma unroll
      for (int j = 0; j < kPieces; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          y[j][e] = x[c][j][e / 4][e % 4];
          if (has_bias) y[j][e] += elem16(bias[c][j], e);
          ss += y[j][e] * y[j][e];
        }
      if (has_gamma) {
        ss += __shfl_xor(ss, 16, kWave);
        ss += __shfl_xor(ss, 32, kWave);
        const float norm = 1.0f / sqrtf(ss / static_cast<float>(HD) + p.eps);
#pragma unroll
        for (int j = 0; j < kPieces; ++j)
#pragma unroll
          for (int e = 0; e < 8; ++e) y[j][e] *= norm * elem16(gamma[j], e);
      }
      if (has_rope) {
#pragma unroll
        for (int j = 0; j < kHalf; ++j)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float y0 = y[j][e], y1 = y[j + kHalf][e], co = rc[c][j][e / 4][e % 4], si = rs[c][j][e / 4][e % 4];
            y[j][e] = y0 * co - y1 * si;
            y[j + kHalf][e] = y1 * co + y0 * si;
          }
      }
      float up = scale;
      down[c] = 1.0f;
      if constexpr (kScaled) {
        float largest = 0.0f;
#pragma unroll
        for (int j = 0; j < kPieces; ++j)
#pragma unroll
          for (int e = 0; e < 8; ++e) largest = fmaxf(largest, fabsf(y[j][e]));
        largest = fmaxf(largest, __shfl_xor(largest, 16, kWave));
        largest = fmaxf(largest, __shfl_xor(largest, 32, kWave));
        const int shift = attn_query_exponent(largest * scale);
        up = ldexpf(scale, shift);
        down[c] = ldexpf(1.0f, -shift);
      }
#pragma unroll
      for (int j = 0; j < kPieces; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          uint16_t h0, l0, h1, l1;
          split16<DT>(y[j][2 * e] * up, h0, l0);
          split16<DT>(y[j][2 * e + 1] * up, h1, l1);
          qhi[c][j][e] = h0 | (static_cast<uint32_t>(h1) << 16);
          qlo[c][j][e] = l0 | (static_cast<uint32_t>(l1) << 16);
        }
    }
  }
  const bool wave_on = wave_first < T;
  const uint32_t least_keys = p.position + min(wave_first, T - 1) + 1;                            // of any column of the wave,
  const uint32_t most_keys = p.position + min(wave_first + kTokensPerWave - 1, T - 1) + 1;        // and the most of any

  float m[NC], l[NC];
  f32x4_t acc[NC][HD / 16];   // O^T[dims s*16 + grp*4 .. +3][column]
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    m[c] = -INFINITY;
    l[c] = 0.0f;
#pragma unroll
    for (int s2 = 0; s2 < HD / 16; ++s2) acc[c][s2] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(NV_PR_LDS(smem))) + lane * 16u;

  // ---- the three parts of a step (skipped where no column of the wave sees it)
  f32x4_t sc[NC][kStepBlocks];   // scores of keys key0 + 16 t + 4 grp + r, then the bits of their probabilities: two words hi, two lo
  auto sees = [&](uint32_t step) { return wave_on && (b0 + step * kStepBlocks) * kKvBlockTokens < most_keys; };
  auto scores = [&](uint32_t step) {
    if (!sees(step)) return;
    const uint32_t at = lds0 + (step % kStages) * kStage;
    u32x4_t k[2][kPieces];
#pragma unroll
    for (int j = 0; j < kPieces; ++j) NV_PR_READ(k[0][j], at, j * 1024);
#pragma unroll
    for (uint32_t t = 0; t < kStepBlocks; ++t) {
      if (t + 1 < kStepBlocks) {
#pragma unroll
        for (int j = 0; j < kPieces; ++j) NV_PR_READ(k[(t + 1) & 1][j], at, (t + 1) * 2 * kTile + j * 1024);
      }
#pragma unroll
      for (int j = 0; j < kPieces; j += 2) {
        if (t + 1 < kStepBlocks) NV_PR_AWAIT2(kPieces, k[t & 1][j], k[t & 1][j + 1]);
        else NV_PR_AWAIT2(0, k[t & 1][j], k[t & 1][j + 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < NC; ++c) sc[c][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < kPieces; ++j)
#pragma unroll
        for (int c = 0; c < NC; ++c) sc[c][t] = mfma_k32<DT>(k[t & 1][j], qhi[c][j], sc[c][t]);
#pragma unroll
      for (int j = 0; j < kPieces; ++j)
#pragma unroll
        for (int c = 0; c < NC; ++c) sc[c][t] = mfma_k32<DT>(k[t & 1][j], qlo[c][j], sc[c][t]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto softmax = [&](uint32_t step) {
    if (!sees(step)) return;
    const uint32_t key0 = (b0 + step * kStepBlocks) * kKvBlockTokens;
    if (key0 + kStepBlocks * kKvBlockTokens > least_keys) {   // some column ends inside this step (or before it)
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (uint32_t t = 0; t < kStepBlocks; ++t)
#pragma unroll
          for (uint32_t r = 0; r < 4; ++r) sc[c][t][r] = key0 + t * 16u + grp * 4u + r < n_keys[c] ? sc[c][t][r] : -INFINITY;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float mb = fmaxf(fmaxf(sc[c][0][0], sc[c][0][1]), fmaxf(sc[c][0][2], sc[c][0][3]));
#pragma unroll
      for (uint32_t t = 1; t < kStepBlocks; ++t) mb = fmaxf(fmaxf(mb, fmaxf(sc[c][t][0], sc[c][t][1])), fmaxf(sc[c][t][2], sc[c][t][3]));
      mb = fmaxf(mb, __shfl_xor(mb, 16, kWave));
      mb = fmaxf(mb, __shfl_xor(mb, 32, kWave));
      if constexpr (kScaled) mb *= down[c];
      const float m_new = fmaxf(m[c], mb);
      const float m_ref = fmaxf(m_new, -3.0e38f);   // a column with nothing to see yet: exponentials against a finite stand-in
      const float alpha = attn_exp2(m[c] - m_ref);
      const float m_low = kScaled ? m_ref - kAttnWeightShift : m_ref;
      float psum = 0.0f;
#pragma unroll
      for (uint32_t t = 0; t < kStepBlocks; ++t) {
        float e[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) e[r] = attn_exp2(kScaled ? fmaf(sc[c][t][r], down[c], -m_low) : sc[c][t][r] - m_low);
        psum += (e[0] + e[1]) + (e[2] + e[3]);
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          uint16_t h0, l0, h1, l1;
          split16<DT>(e[r], h0, l0);
          split16<DT>(e[r + 1], h1, l1);
          sc[c][t][r / 2] = __uint_as_float(h0 | (static_cast<uint32_t>(h1) << 16));
          sc[c][t][2 + r / 2] = __uint_as_float(l0 | (static_cast<uint32_t>(l1) << 16));
        }
      }
      l[c] = l[c] * alpha + psum;
      m[c] = m_new;
      if (__any(alpha != 1.0f)) {
#pragma unroll
        for (int s2 = 0; s2 < HD / 16; ++s2) acc[c][s2] *= alpha;
      }
    }
  };
  // O^T += V^T . P, two tiles of keys at a time
  auto values = [&](uint32_t step) {
    if (!sees(step)) return;
    const uint32_t at = lds0 + (step % kStages) * kStage + kTile;
    u32x4_t v[2][2];   // a piece of each of the two tiles, this group's and the next one's
    NV_PR_READ(v[0][0], at, 0);
    NV_PR_READ(v[0][1], at, 2 * kTile);
    constexpr int kGroups = 2 * kPieces;   // (pair of tiles, piece)
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      if (g + 1 < kGroups) {
        NV_PR_READ(v[(g + 1) & 1][0], at, ((g + 1) / kPieces) * 4 * kTile + ((g + 1) % kPieces) * 1024);
        NV_PR_READ(v[(g + 1) & 1][1], at, ((g + 1) / kPieces) * 4 * kTile + 2 * kTile + ((g + 1) % kPieces) * 1024);
        NV_PR_AWAIT2(2, v[g & 1][0], v[g & 1][1]);
      } else {
        NV_PR_AWAIT2(0, v[g & 1][0], v[g & 1][1]);
      }
      __builtin_amdgcn_sched_barrier(0);
      const int pair = g / kPieces, j = g % kPieces;
      const u32x4_t &a = v[g & 1][0], &b = v[g & 1][1];
      const u32x4_t lo_slab = {a[0], a[1], b[0], b[1]}, hi_slab = {a[2], a[3], b[2], b[3]};
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const u32x4_t pa = __builtin_bit_cast(u32x4_t, sc[c][2 * pair]), pb = __builtin_bit_cast(u32x4_t, sc[c][2 * pair + 1]);
        const u32x4_t bh = {pa[0], pa[1], pb[0], pb[1]};
        acc[c][2 * j] = mfma_k32<DT>(lo_slab, bh, acc[c][2 * j]);
        acc[c][2 * j + 1] = mfma_k32<DT>(hi_slab, bh, acc[c][2 * j + 1]);
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const u32x4_t pa = __builtin_bit_cast(u32x4_t, sc[c][2 * pair]), pb = __builtin_bit_cast(u32x4_t, sc[c][2 * pair + 1]);
        const u32x4_t bl = {pa[2], pa[3], pb[2], pb[3]};
        acc[c][2 * j] = mfma_k32<DT>(lo_slab, bl, acc[c][2 * j]);
        acc[c][2 * j + 1] = mfma_k32<DT>(hi_slab, bl, acc[c][2 * j + 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- the walk, in two phases a step: while waves 0..3 (one a SIMD) multiply, waves 4..7 work on their probabilities, and
  // the other way round. Phase 2k: first half V(k-1) and K(k), second half softmax(k-1); phase 2k+1: first half
  // softmax(k), second half V(k-1) and K(k). A stage is free when the second half has left V of its step, two phases
  // before it is filled again.
  // With one wave a SIMD nobody takes turns: a step's three parts follow one another, behind one barrier - which also says
  // that the stage of the step before is free.
  const bool first_half = wave < PW / 2;
  if constexpr (PW != kWideWaves) {
    for (uint32_t k = 0; k < steps; ++k) {
      if (k == 0 && steps > 1) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kPieces * kWaveTiles) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
      if (k > 0 && k + 1 < steps) request(k + 1);
      scores(k);
      softmax(k);
      values(k);
    }
  } else
  for (uint32_t k = 0; k <= steps; ++k) {
    // this wave's part of step k has arrived (step k + 1 may be on its way)
    if (k + 1 < steps) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kPieces) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    if (k + 2 < steps) request(k + 2);
    if (!first_half) {
      if (k > 0) softmax(k - 1);
      asm volatile("s_barrier" ::: "memory");
    }
    if (k > 0) values(k - 1);
    if (k < steps) scores(k);
    if (first_half) {
      asm volatile("s_barrier" ::: "memory");
      if (k < steps) softmax(k);
    }
  }
  if (!wave_on) return;

  // ---- results of the wave's pairs: token rows of the four lane groups
  const uint64_t ml_off = reinterpret_cast<char *>(p.part_m) - reinterpret_cast<char *>(p.part_acc);
  const uint64_t l_off = reinterpret_cast<char *>(p.part_l) - reinterpret_cast<char *>(p.part_acc);
  uint32_t spoilt[NC];   // columns with a sum that is not finite
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    float zero = 0.0f;
#pragma unroll
    for (int s2 = 0; s2 < HD / 16; ++s2)
#pragma unroll
      for (int r = 0; r < 4; ++r) zero = fmaf(acc[c][s2][r], 0.0f, zero);
    const uint64_t lanes = __ballot(zero != 0.0f);   // (NaN)
    spoilt[c] = static_cast<uint32_t>(lanes | (lanes >> 16) | (lanes >> 32) | (lanes >> 48)) & 0xffffu;
  }
  const auto any_spoilt = [&] { return (spoilt[0] | spoilt[NC - 1]) != 0; };
  if (any_spoilt()) {
    // 0 x NaN or infinity is NaN: a value that is not finite may have come in by a key that the column does not see - of a
    // later token of its step, or a row not written yet. Where there is such a value behind the least limit of the wave's
    // columns, their sums are formed once more below, over the keys they see.
    uint32_t found = 0;
    for (uint32_t b = max(b0, least_keys / kKvBlockTokens); b < nblk; ++b) {
      const uint16_t *tile = p.v_cache + kv_tile_offset(p.block_count, p.kv_heads, HD, p.layer, p.table[b], kvh) + lane * 8;
#pragma unroll
      for (int i = 0; i < kPieces * 8; ++i) found |= finite16<DT>(tile[i / 8 * 512 + i % 8]) ? 0u : 1u;
    }
    if (!__any(found != 0)) spoilt[0] = spoilt[NC - 1] = 0;
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    float lc = l[c];
    lc += __shfl_xor(lc, 16, kWave);
    lc += __shfl_xor(lc, 32, kWave);
    l[c] = lc;
    const int pair = c * 16 + col;
    const uint32_t tok = wave_first + pair / G, h = kvh * G + pair % G;
    if (pair >= kPairs || tok >= T) continue;
    const float inv = lc > 0.0f && isfinite(lc) ? 1.0f / lc : 1.0f;
    char *ws = reinterpret_cast<char *>(p.part_acc) + static_cast<uint64_t>(tok) * p.ws_token_stride;
    if (((spoilt[c] >> col) & 1u) == 0) {
#pragma unroll
      for (int s2 = 0; s2 < HD / 16; ++s2) {
        const float4 o = make_float4(acc[c][s2][0], acc[c][s2][1], acc[c][s2][2], acc[c][s2][3]);
        const uint32_t d = s2 * 16 + grp * 4;
        if (active == 1) {
          // a single split holds every key: final
          uint2 packed;
          packed.x = enc16<DT>(o.x * inv) | (static_cast<uint32_t>(enc16<DT>(o.y * inv)) << 16);
          packed.y = enc16<DT>(o.z * inv) | (static_cast<uint32_t>(enc16<DT>(o.w * inv)) << 16);
          *reinterpret_cast<uint2 *>(p.out16 + attn_out_token(p, tok) + attn_out_elem(p, h * HD + d)) = packed;   // d % 4 == 0
        } else {
          *reinterpret_cast<float4 *>(reinterpret_cast<float *>(ws) + (static_cast<uint64_t>(h) * S + split) * HD + d) = o;
        }
      }
    }
    if (active != 1 && grp == 0) {
      reinterpret_cast<float *>(ws + ml_off)[h * S + split] = m[c];
      reinterpret_cast<float *>(ws + l_off)[h * S + split] = lc;
    }
  }
  // ---- the sums of spoilt columns, one after the other: the query again (a lane has a rotation's two ends), scores of 64
  // keys at a time (a lane a key), then their values in key order (a lane its two dims)
  if (__builtin_expect(!any_spoilt(), 1)) return;
  for (int pair = 0; pair < kPairs; ++pair) {
    const uint32_t tok = wave_first + pair / G, h = kvh * G + pair % G;
    if ((((pair < 16 ? spoilt[0] : spoilt[NC - 1]) >> (pair % 16)) & 1u) == 0 || tok >= T) continue;
    const int at = pair_of<HD>(lane);
    const float *src = p.qkv + static_cast<uint64_t>(tok) * p.qkv_token_stride + h * HD;
    const float *rope = p.rope_freq != nullptr ? p.rope_cs + static_cast<uint64_t>(tok) * p.rope_token_stride : p.qkv;
    const bool has_bias = p.q_bias != nullptr, has_gamma = p.q_norm != nullptr;
    float q0 = src[at], q1 = src[at + HD / 2];
    head_values<DT, HD>(q0, q1, has_bias, has_bias ? dec16<DT>(p.q_bias[h * HD + at]) : 0.0f,
                        has_bias ? dec16<DT>(p.q_bias[h * HD + at + HD / 2]) : 0.0f, has_gamma, has_gamma ? dec16<DT>(p.q_norm[at]) : 0.0f,
                        has_gamma ? dec16<DT>(p.q_norm[at + HD / 2]) : 0.0f, p.rope_freq != nullptr, rope[at], rope[HD / 2 + at], p.eps);
    const float scale = kLog2e / sqrtf(static_cast<float>(HD));
    q0 *= scale;
    q1 *= scale;
    const float most = __shfl(pair < 16 ? m[0] : m[NC - 1], pair % 16, kWave), sum = __shfl(pair < 16 ? l[0] : l[NC - 1], pair % 16, kWave);
    const uint32_t end = min((b0 + steps * kStepBlocks) * kKvBlockTokens, p.position + tok + 1);
    float o0 = 0.0f, o1 = 0.0f;
    for (uint32_t k0 = b0 * kKvBlockTokens; k0 < end; k0 += kWave) {
      const uint32_t key = min(k0 + lane, end - 1);
      const uint64_t tile = kv_tile_offset(p.block_count, p.kv_heads, HD, p.layer, p.table[key / kKvBlockTokens], kvh);
      float score = 0.0f;
      for (uint32_t d = 0; d < HD / 2; ++d) {
        score = fmaf(__shfl(q0, d, kWave), dec16<DT>(p.k_cache[tile + kv_k_elem(HD, key % kKvBlockTokens, d)]), score);
        score = fmaf(__shfl(q1, d, kWave), dec16<DT>(p.k_cache[tile + kv_k_elem(HD, key % kKvBlockTokens, d + HD / 2)]), score);
      }
      const float weight = attn_exp2(score - (kScaled ? most - kAttnWeightShift : most));
      for (uint32_t i = 0; i < min(end - k0, static_cast<uint32_t>(kWave)); ++i) {
        const uint64_t row = kv_tile_offset(p.block_count, p.kv_heads, HD, p.layer, p.table[(k0 + i) / kKvBlockTokens], kvh);
        const float w = __shfl(weight, i, kWave);
        o0 = fmaf(w, dec16<DT>(p.v_cache[row + kv_v_elem(HD, (k0 + i) % kKvBlockTokens, at)]), o0);
        o1 = fmaf(w, dec16<DT>(p.v_cache[row + kv_v_elem(HD, (k0 + i) % kKvBlockTokens, at + HD / 2)]), o1);
      }
    }
    if (lane >= HD / 2) continue;
    if (active == 1) {
      const float inv = sum > 0.0f && isfinite(sum) ? 1.0f / sum : 1.0f;
      uint16_t *out = p.out16 + attn_out_token(p, tok);
      out[attn_out_elem(p, h * HD + at)] = enc16<DT>(o0 * inv);
      out[attn_out_elem(p, h * HD + at + HD / 2)] = enc16<DT>(o1 * inv);
    } else {
      float *part = reinterpret_cast<float *>(reinterpret_cast<char *>(p.part_acc) + static_cast<uint64_t>(tok) * p.ws_token_stride) +
                    (static_cast<uint64_t>(h) * S + split) * HD;
      part[at] = o0;
      part[at + HD / 2] = o1;
    }
  }
}
#undef NV_PR_LDS
#undef NV_PR_READ
#undef NV_PR_AWAIT2

// Second launch: grid (head, token), one lane per dim; splits in order, kRound of them requested at a time
// (4 where the launch has no more splits than that: the same sums in the same order with a quarter of the loads).
template <uint32_t DT, int HD, int kRound>
__global__ __launch_bounds__(HD) void attn_prompt_merge_kernel(AttnParams p, uint32_t S, uint32_t group_tokens) {
  const uint32_t h = blockIdx.x, tok = blockIdx.y, d = threadIdx.x;
  const uint32_t group_last = min(p.tokens, (tok / group_tokens + 1) * group_tokens) - 1;
  uint32_t bps, active, nblk;
  prompt_splits(p.position + group_last, S, bps, active, nblk);
  if (active == 1) return;   // the first launch wrote the final rows
  const char *ws = reinterpret_cast<const char *>(p.part_acc) + static_cast<uint64_t>(tok) * p.ws_token_stride;
  const float *acc = reinterpret_cast<const float *>(ws) + static_cast<uint64_t>(h) * S * HD + d;
  const float *pm = reinterpret_cast<const float *>(ws + (reinterpret_cast<const char *>(p.part_m) - reinterpret_cast<const char *>(p.part_acc))) + h * S;
  const float *pl = reinterpret_cast<const float *>(ws + (reinterpret_cast<const char *>(p.part_l) - reinterpret_cast<const char *>(p.part_acc))) + h * S;
  // rounds of kRound splits, every load of a round unconditional (index clamped) and in flight at once
  float M = -INFINITY, L = 0.0f, o = 0.0f;
  for (uint32_t s0 = 0; s0 < active; s0 += kRound) {
    float mm[kRound], ll[kRound], aa[kRound];
#pragma unroll
    for (int i = 0; i < kRound; ++i) {
      const uint32_t si = min(s0 + i, active - 1);
      mm[i] = pm[si];
      ll[i] = pl[si];
      aa[i] = acc[static_cast<uint64_t>(si) * HD];
    }
    float Mc = M;
#pragma unroll
    for (int i = 0; i < kRound; ++i) {
      // a split past this token's position saw no key: m = -inf, and its accumulator may hold anything
      const bool on = s0 + i < active && mm[i] > -INFINITY;
      mm[i] = on ? mm[i] : -INFINITY;
      ll[i] = on ? ll[i] : 0.0f;
      aa[i] = on ? aa[i] : 0.0f;
      Mc = fmaxf(Mc, mm[i]);
    }
    const float keep = M > -INFINITY ? attn_exp2(M - Mc) : 0.0f;
    L *= keep;
    o *= keep;
#pragma unroll
    for (int i = 0; i < kRound; ++i) {
      const float f = mm[i] > -INFINITY ? attn_exp2(mm[i] - Mc) : 0.0f;
      L = fmaf(ll[i], f, L);
      o = fmaf(aa[i], f, o);
    }
    M = Mc;
  }
  if (L > 0.0f && isfinite(L)) o /= L;
  p.out16[attn_out_token(p, tok) + attn_out_elem(p, h * HD + d)] = enc16<DT>(o);
}

template <uint32_t DT, int HD, int G, int PW, int NC>
hipError_t launch_shape(const AttnParams &p, uint32_t splits, hipStream_t stream) {
  constexpr size_t lds = static_cast<size_t>(stages_of(PW)) * prompt_stage_bytes(HD);
  // more than the default dynamic LDS limit: raised once per kernel (never under stream capture)
  static std::once_flag once;
  static hipError_t raised = hipSuccess;
  std::call_once(once, [] {
    raised = hipFuncSetAttribute(reinterpret_cast<const void *>(&attn_prompt_kernel<DT, HD, G, PW, NC>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
  });
  if (raised != hipSuccess) return raised;
  constexpr uint32_t group_tokens = PW * (16 * NC / G);
  hipLaunchKernelGGL((attn_prompt_kernel<DT, HD, G, PW, NC>), dim3(p.kv_heads, splits, (p.tokens + group_tokens - 1) / group_tokens),
                     dim3(PW * kWave), lds, stream, p);
  return hipGetLastError();
}
template <uint32_t DT, int HD, int G>
hipError_t launch_group(const AttnParams &p, bool wide, uint32_t splits, hipStream_t stream) {
  return wide ? launch_shape<DT, HD, G, kWideWaves, kWideTiles>(p, splits, stream) : launch_shape<DT, HD, G, kNarrowWaves, kNarrowTiles>(p, splits, stream);
}

template <uint32_t DT, int HD>
hipError_t launch_hd(const AttnParams &p, bool wide, uint32_t splits, hipStream_t stream) {
  const uint32_t group = p.heads / p.kv_heads, group_tokens = group_tokens_of(wide, group);
  hipError_t err = hipSuccess;
  switch (group) {
    case 1: err = launch_group<DT, HD, 1>(p, wide, splits, stream); break;
    case 2: err = launch_group<DT, HD, 2>(p, wide, splits, stream); break;
    case 3: err = launch_group<DT, HD, 3>(p, wide, splits, stream); break;
    case 4: err = launch_group<DT, HD, 4>(p, wide, splits, stream); break;
    case 5: err = launch_group<DT, HD, 5>(p, wide, splits, stream); break;
    case 6: err = launch_group<DT, HD, 6>(p, wide, splits, stream); break;
    case 7: err = launch_group<DT, HD, 7>(p, wide, splits, stream); break;
    default: err = launch_group<DT, HD, 8>(p, wide, splits, stream); break;
  }
  if (err != hipSuccess || splits == 1) return err;
  if (splits <= 4)
    hipLaunchKernelGGL((attn_prompt_merge_kernel<DT, HD, 4>), dim3(p.heads, p.tokens), dim3(HD), 0, stream, p, splits, group_tokens);
  else
    hipLaunchKernelGGL((attn_prompt_merge_kernel<DT, HD, 16>), dim3(p.heads, p.tokens), dim3(HD), 0, stream, p, splits, group_tokens);
  return hipGetLastError();
}

template <uint32_t DT>
hipError_t launch_dt(const AttnParams &p, bool wide, uint32_t splits, hipStream_t stream) {
  return p.head_dim == 64 ? launch_hd<DT, 64>(p, wide, splits, stream) : launch_hd<DT, 128>(p, wide, splits, stream);
}

}  // namespace

namespace {

struct PromptShape {
  bool wide;
  uint32_t splits;
  double us;   // of the launch and its merge
};
// A launch's time: its start (queries, first tiles), and the longest workgroup's steps or, past the workgroups the chip holds
// at once (one wide one a CU, two narrow ones, the longest first), all of them and a share of the longest's. A merge costs a
// launch, and the partial sums' way to memory and back. Fitted on heads of 128 (32 on 8, tokens x first position, us):
//                  146 x 0   512 x 0   88 x 512   512 x 512   1024 x 0   2048 x 0   4096 x 0   4096 x 4096   8 x 4096
//   wide             20.8      38.6       29.3        44.5       64.7        116        241          607        23.5
//   narrow           11.4      18.7       19.2        31.3       34.2         89        267          723        13
// (wide in four or more splits where that is better, as it was before there were narrow ones.) Heads of 64, and of 128 with any number of query heads a
// key head, go by the same constants, too high for heads of 64 on both sides: of 260 launches drawn over both, 1 to 8 query heads a key head, 2 to 4096
// tokens behind 0 to 8000, none is slower than with wide workgroups alone, and all take 7.3 ms instead of 13.4 (64 wide, 4 of a key head: 18 tokens
// 10.2 -> 5.9 us, 267 tokens 18.7 -> 9.8; 128 wide, 7 of a key head: 140 tokens 21.3 -> 11.2, 2902 tokens 152 -> 119).
PromptShape shape_at(bool wide, uint32_t splits, uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t position, uint32_t tokens) {
  const uint32_t group_tokens = group_tokens_of(wide, heads / kv_heads), groups = (tokens + group_tokens - 1) / group_tokens;
  constexpr uint32_t kKeys = kStepBlocks * kKvBlockTokens;
  const double longest = ((position + tokens - 1) / kKeys + splits) / splits;
  const double workgroups = static_cast<double>(kv_heads) * groups * splits;
  const double all = static_cast<double>(kv_heads) * groups * ((position + std::min(tokens, (tokens + group_tokens) / 2)) / kKeys + 1.0);
  const double path = wide ? 3.3 : workgroups <= 256 ? 1.45 : 1.7;
  const double steps = std::max(path * longest, wide ? 3.0 * all / 256 + 0.3 * longest : 1.7 * all / 512 + 0.6 * longest);
  const double merge = splits == 1 ? 0.0 : 3.0 + static_cast<double>(tokens) * heads * head_dim * splits * 4 / 1.4e6;
  return PromptShape{wide, splits, (wide ? 12.0 : 7.0) + steps + merge};
}
// The best of both shapes and of splits 1, 2, 4, ... (splits != 0: that many).
PromptShape prompt_shape(uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t position, uint32_t tokens, uint32_t splits) {
  const int forced = tuning(kTunePromptWaves);
  const uint32_t most = std::min(kAttnMaxSplits, (position + tokens - 1) / (kStepBlocks * kKvBlockTokens) + 1);
  PromptShape best{true, 1, 1e30};
  for (const bool wide : {true, false}) {
    if (forced == (wide ? kNarrowWaves : kWideWaves)) continue;
    for (uint32_t s = splits != 0 ? std::min(splits, most) : 1u; s <= most; s *= 2) {
      const PromptShape shape = shape_at(wide, s, heads, kv_heads, head_dim, position, tokens);
      if (shape.us < best.us) best = shape;
      if (splits != 0) break;
    }
  }
  return best;
}

}  // namespace

// Several blocks in one launch have no splits: that, or a launch a block with as many as are best for it.
uint32_t attn_prompt_launch_tokens(uint32_t heads, uint32_t kv_heads, uint32_t head_dim, uint32_t position, uint32_t tokens, uint32_t block) {
  if (tokens <= block) return tokens;
  const double together = prompt_shape(heads, kv_heads, head_dim, position, tokens, 1).us;
  double apart = 0.0;
  for (uint32_t at = 0; at < tokens && apart < together; at += block)
    apart += prompt_shape(heads, kv_heads, head_dim, position + at, std::min(block, tokens - at), 0).us;
  return together <= apart ? tokens : block;
}

hipError_t launch_attn_prompt(uint32_t dtype, const AttnParams &p, hipStream_t stream) {
  if (p.qkv == nullptr || p.k_cache == nullptr || p.v_cache == nullptr || p.table == nullptr || p.out16 == nullptr ||
      p.part_acc == nullptr || p.part_m == nullptr || p.part_l == nullptr)
    return hipErrorInvalidValue;
  if (!attn_matrix_cores(p.heads, p.kv_heads, p.head_dim) || p.tokens == 0 || p.tokens > 65535 || p.block_count == 0)
    return hipErrorInvalidValue;
  if (static_cast<uint64_t>(p.position) + p.tokens > static_cast<uint64_t>(p.block_count) * kKvBlockTokens)
    return hipErrorInvalidValue;
  if (p.rope_freq != nullptr && p.rope_cs == nullptr) return hipErrorInvalidValue;   // rotation tables per token row
  if (p.out_packed_tiles != 0 && p.out_packed_tiles * 16u < p.tokens) return hipErrorInvalidValue;
  const PromptShape shape = prompt_shape(p.heads, p.kv_heads, p.head_dim, p.position, p.tokens, std::min<uint32_t>(p.splits, kAttnMaxSplits));
  if (dtype == kBF16) return launch_dt<kBF16>(p, shape.wide, shape.splits, stream);
  if (dtype == kF16) return launch_dt<kF16>(p, shape.wide, shape.splits, stream);
  return hipErrorInvalidValue;
}

}  // namespace nv
