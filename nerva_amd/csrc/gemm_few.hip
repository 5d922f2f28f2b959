// Multi-row projection for up to 32 token rows (a batch step, drafts to check) of matrices that a launch is over with in a few
// microseconds: there the chain of one launch counts, not the stream, and how many launches the layer has.
//
// A workgroup owns 16 weight rows (NR = 2: 32, or 16 gate rows and their 16 up rows) over the whole of K and its waves
// split K in blocks of 64 columns, so there are no K slices, no partial sums in memory and no launch that adds them. Both
// operands go from global memory straight into the registers the matrix cores read: a request covers 16 rows x 64 bytes, the
// next one the other halves of those cache lines (which has to find them in the L2: with streaming loads, which are not kept there,
// every line came from memory twice), and every request of a wave's first DEPTH blocks is out before the first is awaited. The waves' sums meet in LDS, in wave order.
// kFewNorm: the launch normalises its input itself - the f32 rows instead of X, with the norm's weight. A wave reads its
// columns of the rows, the waves' sums of squares meet in LDS while the weights are on their way, and the values are scaled and
// rounded in the operand registers: a launch and a round trip of X through memory less. Every workgroup reads all of the rows
// for that and rounds them, which is what limits it to 1024 columns, 16 tokens and a workgroup a CU.
// 6 rows, us of the launches before (in K slices and with the launch that adds them, but for the pairs) -> here: 4096 x 1024 7.9 -> 4.0,
// 1024 x 2048 7.2 -> 4.8, 1024 x 3072 9.0 -> 6.5, 3072 x 1024 pairs 7.8 -> 5.4; with the norm in front 10.0 -> 5.9 (4096 x 1024), 10.7 -> 7.6
// (pairs). What bounds it there is the chain: launch, one round trip to memory, two barriers.
#include "gemm_epilogue.cuh"

#include <algorithm>

namespace nv {

namespace {

constexpr int kFewK = 64;        // columns of a block: one cache line a row
constexpr int kFewRow = 20;      // floats between the tokens of a 16-row tile of sums in LDS (16 and padding)
enum : int { kFewOperand = 0, kFewNorm = 1 };

// Eight normalised values: in every workgroup all rows are rounded once more, and with enc16's integer steps that took 1.5 us of a launch.
template <uint32_t DT>
__device__ __forceinline__ u32x4_t few_norm8(const f32x4_t &a, const f32x4_t &b, float scale, const u32x4_t &gamma) {
  u32x4_t out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float g0, g1;
    unpack2<DT>(gamma[i], g0, g1);
    const f32x4_t &v = i < 2 ? a : b;
    const float y0 = v[i % 2 * 2] * scale * g0, y1 = v[i % 2 * 2 + 1] * scale * g1;
    out[i] = enc16_pair<DT>(y0, y1);
  }
  return out;
}

// TT: token tiles of 16 (1 or 2). NW: waves. DEPTH: blocks of a wave requested ahead (kFewNorm: all of them).
template <uint32_t DT, int EPI, int NR, int TT, int NW, int IN, int DEPTH>
__global__ __launch_bounds__(NW *kWave, NW / 4) void gemm_few_kernel(GemmRowsParams p) {
  static_assert(EPI != kGemmSwiglu || NR == 2, "a gate tile and its up tile");
  static_assert(IN != kFewNorm || TT == 1, "the normalised rows are held in registers");
  __shared__ __align__(16) float red[NW][NR][TT][16][kFewRow];
  __shared__ float squares[IN == kFewNorm ? NW : 1][16];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t n = lane & 15, q = lane >> 4;
  const uint32_t cols = p.cols, T = p.tokens, rows = p.rows;
  const uint32_t row0 = blockIdx.x * (EPI == kGemmSwiglu ? 16u : 16u * NR);
  const uint32_t nblk = cols / kFewK, mine = static_cast<uint32_t>(wave) < nblk ? (nblk - wave + NW - 1) / NW : 0u;   // blocks wave, wave + NW, ...

  const uint16_t *wp[NR];
#pragma unroll
  for (int j = 0; j < NR; ++j) {   // (rows past the matrix: its last one again, never stored)
    const uint32_t row = min(row0 + (EPI == kGemmSwiglu ? 0u : j * 16u) + n, rows - 1);
    const bool up = EPI == kGemmSwiglu && j == 1;
    wp[j] = p.w + static_cast<uint64_t>(up ? rows + row : row) * cols + (up ? p.pair_gap : 0u) + wave * kFewK + q * 8;
  }
  u32x4_t a[DEPTH][NR][2], x[DEPTH][TT][2];
  auto load_w = [&](int slot, uint32_t i) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int j = 0; j < NR; ++j)
        a[slot][j][e] = *reinterpret_cast<const u32x4_t *>(wp[j] + static_cast<uint64_t>(i) * (NW * kFewK) + e * 32);
  };
  f32x4_t acc[NR][TT];
#pragma unroll
  for (int j = 0; j < NR; ++j)
#pragma unroll
    for (int c = 0; c < TT; ++c) acc[j][c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](int slot) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int j = 0; j < NR; ++j)
#pragma unroll
        for (int c = 0; c < TT; ++c) acc[j][c] = mfma_k32<DT>(a[slot][j][e], x[slot][c][e], acc[j][c]);
  };

  if constexpr (IN == kFewNorm) {
    // (the launch rule: no wave has more than DEPTH blocks; a block that a wave does not have is read as its last and left out)
    const uint32_t t = min(n, T - 1);
    const float *row = p.norm_in + static_cast<uint64_t>(t) * cols + q * 8;
    const uint16_t *gamma = p.norm_in_gamma + q * 8;
    f32x4_t v[DEPTH][2][2];
    u32x4_t g[DEPTH][2];
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
      const uint32_t at = min(wave + i * static_cast<uint32_t>(NW), nblk - 1) * kFewK;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        v[i][e][0] = *reinterpret_cast<const f32x4_t *>(row + at + e * 32);
        v[i][e][1] = *reinterpret_cast<const f32x4_t *>(row + at + e * 32 + 4);
        g[i][e] = *reinterpret_cast<const u32x4_t *>(gamma + at + e * 32);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (mine == DEPTH) {
#pragma unroll
      for (int i = 0; i < DEPTH; ++i) load_w(i, i);
    } else {
#pragma unroll
      for (int i = 0; i < DEPTH; ++i)
        if (static_cast<uint32_t>(i) < mine) load_w(i, i);
    }
    __builtin_amdgcn_sched_barrier(0);
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
      float part = 0.0f;
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int r = 0; r < 4; ++r) part = fmaf(v[i][e][h][r], v[i][e][h][r], part);
      if (static_cast<uint32_t>(i) < mine) ss += part;
    }
    ss += __shfl_xor(ss, 16, kWave);
    ss += __shfl_xor(ss, 32, kWave);
    if (lane < 16) squares[wave][lane] = ss;
    // (not __syncthreads(): that waits for the weights as well)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    float total = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) total += squares[w][n];
    const float scale = 1.0f / sqrtf(total / static_cast<float>(cols) + p.norm_eps);
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
      if (static_cast<uint32_t>(i) < mine) {
#pragma unroll
        for (int e = 0; e < 2; ++e) x[i][0][e] = few_norm8<DT>(v[i][e][0], v[i][e][1], scale, g[i][e]);
        multiply(i);
      }
    }
  } else {
    const uint16_t *xp[TT];
#pragma unroll
    for (int c = 0; c < TT; ++c) {
      const uint32_t t = min(c * 16u + n, T - 1);   // lanes past the block's tokens read its last one again
      xp[c] = p.x16 + static_cast<uint64_t>(wave) * (2 * 512u) * p.x_packed + (t / 16u) * 512u + (q * 16u + t % 16u) * 8u;
    }
    const uint64_t x_step = 512u * p.x_packed;
    auto load = [&](int slot, uint32_t i) {
      load_w(slot, i);
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int c = 0; c < TT; ++c)
          x[slot][c][e] = *reinterpret_cast<const u32x4_t *>(xp[c] + (static_cast<uint64_t>(i) * (2 * NW) + e) * x_step);
    };
    if (mine >= DEPTH) {   // requests under no branch keep the compiler's waits exact
#pragma unroll
      for (int s = 0; s < DEPTH; ++s) load(s, s);
      uint32_t i = 0;
      for (; i + 2 * DEPTH <= mine; i += DEPTH) {
#pragma unroll
        for (int s = 0; s < DEPTH; ++s) {
          multiply(s);
          load(s, i + s + DEPTH);
        }
      }
      const uint32_t left = mine - i;   // DEPTH .. 2 DEPTH - 1
#pragma unroll
      for (int s = 0; s < DEPTH; ++s) {
        multiply(s);
        if (s + DEPTH < left) load(s, i + s + DEPTH);
      }
#pragma unroll
      for (int s = 0; s < DEPTH; ++s)
        if (s + DEPTH < left) multiply(s);
    } else {
#pragma unroll
      for (int s = 0; s < DEPTH; ++s)
        if (static_cast<uint32_t>(s) < mine) load(s, s);
#pragma unroll
      for (int s = 0; s < DEPTH; ++s)
        if (static_cast<uint32_t>(s) < mine) multiply(s);
    }
  }

  // ---- the waves' sums, four rows of a token a thread
#pragma unroll
  for (int j = 0; j < NR; ++j)
#pragma unroll
    for (int c = 0; c < TT; ++c) *reinterpret_cast<f32x4_t *>(&red[wave][j][c][n][q * 4]) = acc[j][c];
  __syncthreads();
  constexpr int kOutTiles = EPI == kGemmSwiglu ? 1 : NR;
  const uint32_t out = threadIdx.x / 64u, t = out % TT * 16u + n, j = out / TT;   // a wave an output tile: its sixteen tokens and four row groups
  if (j >= kOutTiles || t >= T) return;
  f32x4_t y{0.0f, 0.0f, 0.0f, 0.0f}, up{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    y += *reinterpret_cast<const f32x4_t *>(&red[w][j][out % TT][n][q * 4]);
    if constexpr (EPI == kGemmSwiglu) up += *reinterpret_cast<const f32x4_t *>(&red[w][1][out % TT][n][q * 4]);
  }
  const uint32_t row = row0 + j * 16u + q * 4u;
  if (row < rows) block_epilogue<DT, EPI>(p, t, row, y, up, epilogue_act<DT, EPI>(p));
}

// Waves: sixteen for the normalising launch (a block each), eight otherwise (a wave has its whole DEPTH in flight: 4096 x 1024
// 5.6 us with sixteen, 4.0 with eight). NR = 1 for plain projections (32 rows a workgroup: 4.6, and 11.9 against 8.6 at 4096 x 4096).
template <uint32_t DT, int EPI>
hipError_t launch_epi(const GemmRowsParams &p, uint32_t workgroups, hipStream_t stream) {
  constexpr int NR = EPI == kGemmSwiglu ? 2 : 1;
  const dim3 grid(workgroups);
  if (p.norm_in != nullptr) hipLaunchKernelGGL((gemm_few_kernel<DT, EPI, NR, 1, 16, kFewNorm, 1>), grid, dim3(16 * kWave), 0, stream, p);
  else if (p.tokens <= 16) hipLaunchKernelGGL((gemm_few_kernel<DT, EPI, NR, 1, 8, kFewOperand, 4>), grid, dim3(8 * kWave), 0, stream, p);
  else hipLaunchKernelGGL((gemm_few_kernel<DT, EPI, NR, 2, 8, kFewOperand, 4>), grid, dim3(8 * kWave), 0, stream, p);
  return hipGetLastError();
}
template <uint32_t DT>
hipError_t launch_dt(int epilogue, const GemmRowsParams &p, uint32_t workgroups, hipStream_t stream) {
  switch (epilogue) {
    case kGemmF32: return launch_epi<DT, kGemmF32>(p, workgroups, stream);
    case kGemmResidual: return launch_epi<DT, kGemmResidual>(p, workgroups, stream);
    case kGemmSwiglu: return launch_epi<DT, kGemmSwiglu>(p, workgroups, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

uint32_t gemm_few_workgroups(int epilogue, uint32_t rows, uint32_t cols, uint32_t tokens) {
  if (tokens == 0 || tokens > kGemmFewMaxTokens || epilogue == kGemmXielu || rows % 4 != 0 || rows < 16 || cols % kFewK != 0) return 0;
  return (rows + 15u) / 16u;
}

// What a CU fetches of W and X at the rate one is served at (52 KiB a us up to 8 tokens, 46 to 16, 44 with two token tiles) and 2.5 us
// for the start of the second workgroup where there are more than CUs, or W at the rate of memory. (Plain projections and pairs of 2 to 32 rows
// as measured: 0.73 to 1.04 times this for nine in ten. One rate of 54 up to 16 tokens and no second start fell short of 7168 x 5120 by a
// fourth and of pairs of 5120 x 2048 by a third, at 9 to 16 tokens.)
double gemm_few_us(int epilogue, uint32_t rows, uint32_t cols, uint32_t tokens) {
  const double pair = epilogue == kGemmSwiglu ? 2.0 : 1.0, tiles = tokens > 16 ? 2.0 : 1.0;
  const uint32_t rounds = ((rows + 15u) / 16u + 255u) / 256u;
  const double a_cu = rounds * (pair + tiles) * 16.0 * cols * 2.0 / 1024.0;
  return 3.0 + (rounds > 1 ? 2.5 : 0.0) + std::max(a_cu / (tokens > 16 ? 44.0 : tokens > 8 ? 46.0 : 52.0), pair * rows * cols * 2.0 / 6.3e6);
}

hipError_t launch_gemm_few(uint32_t dtype, int epilogue, const GemmRowsParams &p, hipStream_t stream) {
  const uint32_t workgroups = gemm_few_workgroups(epilogue, p.rows, p.cols, p.tokens);
  if (workgroups == 0 || p.x_packed == 0) return hipErrorInvalidValue;
  if (dtype == kBF16) return launch_dt<kBF16>(epilogue, p, workgroups, stream);
  if (dtype == kF16) return launch_dt<kF16>(epilogue, p, workgroups, stream);
  return hipErrorInvalidValue;
}

}  // namespace nv
