// Multi-row projection for token blocks of up to 128 rows (X in matrix-operand order) of any number of weight rows and
// any K that is a multiple of 32: the shapes whose K does not divide into the rings of gemm_block.hip (a width of 896 or
// 1344, a vocabulary of any size), or not into enough slices of them (a feed-forward of 9728 or 18944).
//
// What bounds it is the weight stream, so a workgroup keeps as much of it in flight as LDS holds: the K-blocks of 64
// columns - 64 RT weight rows of 128 bytes and the block's X pieces - go from global memory straight into a ring of
// LDS stages (global_load_lds_dwordx4, no registers), kDepth - 1 blocks ahead, with two workgroups a CU (RT = 1: 40 to
// 60 KiB of W in flight a CU, RT = 2: 96). A request covers 8 rows x 128 bytes, whole cache lines; the 16-byte pieces
// of a row are XORed with the row number (mod 8) on the way in, which makes the operand reads conflict-free. One
// barrier a K-block: a wave waits until its own requests of the block are in, everyone meets, the stage of the block
// before is free and takes the requests of the block kDepth - 1 ahead.
// K slices are runs of whole K-blocks, as even as they come (any count: K need not divide); rows past the matrix and
// columns past K are fetched again from its last row or column and never multiplied into anything that is stored.
#include "gemm_epilogue.cuh"

#include <algorithm>
#include <mutex>

namespace nv {

namespace {

constexpr int kFW = 4;                        // waves per workgroup: they split the rows
constexpr int kFK = 64;                       // columns per K-block
constexpr uint32_t kFTokCap = 128;            // token rows at most; the token stride of the partial sums
constexpr int kFWTile = 16 * kFK * 2;         // bytes of 16 rows of a K-block: 2 KiB

constexpr int flow_stage_bytes(int tt, int rt) { return kFW * rt * kFWTile + 2 * tt * 1024; }
// Stages that fit two workgroups into a CU's 160 KiB, or one where that would leave fewer than three
constexpr int flow_depth(int tt, int rt) {
  const int two = 80 * 1024 / flow_stage_bytes(tt, rt);
  return std::min(6, two >= 3 ? two : 160 * 1024 / flow_stage_bytes(tt, rt));
}

#define NV_FLOW_LDS(P) ((__attribute__((address_space(3))) void *)(P))

// Waits until at most N of this wave's requests are outstanding.
template <int N>
__device__ __forceinline__ void wait_requests() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Grid (row groups, K slices). TT: token tiles of the block (x_packed). RT: row tiles a wave (SwiGLU: a gate tile and its
// up tile). A workgroup has 64 RT rows of W (SwiGLU: 64 gate and 64 up rows).
template <uint32_t DT, int EPI, int TT, int RT>
__global__ __launch_bounds__(kFW *kWave, TT == 8 && RT == 2 ? 1 : 2) void gemm_flow_kernel(GemmRowsParams p, float *partials) {
  static_assert(EPI != kGemmSwiglu || RT == 2, "a gate tile and its up tile");
  constexpr int kStage = flow_stage_bytes(TT, RT), kDepth = flow_depth(TT, RT);
  constexpr int kWReq = 2 * RT, kXReq = TT / 2, kReq = kWReq + kXReq;   // requests of a wave and K-block, 1 KiB each
  static_assert(kDepth >= 3 && (kDepth - 2) * kReq <= 63, "the wait counter holds 63 requests");
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t n = lane & 15, q = lane >> 4;
  const uint32_t cols = p.cols, T = p.tokens, rows = p.rows;
  const uint32_t slices = gridDim.y, all = (cols + kFK - 1) / kFK;
  const uint32_t first = blockIdx.y * all / slices, last = (blockIdx.y + 1) * all / slices, nblk = last - first;

  // first output row of this wave's tile j (SwiGLU: tile 1 is the up tile of the same outputs)
  uint32_t trow[RT];
#pragma unroll
  for (int j = 0; j < RT; ++j)
    trow[j] = EPI == kGemmSwiglu ? blockIdx.x * (16u * kFW) + wave * 16u : blockIdx.x * (16u * kFW * RT) + (wave * RT + j) * 16u;
  // W request i: rows 8 (i % 2) .. + 7 of tile i / 2; lane (r, c) asks for piece c ^ r of row r
  const char *wsrc[kWReq];
#pragma unroll
  for (int i = 0; i < kWReq; ++i) {
    const uint32_t row = min(trow[i / 2] + (i % 2) * 8u + (lane >> 3), rows - 1);
    const bool up = EPI == kGemmSwiglu && i / 2 == 1;
    wsrc[i] = reinterpret_cast<const char *>(p.w) +
              (static_cast<uint64_t>(up ? rows + row : row) * cols + (up ? p.pair_gap : 0u)) * sizeof(uint16_t);
  }
  const uint32_t wpiece = static_cast<uint32_t>((lane & 7) ^ (lane >> 3)) * 16u, wlast = cols * 2u - 16u;
  // X request i: piece wave * kXReq + i of the block's 2 TT (K-step, token tile) pieces
  const uint32_t ksteps = cols / 32u;
  const char *xsrc = reinterpret_cast<const char *>(p.x16) + lane * 16u;

  f32x4_t acc[RT][TT];
#pragma unroll
  for (int j = 0; j < RT; ++j)
#pragma unroll
    for (int c = 0; c < TT; ++c) acc[j][c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  auto request = [&](uint32_t b, uint32_t stage) {
    unsigned char *at = smem + stage * kStage;
    const uint32_t blk = first + b;
    const uint32_t woff = min(blk * (kFK * 2u) + wpiece, wlast);
#pragma unroll
    for (int i = 0; i < kWReq; ++i)
      __builtin_amdgcn_global_load_lds(reinterpret_cast<const u32x4_t *>(wsrc[i] + woff), NV_FLOW_LDS(at + (wave * kWReq + i) * 1024),
                                       16, 0, 0);
#pragma unroll
    for (int i = 0; i < kXReq; ++i) {
      const uint32_t piece = wave * kXReq + i, kstep = min(blk * 2u + piece / TT, ksteps - 1);
      __builtin_amdgcn_global_load_lds(
          reinterpret_cast<const u32x4_t *>(xsrc + (static_cast<uint64_t>(kstep) * TT + piece % TT) * 1024u),
          NV_FLOW_LDS(at + kFW * RT * kFWTile + piece * 1024), 16, 0, 0);
    }
  };

  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(NV_FLOW_LDS(smem)));
  // operands of K-step e: A at piece 4 e + q of row n, B at piece (e TT + c) of the X pieces
  uint32_t a_off[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) a_off[e] = lds0 + wave * RT * kFWTile + n * 128u + (((e * 4 + q) ^ (n & 7)) << 4);
  const uint32_t b_off = lds0 + kFW * RT * kFWTile + lane * 16u;

#pragma unroll
  for (int b = 0; b < kDepth - 1; ++b)
    if (static_cast<uint32_t>(b) < nblk) request(b, b);
  uint32_t stage = 0;
  for (uint32_t b = 0; b < nblk; ++b) {
    // requests of younger blocks in flight: kDepth - 2 blocks', fewer at the end
    const uint32_t behind = min(nblk - 1u - b, static_cast<uint32_t>(kDepth - 2));
    switch (behind) {
      case 0u: wait_requests<0>(); break;
      case 1u: wait_requests<kReq>(); break;
      case 2u: wait_requests<kDepth >= 4 ? 2 * kReq : 0>(); break;
      case 3u: wait_requests<kDepth >= 5 ? 3 * kReq : 0>(); break;
      default: wait_requests<kDepth >= 6 ? 4 * kReq : 0>(); break;
    }
    asm volatile("s_barrier" ::: "memory");
    if (b + kDepth - 1u < nblk) request(b + kDepth - 1u, stage == 0 ? kDepth - 1u : stage - 1u);
    const uint32_t at = stage * kStage;
    // (the second K-step of the last block lies past the matrix when K is an odd multiple of 32)
    const uint32_t steps = min(2u, ksteps - (first + b) * 2u);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (e == 1 && steps < 2u) break;
      // the reads and their wait in one statement: nothing that uses the operands can come before it
      u32x4_t a[2], x[8];
      const uint32_t aa = a_off[e] + at, ba = b_off + at + e * TT * 1024u;
      if constexpr (TT == 2 && RT == 1)
        asm volatile("ds_read_b128 %0, %3\n\tds_read_b128 %1, %4\n\tds_read_b128 %2, %4 offset:1024\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(a[0]), "=&v"(x[0]), "=&v"(x[1])
                     : "v"(aa), "v"(ba)
                     : "memory");
      else if constexpr (TT == 2)
        asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:2048\n\tds_read_b128 %2, %5\n\tds_read_b128 %3, %5 offset:1024\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(a[0]), "=&v"(a[1]), "=&v"(x[0]), "=&v"(x[1])
                     : "v"(aa), "v"(ba)
                     : "memory");
      else if constexpr (TT == 4)
        asm volatile("ds_read_b128 %0, %6\n\tds_read_b128 %1, %6 offset:%8\n\tds_read_b128 %2, %7\n\tds_read_b128 %3, %7 offset:1024\n\t"
                     "ds_read_b128 %4, %7 offset:2048\n\tds_read_b128 %5, %7 offset:3072\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(a[0]), "=&v"(a[1]), "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3])
                     : "v"(aa), "v"(ba), "n"(RT == 2 ? kFWTile : 0)
                     : "memory");
      else
        asm volatile("ds_read_b128 %0, %10\n\tds_read_b128 %1, %10 offset:%12\n\tds_read_b128 %2, %11\n\tds_read_b128 %3, %11 offset:1024\n\t"
                     "ds_read_b128 %4, %11 offset:2048\n\tds_read_b128 %5, %11 offset:3072\n\tds_read_b128 %6, %11 offset:4096\n\t"
                     "ds_read_b128 %7, %11 offset:5120\n\tds_read_b128 %8, %11 offset:6144\n\tds_read_b128 %9, %11 offset:7168\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(a[0]), "=&v"(a[1]), "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(x[4]), "=&v"(x[5]),
                       "=&v"(x[6]), "=&v"(x[7])
                     : "v"(aa), "v"(ba), "n"(RT == 2 ? kFWTile : 0)
                     : "memory");
#pragma unroll
      for (int c = 0; c < TT; ++c)
#pragma unroll
        for (int j = 0; j < RT; ++j) acc[j][c] = mfma_k32<DT>(a[j], x[c], acc[j][c]);
    }
    stage = stage + 1u == kDepth ? 0u : stage + 1u;
  }

  // D layout: lane (n, q) holds rows q*4 .. q*4+3 of a row tile for token n of a token tile
  const XieluParams act = slices == 1 ? epilogue_act<DT, EPI>(p) : XieluParams{};
  const uint32_t wrows = EPI == kGemmSwiglu ? 2u * rows : rows;
  float *part = partials + static_cast<uint64_t>(blockIdx.y) * kFTokCap * wrows;
#pragma unroll
  for (int c = 0; c < TT; ++c) {
    const uint32_t t = c * 16u + n;
    if (t >= T) continue;
#pragma unroll
    for (int j = 0; j < RT; ++j) {
      const uint32_t row = trow[j] + q * 4u;
      if (row >= rows) continue;
      if (slices > 1) {   // (rows % 4 == 0: the plan)
        const uint32_t at = EPI == kGemmSwiglu && j == 1 ? rows + row : row;
        *reinterpret_cast<float4 *>(part + static_cast<uint64_t>(t) * wrows + at) =
            make_float4(acc[j][c][0], acc[j][c][1], acc[j][c][2], acc[j][c][3]);
      } else if (EPI == kGemmF32 && rows % 4u != 0) {   // a head of any vocabulary
        for (uint32_t r = 0; r < 4 && row + r < rows; ++r)
          p.out_f32[static_cast<uint64_t>(t) * rows + row + r] = acc[j][c][r] + (p.bias != nullptr ? dec16<DT>(p.bias[row + r]) : 0.0f);
      } else if constexpr (EPI == kGemmSwiglu) {
        if (j == 0) block_epilogue<DT, EPI>(p, t, row, acc[0][c], acc[RT - 1][c], act);
      } else {
        block_epilogue<DT, EPI>(p, t, row, acc[j][c], acc[j][c], act);
      }
    }
  }
}
#undef NV_FLOW_LDS

template <uint32_t DT, int EPI, int TT, int RT>
hipError_t launch_flow_rt(const GemmRowsParams &p, uint32_t kslices, hipStream_t stream) {
  constexpr size_t lds = static_cast<size_t>(flow_stage_bytes(TT, RT)) * flow_depth(TT, RT);
  // more than the default dynamic LDS limit: raised once per kernel (never under stream capture)
  static std::once_flag once;
  static hipError_t raised = hipSuccess;
  std::call_once(once, [] {
    raised = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_flow_kernel<DT, EPI, TT, RT>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
  });
  if (raised != hipSuccess) return raised;
  const uint32_t wg_rows = EPI == kGemmSwiglu ? 16u * kFW : 16u * kFW * RT;
  hipLaunchKernelGGL((gemm_flow_kernel<DT, EPI, TT, RT>), dim3((p.rows + wg_rows - 1) / wg_rows, kslices), dim3(kFW * kWave), lds,
                     stream, p, static_cast<float *>(p.workspace));
  return hipGetLastError();
}

template <uint32_t DT, int EPI, int TT>
hipError_t launch_flow_tt(const GemmRowsParams &p, const GemmFlowPlan &plan, hipStream_t stream) {
  if constexpr (EPI == kGemmSwiglu) return launch_flow_rt<DT, EPI, TT, 2>(p, plan.kslices, stream);
  else return plan.row_tiles == 2 ? launch_flow_rt<DT, EPI, TT, 2>(p, plan.kslices, stream) : launch_flow_rt<DT, EPI, TT, 1>(p, plan.kslices, stream);
}

template <uint32_t DT, int EPI>
hipError_t launch_flow(const GemmRowsParams &p, const GemmFlowPlan &plan, hipStream_t stream) {
  switch (p.x_packed) {
    case 2: return launch_flow_tt<DT, EPI, 2>(p, plan, stream);
    case 4: return launch_flow_tt<DT, EPI, 4>(p, plan, stream);
    case 8: return launch_flow_tt<DT, EPI, 8>(p, plan, stream);
    default: return hipErrorInvalidValue;
  }
}

template <uint32_t DT>
hipError_t launch_flow_dt(int epilogue, const GemmRowsParams &p, const GemmFlowPlan &plan, hipStream_t stream) {
  switch (epilogue) {
    case kGemmF32: return launch_flow<DT, kGemmF32>(p, plan, stream);
    case kGemmResidual: return launch_flow<DT, kGemmResidual>(p, plan, stream);
    case kGemmXielu: return launch_flow<DT, kGemmXielu>(p, plan, stream);
    case kGemmSwiglu: return launch_flow<DT, kGemmSwiglu>(p, plan, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

// K slices until every CU has a workgroup and no further (what is left over from a second round costs more than it
// spreads: 2 rows of 5120 x 5120 in 3 / 4 / 6 slices of 80 row groups 15.0 / 18.4 / 15.9 us, of 2560 x 9728 in 4 / 6 / 8
// slices of 40 17.2 / 14.5 / 18.1), each of at least eight K-blocks (its pipeline has to fill: 4096 x 1024 in 1 / 2 / 4
// slices 7.0 / 7.3 / 6.8 us, 11 and 12 us at 128 rows), the partial sums within the workspace. Two row tiles a wave only
// for a gate/up pair and for heads of so many rows that every CU still has three rounds of workgroups.
GemmFlowPlan gemm_flow_plan(int epilogue, uint32_t rows, uint32_t cols, uint32_t tokens, uint64_t workspace_bytes) {
  GemmFlowPlan plan{};
  if (tokens == 0 || tokens > kFTokCap || cols == 0 || cols % 32u != 0 || rows == 0 || (epilogue != kGemmF32 && rows % 4u != 0)) return plan;
  const uint32_t wrows = epilogue == kGemmSwiglu ? 2u * rows : rows;
  plan.row_tiles = epilogue == kGemmSwiglu || rows >= 128u * 768u ? 2u : 1u;
  const uint32_t wg_rows = epilogue == kGemmSwiglu ? 64u : 64u * plan.row_tiles;
  const uint32_t groups = (rows + wg_rows - 1) / wg_rows, blocks = (cols + kFK - 1) / kFK;
  uint32_t slices = rows % 4u != 0 ? 1u : std::max(1u, std::min({256u / groups, blocks / 8u, 8u}));
  const uint64_t one = static_cast<uint64_t>(kFTokCap) * wrows * sizeof(float);
  if (slices > 1 && slices * one > workspace_bytes) slices = std::max<uint32_t>(1u, static_cast<uint32_t>(workspace_bytes / one));
  plan.kslices = slices;
  plan.workgroups = groups * slices;
  return plan;
}

hipError_t launch_gemm_flow(uint32_t dtype, int epilogue, const GemmRowsParams &p, const GemmFlowPlan &plan, hipStream_t stream) {
  if (plan.kslices == 0 || p.x_packed == 0 || p.x_packed != gemm_packed_tiles(p.tokens)) return hipErrorInvalidValue;
  if (plan.kslices > 1 && p.workspace == nullptr) return hipErrorInvalidValue;
  hipError_t err = dtype == kBF16  ? launch_flow_dt<kBF16>(epilogue, p, plan, stream)
                   : dtype == kF16 ? launch_flow_dt<kF16>(epilogue, p, plan, stream)
                                   : hipErrorInvalidValue;
  if (err == hipSuccess && plan.kslices > 1 && !(epilogue == kGemmF32 && p.keep_partials != 0))
    err = launch_gemm_finish(dtype, epilogue, p, static_cast<const float *>(p.workspace), plan.kslices, kFTokCap, stream);
  return err;
}

}  // namespace nv
