// What the multi-row projection kernels (gemm_block.hip, gemm_flow.hip) share: the matrix-core step, the epilogue of
// four output rows, and the launch that adds the partial sums of K slices.
#pragma once

#include "activations.cuh"
#include "gemm_rows.cuh"

namespace nv {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));   // a 16-byte piece as a first-class value

template <uint32_t DT>
__device__ __forceinline__ f32x4_t mfma_k32(u32x4_t a, u32x4_t b, f32x4_t c) {
  if constexpr (DT == kBF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                  0, 0);
}

// The activation's numbers of a launch, fetched and worked out once a thread and not with every four results (the stores between
// them keep the compiler from seeing that they do not change).
template <uint32_t DT, int EPI>
__device__ __forceinline__ XieluParams epilogue_act(const GemmRowsParams &p) {
  if constexpr (EPI == kGemmXielu) return xielu_params<DT>(p.act);
  else return XieluParams{};
}
// Epilogue of four consecutive output rows (row .. row + 3) of token t. For SwiGLU `up` holds the up
// rows' sums, otherwise it is unused. The arithmetic of the activations counts: a workgroup has its CU to itself at the end of a
// launch, and with expf, a division and integer rounding a gate/up pair's took 9 of 98 us of 256 rows x 256 tokens x 4096 columns.
template <uint32_t DT, int EPI>
__device__ __forceinline__ void block_epilogue(const GemmRowsParams &p, uint32_t t, uint32_t row, f32x4_t y, f32x4_t up, const XieluParams &act) {
  if (p.bias != nullptr) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      y[r] += dec16<DT>(p.bias[row + r]);
      if constexpr (EPI == kGemmSwiglu) up[r] += dec16<DT>(p.bias[p.rows + row + r]);
    }
  }
  const uint64_t at = static_cast<uint64_t>(t) * p.rows + row;
  if constexpr (EPI == kGemmSwiglu) {
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = gated(y[r], 1.0f) * up[r];
    const uint64_t at16 = p.out_packed_tiles != 0 ? gemm_x_packed_index(p.out_packed_tiles, t, row) : at;
    *reinterpret_cast<uint2 *>(p.out16 + at16) = make_uint2(enc16_pair<DT>(y[0], y[1]), enc16_pair<DT>(y[2], y[3]));
  } else if constexpr (EPI == kGemmXielu) {
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = xielu(y[r], act);
    const uint64_t at16 = p.out_packed_tiles != 0 ? gemm_x_packed_index(p.out_packed_tiles, t, row) : at;
    *reinterpret_cast<uint2 *>(p.out16 + at16) = make_uint2(enc16_pair<DT>(y[0], y[1]), enc16_pair<DT>(y[2], y[3]));
  } else {
    if constexpr (EPI == kGemmResidual) {
      const float4 res = *reinterpret_cast<const float4 *>(p.residual + at);
      y[0] += res.x;
      y[1] += res.y;
      y[2] += res.z;
      y[3] += res.w;
      if (p.round_out) {
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = round16<DT>(y[r]);
      }
    }
    *reinterpret_cast<float4 *>(p.out_f32 + at) = make_float4(y[0], y[1], y[2], y[3]);
  }
}

// Adds the slices' partial sums ([slice][tokcap][W rows] f32) in slice order and applies the epilogue, with the RMSNorm
// behind it where p.norm_gamma asks for one (gemm_block.hip). rows % 4 == 0.
hipError_t launch_gemm_finish(uint32_t dtype, int epilogue, const GemmRowsParams &p, const float *partials, uint32_t kslices,
                              uint32_t tokcap, hipStream_t stream);

}  // namespace nv
