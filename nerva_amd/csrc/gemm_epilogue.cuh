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

// Epilogue of four consecutive output rows (row .. row + 3) of token t. For SwiGLU `up` holds the up
// rows' sums, otherwise it is unused.
template <uint32_t DT, int EPI>
__device__ __forceinline__ void block_epilogue(const GemmRowsParams &p, uint32_t t, uint32_t row, f32x4_t y, f32x4_t up) {
  if (p.bias != nullptr) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      y[r] += dec16<DT>(p.bias[row + r]);
      if constexpr (EPI == kGemmSwiglu) up[r] += dec16<DT>(p.bias[p.rows + row + r]);
    }
  }
  const uint64_t at = static_cast<uint64_t>(t) * p.rows + row;
  if constexpr (EPI == kGemmSwiglu) {
    uint16_t h[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) h[r] = enc16<DT>(silu(y[r]) * up[r]);
    const uint64_t at16 = p.out_packed_tiles != 0 ? gemm_x_packed_index(p.out_packed_tiles, t, row) : at;
    *reinterpret_cast<uint2 *>(p.out16 + at16) =
        make_uint2(h[0] | (static_cast<uint32_t>(h[1]) << 16), h[2] | (static_cast<uint32_t>(h[3]) << 16));
  } else if constexpr (EPI == kGemmXielu) {
    const XieluParams act = xielu_params<DT>(p.act);
    uint16_t h[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) h[r] = enc16<DT>(xielu(y[r], act));
    const uint64_t at16 = p.out_packed_tiles != 0 ? gemm_x_packed_index(p.out_packed_tiles, t, row) : at;
    *reinterpret_cast<uint2 *>(p.out16 + at16) =
        make_uint2(h[0] | (static_cast<uint32_t>(h[1]) << 16), h[2] | (static_cast<uint32_t>(h[3]) << 16));
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
