// Decode-step projections of a parallel layer (see gemv_layer.cuh).
#include "gemv_layer.cuh"

#include <algorithm>

#include "gemv_layer_walk.cuh"
#include "moe_rows.cuh"

namespace nv {

namespace {

using namespace layer;

constexpr int kWaves = 8, kThreads = kWaves * kWave;
constexpr uint32_t kMaxWorkgroups = 512;     // two a CU
// round16(x * rsqrt(mean(x^2) + eps) * gamma) of a row, for one or two gammas. cols % 8 == 0.
template <uint32_t DT>
__device__ __forceinline__ void rms_stage(const float *x, uint32_t cols, float eps, const uint16_t *g0, uint16_t *xs0, const uint16_t *g1,
                                          uint16_t *xs1, float *red) {
  float ss = 0.0f;
  for (uint32_t c = threadIdx.x * 8u; c < cols; c += kThreads * 8u) {
    const float4 a = *reinterpret_cast<const float4 *>(x + c), b = *reinterpret_cast<const float4 *>(x + c + 4);
    ss += a.x * a.x + a.y * a.y + a.z * a.z + a.w * a.w + b.x * b.x + b.y * b.y + b.z * b.z + b.w * b.w;
  }
  const float scale = 1.0f / sqrtf(block_sum_n<kWaves>(ss, red) / static_cast<float>(cols) + eps);
  for (uint32_t c = threadIdx.x * 8u; c < cols; c += kThreads * 8u) {
    const float4 a = *reinterpret_cast<const float4 *>(x + c), b = *reinterpret_cast<const float4 *>(x + c + 4);
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    const auto put = [&](const uint16_t *gamma, uint16_t *xs) {
      const uint4 g = *reinterpret_cast<const uint4 *>(gamma + c);
      float w[8];
      unpack8<DT>(g, w);
      uint32_t o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o[e] = enc16<DT>(v[2 * e] * scale * w[2 * e]) | (static_cast<uint32_t>(enc16<DT>(v[2 * e + 1] * scale * w[2 * e + 1])) << 16);
      *reinterpret_cast<uint4 *>(xs + c) = make_uint4(o[0], o[1], o[2], o[3]);
    };
    put(g0, xs0);
    if (g1 != nullptr) put(g1, xs1);
  }
  clear_tail<kThreads>(xs0, cols);
  if (g1 != nullptr) clear_tail<kThreads>(xs1, cols);
}

// ---- front, middle ---------------------------------------------------------------------------

template <uint32_t DT>
__global__ __launch_bounds__(kThreads, 4) void layer_front_kernel(LayerFront p) {
  extern __shared__ __align__(16) uint16_t xs[];   // the mixer's row, the feed-forward's
  __shared__ float red[kWaves];
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t n_in = (p.in_rows + 1) / 2, n_router = (p.experts + 1) / 2, units = n_in + n_router + p.shared_ff;
  const auto unit_at = [&](uint32_t i) {
    if (i < n_router) return two_rows(p.router, p.hidden, p.experts, i, padded(p.hidden), p.logits);
    i -= n_router;
    if (i < n_in) return two_rows(p.w_in, p.hidden, p.in_rows, i, 0u, p.in);
    return gate_and_up(p.shared_in, p.hidden, p.shared_ff, i - n_in, padded(p.hidden), p.shared_act, p.shared_limit);
  };
  // (consecutive units go to different workgroups)
  PairWalk<DT, decltype(unit_at)> walk(unit_at, units, wave * gridDim.x + blockIdx.x, gridDim.x * kWaves);
  walk.start();
  if (*p.cursor >= p.max_steps) return;   // (after the requests, which do not depend on it)
  uint16_t *xs2 = xs + padded(p.hidden);
  rms_stage<DT>(p.x, p.hidden, p.eps, p.mixer_norm, xs, p.ff_norm, xs2, red);
  __syncthreads();
  if (p.ff_norm != nullptr && blockIdx.x == 0)
    for (uint32_t c = threadIdx.x * 8u; c < p.hidden; c += kThreads * 8u) *reinterpret_cast<uint4 *>(p.h16 + c) = *reinterpret_cast<const uint4 *>(xs2 + c);
  walk.run(xs);
}

template <uint32_t DT, bool RIDES>
__global__ __launch_bounds__(kThreads, 4) void layer_middle_kernel(LayerMiddle p) {
  extern __shared__ __align__(16) uint16_t xs[];   // the query latent, the feed-forward's row
  __shared__ float red[kWaves];
  __shared__ float score[kMaxExperts];
  __shared__ uint32_t id_s[kMaxTop];
  __shared__ float s_s[kMaxTop];
  uint16_t *xs2 = xs + padded(p.q_rank);
  const uint32_t tid = threadIdx.x;
  const auto choose = [&] {
    for (uint32_t e = tid; e < p.experts; e += kThreads) score[e] = 1.0f / (1.0f + expf(-p.logits[e]));
    if (tid < kMaxTop) {   // (scores that are no numbers choose nothing: some expert that exists)
      id_s[tid] = 0u;
      s_s[tid] = 0.0f;
    }
    __syncthreads();
    // an expert's place is the number of experts ahead of it
    for (uint32_t e = tid; e < p.experts; e += kThreads) {
      const float s = score[e];
      uint32_t ahead = 0;
#pragma unroll 8
      for (uint32_t j = 0; j < p.experts; ++j) ahead += score[j] > s || (score[j] == s && j < e) ? 1u : 0u;
      if (ahead < p.top) {
        id_s[ahead] = e;
        s_s[ahead] = s;
      }
    }
    __syncthreads();
  };
  const auto publish = [&] {
    if (tid >= p.top) return;
    float sum = 0.0f;
    for (uint32_t k = 0; k < p.top; ++k) sum += s_s[k];
    p.ids[tid] = id_s[tid];
    p.weights[tid] = s_s[tid] / (sum + 1e-20f);
  };
  if constexpr (RIDES) {
    if (blockIdx.x == gridDim.x - 1) {   // a workgroup of its own: who is chosen is wanted by the next launch
      if (*p.cursor >= p.max_steps) return;
      choose();
      publish();
      return;
    }
  } else if (p.experts != 0) {
    choose();   // (whose rows this launch walks, everyone has to know)
  }
  const uint32_t blocks = gridDim.x - (RIDES ? 1u : 0u);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const uint32_t pairs = RIDES ? p.shared_ff : p.experts != 0 ? p.top * p.ff : 0u, units = pairs + (p.q_rows + 1) / 2;
  const auto unit_at = [&](uint32_t i) {
    if (i >= pairs) return two_rows(p.w_uq, p.q_rank, p.q_rows, i - pairs, 0u, p.q);
    if (RIDES) return gate_and_up(p.shared_in, p.hidden, p.shared_ff, i, padded(p.q_rank), p.shared_act, p.shared_limit);
    const uint32_t k = i / p.ff, e = __builtin_amdgcn_readfirstlane(id_s[k]);
    return gate_and_up(p.e_in + static_cast<uint64_t>(e) * 2u * p.ff * p.hidden, p.hidden, p.ff, i - k * p.ff, padded(p.q_rank), p.act + k * p.ff,
                       p.limit);
  };
  PairWalk<DT, decltype(unit_at)> walk(unit_at, units, wave * blocks + blockIdx.x, blocks * kWaves);
  walk.start();
  if (*p.cursor >= p.max_steps) return;   // (after the requests, which do not depend on it)
  if (pairs != 0) stage_vector<kThreads>(xs2, p.h16, p.hidden);
  rms_stage<DT>(p.latent, p.q_rank, p.eps, p.latent_norm, xs, nullptr, nullptr, red);
  __syncthreads();
  if (!RIDES && p.experts != 0 && blockIdx.x == 0) publish();
  walk.run(xs);
}

// ---- back ------------------------------------------------------------------------------------

template <uint32_t DT>
__global__ __launch_bounds__(kThreads, 4) void layer_back_kernel(LayerBack p) {
  extern __shared__ __align__(16) uint16_t xs[];   // the pieces' inputs
  __shared__ __align__(16) Chunk table[kMaxChunks + kBackBatch];
  walk_back<DT, kWaves>(p, xs, table, blockIdx.x, gridDim.x);
}

uint32_t workgroups(uint32_t units) { return std::max(1u, std::min(kMaxWorkgroups, (units + kWaves - 1) / kWaves)); }
bool whole(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

bool layer_gemv_takes(uint32_t hidden, uint32_t q_rank, uint32_t mix_cols, uint32_t experts, uint32_t top, uint32_t ff, uint32_t shared_ff) {
  return hidden % 8 == 0 && q_rank % 8 == 0 && mix_cols % 8 == 0 && ff % 8 == 0 && shared_ff % 8 == 0 && experts <= kMaxExperts && top <= kMaxTop &&
         2u * 2u * padded(hidden) <= kMaxLds && 2u * (padded(q_rank) + padded(hidden)) <= kMaxLds && 2u * back_columns(mix_cols, top, ff, shared_ff) <= kMaxLds;
}

hipError_t launch_layer_front(uint32_t dtype, const LayerFront &p, hipStream_t stream) {
  const bool ff = p.ff_norm != nullptr;
  if (dtype != kBF16 || p.x == nullptr || p.mixer_norm == nullptr || p.w_in == nullptr || p.in == nullptr || p.in_rows == 0 || p.cursor == nullptr ||
      p.hidden == 0 || !layer_gemv_takes(p.hidden, 8, 8, p.experts, 0, 0, p.shared_ff) || (!ff && (p.experts != 0 || p.shared_ff != 0)) ||
      (ff && p.h16 == nullptr) || (p.experts != 0 && (p.router == nullptr || p.logits == nullptr)) ||
      (p.shared_ff != 0 && (p.shared_in == nullptr || p.shared_act == nullptr)) || !whole(p.x) || !whole(p.w_in) || !whole(p.router) ||
      !whole(p.shared_in) || !whole(p.mixer_norm) || !whole(p.ff_norm) || !whole(p.h16))
    return hipErrorInvalidValue;
  const uint32_t units = (p.in_rows + 1) / 2 + (p.experts + 1) / 2 + p.shared_ff;
  hipLaunchKernelGGL(layer_front_kernel<kBF16>, dim3(workgroups(units)), dim3(kThreads), 2u * 2u * padded(p.hidden), stream, p);
  return hipGetLastError();
}

hipError_t launch_layer_middle(uint32_t dtype, const LayerMiddle &p, hipStream_t stream) {
  if (dtype != kBF16 || p.latent == nullptr || p.latent_norm == nullptr || p.w_uq == nullptr || p.q == nullptr || p.q_rows == 0 || p.q_rank == 0 ||
      p.cursor == nullptr || !layer_gemv_takes(p.experts != 0 ? p.hidden : 8, p.q_rank, 8, p.experts, 0, p.experts != 0 ? p.ff : 0, 0) ||
      (p.experts != 0 && (p.h16 == nullptr || p.logits == nullptr || p.top == 0 || p.top > p.experts || p.top > kMaxTop || p.e_in == nullptr ||
                          p.ff == 0 || p.act == nullptr || p.ids == nullptr || p.weights == nullptr)) ||
      !whole(p.latent) || !whole(p.latent_norm) || !whole(p.w_uq) || !whole(p.h16) || !whole(p.e_in))
    return hipErrorInvalidValue;
  if (p.rides != 0 && (p.experts == 0 || (p.shared_ff != 0 && (p.shared_in == nullptr || p.shared_act == nullptr || !whole(p.shared_in))))) return hipErrorInvalidValue;
  const uint32_t units = (p.q_rows + 1) / 2 + (p.rides != 0 ? p.shared_ff : p.experts != 0 ? p.top * p.ff : 0u);
  const size_t lds = 2u * (padded(p.q_rank) + (p.experts != 0 ? padded(p.hidden) : 0u));
  if (p.rides != 0) hipLaunchKernelGGL((layer_middle_kernel<kBF16, true>), dim3(workgroups(units) + 1), dim3(kThreads), lds, stream, p);
  else hipLaunchKernelGGL((layer_middle_kernel<kBF16, false>), dim3(workgroups(units)), dim3(kThreads), lds, stream, p);
  return hipGetLastError();
}

hipError_t launch_layer_back(uint32_t dtype, const LayerBack &p, hipStream_t stream) {
  if (dtype != kBF16 || p.x == nullptr || p.w_o == nullptr || p.mixed == nullptr || p.hidden == 0 || p.mix_cols == 0 || p.y != nullptr || p.cursor == nullptr ||
      !layer_gemv_takes(8, 8, p.mix_cols, 0, p.top, p.top != 0 ? p.ff : 0, p.shared_ff) ||
      (p.top != 0 && (p.e_out == nullptr || p.act == nullptr || p.ids == nullptr || p.weights == nullptr || p.ff == 0 || p.experts == 0)) ||
      (p.shared_ff != 0 && (p.shared_out == nullptr || p.shared_act == nullptr)) || !whole(p.w_o) || !whole(p.mixed) || !whole(p.e_out) ||
      !whole(p.act) || !whole(p.shared_out) || !whole(p.shared_act))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(layer_back_kernel<kBF16>, dim3(workgroups(p.hidden)), dim3(kThreads), 2u * back_columns(p.mix_cols, p.top, p.ff, p.shared_ff), stream, p);
  return hipGetLastError();
}

}  // namespace nv
