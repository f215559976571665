// Router top-k: expert scores from the router logits, the top_k picks and their mixing weights in one
// launch -- the inputs of the fused MoE ops.  One workgroup (256 threads) per token computes the E <= 1024 scores;
// then one wave picks: a lane holds NV neighbouring scores + biases in registers, a pick is an arg-max over the wave
// (largest, smallest index on ties) after which the winner leaves the pool.  What bounds it is the chain of picks: as
// workgroup arg-maxes (two barriers and a serial look at the waves' winners each) it took, us before / now: 1 token, 128
// experts, top 8, 10.3 / 4.0; 1000 tokens 12.9 / 4.7; 1 token, 8 experts, top 2, 4.4 / 2.7; 64 tokens, 1024 experts, top 16,
// 25.1 / 17.9.  All math in f32.  Semantics of the reference's kq_moe_router_topk
// (metal/mlx/backend/metal/kernels/kq_moe_glu_kq.h:1215-1358; op contract src/kquant_moe_glu.cpp:1366-1441).
#include <type_traits>

#include "kq_decode.h"

namespace {

constexpr int RT_THREADS = 256;
constexpr int RT_WAVES = RT_THREADS / 64;
constexpr int RT_MAX_E = 1024;

struct RouterArgs {
  const void* logits;  // [T][E + shared]
  uint32_t* indices;   // [T][R]
  float* scores;       // [T][R + shared]
  const float* pes;    // per-expert scale [E] or null
  const float* bias;   // selection bias [E] or null
  int E, R, norm, shared, scoring;
  float scale;
};

template <int DT>
__device__ __forceinline__ float load_logit(const void* p, size_t i) {
  if constexpr (DT == KQ_F32) return static_cast<const float*>(p)[i];
  const uint16_t h = static_cast<const uint16_t*>(p)[i];
  return DT == KQ_F16 ? kq::h2f(h) : kq::bf162f(h);
}

// largest value over the wave, in every lane
__device__ __forceinline__ float wave_max(float v) {
  auto with = [&](auto ctrl) {
    v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xf, 0xf, false)));
  };
  with(std::integral_constant<int, 0xB1>{});   // neighbours
  with(std::integral_constant<int, 0x4E>{});   // pairs of a quad
  with(std::integral_constant<int, 0x141>{});  // quads of eight lanes
  with(std::integral_constant<int, 0x140>{});  // halves of a row of 16
  float m = v;
#pragma unroll
  for (int row = 0; row < 64; row += 16)
    m = fmaxf(m, __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), row)));
  return m;
}

template <int DT, int NV>
__global__ __launch_bounds__(RT_THREADS) void router_topk_kernel(RouterArgs a) {
  __shared__ float p[RT_MAX_E];
  __shared__ float red_m[RT_WAVES], red_s[RT_WAVES];
  constexpr int PT = (64 * NV + RT_THREADS - 1) / RT_THREADS;  // logits per thread
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int E = a.E, R = a.R;
  const size_t row = (size_t)blockIdx.x * (E + a.shared);
  float x[PT];
#pragma unroll
  for (int i = 0; i < PT; i++) x[i] = tid + RT_THREADS * i < E ? load_logit<DT>(a.logits, row + tid + RT_THREADS * i) : -INFINITY;

  float gsum = 1.0f;
  if (a.scoring == 1) {
#pragma unroll
    for (int i = 0; i < PT; i++) {
      const int e = tid + RT_THREADS * i;
      // stable softplus: max(x, 0) + log1p(exp(-|x|)), series where log(1 + z) loses bits
      const float z = expf(-fabsf(x[i]));
      const float l1p = z < 1e-4f ? fmaf(-0.5f * z, z, z) : logf(1.0f + z);
      if (e < E) p[e] = sqrtf(fmaxf(x[i], 0.0f) + l1p);
    }
    __syncthreads();
  } else {
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < PT; i++) m = fmaxf(m, x[i]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if (lane == 0) red_m[wave] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red_m[0], red_m[1]), fmaxf(red_m[2], red_m[3]));
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < PT; i++) {
      const int e = tid + RT_THREADS * i;
      if (e < E) {
        const float v = expf(x[i] - m);
        p[e] = v;
        s += v;
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane == 0) red_s[wave] = s;
    __syncthreads();
    gsum = (red_s[0] + red_s[1]) + (red_s[2] + red_s[3]);
  }
  if (wave != 0) return;

  // lane l: experts NV l ... NV l + NV - 1, so that the lowest lane with the largest value has the smallest index
  float v[NV], bias[NV];
#pragma unroll
  for (int j = 0; j < NV; j++) {
    const int e = NV * lane + j;
    bias[j] = a.bias && e < E ? a.bias[e] : 0.f;
    v[j] = e < E ? p[e] + bias[j] : NAN;  // (NaN is never picked)
  }
  float won = 0.f;     // lane r: the r-th pick, its score without the bias
  uint32_t pick = 0u;
  for (int r = 0; r < R; r++) {
    float bv = -INFINITY;
    uint32_t bi = 0xffffffffu;
#pragma unroll
    for (int j = 0; j < NV; j++)
      if (v[j] > bv || (v[j] == bv && bi == 0xffffffffu)) {
        bv = v[j];
        bi = (uint32_t)(NV * lane + j);
      }
    const float m = wave_max(bv);
    const uint64_t best = __builtin_amdgcn_ballot_w64(bv == m && bi != 0xffffffffu);
    // every value NaN: index 0
    const uint32_t wi = best ? (uint32_t)__builtin_amdgcn_readlane((int)bi, __builtin_ctzll(best)) : 0u;
    if (lane == r) {
      won = p[wi];
      pick = wi;
    }
    if (lane == 0) p[wi] = -INFINITY;  // a wave's LDS accesses are in order
#pragma unroll
    for (int j = 0; j < NV; j++)
      if (wi == (uint32_t)(NV * lane + j)) v[j] = -INFINITY + bias[j];
  }
  float ps = 0.f;
  for (int r = 0; r < R; r++) ps += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, won), r));
  const float denom = a.norm ? (a.scoring == 1 ? ps + 1e-20f : ps) : gsum;
  float* srow = a.scores + (size_t)blockIdx.x * (R + a.shared);
  if (lane < R) {
    a.indices[(size_t)blockIdx.x * R + lane] = pick;
    float sv = won / denom;
    if (a.pes) sv *= a.pes[pick];
    srow[lane] = sv * a.scale;
  }
  if (a.shared && lane == 0) srow[R] = 1.0f / (1.0f + expf(-load_logit<DT>(a.logits, row + E)));
}

template <int DT>
void launch_router(const RouterArgs& a, int T, hipStream_t s) {
  auto kern = a.E <= 128 ? router_topk_kernel<DT, 2> : a.E <= 256 ? router_topk_kernel<DT, 4> : router_topk_kernel<DT, 16>;
  hipLaunchKernelGGL(kern, dim3(T), dim3(RT_THREADS), 0, s, a);
}

}  // namespace

int kq_launch_router_topk(const void* logits, int dtype, int T, int E, int top_k, int norm, int shared, const float* pes,
                          const float* bias, int scoring, float scale, uint32_t* indices, float* scores, hipStream_t s) {
  if (T <= 0) return KQ_OK;
  RouterArgs a{logits, indices, scores, pes, bias, E, top_k, norm, shared ? 1 : 0, scoring, scale};
  if (dtype == KQ_F32)
    launch_router<KQ_F32>(a, T, s);
  else if (dtype == KQ_F16)
    launch_router<KQ_F16>(a, T, s);
  else
    launch_router<KQ_BF16>(a, T, s);
  KQ_HIP_CHECK(hipGetLastError());
  return KQ_OK;
}
