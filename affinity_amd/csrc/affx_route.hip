// Routing on the device: the router's top-k over a batch's logits, writing
// the [n_tok][top_k] expert ids and weights that the decode and grouped entries read, so a layer
// goes from logits to expert output without routes passing through the host.
//
// Two rules:
//  * the engine's (src/engine/ops.cpp:62-92, the device form src/gpu/batch_kernels.hip:2964-3031):
//    score = sqrt(softplus(logit)) with the x > 20 guard; the k best of score + bias (the bias
//    chooses, it never weighs), ties to the lower id; weight = score * inv * routed_scaling with
//    inv = 1 / (sum of the k scores, in double, floored at the fp16 least normal) when the
//    weights are renormalised, else 1;
//  * the benchmark configs' softmax top-k: the k largest logits (ties to the lower id), weights
//    the softmax over those k, in double.
#include "affx_common.h"

namespace affx {

constexpr int kRouteWaves = 4;  // waves of a workgroup: that many tokens, or one token's

// The order of the choice as an integer: the larger key first, then the lower id (equal float keys,
// the two zeros included, have equal high words). Never 0, which marks an expert already taken.
__device__ __forceinline__ uint64_t route_rank(float key, uint32_t id) {
  const uint32_t u = __float_as_uint(key + 0.0f);
  return ((uint64_t)(u & 0x80000000u ? ~u : u | 0x80000000u) << 32) | (0xFFFFFFFFu - id);
}

// Maximum over the wave, in every lane: four DPP row shifts leave each row's in its last lane (a
// shuffle through the LDS costs several times a DPP op, and the k picks are a serial chain of them).
template <int N>
__device__ __forceinline__ uint64_t row_max_step(uint64_t x) {
  const uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
  const uint32_t sl = (uint32_t)__builtin_amdgcn_update_dpp((int)lo, (int)lo, 0x110 + N, 0xF, 0xF, false);
  const uint32_t sh = (uint32_t)__builtin_amdgcn_update_dpp((int)hi, (int)hi, 0x110 + N, 0xF, 0xF, false);
  const uint64_t y = ((uint64_t)sh << 32) | sl;
  return x > y ? x : y;
}
__device__ __forceinline__ uint64_t wave_max(uint64_t x) {
  x = row_max_step<1>(x);
  x = row_max_step<2>(x);
  x = row_max_step<4>(x);
  x = row_max_step<8>(x);
  uint64_t m = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const uint64_t y = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), 16 * r + 15) << 32) |
                       (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, 16 * r + 15);
    m = m > y ? m : y;
  }
  return m;
}

// The engine router's score. expf and log1pf are evaluated in double and rounded once, which is
// within an ulp of the host's float functions (their results are not always correctly rounded).
__device__ __forceinline__ float route_score(float x) {
  if (x > 20.0f) return sqrtf(x);
  const float e = (float)exp((double)x);
  const float sp = (float)log1p((double)e);
  return sqrtf(sp);
}

// WPT: waves per token. All of them score the token's experts (double-precision exp and log1p, the
// longest part); its first wave then takes the k best, one wave_max each. Latency-bound: one token of
// 256 experts took 10.1 us with a wave a token, shuffles and the weights in one lane, now 4.7 (launches in
// a graph); 1024 tokens 11.1, now 6.5 (WPT = 4) against 7.5 (WPT = 1). From kRouteWide tokens on there
// are waves enough either way (2048 tokens: 9.2 and 9.1, 16384: 41.7 and 39.3), and a wave a token does
// without the idle waves of the picks.
constexpr uint32_t kRouteWide = 2048;
template <int RULE, int WPT>
__global__ void __launch_bounds__(kRouteWaves * 64) route_topk_kernel(
    const float* __restrict__ logits, uint64_t tok_stride, uint64_t exp_stride, const float* __restrict__ bias,
    uint32_t n_tok, uint32_t n_expert, uint32_t k, int norm_topk_prob, float routed_scaling,
    uint32_t* __restrict__ sel, float* __restrict__ wout) {
  constexpr int NT = kRouteWaves / WPT;                  // tokens a workgroup
  constexpr int NV = AFFX_MAX_EXPERTS / 64, NS = NV / WPT;  // experts per lane: of a wave, when scored
  __shared__ float val_s[NT][AFFX_MAX_EXPERTS];         // what the weights are made of
  __shared__ uint64_t rank_s[WPT > 1 ? AFFX_MAX_EXPERTS : 1];
  __shared__ double ex_s[NT][AFFX_MAX_TOPK];
  __shared__ uint32_t id_s[NT][AFFX_MAX_TOPK];
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6, tl = wv / WPT, sub = wv % WPT;
  const uint32_t t = blockIdx.x * NT + tl;
  const bool live = t < n_tok, pick = live && sub == 0;
  uint64_t rank[NV];  // lane holds experts lane + 64 v
#pragma unroll
  for (int v = 0; v < NV; ++v) rank[v] = 0;
  if (live) {
#pragma unroll
    for (int v = 0; v < NS; ++v) {
      const uint32_t e = (WPT > 1 ? sub * 64u + 256u * v : 64u * v) + lane;
      if (e < n_expert) {
        const float x = logits[(uint64_t)t * tok_stride + (uint64_t)e * exp_stride];
        float val = x, key = x;
        if constexpr (RULE == AFFX_ROUTE_ENGINE) {
          val = route_score(x);
          key = val + (bias ? bias[e] : 0.0f);
        }
        val_s[tl][e] = val;
        rank[v] = route_rank(key, e);
        if constexpr (WPT > 1) rank_s[e] = rank[v];
      }
    }
  }
  __syncthreads();
  if (pick) {
    if constexpr (WPT > 1) {
#pragma unroll
      for (int v = 0; v < NV; ++v) rank[v] = 64u * v + lane < n_expert ? rank_s[64u * v + lane] : 0;
    }
    for (uint32_t r = 0; r < k; ++r) {
      uint64_t best = rank[0];
#pragma unroll
      for (int v = 1; v < NV; ++v)
        if (64u * v < n_expert) best = best > rank[v] ? best : rank[v];
      best = wave_max(best);  // (k <= n_expert: there is one)
#pragma unroll
      for (int v = 0; v < NV; ++v)
        if (rank[v] == best) rank[v] = 0;
      if (lane == 0) id_s[tl][r] = 0xFFFFFFFFu - (uint32_t)best;
    }
  }
  __syncthreads();
  // the weights, a lane each (every lane adds the same terms in the same order)
  const uint32_t id = pick && lane < k ? id_s[tl][lane] : 0u;
  if constexpr (RULE == AFFX_ROUTE_ENGINE) {
    if (pick && lane < k) {
      double sum = 0.0;
      for (uint32_t j = 0; j < k; ++j) sum += val_s[tl][id_s[tl][j]];
      if (sum < 6.103515625e-5) sum = 6.103515625e-5;
      const double inv = norm_topk_prob ? 1.0 / sum : 1.0;
      sel[(uint64_t)t * k + lane] = id;
      wout[(uint64_t)t * k + lane] = (float)((double)val_s[tl][id] * inv * (double)routed_scaling);
    }
  } else {
    // softmax over the k: the first is the largest logit of all
    if (pick && lane < k) ex_s[tl][lane] = exp((double)val_s[tl][id] - (double)val_s[tl][id_s[tl][0]]);
    __syncthreads();
    if (pick && lane < k) {
      double sum = 0.0;
      for (uint32_t j = 0; j < k; ++j) sum += ex_s[tl][j];
      sel[(uint64_t)t * k + lane] = id;
      wout[(uint64_t)t * k + lane] = (float)(ex_s[tl][lane] / sum);
    }
  }
}

}  // namespace affx

using namespace affx;

extern "C" int affx_route_topk(const float* logits, uint64_t tok_stride, uint64_t expert_stride,
                               const float* bias, uint32_t n_tok, uint32_t n_expert, uint32_t top_k, int rule,
                               int norm_topk_prob, float routed_scaling, uint32_t* sel, float* w,
                               void* stream) {
  if (!logits || !sel || !w) return set_error(AFFX_ERR_ARG, "route_topk: null pointer");
  if (n_tok == 0) return AFFX_OK;
  if (n_expert == 0 || n_expert > AFFX_MAX_EXPERTS || top_k == 0 || top_k > AFFX_MAX_TOPK || top_k > n_expert)
    return set_error(AFFX_DECLINED, "route_topk: n_expert must be 1..%d and top_k 1..min(%d, n_expert)",
                     AFFX_MAX_EXPERTS, AFFX_MAX_TOPK);
  if (rule != AFFX_ROUTE_ENGINE && rule != AFFX_ROUTE_SOFTMAX)
    return set_error(AFFX_ERR_ARG, "route_topk: unknown rule %d", rule);
  hipStream_t s = (hipStream_t)stream;
  auto launch = [&](auto* kernel, uint32_t per) {
    hipLaunchKernelGGL(kernel, dim3((n_tok + per - 1) / per), dim3(kRouteWaves * 64), 0, s, logits, tok_stride,
                       expert_stride, bias, n_tok, n_expert, top_k, norm_topk_prob, routed_scaling, sel, w);
  };
  const bool few = n_tok < kRouteWide;
  if (rule == AFFX_ROUTE_ENGINE)
    few ? launch(route_topk_kernel<AFFX_ROUTE_ENGINE, kRouteWaves>, 1) : launch(route_topk_kernel<AFFX_ROUTE_ENGINE, 1>, kRouteWaves);
  else
    few ? launch(route_topk_kernel<AFFX_ROUTE_SOFTMAX, kRouteWaves>, 1) : launch(route_topk_kernel<AFFX_ROUTE_SOFTMAX, 1>, kRouteWaves);
  return check_launch("route_topk_kernel");
}
