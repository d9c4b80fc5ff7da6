// Gradient of the router's logits from that of the renormalised top-k weights
// (torch autograd over astrai/model/components/mlp.py:84-87).
//
// p = softmax(logits) in float, v_k = p at the chosen experts rounded to the
// element type, S = sum v rounded, w_k = v_k / S:
//   dv_k = (dw_k - sum_j dw_j w_j) / S,  dl_e = p_e (dp_e - sum_j dp_j p_j)
// with dp = dv at the chosen experts and zero elsewhere, in float throughout
// (autograd rounds to the element type after each of its operators).
//
// One wave per token, lane l holding logits l, l + 64, ...: latency-bound, a
// few us. It takes the place of the torch operators that rebuilt the weights
// for autograd, two dozen launches of 2 to 8 us in a training step and as many
// host calls: 700 bf16 tokens of D 2048, F 1408, 16 experts, top-4 and a shared
// expert 1282 -> 1060 us a step, bound by the host before and after.
#include "moe_common.h"

namespace astrai_moe {
namespace {

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

template <typename T, int ITER>
__global__ __launch_bounds__(256) void route_grad_kernel(const T* __restrict__ logits,
                                                         const int32_t* __restrict__ topk_idx,
                                                         const T* __restrict__ dw, int64_t n_tokens, int n_experts,
                                                         int top_k, T* __restrict__ dlogits) {
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (t >= n_tokens) return;
  const bool mine = lane < top_k;
  const int idx = mine ? topk_idx[t * top_k + lane] : -1;
  const float g = mine ? Elem<T>::to_f32(dw[t * top_k + lane]) : 0.0f;
  const T* const row = logits + t * n_experts;
  float l[ITER], mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < ITER; ++i) {
    const int c = lane + i * 64;
    l[i] = c < n_experts ? Elem<T>::to_f32(row[c]) : -INFINITY;
    mx = fmaxf(mx, l[i]);
  }
  const float chosen = (mine && idx >= 0 && idx < n_experts) ? Elem<T>::to_f32(row[idx]) : -INFINITY;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < ITER; ++i) {
    l[i] = expf(l[i] - mx);
    sum += l[i];
  }
  sum = wave_sum(sum);
  const float p = mine ? expf(chosen - mx) / sum : 0.0f;
  const float v = Elem<T>::round(p);
  const float S = Elem<T>::round(wave_sum(v));
  const float dot = wave_sum(g * (v / S));
  const float dv = mine ? (g - dot) / S : 0.0f;
  const float dp_p = wave_sum(dv * p);
#pragma unroll
  for (int i = 0; i < ITER; ++i) {
    const int c = lane + i * 64;
    float dp = 0.0f;
    for (int k = 0; k < top_k; ++k) {
      const int e = __shfl(idx, k, 64);
      const float d = __shfl(dv, k, 64);
      if (e == c) dp = d;
    }
    if (c < n_experts) dlogits[t * n_experts + c] = Elem<T>::from_f32(l[i] / sum * (dp - dp_p));
  }
}

template <typename T>
int launch_route_grad(const void* logits, const int32_t* topk_idx, const void* dw, int64_t n_tokens, int n_experts,
                      int top_k, void* dlogits, hipStream_t s) {
  auto kernel = n_experts <= 64    ? &route_grad_kernel<T, 1>
                : n_experts <= 128 ? &route_grad_kernel<T, 2>
                : n_experts <= 256 ? &route_grad_kernel<T, 4>
                                   : &route_grad_kernel<T, ASTRAI_MOE_MAX_EXPERTS / 64>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div(n_tokens, 4)), dim3(256), 0, s, static_cast<const T*>(logits),
                     topk_idx, static_cast<const T*>(dw), n_tokens, n_experts, top_k, static_cast<T*>(dlogits));
  return check_launch("route_grad_kernel");
}

}  // namespace
}  // namespace astrai_moe

using namespace astrai_moe;

extern "C" int astrai_moe_route_grad(const void* logits, const int32_t* topk_idx, const void* dw, int dtype,
                                     int64_t n_tokens, int n_experts, int top_k, void* dlogits, void* stream) {
  clear_error();
  ASTRAI_REQUIRE(n_tokens >= 0 && n_tokens < (1ll << 31), "route_grad: n_tokens must be in [0, 2^31)");
  ASTRAI_REQUIRE(n_experts >= 1 && n_experts <= ASTRAI_MOE_MAX_EXPERTS,
                 "route_grad: n_experts must be in [1, %d] (got %d)", ASTRAI_MOE_MAX_EXPERTS, n_experts);
  ASTRAI_REQUIRE(top_k >= 1 && top_k <= n_experts && top_k <= ASTRAI_MOE_MAX_TOPK,
                 "route_grad: top_k must be in [1, min(n_experts, %d)] (got %d)", ASTRAI_MOE_MAX_TOPK, top_k);
  ASTRAI_REQUIRE(dtype == ASTRAI_MOE_BF16 || dtype == ASTRAI_MOE_F32, "route_grad: unsupported dtype %d", dtype);
  if (n_tokens == 0) return ASTRAI_MOE_OK;
  ASTRAI_REQUIRE(logits && topk_idx && dw && dlogits, "route_grad: null buffer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == ASTRAI_MOE_BF16)
    return launch_route_grad<bf16_t>(logits, topk_idx, dw, n_tokens, n_experts, top_k, dlogits, s);
  return launch_route_grad<float>(logits, topk_idx, dw, n_tokens, n_experts, top_k, dlogits, s);
}
