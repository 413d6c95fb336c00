// Expert selection of the Kimi-K3 MoE router on the GPU (lazy_lora/core/moe_router.py:55-123).
//
// The gate product logits = x . W^T is a plain dense GEMM and runs in the platform BLAS; this
// kernel does the rest per token, one wave per token: scores = sigmoid(logits), the top_k
// largest of scores + bias (the bias steers selection only), the unbiased scores of the chosen
// experts renormalised by their sum + 1e-20 and multiplied by the scaling factor. The indices
// are written in descending order of the biased score, like torch.topk(sorted=True); equal
// scores go to the lower expert id first.
#include "mx_device.h"
#include "mx_kernels.h"

namespace mx {

namespace {

// The choice values as whole numbers in selection order: NaN first (torch.topk ranks NaN above every
// number), then the larger value; 0 stands for "not selectable" (below every float's key). A choice
// is never -0 (a score is at least +0), so equal values have equal keys.
__device__ __forceinline__ uint32_t order_key(float v)
{
  const uint32_t u = f_bits(v);
  return v != v ? 0xFFFFFFFFu : u & 0x80000000u ? ~u : u | 0x80000000u;
}
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_umax(uint32_t v)
{
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false));
}
// Largest key of the wave: a DPP butterfly within each row of 16 lanes, then the four rows' lanes.
__device__ __forceinline__ uint32_t wave_max_key(uint32_t v)
{
  v = dpp_umax<kDppXor1>(v);
  v = dpp_umax<kDppXor2>(v);
  v = dpp_umax<kDppHalfMirror>(v);
  v = dpp_umax<kDppMirror>(v);
  const uint32_t a = __builtin_amdgcn_readlane((int)v, 0), b = __builtin_amdgcn_readlane((int)v, 16);
  const uint32_t c = __builtin_amdgcn_readlane((int)v, 32), d = __builtin_amdgcn_readlane((int)v, 48);
  return max(max(a, b), max(c, d));
}

// One wave per token, lane l holding experts l + 64 m. A selection round is bound by its serial
// chain, not by data (1024 x 896 logits are 3.7 MB): the lanes' largest open keys meet in four DPP
// steps and four lane reads, one ballot names the owner (a second one only if several lanes tie),
// which retires the expert and hands over its score from a register. Rounds of twelve cross-lane
// shuffles and a dependent load of the winner's logit took 49 us for 1024 tokens, top-16 of 896;
// this form 14.
template <int PER_LANE>
__global__ __launch_bounds__(256) void router_topk_kernel(long long* __restrict__ topk_idx, float* __restrict__ topk_w,
                                                          const float* __restrict__ logits,
                                                          const float* __restrict__ bias, int N, int E, int top_k,
                                                          float scale, int renormalize)
{
  const int lane = threadIdx.x & 63;
  const int token = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (token >= N) return;  // whole waves leave together
  const float* row = logits + (long long)token * E;

  float score[PER_LANE];
  uint32_t key[PER_LANE];  // 0: absent or already chosen
  uint32_t best = 0;
  // (static_for: the arrays' indices are constants from the start, so they are registers of their own and
  // not one tuple that every branch below copies)
  static_for<PER_LANE>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    const int e = lane + 64 * m;
    score[m] = e < E ? row[e] : 0.f;
  });
  static_for<PER_LANE>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    const int e = lane + 64 * m;
    key[m] = 0;
    if (e < E) {
      score[m] = 1.0f / (1.0f + expf(-score[m]));
      key[m] = order_key(bias ? score[m] + bias[e] : score[m]);
    }
    best = max(best, key[m]);
  });

  float sum = 0.f;
  float mine = 0.f;  // lane t keeps the t-th chosen score
  int mine_idx = 0;
  for (int t = 0; t < top_k; ++t) {
    const uint32_t win = wave_max_key(best);
    // the lowest expert id among the open entries with this key: every lane's lowest m, then, if
    // several lanes hold one, the lowest id
    int mm = PER_LANE;
    float s_mm = 0.f;
    static_for<PER_LANE>([&](auto mc) {
      constexpr int m = PER_LANE - 1 - decltype(mc)::value;
      const bool hit = key[m] == win;
      mm = hit ? m : mm;
      s_mm = hit ? score[m] : s_mm;
    });
    const uint64_t holders = __builtin_amdgcn_ballot_w64(best == win);
    int owner = __builtin_ctzll(holders);
    if (holders & (holders - 1)) {  // uniform, rare
      int id = best == win ? lane + 64 * mm : 0x7fffffff;
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) id = min(id, __shfl_xor(id, off, 64));
      owner = id & 63;
    }
    owner = __builtin_amdgcn_readfirstlane(owner);
    const int e = owner + 64 * __builtin_amdgcn_readlane(mm, owner);
    const float s = bits_f((uint32_t)__builtin_amdgcn_readlane((int)f_bits(s_mm), owner));  // the unbiased score
    // the owner retires it
    uint32_t nb = 0;
    static_for<PER_LANE>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      key[m] = lane == owner && m == mm ? 0u : key[m];
      nb = max(nb, key[m]);
    });
    best = nb;
    sum += s;
    if (lane == t) {
      mine = s;
      mine_idx = e;
    }
  }
  if (lane < top_k) {
    float w = mine;
    if (renormalize && top_k > 1) w = w / (sum + 1e-20f);
    topk_idx[(long long)token * top_k + lane] = mine_idx;
    topk_w[(long long)token * top_k + lane] = w * scale;
  }
}

// Gradient of the combine weights with respect to the logits, the autograd of the torch
// branch (moe_router.py:86-98), which the trainer relies on to carry dL/dtopk_w back into the
// router's input (lazy_lora/trainer/lazy_trainer.py:842-844). With s_j the chosen scores,
// S = sum_j s_j + 1e-20 and c the scaling factor:
//   w_j = c s_j / S          (renormalised)  =>  dL/ds_i = c (g_i / S - sum_j g_j s_j / S^2)
//   w_j = c s_j              (otherwise)     =>  dL/ds_i = c g_i
// and dL/dlogit_i = dL/ds_i s_i (1 - s_i) for chosen experts, 0 for the others (the selection
// itself has no gradient, and neither has the bias). One wave per token writes its whole row.
template <int PER_LANE>
__global__ __launch_bounds__(256) void router_topk_bwd_kernel(float* __restrict__ grad_logits,
                                                              const long long* __restrict__ topk_idx,
                                                              const float* __restrict__ grad_w,
                                                              const float* __restrict__ logits, int N, int E,
                                                              int top_k, float scale, int renormalize)
{
  const int lane = threadIdx.x & 63;
  const int token = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (token >= N) return;
  const float* row = logits + (long long)token * E;

  int e = -1;
  float s = 0.f, sm = 0.f, g = 0.f;  // sm = sigmoid(-x) = 1 - s, without the cancellation of 1 - s
  if (lane < top_k) {
    const long long v = topk_idx[(long long)token * top_k + lane];
    if (v >= 0 && v < E) {
      e = (int)v;
      s = 1.0f / (1.0f + expf(-row[e]));
      sm = 1.0f / (1.0f + expf(row[e]));
      g = grad_w[(long long)token * top_k + lane];
    }
  }
  float S = s, G = g * s;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    S += __shfl_xor(S, off, 64);
    G += __shfl_xor(G, off, 64);
  }
  float ds;
  if (renormalize && top_k > 1) {
    const float den = S + 1e-20f;
    ds = scale * (g / den - G / (den * den));
  } else {
    ds = scale * g;
  }
  const float val = ds * s * sm;  // sigmoid'(x) = s (1 - s), its small factor computed directly

  float out[PER_LANE];
#pragma unroll
  for (int m = 0; m < PER_LANE; ++m) out[m] = 0.f;
  for (int j = 0; j < top_k; ++j) {
    const int ej = __builtin_amdgcn_readlane(e, j);
    const float vj = bits_f((uint32_t)__builtin_amdgcn_readlane((int)f_bits(val), j));
    if (ej < 0) continue;  // uniform
#pragma unroll
    for (int m = 0; m < PER_LANE; ++m)
      if (lane + 64 * m == ej) out[m] += vj;
  }
  float* orow = grad_logits + (long long)token * E;
#pragma unroll
  for (int m = 0; m < PER_LANE; ++m) {
    const int c = lane + 64 * m;
    if (c < E) orow[c] = out[m];
  }
}

}  // namespace

hipError_t launch_router_topk_bwd(float* grad_logits, const long long* topk_idx, const float* grad_w,
                                  const float* logits, int N, int E, int top_k, float scale, int renormalize,
                                  hipStream_t s)
{
  if (N <= 0) return hipSuccess;
  dim3 grid((unsigned)((N + 3) / 4)), block(256);
  if (E <= 16 * 64)
    hipLaunchKernelGGL(router_topk_bwd_kernel<16>, grid, block, 0, s, grad_logits, topk_idx, grad_w, logits, N, E,
                       top_k, scale, renormalize);
  else
    hipLaunchKernelGGL(router_topk_bwd_kernel<64>, grid, block, 0, s, grad_logits, topk_idx, grad_w, logits, N, E,
                       top_k, scale, renormalize);
  return hipGetLastError();
}

hipError_t launch_router_topk(long long* topk_idx, float* topk_w, const float* logits, const float* bias, int N,
                              int E, int top_k, float scale, int renormalize, hipStream_t s)
{
  if (N <= 0) return hipSuccess;
  dim3 grid((unsigned)((N + 3) / 4)), block(256);
  if (E <= 16 * 64)
    hipLaunchKernelGGL(router_topk_kernel<16>, grid, block, 0, s, topk_idx, topk_w, logits, bias, N, E, top_k, scale,
                       renormalize);
  else
    hipLaunchKernelGGL(router_topk_kernel<64>, grid, block, 0, s, topk_idx, topk_w, logits, bias, N, E, top_k, scale,
                       renormalize);
  return hipGetLastError();
}

}  // namespace mx
