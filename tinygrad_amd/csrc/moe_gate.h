// Expert gating + pairwise top-k of one token on one wave (tinygrad/llm/model.py:35-41, 110-121); shared by the MoE kernels and the
// expert GEMV that routes for itself.
#pragma once
#include "common.h"

// At most 64 experts of which few are taken (every model of the benchmarks): expert = lane, nothing in LDS.  The k largest scores are taken one after the other, the largest first - the wave's
// maximum, of the lanes that hold it the lowest - which is the pairwise rank below as long as no score is NaN (those rank by themselves: the general way).  k steps of a reduction in registers,
// about 80 cycles each, against as many reads of LDS as there are experts, with their comparisons, and a maximum by way of LDS.  A launch of moe_gate_kernel, us, in lanes / the general way: 64 experts, one token,
// k 1 / 8 / 16: 2.9 / 2.9 / 3.4 against 5.6; 4096 tokens 3.0 / 3.8 / 5.0 against 7.5; 16 experts, 4096 tokens, k 4 / 8 3.3 / 3.8 against 4.5, k 16 5.0 against 4.5 (not taken).
__host__ __device__ __forceinline__ bool gate_in_lanes(int n_experts, int k) { return n_experts <= 64 && (k <= 8 || (k <= 16 && 2 * k <= n_experts)); }
__device__ __forceinline__ int gate_kind(int gating, int norm_topk) { return gating == 1 && norm_topk ? 3 : gating; }      // model.py:116-117: softmax over the selected is all there is to it
// the score of expert `lane` from its logit v (lanes behind the last expert: any v); false: a score is NaN
__device__ __forceinline__ bool gate_score_lane(float v, int n_experts, int kind, int lane, float& s) {
  const bool has = lane < n_experts;
  if (kind == 3) s = v;
  else if (kind == 1) {
    const float mx = wave_max_dpp(has ? v : -INFINITY), e = has ? expf(v - mx) : 0.f, sum = wave_sum(e);
    s = e * (1.0f / sum);
  } else if (kind == 2) s = 1.0f / (1.0f + expf(-v));
  else s = sqrtf(log1pf(expf(v)));
  return __ballot(has && !(s == s)) == 0;
}
// the experts of the slots k - 1 down to `slot`: lane j holds slot j's expert and score, the result is slot's expert
__device__ __forceinline__ int gate_pick_lanes(float s, int n_experts, int k, int slot, int lane, int& sel, float& p) {
  unsigned long long left = n_experts >= 64 ? ~0ull : (1ull << n_experts) - 1;
  float c = lane < n_experts ? s : -INFINITY;
  int e = 0;
  sel = 0; p = 0.f;
  for (int j = k - 1; j >= slot; j--) {
    e = __builtin_ctzll(__ballot(c == wave_max_dpp(c)) & left);
    left &= ~(1ull << e);
    const float se = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, s), e));
    if (lane == e) c = -INFINITY;
    if (lane == j) { sel = e; p = se; }
  }
  return e;
}
// the weight of slot `lane` (below k) from the slots' scores
__device__ __forceinline__ float gate_weight_lanes(float p, int k, int gating, int norm_topk, float scale, int lane) {
  auto sum = [&](float v) { float z = 0.f; for (int j = 0; j < k; j++) z += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), j)); return z; };
  if (gate_kind(gating, norm_topk) == 3) {                // softmax over the selected logits
    const float e = expf(p - wave_max_dpp(lane < k ? p : -INFINITY));
    p = e * (1.0f / sum(e));
    if (gating == 1) norm_topk = 0;
  }
  if (norm_topk) p = p / sum(p);
  return p * scale;
}

// scores per ExpertGating (model.py:9-13, 116-121): 1 SOFTMAX, 2 SIGMOID, 3 SOFTMAX_WEIGHT (softmax over the selected logits),
// 4 SQRT_SOFTPLUS.  Top-k by pairwise rank exactly as pairwise_topk (model.py:35-41): rank_i = #{j: s_i > s_j or (s_i == s_j and
// i < j)}; the k highest ranks are emitted in ASCENDING rank order (the largest last), so among equal scores the lower index
// ranks higher.  Runs on ONE wave (lane = threadIdx.x & 63 of the calling wave); lg may live in LDS or global memory, sc is
// n_experts floats of LDS, tmp 192 floats of LDS.  The caller separates the call from earlier LDS writes with a barrier.
// bias (optional, n_experts floats): the expert selection bias of model.py:113, 123 - experts are ranked by score + bias, the weights are
// gathered from the unbiased scores; scb is then n_experts more floats of LDS for the biased scores (without a bias pass scb = sc).
__device__ __forceinline__ void gate_topk_wave(const float* lg, int n_experts, int k, int gating, int norm_topk, float scale,
                                               int* __restrict__ sel, float* __restrict__ probs, float* sc, float* tmp, int lane,
                                               const float* bias = nullptr, float* scb = nullptr) {
  int* s_sel = (int*)tmp; float* s_p = tmp + 64; float* s_q = tmp + 128;
  if (!bias && gate_in_lanes(n_experts, k)) {
    float s, p; int e;
    if (gate_score_lane(lg[lane < n_experts ? lane : n_experts - 1], n_experts, gate_kind(gating, norm_topk), lane, s)) {
      gate_pick_lanes(s, n_experts, k, 0, lane, e, p);
      p = gate_weight_lanes(p, k, gating, norm_topk, scale, lane);
      if (lane < k) { s_sel[lane] = e; sel[lane] = e; probs[lane] = p; }
      return;
    }
  }
  if (!bias) scb = sc;
  if (gating == 1 && norm_topk && !bias) { gating = 3; norm_topk = 0; }   // model.py:116-117 fast path (only without a selection bias)
  float mx = -INFINITY;
  for (int i = lane; i < n_experts; i += 64) mx = fmaxf(mx, lg[i]);
  mx = wave_max(mx);
  float sum = 0.f;
  if (gating == 1) { for (int i = lane; i < n_experts; i += 64) sum += expf(lg[i] - mx); sum = wave_sum(sum); }
  for (int i = lane; i < n_experts; i += 64) {
    const float v = lg[i];
    float s;
    if (gating == 3) s = v;
    else if (gating == 1) s = expf(v - mx) * (1.0f / sum);
    else if (gating == 2) s = 1.0f / (1.0f + expf(-v));
    else s = sqrtf(log1pf(expf(v)));
    sc[i] = s;
    if (bias) scb[i] = s + bias[i];
  }
  s_sel[lane] = 0; s_p[lane] = 0.f;                       // a slot no rank lands in (NaN scores compare false with everything) selects expert 0, like the reference's zero-filled scatter
  __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_s_waitcnt(0xc07f);   // this wave's LDS writes are visible to its own lanes
  for (int i = lane; i < n_experts; i += 64) {
    const float si = scb[i];
    int rank = 0;
    for (int j = 0; j < n_experts; j++) { const float sj = scb[j]; rank += (si > sj) || (si == sj && i < j); }
    const int slot = rank - (n_experts - k);
    if (slot >= 0) { s_sel[slot] = i; s_p[slot] = sc[i]; }
  }
  __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_s_waitcnt(0xc07f);
  float p = lane < k ? s_p[lane] : 0.f;
  if (gating == 3 && lane < k) {                          // softmax over the selected logits
    float m2 = -INFINITY; for (int j = 0; j < k; j++) m2 = fmaxf(m2, s_p[j]);
    float z = 0.f; for (int j = 0; j < k; j++) z += expf(s_p[j] - m2);
    p = expf(p - m2) * (1.0f / z);
  }
  s_q[lane] = p;
  __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_s_waitcnt(0xc07f);
  if (lane < k) {
    if (norm_topk) { float z = 0.f; for (int j = 0; j < k; j++) z += s_q[j]; p = p / z; }
    sel[lane] = s_sel[lane];
    probs[lane] = p * scale;
  }
}

