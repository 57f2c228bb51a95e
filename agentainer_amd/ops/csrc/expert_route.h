// The router of a mixture, for packed rows (stream_gemm.hip) and row-major
// ones (expert_rows.hip).
#pragma once

#include "common.h"

namespace {

constexpr int MAX_EXPERTS = 16;

// One token per workgroup: fp32 logits of E experts, the top_k largest (lowest
// index first among equals), softmax weights over the chosen ones. Rows are
// packed in `groups` 16-row groups, or row-major.
template <bool PACKED>
__global__ __launch_bounds__(256) void route_kernel(
    int* __restrict__ choice, float* __restrict__ weight,
    const short* __restrict__ x, const short* __restrict__ router, int K,
    int groups, int E, int top_k) {
  const long row = blockIdx.x;
  float acc[MAX_EXPERTS];
#pragma unroll
  for (int e = 0; e < MAX_EXPERTS; ++e) acc[e] = 0.f;
  for (int k = threadIdx.x * 8; k < K; k += 256 * 8) {
    const bf16x8 v = *reinterpret_cast<const bf16x8*>(
        x + (PACKED ? packed_at((int)row, k, groups) : row * K + k));
#pragma unroll
    for (int e = 0; e < MAX_EXPERTS; ++e) {
      if (e >= E) break;
      const bf16x8 r =
          *reinterpret_cast<const bf16x8*>(router + (long)e * K + k);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        acc[e] = fmaf(bits2f(v[j]), bits2f(r[j]), acc[e]);
    }
  }
  __shared__ float red[4][MAX_EXPERTS];
#pragma unroll
  for (int e = 0; e < MAX_EXPERTS; ++e) {
    if (e >= E) break;
    const float s = wave_sum(acc[e]);
    if (threadIdx.x % WAVE == 0) red[threadIdx.x / WAVE][e] = s;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  float logit[MAX_EXPERTS], mx = -INFINITY;
  for (int e = 0; e < E; ++e) {
    logit[e] = red[0][e] + red[1][e] + red[2][e] + red[3][e];
    mx = fmaxf(mx, logit[e]);
  }
  // the softmax's denominator cancels in the renormalized weights
  unsigned taken = 0;
  float sum = 0.f;
  for (int i = 0; i < top_k; ++i) {
    int best = -1;
    for (int e = 0; e < E; ++e)
      if (!(taken >> e & 1) && (best < 0 || logit[e] > logit[best])) best = e;
    taken |= 1u << best;
    choice[row * top_k + i] = best;
    const float p = __expf(logit[best] - mx);
    weight[row * top_k + i] = p;
    sum += p;
  }
  for (int i = 0; i < top_k; ++i) weight[row * top_k + i] /= sum;
}

}  // namespace
