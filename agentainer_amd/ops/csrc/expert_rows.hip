// Mixture-of-experts rows of a prompt step (gfx950): router, expert order,
// gather and weighted return around the per-expert library products.
//
// The products need each expert's rows side by side and their number on the
// host. Finding them expert by expert with tensor ops took some 20 launches
// and a host wait per expert; here the (token, choice) pairs are sorted by
// expert in one launch, the host waits once a layer for the counts, and the
// rows move in one gather and one return for all experts. All four kernels
// are bound by memory (rows in, rows out); none measures above 20 us at 1536
// rows of 4096, two choices of eight experts.

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include "expert_route.h"

namespace {

// Workgroup e: the pairs that chose expert e, in order, behind those of the
// experts below it. place[pair] is where the pair's row goes.
__global__ __launch_bounds__(256) void sort_pairs_kernel(
    int* __restrict__ order, int* __restrict__ place, int* __restrict__ counts,
    const int* __restrict__ choice, int pairs) {
  const int e = blockIdx.x;
  const int lane = threadIdx.x % WAVE, wid = threadIdx.x / WAVE;
  __shared__ int tot[2][4];
  int below = 0;
  for (int p = threadIdx.x; p < pairs; p += 256) below += choice[p] < e;
  below = (int)wave_sum((float)below);  // exact: at most 2^24 pairs
  if (lane == 0) tot[0][wid] = below;
  __syncthreads();
  const int base = tot[0][0] + tot[0][1] + tot[0][2] + tot[0][3];
  int at = base;
  for (int p0 = 0; p0 < pairs; p0 += 256) {
    const int p = p0 + threadIdx.x;
    const bool mine = p < pairs && choice[p] == e;
    const unsigned long long all = __ballot(mine);
    if (lane == 0) tot[1][wid] = __popcll(all);
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w < wid) before += tot[1][w];
      total += tot[1][w];
    }
    if (mine) {
      const int pos = at + before + __popcll(all & ((1ull << lane) - 1));
      order[pos] = p;
      place[p] = pos;
    }
    at += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) counts[e] = at - base;
}

__global__ __launch_bounds__(256) void gather_pairs_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    const int* __restrict__ order, int top_k, int h8) {
  const long pos = blockIdx.x;
  const bf16x8* src =
      reinterpret_cast<const bf16x8*>(x) + (long)(order[pos] / top_k) * h8;
  bf16x8* dst = reinterpret_cast<bf16x8*>(out) + pos * h8;
  for (int i = threadIdx.x; i < h8; i += 256) dst[i] = src[i];
}

// out[t] = sum over choices of weight * row, fp32
__global__ __launch_bounds__(256) void return_pairs_kernel(
    short* __restrict__ out, const short* __restrict__ y,
    const int* __restrict__ place, const float* __restrict__ weight, int top_k,
    int h8) {
  const long t = blockIdx.x;
  for (int i = threadIdx.x; i < h8; i += 256) {
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.f;
    for (int c = 0; c < top_k; ++c) {
      const float w = weight[t * top_k + c];
      const bf16x8 v = reinterpret_cast<const bf16x8*>(
          y)[(long)place[t * top_k + c] * h8 + i];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = fmaf(w, bits2f(v[j]), acc[j]);
    }
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = f2bits(acc[j]);
    reinterpret_cast<bf16x8*>(out)[t * h8 + i] = o;
  }
}

void check_rows(const torch::Tensor& x) {
  TORCH_CHECK(x.is_contiguous() && x.scalar_type() == at::kBFloat16 &&
              x.dim() == 2 && x.size(1) % 8 == 0 &&
              reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0);
}
void check_ints(const torch::Tensor& x, long n) {
  TORCH_CHECK(x.is_contiguous() && x.scalar_type() == at::kInt &&
              x.numel() == n);
}

}  // namespace

// choice [T, top_k], weight [T, top_k]; order, place [T * top_k]; counts [E]
void route_rows(torch::Tensor choice, torch::Tensor weight, torch::Tensor order,
                torch::Tensor place, torch::Tensor counts, torch::Tensor x,
                torch::Tensor router) {
  check_rows(x);
  check_rows(router);
  const int T = x.size(0), K = x.size(1), E = router.size(0);
  const int top_k = choice.size(1);
  TORCH_CHECK(router.size(1) == K && E <= MAX_EXPERTS && top_k <= E);
  TORCH_CHECK((long)T * top_k < (1 << 24));
  check_ints(choice, (long)T * top_k);
  check_ints(order, (long)T * top_k);
  check_ints(place, (long)T * top_k);
  check_ints(counts, E);
  TORCH_CHECK(weight.is_contiguous() && weight.scalar_type() == at::kFloat &&
              weight.numel() == choice.numel());
  if (T == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(route_kernel<false>, dim3(T), dim3(256), 0, stream,
                     choice.data_ptr<int>(), weight.data_ptr<float>(),
                     (const short*)x.data_ptr(), (const short*)router.data_ptr(),
                     K, 0, E, top_k);
  hipLaunchKernelGGL(sort_pairs_kernel, dim3(E), dim3(256), 0, stream,
                     order.data_ptr<int>(), place.data_ptr<int>(),
                     counts.data_ptr<int>(), choice.data_ptr<int>(),
                     T * top_k);
}

void gather_pairs(torch::Tensor out, torch::Tensor x, torch::Tensor order,
                  long top_k) {
  check_rows(x);
  check_rows(out);
  const long pairs = x.size(0) * top_k;
  check_ints(order, pairs);
  TORCH_CHECK(out.size(0) == pairs && out.size(1) == x.size(1));
  if (pairs == 0) return;
  hipLaunchKernelGGL(gather_pairs_kernel, dim3(pairs), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), (short*)out.data_ptr(),
                     (const short*)x.data_ptr(), order.data_ptr<int>(),
                     (int)top_k, (int)(x.size(1) / 8));
}

void return_pairs(torch::Tensor out, torch::Tensor y, torch::Tensor place,
                  torch::Tensor weight, long top_k) {
  check_rows(y);
  check_rows(out);
  const long pairs = out.size(0) * top_k;
  check_ints(place, pairs);
  TORCH_CHECK(y.size(0) == pairs && y.size(1) == out.size(1));
  TORCH_CHECK(weight.is_contiguous() && weight.scalar_type() == at::kFloat &&
              weight.numel() == pairs);
  if (pairs == 0) return;
  hipLaunchKernelGGL(return_pairs_kernel, dim3(out.size(0)), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), (short*)out.data_ptr(),
                     (const short*)y.data_ptr(), place.data_ptr<int>(),
                     weight.data_ptr<float>(), (int)top_k,
                     (int)(out.size(1) / 8));
}
