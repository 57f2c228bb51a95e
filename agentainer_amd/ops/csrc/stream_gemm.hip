// Decode projections (gfx950): x[M, K] @ W[N, K]^T for few rows, with bf16
// weights in the fragment-linear layout of ops.pack_weight, dense or as the
// experts of a mixture.
//
// HBM-bound: W is read once, everything else is small. Each workgroup owns NT
// 16-column tiles and splits K over its WV waves, so no wave waits for another
// until the end: a wave streams its own contiguous run of every tile (one
// fragment per load instruction, non-temporal, U fragments a tile in flight
// while the previous U multiply) and reads the x fragments it needs, packed,
// from L2. The waves' sums meet in LDS once, where one thread per four values
// adds them and applies the epilogue:
//
//   BF16   out bf16 [M, N]
//   PARTS  out fp32 [split, M, N], summed by the kernel that consumes it
//          (add_parts_rmsnorm); split > 1 where one split would leave CUs idle
//   SILU   W = [gate; up]: a workgroup holds both tiles of its columns and
//          writes silu(gate) * up as packed rows of N / 2; the products
//          never round to bf16 in between
//
// GROUPED: blockIdx.y is an expert, its rows are the (token, choice) pairs
// routed to it (listed from the choices by every workgroup for itself; an
// expert nobody chose costs nothing). The rows are gathered out of the packed
// x in place. SILU writes row `pair`, PARTS writes weight * product into part
// `choice` of its token.
//
// Up to 64 rows; 65 to 128 rows take wide_gemm_kernel below.
//
// W is the A operand and x^T the B operand, so a lane ends up with four
// consecutive output columns of one row.

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <algorithm>
#include <vector>
#include "common.h"
#include "expert_route.h"

namespace {

typedef __bf16 bf16v8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16v4 __attribute__((ext_vector_type(4)));
typedef int i32x4v __attribute__((ext_vector_type(4)));

enum Mode { BF16 = 0, PARTS = 1, SILU = 2 };
constexpr int MAX_PAIRS = 128;

constexpr int FRAG_K = 32;           // k per fragment
constexpr int LANE_BYTES = 16;       // what a lane holds of one
constexpr int FRAG_BYTES = LANE_BYTES * WAVE;

struct StreamArgs {
  void* out;
  const char* x;        // packed rows
  int M, N, steps, steps_per_split;
  int x_groups;         // 16-row groups of the packed x
  // GROUPED
  const int* choice;    // [M, top_k] expert of each pair
  const float* weight;  // [M, top_k]
  int n_pairs, top_k, out_groups;
};

// weights per expert
template <bool GROUPED>
struct Weights {
  const char* w[GROUPED ? MAX_EXPERTS : 1];
};

// At most four waves a SIMD: aiming higher, the compiler moves the loads down
// to their uses to save registers (gate_up at one row 40.9 instead of 40.2 us).
template <int MODE, int MS, int NT, int WV, int U, bool GROUPED>
__global__ __launch_bounds__(WV * WAVE)
__attribute__((amdgpu_waves_per_eu(WV / 4, 4))) void stream_gemm_kernel(
    const StreamArgs a, const Weights<GROUPED> weights) {
  typedef bf16v8 frag;
  constexpr int LB = LANE_BYTES, FB = FRAG_BYTES;
  const int lane = threadIdx.x % WAVE;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int l16 = lane % 16, lg = lane / 16;
  const int n_tiles = a.N / 16;
  const int expert = GROUPED ? blockIdx.y : 0;
  const int s_begin = GROUPED ? 0 : blockIdx.y * a.steps_per_split;
  const int s_end = min(s_begin + a.steps_per_split, a.steps);
  const int per = (s_end - s_begin + WV - 1) / WV;
  const int first = s_begin + wid * per;
  const int last = min(first + per, s_end);

  // this expert's pairs
  __shared__ int list[GROUPED ? MAX_PAIRS : 1];
  int count = a.M;
  if (GROUPED) {
    count = 0;
#pragma unroll
    for (int h = 0; h < MAX_PAIRS / WAVE; ++h) {
      const int p = h * WAVE + lane;
      const bool mine = p < a.n_pairs && a.choice[p] == expert;
      const unsigned long long all = __ballot(mine);
      if (mine && wid == 0)
        list[count + __popcll(all & ((1ull << lane) - 1))] = p;
      count += __popcll(all);
    }
    if (count == 0) return;
    __syncthreads();
  }

  auto tile_of = [&](int nt) {
    const int t = MODE == SILU
                      ? (nt < NT / 2 ? (int)blockIdx.x * (NT / 2) + nt
                                     : n_tiles / 2 + (int)blockIdx.x * (NT / 2) +
                                           nt - NT / 2)
                      : (int)blockIdx.x * NT + nt;
    return min(t, n_tiles - 1);
  };
  // uniform bases with 32-bit lane offsets: the loads take them apart, and no
  // VGPR pair goes to an address
  const char* x = a.x;
  const int x_groups = GROUPED ? a.x_groups : MS;
  const unsigned w_off = lane * LB;
  const char* wt[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    wt[nt] = weights.w[expert] + (long)tile_of(nt) * a.steps * FB;

  __shared__ f32x4 red[WV][MS][WAVE];
  constexpr int ITEMS = MS * WAVE;

  for (int r0 = 0; r0 < count; r0 += MS * 16) {
    // row of x behind slot m (slots past the last one repeat the first)
    auto pair_of = [&](int m) { return GROUPED ? list[m < count ? m : 0] : m; };
    unsigned x_off[MS];
#pragma unroll
    for (int ms = 0; ms < MS; ++ms) {
      if (!GROUPED) {
        x_off[ms] = ms * FB + lane * LB;
        continue;
      }
      const int p = pair_of(r0 + ms * 16 + l16);
      const int t = GROUPED && MODE == SILU ? p / a.top_k : p;
      x_off[ms] = t / 16 * FB + (lg * 16 + t % 16) * LB;
    }

    f32x4 acc[NT][MS];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) acc[nt][ms] = f32x4{0.f, 0.f, 0.f, 0.f};

    frag wa[U][NT], xa[U][MS], wb[U][NT], xb[U][MS];
    auto load = [&](frag (&wf)[U][NT], frag (&xf)[U][MS], int step) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int s = min(step + u, last - 1);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const char* ws = wt[nt] + (long)s * FB;
          wf[u][nt] = __builtin_nontemporal_load(
              reinterpret_cast<const frag*>(ws + w_off));
        }
        const char* xs = x + (long)s * (x_groups * FB);
#pragma unroll
        for (int ms = 0; ms < MS; ++ms)
          xf[u][ms] = *reinterpret_cast<const frag*>(xs + x_off[ms]);
      }
    };
    auto multiply = [&](frag (&wf)[U][NT], frag (&xf)[U][MS], int step) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (u == 0 || step + u < last) {
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int ms = 0; ms < MS; ++ms)
              acc[nt][ms] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  wf[u][nt], xf[u][ms], acc[nt][ms], 0, 0, 0);
        }
    };
    // No load of the main loop is conditional: behind a branch that may or may
    // not have issued loads the compiler has to wait for all of them.
    if (first < last) {
      int s = first;
      load(wa, xa, s);
      while (s + 2 * U < last) {
        load(wb, xb, s + U);
        multiply(wa, xa, s);
        load(wa, xa, s + 2 * U);
        multiply(wb, xb, s + U);
        s += 2 * U;
      }
      if (s + U < last) {
        load(wb, xb, s + U);
        multiply(wa, xa, s);
        multiply(wb, xb, s + U);
      } else {
        multiply(wa, xa, s);
      }
    }

    // the waves' sums, one tile (SILU: one gate tile, then its up tile) a
    // round
    f32x4 gate[(ITEMS + WV * WAVE - 1) / (WV * WAVE)];
#pragma unroll
    for (int r = 0; r < NT; ++r) {
      const int nt = MODE == SILU ? (r % 2) * (NT / 2) + r / 2 : r;
      if (r || (GROUPED && r0)) __syncthreads();
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) red[wid][ms][lane] = acc[nt][ms];
      __syncthreads();
#pragma unroll
      for (int i = 0; i * WV * WAVE < ITEMS; ++i) {
        const int e = i * WV * WAVE + threadIdx.x;
        if (e >= ITEMS) continue;
        f32x4 v = red[0][e / WAVE][e % WAVE];
#pragma unroll
        for (int q = 1; q < WV; ++q) {
          const f32x4 o = red[q][e / WAVE][e % WAVE];
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] += o[j];
        }
        // value j is slot m, column n + j
        const int m = r0 + (e / WAVE) * 16 + e % 16;
        const int t = MODE == SILU ? (int)blockIdx.x * (NT / 2) + r / 2
                                   : (int)blockIdx.x * NT + nt;
        if (MODE == SILU && r % 2 == 0) {
          gate[i] = v;
          continue;
        }
        if (t >= (MODE == SILU ? n_tiles / 2 : n_tiles)) continue;
        if (MODE == SILU) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float g = gate[i][j];
            v[j] = g / (1.f + __expf(-g)) * v[j];
          }
        }
        const int n = t * 16 + (e % WAVE) / 16 * 4;
        if (m >= count) continue;
        auto at = [&]() -> long {
          if (MODE == SILU)
            return packed_at(pair_of(m), n, GROUPED ? a.out_groups : MS);
          if (MODE == PARTS && GROUPED) {
            const int p = pair_of(m);
            return ((long)(p % a.top_k) * a.M + p / a.top_k) * a.N + n;
          }
          return (MODE == PARTS ? (long)blockIdx.y * a.M * a.N : 0) +
                 (long)m * a.N + n;
        };
        if (MODE == PARTS) {
          const float f = GROUPED ? a.weight[pair_of(m)] : 1.f;
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] *= f;
          *reinterpret_cast<f32x4*>((float*)a.out + at()) = v;
        } else {
          bf16x4 o;
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = f2bits(v[j]);
          *reinterpret_cast<bf16x4*>((short*)a.out + at()) = o;
        }
      }
    }
    if (!GROUPED) break;
  }
}

template <int MODE, int MS, int NT, int WV, bool GROUPED>
void launch(const StreamArgs& a, const Weights<GROUPED>& w, int grid_y) {
  // fragments in flight: about 8 KB of W a wave, less where x takes the room
  constexpr int U = NT * MS >= 8 ? 2 : NT * MS >= 2 ? 4 : 8;
  hipLaunchKernelGGL((stream_gemm_kernel<MODE, MS, NT, WV, U, GROUPED>),
                     dim3((a.N / 16 + NT - 1) / NT, grid_y), dim3(WV * WAVE),
                     0, at::hip::getCurrentHIPStream(), a, w);
}

template <int MODE, int NT, int WV>
void by_rows(const StreamArgs& a, const Weights<false>& w, int split) {
  switch (packed_groups(a.M)) {
    case 1: return launch<MODE, 1, NT, WV, false>(a, w, split);
    case 2: return launch<MODE, 2, NT, WV, false>(a, w, split);
    default: return launch<MODE, 4, NT, WV, false>(a, w, split);
  }
}

// Tiles per workgroup and waves, from a sweep over 1, 13, 32 and 64 rows of
// the 4096- and 8192-wide layers (us; best row-major library call, silu and
// split-K passes not counted):
//   gate_up 28672 x 4096    1 row 39 (62), 13: 39 (63), 32: 42 (54), 64: 46 (52)
//   down     4096 x 14336   1 row 20 (26), 13: 20 (27), 32: 22 (34), 64: 29 (41)
//   o        4096 x 4096    1 row  7 (15), 13:  8 (16), 32:  9 (13), 64: 11 (15)
//   qkv      6144 x 4096    1 row 11 (14), 13: 11 (16), 32: 13 (16), 64: 17 (18)
//   lm_head 128256 x 4096   1 row 163 (186), 13: 166 (187), 32: 182 (198),
//                           64: 213 (211)
// More rows mean more x per byte of W: four tiles share a fragment then, where
// N still gives enough workgroups.
void dispatch(const StreamArgs& a, const Weights<false>& w, int mode,
              int split) {
  if (mode == PARTS) return by_rows<PARTS, 2, 8>(a, w, split);
  if (mode == SILU)
    return a.M <= 16 ? by_rows<SILU, 2, 8>(a, w, 1)
                     : by_rows<SILU, 4, 4>(a, w, 1);
  if (a.M > 16 && a.N >= 32768)
    by_rows<BF16, 4, 4>(a, w, 1);
  else
    by_rows<BF16, 2, 8>(a, w, 1);
}

void dispatch_grouped(const StreamArgs& a, const Weights<true>& w, int mode,
                      int experts) {
  // rows of one expert: a choice in 16 of a batch's fits one group up to 16
  // rows; larger batches take two groups at a time and come back for more
  if (mode == PARTS) {
    if (a.n_pairs <= 16) launch<PARTS, 1, 2, 8, true>(a, w, experts);
    else launch<PARTS, 2, 2, 8, true>(a, w, experts);
  } else {
    if (a.n_pairs <= 16) launch<SILU, 1, 2, 8, true>(a, w, experts);
    else launch<SILU, 2, 2, 8, true>(a, w, experts);
  }
}

// ---- 65 to 128 rows, bf16 ----
//
// With more rows the packed x outweighs W: read by every workgroup out of L2
// it would bound the step (8 KB of x per KB of W and tile). Here a workgroup of
// 4 waves owns 8 tiles (two a wave) and stages x in LDS, two k steps (16 KB)
// at a time, double-buffered; the fragment order makes the staging a plain
// copy and every LDS access 1 KB contiguous. W goes straight to registers. A
// wave's two tiles are gate and up of the same columns in SILU; nothing
// crosses waves, so there is no reduction.
//
// Bound by the latency of one stage while a CU has one workgroup, hence the
// splits. 128 rows, us (best row-major library call, its silu not counted):
//   gate_up 28672 x 4096  58 (57)    down 4096 x 14336  32 (75)
//   o        4096 x 4096  14 (24)    lm_head           210 (234)
//   8192 x 28672          94 (200)   8192 x 8192        32 (48)
// A projection that is neither split nor large (qkv: 48 workgroups, 52 us
// against 26) is left to the library (ops.streams has the line), and so are
// more than 128 rows, where twice the x makes gate_up 81 us against 70. Two
// passes of 125 rows lose as well: gate_up 130 us against 88 with the library's
// silu, qkv 104 against 28, o 28 against 23, down 70 against 63.
template <int MODE>
__global__ __launch_bounds__(256, 2) void wide_gemm_kernel(
    void* __restrict__ out, const char* __restrict__ x,
    const char* __restrict__ w, int M, int N, int steps, int steps_per_split) {
  constexpr int MS = PACKED_ROWS / 16;
  constexpr int U = 2;                   // k steps per stage
  constexpr int STAGE = U * MS * 1024;   // bytes
  constexpr int CP = STAGE / (256 * 16); // 16-byte pieces per thread
  const int lane = threadIdx.x % WAVE;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int n_tiles = N / 16;
  const int s0 = blockIdx.y * steps_per_split;
  const int s1 = min(s0 + steps_per_split, steps);
  // one stage more than needed may be read: clamped to the last pair of steps
  __shared__ __attribute__((aligned(16))) char lds[2][STAGE];

  auto tile_of = [&](int nt) {
    const int t = MODE == SILU
                      ? nt * (n_tiles / 2) + (int)blockIdx.x * 4 + wid
                      : (int)blockIdx.x * 8 + wid * 2 + nt;
    return min(t, n_tiles - 1);
  };
  const char* wt[2];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) wt[nt] = w + (long)tile_of(nt) * steps * 1024;

  f32x4 acc[2][MS];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
#pragma unroll
    for (int ms = 0; ms < MS; ++ms) acc[nt][ms] = f32x4{0.f, 0.f, 0.f, 0.f};

  bf16v8 wa[U][2], wb[U][2];
  i32x4v st[CP];
  auto load_w = [&](bf16v8 (&wf)[U][2], int s) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
        wf[u][nt] = __builtin_nontemporal_load(reinterpret_cast<const bf16v8*>(
            wt[nt] + (long)min(s + u, s1 - 1) * 1024 + lane * 16));
  };
  auto load_x = [&](int s) {
#pragma unroll
    for (int i = 0; i < CP; ++i) {
      // piece i lies in one k step: its step is clamped like W's
      const int at = (i * 256 + (int)threadIdx.x) * 16;
      const int u = i * 256 * 16 / (MS * 1024);
      st[i] = *reinterpret_cast<const i32x4v*>(
          x + (long)min(s + u, s1 - 1) * (MS * 1024) + (at - u * MS * 1024));
    }
  };
  auto store_x = [&](int buf) {
#pragma unroll
    for (int i = 0; i < CP; ++i)
      *reinterpret_cast<i32x4v*>(lds[buf] + (i * 256 + threadIdx.x) * 16) =
          st[i];
  };
  auto multiply = [&](bf16v8 (&wf)[U][2], int s, int buf) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u == 0 || s + u < s1) {
#pragma unroll
        for (int ms = 0; ms < MS; ++ms) {
          const bf16v8 xf = *reinterpret_cast<const bf16v8*>(
              lds[buf] + (u * MS + ms) * 1024 + lane * 16);
#pragma unroll
          for (int nt = 0; nt < 2; ++nt)
            acc[nt][ms] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                wf[u][nt], xf, acc[nt][ms], 0, 0, 0);
        }
      }
  };
  load_x(s0);
  load_w(wa, s0);
  store_x(0);
  __syncthreads();
  // loads run one stage past the end (clamped), so none is conditional
  for (int s = s0; s < s1; s += 2 * U) {
    load_x(s + U);
    load_w(wb, s + U);
    multiply(wa, s, 0);
    store_x(1);
    __syncthreads();
    if (s + U >= s1) break;
    load_x(s + 2 * U);
    load_w(wa, s + 2 * U);
    multiply(wb, s + U, 1);
    store_x(0);
    __syncthreads();
  }

  const int l16 = lane % 16, quad = lane / 16 * 4;
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) {
    const int m = ms * 16 + l16;
    if (m >= M) continue;
#pragma unroll
    for (int nt = 0; nt < (MODE == SILU ? 1 : 2); ++nt) {
      const int t = MODE == SILU ? (int)blockIdx.x * 4 + wid
                                 : (int)blockIdx.x * 8 + wid * 2 + nt;
      if (t >= (MODE == SILU ? n_tiles / 2 : n_tiles)) continue;
      const int n = t * 16 + quad;
      if (MODE == PARTS) {
        *reinterpret_cast<f32x4*>(
            (float*)out + ((long)blockIdx.y * M + m) * N + n) = acc[nt][ms];
        continue;
      }
      f32x4 v = acc[nt][ms];
      if (MODE == SILU)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          v[j] = v[j] / (1.f + __expf(-v[j])) * acc[1][ms][j];
      *reinterpret_cast<bf16v4*>(
          (short*)out + (MODE == SILU ? packed_at(m, n, MS)
                                      : (long)m * N + n)) =
          __builtin_convertvector(v, bf16v4);
    }
  }
}

template <int MODE>
void launch_wide(const StreamArgs& a, const Weights<false>& w, int split) {
  const int tiles = a.N / 16;
  const dim3 grid(MODE == SILU ? (tiles / 2 + 3) / 4 : (tiles + 7) / 8, split);
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL((wide_gemm_kernel<MODE>), grid, dim3(256), 0, stream,
                     a.out, a.x, w.w[0], a.M, a.N, a.steps, a.steps_per_split);
}

void check_weight(const torch::Tensor& w, long N, long K) {
  TORCH_CHECK(w.is_contiguous() && w.scalar_type() == at::kBFloat16 &&
              w.numel() == N * K);
}
void check_packed(const torch::Tensor& x, long groups, long K) {
  TORCH_CHECK(x.is_contiguous() && x.scalar_type() == at::kBFloat16 &&
              x.numel() == groups * 16 * K);
}

}  // namespace

// Splits of K that give every CU a workgroup: N = 4096 (128 workgroups of two
// tiles) takes 2, N >= 8192 has 256 and fills the chip alone. Above
// 64 rows a workgroup has eight tiles and one stage's latency to hide (4096 x
// 4096 at 128 rows: 51 us unsplit, 29, 18 and 14 in 2, 4 and 8).
long stream_splits(long M, long N, long K) {
  long split = 1;
  if (M > 64) {
    while (split < 8 && N / 128 * split < 256 && K >= 1024 * split) split *= 2;
    return split;
  }
  while (split < 4 && N / 32 * split < 256 && K / 32 >= 64 * split) split *= 2;
  return split;
}

// mode 0: out bf16 [M, N]; 1: out fp32 [split, M, N]; 2: w = [gate; up], out
// packed rows of N / 2. x: packed rows of K.
void stream_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w, long M,
                 long N, long K, long mode, long split) {
  TORCH_CHECK(M >= 0 && M <= PACKED_ROWS && N % 32 == 0 && K % FRAG_K == 0,
              "stream_gemm: M <= 128, N and K multiples of a fragment");
  const long groups = packed_groups(M);
  check_packed(x, groups, K);
  check_weight(w, N, K);
  TORCH_CHECK(out.is_contiguous());
  const int steps = K / FRAG_K;
  TORCH_CHECK(split >= 1 && split <= steps &&
              (split - 1) * ((steps + split - 1) / split) < steps);
  TORCH_CHECK(mode >= BF16 && mode <= SILU);
  TORCH_CHECK(mode == PARTS || split == 1, "only parts are split");
  TORCH_CHECK(mode != SILU || N % 64 == 0,
              "stream_gemm: gate and up in whole fragments");
  TORCH_CHECK(out.numel() == (mode == PARTS  ? split * M * N
                              : mode == SILU ? groups * 16 * (N / 2)
                                             : M * N));
  TORCH_CHECK(out.scalar_type() ==
              (mode == PARTS ? at::kFloat : at::kBFloat16));
  if (M == 0) return;
  StreamArgs a{};
  a.out = out.data_ptr();
  a.x = (const char*)x.data_ptr();
  const Weights<false> wt{{(const char*)w.data_ptr()}};
  a.M = M;
  a.N = N;
  a.steps = steps;
  a.steps_per_split = (steps + split - 1) / split;
  a.x_groups = groups;
  if (M > 64) {
    if (mode == PARTS) launch_wide<PARTS>(a, wt, split);
    else if (mode == SILU) launch_wide<SILU>(a, wt, 1);
    else launch_wide<BF16>(a, wt, 1);
    return;
  }
  dispatch(a, wt, mode, split);
}

// The experts' half of a mixture: mode 2 (SILU) turns packed rows of T tokens
// into packed rows of T * top_k pairs, mode 1 (PARTS) those into fp32
// [top_k, T, N], each times its pair's weight.
void stream_gemm_experts(torch::Tensor out, torch::Tensor x,
                         std::vector<torch::Tensor> w, torch::Tensor choice,
                         torch::Tensor weight, long N, long K, long mode) {
  const int T = choice.size(0), top_k = choice.size(1);
  const int experts = w.size();
  TORCH_CHECK(choice.is_contiguous() && choice.scalar_type() == at::kInt &&
              weight.is_contiguous() && weight.scalar_type() == at::kFloat &&
              weight.numel() == choice.numel());
  TORCH_CHECK(experts >= 1 && experts <= MAX_EXPERTS);
  TORCH_CHECK(T <= 64 && T * top_k <= MAX_PAIRS);
  TORCH_CHECK(mode == PARTS || mode == SILU);
  TORCH_CHECK(N % (mode == SILU ? 64 : 32) == 0 && K % FRAG_K == 0);
  const int rows = mode == SILU ? T : T * top_k;
  const int x_groups = mode == SILU ? packed_groups(T) : (rows + 15) / 16;
  const int pair_groups = (T * top_k + 15) / 16;
  check_packed(x, x_groups, K);
  TORCH_CHECK(out.is_contiguous() &&
              out.scalar_type() ==
                  (mode == PARTS ? at::kFloat : at::kBFloat16) &&
              out.numel() == (mode == PARTS ? (long)top_k * T * N
                                            : (long)pair_groups * 16 * (N / 2)));
  if (T == 0) return;
  StreamArgs a{};
  a.out = out.data_ptr();
  a.x = (const char*)x.data_ptr();
  Weights<true> wt{};
  for (int e = 0; e < experts; ++e) {
    check_weight(w[e], N, K);
    wt.w[e] = (const char*)w[e].data_ptr();
  }
  a.M = T;
  a.N = N;
  a.steps = a.steps_per_split = K / FRAG_K;
  a.x_groups = x_groups;
  a.choice = choice.data_ptr<int>();
  a.weight = weight.data_ptr<float>();
  a.n_pairs = T * top_k;
  a.top_k = top_k;
  a.out_groups = pair_groups;
  dispatch_grouped(a, wt, mode, experts);
}

// ---------------------------------------------------------------------------
// The elementwise steps between the projections.

namespace {

// residual += sum of the parts (rounded once), out = rmsnorm(residual) as
// packed rows (ms > 0) or row-major (ms = 0). One row per workgroup, held in
// registers between the reduction and the stores. n_parts 0: only the norm.
template <int VPT>
__global__ __launch_bounds__(512) void add_parts_rmsnorm_kernel(
    short* __restrict__ out, short* __restrict__ residual, const float* __restrict__ parts, int n_parts,
    long part_stride, const short* __restrict__ w, float eps, int H, int ms) {
  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  const long base = (long)row * H;
  __shared__ float red[8];
  bf16x8 v[VPT];
  float ss = 0.f;
#pragma unroll
  for (int r = 0; r < VPT; ++r) {
    const int i = (tid + r * 512) * 8;
    v[r] = bf16x8{};
    if (i >= H) continue;
    v[r] = *reinterpret_cast<const bf16x8*>(residual + base + i);
    if (n_parts > 0) {
      f32x4 s0{0.f, 0.f, 0.f, 0.f}, s1 = s0;
      for (int p = 0; p < n_parts; ++p) {
        const float* pp = parts + p * part_stride + base + i;
        const f32x4 a = *reinterpret_cast<const f32x4*>(pp);
        const f32x4 b = *reinterpret_cast<const f32x4*>(pp + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          s0[j] += a[j];
          s1[j] += b[j];
        }
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
        v[r][j] = f2bits(bits2f(v[r][j]) + (j < 4 ? s0[j % 4] : s1[j % 4]));
      *reinterpret_cast<bf16x8*>(residual + base + i) = v[r];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float f = bits2f(v[r][j]);
      ss = fmaf(f, f, ss);
    }
  }
  ss = wave_sum(ss);
  if ((tid & (WAVE - 1)) == 0) red[tid / WAVE] = ss;
  __syncthreads();
  ss = 0.f;
#pragma unroll
  for (int q = 0; q < 8; ++q) ss += red[q];
  const float rms = rsqrtf(ss / (float)H + eps);
#pragma unroll
  for (int r = 0; r < VPT; ++r) {
    const int i = (tid + r * 512) * 8;
    if (i >= H) continue;
    const bf16x8 wv = *reinterpret_cast<const bf16x8*>(w + i);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[r][j] = f2bits(bits2f(v[r][j]) * rms * bits2f(wv[j]));
    *reinterpret_cast<bf16x8*>(out + (ms ? packed_at(row, i, ms) : base + i)) =
        v[r];
  }
}

__global__ void pack_rows_kernel(short* __restrict__ out,
                                 const short* __restrict__ x, int K, int ms,
                                 long stride, long n8) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n8) return;
  const int row = (int)(i / (K / 8)), k = (int)(i % (K / 8)) * 8;
  *reinterpret_cast<bf16x8*>(out + packed_at(row, k, ms)) =
      *reinterpret_cast<const bf16x8*>(x + row * stride + k);
}

}  // namespace

// out: packed or row-major rows
void add_parts_rmsnorm(torch::Tensor out, torch::Tensor residual,
                       c10::optional<torch::Tensor> parts, torch::Tensor w,
                       double eps, bool packed) {
  TORCH_CHECK(residual.is_contiguous() && w.is_contiguous() &&
              out.is_contiguous());
  TORCH_CHECK(residual.scalar_type() == at::kBFloat16 &&
              w.scalar_type() == at::kBFloat16 &&
              out.scalar_type() == at::kBFloat16);
  const int T = residual.size(0), H = residual.size(1);
  TORCH_CHECK(w.numel() == H && H % 8 == 0 && H <= 16384);
  TORCH_CHECK(!packed || (T <= PACKED_ROWS && H % FRAG_K == 0));
  const int ms = packed ? packed_groups(T) : 0;
  TORCH_CHECK(out.numel() == (packed ? (long)ms * 16 : (long)T) * H);
  int n_parts = 0;
  const float* pp = nullptr;
  if (parts.has_value()) {
    TORCH_CHECK(parts->is_contiguous() &&
                parts->scalar_type() == at::kFloat && parts->dim() == 3 &&
                parts->size(1) == T && parts->size(2) == H);
    n_parts = parts->size(0);
    pp = parts->data_ptr<float>();
  }
  if (T == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
#define AP_LAUNCH(VPT)                                                         \
  hipLaunchKernelGGL((add_parts_rmsnorm_kernel<VPT>), dim3(T), dim3(512), 0,   \
                     stream, (short*)out.data_ptr(),                           \
                     (short*)residual.data_ptr(), pp, n_parts, (long)T * H,    \
                     (const short*)w.data_ptr(), (float)eps, H, ms)
  if (H <= 4096) AP_LAUNCH(1);
  else if (H <= 8192) AP_LAUNCH(2);
  else AP_LAUNCH(4);
#undef AP_LAUNCH
}

void pack_rows(torch::Tensor out, torch::Tensor x) {
  const int T = x.size(0), K = x.size(1);
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 && x.stride(1) == 1 &&
              x.stride(0) % 8 == 0 && x.storage_offset() % 8 == 0);
  TORCH_CHECK(T <= PACKED_ROWS && K % 32 == 0 && out.is_contiguous() &&
              out.scalar_type() == at::kBFloat16 &&
              out.numel() == (long)packed_groups(T) * 16 * K);
  const long n8 = (long)T * (K / 8);
  if (n8 == 0) return;
  hipLaunchKernelGGL(pack_rows_kernel, dim3((n8 + 255) / 256), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), (short*)out.data_ptr(),
                     (const short*)x.data_ptr(), K, packed_groups(T),
                     (long)x.stride(0), n8);
}

void route_packed(torch::Tensor choice, torch::Tensor weight, torch::Tensor x,
                  torch::Tensor router) {
  const int T = choice.size(0), top_k = choice.size(1);
  const int E = router.size(0), K = router.size(1);
  TORCH_CHECK(E <= MAX_EXPERTS && top_k <= E && K % 32 == 0 && T <= 64);
  TORCH_CHECK(router.is_contiguous() &&
              router.scalar_type() == at::kBFloat16);
  TORCH_CHECK(choice.is_contiguous() && choice.scalar_type() == at::kInt &&
              weight.is_contiguous() && weight.scalar_type() == at::kFloat &&
              weight.numel() == choice.numel());
  const int groups = packed_groups(T);
  TORCH_CHECK(x.is_contiguous() && x.scalar_type() == at::kBFloat16 &&
              x.numel() == (long)groups * 16 * K);
  if (T == 0) return;
  hipLaunchKernelGGL(route_kernel<true>, dim3(T), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), choice.data_ptr<int>(),
                     weight.data_ptr<float>(), (const short*)x.data_ptr(),
                     (const short*)router.data_ptr(), K, groups, E, top_k);
}
