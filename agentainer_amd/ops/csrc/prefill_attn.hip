// Paged varlen causal prefill attention (gfx950, MFMA bf16).
//
// Flash-style online-softmax attention for the batched prefill phase of
// the continuous-batching scheduler. Q rows are the batch's NEW tokens
// (varlen-packed); K/V are read from the paged pools, so a conversation's
// cached prefix is attended without re-prefilling it (the
// agent-KV-persistence contract).
//
// Geometry: one workgroup = 4 waves = one 32-row Q tile of 4 GQA heads that
// share a kv head; wave w owns head group*4 + w. KV tile = 64 tokens, staged
// once per workgroup in LDS (double-buffered, the next tile's loads are in
// flight during the current tile's MFMAs, one barrier per tile).
//
//   S^T[kv, q]  = mfma_f32_32x32x16_bf16(A = K, B = Q^T)   2 x 8 steps
//   O^T[d, q]  += mfma_f32_32x32x16_bf16(A = V^T, B = P^T) 4 x 4 steps
//
// Both products are kept transposed because the accumulator of the first is
// then laid out like the B operand of the second: lane l holds q column
// l % 32 and, of every 16 kv rows, rows {0..3} and {8..11} offset by
// 4 * (l / 32). Probabilities go from accumulator to operand with a convert
// and no exchange; the row maximum is an in-lane chain plus one half-wave
// swap, and the rescale of O is one factor per lane. V^T comes out of the
// row-major V tile with the transposing LDS read (16 lanes read a 4 x 16
// block, lane i gets column i), in that same kv order.
//
// What bounds it: per wave and tile 1024 cycles of MFMA, about as many of
// VALU (32 exponentials per lane) and 128 KB of LDS reads per workgroup, so
// two workgroups per CU (73 KB LDS, <= 256 VGPRs) overlap one's exponentials
// with the other's MFMAs. The accumulator is only rescaled when a row's
// maximum grew by more than 2^8 since the last rescale.
//
// Measured (32 heads on 8, bf16 cache), against the 16x16 tiles of 32 tokens
// with probabilities going through LDS that were here before: one prompt of
// 7900 tokens 620 us, 0.82 PFLOP/s (5193 us); 32 prompts of 256 63 us (364);
// 45 rows over 1245 tokens 10.3 us + 5.8 us merge (198).
//
// LDS: K keeps the pool's order [16-token group][d/8][16 tokens][8], whose
// fragment reads are 256 contiguous bytes per 16 lanes; V rows are padded to
// 320 B so the four rows x two column blocks that 32 lanes of a transposing
// read touch cover all 64 banks once.

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <algorithm>
#include <cfloat>
#include <cmath>
#include "common.h"
#include "pool_tiles.h"

namespace {

constexpr int QBLK = 32;
constexpr int KVBLK = 64;
constexpr int D = 128;
constexpr int K_TILE = KVBLK * D;       // shorts
constexpr int V_STRIDE = 160;           // shorts per padded V row
constexpr int V_TILE = KVBLK * V_STRIDE;
constexpr int O_STRIDE = D + 8;         // shorts per output row in LDS
constexpr float LAZY_LOG2 = 8.f;
constexpr int PART = D + 2;             // o, m, l of one (split, row, head)

// maximum over the two halves of the wave, in every lane
__device__ __forceinline__ float half_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x),
                                                  __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x),
                                                  __float_as_uint(x), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// SPLIT: blockIdx.z = seq * n_split + split; the workgroup covers one of
// n_split equal runs of KV tiles and writes unnormalized partials.
// PAGE16: page size is a power of two >= 16, so the 16 tokens of a staging
// group lie in one page and the page lookup is uniform.
template <typename CT, bool SPLIT, bool PAGE16>
__global__ __launch_bounds__(256, 2) void prefill_attn_kernel(
    short* __restrict__ out,            // [Tq, n_q, D] or packed rows
    float* __restrict__ part,           // [n_split, Tq, n_q, PART]
    const short* __restrict__ q,        // [Tq, n_q, D]
    const CT* __restrict__ k_cache,     // [P, n_kv, D/8, PS, 8]
    const CT* __restrict__ v_cache,     // [P, n_kv, PS, D]
    const int* __restrict__ page_table, // [B, max_pages]
    const int* __restrict__ seq_lens,   // [B] total context length
    const int* __restrict__ q_starts,   // [B] row offset into q
    const int* __restrict__ q_lens,     // [B]
    float c, bool negate, int n_q, int n_kv, int PS, int ps_shift,
    int max_pages, long q_ts, int n_split, long t_rows, int ms) {
  // head groups go round the 8 XCDs first (workgroups are dealt to XCDs in
  // turn), so the groups of one kv head meet in one L2; the longest causal
  // ranges (last Q tiles) start first
  const int n_groups = gridDim.x;
  int group = blockIdx.x;
  if (n_groups % 8 == 0) {
    const int per = n_groups / 8;
    group = (blockIdx.x % 8) * per + blockIdx.x / 8;
  }
  const int qtile = gridDim.y - 1 - blockIdx.y;
  const int b = SPLIT ? blockIdx.z / n_split : blockIdx.z;
  const int split = SPLIT ? blockIdx.z % n_split : 0;
  const int qlen = q_lens[b];
  if (qtile * QBLK >= qlen) return;
  const int lane = threadIdx.x % WAVE;
  const int wid = threadIdx.x / WAVE;
  const int l32 = lane % 32;
  const int h = lane / 32;
  const int head = group * 4 + wid;
  const int g = head / (n_q / n_kv);
  const int ctx_start = seq_lens[b] - qlen;  // new tokens sit at the end

  __shared__ __attribute__((aligned(16))) short lds[2 * (K_TILE + V_TILE)];

  const int* pt = page_table + (long)b * max_pages;
  const long q_row0 = q_starts[b] + (long)qtile * QBLK;

  // Q^T operand: lane holds Q[l32][s*16 + h*8 .. +8]
  bf16v8 qf[8];
  {
    const bool live = qtile * QBLK + l32 < qlen;
    const short* p = q + (q_row0 + l32) * q_ts + (long)head * D + h * 8;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      bf16x8 v{};
      if (live) v = *reinterpret_cast<const bf16x8*>(p + s * 16);
      if (negate)
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (short)(v[j] ^ (short)0x8000);
      qf[s] = *reinterpret_cast<bf16v8*>(&v);
    }
  }

  f32x16 o[4];  // O^T d tiles
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m_ref = -FLT_MAX, l_run = 0.f;

  const int q_last = min(qtile * QBLK + QBLK - 1, qlen - 1);
  const int kv_end = ctx_start + q_last + 1;
  const int n_tiles = (kv_end + KVBLK - 1) / KVBLK;
  int t0 = 0, t1 = n_tiles;
  if (SPLIT) {
    const int per = (n_tiles + n_split - 1) / n_split;
    t0 = split * per;
    t1 = min(t0 + per, n_tiles);
  }
  const int q_first = ctx_start + qtile * QBLK;  // position of column 0

  // staging: per 16-token group i of a tile this thread moves K chunk
  // (token 16i + tid%16, d8 = tid/16) and V chunk (token 16i + tid/16,
  // columns 8 * (tid%16)). Tokens past the last visible one load it again, so
  // nothing stale is ever multiplied, and their values are zeroed on the way
  // to LDS: under a probability of 0 an infinite one would make NaN.
  typedef typename Raw<CT>::type raw;
  raw st_k[4], st_v[4];
  const int lo = threadIdx.x % 16, hi = threadIdx.x / 16;
  auto stage_load = [&](int t) {
    const int kv0 = t * KVBLK;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tk = min(kv0 + 16 * i + lo, kv_end - 1);
      const int tv = min(kv0 + 16 * i + hi, kv_end - 1);
      long kb, vb;
      if (PAGE16) {
        const int pi = min(kv0 + 16 * i, kv_end - 1) >> ps_shift;
        const long pg = (long)pt[pi] * n_kv + g;
        kb = ((pg * (D / 8) + hi) << ps_shift) + (tk & (PS - 1));
        vb = (pg << ps_shift) + (tv & (PS - 1));
      } else {
        kb = (((long)pt[tk / PS] * n_kv + g) * (D / 8) + hi) * PS + tk % PS;
        vb = ((long)pt[tv / PS] * n_kv + g) * PS + tv % PS;
      }
      st_k[i] = *reinterpret_cast<const raw*>(k_cache + kb * 8);
      st_v[i] = *reinterpret_cast<const raw*>(v_cache + vb * D + lo * 8);
    }
  };
  auto stage_write = [&](int buf, int t) {
    const int left = kv_end - t * KVBLK;
    if (left < KVBLK) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (16 * i + hi >= left) st_v[i] = raw{};
    }
    short* kl = lds + buf * (K_TILE + V_TILE);
    short* vl = kl + K_TILE;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<bf16x8*>(kl + (i * 256 + threadIdx.x) * 8) =
          to_bf16(st_k[i]);
      *reinterpret_cast<bf16x8*>(vl + (16 * i + hi) * V_STRIDE + lo * 8) =
          to_bf16(st_v[i]);
    }
  };

  if (t0 < t1) {
    stage_load(t0);
    stage_write(0, t0);
  }
  __syncthreads();
  // fragment bases: K chunk of (token l32, d8 = h); V block of the 16-lane
  // group: rows 4h + i/4, columns 16 * (group % 2) + 4 * (i % 4)
  const int k_off = ((l32 / 16) * 256 + h * 16 + l32 % 16) * 8;
  const int v_off = (4 * h + (lane % 16) / 4) * V_STRIDE +
                    16 * ((lane / 16) % 2) + 4 * (lane % 4);
  int buf = 0;
  for (int t = t0; t < t1; ++t) {
    const int kv0 = t * KVBLK;
    const bool has_next = t + 1 < t1;
    if (has_next) stage_load(t + 1);
    const short* kl = lds + buf * (K_TILE + V_TILE) + k_off;
    const short* vl = lds + buf * (K_TILE + V_TILE) + K_TILE + v_off;

    f32x16 s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[u][r] = 0.f;
#pragma unroll
      for (int st = 0; st < 8; ++st) {
        const bf16v8 kf =
            *reinterpret_cast<const bf16v8*>(kl + u * 4096 + st * 256);
        s[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[st], s[u], 0, 0,
                                                       0);
      }
    }
    if (kv0 + KVBLK - 1 > q_first) {  // the tile crosses the diagonal
      const int last = q_first + l32 - kv0 - 4 * h;  // last visible row
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (32 * u + (r / 4) * 8 + r % 4 > last) s[u][r] = -INFINITY;
    }
    float mx = m_ref;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[u][r]);
    mx = half_max(mx);
    if (__any((mx - m_ref) * c > LAZY_LOG2)) {
      const float alpha = __builtin_amdgcn_exp2f(fmaxf((m_ref - mx) * c,
                                                       -FLT_MAX));
      m_ref = mx;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
    }
    const float mc = fmaxf(m_ref * c, -FLT_MAX);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float sum = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[u][r] = __builtin_amdgcn_exp2f(fmaf(s[u][r], c, -mc));
        sum += s[u][r];
      }
      l_run += sum;
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        f32v8 pv;
#pragma unroll
        for (int j = 0; j < 8; ++j) pv[j] = s[u][8 * st + j];
        const bf16v8 pf = __builtin_convertvector(pv, bf16v8);
        const short* vr = vl + (32 * u + 16 * st) * V_STRIDE;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
          union {
            s16x4 half[2];
            bf16v8 v;
          } vf;
          vf.half[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_s16x4*)(vr + 32 * dt));
          vf.half[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_s16x4*)(vr + 8 * V_STRIDE + 32 * dt));
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.v, pf, o[dt], 0,
                                                          0, 0);
        }
      }
    }
    if (has_next) stage_write(buf ^ 1, t + 1);
    __syncthreads();
    buf ^= 1;
  }

  const float l_all = half_sum(l_run);
  if (SPLIT) {
    if (qtile * QBLK + l32 < qlen) {
      float* pp = part + (((long)split * t_rows + q_row0 + l32) * n_q + head) *
                             PART;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          pp[dt * 32 + (r / 4) * 8 + 4 * h + r % 4] = o[dt][r];
      if (h == 0) {
        pp[D] = m_ref;
        pp[D + 1] = l_all;
      }
    }
    return;
  }
  // O^T -> rows through LDS, so the stores are whole 256-byte head rows
  const float inv = l_all > 0.f ? 1.f / l_all : 0.f;
  short* ol = lds + wid * QBLK * O_STRIDE;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      bf16x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = f2bits(o[dt][r4 * 4 + j] * inv);
      *reinterpret_cast<bf16x4*>(ol + l32 * O_STRIDE + dt * 32 + r4 * 8 +
                                 4 * h) = v;
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = i * 4 + lane / 16;
    if (qtile * QBLK + row < qlen)
      *reinterpret_cast<bf16x8*>(
          out + (ms ? packed_at((int)q_row0 + row, head * D + lane % 16 * 8, ms)
                    : ((q_row0 + row) * n_q + head) * D + lane % 16 * 8)) =
          *reinterpret_cast<const bf16x8*>(ol + row * O_STRIDE +
                                           (lane % 16) * 8);
  }
}

// Merges the splits' partials of one (row, head) per wave: lane s holds split
// s's maximum and sum, so all of them are one load; the values then come eight
// splits at a time (one at a time, each behind its weight: 10 us for 48 rows
// of 32 heads in 16 splits; now 6).
__global__ __launch_bounds__(256) void prefill_combine_kernel(
    short* __restrict__ out, const float* __restrict__ part,
    const int* __restrict__ q_starts, const int* __restrict__ q_lens, float c,
    int n_q, int n_split, long t_rows, int ms) {
  const int b = blockIdx.y;
  const int item = blockIdx.x * 4 + threadIdx.x / WAVE;
  const int row = item / n_q, head = item % n_q;
  if (row >= q_lens[b]) return;
  const int lane = threadIdx.x % WAVE;
  const long r = q_starts[b] + row;
  const float* first = part + (r * n_q + head) * PART;
  const long step = t_rows * n_q * PART;
  float m_s = -FLT_MAX, l_s = 0.f;
  if (lane < n_split) {
    m_s = first[lane * step + D];
    l_s = first[lane * step + D + 1];
  }
  const float m = wave_max(m_s);
  // a split in which nothing is visible has l = 0 and holds no values
  float w_s = l_s != 0.f
                  ? __builtin_amdgcn_exp2f(fmaxf((m_s - m) * c, -FLT_MAX))
                  : 0.f;
  const float l = wave_sum(w_s * l_s);
  float o0 = 0.f, o1 = 0.f;
  for (int s0 = 0; s0 < n_split; s0 += 8) {
    float v0[8], v1[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float* pp = first + min(s0 + j, n_split - 1) * step + 2 * lane;
      v0[j] = pp[0];
      v1[j] = pp[1];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (s0 + j >= n_split) break;
      const float w = __shfl(w_s, s0 + j, WAVE);
      o0 = fmaf(w, v0[j], o0);
      o1 = fmaf(w, v1[j], o1);
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  short* op = out + (ms ? packed_at((int)r, head * D + 2 * lane, ms)
                        : (r * n_q + head) * D + 2 * lane);
  op[0] = f2bits(o0 * inv);
  op[1] = f2bits(o1 * inv);
}

}  // namespace

void paged_prefill_attention(torch::Tensor out, torch::Tensor q,
                             torch::Tensor k_cache, torch::Tensor v_cache,
                             torch::Tensor page_table, torch::Tensor seq_lens,
                             torch::Tensor query_starts, torch::Tensor query_lens,
                             double scale, long max_qlen, bool packed) {
  TORCH_CHECK(out.is_contiguous());
  TORCH_CHECK(q.scalar_type() == at::kBFloat16);
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == q.size(2));
  const int n_q = q.size(1), Dh = q.size(2);
  const int n_kv = k_cache.size(1), PS = k_cache.size(3);
  const int B = seq_lens.size(0);
  const int max_pages = page_table.size(1);
  TORCH_CHECK(Dh == 128, "prefill attention: head_dim 128 only");
  TORCH_CHECK(n_q % 4 == 0, "n_q must be a multiple of 4");
  const int ratio = n_q / n_kv;
  TORCH_CHECK(ratio % 4 == 0 || ratio == n_q,
              "GQA ratio must be a multiple of 4 (waves of a workgroup share "
              "one kv head)");
  if (max_qlen <= 0) {
    // fallback: derive from the device tensor. This D2H copy BLOCKS the
    // host until the stream drains (measured ~2 ms/call under serving
    // load with a deep queue — 32x per prefill); hot callers pass
    // max_qlen explicitly (AttnMetadata.max_qlen).
    auto q_lens_cpu = query_lens.to(torch::kCPU);
    auto* ql = q_lens_cpu.data_ptr<int>();
    for (int i = 0; i < B; ++i)
      max_qlen = std::max<long>(max_qlen, ql[i]);
    if (max_qlen == 0) return;
  }
  // rows are read and written 16 bytes at a time; others go through copies
  auto aligned = [](const torch::Tensor& x) {
    return reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0;
  };
  if (q.stride(0) % 8 != 0 || !aligned(q))
    q = q.clone(at::MemoryFormat::Contiguous);
  const long t_rows = q.size(0);
  TORCH_CHECK(!packed || t_rows <= PACKED_ROWS);
  const int ms = packed ? packed_groups(t_rows) : 0;
  const long out_size = (packed ? (long)ms * 16 : t_rows) * n_q * Dh;
  TORCH_CHECK(!packed || out.numel() == out_size);
  // more rows than q's are left alone; fewer are enough where the sequences
  // cover no more
  if (!aligned(out) || out.numel() < out_size) {
    auto rows = torch::empty({out_size}, out.options());
    auto all = out.view({-1});
    const long n = std::min<long>(out_size, all.numel());
    auto part = all.narrow(0, 0, n), mine = rows.narrow(0, 0, n);
    mine.copy_(part);
    paged_prefill_attention(rows, q, k_cache, v_cache, page_table, seq_lens,
                            query_starts, query_lens, scale, max_qlen, packed);
    part.copy_(mine);
    return;
  }
  const int qtiles = (max_qlen + QBLK - 1) / QBLK;
  auto stream = at::hip::getCurrentHIPStream();
  // Few Q tiles (the next turn of one conversation) leave most of the chip
  // idle while each workgroup walks the whole context alone: split the KV
  // range until two workgroups per CU are in flight, each still with at
  // least two tiles. From 384 workgroups on (1.5 per CU) a split would only
  // add the partials' round trip through memory.
  const long blocks = (long)qtiles * B * (n_q / 4);
  if (blocks == 0) return;
  const long ctx_tiles = ((long)max_pages * PS + KVBLK - 1) / KVBLK;
  int n_split = 1;
  if (blocks < 384)
    n_split = (int)std::max<long>(
        1, std::min<long>({16, 512 / blocks, ctx_tiles / 2}));
  torch::Tensor part;
  if (n_split > 1)
    part = torch::empty({n_split * t_rows * n_q * PART},
                        torch::TensorOptions().dtype(torch::kFloat).device(
                            q.device()));
  int ps_shift = 0;
  while ((1 << ps_shift) < PS) ++ps_shift;
  const bool page16 = PS >= 16 && (1 << ps_shift) == PS;
  // exponents in base 2; a negative scale is moved into Q's signs
  const float c = std::max((float)(std::fabs(scale) * 1.4426950408889634),
                           1e-30f);
#define PF_LAUNCH(CT, SPLIT_, P16_)                                            \
  hipLaunchKernelGGL((prefill_attn_kernel<CT, SPLIT_, P16_>),                  \
                     dim3(n_q / 4, qtiles, B * n_split), dim3(256), 0, stream, \
                     (short*)out.data_ptr(),                                   \
                     SPLIT_ ? part.data_ptr<float>() : nullptr,                \
                     (const short*)q.data_ptr(),                               \
                     (const CT*)k_cache.data_ptr(),                            \
                     (const CT*)v_cache.data_ptr(),                            \
                     page_table.data_ptr<int>(), seq_lens.data_ptr<int>(),     \
                     query_starts.data_ptr<int>(), query_lens.data_ptr<int>(), \
                     c, scale < 0, n_q, n_kv, PS, ps_shift, max_pages,         \
                     (long)q.stride(0), n_split, t_rows, ms)
#define PF_TYPE(CT)                                                            \
  do {                                                                         \
    if (n_split > 1) {                                                         \
      if (page16) PF_LAUNCH(CT, true, true);                                   \
      else PF_LAUNCH(CT, true, false);                                         \
    } else {                                                                   \
      if (page16) PF_LAUNCH(CT, false, true);                                  \
      else PF_LAUNCH(CT, false, false);                                        \
    }                                                                          \
  } while (0)
  if (k_cache.scalar_type() == at::kFloat8_e4m3fn) {
    PF_TYPE(unsigned char);
  } else {
    TORCH_CHECK(k_cache.scalar_type() == at::kBFloat16);
    PF_TYPE(short);
  }
#undef PF_TYPE
#undef PF_LAUNCH
  if (n_split > 1)
    hipLaunchKernelGGL(prefill_combine_kernel,
                       dim3((unsigned)(max_qlen * n_q / 4), B), dim3(256), 0,
                       stream, (short*)out.data_ptr(), part.data_ptr<float>(),
                       query_starts.data_ptr<int>(),
                       query_lens.data_ptr<int>(), c, n_q, n_split, t_rows, ms);
}
