// Paged GQA decode attention (gfx950): one query token per sequence.
//
// HBM-bound: the op streams seq_len * 2 * D pool values per (sequence, kv
// head) once; the GQA group's RATIO query heads share every value loaded.
//
// One workgroup of 4 waves owns (kv head, split, sequence): a run of the
// sequence's tokens that its waves walk in tiles of 32, each wave on its own
// with its own online softmax, merged through LDS at the end. Per tile and
// wave (mfma_f32_16x16x32_bf16 throughout):
//
//   S^T[token, column] = K . Q^T    K fragments come straight from the pool:
//       its [d/8][token][8] page order IS the fragment order, so a load
//       instruction is one contiguous KB. bf16 queries are used as they are
//       for fp8 pools too (every e4m3 value is a bf16 value).
//   O^T[d, column]    += V^T . P^T  V rows go through a wave-private LDS tile
//       (no barrier) and come back transposed by ds_read_b64_tr_b16; P^T is
//       the accumulator of the first product, converted in place.
//
// The 16 columns hold at most 8 heads twice, and every V tile is multiplied
// twice, so a probability enters as four bf16 parts whose sum is its fp32 value
// exactly: columns 0..7 take about half of it and what that half leaves, to 9
// bits, columns 8..15 two parts of the rest; the two halves of O are added at
// the end. That costs, against one product with 16 bits of a probability, 0.3
// us where latency counts (1 x 320 tokens 9.5 against 9.2, with the op's clear)
// and nothing to 3 % where bytes do (48 x 4800: 161.4 against 161.0; 250 x 600
// of fp8: 58.2 against 56.5).
//
// The next tile's 16 KB (8 KB for fp8) per wave are in flight during the
// current tile; at 3 workgroups per CU that is 192 KB, several times what
// covers the memory's latency.
//
// Splits: a run is at least `chunk` tokens, so a short sequence uses one
// workgroup per kv head and writes its result directly, a long one as many
// as its length asks for (the grid covers the longest the page table could
// hold, see splits_of). Partials of several runs are
// merged by the workgroup that finishes last, told by a counter per (sequence,
// kv head) that a kernel earlier in the stream has cleared.
//
// The pool is read with non-temporal loads: a layer's cache is mostly not seen
// again until the next step (48 x 4800 tokens: 188 -> 168 us, 64 x 1100: 61 ->
// 56). Pages of a prefix that the sequences share are, and the hint costs there,
// but less: 4096 of 4800 tokens shared by 48 sequences 72.6 -> 74.1 us, 1024 of
// 1100 by 64 28.7 -> 28.3, by 250 66.0 -> 70.2.
//
// Measured (32 heads on 8, page 16, tables of 512 pages, cold cache, the op
// with the clearing of its counters), against one-wave workgroups that score
// with dot instructions, sum V on the VALU and merge 8 fixed splits in a second
// kernel (decode_attn_fixed.hip):
//   1 x 320 tokens     9.1 us (14.5)     64 x 290     18.8 us (30.0)
//   13 x 1500, fp8    18.7 us (50.6)     48 x 4800     168 us, 5.6 TB/s (253)
//   250 x 600, fp8    59.7 us (111)      16 x 1300, 64 heads  26.1 us (79)

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <algorithm>
#include <cfloat>
#include <cmath>
#include "common.h"
#include "pool_tiles.h"

namespace {

constexpr int D = 128;
constexpr int TILE = 32;              // tokens per wave and step
constexpr int WAVES = 4;
constexpr int PART = D + 2;           // o, m, l of one (split, head)
constexpr int MAX_SPLITS = 64;
constexpr long CAP = 2048;            // workgroups of a split grid
constexpr float LAZY_LOG2 = 8.f;

// reductions over the four lanes that share a column (lanes 16 apart)
__device__ __forceinline__ float col_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x),
                                            __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x),
                                       false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float col_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x),
                                            __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x),
                                       false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// value of the lane 8 columns away within a row of 16 lanes
__device__ __forceinline__ float other_half(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x128, 0xf,
                                                 0xf, true));
}

// device-scope partials (see the merge)
__device__ __forceinline__ void put(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float get(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// PAGE: 16 = that page size, 1 = another power of two above it, 0 = any.
// Unless 0, a 16-token group lies in one page: its lookup is a scalar load and
// its addresses are a scalar base plus a lane offset.
template <int RATIO, typename CT, int PAGE>
__global__ __launch_bounds__(WAVES * WAVE, 3) void decode_attn_kernel(
    short* __restrict__ out,            // [B, n_q, D] or packed rows
    float* __restrict__ part,           // [B, n_kv, n_split, RATIO, PART]
    int* __restrict__ arrived,          // [B, n_kv], zero
    const short* __restrict__ q,        // [B, n_q, D]
    const CT* __restrict__ k_cache,     // [P, n_kv, D/8, PS, 8]
    const CT* __restrict__ v_cache,     // [P, n_kv, PS, D]
    const int* __restrict__ page_table, // [B, max_pages]
    const int* __restrict__ seq_lens,   // [B]
    float c, bool negate, int n_kv, int page_size, int ps_shift,
    int max_pages, long q_ts, int min_chunk, int ms) {
  const int PS = PAGE == 16 ? 16 : page_size;
  const int shift = PAGE == 16 ? 4 : ps_shift;
  const int g = blockIdx.x, b = blockIdx.y, split = blockIdx.z;
  const int n_split = gridDim.z;
  // where value d of head h goes: a row of [B, n_q, D], or packed rows (ms)
  auto out_at = [&](int h, int d) {
    const int k = (g * RATIO + h) * D + d;
    return ms ? packed_at(b, k, ms) : (long)b * n_kv * RATIO * D + k;
  };
  const int len = seq_lens[b];
  if (len <= 0) return;
  // tokens per run: at least min_chunk, more when the grid has too few runs
  int chunk = min_chunk;
  if ((long)chunk * n_split < len)
    chunk = ((len + n_split - 1) / n_split + 127) / 128 * 128;
  const int n_act = (len + chunk - 1) / chunk;
  if (split >= n_act) return;
  const int t_begin = split * chunk, t_end = min(t_begin + chunk, len);
  const int lane = threadIdx.x % WAVE;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int col = lane % 16;
  const int lg = lane / 16;

  typedef typename Raw<CT>::type raw;
  __shared__ __attribute__((aligned(16))) short v_lds[WAVES][TILE * D];
  const int* pt = page_table + (long)b * max_pages;

  // Q^T operand: column `col` is head col % 8 % RATIO, dims s*32 + lg*8 ..+8
  bf16v8 qf[4];
  {
    const short* qp = q + (long)b * q_ts +
                      (long)(g * RATIO + col % 8 % RATIO) * D + lg * 8;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      bf16x8 v = *reinterpret_cast<const bf16x8*>(qp + s * 32);
      if (negate)
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (short)(v[j] ^ (short)0x8000);
      qf[s] = *reinterpret_cast<bf16v8*>(&v);
    }
  }

  // one tile: K chunk (token 16i + col, d8 = 4s + lg), V chunk (token
  // 4i + lg, dims 8*col ..+8). Tokens past the run repeat its last one, so
  // nothing stale is ever multiplied.
  raw rk[2][4], rv[8];
  // pages of a tile's two groups, looked up one tile ahead
  int pg[2];
  auto look = [&](int t) {
    if (PAGE)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        pg[i] = pt[min(t + 16 * i, t_end - 1) >> shift];
  };
  auto load = [&](int t) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int tk = min(t + 16 * i + col, t_end - 1);
      if (PAGE) {
        const long head = ((long)pg[i] * n_kv + g) << shift;
        const CT* kb = k_cache + head * D;
        const CT* vb = v_cache + head * D;
        const int k_off = (lg * PS + (tk & (PS - 1))) * 8;
#pragma unroll
        for (int s = 0; s < 4; ++s)
          rk[i][s] = __builtin_nontemporal_load(
              reinterpret_cast<const raw*>(kb + k_off + s * 32 * PS));
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int tv = min(t + 16 * i + 4 * k + lg, t_end - 1);
          rv[4 * i + k] = __builtin_nontemporal_load(
              reinterpret_cast<const raw*>(vb + (tv & (PS - 1)) * D +
                                           col * 8));
        }
      } else {
        const CT* kb = k_cache + ((((long)pt[tk / PS] * n_kv + g) * (D / 8) +
                                   lg) * PS + tk % PS) * 8;
#pragma unroll
        for (int s = 0; s < 4; ++s)
          rk[i][s] = *reinterpret_cast<const raw*>(kb + (long)s * 32 * PS);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int tv = min(t + 16 * i + 4 * k + lg, t_end - 1);
          rv[4 * i + k] = *reinterpret_cast<const raw*>(
              v_cache +
              (((long)pt[tv / PS] * n_kv + g) * PS + tv % PS) * D + col * 8);
        }
      }
    }
  };

  f32x4 o[8];  // O^T d tiles
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_ref = -FLT_MAX, l_run = 0.f;

  // V tile rows are 256 B, i.e. all 64 banks; 16-byte slots are permuted by
  // the row so the 8 rows x 32 B that half a wave reads transposed are apart
  short* vl = v_lds[wid];
  const int w_slot = lane / 16;  // + 4i = row written
  // transposing read: this lane points at row 4*lg + col/4 (+16) and the
  // 8-byte piece col%4 of the d tile's 32 bytes
  const int r_row = 4 * lg + col / 4;
  const short* r_base = vl + r_row * D;
  const int r_piece = (col % 4) * 4;

  int t = t_begin + wid * TILE;
  if (t < t_end) {
    look(t);
    load(t);
    look(t + WAVES * TILE);
  }
  for (; t < t_end; t += WAVES * TILE) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = 4 * i + w_slot;
      *reinterpret_cast<bf16x8*>(vl + row * D +
                                 ((col ^ (2 * (row % 8))) * 8)) =
          to_bf16(rv[i]);
    }
    f32x4 s[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const bf16x8 kv = to_bf16(rk[i][st]);
        s[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<const bf16v8*>(&kv), qf[st], s[i], 0, 0, 0);
      }
    }
    const int left = t_end - t;  // tokens of this tile that exist
    if (t + WAVES * TILE < t_end) {
      load(t + WAVES * TILE);
      look(t + 2 * WAVES * TILE);
    }
    if (left < TILE) {
      // The last token and its repetitions share its probability. (Masked,
      // a repetition would be 0 times its value, NaN where that is infinite;
      // zeroing values instead costs the loads their registers, 180 instead
      // of 161 us for 48 x 4800.)
      const float share =
          -__builtin_amdgcn_logf((float)(TILE - left + 1)) / c;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (16 * i + 4 * lg + r >= left - 1) s[i][r] += share;
    }
    float mx = m_ref;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[i][r]);
    mx = col_max(mx);
    if (__any((mx - m_ref) * c > LAZY_LOG2)) {
      const float alpha =
          __builtin_amdgcn_exp2f(fmaxf((m_ref - mx) * c, -FLT_MAX));
      m_ref = mx;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[dt][r] *= alpha;
    }
    const float mc = fmaxf(m_ref * c, -FLT_MAX);
    f32v8 p;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p[4 * i + r] = __builtin_amdgcn_exp2f(fmaf(s[i][r], c, -mc));
        l_run += p[4 * i + r];
      }
    // p = half + rest, both about p / 2; what their bf16 values leave has at
    // most 15 bits, which the two parts of the upper columns hold
    bf16v8 pa = __builtin_convertvector(p * 0.5f, bf16v8);
    const f32v8 rest = p - __builtin_convertvector(pa, f32v8);
    bf16v8 pb = __builtin_convertvector(rest, bf16v8);
    if (col >= 8) {
      const f32v8 low = rest - __builtin_convertvector(pb, f32v8);
      pa = __builtin_convertvector(low, bf16v8);
      pb = __builtin_convertvector(low - __builtin_convertvector(pa, f32v8),
                                   bf16v8);
    }
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      // the two 16-byte slots of a d tile stay a pair under the permutation
      const short* rp = r_base + ((2 * dt) ^ (2 * (r_row % 8))) * 8 + r_piece;
      union {
        s16x4 half[2];
        bf16v8 v;
      } vf;
      vf.half[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)rp);
      vf.half[1] =
          __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(rp + 16 * D));
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, pa, o[dt], 0, 0,
                                                      0);
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, pb, o[dt], 0, 0,
                                                      0);
    }
  }

  // fold the low parts in, then merge the four waves through LDS (each wave
  // writes over its own V tile)
  float* red = reinterpret_cast<float*>(v_lds);
  constexpr int WAVE_RED = TILE * D / 2;  // floats of one wave's region
  static_assert(RATIO * PART <= WAVE_RED, "merge area");
  const float l_all = col_sum(l_run);
  {
    float* mine = red + wid * WAVE_RED;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // A low part is often exactly 0, and 0 times an infinite value is
        // NaN; the upper parts of a probability above 0 are above 0 too, so
        // their half alone has the answer whenever it is not finite.
        const float low = other_half(o[dt][r]);
        const float v = __builtin_isfinite(o[dt][r]) ? o[dt][r] + low
                                                     : o[dt][r];
        if (col < RATIO) mine[col * PART + dt * 16 + lg * 4 + r] = v;
      }
    if (lg == 0 && col < RATIO) {
      mine[col * PART + D] = m_ref;
      mine[col * PART + D + 1] = l_all;
    }
  }
  __syncthreads();
  float* my_part = part + ((((long)b * n_kv + g) * n_split + split) * RATIO) *
                              PART;
  for (int e = threadIdx.x; e < RATIO * D; e += WAVES * WAVE) {
    const int h = e / D, d = e % D;
    float m = -FLT_MAX;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
      m = fmaxf(m, red[w * WAVE_RED + h * PART + D]);
    float l = 0.f, ov = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float* rw = red + w * WAVE_RED + h * PART;
      const float f =
          __builtin_amdgcn_exp2f(fmaxf((rw[D] - m) * c, -FLT_MAX));
      l = fmaf(f, rw[D + 1], l);
      ov = fmaf(f, rw[d], ov);
    }
    if (n_act == 1) {
      const float inv = l > 0.f ? 1.f / l : 0.f;
      out[out_at(h, d)] = f2bits(ov * inv);
    } else {
      put(my_part + h * PART + d, ov);
      if (d == 0) {
        put(my_part + h * PART + D, m);
        put(my_part + h * PART + D + 1, l);
      }
    }
  }
  if (n_act == 1) return;

  // The workgroup that arrives last merges all runs of this (b, g). The
  // partials are device-scope stores and loads (they pass the XCD's own L2
  // by), so it takes only this workgroup's stores to be complete before its
  // arrival counts, not a write-back and invalidation of whole caches: the
  // fences that do that cost 500 us per layer at 48 x 4800 tokens.
  __shared__ int last;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0)
    last = __hip_atomic_fetch_add(arrived + (long)b * n_kv + g, 1,
                                  __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT) == n_act - 1;
  __syncthreads();
  if (!last) return;
  const float* all = part + (((long)b * n_kv + g) * n_split * RATIO) * PART;
  // every run's m and l once into LDS, then the values eight runs at a time
  float* ml = red;  // [n_act * RATIO][2]
  for (int e = threadIdx.x; e < n_act * RATIO; e += WAVES * WAVE) {
    const float m = get(all + (long)e * PART + D);
    const float l = get(all + (long)e * PART + D + 1);
    ml[2 * e] = m;
    ml[2 * e + 1] = l;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < RATIO * D; e += WAVES * WAVE) {
    const int h = e / D, d = e % D;
    float m = -FLT_MAX;
    for (int s = 0; s < n_act; ++s) m = fmaxf(m, ml[2 * (s * RATIO + h)]);
    float l = 0.f, ov = 0.f;
    for (int s0 = 0; s0 < n_act; s0 += 8) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        v[j] = get(all + (long)(min(s0 + j, n_act - 1) * RATIO + h) * PART + d);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (s0 + j < n_act) {
          const float* x = ml + 2 * ((s0 + j) * RATIO + h);
          const float f =
              __builtin_amdgcn_exp2f(fmaxf((x[0] - m) * c, -FLT_MAX));
          l = fmaf(f, x[1], l);
          ov = fmaf(f, v[j], ov);
        }
    }
    const float inv = l > 0.f ? 1.f / l : 0.f;
    out[out_at(h, d)] = f2bits(ov * inv);
  }
}

// Shortest run worth a workgroup. Few (sequence, kv head) pairs: 128 tokens,
// one tile per wave, so a single conversation spreads over the chip; many
// pairs: 512, which keeps a 300-token sequence in one workgroup (no merge)
// and still cuts long ones finely enough that uneven lengths even out.
int chunk_of(long pairs) {
  return pairs <= 64 ? 128 : pairs <= 256 ? 256 : 512;
}

int splits_of(long pairs, long max_tokens) {
  // Enough runs for the longest sequence the table can hold, up to a grid of
  // CAP. Workgroups past a sequence's end leave at once but take a slot for
  // a microsecond; the runs are the grid's slowest dimension so that they
  // come after the ones that work (64 x 290 tokens, with two parts of a
  // probability: 15 us, 31 us with the runs inside the sequences). Caps of 1024 and 4096 measured 0 to 17 %
  // slower at 250 sequences and within 4 % elsewhere.
  const long want = (max_tokens + chunk_of(pairs) - 1) / chunk_of(pairs);
  return (int)std::max<long>(
      1, std::min<long>(std::min<long>(want, MAX_SPLITS), CAP / pairs));
}

}  // namespace

// `arrived` [B * n_kv] int32 has to be zero when the kernel starts.
void decode_attention_counted(torch::Tensor out, torch::Tensor q,
                              torch::Tensor k_cache, torch::Tensor v_cache,
                              torch::Tensor page_table, torch::Tensor seq_lens,
                              torch::Tensor arrived, double scale, bool packed) {
  TORCH_CHECK(out.is_contiguous());
  TORCH_CHECK(q.scalar_type() == at::kBFloat16);
  TORCH_CHECK(page_table.scalar_type() == at::kInt &&
              seq_lens.scalar_type() == at::kInt);
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == q.size(2));
  const int B = q.size(0), n_q = q.size(1), Dh = q.size(2);
  const int n_kv = k_cache.size(1), PS = k_cache.size(3);
  const int max_pages = page_table.size(1);
  const int ratio = n_q / n_kv;
  TORCH_CHECK(Dh == 128, "decode attention: head_dim 128 only");
  TORCH_CHECK(n_q % n_kv == 0);
  if (B == 0) return;
  // query rows are read 16 bytes at a time; others are accepted as copies
  if (q.stride(0) % 8 != 0 ||
      reinterpret_cast<uintptr_t>(q.data_ptr()) % 16 != 0)
    q = q.clone(at::MemoryFormat::Contiguous);
  TORCH_CHECK(arrived.scalar_type() == at::kInt &&
              arrived.numel() >= (long)B * n_kv);
  TORCH_CHECK(!packed || B <= PACKED_ROWS);
  const int ms = packed ? packed_groups(B) : 0;
  const long out_size = (packed ? (long)ms * 16 : (long)B) * n_q * Dh;
  TORCH_CHECK(packed ? out.numel() == out_size : out.numel() >= out_size);
  const long pairs = (long)B * n_kv;
  const int n_split = splits_of(pairs, (long)max_pages * PS);
  auto part = torch::empty(
      {n_split > 1 ? pairs * n_split * ratio * PART : 1},
      torch::TensorOptions().dtype(torch::kFloat).device(q.device()));
  int ps_shift = 0;
  while ((1 << ps_shift) < PS) ++ps_shift;
  const int page = PS == 16 ? 16 : PS > 16 && (1 << ps_shift) == PS ? 1 : 0;
  // exponents in base 2; a negative scale is moved into Q's signs
  const float c = std::max((float)(std::fabs(scale) * 1.4426950408889634),
                           1e-30f);
  auto stream = at::hip::getCurrentHIPStream();
  const bool fp8 = k_cache.scalar_type() == at::kFloat8_e4m3fn;
  TORCH_CHECK(fp8 || k_cache.scalar_type() == at::kBFloat16);
#define DA_LAUNCH(R, CT, PAGE_)                                                \
  hipLaunchKernelGGL((decode_attn_kernel<R, CT, PAGE_>),                         \
                     dim3(n_kv, B, n_split), dim3(WAVES * WAVE), 0, stream,    \
                     (short*)out.data_ptr(), part.data_ptr<float>(),           \
                     arrived.data_ptr<int>(), (const short*)q.data_ptr(),      \
                     (const CT*)k_cache.data_ptr(),                            \
                     (const CT*)v_cache.data_ptr(),                            \
                     page_table.data_ptr<int>(), seq_lens.data_ptr<int>(), c,  \
                     scale < 0, n_kv, PS, ps_shift, max_pages,                 \
                     (long)q.stride(0), chunk_of(pairs), ms)
#define DA_PAGE(R, CT)                                                         \
  do {                                                                         \
    if (page == 16) DA_LAUNCH(R, CT, 16);                                      \
    else if (page == 1) DA_LAUNCH(R, CT, 1);                                   \
    else DA_LAUNCH(R, CT, 0);                                                  \
  } while (0)
#define DA_RATIO(R)                                                            \
  do {                                                                         \
    if (fp8) DA_PAGE(R, unsigned char);                                        \
    else DA_PAGE(R, short);                                                    \
  } while (0)
  switch (ratio) {
    case 1: DA_RATIO(1); break;
    case 2: DA_RATIO(2); break;
    case 4: DA_RATIO(4); break;
    case 8: DA_RATIO(8); break;
    default:
      TORCH_CHECK(false, "decode attention: GQA ratio must be 1/2/4/8, got ",
                  ratio);
  }
#undef DA_RATIO
#undef DA_PAGE
#undef DA_LAUNCH
}

void paged_decode_attention(torch::Tensor out, torch::Tensor q,
                            torch::Tensor k_cache, torch::Tensor v_cache,
                            torch::Tensor page_table, torch::Tensor seq_lens,
                            double scale) {
  auto arrived = torch::zeros(
      {(long)q.size(0) * k_cache.size(1)},
      torch::TensorOptions().dtype(torch::kInt).device(q.device()));
  decode_attention_counted(out, q, k_cache, v_cache, page_table, seq_lens,
                           arrived, scale, false);
}
