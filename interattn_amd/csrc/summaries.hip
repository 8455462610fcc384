// Per-block summaries of a paged K/V pool for gfx950 (the paged form of
// _build_prompt_blocks, CBT/core.py:449-500).
//
//   grid = (block groups x Hkv, batch), the kv head fastest, 256 threads; a block's keys
//   are summarised by one wave and its values by another (four blocks a workgroup where
//   only the mean keys are asked for, else two; more in large launches).  Tokens are read 16 at a time (one
//   page-resident subtile), 4 token rows per wave-wide load, 16 lanes per row
//   (DPL = D/16 dims per lane).  Sums are fp32 (the reference's
//   dtype=torch.float32 accumulation), extrema are exact copies, and the value
//   norm of each token is a DPP row sum of squares.  A second tiny kernel folds
//   v_norm_max into v_norm_all.
//
//   The kernel is bound by HBM reads, so what matters is that a wave always has row
//   loads in flight:
//   * a wave's subtiles' page ids, offsets and (fp8) scales are fetched at the start, one
//     subtile per lane, and read back with readlane: one dependent round trip per wave
//     instead of one per subtile;
//   * the subtiles run through a ring of register buffers, across the wave's consecutive
//     blocks: the next three subtiles' rows load while one is summed;
//   * K and V are read by different waves (their sums, extrema and norms together left
//     room for one subtile in flight per wave at half the waves), and V is not read
//     unless v_bar or its norms are asked for: a top-k program keeps only the mean keys
//     (with the extrema alone the values' waves are launched and leave at once);
//   * a block's rows are stored as 16-byte pieces, one array per lane row.
//   Measured (8 sequences of 40-64K tokens, 8 kv heads, D = 128, 64-token blocks, 16-token
//   pages; before -> after): bf16, every output 381 -> 319 us (5.3 TB/s of the bytes read
//   once and written once; without the extrema's and norms' arithmetic it measures 313),
//   mean keys 323 -> 144 us (5.8 TB/s); fp8 312 -> 202 and 290 -> 86 us.  The sums, extrema and
//   norms keep their order, hence their bits.
#include <algorithm>
#include <type_traits>

#include "ia_common.hpp"

namespace ia {
namespace {

struct SummaryParams {
  ia_paged_kv kv;
  const int32_t* seq_lens;
  int32_t n_kv_heads, block_size, nb_max;
  void* k_bar;
  void* v_bar;
  void* k_max;
  void* k_min;
  int32_t k_bar_dtype, v_bar_dtype, bounds_dtype;
  float* v_norm_max;
  float* v_norm_all;
  int32_t* counts;
  // incremental mode: blocks [old_seq_lens[b] / block_size, ceil(seq_lens[b] / block_size))
  // only, v_norm_all raised by atomic max (null: every block, full build)
  const int32_t* old_seq_lens;
  int32_t vec_store;      // every summary array is 16-byte aligned
  int32_t window_blocks;  // blocks per sequence this launch covers
  int32_t wave_blocks;    // consecutive blocks per wave
};

// One token row slice of DPL elements as raw words, loaded before any use.
template <int DPL, int EB>
struct RowWords {
  static constexpr int kWords = DPL * EB / 4;
  u32 w[kWords];
  __device__ __forceinline__ void load(const char* p) {
    if constexpr (kWords >= 4) {
#pragma unroll
      for (int i = 0; i < kWords; i += 4) {
        const u32x4_t a = ld_stream16(p + 4 * i);
        w[i] = a[0]; w[i + 1] = a[1]; w[i + 2] = a[2]; w[i + 3] = a[3];
      }
    } else if constexpr (kWords == 2) {
      const u32x2_t a = ld_stream8(p);
      w[0] = a[0]; w[1] = a[1];
    } else {
      w[0] = ld_stream4(p);
    }
  }
  __device__ __forceinline__ void get(float* out) const {
    if constexpr (EB == 4) {
#pragma unroll
      for (int e = 0; e < DPL; ++e) out[e] = __uint_as_float(w[e]);
    } else if constexpr (EB == 2) {
#pragma unroll
      for (int e = 0; e < DPL / 2; ++e) {
        out[2 * e] = bf16_lo(w[e]);
        out[2 * e + 1] = bf16_hi(w[e]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < DPL / 4; ++e) fp8x4_to_f32(w[e], out + 4 * e);
    }
  }
};

// Subtile buffers of a wave's ring: four of 16 rows (three in flight while one is
// summed), two for fp32 rows of 128 dims (registers).
template <int D, int EB>
constexpr int summary_ring() { return D * EB > 256 ? 2 : 4; }

// v + v[lane ^ 16], then + the same of lane ^ 32: the order of the four token rows' sum
__device__ __forceinline__ float fold_rows_sum(float v) {
  auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(t[0]) + __uint_as_float(t[1]);
  t = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(t[0]) + __uint_as_float(t[1]);
}

// DPL values of one summary row slice; vec: the arrays are 16-byte aligned.
template <int DPL>
__device__ __forceinline__ void store_slice(void* base, int64_t off, bool bf16, bool vec, const float* v) {
  if (bf16) {
    u32 w[DPL / 2];
#pragma unroll
    for (int e = 0; e < DPL / 2; ++e) w[e] = pack_bf16x2(v[2 * e], v[2 * e + 1]);
    unsigned short* p = reinterpret_cast<unsigned short*>(base) + off;
    if (vec) {
      if constexpr (DPL == 8) *reinterpret_cast<u32x4_t*>(p) = u32x4_t{w[0], w[1], w[2], w[3]};
      else *reinterpret_cast<u32x2_t*>(p) = u32x2_t{w[0], w[1]};
    } else {
#pragma unroll
      for (int e = 0; e < DPL; ++e) p[e] = (unsigned short)(w[e >> 1] >> (16 * (e & 1)));
    }
  } else {
    float* p = reinterpret_cast<float*>(base) + off;
    if (vec) {
#pragma unroll
      for (int e = 0; e < DPL; e += 4) *reinterpret_cast<f32x4_t*>(p + e) = f32x4_t{v[e], v[e + 1], v[e + 2], v[e + 3]};
    } else {
#pragma unroll
      for (int e = 0; e < DPL; ++e) p[e] = v[e];
    }
  }
}

// What a wave reads of its block: K for the mean keys alone, K for the means and
// extrema, or V for the means and norms.
enum { kMeanKeys = 0, kKeys = 1, kValues = 2 };

template <int D, int EB, int ROLE>
__device__ __forceinline__ void summarise_blocks(const SummaryParams& p, int b, int h, int j0, int j1, int seq_len) {
  constexpr int DPL = D / 16;
  constexpr int NBUF = summary_ring<D, EB>();
  constexpr bool kV = ROLE == kValues;
  const int lane = threadIdx.x & 63;
  const int c16 = lane & 15;
  const int r = lane >> 4;
  const ia_paged_kv& kv = p.kv;
  const int nsb = p.block_size / 16;  // subtiles per block
  const int32_t* bt_row = kv.block_table ? kv.block_table + (int64_t)b * kv.bt_stride : nullptr;
  const int64_t bh = (int64_t)b * p.n_kv_heads + h;

  float sum[DPL], mx[DPL], mn[DPL];
  float sq_max;  // largest squared value norm (its root is taken once: sqrt is monotone)
  int cnt;
  auto clear = [&]() {
#pragma unroll
    for (int e = 0; e < DPL; ++e) {
      sum[e] = 0.f;
      mx[e] = kNegInf;
      mn[e] = -kNegInf;
    }
    sq_max = kNegInf;
    cnt = 0;
  };
  // block j's results: the 4 token rows folded; every lane row then holds the block's
  // values and stores one of the wave's arrays
  auto flush = [&](int j) {
    const float inv = 1.0f / (float)max(cnt, 1);
    float o[DPL];
#pragma unroll
    for (int e = 0; e < DPL; ++e) {
      o[e] = fold_rows_sum(sum[e]) * inv;
      if constexpr (ROLE == kKeys) {
        const float hi = rows_max(mx[e]), lo = -rows_max(-mn[e]);
        o[e] = r == 0 ? o[e] : r == 1 ? hi : lo;
      }
    }
    void* dst = kV ? p.v_bar : r == 0 ? p.k_bar : r == 1 ? p.k_max : p.k_min;
    const int dt = kV ? p.v_bar_dtype : r == 0 ? p.k_bar_dtype : p.bounds_dtype;
    if (dst && r < (ROLE == kKeys ? 3 : 1))
      store_slice<DPL>(dst, (bh * p.nb_max + j) * D + c16 * DPL, dt == IA_BF16, p.vec_store, o);
    if constexpr (kV) {
      sq_max = wave_max(sq_max);
      if (lane == 0) {
        const float vn = sq_max == kNegInf ? kNegInf : sqrtf(sq_max);
        if (p.v_norm_max) p.v_norm_max[bh * p.nb_max + j] = vn;
        // a refreshed block's norm only grows (tokens are appended), so the running
        // maximum stays exact; values are >= 0 or -inf, whose int32 bit patterns
        // order like the floats
        if (p.old_seq_lens && p.v_norm_all)
          atomicMax(reinterpret_cast<int*>(p.v_norm_all) + bh, __float_as_int(vn));
      }
    } else if (lane == 0 && h == 0) {
      p.counts[(int64_t)b * p.nb_max + j] = cnt;
    }
    clear();
  };
  clear();
  int cur = j0;  // the block being summed

  // row 4 i + r of a subtile at this lane's dims: 4 i ts + row_off bytes past its first row
  const int64_t ts = (kV ? kv.v_token_stride : kv.k_token_stride) * EB;
  const int64_t lane_off = c16 * DPL * EB;
  const int64_t row_off = r * ts + lane_off;
  const char* base = reinterpret_cast<const char*>(kV ? kv.v : kv.k) +
                     (int64_t)h * (kV ? kv.v_head_stride : kv.k_head_stride) * EB;

  const int n_all = (j1 - j0) * nsb;
  for (int s0 = 0; s0 < n_all; s0 += 64) {
    // lane l: subtile s0 + l of the wave's blocks, its valid rows, offset and scale
    int nv_l = 0;
    int64_t off_l = 0;
    float sc_l = 1.f;
    const int64_t tok = (int64_t)j0 * p.block_size + 16 * (s0 + lane);
    const int blk_l = j0 + (s0 + lane) / nsb;
    if (s0 + lane < n_all && tok < seq_len) {
      const int lp = (int)tok / kv.page_size;
      int64_t pg = lp;
      if (bt_row) pg = lp < kv.bt_cols ? (int64_t)bt_row[lp] : -1;
      if (pg >= 0 && pg < kv.n_pages) {
        nv_l = min(16, seq_len - (int)tok);
        off_l = pg * (kV ? kv.v_page_stride : kv.k_page_stride) * EB + (int64_t)((int)tok - lp * kv.page_size) * ts;
        if constexpr (EB == 1) sc_l = (kV ? kv.v_scale : kv.k_scale)[pg * kv.scale_page_stride + h];
      }
    }
    unsigned long long todo = __ballot(nv_l > 0);  // subtiles with rows, ascending
    const int n = __popcll(todo);
    if (n == 0) continue;

    struct Sub {
      int nv;   // valid rows (0: a placeholder past the list)
      int blk;  // its block
      float sc;
    };
    RowWords<DPL, EB> buf[NBUF][4];
    Sub ring[NBUF];
    int src = 0;
    // the next subtile of the list; past it the loads stay unconditional (one row already
    // read, so every path issues the same loads and the wait counts stay exact)
    auto issue = [&](RowWords<DPL, EB>* rows, Sub& sb) {
      const bool more = todo != 0ull;
      src = more ? __ffsll((long long)todo) - 1 : src;
      todo &= todo - 1ull;
      const u32 lo = (u32)__builtin_amdgcn_readlane((int)(u32)off_l, src);
      const u32 hi = (u32)__builtin_amdgcn_readlane((int)(u32)((uint64_t)off_l >> 32), src);
      const char* p0 = base + (int64_t)((uint64_t)hi << 32 | lo);
      sb.nv = more ? __builtin_amdgcn_readlane(nv_l, src) : 0;
      sb.blk = __builtin_amdgcn_readlane(blk_l, src);
      sb.sc = EB == 1 ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sc_l), src)) : 1.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) rows[i].load(p0 + (4 * i + r < sb.nv ? 4 * i * ts + row_off : lane_off));
    };
    auto sum_rows = [&](auto full, const RowWords<DPL, EB>* rows, const Sub& sb) {
      // (written out, so that every instance sums an fp8 row with the same roundings)
#pragma clang fp contract(off)
      constexpr bool kFull = decltype(full)::value;
      float sq[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool valid = kFull || 4 * i + r < sb.nv;
        float f[DPL], a = 0.f;
        rows[i].get(f);
#pragma unroll
        for (int e = 0; e < DPL; ++e) {
          const float x = EB == 1 ? f[e] * sb.sc : f[e];
          if constexpr (kV) a = fmaf(x, x, a);
          if (valid) {
            sum[e] = EB == 1 && !kV ? fmaf(f[e], sb.sc, sum[e]) : sum[e] + x;
            if constexpr (ROLE == kKeys) {
              mx[e] = fmaxf(mx[e], x);
              mn[e] = fminf(mn[e], x);
            }
          }
        }
        sq[i] = a;
      }
      if constexpr (kV) {
        // lane c16 of a row ends with the squared norm of token 4 (c16 >> 2) + r (the
        // same pairs added in the same tree as a row sum per token)
        reduce_scatter16<4>(sq, lane);
        if (kFull || 4 * (c16 >> 2) + r < sb.nv) sq_max = fmaxf(sq_max, sq[0]);
      }
    };
    auto step = [&](auto kc) {
      constexpr int k = decltype(kc)::value;
      constexpr int fk = (k + NBUF - 1) % NBUF;
      issue(buf[fk], ring[fk]);
      __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the older subtile's sums
      if (ring[k].nv == 0) return;
      while (cur < ring[k].blk) flush(cur++);
      if (ring[k].nv == 16) sum_rows(std::true_type{}, buf[k], ring[k]);
      else sum_rows(std::false_type{}, buf[k], ring[k]);
      cnt += ring[k].nv;
    };
#pragma unroll
    for (int k = 0; k < NBUF - 1; ++k) {
      issue(buf[k], ring[k]);
      __builtin_amdgcn_sched_barrier(0);
    }
    for (int k = 0; k < n; k += NBUF) {  // whole rotations (the last may end in placeholders)
      step(std::integral_constant<int, 0>{});
      step(std::integral_constant<int, 1>{});
      if constexpr (NBUF > 2) {
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
      }
    }
  }
  while (cur < j1) flush(cur++);
}

// ALL: a block's K and V by two waves (every output; null ones skipped); else one wave
// per block, k_bar and counts only, and V is not read.  A wave takes p.wave_blocks
// consecutive blocks.
template <int D, int EB, bool ALL>
__global__ __launch_bounds__(256) void ia_condition_block_summaries(SummaryParams p) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.x % p.n_kv_heads;
  const int x = blockIdx.x / p.n_kv_heads;
  const int b = blockIdx.y;
  const int seq_len = max(p.seq_lens[b], 0);
  int j0 = (ALL ? x * 2 + (wave >> 1) : x * 4 + wave) * p.wave_blocks;
  int j1 = min(j0 + p.wave_blocks, p.window_blocks);
  if (p.old_seq_lens) {  // only blocks holding tokens are refreshed
    const int first = max(p.old_seq_lens[b], 0) / p.block_size;
    j0 += first;
    j1 = min(j1 + first, seq_len / p.block_size + (seq_len % p.block_size != 0));
  }
  j1 = min(j1, p.nb_max);
  if (j0 >= j1) return;
  if constexpr (!ALL) summarise_blocks<D, EB, kMeanKeys>(p, b, h, j0, j1, seq_len);
  else if (wave & 1) {
    if (p.v_bar || p.v_norm_max) summarise_blocks<D, EB, kValues>(p, b, h, j0, j1, seq_len);
  } else {
    summarise_blocks<D, EB, kKeys>(p, b, h, j0, j1, seq_len);
  }
}

__global__ __launch_bounds__(256) void ia_condition_block_vnorm_all(const float* v_norm_max, float* v_norm_all,
                                                                    int32_t nb_max) {
  __shared__ float red[4];
  const int bh = blockIdx.x;
  float m = kNegInf;
  for (int j = threadIdx.x; j < nb_max; j += 256) m = fmaxf(m, v_norm_max[(int64_t)bh * nb_max + j]);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) v_norm_all[bh] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

template <int D, bool ALL>
void launch_summaries(const SummaryParams& p, int eb, dim3 grid, hipStream_t st) {
  if (eb == 4) hipLaunchKernelGGL((ia_condition_block_summaries<D, 4, ALL>), grid, dim3(256), 0, st, p);
  else if (eb == 2) hipLaunchKernelGGL((ia_condition_block_summaries<D, 2, ALL>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((ia_condition_block_summaries<D, 1, ALL>), grid, dim3(256), 0, st, p);
}

}  // namespace
}  // namespace ia

namespace ia {
namespace {

int run_summaries(const ia_paged_kv* kv, const int32_t* old_seq_lens, const int32_t* seq_lens, int32_t batch,
                  int32_t n_kv_heads, int32_t head_dim, int32_t block_size, int32_t nb_max, int32_t window_blocks,
                  void* k_bar, int32_t k_bar_dtype, void* v_bar, int32_t v_bar_dtype, void* k_max, void* k_min,
                  int32_t bounds_dtype, float* v_norm_max, float* v_norm_all, int32_t* counts, void* stream) {
  if (!kv || !kv->k || !kv->v || !seq_lens || !counts) return fail(IA_ERR_INVALID, "null pointer argument");
  if (head_dim != 64 && head_dim != 128) return fail(IA_ERR_UNSUPPORTED, "head_dim must be 64 or 128");
  if (block_size <= 0 || block_size % 16) return fail(IA_ERR_INVALID, "block_size must be a positive multiple of 16");
  if (kv->page_size <= 0 || kv->page_size % 16) return fail(IA_ERR_INVALID, "page_size must be a positive multiple of 16");
  if (batch < 0 || n_kv_heads <= 0 || nb_max < 0) return fail(IA_ERR_INVALID, "batch/heads/nb_max");
  const int32_t dts[3] = {k_bar_dtype, v_bar_dtype, bounds_dtype};
  for (int32_t dt : dts)
    if (dt != IA_F32 && dt != IA_BF16) return fail(IA_ERR_INVALID, "summary dtypes must be IA_F32 or IA_BF16");
  if (kv->dtype == IA_FP8_E4M3 && (!kv->k_scale || !kv->v_scale)) return fail(IA_ERR_INVALID, "fp8 needs scales");
  if (v_norm_all && !v_norm_max) return fail(IA_ERR_INVALID, "v_norm_all needs v_norm_max");
  const int eb = kv->dtype == IA_F32 ? 4 : (kv->dtype == IA_BF16 ? 2 : 1);
  if ((kv->k_token_stride * eb) % 16 || (kv->v_token_stride * eb) % 16 || (kv->k_page_stride * eb) % 16 ||
      (kv->v_page_stride * eb) % 16 || (kv->k_head_stride * eb) % 16 || (kv->v_head_stride * eb) % 16)
    return fail(IA_ERR_INVALID, "kv strides must be 16-byte multiples");
  if (batch == 0 || nb_max == 0 || window_blocks == 0) return IA_OK;
  SummaryParams p{};
  p.kv = *kv;
  p.seq_lens = seq_lens;
  p.old_seq_lens = old_seq_lens;
  p.n_kv_heads = n_kv_heads;
  p.block_size = block_size;
  p.nb_max = nb_max;
  p.k_bar = k_bar;
  p.v_bar = v_bar;
  p.k_max = k_max;
  p.k_min = k_min;
  p.k_bar_dtype = k_bar_dtype;
  p.v_bar_dtype = v_bar_dtype;
  p.bounds_dtype = bounds_dtype;
  p.v_norm_max = v_norm_max;
  p.v_norm_all = v_norm_all;
  p.counts = counts;
  p.vec_store = ((reinterpret_cast<uintptr_t>(k_bar) | reinterpret_cast<uintptr_t>(v_bar) |
                  reinterpret_cast<uintptr_t>(k_max) | reinterpret_cast<uintptr_t>(k_min)) % 16) == 0;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool all = v_bar || k_max || k_min || v_norm_max;
  p.window_blocks = window_blocks;
  // Consecutive blocks per wave: enough that a wave's ring runs over about 16 subtiles
  // (8 where only the mean keys are asked for) instead of draining at every block, as long
  // as the launch keeps 48 waves per CU: four rounds of the D = 128 instances with every
  // output (12 resident waves per CU), three of the mean keys' (16), fewer of the D = 64
  // ones (16 to 32).  Measured, 8 x 40-64K tokens of
  // bf16 D = 128, every output: 64-token blocks 343 us with one block per wave, 326 / 319
  // / 326 us with 8 / 16 / 32 subtiles; 16-token blocks 721 -> 422 us; mean keys only,
  // 144 / 144 / 146 / 151 us with 4 / 8 / 16 / 32.  A batch of 2 x 30K: 49.7 us with one
  // block per wave, 51.6 with two.
  const int64_t waves = (int64_t)window_blocks * n_kv_heads * batch * (all ? 2 : 1);
  p.wave_blocks = (int)std::max<int64_t>(1, std::min<int64_t>((all ? 16 : 8) / (block_size / 16), waves / (48 * device_cus())));
  const int per_wg = (all ? 2 : 4) * p.wave_blocks;  // blocks per workgroup
  dim3 grid((window_blocks + per_wg - 1) / per_wg * n_kv_heads, batch);
  if (head_dim == 128) all ? launch_summaries<128, true>(p, eb, grid, st) : launch_summaries<128, false>(p, eb, grid, st);
  else all ? launch_summaries<64, true>(p, eb, grid, st) : launch_summaries<64, false>(p, eb, grid, st);
  int rc = check_launch("block summaries");
  if (rc) return rc;
  if (v_norm_all && !old_seq_lens) {
    hipLaunchKernelGGL(ia_condition_block_vnorm_all, dim3(batch * n_kv_heads), dim3(256), 0, st, v_norm_max,
                       v_norm_all, nb_max);
    rc = check_launch("v_norm_all");
  }
  return rc;
}

}  // namespace
}  // namespace ia

extern "C" int ia_build_block_summaries(const ia_paged_kv* kv, const int32_t* seq_lens, int32_t batch,
                                        int32_t n_kv_heads, int32_t head_dim, int32_t block_size, int32_t nb_max,
                                        void* k_bar, int32_t k_bar_dtype, void* v_bar, int32_t v_bar_dtype,
                                        void* k_max, void* k_min, int32_t bounds_dtype, float* v_norm_max,
                                        float* v_norm_all, int32_t* counts, void* stream) {
  return ia::run_summaries(kv, nullptr, seq_lens, batch, n_kv_heads, head_dim, block_size, nb_max, nb_max, k_bar,
                           k_bar_dtype, v_bar, v_bar_dtype, k_max, k_min, bounds_dtype, v_norm_max, v_norm_all,
                           counts, stream);
}

extern "C" int ia_update_block_summaries(const ia_paged_kv* kv, const int32_t* old_seq_lens, const int32_t* seq_lens,
                                         int32_t batch, int32_t n_kv_heads, int32_t head_dim, int32_t block_size,
                                         int32_t nb_max, int32_t max_new_tokens, void* k_bar, int32_t k_bar_dtype,
                                         void* v_bar, int32_t v_bar_dtype, void* k_max, void* k_min,
                                         int32_t bounds_dtype, float* v_norm_max, float* v_norm_all, int32_t* counts,
                                         void* stream) {
  using namespace ia;
  if (!old_seq_lens) return fail(IA_ERR_INVALID, "old_seq_lens must be non-null");
  if (max_new_tokens < 0) return fail(IA_ERR_INVALID, "max_new_tokens must be >= 0");
  if (block_size <= 0) return fail(IA_ERR_INVALID, "block_size must be a positive multiple of 16");
  // the partial block at the old end plus every block the new tokens can reach
  const int64_t window = std::min<int64_t>((int64_t)nb_max, ((int64_t)max_new_tokens + block_size - 1) / block_size + 1);
  return run_summaries(kv, old_seq_lens, seq_lens, batch, n_kv_heads, head_dim, block_size, nb_max, (int32_t)window,
                       k_bar, k_bar_dtype, v_bar, v_bar_dtype, k_max, k_min, bounds_dtype, v_norm_max, v_norm_all,
                       counts, stream);
}
