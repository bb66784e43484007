// The router's selection for one wave, as device functions: the select kernels (router.hip; the selection itself is described
// there) and the launch that selects beside a projection (few_tokens.hip) share them.
#pragma once
#include "common.h"

namespace omni {

// Storage dtype handled at run time, one uniform branch per access: for the norms' buffers, whose dtype is their own.  (The scores' dtype is a template
// parameter: with a branch to every load and rounding a token was 142 branches to 817 vector instructions, and its loads waited for one another.)
__device__ __forceinline__ float load_score(const void* p, int64_t i, int dt) {
  return dt == kBF16 ? Elem<kBF16>::load(p, i) : dt == kF16 ? Elem<kF16>::load(p, i) : Elem<kF32>::load(p, i);
}
__device__ __forceinline__ void store_score(void* p, int64_t i, float v, int dt) {
  if (dt == kBF16) Elem<kBF16>::store(p, i, v);
  else if (dt == kF16) Elem<kF16>::store(p, i, v);
  else Elem<kF32>::store(p, i, v);
}

constexpr int kRouterWaves = 4;
constexpr int kUnrollMaxR = 2;     // lists of <= 128 items use the unrolled, LDS-free exchanges
constexpr int kMaxKeys = 1024;        // keys per half that the select kernels hold in registers (16 per lane)
constexpr int kMaxKeysChunked = 16384; // ... that the chunked kernel walks (16-bit scores, at most 64 candidates per half)
constexpr float kNegInf = -__builtin_huge_valf();

struct SelectArgs {
  const void* lx;        // x-half scores of token t at lx[t*row_stride + key]
  const void* ly;
  int64_t row_stride;
  const float* stats;    // NULL, or [4][r] fp32: mean_x, rstd_x, mean_y, rstd_y -> the inputs are raw
                         // projections; normalise and log-softmax them before selecting
  const void* run_mean[2];  // instead of stats (eval-mode BatchNorm): the two halves' running_mean / running_var
  const void* run_var[2];   //   [r] of dtype stat_dt; mean and 1/sqrt(var + eps) are formed here, and block 0
  float* stats_out;         //   also leaves them at stats_out [4][r] (may be NULL) for a backward pass
  int stat_dt;
  float eps;
  void* scores;          // [T,k] storage dtype, may be NULL
  void* gates;           // [T,k] storage dtype = exp(score), may be NULL
  int32_t* indices;      // [T,k]
  int num_tokens, r, k, kp, dt;
  uint8_t row_cells[128]; // candidate cells in row a: min(kp, k/(a+1)), filled by select_dispatch
  int64_t* count_batch[2]; // NULL, or BatchNorm's num_batches_tracked of the two halves: incremented here, behind the
                           // kernel that read them (train-mode router stage)
  const float* part_mean;  // NULL, or the projection's column statistics [strips][2r] of every 32 rows (training; joint launches): each block merges them
  const float* part_m2;    //   itself (merge_statistics); block 0 moves run_mean / run_var with `momentum` and leaves the result at stats_out
  int strips;
  float momentum;          // < 0: cumulative average, factor 1 / (batches tracked so far + 1)
};
constexpr int kMergeKeys = 128;    // keys per half up to which a block merges batch statistics itself
constexpr int kBnRows = 32;       // rows per strip: one 32-row MFMA tile of the projection GEMM

// One column's batch statistics from its strips' sums (mean = sum n_s mean_s / n, M2 = sum M2_s + n_s mean_s^2 - n mean^2, in double: 29 bits more than
// the fp32 result keeps, so the difference stays exact to fp32 while mean^2 / variance < 2^29).
struct ColumnSums { double weighted, squares; };
__device__ __forceinline__ void add_strip(ColumnSums& c, float mean, float m2, int strip, int num_rows) {
  const double ns = (double)min(kBnRows, num_rows - strip * kBnRows), ms = (double)mean;
  c.weighted += ns * ms;
  c.squares += (double)m2 + ns * ms * ms;
}
__device__ __forceinline__ void add_strip(ColumnSums& c, const float* part_mean, const float* part_m2, int strip, int cols, int col, int num_rows) {
  const int64_t at = int64_t(strip) * cols + col;
  add_strip(c, part_mean[at], part_m2[at], strip, num_rows);
}
// ... of up to N strips first, first + step, ..: all requested before the first is waited for, the last strip again in place of those behind it
template <int N>
__device__ __forceinline__ void add_batch(ColumnSums& c, const float* part_mean, const float* part_m2, int first, int step, int strips, int cols, int col, int num_rows) {
  float mean[N], m2[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int64_t at = int64_t(min(first + j * step, strips - 1)) * cols + col;
    mean[j] = part_mean[at];
    m2[j] = part_m2[at];
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < N; ++j)
    if (first + j * step < strips) add_strip(c, mean[j], m2[j], first + j * step, num_rows);
}
struct ColumnStats { float mean, var, unbiased; };             // var: biased, normalises the batch
__device__ __forceinline__ ColumnStats column_stats(const ColumnSums& c, int num_rows) {
  const double n = (double)num_rows, mu = c.weighted / n, m2 = fmax(c.squares - n * mu * mu, 0.);
  return {(float)mu, (float)(m2 / n), (float)(m2 / (n > 1. ? n - 1. : 1.))};
}
__device__ __forceinline__ float rstd_of(float var, float eps) { return 1.0f / sqrtf(var + eps); }

// Batch statistics for a block of `threads` that selects, beside another kernel's tiles or (router_fwd says where) by itself: every such block merges all columns, 2r of
// them with 16384 strip values in all at most (merge_here), where a merge of its own is a 4-5 us launch between projection and selection.  Strips are requested eight at
// a time and those left over, up to seven a thread, at once: batches of eight alone left the remainder to a wait each (512 tokens x 32 keys in single precision 25.3 us,
// not unrolled 25.2, now 24.8; 2000 tokens 44.8, 46.8, 43.3).  lds: merge_lds_floats(r, threads) floats, 16-byte aligned; the first 4r hold mean_x, rstd_x,
// mean_y, rstd_y afterwards.
__device__ __host__ constexpr int merge_lds_floats(int r, int threads) { return (4 * r + 3) / 4 * 4 + 4 * threads; }
constexpr int kF32MergeThreads = 256;                         // of a block that merges in the single-precision layer's joint launches
__device__ __host__ constexpr int merge_parts(int r, int threads) { return threads / (2 * r) > 1 ? threads / (2 * r) : 1; }      // a column's sums are the parts' strided ones, in their order
__device__ __forceinline__ void merge_statistics(const SelectArgs& g, float* lds, const int threads) {
  const int cols = 2 * g.r, tid = threadIdx.x, parts = merge_parts(g.r, threads);
  ColumnSums* sums = (ColumnSums*)(lds + (4 * g.r + 3) / 4 * 4);
  for (int c0 = 0; c0 < cols; c0 += threads) {                  // (one round up to threads / 2 keys)
    const int part = tid / cols, col = c0 + (parts > 1 ? tid - part * cols : tid);
    if (part < parts && col < cols) {
      ColumnSums c{0., 0.};
      int strip = part;
      for (; strip + 7 * parts < g.strips; strip += 8 * parts)
#pragma unroll
        for (int j = 0; j < 8; ++j) add_strip(c, g.part_mean, g.part_m2, strip + j * parts, cols, col, g.num_tokens);
      if (strip < g.strips) add_batch<7>(c, g.part_mean, g.part_m2, strip, parts, g.strips, cols, col, g.num_tokens);
      sums[tid] = c;
    }
    __syncthreads();
    const int mine = c0 + tid;
    if (tid < min(cols - c0, threads)) {
      ColumnSums c = sums[tid];
      for (int q = 1; q < parts; ++q) {
        c.weighted += sums[q * cols + tid].weighted;
        c.squares += sums[q * cols + tid].squares;
      }
      const ColumnStats v = column_stats(c, g.num_tokens);
      const int half = mine >= g.r, key = mine - half * g.r;
      const float rstd = rstd_of(v.var, g.eps);
      lds[(2 * half) * g.r + key] = v.mean;
      lds[(2 * half + 1) * g.r + key] = rstd;
      if (blockIdx.x == 0) {
        const float f = g.momentum >= 0.f ? g.momentum : 1.0f / (float)(*g.count_batch[half] + 1);
        const float rm = load_score(g.run_mean[half], key, g.stat_dt), rv = load_score(g.run_var[half], key, g.stat_dt);
        store_score((void*)g.run_mean[half], key, (1.f - f) * rm + f * v.mean, g.stat_dt);
        store_score((void*)g.run_var[half], key, (1.f - f) * rv + f * v.unbiased, g.stat_dt);
        if (g.stats_out) {
          g.stats_out[(2 * half) * g.r + key] = v.mean;
          g.stats_out[(2 * half + 1) * g.r + key] = rstd;
        }
      }
    }
    __syncthreads();
  }
}

// (behind merge_statistics, which reads the counts)
__device__ __forceinline__ void count_batch(const SelectArgs& g) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (g.count_batch[0]) *g.count_batch[0] += 1;
    if (g.count_batch[1]) *g.count_batch[1] += 1;
  }
  if (blockIdx.x == 0 && !g.stats && !g.part_mean && g.run_mean[0] && g.stats_out) {   // eval mode: the statistics a backward pass reads
    for (int i = threadIdx.x; i < 2 * g.r; i += blockDim.x) {
      const int half = i >= g.r, key = i - half * g.r;
      g.stats_out[(2 * half) * g.r + key] = load_score(g.run_mean[half], key, g.stat_dt);
      g.stats_out[(2 * half + 1) * g.r + key] = __builtin_amdgcn_rsqf(load_score(g.run_var[half], key, g.stat_dt) + g.eps);
    }
  }
}

// BatchNorm (affine-free) of one raw projection value, rounded to the storage dtype as the reference's BatchNorm output is
template <int DT>
__device__ __forceinline__ float normalise_one(float v, const SelectArgs& g, const int half, const int key, const int r) {
  float mean, rstd;
  if (g.stats) {
    mean = g.stats[(2 * half) * r + key];
    rstd = g.stats[(2 * half + 1) * r + key];
  } else {
    mean = load_score(g.run_mean[half], key, g.stat_dt);
    rstd = __builtin_amdgcn_rsqf(load_score(g.run_var[half], key, g.stat_dt) + g.eps);
  }
  return Elem<DT>::round((v - mean) * rstd);
}

// Mean and 1/sqrt(var + eps) of this lane's keys: g.stats, or (eval mode) the running buffers with the hardware's reciprocal square root (1 ulp), as in
// stats_out, or a block's own merge (merged: the LDS that merge_statistics filled).  Held for all of a wave's tokens up to 8 keys a lane.
template <int R>
struct NormKeys {
  static constexpr bool kHeld = R <= 8;
  float mean[2][kHeld ? R : 1], rstd[2][kHeld ? R : 1];
  __device__ __forceinline__ static void one(const SelectArgs& g, const float* stats, int half, int key, float& mean, float& rstd) {
    if (stats) {
      mean = stats[(2 * half) * g.r + key];
      rstd = stats[(2 * half + 1) * g.r + key];
    } else {
      mean = load_score(g.run_mean[half], key, g.stat_dt);
      rstd = __builtin_amdgcn_rsqf(load_score(g.run_var[half], key, g.stat_dt) + g.eps);
    }
  }
  template <class Mean, class Rstd>
  __device__ __forceinline__ void fill(const SelectArgs& g, int lane, Mean&& mean_of, Rstd&& rstd_of) {
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int a = 0; a < R; ++a) {
        const int key = min(a * kWave + lane, g.r - 1);
        mean[half][a] = mean_of(half, key);
        rstd[half][a] = rstd_of(half, key);
      }
  }
  __device__ __forceinline__ NormKeys(const SelectArgs& g, const float* stats, int lane) {
    if constexpr (kHeld) {
      if (stats) {
        fill(g, lane, [&](int half, int key) { return stats[(2 * half) * g.r + key]; }, [&](int half, int key) { return stats[(2 * half + 1) * g.r + key]; });
      } else if (g.run_mean[0]) {
        auto buffers = [&](auto dt) {
          using B = Elem<decltype(dt)::value>;
          fill(g, lane, [&](int half, int key) { return B::load(g.run_mean[half], key); },
               [&](int half, int key) { return __builtin_amdgcn_rsqf(B::load(g.run_var[half], key) + g.eps); });
        };
        if (g.stat_dt == kBF16) buffers(std::integral_constant<int, kBF16>{});
        else if (g.stat_dt == kF16) buffers(std::integral_constant<int, kF16>{});
        else buffers(std::integral_constant<int, kF32>{});
      }
    }
  }
};

// BatchNorm (affine-free) then log-softmax of one half, in place: v holds the raw projection
// of key a*64+lane (NaN-free -inf padding past r).  Each stage rounds to the storage dtype
// where the reference's torch ops do (BN output, log-softmax output; omni_moe.py:70-78).
template <int DT, int R>
__device__ __forceinline__ void normalise_half(float (&v)[R], const SelectArgs& g, const NormKeys<R>& norm, const float* stats, const int half, int r, int lane) {
  float m = kNegInf;
#pragma unroll
  for (int a = 0; a < R; ++a) {
    const int key = a * kWave + lane;
    if (key < r) {
      float mean, rstd;
      if constexpr (NormKeys<R>::kHeld) { mean = norm.mean[half][a]; rstd = norm.rstd[half][a]; }
      else NormKeys<R>::one(g, stats, half, key, mean, rstd);
      v[a] = Elem<DT>::round((v[a] - mean) * rstd);
    }
    m = fmaxf(m, v[a]);
  }
  m = wave_max(m);
  float e = 0.f;
#pragma unroll
  for (int a = 0; a < R; ++a) e += (a * kWave + lane < r) ? expf(v[a] - m) : 0.f;
  const float lse = logf(wave_sum(e));
#pragma unroll
  for (int a = 0; a < R; ++a)
    if (a * kWave + lane < r) v[a] = Elem<DT>::round(v[a] - m - lse);
}

// This lane's candidate cells: cell index ci = c*64+lane enumerates rows a = 0..kp-1 with
// min(kp, k/(a+1)) cells each.  Payload (a<<8)|b orders like position a*kp+b.  The row counts
// come with the arguments: the lanes fetch them all at once (row a in lane a%64) and the uniform
// loop hands them round by readlane, so it waits for memory once, not once per row.
template <int R, int C>
__device__ __forceinline__ void candidate_cells(int (&cell)[C], const SelectArgs& g, const int kp, const int lane) {
#pragma unroll
  for (int c = 0; c < C; ++c) cell[c] = -1;
  // Measured per shape: with 4 or 8 keys and fewer than 8 cells per lane the plain loop, one load per row, is the faster
  // one by 3-6 % of the kernel (32768 tokens, 256-512 keys per half, k = 32); everywhere else the lanes' loop is, by 1-6 %.
  if constexpr (R > 2 && C < 8) {
    for (int a = 0, start = 0; a < kp; ++a) {
      const int cnt = g.row_cells[a];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int b = c * kWave + lane - start;
        cell[c] = (unsigned)b < (unsigned)cnt ? (a << 8) | b : cell[c];
      }
      start += cnt;
    }
    return;
  }
  const int cnt_lo = lane < kp ? g.row_cells[lane] : 0;
  const int cnt_hi = lane + kWave < kp ? g.row_cells[lane + kWave] : 0;
  int start = 0;
  for (int a = 0; a < min(kp, kWave); ++a) {
    const int cnt = __builtin_amdgcn_readlane(cnt_lo, a);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int b = c * kWave + lane - start;
      cell[c] = (unsigned)b < (unsigned)cnt ? (a << 8) | b : cell[c];
    }
    start += cnt;
  }
  for (int a = kWave; a < kp; ++a) {
    const int cnt = __builtin_amdgcn_readlane(cnt_hi, a - kWave);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int b = c * kWave + lane - start;
      cell[c] = (unsigned)b < (unsigned)cnt ? (a << 8) | b : cell[c];
    }
    start += cnt;
  }
}

// ---- scores and payloads as pairs -------------------------------------------------------------
// strict "a goes before b": higher score first, then lower payload
__device__ __forceinline__ bool goes_before(float sa, int pa, float sb, int pb) {
  return (sa > sb) || (sa == sb && pa < pb);
}

// Compare-exchange step with a compile-time lane distance, fully unrolled (small R only).
template <int R, int SIZE, int STRIDE>
__device__ __forceinline__ void lane_stage_ct(float (&s)[R], int (&p)[R], const int lane) {
#pragma unroll
  for (int a = 0; a < R; ++a) {
    const float os = xor_lane_f<STRIDE>(s[a], lane);
    const int op = xor_lane_i<STRIDE>(p[a], lane);
    const bool up = (((a * kWave) | lane) & SIZE) == 0;
    const bool lower = (lane & STRIDE) == 0;
    const bool take_other = (lower == up) != goes_before(s[a], p[a], os, op);
    s[a] = take_other ? os : s[a];
    p[a] = take_other ? op : p[a];
  }
}
// strides STRIDE, STRIDE/2, ..., 1 of the merge for block size SIZE, on NL lists in lockstep
template <int R, int SIZE, int STRIDE>
__device__ __forceinline__ void lane_stages_ct(float (&s0)[R], int (&p0)[R], float (&s1)[R], int (&p1)[R], const int lane, const bool two) {
  if constexpr (STRIDE >= 1) {
    lane_stage_ct<R, SIZE, STRIDE>(s0, p0, lane);
    if (two) lane_stage_ct<R, SIZE, STRIDE>(s1, p1, lane);
    lane_stages_ct<R, SIZE, STRIDE / 2>(s0, p0, s1, p1, lane, two);
  }
}
template <int R, int SIZE>
__device__ __forceinline__ void small_sizes_ct(float (&s0)[R], int (&p0)[R], float (&s1)[R], int (&p1)[R], const int lane, const bool two) {
  if constexpr (SIZE <= kWave) {
    lane_stages_ct<R, SIZE, SIZE / 2>(s0, p0, s1, p1, lane, two);
    small_sizes_ct<R, SIZE * 2>(s0, p0, s1, p1, lane, two);
  }
}

// One compare-exchange step between lanes `stride` apart (stride < 64), all R registers.
template <int R>
__device__ __forceinline__ void lane_stage(float (&s)[R], int (&p)[R], const int lane, const int size, const int stride) {
#pragma unroll
  for (int a = 0; a < R; ++a) {
    const float os = __shfl_xor(s[a], stride, kWave);
    const int op = __shfl_xor(p[a], stride, kWave);
    const bool up = (((a * kWave) | lane) & size) == 0;
    const bool lower = (lane & stride) == 0;
    const bool take_other = (lower == up) != goes_before(s[a], p[a], os, op);
    s[a] = take_other ? os : s[a];
    p[a] = take_other ? op : p[a];
  }
}

// One compare-exchange step between registers RS apart (element stride 64*RS).
template <int R, int SIZE, int RS>
__device__ __forceinline__ void reg_stage(float (&s)[R], int (&p)[R]) {
#pragma unroll
  for (int a = 0; a < R; ++a) {
    if ((a & RS) == 0) {
      const int b = a | RS;
      const bool up = ((a * kWave) & SIZE) == 0;
      const bool swap = goes_before(s[a], p[a], s[b], p[b]) != up;
      const float ts = swap ? s[b] : s[a];
      const int tp = swap ? p[b] : p[a];
      s[b] = swap ? s[a] : s[b];
      p[b] = swap ? p[a] : p[b];
      s[a] = ts;
      p[a] = tp;
    }
  }
}

template <int R, int SIZE, int RS>
__device__ __forceinline__ void reg_stages_down(float (&s)[R], int (&p)[R]) {
  if constexpr (RS >= 1) {
    reg_stage<R, SIZE, RS>(s, p);
    reg_stages_down<R, SIZE, RS / 2>(s, p);
  }
}

// Merge steps for block size SIZE (> 64) and the sizes above it, up to 64*R.

template <int R, int SIZE>
__device__ __forceinline__ void big_sizes(float (&s)[R], int (&p)[R], const int lane) {
  if constexpr (SIZE <= kWave * R) {
    reg_stages_down<R, SIZE, SIZE / (2 * kWave)>(s, p);
    if constexpr (R <= kUnrollMaxR) {
      lane_stages_ct<R, SIZE, kWave / 2>(s, p, s, p, lane, false);
    } else {
#pragma nounroll
      for (int stride = kWave / 2; stride >= 1; stride >>= 1) lane_stage<R>(s, p, lane, SIZE, stride);
    }
    big_sizes<R, SIZE * 2>(s, p, lane);
  }
}

// Sorts the 64*R (score, payload) items held as item e = reg*64 + lane with a bitonic
// network.  Steps between lanes run as rolled loops (the shuffle distance is a run-time
// value); steps between registers are unrolled so that register indices are constants.
template <int R>
__device__ __forceinline__ void bitonic_sort(float (&s)[R], int (&p)[R], const int lane) {
  if constexpr (R <= kUnrollMaxR) {
    small_sizes_ct<R, 2>(s, p, s, p, lane, false);
  } else {
#pragma nounroll
    for (int size = 2; size <= kWave; size <<= 1) {
#pragma nounroll
      for (int stride = size >> 1; stride >= 1; stride >>= 1) lane_stage<R>(s, p, lane, size, stride);
    }
  }
  big_sizes<R, 2 * kWave>(s, p, lane);
}

// Two independent lists sorted in lockstep: the two dependency chains interleave, which
// hides most of the cross-lane exchange latency.
template <int R, int SIZE>
__device__ __forceinline__ void big_sizes2(float (&s0)[R], int (&p0)[R], float (&s1)[R], int (&p1)[R], const int lane) {
  if constexpr (SIZE <= kWave * R) {
    reg_stages_down<R, SIZE, SIZE / (2 * kWave)>(s0, p0);
    reg_stages_down<R, SIZE, SIZE / (2 * kWave)>(s1, p1);
    if constexpr (R <= kUnrollMaxR) {
      lane_stages_ct<R, SIZE, kWave / 2>(s0, p0, s1, p1, lane, true);
    } else {
#pragma nounroll
      for (int stride = kWave / 2; stride >= 1; stride >>= 1) {
        lane_stage<R>(s0, p0, lane, SIZE, stride);
        lane_stage<R>(s1, p1, lane, SIZE, stride);
      }
    }
    big_sizes2<R, SIZE * 2>(s0, p0, s1, p1, lane);
  }
}
template <int R>
__device__ __forceinline__ void bitonic_sort2(float (&s0)[R], int (&p0)[R], float (&s1)[R], int (&p1)[R], const int lane) {
  if constexpr (R <= kUnrollMaxR) {
    small_sizes_ct<R, 2>(s0, p0, s1, p1, lane, true);
  } else {
#pragma nounroll
    for (int size = 2; size <= kWave; size <<= 1) {
#pragma nounroll
      for (int stride = size >> 1; stride >= 1; stride >>= 1) {
        lane_stage<R>(s0, p0, lane, size, stride);
        lane_stage<R>(s1, p1, lane, size, stride);
      }
    }
  }
  big_sizes2<R, 2 * kWave>(s0, p0, s1, p1, lane);
}

// value of sorted item `i` (i < 128) of a list held as item = reg*64+lane
template <int R, typename T>
__device__ __forceinline__ T sorted_item(const T (&v)[R], int i) {
  T r0 = __shfl(v[0], i & 63, kWave);
  if constexpr (R >= 2) {
    T r1 = __shfl(v[1], i & 63, kWave);
    r0 = (i >= kWave) ? r1 : r0;
  }
  return r0;
}

// The tokens of wave `wave` of `num_waves`, fp32 scores; stats: g.stats, or what the block merged.
// R = half keys per lane (r <= 64*R); C = candidate cells per lane.  With few keys per lane a wave requests
// the raw scores of its first token before anything else and those of its next token as soon as the current
// token's are consumed.
template <int R, int C>
__device__ __forceinline__ void select_pairs(const SelectArgs& g, const int wave, const int num_waves, const float* stats) {
  const int lane = lane_id();
  using S = Elem<kF32>;                           // (16-bit scores travel packed)
  const int r = g.r, k = g.k, kp = g.kp;

  float rx[R], ry[R];                             // raw scores of the token about to be selected
  auto load_raw = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < R; ++a) {
      const int key = a * kWave + lane;
      const bool ok = key < r;
      rx[a] = ok ? S::load(g.lx, int64_t(t) * g.row_stride + key) : kNegInf;
      ry[a] = ok ? S::load(g.ly, int64_t(t) * g.row_stride + key) : kNegInf;
    }
  };
  constexpr bool kPrefetch = R <= 2;              // beyond that the extra live registers cost a wave per SIMD
  if (kPrefetch && wave < g.num_tokens) load_raw(wave);
  const NormKeys<R> norm(g, stats, lane);
  int cell[C];
  candidate_cells<R, C>(cell, g, kp, lane);

  for (int t = wave; t < g.num_tokens; t += num_waves) {
    float sx[R], sy[R];
    int px[R], py[R];
#pragma unroll
    for (int a = 0; a < R; ++a) {
      const int key = a * kWave + lane;
      const bool ok = key < r;
      sx[a] = kPrefetch ? rx[a] : ok ? S::load(g.lx, int64_t(t) * g.row_stride + key) : kNegInf;
      sy[a] = kPrefetch ? ry[a] : ok ? S::load(g.ly, int64_t(t) * g.row_stride + key) : kNegInf;
      px[a] = py[a] = key;
    }
    if (kPrefetch && t + num_waves < g.num_tokens) load_raw(t + num_waves);
    if (stats || g.run_mean[0]) {
      normalise_half<kF32, R>(sx, g, norm, stats, 0, r, lane);
      normalise_half<kF32, R>(sy, g, norm, stats, 1, r, lane);
    }
    bitonic_sort2<R>(sx, px, sy, py, lane);

    float cs[C];
    int cp[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const bool ok = cell[c] >= 0;
      const int a = ok ? (cell[c] >> 8) : 0, b = ok ? (cell[c] & 255) : 0;
      const float va = sorted_item<R>(sx, a), vb = sorted_item<R>(sy, b);
      cs[c] = ok ? va + vb : kNegInf;
      cp[c] = ok ? cell[c] : (0x40000000 | (c * kWave + lane));
    }
    bitonic_sort<C>(cs, cp, lane);

    constexpr int kOut = (C >= 2) ? 2 : 1;          // k <= 128 -> winners live in regs 0..1
#pragma unroll
    for (int c = 0; c < kOut; ++c) {
      const int j = c * kWave + lane;
      const bool ok = j < k;
      const int a = ok ? (cp[c] >> 8) & 255 : 0, b = ok ? (cp[c] & 255) : 0;
      const int ia = sorted_item<R>(px, a), ib = sorted_item<R>(py, b);
      if (ok) {
        const int64_t o = int64_t(t) * k + j;
        if (g.scores) S::store(g.scores, o, cs[c]);
        if (g.gates) S::store(g.gates, o, expf(cs[c]));      // gate = P(x key) * P(y key)
        g.indices[o] = ia * r + ib;
      }
    }
  }
}

// ---- 16-bit scores: (score, payload) packed into one ordered 32-bit key ---------------------
// key = order-preserving image of the 16-bit score << 16 | (0xFFFF - payload): a larger key goes
// first, equal scores resolve to the lower payload, and a compare-exchange is one max / min.
// Four times fewer VALU instructions than the (float, int) pairs the fp32 path needs.
__device__ __forceinline__ uint32_t ord16(uint32_t bits) { return bits ^ ((bits & 0x8000u) ? 0xFFFFu : 0x8000u); }
__device__ __forceinline__ uint32_t unord16(uint32_t u) { return u ^ ((u & 0x8000u) ? 0x8000u : 0xFFFFu); }
template <int DT>
__device__ __forceinline__ uint32_t make_key(float v, int payload) {              // v is representable in DT
  v += 0.0f;                                                                      // -0 -> +0: they compare equal as floats
  const uint32_t bits = DT == kBF16 ? __float_as_uint(v) >> 16 : (uint32_t)f32_to_f16_bits(v);
  return (ord16(bits) << 16) | (0xFFFFu - (uint32_t)payload);
}
template <int DT>
__device__ __forceinline__ float key_score(uint32_t key) {
  const uint32_t bits = unord16(key >> 16);
  return DT == kBF16 ? bf16_bits_to_f32((uint16_t)bits) : f16_bits_to_f32((uint16_t)bits);
}
__device__ __forceinline__ int key_payload(uint32_t key) { return (int)(0xFFFFu - (key & 0xFFFFu)); }

// A compare-exchange of a key with its partner's: the lanes whose mask is all ones keep the larger, those whose mask is 0 the smaller (v_med3_u32)
__device__ __forceinline__ uint32_t keep_one(uint32_t a, uint32_t b, uint32_t mask) { return max(min(a, b), min(max(a, b), mask)); }
// lanes with this bit clear keep the larger
__device__ __forceinline__ uint32_t keep_mask(int lane, int bit) { return ((uint32_t)(lane / bit) & 1u) - 1u; }

// Sorting networks, every list descending (item e = reg*64 + lane): blocks of SIZE items are made of two sorted halves by a first exchange with the block's mirror
// image, e ^ (SIZE - 1), and exchanges at distances SIZE/4 .. 1.  No block is ever ascending, so the lanes that keep the larger key are those with one bit clear,
// whatever the size: six masks in all (a network of alternating directions has 21).  A compare-exchange is a DPP move and a v_med3 (it was a copy, a move, a
// minimum, a maximum and a choice): router with batch statistics, 4096 tokens x 64 keys 17.6 -> 16.3 us, selection of 32768 tokens x 512 keys 105 -> 92.
template <int DIST>
__device__ __forceinline__ uint32_t exchanged(uint32_t k, int lane) {             // at lane distance DIST
  const uint32_t mask = keep_mask(lane, DIST);
  if constexpr (DIST == 32) {
    const auto s = __builtin_amdgcn_permlane32_swap(k, k, false, false);          // (own and other, in one order or the other)
    return keep_one(s[0], s[1], mask);
  } else if constexpr (DIST == 16) {
    const auto s = __builtin_amdgcn_permlane16_swap(k, k, false, false);
    return keep_one(s[0], s[1], mask);
  } else {
    return keep_one(k, (uint32_t)xor_lane_i<DIST>((int)k, lane), mask);
  }
}
template <int SIZE>
__device__ __forceinline__ uint32_t mirrored(uint32_t k, int lane) {              // the value of lane ^ (SIZE - 1)
  if constexpr (SIZE == 2) return (uint32_t)dpp_i<kQuadXor1>((int)k);
  else if constexpr (SIZE == 4) return (uint32_t)dpp_i<kQuadXor3>((int)k);
  else if constexpr (SIZE == 8) return (uint32_t)dpp_i<kRowXor7>((int)k);
  else if constexpr (SIZE == 16) return (uint32_t)dpp_i<kRowXor15>((int)k);
  else if constexpr (SIZE == 32) return (uint32_t)__builtin_amdgcn_ds_swizzle((int)k, 0x7C1F);
  else return (uint32_t)__shfl((int)k, 63 - lane, kWave);
}
// lane distances DIST..1, on one or two lists in lockstep: the two dependency chains interleave
template <int R, int DIST>
__device__ __forceinline__ void kdistances(uint32_t (&k0)[R], uint32_t (&k1)[R], const int lane, const bool two) {
  if constexpr (DIST >= 1) {
#pragma unroll
    for (int a = 0; a < R; ++a) {
      k0[a] = exchanged<DIST>(k0[a], lane);
      if (two) k1[a] = exchanged<DIST>(k1[a], lane);
    }
    kdistances<R, DIST / 2>(k0, k1, lane, two);
  }
}
// every register by itself, up to blocks of 64
template <int R, int SIZE>
__device__ __forceinline__ void ksort_lanes(uint32_t (&k0)[R], uint32_t (&k1)[R], const int lane, const bool two) {
  if constexpr (SIZE <= kWave) {
    const uint32_t mask = keep_mask(lane, SIZE / 2);
#pragma unroll
    for (int a = 0; a < R; ++a) {
      k0[a] = keep_one(k0[a], mirrored<SIZE>(k0[a], lane), mask);
      if (two) k1[a] = keep_one(k1[a], mirrored<SIZE>(k1[a], lane), mask);
    }
    kdistances<R, SIZE / 4>(k0, k1, lane, two);
    ksort_lanes<R, SIZE * 2>(k0, k1, lane, two);
  }
}
// the same at run time, for many registers
template <int R>
__device__ __forceinline__ void kdistances_rt(uint32_t (&k)[R], const int lane) {
#pragma nounroll
  for (int dist = kWave / 2; dist >= 1; dist >>= 1) {
    const uint32_t mask = keep_mask(lane, dist);
#pragma unroll
    for (int a = 0; a < R; ++a) k[a] = keep_one(k[a], (uint32_t)__shfl_xor((int)k[a], dist, kWave), mask);
  }
}
template <int R, int RS>
__device__ __forceinline__ void kreg_distances(uint32_t (&k)[R]) {
  if constexpr (RS >= 1) {
#pragma unroll
    for (int a = 0; a < R; ++a) {
      if ((a & RS) == 0) {
        const uint32_t hi = max(k[a], k[a | RS]), lo = min(k[a], k[a | RS]);
        k[a] = hi;
        k[a | RS] = lo;
      }
    }
    kreg_distances<R, RS / 2>(k);
  }
}
// blocks of REGS sorted registers from two halves each, and the sizes above
template <int R, int REGS>
__device__ __forceinline__ void kmerge(uint32_t (&k0)[R], uint32_t (&k1)[R], const int lane, const bool two) {
  if constexpr (REGS <= R) {
    auto mirror = [&](uint32_t (&k)[R]) __attribute__((always_inline)) {
#pragma unroll
      for (int base = 0; base < R; base += REGS)
#pragma unroll
        for (int i = 0; i < REGS / 2; ++i) {
          const int a = base + i, b = base + REGS - 1 - i;
          const uint32_t ma = mirrored<kWave>(k[a], lane), mb = mirrored<kWave>(k[b], lane);
          k[a] = max(k[a], mb);
          k[b] = min(k[b], ma);
        }
      kreg_distances<R, REGS / 4>(k);
    };
    mirror(k0);
    if (two) mirror(k1);
    if constexpr (R <= kUnrollMaxR) {
      kdistances<R, kWave / 2>(k0, k1, lane, two);
    } else {
      kdistances_rt<R>(k0, lane);
      if (two) kdistances_rt<R>(k1, lane);
    }
    kmerge<R, REGS * 2>(k0, k1, lane, two);
  }
}
// sorts the 64*R keys of each list
template <int R> __device__ __forceinline__ void ksort(uint32_t (&k)[R], const int lane) {
  ksort_lanes<R, 2>(k, k, lane, false);
  kmerge<R, 2>(k, k, lane, false);
}
template <int R> __device__ __forceinline__ void ksort2(uint32_t (&k0)[R], uint32_t (&k1)[R], const int lane) {
  ksort_lanes<R, 2>(k0, k1, lane, true);
  kmerge<R, 2>(k0, k1, lane, true);
}

// The 64 largest keys of each list (64*R keys, item = reg*64 + lane), descending, into register 0 -- all that the
// candidate stage reads when k' <= 64.  Every register is sorted across the lanes by itself (compile-time lane
// distances, no LDS), then the registers are merged pairwise: for two descending runs A and B, max(A[i], B[63-i])
// holds the 64 largest of both as a bitonic sequence, which six more compare-exchange steps put in order.  About a
// third of the compare-exchanges of a full sort of 512 keys, and none of them through run-time lane distances.
template <int R>
__device__ __forceinline__ void ktop64_2(uint32_t (&k0)[R], uint32_t (&k1)[R], const int lane) {
#pragma unroll
  for (int a = 0; a < R; ++a) {
    uint32_t x[1] = {k0[a]}, y[1] = {k1[a]};
    ksort2<1>(x, y, lane);
    k0[a] = x[0];
    k1[a] = y[0];
  }
#pragma unroll
  for (int width = R; width > 1; width /= 2) {
#pragma unroll
    for (int a = 0; a < width / 2; ++a) {
      uint32_t x[1] = {max(k0[a], mirrored<kWave>(k0[a + width / 2], lane))};
      uint32_t y[1] = {max(k1[a], mirrored<kWave>(k1[a + width / 2], lane))};
      kdistances<1, kWave / 2>(x, y, lane, true);
      k0[a] = x[0];
      k1[a] = y[0];
    }
  }
}

// The same for the kp <= 32 largest alone, from the few keys that can be among them: of 64 lanes' largest keys the kp-th is a bound that kp keys reach, so
// every key below it is out; what is left (for scores in no particular order about 42 of 512 keys at kp = 32) goes into one register and is
// sorted there.  Two sorts of 64 keys instead of R and the merges: 32768 tokens, 2 x 512 keys, k = 32: 211 -> 165 us.  More than 64 left, or fewer than kp lanes with a key: false, and the keys as they were.
// The way there is a permutation of the lanes (ds_permute_b32) and no LDS: beside the 256 x 256 tile GEMM, whose ring takes all of a CU's, a block with any finds no place.
constexpr int kPruneTop = 32;
// Appends the keys that reach `least` to list[0..n), which has room for them (list: zeros beyond n): in order of lanes, the other lanes' places go round behind them (modulo 64, as
// the instruction takes them) with a zero each
__device__ __forceinline__ void kappend(uint32_t& list, int& n, const uint32_t key, const uint32_t least, const int lane) {
  const uint64_t in = __ballot(key >= least);
  const int count = __popcll(in), mine = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(in >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)in, (uint32_t)n));
  const int to = key >= least ? mine : 2 * n + count + lane - mine;
  list |= (uint32_t)__builtin_amdgcn_ds_permute(to * 4, (int)(key >= least ? key : 0u));
  n += count;
}
template <int R>
__device__ __forceinline__ bool ktop_pruned_2(uint32_t (&k0)[R], uint32_t (&k1)[R], const int kp, const int lane) {
  uint32_t m0[1] = {k0[0]}, m1[1] = {k1[0]};
#pragma unroll
  for (int a = 1; a < R; ++a) {
    m0[0] = max(m0[0], k0[a]);
    m1[0] = max(m1[0], k1[a]);
  }
  ksort2<1>(m0, m1, lane);
  const uint32_t t0 = (uint32_t)__builtin_amdgcn_readlane((int)m0[0], kp - 1), t1 = (uint32_t)__builtin_amdgcn_readlane((int)m1[0], kp - 1);
  int n0 = 0, n1 = 0;
#pragma unroll
  for (int a = 0; a < R; ++a) {
    n0 += __popcll(__ballot(k0[a] >= t0));
    n1 += __popcll(__ballot(k1[a] >= t1));
  }
  if (t0 == 0u || t1 == 0u || n0 > kWave || n1 > kWave) return false;
  uint32_t x[1] = {0u}, y[1] = {0u};
  n0 = n1 = 0;
#pragma unroll
  for (int a = 0; a < R; ++a) {
    kappend(x[0], n0, k0[a], t0, lane);
    kappend(y[0], n1, k1[a], t1, lane);
  }
  ksort2<1>(x, y, lane);
  k0[0] = x[0];
  k1[0] = y[0];
  return true;
}

template <int R>
__device__ __forceinline__ uint32_t sorted_key(const uint32_t (&v)[R], int i) {
  uint32_t r0 = (uint32_t)__shfl((int)v[0], i & 63, kWave);
  if constexpr (R >= 2) {
    const uint32_t r1 = (uint32_t)__shfl((int)v[1], i & 63, kWave);
    r0 = (i >= kWave) ? r1 : r0;
  }
  return r0;
}

// Same selection as select_pairs for bf16 / f16 storage, on packed keys: the tokens of wave `wave` of `num_waves`.  stats: g.stats, or what the
// block merged.
template <int DT, int R, int C>
__device__ __forceinline__ void select_packed(const SelectArgs& g, const int wave, const int num_waves, const float* stats) {
  const int lane = lane_id();
  const int r = g.r, k = g.k, kp = g.kp;

  float rx[R], ry[R];                             // as in select_pairs
  auto load_raw = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < R; ++a) {
      const int key = a * kWave + lane;
      const bool ok = key < r;
      rx[a] = ok ? Elem<DT>::load(g.lx, int64_t(t) * g.row_stride + key) : kNegInf;
      ry[a] = ok ? Elem<DT>::load(g.ly, int64_t(t) * g.row_stride + key) : kNegInf;
    }
  };
  constexpr bool kPrefetch = R <= 2;              // beyond that the extra live registers cost a wave per SIMD
  if (kPrefetch && wave < g.num_tokens) load_raw(wave);
  const NormKeys<R> norm(g, stats, lane);
  int cell[C];
  candidate_cells<R, C>(cell, g, kp, lane);

  for (int t = wave; t < g.num_tokens; t += num_waves) {
    float sx[R], sy[R];
#pragma unroll
    for (int a = 0; a < R; ++a) {
      const int key = a * kWave + lane;
      const bool ok = key < r;
      sx[a] = kPrefetch ? rx[a] : ok ? Elem<DT>::load(g.lx, int64_t(t) * g.row_stride + key) : kNegInf;
      sy[a] = kPrefetch ? ry[a] : ok ? Elem<DT>::load(g.ly, int64_t(t) * g.row_stride + key) : kNegInf;
    }
    if (kPrefetch && t + num_waves < g.num_tokens) load_raw(t + num_waves);
    if (stats || g.run_mean[0]) {
      normalise_half<DT, R>(sx, g, norm, stats, 0, r, lane);
      normalise_half<DT, R>(sy, g, norm, stats, 1, r, lane);
    }
    // (With most keys the sorts' masks are made anew for each token: held from one to the next they are six registers where there are none to spare, kSelectWaves)
    int here = lane;
    if constexpr (R > 8) asm volatile("" : "+v"(here));
    uint32_t kx[R], ky[R];
#pragma unroll
    for (int a = 0; a < R; ++a) {
      const int key = a * kWave + lane;
      kx[a] = key < r ? make_key<DT>(sx[a], key) : 0u;          // 0 sorts behind every real key
      ky[a] = key < r ? make_key<DT>(sy[a], key) : 0u;
    }
    if constexpr (R > kUnrollMaxR) {                             // uniform: kp comes with the arguments
      if (kp > kWave) ksort2<R>(kx, ky, here);
      else if (kp > kPruneTop || !ktop_pruned_2<R>(kx, ky, kp, here)) ktop64_2<R>(kx, ky, here);
    } else {
      ksort2<R>(kx, ky, here);
    }

    uint32_t ck[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const bool ok = cell[c] >= 0;
      const int a = ok ? (cell[c] >> 8) : 0, b = ok ? (cell[c] & 255) : 0;
      const float va = key_score<DT>(sorted_key<R>(kx, a)), vb = key_score<DT>(sorted_key<R>(ky, b));
      ck[c] = ok ? make_key<DT>(Elem<DT>::round(va + vb), cell[c]) : 0u;
    }
    ksort<C>(ck, here);

    constexpr int kOut = (C >= 2) ? 2 : 1;          // k <= 128 -> winners live in regs 0..1
#pragma unroll
    for (int c = 0; c < kOut; ++c) {
      const int j = c * kWave + lane;
      const bool ok = j < k;
      const int pl = ok ? key_payload(ck[c]) : 0;
      const int ia = key_payload(sorted_key<R>(kx, pl >> 8)), ib = key_payload(sorted_key<R>(ky, pl & 255));
      if (ok) {
        const int64_t o = int64_t(t) * k + j;
        const float sc = key_score<DT>(ck[c]);
        if (g.scores) Elem<DT>::store(g.scores, o, sc);
        if (g.gates) Elem<DT>::store(g.gates, o, expf(sc));         // gate = P(x key) * P(y key)
        g.indices[o] = ia * r + ib;
      }
    }
  }
}

static inline int num_cells(int k, int kp) {
  int n = 0;
  for (int a = 0; a < kp; ++a) n += (kp < k / (a + 1)) ? kp : k / (a + 1);
  return n;
}

// Whether the selecting blocks merge the batch statistics: up to 128 KiB of them to a block.  Both sides of the line, the router alone, its own launch / merged in the blocks:
// 64 keys 4096 tokens 18.4 / 17.3 us, 4200 20.6 / 23.1, 5000 21.2 / 23.8, 8000 25.3 / 26.1; 32 keys 8192 27.6 / 25.6, 8300 23.7 / 25.5, 10000 25.1 / 27.1 (each pair on one box).
static inline bool merge_here(int64_t num_tokens, int r) { return r <= kMergeKeys && (num_tokens + kBnRows - 1) / kBnRows * 2 * r <= 16384; }

// What select_packed and its kernels want filled in beside the caller's fields; returns the candidate cells per lane
static inline int prepare_select(SelectArgs& g) {
  g.kp = g.r < g.k ? g.r : g.k;
  for (int a = 0; a < 128; ++a) g.row_cells[a] = a < g.kp ? (uint8_t)(g.kp < g.k / (a + 1) ? g.kp : g.k / (a + 1)) : 0;
  return (num_cells(g.k, g.kp) + kWave - 1) / kWave;            // <= 11 for k <= 128
}

}  // namespace omni
