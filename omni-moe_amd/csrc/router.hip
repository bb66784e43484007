// Cartesian-product router selection for gfx950.
//
// Replaces the reference's two torch.topk launches plus its serial max/argmax
// Triton kernel (omni_moe/ops/triton/omni_router.py:8-95, 167-232).  One 64-lane
// wave owns one token and never leaves registers:
//   1. each half's r scores sit `R` per lane and are sorted descending by a bitonic
//      network (cross-lane exchanges for strides < 64, register exchanges above),
//      ordered by (score desc, key index asc) -- a total order, so ties resolve to
//      the lower key index;
//   2. candidate sums sx[a]+sy[b] are formed in the storage dtype, but only for the
//      cells with (a+1)(b+1) <= k: both half lists are sorted, so a cell (a,b) is
//      preceded by the (a+1)(b+1)-1 cells it is dominated by (each has a score >= its
//      own and a lower position a*k'+b), and cannot be among the first k otherwise.
//      That is 50 cells instead of 256 at k=16, 119 instead of 1024 at k=32;
//   3. the candidates are sorted by (score desc, position asc) with the same
//      network and the first k are written out with id = ix[a]*r + iy[b].
#include "common.h"
#include "omni_moe_hip.h"
#include "select.h"

#include <algorithm>

// defined beside the GEMM kernels: z = x [Wx;Wy]^T, optionally with per-32-row column
// partial statistics (mean, M2) [ceil(T/32)][2r] of the rounded z
int omni_gemm_router_projection(const void* x, const void* wx, const void* wy, void* z, float* part_mean, float* part_m2,
                                int64_t T, int H, int r, int dtype, void* stream, bool exclusive = true);

namespace omni {

template <int R, int C>
__global__ __launch_bounds__(kRouterWaves* kWave) void router_select_kernel(const SelectArgs g) {
  count_batch(g);
  select_pairs<R, C>(g, blockIdx.x * kRouterWaves + (threadIdx.x >> 6), gridDim.x * kRouterWaves, g.stats);
}

// Waves to a SIMD that the registers have to leave room for, where a few more of them would cost one (router of 32768 tokens, hidden 256, 1000 keys a half, top-16: with 169
// registers, two waves, 435 us; with 168, three, 355)
template <int R, int C>
constexpr int kSelectWaves = R == 16 && C <= 4 ? 3 : 1;
template <int DT, int R, int C>
__global__ __launch_bounds__(kRouterWaves* kWave, (kSelectWaves<R, C>)) void router_select_packed_kernel(const SelectArgs g) {
  count_batch(g);
  select_packed<DT, R, C>(g, blockIdx.x * kRouterWaves + (threadIdx.x >> 6), gridDim.x * kRouterWaves, g.stats);
}

// Training: the blocks merge the projection's column statistics themselves, W waves to a block.
template <int DT, int R, int C, int W>
__global__ __launch_bounds__(W* kWave) void router_select_merge_kernel(const SelectArgs g) {
  extern __shared__ __align__(16) float stats[];
  merge_statistics(g, stats, W * kWave);
  count_batch(g);
  select_packed<DT, R, C>(g, blockIdx.x * W + (threadIdx.x >> 6), gridDim.x * W, stats);
}

// More keys per half than a wave's registers hold (r > 1024): 16-bit scores, k' <= 64.  The row is walked in chunks of
// 512 keys per half: each chunk's 64 best (ktop64_2) are merged into the running 64 best by the same max(A[i], B[63-i])
// step.  With the BatchNorm + log-softmax front the row is read three times (maximum, sum of exponentials, keys), each
// time with the arithmetic and the per-lane summation order of normalise_half, so a row gives the bits it would give there.
template <int DT, int C>
__global__ __launch_bounds__(kRouterWaves* kWave) void router_select_chunked_kernel(const SelectArgs g) {
  constexpr int RC = 8, kChunk = RC * kWave;
  count_batch(g);
  const int lane = lane_id();
  const int wave = blockIdx.x * kRouterWaves + (threadIdx.x >> 6);
  const int num_waves = gridDim.x * kRouterWaves;
  const int r = g.r, k = g.k, kp = g.kp;
  const int chunks = (r + kChunk - 1) / kChunk;
  const bool norm = g.stats || g.run_mean[0];
  int cell[C];
  candidate_cells<1, C>(cell, g, kp, lane);

  for (int t = wave; t < g.num_tokens; t += num_waves) {
    const int64_t row = int64_t(t) * g.row_stride;
    float mx[2] = {0.f, 0.f}, lse[2] = {0.f, 0.f};
    if (norm) {
      for (int half = 0; half < 2; ++half) {
        const void* src = half ? g.ly : g.lx;
        float m = kNegInf;
        for (int c = 0; c < chunks; ++c)
#pragma unroll
          for (int a = 0; a < RC; ++a) {
            const int key = c * kChunk + a * kWave + lane;
            if (key < r) m = fmaxf(m, normalise_one<DT>(Elem<DT>::load(src, row + key), g, half, key, r));
          }
        m = wave_max(m);
        float e = 0.f;
        for (int c = 0; c < chunks; ++c)
#pragma unroll
          for (int a = 0; a < RC; ++a) {
            const int key = c * kChunk + a * kWave + lane;
            e += key < r ? expf(normalise_one<DT>(Elem<DT>::load(src, row + key), g, half, key, r) - m) : 0.f;
          }
        mx[half] = m;
        lse[half] = logf(wave_sum(e));
      }
    }
    uint32_t bx = 0u, by = 0u;                      // the 64 best keys so far of each half, descending across the lanes
    for (int c = 0; c < chunks; ++c) {
      uint32_t kx[RC], ky[RC];
#pragma unroll
      for (int a = 0; a < RC; ++a) {
        const int key = c * kChunk + a * kWave + lane;
        const bool ok = key < r;
        float vx = ok ? Elem<DT>::load(g.lx, row + key) : 0.f, vy = ok ? Elem<DT>::load(g.ly, row + key) : 0.f;
        if (norm && ok) {
          vx = Elem<DT>::round(normalise_one<DT>(vx, g, 0, key, r) - mx[0] - lse[0]);
          vy = Elem<DT>::round(normalise_one<DT>(vy, g, 1, key, r) - mx[1] - lse[1]);
        }
        kx[a] = ok ? make_key<DT>(vx, key) : 0u;    // 0 sorts behind every real key
        ky[a] = ok ? make_key<DT>(vy, key) : 0u;
      }
      ktop64_2<RC>(kx, ky, lane);
      uint32_t x[1] = {max(bx, mirrored<kWave>(kx[0], lane))};
      uint32_t y[1] = {max(by, mirrored<kWave>(ky[0], lane))};
      kdistances<1, kWave / 2>(x, y, lane, true);
      bx = c == 0 ? kx[0] : x[0];
      by = c == 0 ? ky[0] : y[0];
    }
    const uint32_t sx[1] = {bx}, sy[1] = {by};

    uint32_t ck[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const bool ok = cell[c] >= 0;
      const int a = ok ? (cell[c] >> 8) : 0, b = ok ? (cell[c] & 255) : 0;
      const float va = key_score<DT>(sorted_key<1>(sx, a)), vb = key_score<DT>(sorted_key<1>(sy, b));
      ck[c] = ok ? make_key<DT>(Elem<DT>::round(va + vb), cell[c]) : 0u;
    }
    ksort<C>(ck, lane);

    constexpr int kOut = (C >= 2) ? 2 : 1;
#pragma unroll
    for (int c = 0; c < kOut; ++c) {
      const int j = c * kWave + lane;
      const bool ok = j < k;
      const int pl = ok ? key_payload(ck[c]) : 0;
      const int ia = key_payload(sorted_key<1>(sx, pl >> 8)), ib = key_payload(sorted_key<1>(sy, pl & 255));
      if (ok) {
        const int64_t o = int64_t(t) * k + j;
        const float sc = key_score<DT>(ck[c]);
        if (g.scores) Elem<DT>::store(g.scores, o, sc);
        if (g.gates) Elem<DT>::store(g.gates, o, expf(sc));
        g.indices[o] = ia * r + ib;
      }
    }
  }
}

template <int C>
static hipError_t launch_select_chunked(const SelectArgs& g, hipStream_t s) {
  int64_t blocks = ((int64_t)g.num_tokens + kRouterWaves - 1) / kRouterWaves;
  if (blocks > 256 * 16) blocks = 256 * 16;
  if (g.dt == kBF16) hipLaunchKernelGGL((router_select_chunked_kernel<kBF16, C>), dim3((unsigned)blocks), dim3(kRouterWaves * kWave), 0, s, g);
  else hipLaunchKernelGGL((router_select_chunked_kernel<kF16, C>), dim3((unsigned)blocks), dim3(kRouterWaves * kWave), 0, s, g);
  return hipGetLastError();
}

// What the select kernels take: r <= 1024 with every dtype and k <= 128; beyond that 16-bit scores with k <= 64.
bool select_covers(int r, int k, int dtype) {
  if (r <= kMaxKeys) return true;
  return r <= kMaxKeysChunked && dtype != kF32 && k <= kWave;
}

template <int R, int C>
static hipError_t launch_select(const SelectArgs& g, hipStream_t s) {
  int64_t blocks = ((int64_t)g.num_tokens + kRouterWaves - 1) / kRouterWaves;
  if (blocks > 256 * 16) blocks = 256 * 16;     // waves loop over tokens beyond that
  if (g.dt == kF32)
    hipLaunchKernelGGL((router_select_kernel<R, C>), dim3((unsigned)blocks), dim3(kRouterWaves * kWave), 0, s, g);
  else if (g.dt == kBF16)
    hipLaunchKernelGGL((router_select_packed_kernel<kBF16, R, C>), dim3((unsigned)blocks), dim3(kRouterWaves * kWave), 0, s, g);
  else
    hipLaunchKernelGGL((router_select_packed_kernel<kF16, R, C>), dim3((unsigned)blocks), dim3(kRouterWaves * kWave), 0, s, g);
  return hipGetLastError();
}

template <int R>
static hipError_t select_by_cells(int cpl, const SelectArgs& g, hipStream_t s) {
  if (cpl <= 1) return launch_select<R, 1>(g, s);
  if (cpl <= 2) return launch_select<R, 2>(g, s);
  if (cpl <= 4) return launch_select<R, 4>(g, s);
  if (cpl <= 8) return launch_select<R, 8>(g, s);
  return launch_select<R, 16>(g, s);
}

static int select_dispatch(SelectArgs g, hipStream_t s) {
  const int cpl = prepare_select(g);
  const int rpl = (g.r + kWave - 1) / kWave;
  hipError_t err;
  if (rpl <= 1) err = select_by_cells<1>(cpl, g, s);
  else if (rpl <= 2) err = select_by_cells<2>(cpl, g, s);
  else if (rpl <= 4) err = select_by_cells<4>(cpl, g, s);
  else if (rpl <= 8) err = select_by_cells<8>(cpl, g, s);
  else if (rpl <= 16) err = select_by_cells<16>(cpl, g, s);
  else if (!select_covers(g.r, g.k, g.dt)) return OMNI_ERR_UNSUPPORTED;   // the entry points refuse it before anything is enqueued
  else if (cpl <= 1) err = launch_select_chunked<1>(g, s);
  else if (cpl <= 2) err = launch_select_chunked<2>(g, s);
  else if (cpl <= 4) err = launch_select_chunked<4>(g, s);
  else err = launch_select_chunked<8>(g, s);                // k <= 64: at most 280 cells
  return err == hipSuccess ? OMNI_OK : OMNI_ERR_HIP_BASE + (int)err;
}

static int merge_cells(int r, int k) { return (num_cells(k, r < k ? r : k) + kWave - 1) / kWave; }      // candidates per lane
template <int W>
static hipError_t launch_select_merge(SelectArgs g, hipStream_t s) {
  const int cpl = prepare_select(g);
  const int64_t blocks = std::min<int64_t>(((int64_t)g.num_tokens + W - 1) / W, 256 * 16 / W);
  auto start = [&](auto cells) {
    constexpr int C = decltype(cells)::value;
    const int bytes = 4 * merge_lds_floats(g.r, W * kWave);
    if (g.dt == kBF16) hipLaunchKernelGGL((router_select_merge_kernel<kBF16, 1, C, W>), dim3((unsigned)blocks), dim3(W * kWave), bytes, s, g);
    else hipLaunchKernelGGL((router_select_merge_kernel<kF16, 1, C, W>), dim3((unsigned)blocks), dim3(W * kWave), bytes, s, g);
    return hipGetLastError();
  };
  return cpl <= 1 ? start(std::integral_constant<int, 1>{}) : start(std::integral_constant<int, 2>{});
}

// ---- BatchNorm1d(affine=False) statistics over the T rows of z [T, C] -------------------
struct BnFinalArgs {
  const float* part_mean;   // [strips][2r] (training)
  const float* part_m2;
  float* stats;             // [4][r]: mean_x, rstd_x, mean_y, rstd_y
  void* running_mean[2];    // [r] each, dtype stat_dt; read in eval, updated in training
  void* running_var[2];
  int64_t* num_batches_tracked[2];   // may be NULL; read for the cumulative average (momentum < 0)
  int num_rows, r, strips, training, stat_dt;
  int count_here;                    // increment num_batches_tracked in this kernel (no select kernel follows; momentum >= 0 only)
  float momentum, eps;               // momentum < 0: cumulative moving average, factor 1 / (batches tracked so far + 1)
  int parts;                         // 0, or the parts of merge_statistics whose order of the sums is taken
};

__device__ __forceinline__ double of_lane(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane), __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// A column's sums in the order of merge_statistics: part p over the strips p, p + parts, ..., then part after part.  Every lane ends with them.
// (A lane to a part, where the 64 folded sums use all lanes; eight strips requested ahead make up for it: two-stream layer of hidden 1024 x 4096, 4096 tokens x 64 keys
// 123.4 us with the folded sums, 123.1 with these, 8192 x 32 keys 211.9 / 212.0.  Strips one after the other: 120.8 / 124.3 at 4096.)
__device__ __forceinline__ ColumnSums sums_by_parts(const BnFinalArgs& g, const int col) {
  const int lane = lane_id();
  ColumnSums all{0., 0.};
  for (int p0 = 0; p0 < g.parts; p0 += kWave) {
    ColumnSums c{0., 0.};
    if (p0 + lane < g.parts)
      for (int first = p0 + lane; first < g.strips; first += 8 * g.parts) add_batch<8>(c, g.part_mean, g.part_m2, first, g.parts, g.strips, 2 * g.r, col, g.num_rows);
    for (int q = 0; q < min(kWave, g.parts - p0); ++q) {
      all.weighted += of_lane(c.weighted, q);
      all.squares += of_lane(c.squares, q);
    }
  }
  return all;
}

// One wave per column: merges the strip partials, writes mean and 1/sqrt(var+eps), and in
// training moves the running buffers (unbiased variance) as nn.BatchNorm1d does.  In eval
// the running buffers provide mean and variance.
__global__ __launch_bounds__(256) void bn_finalize_kernel(const BnFinalArgs g) {
  const int col = blockIdx.x * (256 / kWave) + (threadIdx.x >> 6), lane = lane_id();
  if (col == 0 && lane == 0 && g.training && g.count_here) {
    if (g.num_batches_tracked[0]) *g.num_batches_tracked[0] += 1;
    if (g.num_batches_tracked[1]) *g.num_batches_tracked[1] += 1;
  }
  if (col >= 2 * g.r) return;
  const int half = col >= g.r, key = col - half * g.r;
  float mean, var;
  if (g.training) {
    // the running buffers (and the batch count) are requested first: their latency passes beside the strips'
    const float rm = load_score(g.running_mean[half], key, g.stat_dt), rv = load_score(g.running_var[half], key, g.stat_dt);
    const float f = g.momentum >= 0.f ? g.momentum : 1.0f / (float)(*g.num_batches_tracked[half] + 1);
    ColumnSums c{0., 0.};
    if (g.parts) {
      c = sums_by_parts(g, col);
    } else {
      for (int strip = lane; strip < g.strips; strip += kWave) add_strip(c, g.part_mean, g.part_m2, strip, 2 * g.r, col, g.num_rows);
#pragma unroll
      for (int m = kWave / 2; m >= 1; m >>= 1) {
        const double o0 = __shfl_xor(c.weighted, m, kWave), o1 = __shfl_xor(c.squares, m, kWave);
        c.weighted += o0;
        c.squares += o1;
      }
    }
    const ColumnStats v = column_stats(c, g.num_rows);
    mean = v.mean;
    var = v.var;
    if (lane == 0) {
      // nn.BatchNorm1d(momentum=None): the factor f is 1 / num_batches_tracked AFTER this batch has been counted
      store_score(g.running_mean[half], key, (1.f - f) * rm + f * mean, g.stat_dt);
      store_score(g.running_var[half], key, (1.f - f) * rv + f * v.unbiased, g.stat_dt);
    }
  } else {
    mean = load_score(g.running_mean[half], key, g.stat_dt);
    var = load_score(g.running_var[half], key, g.stat_dt);
  }
  if (lane == 0) {
    g.stats[(2 * half) * g.r + key] = mean;
    g.stats[(2 * half + 1) * g.r + key] = rstd_of(var, g.eps);
  }
}

// The selection for the layer call, which fills the arguments itself; with column statistics in them the launch that merges those in front of it
int launch_router_select(const SelectArgs& args, hipStream_t s) {
  SelectArgs g = args;
  if (g.part_mean) {
    const BnFinalArgs b{g.part_mean, g.part_m2, g.stats_out, {(void*)g.run_mean[0], (void*)g.run_mean[1]}, {(void*)g.run_var[0], (void*)g.run_var[1]},
                        {g.count_batch[0], g.count_batch[1]}, g.num_tokens, g.r, g.strips, 1, g.stat_dt, 0, g.momentum, g.eps};
    hipLaunchKernelGGL(bn_finalize_kernel, dim3((2 * g.r + 3) / 4), dim3(256), 0, s, b);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return OMNI_ERR_HIP_BASE + (int)e;
    g.stats = g.stats_out;
    g.part_mean = g.part_m2 = nullptr;
  }
  return select_dispatch(g, s);
}

static inline size_t align256(size_t v) { return (v + 255) / 256 * 256; }

}  // namespace omni

extern "C" OMNI_API int32_t omni_router_select(const void* logits_x, const void* logits_y, void* scores, int32_t* indices,
                                               int64_t num_tokens, int32_t num_expert_sqrt, int32_t num_experts_per_token,
                                               int32_t dtype, void* stream) {
  using namespace omni;
  const int r = num_expert_sqrt, k = num_experts_per_token;
  if (num_tokens < 0 || num_tokens > INT32_MAX / 256 || r <= 0) return OMNI_ERR_SHAPE;
  if (k < 0 || (int64_t)k > (int64_t)r * r || k > 128 || (k & 1)) return OMNI_ERR_TOPK;
  if (dtype != OMNI_BF16 && dtype != OMNI_F16 && dtype != OMNI_F32) return OMNI_ERR_DTYPE;
  if (num_tokens == 0 || k == 0) return OMNI_OK;
  if (!logits_x || !logits_y || !scores || !indices) return OMNI_ERR_NULL;
  if (!select_covers(r, k, dtype)) return OMNI_ERR_UNSUPPORTED;
  SelectArgs g{};
  g.lx = logits_x; g.ly = logits_y; g.row_stride = r; g.scores = scores; g.indices = indices;
  g.num_tokens = (int)num_tokens; g.r = r; g.k = k; g.dt = dtype;
  return select_dispatch(g, (hipStream_t)stream);
}

// workspace layout of omni_router_fwd: z [T,2r] | stats [4r] f32 | part_mean | part_m2
extern "C" OMNI_API size_t omni_router_workspace_bytes(int64_t num_tokens, int32_t num_expert_sqrt, int32_t dtype) {
  using namespace omni;
  if (num_tokens < 0 || num_expert_sqrt <= 0) return 0;
  const size_t es = dtype == OMNI_F32 ? 4 : 2, r = (size_t)num_expert_sqrt;
  const size_t strips = ((size_t)num_tokens + kBnRows - 1) / kBnRows;
  return align256((size_t)num_tokens * 2 * r * es) + align256(4 * r * 4) + 2 * align256(strips * 2 * r * 4);
}

// After omni_router_fwd the workspace still holds what a backward pass needs: z at offset 0 and,
// at this offset, the fp32 statistics [mean_x | rstd_x | mean_y | rstd_y], r values each.
extern "C" OMNI_API size_t omni_router_workspace_stats_offset(int64_t num_tokens, int32_t num_expert_sqrt, int32_t dtype) {
  using namespace omni;
  if (num_tokens < 0 || num_expert_sqrt <= 0) return 0;
  const size_t es = dtype == OMNI_F32 ? 4 : 2;
  return align256((size_t)num_tokens * 2 * (size_t)num_expert_sqrt * es);
}

namespace omni {
// exclusive: nothing is meant to run beside the call.  order_threads: 0, or the block size of the joint launches whose order the batch statistics' sums take
int router_fwd(const void* x, const void* weight_x, const void* weight_y,
               void* running_mean_x, void* running_var_x, int64_t* num_batches_tracked_x,
               void* running_mean_y, void* running_var_y, int64_t* num_batches_tracked_y,
               int32_t training, float momentum, float eps, void* gates, int32_t* indices,
               void* scores, int64_t num_tokens, int32_t hidden_size, int32_t num_expert_sqrt,
               int32_t num_experts_per_token, int32_t dtype, int32_t stats_dtype,
               void* workspace, void* stream, bool exclusive, int order_threads) {
  const int r = num_expert_sqrt, k = num_experts_per_token;
  if (num_tokens < 0 || num_tokens > INT32_MAX / 256 || r <= 0 || hidden_size <= 0) return OMNI_ERR_SHAPE;
  if (k < 0 || (int64_t)k > (int64_t)r * r || k > 128 || (k & 1)) return OMNI_ERR_TOPK;
  if (dtype != OMNI_BF16 && dtype != OMNI_F16 && dtype != OMNI_F32) return OMNI_ERR_DTYPE;
  if (stats_dtype != OMNI_BF16 && stats_dtype != OMNI_F16 && stats_dtype != OMNI_F32) return OMNI_ERR_DTYPE;
  if (num_tokens == 0) return OMNI_OK;
  if (training && num_tokens == 1) return OMNI_ERR_SHAPE;   // batch statistics of one sample: nn.BatchNorm1d raises
  if (!x || !weight_x || !weight_y || !running_mean_x || !running_var_x || !running_mean_y || !running_var_y) return OMNI_ERR_NULL;
  if (training && momentum < 0.f && (!num_batches_tracked_x || !num_batches_tracked_y)) return OMNI_ERR_NULL;   // the cumulative average needs the counts
  if (training && momentum < 0.f && k == 0) return OMNI_ERR_UNSUPPORTED;
  if (k > 0 && !select_covers(r, k, dtype)) return OMNI_ERR_UNSUPPORTED;   // the select kernels' limit, checked before the projection is enqueued
  if (k > 0 && (!gates || !indices)) return OMNI_ERR_NULL;
  if (!workspace) return OMNI_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  const size_t strips = ((size_t)num_tokens + kBnRows - 1) / kBnRows;
  char* w = (char*)workspace;
  const size_t es = dtype == OMNI_F32 ? 4 : 2;
  void* z = w;                       w += align256((size_t)num_tokens * 2 * r * es);
  float* stats = (float*)w;          w += align256((size_t)4 * r * 4);
  float* part_mean = (float*)w;      w += align256(strips * 2 * r * 4);
  float* part_m2 = (float*)w;

  // z = x [Wx;Wy]^T on the matrix cores
  // (in training its epilogue also leaves the per-32-row column statistics)
  if (int e = omni_gemm_router_projection(x, weight_x, weight_y, z, training ? part_mean : nullptr, training ? part_m2 : nullptr,
                                          num_tokens, hidden_size, r, dtype, stream, exclusive)) return e;
  // Training, up to 64 keys per half and 128 KiB of partial statistics: the selecting blocks merge them themselves.  16 waves to a block beyond 2048 tokens (as many
  // merges as CUs), 8 below (more CUs).  Whole call in three launches / two, top-16 and 64 keys: 1024 tokens 15.0 -> 13.7 us, 2048 15.7 -> 14.4 (16 waves 15.9), 4096
  // 18.4 -> 17.3 (8 waves 18.5); 32 keys: 256 13.3 -> 11.8, 8192 27.6 -> 25.6.  More keys: 2048 x 100 17.8 -> 23-30, 1500 x 128 21 -> 28-30.  Beside another stream's
  // kernels, which hide the launch, whole blocks of 16 waves would wait for a CU: there it stays, and takes the blocks' order of the sums, so that the sizes
  // alone give the bits.
  const bool block_order = training && k > 0 && dtype != OMNI_F32 && r <= kWave && merge_here(num_tokens, r) && merge_cells(r, k) <= 2, merge = block_order && exclusive;
  const int merge_waves = num_tokens > 2048 ? 16 : 8;
  SelectArgs g{};
  g.lx = z; g.ly = (const char*)z + (size_t)r * es; g.row_stride = 2 * r;
  g.scores = scores; g.gates = gates; g.indices = indices;
  g.num_tokens = (int)num_tokens; g.r = r; g.k = k; g.dt = dtype;
  if (!training || merge) {
    g.run_mean[0] = running_mean_x; g.run_mean[1] = running_mean_y;
    g.run_var[0] = running_var_x; g.run_var[1] = running_var_y;
    g.stats_out = stats; g.stat_dt = stats_dtype; g.eps = eps;
  }
  if (training) {
    g.count_batch[0] = num_batches_tracked_x; g.count_batch[1] = num_batches_tracked_y;
  }
  if (merge) {
    g.part_mean = part_mean; g.part_m2 = part_m2; g.strips = (int)strips; g.momentum = momentum;
    const hipError_t err = merge_waves == 16 ? launch_select_merge<16>(g, s) : launch_select_merge<8>(g, s);
    return err == hipSuccess ? OMNI_OK : OMNI_ERR_HIP_BASE + (int)err;
  }
  // Training: one more launch merges the partial statistics and moves the running buffers.  In eval mode the
  // select kernel reads the running buffers itself (and leaves mean and 1/sqrt(var + eps) in `stats`).
  if (training || k == 0) {
    BnFinalArgs b{part_mean, part_m2, stats, {running_mean_x, running_mean_y}, {running_var_x, running_var_y},
                  {num_batches_tracked_x, num_batches_tracked_y}, (int)num_tokens, r, (int)strips, training ? 1 : 0, stats_dtype,
                  k == 0 ? 1 : 0, momentum, eps, order_threads ? merge_parts(r, order_threads) : block_order ? merge_parts(r, merge_waves * kWave) : 0};
    hipLaunchKernelGGL(bn_finalize_kernel, dim3((2 * r + 3) / 4), dim3(256), 0, s, b);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return OMNI_ERR_HIP_BASE + (int)err;
    if (k == 0) return OMNI_OK;
  }
  if (training) g.stats = stats;
  return select_dispatch(g, s);
}
}  // namespace omni

extern "C" OMNI_API int32_t omni_router_fwd(const void* x, const void* weight_x, const void* weight_y,
                                            void* running_mean_x, void* running_var_x, int64_t* num_batches_tracked_x,
                                            void* running_mean_y, void* running_var_y, int64_t* num_batches_tracked_y,
                                            int32_t training, float momentum, float eps, void* gates, int32_t* indices,
                                            void* scores, int64_t num_tokens, int32_t hidden_size, int32_t num_expert_sqrt,
                                            int32_t num_experts_per_token, int32_t dtype, int32_t stats_dtype,
                                            void* workspace, void* stream) {
  return omni::router_fwd(x, weight_x, weight_y, running_mean_x, running_var_x, num_batches_tracked_x, running_mean_y, running_var_y, num_batches_tracked_y, training, momentum, eps,
                          gates, indices, scores, num_tokens, hidden_size, num_expert_sqrt, num_experts_per_token, dtype, stats_dtype, workspace, stream, true, 0);
}
