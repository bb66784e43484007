// Backward kernels of the three OmniMoE operators for gfx950, so that a layer built on them
// trains.  Each replaces the matching Triton backward of the reference:
//   * router   (omni_moe/ops/triton/omni_router.py:98-164, 235-274): the gradient of the k
//     selected scores scatters back to the two half-logit rows, d_lx[ix] += ds, d_ly[iy] += ds;
//   * experts  (omni_expert.py:375-618, 1067-1277): for a pair (t, e) with s = <x_t, U_e>,
//     a = <dy_t, V_e>:   dg = a silu(s),   ds = a g silu'(s),   dx_t += ds U_e,
//     dU_e += ds x_t,   dV_e += silu(s) g dy_t;
//   * SwiGLU   (omni_mlp.py:102-177 forward, 180-249 backward) as element-wise kernels for
//     the training path, which keeps gate and up (the inference path forms the product in the
//     GEMM epilogue and never stores them).
// All sums are fp32 in a fixed order, rounded once on the way out: no atomics anywhere (the
// reference accumulates dx, dU and dV with atomics in the storage dtype), so gradients are
// run-to-run identical.
//
// Expert backward in two passes.  Token pass: forms dx and dg and, in an fp32 workspace, ds and the forward coefficient silu(s) g of
// every pair, in the organisation that the forward takes at the sizes: gather (one wave owns one token, keeps x_t, dy_t and the fp32 dx
// accumulator in registers and fetches each selected up and down row once) or split (the rows in eight column slices, one to an XCD).
// split takes s from the forward where that kept it; gather, which has the up rows in hand for dx, and split without it form it again.  Weight pass: the pairs are grouped by expert with the
// stable schedule of the forward path; a wave owns a chunk of that list for one part of the columns and
// gathers the parts of its tokens' x or dy rows; long segments, which several waves share, are added by a fix-up, so every dU/dV row
// is written exactly once (zeros for experts nobody selected).
#include "common.h"
#include "expert_split.h"
#include "omni_moe_hip.h"
#include "rows.h"
#include "schedule.h"

namespace omni {

constexpr int kBwdWavesPerBlock = 4;

// ---- router ------------------------------------------------------------------------------------
// One wave per token; lane l accumulates columns l, l+64, ... of both halves (r <= 64 * kCols).
template <int DT, int kCols>
__global__ __launch_bounds__(kBwdWavesPerBlock* kWave) void router_bwd_kernel(
    const void* __restrict__ dscores, const int32_t* __restrict__ ids, void* __restrict__ dlx, void* __restrict__ dly,
    int num_tokens, int r, int top_k) {
  const int lane = lane_id();
  const int t = __builtin_amdgcn_readfirstlane(blockIdx.x * kBwdWavesPerBlock + (threadIdx.x >> 6));
  if (t >= num_tokens) return;
  float ax[kCols], ay[kCols];
#pragma unroll
  for (int c = 0; c < kCols; ++c) ax[c] = ay[c] = 0.f;
  const int64_t base = int64_t(t) * top_k;
  for (int j0 = 0; j0 < top_k; j0 += kWave) {       // k <= 128: at most two rounds
    const int j = j0 + lane;
    const int my_id = j < top_k ? ids[base + j] : -1;
    const float my_ds = j < top_k ? Elem<DT>::load(dscores, base + j) : 0.f;
    // lane j splits slot j's id once; an id outside the product gets coordinates no lane owns
    const bool ok = (uint32_t)my_id < (uint32_t)r * (uint32_t)r;
    const int my_ix = ok ? my_id / r : -1, my_iy = ok ? my_id - my_ix * r : -1;
    const int n = min(kWave, top_k - j0);
    for (int i = 0; i < n; ++i) {                   // slot order: the sum per column is deterministic
      const int ix = __builtin_amdgcn_readlane(my_ix, i), iy = __builtin_amdgcn_readlane(my_iy, i);
      const float ds = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_ds), i));
#pragma unroll
      for (int c = 0; c < kCols; ++c) {
        ax[c] += (ix == c * kWave + lane) ? ds : 0.f;
        ay[c] += (iy == c * kWave + lane) ? ds : 0.f;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < kCols; ++c) {
    const int col = c * kWave + lane;
    if (col < r) {
      Elem<DT>::store(dlx, int64_t(t) * r + col, ax[c]);
      Elem<DT>::store(dly, int64_t(t) * r + col, ay[c]);
    }
  }
}

// ---- router stage: exp, Cartesian select, log-softmax and BatchNorm in reverse -------------------
// The layer's router forward (omni_moe.py:70-86) is  z = x W^T -> n = BN(z) -> l = log_softmax(n)
// -> scores = lx[ix] + ly[iy] -> gates = exp(scores).  Given d(gates), this pass returns d(z); the
// two GEMMs around it (dW = dz^T x, dx = dz W) are the caller's.  One wave owns a token and walks
// both halves with lane = column (R columns per lane and half):
//   d(score_j) = d(gate_j) gate_j;  d(l) = scatter of d(score) by (ix, iy), in slot order;
//   d(n) = d(l) - exp(l) sum(d(l));                      (log-softmax)
//   eval:  d(z) = rstd d(n);   train:  d(z) = rstd (d(n) - mean_T d(n) - nhat mean_T(d(n) nhat)).
// Training needs the two column means over all tokens: the first kernel leaves d(n) in the dz
// buffer and per-block column sums, a one-wave-per-column kernel adds those, a third kernel
// finishes d(z).  Values are rounded to the storage dtype where the reference's torch ops round
// (d(score), d(l), d(n), d(z)); n and l are recomputed from z and the saved statistics.
//
// A token's k slots are walked one after the other (a fixed order of the sums), each slot's id and gradient handed to all lanes by
// v_readlane; what bounds the pass is that chain, so a wave takes few tokens while there are waves to spare (4096 tokens, 64 keys, k = 16:
// eight tokens a wave and ds_bpermute exchanges 29 us).
// Two launches in training: the blocks that finish d(z) add the column sums of their 64 columns themselves, 512 bytes from each block of the first launch, of
// which there are few (4096 tokens: 256).  Neither reads what the experts' weight pass leaves, so the layer's backward puts the first
// beside that pass and the second beside its fix-up.
static inline int norm_tokens_per_wave(int64_t num_tokens) {
  const int64_t t = num_tokens / (kBwdWavesPerBlock * 512);
  return (int)(t < 1 ? 1 : t > 8 ? 8 : t);
}
struct RouterPass {
  const void *dgates, *gates;
  const int32_t* ids;
  const void* z;
  const float* stats;
  void* dz;
  float* partials;                   // training: column sums [block][S1x, S2x, S1y, S2y][r]
  int num_tokens, r, top_k, training, tokens_per_wave, dz_half;
};
// waves of a block: eight, or four where a lane has more than four columns of each half (the sums' LDS).  Sixteen put them on half as many CUs: fix-up and
// router's first launch 13.9 us at 4096 tokens, eight 12.2
constexpr int norm_waves(int cols) { return cols <= 4 ? 8 : kBwdWavesPerBlock; }

template <int DT, int R>
__device__ __forceinline__ void router_norm_bwd_block(const RouterPass& p, const int block) {
  constexpr int W = norm_waves(R);
  __shared__ float red[W][4][R * kWave];                       // per wave: S1x, S2x, S1y, S2y by column
  const int lane = lane_id(), wave = threadIdx.x >> 6, r = p.r;
  const int first = __builtin_amdgcn_readfirstlane((block * W + wave) * p.tokens_per_wave);
  float s1[2][R], s2[2][R];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int a = 0; a < R; ++a) s1[h][a] = s2[h][a] = 0.f;
  float mean[2][R], rstd[2][R];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int a = 0; a < R; ++a) {
      const int key = a * kWave + lane;
      mean[h][a] = key < r ? p.stats[(2 * h) * r + key] : 0.f;
      rstd[h][a] = key < r ? p.stats[(2 * h + 1) * r + key] : 0.f;
    }
  // What a token's sums start from, requested ahead of the one before it: the chain of slots then waits for memory once
  float zv[2][R], my_dg, my_gate;
  int my_slot;
  auto request = [&](int t) __attribute__((always_inline)) {
    const int j = min(lane, p.top_k - 1);
    const int64_t base = int64_t(t) * p.top_k;
    my_slot = p.top_k ? p.ids[base + j] : -1;
    my_dg = p.top_k ? Elem<DT>::load(p.dgates, base + j) : 0.f;
    my_gate = p.top_k ? Elem<DT>::load(p.gates, base + j) : 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int a = 0; a < R; ++a) zv[h][a] = Elem<DT>::load(p.z, int64_t(t) * 2 * r + h * r + min(a * kWave + lane, r - 1));
  };
  const int last = min(first + p.tokens_per_wave, p.num_tokens);
  if (first < last) request(first);
  for (int t = first; t < last; ++t) {
    float zt[2][R];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int a = 0; a < R; ++a) zt[h][a] = zv[h][a];
    int slot = my_slot;
    float dg = my_dg, gate = my_gate;
    if (t + 1 < last) request(t + 1);
    // d(l): scatter of the slot gradients, fp32 sums in slot order, one rounding
    float dl[2][R];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int a = 0; a < R; ++a) dl[h][a] = 0.f;
    for (int j0 = 0; j0 < p.top_k; j0 += kWave) {
      if (j0 > 0) {                                             // k <= 128: a second round
        const int64_t at = int64_t(t) * p.top_k + min(j0 + lane, p.top_k - 1);
        slot = p.ids[at];
        dg = Elem<DT>::load(p.dgates, at);
        gate = Elem<DT>::load(p.gates, at);
      }
      const float my_ds = Elem<DT>::round(dg * gate);
      const bool ok = j0 + lane < p.top_k && (uint32_t)slot < (uint32_t)r * (uint32_t)r;
      const int my_ix = ok ? slot / r : -1, my_iy = ok ? slot - my_ix * r : -1;
      const int n = min(kWave, p.top_k - j0);
      for (int i = 0; i < n; ++i) {
        const int ix = __builtin_amdgcn_readlane(my_ix, i), iy = __builtin_amdgcn_readlane(my_iy, i);
        const float ds = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_ds), i));
#pragma unroll
        for (int a = 0; a < R; ++a) {
          dl[0][a] += (ix == a * kWave + lane) ? ds : 0.f;
          dl[1][a] += (iy == a * kWave + lane) ? ds : 0.f;
        }
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // recompute nhat (fp32), n = round(nhat), l = round(log_softmax(n))
      float nhat[R], l[R];
      float m = -INFINITY;
#pragma unroll
      for (int a = 0; a < R; ++a) {
        const int key = a * kWave + lane;
        nhat[a] = (zt[h][a] - mean[h][a]) * rstd[h][a];
        l[a] = key < r ? Elem<DT>::round(nhat[a]) : -INFINITY;
        m = fmaxf(m, l[a]);
      }
      m = wave_max(m);
      float e = 0.f;
#pragma unroll
      for (int a = 0; a < R; ++a) e += (a * kWave + lane < r) ? expf(l[a] - m) : 0.f;
      const float lse = logf(wave_sum(e));
      float sum_dl = 0.f;
#pragma unroll
      for (int a = 0; a < R; ++a) {
        dl[h][a] = Elem<DT>::round(dl[h][a]);
        sum_dl += dl[h][a];
      }
      sum_dl = wave_sum(sum_dl);
#pragma unroll
      for (int a = 0; a < R; ++a) {
        const int key = a * kWave + lane;
        if (key >= r) {
          if (key < p.dz_half) Elem<DT>::store(p.dz, (int64_t(t) * 2 + h) * p.dz_half + key, 0.f);
          continue;
        }
        const float prob = expf(Elem<DT>::round(l[a] - m - lse));
        const float dn = Elem<DT>::round(dl[h][a] - prob * sum_dl);
        s1[h][a] += dn;
        s2[h][a] += dn * nhat[a];
        Elem<DT>::store(p.dz, (int64_t(t) * 2 + h) * p.dz_half + key, p.training ? dn : dn * rstd[h][a]);
      }
    }
  }
  if (!p.training) return;
  // column sums of the block: waves in order through LDS, then one row of partials per block
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int a = 0; a < R; ++a) {
      red[wave][2 * h][a * kWave + lane] = s1[h][a];
      red[wave][2 * h + 1][a * kWave + lane] = s2[h][a];
    }
  __syncthreads();
  for (int i = threadIdx.x; i < 4 * R * kWave; i += W * kWave) {
    const int q = i / (R * kWave), col = i % (R * kWave);
    if (col >= r) continue;
    float acc = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) acc += red[w][q][col];
    p.partials[(int64_t(block) * 4 + q) * r + col] = acc;
  }
}
template <int DT, int R>
__global__ __launch_bounds__(norm_waves(R)* kWave) void router_norm_bwd_kernel(const RouterPass p) {
  router_norm_bwd_block<DT, R>(p, (int)blockIdx.x);
}

// dz = rstd (dn - mean(dn) - nhat mean(dn nhat)); dn is read from dz.  Blocks alternate between the groups of 64 columns of a half; a block adds its columns'
// sums over the `rows` partials in double, sixteen waves side by side, while its first tokens' values are on their way.
constexpr int kFinishWaves = 16, kFinishRows = 4;               // tokens that a wave has in flight
template <int DT>
__device__ __forceinline__ void router_norm_bwd_finish_block(const RouterPass& p, const int rows, const int block, const int blocks) {
  __shared__ double sums[2][kFinishWaves][kWave];
  __shared__ float means[2][kWave];
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = p.r, per_half = (r + kWave - 1) / kWave, groups = 2 * per_half;
  const int group = block % groups, part = block / groups, parts = blocks / groups;
  const int h = group / per_half, col = (group - h * per_half) * kWave + lane, key = min(col, r - 1);
  const bool live = col < r;
  float zv[kFinishRows], dn[kFinishRows];
  auto at = [&](int t) __attribute__((always_inline)) { return ((int64_t)t * 2 + h) * p.dz_half + key; };
  auto request = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kFinishRows; ++i) {
      const int t = min(t0 + i * kFinishWaves, p.num_tokens - 1);
      zv[i] = Elem<DT>::load(p.z, ((int64_t)t * 2 + h) * r + key);
      dn[i] = Elem<DT>::load(p.dz, at(t));
    }
  };
  constexpr int kStep = kFinishWaves * kFinishRows;
  request(part * kStep + wave);
  const float mu = p.stats[(2 * h) * r + key], rs = p.stats[(2 * h + 1) * r + key];
  double a1 = 0., a2 = 0.;
#pragma unroll 4
  for (int b = wave; b < rows; b += kFinishWaves) {
    const float* row = p.partials + ((int64_t)b * 4 + 2 * h) * r + key;
    a1 += (double)row[0];
    a2 += (double)row[r];
  }
  sums[0][wave][lane] = a1;
  sums[1][wave][lane] = a2;
  __syncthreads();
  if (wave < 2) {
    double acc = 0.;
#pragma unroll
    for (int w = 0; w < kFinishWaves; ++w) acc += sums[wave][w][lane];
    means[wave][lane] = (float)(acc / (double)p.num_tokens);
  }
  __syncthreads();
  const float m1 = means[0][lane], m2 = means[1][lane];
  for (int t0 = part * kStep + wave; t0 < p.num_tokens; t0 += parts * kStep) {
    if (t0 != part * kStep + wave) request(t0);
#pragma unroll
    for (int i = 0; i < kFinishRows; ++i) {
      const int t = t0 + i * kFinishWaves;
      if (live && t < p.num_tokens) Elem<DT>::store(p.dz, at(t), rs * (dn[i] - m1 - (zv[i] - mu) * rs * m2));
    }
  }
}
template <int DT>
__global__ __launch_bounds__(kFinishWaves* kWave) void router_norm_bwd_finish_kernel(const RouterPass p, const int rows) {
  router_norm_bwd_finish_block<DT>(p, rows, (int)blockIdx.x, (int)gridDim.x);
}

// ---- experts, token pass -----------------------------------------------------------------------
// Both organisations are bound as the forward's are: gather by the rows' trip over the fabric, split on the chip, by loads and arithmetic on rows that an XCD's
// L2 holds; split needs the sums over the slices in between, so the forward keeps its <x, U> (4 bytes a pair) and only <dy, V> is formed here.
// The sort of the pairs, which only the weight pass needs, runs beside: the token pass comes in two launches whose first blocks sort, the count
// pass beside the first and the scatter pass beside the second.  All blocks have the sort's threads.
// Sort and token pass, hidden 1024, bf16: 4096 tokens x 16 over 4096 experts 13 + 40 us (gather) -> 11 + 17.5, 1024 x 32 over 16384 18 + 30 -> 7.5 + 15.5.
constexpr int kTokenWaves = kSortWaves;
enum : int { kSortNone = 0, kSortCount = 1, kSortScatter = 2 };
struct SortShare { SortPass pass; int kind, blocks; };          // blocks: a multiple of 8, so that block % 8 names the slice of the others too
__device__ __forceinline__ bool sort_share(const SortShare& s, uint8_t* lds) {       // false: the block is not one of them
  if ((int)blockIdx.x >= s.blocks) return false;
  if (s.kind == kSortScatter) sort_scatter_block(s.pass, (int)blockIdx.x, (int32_t*)lds);
  else if ((int)blockIdx.x < s.pass.tiles) sort_count_block(s.pass, (int)blockIdx.x, (int32_t*)lds);
  return true;
}

struct TokenPass {
  const uint8_t *x, *dy, *up, *down;
  const void* gates;
  const int32_t* ids;
  const float* scores;               // split: NULL: recompute
  uint8_t* dx;
  void* dgates;
  float *ds, *coef;                  // [tokens][top_k]
  float *partial_a, *partial_s;      // split: [slices][tokens][top_k], partial_s without scores only
  int first, last, num_tokens, hidden, top_k;      // gather: the tokens of this launch
  int lanes, slices;                 // split: 16-byte lanes of a row slice, and slices; 0, 0: gather
  uint32_t num_experts;
};
struct PairGrad { float dg, ds, coef; };
__device__ __forceinline__ PairGrad pair_grad(float s, float a, float g) {
  const float sig = sigmoid_f32(s), silu = s * sig, dsilu = sig + silu * (1.0f - sig);
  return {a * silu, a * g * dsilu, silu * g};
}

template <int DT, int NCH, int G>
__global__ __launch_bounds__(kSortThreads, 2) void expert_bwd_token_kernel(const TokenPass p, const SortShare sort) {
  extern __shared__ __align__(16) uint8_t lds[];
  if (sort_share(sort, lds)) return;
  constexpr int E = Row16<DT>::kElems;
  const int lane = lane_id(), hidden = p.hidden, top_k = p.top_k;
  const int t = __builtin_amdgcn_readfirstlane(p.first + ((int)blockIdx.x - sort.blocks) * (int)(blockDim.x / kWave) + (int)(threadIdx.x >> 6));
  if (t >= p.last) return;
  const int64_t row_bytes = int64_t(hidden) * (16 / E);

  bool live[NCH];
  int64_t off[NCH];
  u32x4_t xr[NCH], dyr[NCH];
  float acc[NCH][E];
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    live[c] = (c * kWave + lane) * E < hidden;
    off[c] = int64_t(c * kWave + lane) * 16;
    xr[c] = live[c] ? *(const u32x4_t*)(p.x + t * row_bytes + off[c]) : u32x4_t{0, 0, 0, 0};
    dyr[c] = live[c] ? *(const u32x4_t*)(p.dy + t * row_bytes + off[c]) : u32x4_t{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < E; ++i) acc[c][i] = 0.f;
  }

  const int64_t base = int64_t(t) * top_k;
  for (int j0 = 0; j0 < top_k; j0 += G) {
    int e[G];
    float g[G];
    bool live_slot[G];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int j = min(j0 + i, top_k - 1);
      const int id = p.ids[base + j];
      const float gate = Elem<DT>::load(p.gates, base + j);
      const bool ok = (j0 + i < top_k) && (uint32_t)id < p.num_experts;   // as the forward: such a pair contributes nothing
      e[i] = ok ? id : 0;
      g[i] = ok ? gate : 0.f;
      live_slot[i] = ok;
    }
    u32x4_t ur[G][NCH], vr[G][NCH];
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
      for (int c = 0; c < NCH; ++c)
        ur[i][c] = live[c] ? *(const u32x4_t*)(p.up + e[i] * row_bytes + off[c]) : u32x4_t{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
      for (int c = 0; c < NCH; ++c)
        vr[i][c] = live[c] ? *(const u32x4_t*)(p.down + e[i] * row_bytes + off[c]) : u32x4_t{0, 0, 0, 0};

    float s[G], a[G];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      float ps = 0.f, pa = 0.f;
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        ps = dot16<DT>(xr[c], ur[i][c], ps);
        pa = dot16<DT>(dyr[c], vr[i][c], pa);
      }
      s[i] = ps;
      a[i] = pa;
    }
#pragma unroll
    for (int i = 0; i < G; ++i) {
      s[i] = wave_sum(s[i]);
      a[i] = wave_sum(a[i]);
    }
    // every lane forms the gradients of all of the batch's pairs; lane i keeps pair i's
    PairGrad mine{0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < G; ++i) {
      PairGrad q = pair_grad(s[i], a[i], g[i]);
      if (!live_slot[i]) q = PairGrad{0.f, 0.f, 0.f};
      if (lane == i) mine = q;
      if (live_slot[i]) {                       // not even 0 * row: the stand-in row may hold Inf or NaN
#pragma unroll
        for (int c = 0; c < NCH; ++c) axpy16<DT>(q.ds, ur[i][c], acc[c]);
      }
    }
    if (lane < G && j0 + lane < top_k) {
      Elem<DT>::store(p.dgates, base + j0 + lane, mine.dg);
      p.ds[base + j0 + lane] = mine.ds;
      p.coef[base + j0 + lane] = mine.coef;
    }
  }
#pragma unroll
  for (int c = 0; c < NCH; ++c)
    if (live[c]) *(u32x4_t*)(p.dx + t * row_bytes + off[c]) = pack16<DT>(acc[c]);
}

// Split: partial <dy, V> (and, where the forward kept no scores, <x, U>) of every pair and slice ...
template <int DT, int LPR, int S, bool RAGGED, bool SMALL>
__global__ __launch_bounds__(kSortThreads) void expert_bwd_dots_kernel(const TokenPass p, const SortShare sort) {
  extern __shared__ __align__(16) uint8_t lds[];
  if (sort_share(sort, lds)) return;
  const int block = (int)blockIdx.x - sort.blocks;
  split_dots_block<DT, LPR, S, RAGGED, SMALL, kTokenWaves>(p.dy, p.down, p.ids, p.partial_a, p.num_tokens, p.hidden, p.top_k, p.num_experts, p.lanes, 0, block);
  if (!p.scores) split_dots_block<DT, LPR, S, RAGGED, SMALL, kTokenWaves>(p.x, p.up, p.ids, p.partial_s, p.num_tokens, p.hidden, p.top_k, p.num_experts, p.lanes, 0, block);
}

// ... then the slice of dx = sum of ds U, with ds from the sums over the slices; slice 0 leaves dg, ds and the coefficients
template <int DT, int S, class Off>
struct SplitPairGrad {
  const TokenPass& p;
  bool writes, there, use;
  float part_a[S], part_s[S], gate;
  Off at;
  __device__ __forceinline__ void request(bool there_, int t, Off pair, int j, bool inside) {
    there = there_;
    use = there && inside;
    at = pair;
#pragma unroll
    for (int sl = 0; sl < S; ++sl) part_a[sl] = p.partial_a[(Off(sl) * p.num_tokens + t) * p.top_k + j];
    if (p.scores) part_s[0] = p.scores[pair];
    else
#pragma unroll
      for (int sl = 0; sl < S; ++sl) part_s[sl] = p.partial_s[(Off(sl) * p.num_tokens + t) * p.top_k + j];
    gate = Elem<DT>::load(p.gates, pair);
  }
  __device__ __forceinline__ float value() {
    float a = part_a[0], s = part_s[0];
#pragma unroll
    for (int sl = 1; sl < S; ++sl) a += part_a[sl];
    if (!p.scores)
#pragma unroll
      for (int sl = 1; sl < S; ++sl) s += part_s[sl];
    PairGrad q = pair_grad(s, a, gate);
    if (!use) q = PairGrad{0.f, 0.f, 0.f};
    if (there && writes) {
      Elem<DT>::store(p.dgates, at, q.dg);
      p.ds[at] = q.ds;
      p.coef[at] = q.coef;
    }
    return q.ds;
  }
};
template <int DT, int LPR, int S, bool RAGGED, bool SMALL>
__global__ __launch_bounds__(kSortThreads) void expert_bwd_accumulate_kernel(const TokenPass p, const SortShare sort) {
  extern __shared__ __align__(16) uint8_t lds[];
  if (sort_share(sort, lds)) return;
  using Off = typename SplitOff<SMALL>::type;
  const int block = (int)blockIdx.x - sort.blocks;
  SplitPairGrad<DT, S, Off> pair{p, block % S == 0};
  split_accumulate_block<DT, LPR, S, RAGGED, SMALL, kTokenWaves>(p.up, p.ids, p.dx, p.num_tokens, p.hidden, p.top_k, p.num_experts, p.lanes, 0, block, pair);
}

// ---- experts, weight pass ----------------------------------------------------------------------
// The sorted pair list is cut into chunks of `chunk` consecutive pairs, one wave each, whatever the segment lengths: a popular expert's
// segment is spread over many waves and many rare experts share one.  A wave sums run after run (a run = consecutive pairs of one expert).
// A segment of up to `chunk` pairs is summed, rounded and stored by the wave of the chunk that it begins in, also beyond that chunk's
// border; a longer one is cut at the borders, and every wave leaves its run as an fp32 partial row pair in `partials[chunk][slot]`, slot 0
// if the run starts the chunk, slot 1 otherwise (a chunk has at most one of each); the fix-up kernel then adds an expert's partials in
// chunk order, so the summation order is fixed and nothing is added atomically.  (With every segment cut at the borders, 65536 pairs over 4096
// experts left 33 MB of partial rows: weight pass and fix-up 24.3 + 12.1 -> 24.3 + 9.5 us, 32768 over 16384 18.5 + 6.4 -> 16.4 + 4.6; the
// whole backward at 4096 tokens x 16, hidden 1024, 60.5 -> 54.4, hidden 2048 119.9 -> 102.8.)
//
// Bound by the gathers: a row pair is read for every pair of the list.  What a wave owns is therefore a chunk of one PART of the columns: up to 1 KiB of
// the rows of x (for dU) or of dy (for dV), 16 bytes to a lane, and the parts go to the XCDs one after another, so that an XCD gathers from the one or two
// parts that its L2 holds; with whole rows of both in every wave, all of x and dy went through every L2 and the pass ran at the fabric's 7 TB/s.  A wave's row
// address and factor are scalars, so a narrower part costs no exchange between lanes.  Rows of up to 512 bytes: x in the lower half of the lanes, dy in the
// upper.  The finished rows pass the L2 by (non-temporal), which is left to the rows that are gathered.  The chunks, and with them the order of all sums, do not depend on the parts.  (4096 tokens x 16, hidden 1024, bf16 37.7 -> 24.3 us, 1024 x 32 over 16384
// experts 23.7 -> 18.5.  The parts of a chunk one after the other instead, which keeps whole rows together: the whole backward there 54.4 -> 71.6 and 45.9 -> 51.5,
// at 32768 tokens x 16 over 65536, which no L2 holds, 888 either way.  A recorded call of the experts, eight rows in flight -> four: 16384 x 16 over 4096 265.0 -> 261.5, 8192 x 8 over 16384,
// hidden 2048, 221.6 -> 221.1; finished rows through the L2 -> past it: 261.3 -> 261.0 and 232.1 -> 220.7; sixteen rows or the next batch requested ahead: 1-3 % slower at 1024 and 4096 tokens.)
struct WeightPass {
  const uint8_t *x, *dy;
  const float *ds, *coef;
  const int32_t *ids, *offsets, *pair_ids, *token_ids;
  uint8_t *dup, *ddown;
  float* partials;
  int64_t num_experts;
  int hidden, chunk, num_chunks;
  int lanes, columns;                // 16-byte lanes of a part; parts of a row of x, and as many of dy (0: both in one part)
  int blocks, per_xcd;               // blocks of a part; all parts' blocks on an XCD
};
// R > 0: the launch's first `router_blocks` blocks (a multiple of eight, so that block % 8 names the XCD of the others too) are the router's, R columns of a half to
// a lane.
template <int DT, bool PAIRED, int G, int R>
__global__ __launch_bounds__((R ? norm_waves(R) : kBwdWavesPerBlock) * kWave) void expert_bwd_weight_kernel(const WeightPass p, const RouterPass router, const int router_blocks) {
  constexpr int E = Row16<DT>::kElems, W = R ? norm_waves(R) : kBwdWavesPerBlock;
  if constexpr (R > 0) {
    if ((int)blockIdx.x < router_blocks) {
      if ((int)blockIdx.x * W * router.tokens_per_wave < router.num_tokens) router_norm_bwd_block<DT, R>(router, (int)blockIdx.x);
      return;
    }
  }
  const int lane = lane_id(), at_block = (int)blockIdx.x - router_blocks;
  const int item = (at_block % kXcds) * p.per_xcd + at_block / kXcds, parts = PAIRED ? 1 : 2 * p.columns;
  if (item >= parts * p.blocks) return;
  const int part = item / p.blocks, ci = __builtin_amdgcn_readfirstlane((item - part * p.blocks) * W + (int)(threadIdx.x >> 6));
  if (ci >= p.num_chunks) return;
  const int valid = p.offsets[p.num_experts];         // pairs with an id inside the table
  const int border = ci * p.chunk;
  int first = border, last = min(border + p.chunk, valid);
  if (first >= last) return;
  // the segments that the chunk's first and last pair are of
  auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  const int e0 = uniform(p.ids[p.pair_ids[first]]), e1 = uniform(p.ids[p.pair_ids[last - 1]]);
  const int begin0 = uniform(p.offsets[e0]), end0 = uniform(p.offsets[e0 + 1]), begin1 = uniform(p.offsets[e1]), end1 = uniform(p.offsets[e1 + 1]);
  const bool cut0 = end0 - begin0 > p.chunk, cut1 = end1 - begin1 > p.chunk;
  if (!cut0 && begin0 < border) first = end0;         // the wave that it begins with finishes it
  if (!cut1) last = end1;
  if (first >= last) return;
  const uint32_t row_bytes = (uint32_t)p.hidden * (16 / E);

  const bool second = PAIRED ? lane >= kWave / 2 : part >= p.columns;           // of dy and dV
  const int in_part = PAIRED ? lane % (kWave / 2) : lane, piece = (PAIRED ? 0 : (second ? part - p.columns : part) * p.lanes) + in_part;
  const bool live = in_part < p.lanes && piece * E < p.hidden;
  const uint32_t off = live ? piece * 16u : 0u;       // the other lanes read what the first one does, and store nothing
  const uint8_t* const rows = second ? p.dy : p.x;
  uint8_t* const out_rows = second ? p.ddown : p.dup;
  const float* const factors = PAIRED ? p.ds : second ? p.coef : p.ds;
  float acc[E];
#pragma unroll
  for (int i = 0; i < E; ++i) acc[i] = 0.f;
  // Ends the run [run_first, run_last) of expert e and clears the accumulators
  auto flush = [&](int e, int run_first, int run_last) {
    const bool whole = (run_first != border || !cut0) && (run_last != last || !cut1);
    if (live) {
      if (whole) {
        __builtin_nontemporal_store(pack16<DT>(acc), (u32x4_t*)(out_rows + (int64_t)e * row_bytes + off));
      } else {
        float* out = p.partials + (int64_t(ci) * 2 + (run_first == border ? 0 : 1)) * 2 * p.hidden + (second ? p.hidden : 0) + piece * E;
#pragma unroll
        for (int q = 0; q < E; q += 4) *(f32x4_t*)(out + q) = f32x4_t{acc[q], acc[q + 1], acc[q + 2], acc[q + 3]};
      }
    }
#pragma unroll
    for (int i = 0; i < E; ++i) acc[i] = 0.f;
  };

  int run_e = -1, run_first = first;
  for (int p64 = first; p64 < last; p64 += kWave) {   // list order = (expert, pair) order: a fixed summation order
    // lane i holds what belongs to pair p64 + i: the chain pair -> id is walked once for 64 pairs, and the rows of every batch can be asked for at once
    const int n = min(kWave, last - p64), mine = p64 + min(lane, n - 1), my_pid = p.pair_ids[mine], my_tok = p.token_ids[mine];
    const int my_e = p.ids[my_pid];
    const float my_factor = factors[my_pid], my_coef = PAIRED ? p.coef[my_pid] : 0.f;
    if (run_e < 0) run_e = __builtin_amdgcn_readlane(my_e, 0);
    const int left_e = __shfl_up(my_e, 1, kWave);
    const uint64_t starts = __ballot(my_e != (lane ? left_e : run_e));          // bit i: pair p64 + i begins a run
    auto request = [&](int at) __attribute__((always_inline)) {
      const uint8_t* row = rows + (uint64_t)(uint32_t)__builtin_amdgcn_readlane(my_tok, at) * row_bytes;
      if constexpr (!PAIRED) asm("" : "+s"(row));     // a scalar base and the lane's 32-bit offset, not a 64-bit address for every lane
      return *(const u32x4_t*)(row + off);
    };
    auto add = [&](int at, const u32x4_t& row) __attribute__((always_inline)) {
      float factor = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_factor), at));
      if constexpr (PAIRED) {
        const float coef = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_coef), at));
        factor = second ? coef : factor;
      }
      if (starts >> at & 1) {
        flush(run_e, run_first, p64 + at);
        run_e = __builtin_amdgcn_readlane(my_e, at);
        run_first = p64 + at;
      }
      axpy16<DT>(factor, row, acc);
    };
    u32x4_t row[G];
    int at = 0;
    for (; at + G <= n; at += G) {
#pragma unroll
      for (int i = 0; i < G; ++i) row[i] = request(at + i);
#pragma unroll
      for (int i = 0; i < G; ++i) add(at + i, row[i]);
    }
    if (at < n) {
#pragma unroll
      for (int i = 0; i < G - 1; ++i) row[i] = request(min(at + i, n - 1));
#pragma unroll
      for (int i = 0; i < G - 1; ++i)
        if (at + i < n) add(at + i, row[i]);
    }
  }
  flush(run_e, run_first, last);
}

// One wave per expert: zero rows for an expert nobody selected; for a segment of more than `chunk` pairs the sum of its partial rows,
// first chunk to last.  The others were stored by the pass above.
// FINISH: the launch's first `finish_blocks` blocks finish the router's d(z).  Router and experts, before / now: 4096 tokens x 1024 over 64 x 64, k 16: pass 24.3, fix-up beside
// the first 9.4, finish 7.3 us -> 25.5 + 8.7; 1000 x 512 over 32 x 32, k 8: 6.2 + 4.7 + 6.0 -> 7.2 + 6.0.
template <int DT, int NCH, bool FINISH>
__global__ __launch_bounds__((FINISH ? kFinishWaves : kBwdWavesPerBlock) * kWave) void expert_bwd_weight_fixup_kernel(
    const int32_t* __restrict__ offsets, const float* __restrict__ partials, uint8_t* __restrict__ dup,
    uint8_t* __restrict__ ddown, int64_t num_experts, int hidden, int chunk, const RouterPass router, const int router_rows, const int finish_blocks) {
  constexpr int E = Row16<DT>::kElems, W = FINISH ? kFinishWaves : kBwdWavesPerBlock;
  if constexpr (FINISH) {
    if ((int)blockIdx.x < finish_blocks) {
      router_norm_bwd_finish_block<DT>(router, router_rows, (int)blockIdx.x, finish_blocks);
      return;
    }
  }
  const int lane = lane_id();
  const int64_t e = __builtin_amdgcn_readfirstlane((int)(((int)blockIdx.x - finish_blocks) * W + (int)(threadIdx.x >> 6)));
  if (e >= num_experts) return;
  const int begin = offsets[e], end = offsets[e + 1];
  if (end > begin && end - begin <= chunk) return;
  const int c0 = begin / chunk, c1 = end > begin ? (end - 1) / chunk : c0;
  const int64_t row_bytes = int64_t(hidden) * (16 / E);
  float au[NCH][E], av[NCH][E];
#pragma unroll
  for (int c = 0; c < NCH; ++c)
#pragma unroll
    for (int i = 0; i < E; ++i) au[c][i] = av[c][i] = 0.f;
  if (end > begin) {
    for (int ci = c0; ci <= c1; ++ci) {
      const int slot = (ci == c0 && begin != c0 * chunk) ? 1 : 0;
      const float* in = partials + (int64_t(ci) * 2 + slot) * 2 * hidden;
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const int col = (c * kWave + lane) * E;
        if (col < hidden) {
#pragma unroll
          for (int q = 0; q < E; q += 4) {
            const f32x4_t u = *(const f32x4_t*)(in + col + q), v = *(const f32x4_t*)(in + hidden + col + q);
#pragma unroll
            for (int z = 0; z < 4; ++z) {
              au[c][q + z] += u[z];
              av[c][q + z] += v[z];
            }
          }
        }
      }
    }
  }
#pragma unroll
  for (int c = 0; c < NCH; ++c)
    if ((c * kWave + lane) * E < hidden) {
      *(u32x4_t*)(dup + e * row_bytes + int64_t(c * kWave + lane) * 16) = pack16<DT>(au[c]);
      *(u32x4_t*)(ddown + e * row_bytes + int64_t(c * kWave + lane) * 16) = pack16<DT>(av[c]);
    }
}

// ---- SwiGLU, element-wise ----------------------------------------------------------------------
// 16 bytes per lane.  Forward: out = silu(gate) * up in fp32, one rounding (omni_mlp.py:53-61).
// Backward: with a = gate in fp32, sig = sigmoid(a):  d_up = dout * a sig,
// d_gate = dout * (a sig (1 - sig) + sig) * up  (omni_mlp.py:232-236).
template <int DT, bool BWD>
__global__ __launch_bounds__(256) void swiglu_kernel(const uint8_t* __restrict__ dout, const uint8_t* __restrict__ gate,
                                                    const uint8_t* __restrict__ up, uint8_t* __restrict__ out0,
                                                    uint8_t* __restrict__ out1, int64_t num_chunks) {
  constexpr int E = Row16<DT>::kElems;
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < num_chunks; i += gridDim.x * 256ll) {
    const u32x4_t gw = *(const u32x4_t*)(gate + i * 16), uw = *(const u32x4_t*)(up + i * 16);
    float gv[E], uv[E], r0[E], r1[E];
    unpack16<DT>(gw, gv);
    unpack16<DT>(uw, uv);
    if constexpr (BWD) {
      float dv[E];
      unpack16<DT>(*(const u32x4_t*)(dout + i * 16), dv);
#pragma unroll
      for (int q = 0; q < E; ++q) {
        const float sig = sigmoid_f32(gv[q]), silu = gv[q] * sig;
        r0[q] = dv[q] * (silu * (1.0f - sig) + sig) * uv[q];
        r1[q] = dv[q] * silu;
      }
      *(u32x4_t*)(out0 + i * 16) = pack16<DT>(r0);
      *(u32x4_t*)(out1 + i * 16) = pack16<DT>(r1);
    } else {
#pragma unroll
      for (int q = 0; q < E; ++q) r0[q] = gv[q] * sigmoid_f32(gv[q]) * uv[q];
      *(u32x4_t*)(out0 + i * 16) = pack16<DT>(r0);
    }
  }
}

// ---- host side ---------------------------------------------------------------------------------
static inline size_t up256(size_t v) { return (v + 255) / 256 * 256; }
static int to_code(hipError_t e) { return e == hipSuccess ? OMNI_OK : OMNI_ERR_HIP_BASE + (int)e; }

// pairs per weight-pass chunk: about 2048 chunks (8 waves per CU), at least 16 pairs each
static inline int weight_chunk(size_t pairs) {
  const size_t c = (pairs + 2047) / 2048;
  return (int)(c < 16 ? 16 : c);
}

// What a launch of the token pass takes in LDS: the tables of the sort beside it
template <auto kKernel>
struct TokenLds { static inline LdsKernel entry{(const void*)kKernel, (kSortWaves + 3) * slice_width(kMaxBinsWide) * 4}; };
template <auto kKernel>
static hipError_t start_token(const TokenPass& p, const SortPass* sort, int kind, int64_t blocks, hipStream_t s, int threads = kSortThreads) {
  SortShare share{};
  int bytes = 0;
  if (kind != kSortNone) {
    share = SortShare{*sort, kind, kind == kSortCount ? (sort->tiles + kXcds - 1) / kXcds * kXcds : sort->tiles * kBinSlices};
    bytes = kind == kSortCount ? count_lds(sort->stride) : scatter_lds(sort->width);
    if (bytes > 65536)
      if (hipError_t e = TokenLds<kKernel>::entry.ensure(); e != hipSuccess) return e;
  }
  if (share.blocks + blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(kKernel, dim3((unsigned)(share.blocks + blocks)), dim3(threads), bytes, s, p, share);
  return hipGetLastError();
}
template <int DT>
static hipError_t launch_token_split(const TokenPass& p, const SortPass* sort, hipStream_t s) {
  const bool small = split_offsets_small(p.up, p.down, p.num_tokens, p.hidden, p.top_k, p.num_experts, 1, DT == kF32 ? 4 : 2);
  return split_dispatch(p.lanes, p.slices, [&](auto group, auto s_tag, auto ragged) {
    constexpr int LPR = decltype(group)::value, S = decltype(s_tag)::value;
    constexpr bool RAGGED = decltype(ragged)::value;
    const int64_t blocks = split_blocks(p.num_tokens, kTokenWaves * (kWave / LPR), S);
    const int count = sort && sort->tiles > 1 ? kSortCount : kSortNone, scatter = sort ? kSortScatter : kSortNone;
    if constexpr (LPR < 8) {
      return hipErrorInvalidValue;
    } else {
      const hipError_t e = small ? start_token<expert_bwd_dots_kernel<DT, LPR, S, RAGGED, true>>(p, sort, count, blocks, s)
                                 : start_token<expert_bwd_dots_kernel<DT, LPR, S, RAGGED, false>>(p, sort, count, blocks, s);
      if (e != hipSuccess) return e;
      return small ? start_token<expert_bwd_accumulate_kernel<DT, LPR, S, RAGGED, true>>(p, sort, scatter, blocks, s)
                   : start_token<expert_bwd_accumulate_kernel<DT, LPR, S, RAGGED, false>>(p, sort, scatter, blocks, s);
    }
  });
}
// Gather: the scatter pass has all tokens beside it, from 4096 tokens on (two rounds of waves) the count pass half of them; with nothing to share, blocks of
// four waves, two to a CU (23578 tokens x 6, hidden 1024: 2 % of the whole backward)
template <int DT, int NCH, int G>
static hipError_t launch_token_gather(TokenPass p, const SortPass* sort, hipStream_t s) {
  constexpr auto kKernel = expert_bwd_token_kernel<DT, NCH, G>;
  auto blocks = [](int tokens, int waves) -> int64_t { return (tokens + waves - 1) / waves; };
  p.first = 0;
  p.last = p.num_tokens;
  if (!sort) return start_token<kKernel>(p, nullptr, kSortNone, blocks(p.num_tokens, kBwdWavesPerBlock), s, kBwdWavesPerBlock * kWave);
  p.last = p.num_tokens >= 4096 && sort->tiles > 1 ? p.num_tokens / 2 : 0;
  if (sort->tiles > 1)
    if (hipError_t e = start_token<kKernel>(p, sort, kSortCount, blocks(p.last, kTokenWaves), s); e != hipSuccess) return e;
  p.first = p.last;
  p.last = p.num_tokens;
  return start_token<kKernel>(p, sort, kSortScatter, blocks(p.last - p.first, kTokenWaves), s);
}

// The router's share of a backward pass: blocks of its first launch, and its launches
static int norm_blocks(int64_t num_tokens, int r) {
  const int64_t per_block = (int64_t)norm_waves((r + kWave - 1) / kWave) * norm_tokens_per_wave(num_tokens);
  return (int)((num_tokens + per_block - 1) / per_block);
}
template <int DT>
static hipError_t launch_norm_first(const RouterPass& p, hipStream_t s) {
  const unsigned blocks = (unsigned)norm_blocks(p.num_tokens, p.r);
  if (p.r <= kWave) hipLaunchKernelGGL((router_norm_bwd_kernel<DT, 1>), dim3(blocks), dim3(norm_waves(1) * kWave), 0, s, p);
  else if (p.r <= 4 * kWave) hipLaunchKernelGGL((router_norm_bwd_kernel<DT, 4>), dim3(blocks), dim3(norm_waves(4) * kWave), 0, s, p);
  else hipLaunchKernelGGL((router_norm_bwd_kernel<DT, 16>), dim3(blocks), dim3(norm_waves(16) * kWave), 0, s, p);
  return hipGetLastError();
}
// Blocks that finish d(z): a CU's block for every group of columns, or fewer where 64 tokens to a block are all
static int finish_blocks(const RouterPass& p) {
  const int groups = 2 * ((p.r + kWave - 1) / kWave), want = (p.num_tokens + kFinishWaves * kFinishRows - 1) / (kFinishWaves * kFinishRows), most = groups < 256 ? 256 / groups : 1;
  return groups * (want < most ? want : most);
}
template <int DT>
static hipError_t launch_norm_finish(const RouterPass& p, hipStream_t s) {
  if (!p.training) return hipSuccess;
  hipLaunchKernelGGL(router_norm_bwd_finish_kernel<DT>, dim3((unsigned)finish_blocks(p)), dim3(kFinishWaves * kWave), 0, s, p, norm_blocks(p.num_tokens, p.r));
  return hipGetLastError();
}

template <int DT, int NCH, int G>
static hipError_t launch_expert_bwd(const TokenPass& p, const SortPass* sort, void* dup, void* ddown, const int32_t* offsets, const int32_t* pair_ids,
                                    const int32_t* token_ids, float* partials, const RouterPass* router, hipStream_t s) {
  const int64_t T = p.num_tokens, N = p.num_experts;
  const int H = p.hidden, k = p.top_k;
  const hipError_t te = p.lanes ? launch_token_split<DT>(p, sort, s) : launch_token_gather<DT, NCH, G>(p, sort, s);
  if (te != hipSuccess) return te;
  const size_t P = (size_t)T * (size_t)k;
  const int chunk = weight_chunk(P);
  const int num_chunks = (int)((P + chunk - 1) / chunk);
  // The router beside: up to four columns of a half to a lane, and, in the second launch, rows of up to 4 KiB (16-bit 2048 columns)
  const bool first_beside = router && num_chunks > 0 && router->r <= 4 * kWave, finish_beside = router && router->training && NCH <= 4;
  if (router && !first_beside)
    if (hipError_t e = launch_norm_first<DT>(*router, s); e != hipSuccess) return e;
  if (num_chunks > 0) {
    constexpr int E = Row16<DT>::kElems;
    WeightPass w{p.x, p.dy, p.ds, p.coef, p.ids, offsets, pair_ids, token_ids, (uint8_t*)dup, (uint8_t*)ddown, partials, N, H, chunk, num_chunks};
    const int pieces = H / E;                          // 16-byte pieces of a row
    const bool paired = pieces <= kWave / 2;
    w.columns = paired ? 0 : (pieces + kWave - 1) / kWave;
    w.lanes = paired ? pieces : (pieces + w.columns - 1) / w.columns;
    auto start = [&](auto cols) {
      constexpr int R = decltype(cols)::value, W = R ? norm_waves(R) : kBwdWavesPerBlock;
      w.blocks = (num_chunks + W - 1) / W;
      w.per_xcd = ((paired ? 1 : 2 * w.columns) * w.blocks + kXcds - 1) / kXcds;
      const int router_blocks = R ? (norm_blocks(T, router->r) + kXcds - 1) / kXcds * kXcds : 0;
      const dim3 grid((unsigned)(router_blocks + w.per_xcd * kXcds)), block(W * kWave);
      const RouterPass beside = R ? *router : RouterPass{};
      if (paired) hipLaunchKernelGGL((expert_bwd_weight_kernel<DT, true, 4, R>), grid, block, 0, s, w, beside, router_blocks);
      else hipLaunchKernelGGL((expert_bwd_weight_kernel<DT, false, 4, R>), grid, block, 0, s, w, beside, router_blocks);
      return hipGetLastError();
    };
    const hipError_t e = !first_beside ? start(std::integral_constant<int, 0>{}) : router->r <= kWave ? start(std::integral_constant<int, 1>{}) : start(std::integral_constant<int, 4>{});
    if (e != hipSuccess) return e;
  }
  auto fixup = [&](auto finish) {
    constexpr bool FINISH = decltype(finish)::value;
    constexpr int W = FINISH ? kFinishWaves : kBwdWavesPerBlock;
    const int first = FINISH ? finish_blocks(*router) : 0;
    hipLaunchKernelGGL((expert_bwd_weight_fixup_kernel<DT, NCH, FINISH>), dim3((unsigned)(first + (N + W - 1) / W)), dim3(W * kWave), 0, s, offsets, partials, (uint8_t*)dup,
                       (uint8_t*)ddown, N, H, chunk, FINISH ? *router : RouterPass{}, FINISH ? norm_blocks(T, router->r) : 0, first);
    return hipGetLastError();
  };
  if constexpr (NCH <= 4) {
    if (finish_beside) return fixup(std::true_type{});
  }
  const hipError_t e = fixup(std::false_type{});
  return e != hipSuccess || !router ? e : launch_norm_finish<DT>(*router, s);
}

}  // namespace omni

extern "C" OMNI_API int32_t omni_router_bwd(const void* dscores, const int32_t* indices, void* dlogits_x, void* dlogits_y,
                                            int64_t num_tokens, int32_t num_expert_sqrt, int32_t num_experts_per_token,
                                            int32_t dtype, void* stream) {
  using namespace omni;
  if (num_tokens < 0 || num_tokens > INT32_MAX || num_expert_sqrt <= 0 || num_experts_per_token < 0) return OMNI_ERR_SHAPE;
  if (num_expert_sqrt > 1024) return OMNI_ERR_UNSUPPORTED;
  if (num_experts_per_token > 128) return OMNI_ERR_TOPK;
  if (dtype != OMNI_BF16 && dtype != OMNI_F16 && dtype != OMNI_F32) return OMNI_ERR_DTYPE;
  if (num_tokens == 0) return OMNI_OK;
  if (!dlogits_x || !dlogits_y || (num_experts_per_token > 0 && (!dscores || !indices))) return OMNI_ERR_NULL;
  dim3 grid((unsigned)((num_tokens + kBwdWavesPerBlock - 1) / kBwdWavesPerBlock)), block(kBwdWavesPerBlock * kWave);
  hipStream_t s = (hipStream_t)stream;
  const int T = (int)num_tokens, r = num_expert_sqrt, k = num_experts_per_token;
#define OMNI_ROUTER_BWD_CASE(DT)                                                                                             \
  do {                                                                                                                       \
    if (r <= 64) hipLaunchKernelGGL((router_bwd_kernel<DT, 1>), grid, block, 0, s, dscores, indices, dlogits_x, dlogits_y, T, r, k);        \
    else if (r <= 256) hipLaunchKernelGGL((router_bwd_kernel<DT, 4>), grid, block, 0, s, dscores, indices, dlogits_x, dlogits_y, T, r, k);  \
    else hipLaunchKernelGGL((router_bwd_kernel<DT, 16>), grid, block, 0, s, dscores, indices, dlogits_x, dlogits_y, T, r, k);               \
  } while (0)
  if (dtype == OMNI_BF16) OMNI_ROUTER_BWD_CASE(kBF16);
  else if (dtype == OMNI_F16) OMNI_ROUTER_BWD_CASE(kF16);
  else OMNI_ROUTER_BWD_CASE(kF32);
#undef OMNI_ROUTER_BWD_CASE
  return to_code(hipGetLastError());
}

// workspace of omni_router_norm_bwd: per-block column sums [blocks][4][r] f32
extern "C" OMNI_API size_t omni_router_norm_bwd_workspace_bytes(int64_t num_tokens, int32_t num_expert_sqrt) {
  using namespace omni;
  if (num_tokens < 0 || num_expert_sqrt <= 0) return 0;
  return up256((size_t)norm_blocks(num_tokens, num_expert_sqrt) * 4 * num_expert_sqrt * 4);
}

// Checks the arguments and fills p; num_tokens 0: nothing to do
static int32_t router_pass(omni::RouterPass& p, const void* dgates, const void* gates, const int32_t* indices, const void* z, const float* stats, void* dz, int64_t num_tokens,
                           int r, int k, int32_t dtype, int32_t training, void* workspace, bool padded) {
  using namespace omni;
  if (num_tokens < 0 || num_tokens > INT32_MAX / 4096 || r <= 0 || k < 0) return OMNI_ERR_SHAPE;
  if (r > 1024) return OMNI_ERR_UNSUPPORTED;
  if (k > 128) return OMNI_ERR_TOPK;
  if (dtype != OMNI_BF16 && dtype != OMNI_F16 && dtype != OMNI_F32) return OMNI_ERR_DTYPE;
  if (num_tokens == 0) return OMNI_OK;
  if (!z || !stats || !dz || (k > 0 && (!dgates || !gates || !indices))) return OMNI_ERR_NULL;
  if (training && !workspace) return OMNI_ERR_WORKSPACE;
  p = RouterPass{dgates, gates, indices, z, stats, dz, (float*)workspace, (int)num_tokens, r, k, training, norm_tokens_per_wave(num_tokens), padded ? (r + 7) / 8 * 8 : r};
  return OMNI_OK;
}
static int32_t router_norm_bwd(const void* dgates, const void* gates, const int32_t* indices, const void* z, const float* stats, void* dz,
                               int64_t num_tokens, int32_t num_expert_sqrt, int32_t num_experts_per_token, int32_t dtype, int32_t training,
                               void* workspace, void* stream, bool padded) {
  using namespace omni;
  RouterPass p;
  if (int e = router_pass(p, dgates, gates, indices, z, stats, dz, num_tokens, num_expert_sqrt, num_experts_per_token, dtype, training, workspace, padded)) return e;
  if (num_tokens == 0) return OMNI_OK;
  hipStream_t s = (hipStream_t)stream;
  auto go = [&](auto dt) {
    constexpr int DT = decltype(dt)::value;
    const hipError_t e = launch_norm_first<DT>(p, s);
    return to_code(e != hipSuccess ? e : launch_norm_finish<DT>(p, s));
  };
  if (dtype == OMNI_BF16) return go(std::integral_constant<int, kBF16>{});
  if (dtype == OMNI_F16) return go(std::integral_constant<int, kF16>{});
  return go(std::integral_constant<int, kF32>{});
}

extern "C" OMNI_API int32_t omni_router_norm_bwd(const void* dgates, const void* gates, const int32_t* indices, const void* z,
                                                 const float* stats, void* dz, int64_t num_tokens, int32_t num_expert_sqrt,
                                                 int32_t num_experts_per_token, int32_t dtype, int32_t training, void* workspace,
                                                 void* stream) {
  return router_norm_bwd(dgates, gates, indices, z, stats, dz, num_tokens, num_expert_sqrt, num_experts_per_token, dtype, training, workspace, stream, false);
}

extern "C" OMNI_API int32_t omni_router_norm_bwd_padded(const void* dgates, const void* gates, const int32_t* indices, const void* z,
                                                        const float* stats, void* dz, int64_t num_tokens, int32_t num_expert_sqrt,
                                                        int32_t num_experts_per_token, int32_t dtype, int32_t training, void* workspace,
                                                        void* stream) {
  return router_norm_bwd(dgates, gates, indices, z, stats, dz, num_tokens, num_expert_sqrt, num_experts_per_token, dtype, training, workspace, stream, true);
}

namespace omni {
int resolve_algo(int algo, int64_t T, int H, int64_t N, int k, int dtype);       // defined beside the expert kernels: what AUTO runs
// Slices where the token pass takes the split organisation, else 0: where the forward does, but for sorts of one tile, beside which the gather organisation is
// one launch less (whole backward, bf16, rows of 512 B to 1 KiB, 1100 and 2048 tokens x 2 and 4, split over gather: 1.09-1.18 up to 8192 pairs, 0.97-1.02 at 8800)
static int bwd_split_slices(int64_t T, int H, int64_t N, int k, int dtype) {
  if (T * (int64_t)k <= 8192 || resolve_algo(OMNI_EXPERT_ALGO_AUTO, T, H, N, k, dtype) != OMNI_EXPERT_ALGO_SPLIT) return 0;
  const int es = dtype == OMNI_F32 ? 4 : 2, slices = (int64_t)H * es <= 8192 ? split_slices(H, N, es) : 0;
  return slices && split_lanes_per_row(H, es, slices) >= 5 ? slices : 0;       // (no kernels for groups of four lanes)
}
}  // namespace omni

// workspace: ds [P] f32 | coef [P] f32 | sorted pair ids [P] i32 | sorted token ids [P] i32 | offsets [N+1] i32 |
//            partial rows [chunks][2][2][H] f32 | split: partial <dy, V>, partial <x, U> (without scores) [slices][P] f32 each | schedule workspace
extern "C" OMNI_API size_t omni_expert_bwd_workspace_bytes(int64_t num_tokens, int32_t hidden_size, int64_t num_experts,
                                                           int32_t num_experts_per_token, int32_t dtype) {
  using namespace omni;
  if (num_tokens < 0 || num_experts <= 0 || num_experts_per_token < 0 || hidden_size <= 0) return 0;
  const size_t P = (size_t)num_tokens * (size_t)num_experts_per_token;
  const size_t chunks = (P + weight_chunk(P) - 1) / weight_chunk(P);
  const size_t slices = (size_t)bwd_split_slices(num_tokens, hidden_size, num_experts, num_experts_per_token, dtype);
  return 4 * up256(P * 4) + up256(((size_t)num_experts + 1) * 4) + up256(chunks * 4 * (size_t)hidden_size * 4) + 2 * up256(slices * P * 4) +
         omni_schedule_workspace_bytes(num_tokens, num_experts_per_token, num_experts);
}

extern "C" OMNI_API int32_t omni_expert_bwd_reads_scores(int64_t num_tokens, int32_t hidden_size, int64_t num_experts, int32_t num_experts_per_token, int32_t dtype) {
  if (num_tokens < 0 || num_experts <= 0 || num_experts_per_token < 0 || hidden_size <= 0) return 0;
  return omni::bwd_split_slices(num_tokens, hidden_size, num_experts, num_experts_per_token, dtype) ? 1 : 0;
}

extern "C" OMNI_API int32_t omni_expert_bwd(const void* dy, const void* x, const void* up_weight, const void* down_weight,
                                            const void* routing_weights, const int32_t* indices, void* dx, void* dup_weight,
                                            void* ddown_weight, void* drouting_weights, int64_t num_tokens, int32_t hidden_size,
                                            int64_t num_experts, int32_t num_experts_per_token, int32_t dtype, void* workspace,
                                            void* stream) {
  return omni_expert_bwd_scores(dy, x, up_weight, down_weight, routing_weights, indices, nullptr, dx, dup_weight, ddown_weight, drouting_weights, num_tokens, hidden_size,
                                num_experts, num_experts_per_token, dtype, workspace, stream);
}

// router: NULL, or the router's share, enqueued behind the token pass
static int32_t expert_bwd(const void* dy, const void* x, const void* up_weight, const void* down_weight, const void* routing_weights,
                          const int32_t* indices, const float* scores, void* dx, void* dup_weight, void* ddown_weight, void* drouting_weights,
                          int64_t num_tokens, int32_t hidden_size, int64_t num_experts, int32_t num_experts_per_token, int32_t dtype,
                          void* workspace, void* stream, const omni::RouterPass* router) {
  using namespace omni;
  if (num_tokens < 0 || hidden_size <= 0 || num_experts <= 0 || num_experts_per_token < 0) return OMNI_ERR_SHAPE;
  if (num_tokens > INT32_MAX / 2 || num_experts > INT32_MAX / 2 ||
      num_tokens * (int64_t)num_experts_per_token > INT32_MAX / 2)
    return OMNI_ERR_SHAPE;
  if (dtype != OMNI_BF16 && dtype != OMNI_F16 && dtype != OMNI_F32) return OMNI_ERR_DTYPE;
  if (!dup_weight || !ddown_weight) return OMNI_ERR_NULL;
  if (num_tokens > 0 && (!dy || !x || !dx || !up_weight || !down_weight)) return OMNI_ERR_NULL;
  if (num_tokens > 0 && num_experts_per_token > 0 && (!routing_weights || !indices || !drouting_weights)) return OMNI_ERR_NULL;
  if (!workspace) return OMNI_ERR_WORKSPACE;
  const int E = dtype == OMNI_F32 ? 4 : 8;
  if (hidden_size % E != 0) return OMNI_ERR_SHAPE;
  const int nch = (hidden_size + kWave * E - 1) / (kWave * E);
  if (nch > 8) return OMNI_ERR_UNSUPPORTED;
  const size_t P = (size_t)num_tokens * (size_t)num_experts_per_token;
  char* w = (char*)workspace;
  float* ds = (float*)w;               w += up256(P * 4);
  float* coef = (float*)w;             w += up256(P * 4);
  int32_t* pair_ids = (int32_t*)w;     w += up256(P * 4);
  int32_t* token_ids = (int32_t*)w;    w += up256(P * 4);
  int32_t* offsets = (int32_t*)w;      w += up256(((size_t)num_experts + 1) * 4);
  float* partials = (float*)w;
  {
    const size_t chunks = (P + weight_chunk(P) - 1) / weight_chunk(P);
    w += up256(chunks * 4 * (size_t)hidden_size * 4);
  }
  const int slices = bwd_split_slices(num_tokens, hidden_size, num_experts, num_experts_per_token, dtype);
  const int lanes = slices ? split_lanes_per_row(hidden_size, dtype == OMNI_F32 ? 4 : 2, slices) : 0;
  float *partial_a = nullptr, *partial_s = nullptr;
  if (lanes) {
    partial_a = (float*)w;             w += up256(slices * P * 4);
    partial_s = (float*)w;             w += up256(slices * P * 4);
  }
  hipStream_t s = (hipStream_t)stream;
  // one counting pass: beside the token pass; two: on their own, in front of it
  SortPass pass;
  const bool beside = schedule_single_pass(indices, offsets, pair_ids, token_ids, num_tokens, num_experts_per_token, num_experts, w, &pass);
  if (!beside)
    if (int e = omni_schedule(indices, offsets, pair_ids, token_ids, num_tokens, num_experts_per_token, num_experts, w, stream)) return e;
  const TokenPass p{(const uint8_t*)x, (const uint8_t*)dy, (const uint8_t*)up_weight, (const uint8_t*)down_weight, routing_weights, indices, scores, (uint8_t*)dx,
                    drouting_weights, ds, coef, partial_a, partial_s, 0, (int)num_tokens, (int)num_tokens, hidden_size, num_experts_per_token,
                    lanes, slices, (uint32_t)num_experts};
  hipError_t err;
#define OMNI_BWD_ARGS p, beside ? &pass : nullptr, dup_weight, ddown_weight, offsets, pair_ids, token_ids, partials, router, s
#define OMNI_BWD_CASE(DT)                                                      \
  do {                                                                         \
    if (nch <= 1) err = launch_expert_bwd<DT, 1, 8>(OMNI_BWD_ARGS);            \
    else if (nch <= 2) err = launch_expert_bwd<DT, 2, 8>(OMNI_BWD_ARGS);       \
    else if (nch <= 4) err = launch_expert_bwd<DT, 4, 4>(OMNI_BWD_ARGS);       \
    else err = launch_expert_bwd<DT, 8, 2>(OMNI_BWD_ARGS);                     \
  } while (0)
  if (dtype == OMNI_BF16) OMNI_BWD_CASE(kBF16);
  else if (dtype == OMNI_F16) OMNI_BWD_CASE(kF16);
  else OMNI_BWD_CASE(kF32);
#undef OMNI_BWD_ARGS
#undef OMNI_BWD_CASE
  return to_code(err);
}

extern "C" OMNI_API int32_t omni_expert_bwd_scores(const void* dy, const void* x, const void* up_weight, const void* down_weight, const void* routing_weights,
                                                   const int32_t* indices, const float* scores, void* dx, void* dup_weight, void* ddown_weight, void* drouting_weights,
                                                   int64_t num_tokens, int32_t hidden_size, int64_t num_experts, int32_t num_experts_per_token, int32_t dtype,
                                                   void* workspace, void* stream) {
  return expert_bwd(dy, x, up_weight, down_weight, routing_weights, indices, scores, dx, dup_weight, ddown_weight, drouting_weights, num_tokens, hidden_size, num_experts,
                    num_experts_per_token, dtype, workspace, stream, nullptr);
}

extern "C" OMNI_API size_t omni_expert_router_bwd_workspace_bytes(int64_t num_tokens, int32_t hidden_size, int64_t num_experts, int32_t num_expert_sqrt,
                                                                  int32_t num_experts_per_token, int32_t dtype) {
  return omni::up256(omni_expert_bwd_workspace_bytes(num_tokens, hidden_size, num_experts, num_experts_per_token, dtype)) +
         omni_router_norm_bwd_workspace_bytes(num_tokens, num_expert_sqrt);
}
extern "C" OMNI_API int32_t omni_expert_router_bwd(const void* dy, const void* x, const void* up_weight, const void* down_weight, const void* gates, const int32_t* indices,
                                                   const float* scores, const void* z, const float* stats, void* dx, void* dup_weight, void* ddown_weight, void* dgates,
                                                   void* dz, int64_t num_tokens, int32_t hidden_size, int64_t num_experts, int32_t num_expert_sqrt,
                                                   int32_t num_experts_per_token, int32_t dtype, int32_t training, int32_t padded, void* workspace, void* stream) {
  using namespace omni;
  if (!workspace) return OMNI_ERR_WORKSPACE;
  RouterPass p;
  void* const sums = (char*)workspace + up256(omni_expert_bwd_workspace_bytes(num_tokens, hidden_size, num_experts, num_experts_per_token, dtype));
  if (int e = router_pass(p, dgates, gates, indices, z, stats, dz, num_tokens, num_expert_sqrt, num_experts_per_token, dtype, training, sums, padded != 0)) return e;
  return expert_bwd(dy, x, up_weight, down_weight, gates, indices, scores, dx, dup_weight, ddown_weight, dgates, num_tokens, hidden_size, num_experts, num_experts_per_token,
                    dtype, workspace, stream, num_tokens ? &p : nullptr);
}

static int32_t swiglu_launch(bool bwd, const void* dout, const void* gate, const void* up, void* out0, void* out1,
                             int64_t num_elements, int32_t dtype, void* stream) {
  using namespace omni;
  if (num_elements < 0) return OMNI_ERR_SHAPE;
  if (dtype != OMNI_BF16 && dtype != OMNI_F16 && dtype != OMNI_F32) return OMNI_ERR_DTYPE;
  const int E = dtype == OMNI_F32 ? 4 : 8;
  if (num_elements % E != 0) return OMNI_ERR_SHAPE;
  if (num_elements == 0) return OMNI_OK;
  if (!gate || !up || !out0 || (bwd && (!dout || !out1))) return OMNI_ERR_NULL;
  const int64_t chunks = num_elements / E;
  const int64_t want = (chunks + 255) / 256;
  dim3 grid((unsigned)(want < 8192 ? want : 8192)), block(256);
  hipStream_t s = (hipStream_t)stream;
  const uint8_t *d = (const uint8_t*)dout, *g = (const uint8_t*)gate, *u = (const uint8_t*)up;
  uint8_t *o0 = (uint8_t*)out0, *o1 = (uint8_t*)out1;
#define OMNI_SWIGLU_CASE(DT)                                                                            \
  do {                                                                                                  \
    if (bwd) hipLaunchKernelGGL((swiglu_kernel<DT, true>), grid, block, 0, s, d, g, u, o0, o1, chunks); \
    else hipLaunchKernelGGL((swiglu_kernel<DT, false>), grid, block, 0, s, d, g, u, o0, o1, chunks);    \
  } while (0)
  if (dtype == OMNI_BF16) OMNI_SWIGLU_CASE(kBF16);
  else if (dtype == OMNI_F16) OMNI_SWIGLU_CASE(kF16);
  else OMNI_SWIGLU_CASE(kF32);
#undef OMNI_SWIGLU_CASE
  return to_code(hipGetLastError());
}

extern "C" OMNI_API int32_t omni_swiglu_fwd(const void* gate, const void* up, void* out, int64_t num_elements, int32_t dtype,
                                            void* stream) {
  return swiglu_launch(false, nullptr, gate, up, out, nullptr, num_elements, dtype, stream);
}

extern "C" OMNI_API int32_t omni_swiglu_bwd(const void* dout, const void* gate, const void* up, void* dgate, void* dup,
                                            int64_t num_elements, int32_t dtype, void* stream) {
  return swiglu_launch(true, dout, gate, up, dgate, dup, num_elements, dtype, stream);
}
