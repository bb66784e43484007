// Fused atomic-expert forward for gfx950:
//     y[t,:] = sum_j silu(<x[t,:], U[id[t,j],:]>) * g[t,j] * V[id[t,j],:]
// replacing the reference's schedule + two Triton kernels + fp32 score buffer
// (omni_moe/ops/triton/omni_expert.py:8-168, 920-992) with one launch.
//
// Token-resident gather ("gather" algorithm): one 64-lane wave owns one token.
// The token's row of x stays in registers (16 B per lane per 1 KiB of row), each
// selected expert's up row and down row is fetched with one fully coalesced
// 128-bit load per lane per 1 KiB, the dot product is reduced across the wave,
// and the gate-weighted down rows accumulate in fp32 registers.  Nothing but y
// is written: no score buffer, no atomics, and the summation order is fixed
// (slot 0..k-1), so results are run-to-run identical.
//
// Expert-centric variant ("segment" algorithm), the reference's own organisation
// (omni_expert.py:8-168): the pairs are first grouped by expert (omni_schedule), then
//   A. waves walk the sorted pair list, 16 consecutive pairs each -- so a popular expert's
//      segment is spread over many waves and an unpopular one costs one short visit -- gather
//      the pair's x row and its expert's up row (which repeats along a segment and therefore
//      hits in cache), and write the coefficient silu(<x,u>)*g of the pair;
//   B. a token-resident pass accumulates coefficient * down row into y, in slot order.
// No atomics, same fixed summation order as the gather algorithm, hence identical results;
// it moves the same rows plus the schedule and a [T,k] fp32 coefficient buffer, and exists so
// that the two organisations can be measured side by side.
#include "common.h"
#include "expert_split.h"
#include "omni_moe_hip.h"
#include "rows.h"

// gemm.hip: c[T, 2N] = [round(v) | round(v - round(v))], v = silu(x W^T) * gate
int omni_gemm_gated(const void* x, const void* w, const float* gate, void* c, int64_t T, int64_t N, int64_t K, int dtype, void* stream);

namespace omni {

constexpr int kTokensPerBlock = 4;   // one wave each

// NCH = 16-byte chunks of a row per lane (row bytes / 1024, rounded up);
// G   = experts fetched per batch (their 2*G*NCH loads are all in flight at once).
// kAdd: the layer's final add as well: y holds the shared MLP's rounded rows (parts = NULL), or the K splits' fp32 sums of them are in
// parts [splits][tokens][hidden]; both terms are rounded, then their sum.
// scores: NULL, or [tokens][top_k] where <x, u> of every pair goes, for a backward pass.
struct GatherAdd { const float* parts; int splits; float* scores; };
// W waves share a token's slots, each a run of them, and add up in wave order: with fewer tokens than the chip holds waves a token's batches of G slots are
// a chain of waits.
template <int DT, int NCH, int G, bool kAdd = false, int W = 1>
__global__ __launch_bounds__(kTokensPerBlock* kWave, 2) void expert_gather_kernel(
    const uint8_t* __restrict__ x, const uint8_t* __restrict__ up, const uint8_t* __restrict__ down,
    const void* __restrict__ gates, const int32_t* __restrict__ ids, uint8_t* __restrict__ y,
    int num_tokens, int hidden, int top_k, uint32_t num_experts, GatherAdd add) {
  constexpr int E = Row16<DT>::kElems;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), share = wave % W;
  const int t = __builtin_amdgcn_readfirstlane(blockIdx.x * (kTokensPerBlock / W) + wave / W);
  if (W == 1 && t >= num_tokens) return;
  const int per = W == 1 ? top_k : (top_k + W - 1) / W;
  const int first = share * per, last = t >= num_tokens ? first : min(first + per, top_k);
  const int64_t row_bytes = int64_t(hidden) * (16 / E);

  bool live[NCH];
  int64_t off[NCH];                    // byte offset of this lane's chunk c inside a row
  u32x4_t xr[NCH];
  float acc[NCH][E];
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    live[c] = (c * kWave + lane) * E < hidden && (W == 1 || t < num_tokens);
    off[c] = int64_t(c * kWave + lane) * 16;
    xr[c] = live[c] ? *(const u32x4_t*)(x + t * row_bytes + off[c]) : u32x4_t{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < E; ++i) acc[c][i] = 0.f;
  }

  const int32_t* my_ids = ids + int64_t(t) * top_k;
  for (int j0 = first; j0 < last; j0 += G) {
    int e[G];
    float g[G];
    bool live_slot[G];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int j = min(j0 + i, last - 1);          // always a valid slot: no branch around the loads
      const int id = my_ids[j];
      const float gate = Elem<DT>::load(gates, int64_t(t) * top_k + j);
      // a slot of another wave or past k, or an id outside the table, contributes nothing
      const bool ok = (j0 + i < last) && (uint32_t)id < num_experts;
      e[i] = ok ? id : 0;
      g[i] = ok ? gate : 0.f;
      live_slot[i] = ok;
    }
    u32x4_t ur[G][NCH], vr[G][NCH];
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
      for (int c = 0; c < NCH; ++c)
        ur[i][c] = live[c] ? *(const u32x4_t*)(up + e[i] * row_bytes + off[c]) : u32x4_t{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
      for (int c = 0; c < NCH; ++c)
        vr[i][c] = live[c] ? *(const u32x4_t*)(down + e[i] * row_bytes + off[c]) : u32x4_t{0, 0, 0, 0};

    float s[G];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      float p = 0.f;
#pragma unroll
      for (int c = 0; c < NCH; ++c) p = dot16<DT>(xr[c], ur[i][c], p);
      s[i] = p;
    }
#pragma unroll
    for (int i = 0; i < G; ++i) s[i] = wave_sum(s[i]);
    if (!kAdd && add.scores) {
      float mine = 0.f;
#pragma unroll
      for (int i = 0; i < G; ++i) mine = lane == i ? s[i] : mine;
      if (lane < G && j0 + lane < last) add.scores[int64_t(t) * top_k + j0 + lane] = mine;
    }
#pragma unroll
    for (int i = 0; i < G; ++i) {
      if (!live_slot[i]) continue;                  // not even 0 * row: the stand-in row may hold Inf or NaN
      const float coef = silu_f32(s[i]) * g[i];
#pragma unroll
      for (int c = 0; c < NCH; ++c) axpy16<DT>(coef, vr[i][c], acc[c]);
    }
  }

  if constexpr (W > 1) {
    __shared__ __align__(16) float sums[kTokensPerBlock][NCH * kWave * E];
    if (share > 0)
#pragma unroll
      for (int c = 0; c < NCH; ++c)
#pragma unroll
        for (int q = 0; q < E; q += 4) *(f32x4_t*)(&sums[wave][(c * kWave + lane) * E + q]) = f32x4_t{acc[c][q], acc[c][q + 1], acc[c][q + 2], acc[c][q + 3]};
    __syncthreads();
    if (share > 0 || t >= num_tokens) return;
#pragma unroll
    for (int w = 1; w < W; ++w)
#pragma unroll
      for (int c = 0; c < NCH; ++c)
#pragma unroll
        for (int q = 0; q < E; q += 4) {
          const f32x4_t o = *(const f32x4_t*)(&sums[wave + w][(c * kWave + lane) * E + q]);
#pragma unroll
          for (int z = 0; z < 4; ++z) acc[c][q + z] += o[z];
        }
  }
#pragma unroll
  for (int c = 0; c < NCH; ++c)
    if (live[c]) {
      u32x4_t out = pack16<DT>(acc[c]);
      if constexpr (kAdd) {
        float e[E], m[E];
        unpack16<DT>(out, e);
        if (add.parts) {
#pragma unroll
          for (int i = 0; i < E; ++i) m[i] = 0.f;
          const float* at = add.parts + int64_t(t) * hidden + (c * kWave + lane) * E;
          for (int s = 0; s < add.splits; ++s, at += int64_t(num_tokens) * hidden)
#pragma unroll
            for (int q = 0; q < E; q += 4) {
              const f32x4_t p = *(const f32x4_t*)(at + q);
#pragma unroll
              for (int z = 0; z < 4; ++z) m[q + z] += p[z];
            }
          unpack16<DT>(pack16<DT>(m), m);
        } else {
          unpack16<DT>(*(const u32x4_t*)(y + t * row_bytes + off[c]), m);
        }
#pragma unroll
        for (int i = 0; i < E; ++i) m[i] += e[i];
        out = pack16<DT>(m);
      }
      *(u32x4_t*)(y + t * row_bytes + off[c]) = out;
    }
}

// Waves to a token: while the chip has room for them (2048 at these register counts) and a token's slots are several batches.  Time with 2 and 4 over 1,
// bf16, 4096 experts (65536: the same within 5 %), at 200 / 400 / 613 / 1000 / 1500 tokens:
//   two batches   hidden 256 k 32, 1024 k 16, 2048 k 8:   2: 0.64-0.72 / 0.64-0.74 / 0.81-0.95 / 0.81-0.94 / 0.8-1.03   4: 0.6-0.7 / 0.72-0.82 / 0.86-1.09 / 1.04-1.08
//   four and more hidden 1024 k 32, 2048 k 16 and 32, 4096: 2: 0.60-0.66 / 0.74-0.84 / 0.83-0.97 / 0.88-1.03 / 1.0   4: 0.40-0.58 / 0.63-0.84 / 0.78-1.0 / 0.87-1.08 / 1.0
//   one batch: 1.0-1.25 and 1.0-1.8
// Only where AUTO leads here (`shared` of the launches).  Asked for by name the gather algorithm's sums are those of the segment algorithm, slot by slot, and
// so they are where the layer ends with this kernel.
static inline int gather_waves(int64_t T, int k, int batch) {
  const int batches = (k + batch - 1) / batch;
  return batches < 2 || T > 1024 ? 1 : batches >= 4 && T <= 512 ? 4 : 2;
}
template <int DT, int NCH, int G>
static hipError_t launch_gather(const void* x, const void* up, const void* down, const void* gates,
                                const int32_t* ids, void* y, float* scores, bool shared, int64_t T, int H, int k, int64_t N, hipStream_t s) {
  if (T == 0) return hipSuccess;
  auto go = [&](auto waves) {
    constexpr int W = decltype(waves)::value, kTokens = kTokensPerBlock / W;
    hipLaunchKernelGGL((expert_gather_kernel<DT, NCH, G, false, W>), dim3((unsigned)((T + kTokens - 1) / kTokens)), dim3(kTokensPerBlock * kWave), 0, s, (const uint8_t*)x,
                       (const uint8_t*)up, (const uint8_t*)down, gates, ids, (uint8_t*)y, (int)T, H, k, (uint32_t)N, GatherAdd{nullptr, 0, scores});
    return hipGetLastError();
  };
  switch (shared ? gather_waves(T, k, G) : 1) {
    case 4: return go(std::integral_constant<int, 4>{});
    case 2: return go(std::integral_constant<int, 2>{});
    default: return go(std::integral_constant<int, 1>{});
  }
}

// The gather algorithm (rows of at most 8 KiB) with the layer's final add
hipError_t launch_gather_add(const void* x, const void* up, const void* down, const void* gates, const int32_t* ids, void* y, const float* parts, int splits, bool shared, int64_t T,
                             int H, int k, int64_t N, int dtype, hipStream_t s) {
  auto launch = [&](auto dt, auto nch, auto batch, auto waves) {
    constexpr int W = decltype(waves)::value, kTokens = kTokensPerBlock / W;
    hipLaunchKernelGGL((expert_gather_kernel<decltype(dt)::value, decltype(nch)::value, decltype(batch)::value, true, W>), dim3((unsigned)((T + kTokens - 1) / kTokens)),
                       dim3(kTokensPerBlock * kWave), 0, s, (const uint8_t*)x, (const uint8_t*)up, (const uint8_t*)down, gates, ids, (uint8_t*)y, (int)T, H, k, (uint32_t)N,
                       GatherAdd{parts, splits, nullptr});
    return hipGetLastError();
  };
  auto go = [&](auto dt, auto nch, auto batch) {
    switch (shared ? gather_waves(T, k, decltype(batch)::value) : 1) {
      case 4: return launch(dt, nch, batch, std::integral_constant<int, 4>{});
      case 2: return launch(dt, nch, batch, std::integral_constant<int, 2>{});
      default: return launch(dt, nch, batch, std::integral_constant<int, 1>{});
    }
  };
  auto by_row = [&](auto dt) {
    constexpr int E = Row16<decltype(dt)::value>::kElems;
    const int nch = (H + kWave * E - 1) / (kWave * E);
    if (nch <= 1) return go(dt, std::integral_constant<int, 1>{}, std::integral_constant<int, 16>{});
    if (nch <= 2) return go(dt, std::integral_constant<int, 2>{}, std::integral_constant<int, 8>{});
    if (nch <= 4) return go(dt, std::integral_constant<int, 4>{}, std::integral_constant<int, 4>{});
    return go(dt, std::integral_constant<int, 8>{}, std::integral_constant<int, 2>{});
  };
  return dtype == kBF16 ? by_row(std::integral_constant<int, kBF16>{}) : dtype == kF16 ? by_row(std::integral_constant<int, kF16>{}) : by_row(std::integral_constant<int, kF32>{});
}

template <int DT>
static int expert_gather_dispatch(const void* x, const void* up, const void* down, const void* gates,
                                  const int32_t* ids, void* y, int64_t T, int H, int k, int64_t N, hipStream_t s, float* scores = nullptr, bool shared = false) {
  constexpr int E = Row16<DT>::kElems;
  if (H % E != 0) return OMNI_ERR_SHAPE;              // rows must be 16-byte multiples
  const int nch = (H + kWave * E - 1) / (kWave * E);
  hipError_t err;
  if (nch <= 1) err = launch_gather<DT, 1, 16>(x, up, down, gates, ids, y, scores, shared, T, H, k, N, s);
  else if (nch <= 2) err = launch_gather<DT, 2, 8>(x, up, down, gates, ids, y, scores, shared, T, H, k, N, s);
  else if (nch <= 4) err = launch_gather<DT, 4, 4>(x, up, down, gates, ids, y, scores, shared, T, H, k, N, s);
  else if (nch <= 8) err = launch_gather<DT, 8, 2>(x, up, down, gates, ids, y, scores, shared, T, H, k, N, s);
  else return OMNI_ERR_UNSUPPORTED;
  return err == hipSuccess ? OMNI_OK : OMNI_ERR_HIP_BASE + (int)err;
}

// The gather algorithm alone, for a layer whose schedules must agree on it
int expert_gather_f32(const void* x, const void* up, const void* down, const void* gates, const int32_t* ids, void* y, bool shared, int64_t T, int H, int k, int64_t N, hipStream_t s) {
  return expert_gather_dispatch<kF32>(x, up, down, gates, ids, y, T, H, k, N, s, nullptr, shared);
}

// ---- expert-centric variant -------------------------------------------------------------------
constexpr int kPairsPerWave = 16;

template <int DT, int NCH>
__global__ __launch_bounds__(256, 2) void expert_segment_scores_kernel(
    const uint8_t* __restrict__ x, const uint8_t* __restrict__ up, const void* __restrict__ gates,
    const int32_t* __restrict__ ids, const int32_t* __restrict__ sorted_pair_ids, const int32_t* __restrict__ offsets,
    float* __restrict__ coef, int hidden, int top_k, int64_t num_experts) {
  constexpr int E = Row16<DT>::kElems;
  constexpr int G = (NCH <= 2) ? 8 : (NCH <= 4 ? 4 : 2);       // pairs whose rows are in flight together
  const int lane = lane_id();
  const int num_valid = offsets[num_experts];                   // pairs with an id inside the table
  const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int pos0 = wave * kPairsPerWave;
  if (pos0 >= num_valid) return;
  const int64_t row_bytes = int64_t(hidden) * (16 / E);
  bool live[NCH];
  int64_t off[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    live[c] = (c * kWave + lane) * E < hidden;
    off[c] = int64_t(c * kWave + lane) * 16;
  }
  for (int g0 = 0; g0 < kPairsPerWave; g0 += G) {
    int pid[G];
    bool ok[G];
    u32x4_t xr[G][NCH], ur[G][NCH];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int pos = pos0 + g0 + i;
      ok[i] = pos < num_valid;
      pid[i] = sorted_pair_ids[ok[i] ? pos : pos0];
      const int t = pid[i] / top_k, e = ids[pid[i]];
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        xr[i][c] = live[c] ? *(const u32x4_t*)(x + t * row_bytes + off[c]) : u32x4_t{0, 0, 0, 0};
        ur[i][c] = live[c] ? *(const u32x4_t*)(up + e * row_bytes + off[c]) : u32x4_t{0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int i = 0; i < G; ++i) {
      float p = 0.f;
#pragma unroll
      for (int c = 0; c < NCH; ++c) p = dot16<DT>(xr[i][c], ur[i][c], p);
      const float sdot = wave_sum(p);
      if (ok[i] && lane == 0) coef[pid[i]] = silu_f32(sdot) * Elem<DT>::load(gates, pid[i]);
    }
  }
}

// y[t] = sum_j coef[t,j] * down[id[t,j]] in slot order; coef comes from the scores pass.
template <int DT, int NCH, int G>
__global__ __launch_bounds__(kTokensPerBlock* kWave, 2) void expert_accumulate_kernel(
    const uint8_t* __restrict__ down, const float* __restrict__ coef, const int32_t* __restrict__ ids,
    uint8_t* __restrict__ y, int num_tokens, int hidden, int top_k, uint32_t num_experts) {
  constexpr int E = Row16<DT>::kElems;
  const int lane = lane_id();
  const int t = __builtin_amdgcn_readfirstlane(blockIdx.x * kTokensPerBlock + (threadIdx.x >> 6));
  if (t >= num_tokens) return;
  const int64_t row_bytes = int64_t(hidden) * (16 / E);
  bool live[NCH];
  int64_t off[NCH];
  float acc[NCH][E];
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    live[c] = (c * kWave + lane) * E < hidden;
    off[c] = int64_t(c * kWave + lane) * 16;
#pragma unroll
    for (int i = 0; i < E; ++i) acc[c][i] = 0.f;
  }
  for (int j0 = 0; j0 < top_k; j0 += G) {
    float cf[G];
    bool used[G];
    u32x4_t vr[G][NCH];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int j = min(j0 + i, top_k - 1);
      const int id = ids[int64_t(t) * top_k + j];
      const bool ok = (j0 + i < top_k) && (uint32_t)id < num_experts;
      used[i] = ok;
      cf[i] = ok ? coef[int64_t(t) * top_k + j] : 0.f;
      const int e = ok ? id : 0;
#pragma unroll
      for (int c = 0; c < NCH; ++c)
        vr[i][c] = live[c] ? *(const u32x4_t*)(down + e * row_bytes + off[c]) : u32x4_t{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < G; ++i) {
      if (!used[i]) continue;
#pragma unroll
      for (int c = 0; c < NCH; ++c) axpy16<DT>(cf[i], vr[i][c], acc[c]);
    }
  }
#pragma unroll
  for (int c = 0; c < NCH; ++c)
    if (live[c]) *(u32x4_t*)(y + t * row_bytes + off[c]) = pack16<DT>(acc[c]);
}

static inline size_t align256(size_t v) { return (v + 255) / 256 * 256; }

template <int DT, int NCH, int G>
static hipError_t launch_segment(const void* x, const void* up, const void* down, const void* gates, const int32_t* ids,
                                 const int32_t* sorted_pair_ids, const int32_t* offsets, float* coef, void* y, int64_t T,
                                 int H, int k, int64_t N, hipStream_t s) {
  const int64_t P = T * k;
  const unsigned waves = (unsigned)((P + kPairsPerWave - 1) / kPairsPerWave);
  hipLaunchKernelGGL((expert_segment_scores_kernel<DT, NCH>), dim3((waves + 3) / 4), dim3(256), 0, s, (const uint8_t*)x,
                     (const uint8_t*)up, gates, ids, sorted_pair_ids, offsets, coef, H, k, N);
  hipLaunchKernelGGL((expert_accumulate_kernel<DT, NCH, G>), dim3((unsigned)((T + kTokensPerBlock - 1) / kTokensPerBlock)),
                     dim3(kTokensPerBlock * kWave), 0, s, (const uint8_t*)down, coef, ids, (uint8_t*)y, (int)T, H, k, (uint32_t)N);
  return hipGetLastError();
}

// workspace: offsets [N+1] | sorted pair ids [P] | coefficients [P] f32 | schedule workspace
template <int DT>
static int expert_segment_dispatch(const void* x, const void* up, const void* down, const void* gates, const int32_t* ids,
                                   void* y, int64_t T, int H, int k, int64_t N, void* workspace, hipStream_t s) {
  constexpr int E = Row16<DT>::kElems;
  if (H % E != 0) return OMNI_ERR_SHAPE;
  if (T == 0) return OMNI_OK;
  if (k == 0) return expert_gather_dispatch<DT>(x, up, down, gates, ids, y, T, H, k, N, s);   // writes zeros
  if (!workspace) return OMNI_ERR_WORKSPACE;
  const int64_t P = T * k;
  char* w = (char*)workspace;
  int32_t* offsets = (int32_t*)w;          w += align256((size_t)(N + 1) * 4);
  int32_t* sorted_pair_ids = (int32_t*)w;  w += align256((size_t)P * 4);
  float* coef = (float*)w;                 w += align256((size_t)P * 4);
  if (int e = omni_schedule(ids, offsets, sorted_pair_ids, nullptr, T, k, N, w, s)) return e;
  const int nch = (H + kWave * E - 1) / (kWave * E);
  hipError_t err;
  if (nch <= 1) err = launch_segment<DT, 1, 16>(x, up, down, gates, ids, sorted_pair_ids, offsets, coef, y, T, H, k, N, s);
  else if (nch <= 2) err = launch_segment<DT, 2, 8>(x, up, down, gates, ids, sorted_pair_ids, offsets, coef, y, T, H, k, N, s);
  else if (nch <= 4) err = launch_segment<DT, 4, 4>(x, up, down, gates, ids, sorted_pair_ids, offsets, coef, y, T, H, k, N, s);
  else if (nch <= 8) err = launch_segment<DT, 8, 2>(x, up, down, gates, ids, sorted_pair_ids, offsets, coef, y, T, H, k, N, s);
  else return OMNI_ERR_UNSUPPORTED;
  return err == hipSuccess ? OMNI_OK : OMNI_ERR_HIP_BASE + (int)err;
}

// ---- hidden-split variant ("split" algorithm) ------------------------------------------------
// For tables that fit the chip's caches but not one XCD's 4 MiB L2 (16 MiB at N = 4096,
// H = 1024): the hidden dimension is cut into 8 slices and slice s is only ever touched by
// blocks with blockIdx % 8 == s, which the dispatcher places on XCD s -- or into 4, each for
// the blocks of two XCDs (split_slices).  With 8 an XCD then needs
// N * H/8 elements of each table -- 1 MiB each in that example, 2 with 4 -- and serves every table row
// from its own L2 instead of pulling three quarters of them over the fabric.  The price is a
// cross-slice reduction of the pair scores ([slices][T][k] floats):
//   A. block (token group, slice): partial dot products <x[t, slice], up[id, slice]> for the k pairs
//      of each of its tokens -> partial[slice][t][j];
//   B. block (token group, slice): coefficient silu(sum over slices, in slice order) * gate, then
//      y[t, slice] = sum_j coefficient_j * down[id_j, slice].
// A row slice is up to LPR lanes of 16 bytes, LPR a power of two (64 / LPR tokens to a wave).  Fixed summation
// order, no atomics; results agree with the gather algorithm to fp32 rounding of the dot product.
template <int DT, int LPR, int S, bool RAGGED, bool SMALL>
__global__ __launch_bounds__(kTokensPerBlock* kWave) void expert_split_dots_kernel(
    const uint8_t* __restrict__ x, const uint8_t* __restrict__ up, const int32_t* __restrict__ ids,
    float* __restrict__ partial, int num_tokens, int hidden, int top_k, uint32_t num_experts, int lanes, int col_block) {
  split_dots_block<DT, LPR, S, RAGGED, SMALL, kTokensPerBlock>(x, up, ids, partial, num_tokens, hidden, top_k, num_experts, lanes, col_block, (int)blockIdx.x);
}

// The coefficient of a pair: the sum of the slice partials in slice order (WIDE: column block by column block), silu, gate.
// kScores: the dot products go to `scores` as well, for a backward pass.
template <int DT, int S, bool WIDE, bool kScores, class Off>
struct SplitCoefficient {
  const void* gates;
  const float* partial;
  float* scores;
  int num_tokens, top_k, col_blocks;
  bool writes;                                                   // the block that leaves the scores
  float part[S], gate;
  bool use;
  Off at;
  __device__ __forceinline__ void request(bool there, int t, Off pair, int j, bool inside) {
    use = there && inside;
    at = pair;
#pragma unroll
    for (int sl = 0; sl < S; ++sl) part[sl] = partial[(Off(sl) * num_tokens + t) * top_k + j];
    gate = Elem<DT>::load(gates, pair);
    if constexpr (WIDE) {
      float sum = 0.f;
#pragma unroll
      for (int sl = 0; sl < S; ++sl) sum += part[sl];
      for (int cb = 1; cb < col_blocks; ++cb)
#pragma unroll
        for (int sl = 0; sl < S; ++sl) sum += partial[((Off(cb) * S + sl) * num_tokens + t) * top_k + j];
      part[0] = sum;
    }
  }
  __device__ __forceinline__ float value() {
    float s = part[0];
    if constexpr (!WIDE)
#pragma unroll
      for (int sl = 1; sl < S; ++sl) s += part[sl];
    if (kScores && use && writes) scores[at] = s;
    return use ? silu_f32(s) * gate : 0.f;
  }
};
template <int DT, int LPR, int S, bool RAGGED, bool WIDE, bool SMALL, bool kScores>
__global__ __launch_bounds__(kTokensPerBlock* kWave) void expert_split_accumulate_kernel(
    const uint8_t* __restrict__ down, const void* __restrict__ gates, const int32_t* __restrict__ ids,
    const float* __restrict__ partial, uint8_t* __restrict__ y, float* __restrict__ scores, int num_tokens, int hidden, int top_k, uint32_t num_experts,
    int lanes, int col_block_arg, int col_blocks_arg) {
  using Off = typename SplitOff<SMALL>::type;
  const int col_block = WIDE ? col_block_arg : 0;
  SplitCoefficient<DT, S, WIDE, kScores, Off> pair{gates, partial, scores, num_tokens, top_k, col_blocks_arg, blockIdx.x % S == 0 && col_block == 0};
  split_accumulate_block<DT, LPR, S, RAGGED, SMALL, kTokensPerBlock>(down, ids, y, num_tokens, hidden, top_k, num_experts, lanes, col_block, (int)blockIdx.x, pair);
}

template <int DT, int LPR, int S, bool RAGGED, bool SMALL>
static hipError_t launch_split_as(const void* x, const void* up, const void* down, const void* gates, const int32_t* ids,
                                  float* partial, void* y, float* scores, int64_t T, int H, int k, int64_t N, int lanes, int col_blocks, hipStream_t s) {
  constexpr int kPerBlock = kTokensPerBlock * (kWave / LPR);       // tokens per block
  const unsigned blocks = (unsigned)split_blocks(T, kPerBlock, S);
  for (int cb = 0; cb < col_blocks; ++cb)                            // all partial dot products first: a coefficient needs the whole row
    hipLaunchKernelGGL((expert_split_dots_kernel<DT, LPR, S, RAGGED, SMALL>), dim3(blocks), dim3(kTokensPerBlock * kWave), 0, s, (const uint8_t*)x,
                       (const uint8_t*)up, ids, partial, (int)T, H, k, (uint32_t)N, lanes, cb);
  auto accumulate = [&](auto kernel, int cb) {
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kTokensPerBlock * kWave), 0, s, (const uint8_t*)down, gates, ids, partial, (uint8_t*)y, scores, (int)T, H, k, (uint32_t)N, lanes, cb,
                       col_blocks);
  };
  if (col_blocks == 1) {
    if (scores) accumulate(expert_split_accumulate_kernel<DT, LPR, S, RAGGED, false, SMALL, true>, 0);
    else accumulate(expert_split_accumulate_kernel<DT, LPR, S, RAGGED, false, SMALL, false>, 0);
    return hipGetLastError();
  }
  if constexpr (S == kSlices && !RAGGED)                             // rows of several column blocks are cut into eight slices each
    for (int cb = 0; cb < col_blocks; ++cb) {
      if (scores) accumulate(expert_split_accumulate_kernel<DT, LPR, S, false, true, SMALL, true>, cb);
      else accumulate(expert_split_accumulate_kernel<DT, LPR, S, false, true, SMALL, false>, cb);
    }
  return hipGetLastError();
}

// workspace: partial dot products [slices * column blocks][T][k] f32
template <int DT>
static int expert_split_dispatch(const void* x, const void* up, const void* down, const void* gates, const int32_t* ids,
                                 void* y, float* scores, int64_t T, int H, int k, int64_t N, void* workspace, hipStream_t s) {
  constexpr int es = DT == kF32 ? 4 : 2;
  const SplitCut cut = split_cut(H, N, es);
  if (cut.col_blocks == 0 || k > 2 * kWave) return OMNI_ERR_UNSUPPORTED;
  if (T == 0) return OMNI_OK;
  if (k == 0) return expert_gather_dispatch<DT>(x, up, down, gates, ids, y, T, H, k, N, s);   // writes zeros
  if (!workspace) return OMNI_ERR_WORKSPACE;
  float* partial = (float*)workspace;
  const bool small = split_offsets_small(up, down, T, H, k, N, cut.col_blocks, es);
  const hipError_t err = split_dispatch(cut.lanes, cut.slices, [&](auto group, auto s_tag, auto ragged) {
    constexpr int LPR = decltype(group)::value, S = decltype(s_tag)::value;
    constexpr bool RAGGED = decltype(ragged)::value;
    return small ? launch_split_as<DT, LPR, S, RAGGED, true>(x, up, down, gates, ids, partial, y, scores, T, H, k, N, cut.lanes, cut.col_blocks, s)
                 : launch_split_as<DT, LPR, S, RAGGED, false>(x, up, down, gates, ids, partial, y, scores, T, H, k, N, cut.lanes, cut.col_blocks, s);
  });
  return err == hipSuccess ? OMNI_OK : OMNI_ERR_HIP_BASE + (int)err;
}

// ---- dense variant ("dense" algorithm) --------------------------------------------------------
// The regime of the reference's group path (omni_scheduler.py:58,103-226; omni_expert.py:171-372): so few experts
// that each serves hundreds of tokens (T*k/N > 256).  The reference looks for 16 experts with identical token lists
// and runs those through tl.dot; here the whole op becomes two MFMA GEMMs over ALL experts, which at this density
// cost less than fetching 2k rows per token:
//   G[t, e]  = sum of the gates of token t's slots that name expert e (0 elsewhere)      gate matrix, fp32
//   C        = silu(x U^T) * G, kept as a 16-bit head and a 16-bit remainder [T, 2N]      GEMM with a gate epilogue
//   y        = [C_head | C_rem] [V^T | V^T]^T                                             GEMM over K = 2N
// silu and the gate product are fp32, C carries 16 significant bits, sums are fp32: results agree with the gather
// algorithm to a few units of fp32 rounding of the coefficients.  Duplicate slots add their gates in slot order.
constexpr int kDenseMaxExperts = 2048;

// One wave per token: the token's row of G is built in LDS (slots in order, by one lane) and written out whole.
__global__ __launch_bounds__(256) void dense_gate_rows_kernel(const void* __restrict__ gates, const int32_t* __restrict__ ids,
                                                              float* __restrict__ gate_matrix, int num_tokens, int top_k,
                                                              int num_experts, int dtype) {
  extern __shared__ float rows[];                                  // [4 waves][num_experts]
  const int lane = lane_id(), wave = threadIdx.x >> 6;
  const int t = blockIdx.x * 4 + wave;
  if (t >= num_tokens) return;
  float* row = rows + wave * num_experts;
  for (int e = lane; e < num_experts; e += kWave) row[e] = 0.f;
  __builtin_amdgcn_wave_barrier();
  if (lane == 0) {
    for (int j = 0; j < top_k; ++j) {
      const int id = ids[(int64_t)t * top_k + j];
      if ((uint32_t)id < (uint32_t)num_experts) {
        const float g = dtype == OMNI_BF16 ? Elem<kBF16>::load(gates, (int64_t)t * top_k + j) : Elem<kF16>::load(gates, (int64_t)t * top_k + j);
        row[id] += g;
      }
    }
  }
  __builtin_amdgcn_wave_barrier();
  for (int e = lane; e < num_experts; e += kWave) gate_matrix[(int64_t)t * num_experts + e] = row[e];
}

// vt2[h, c] = v[c % N, h] for c < 2N: the down table transposed, twice side by side (K-contiguous operand of the second GEMM)
__global__ __launch_bounds__(256) void dense_transpose_kernel(const uint16_t* __restrict__ v, uint16_t* __restrict__ vt2, int num_experts, int hidden) {
  __shared__ uint16_t tile[64][66];
  const int e0 = blockIdx.x * 64, h0 = blockIdx.y * 64;
  for (int i = threadIdx.x; i < 64 * 64; i += 256) {
    const int e = i / 64, h = i % 64;
    tile[e][h] = (e0 + e < num_experts && h0 + h < hidden) ? v[(int64_t)(e0 + e) * hidden + h0 + h] : (uint16_t)0;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 64 * 64; i += 256) {
    const int h = i / 64, e = i % 64;
    if (e0 + e < num_experts && h0 + h < hidden) {
      const uint16_t x = tile[e][h];
      vt2[(int64_t)(h0 + h) * 2 * num_experts + e0 + e] = x;
      vt2[(int64_t)(h0 + h) * 2 * num_experts + num_experts + e0 + e] = x;
    }
  }
}

static inline bool dense_covers(int64_t T, int H, int64_t N, int k, int dtype) {
  return dtype != OMNI_F32 && N % 32 == 0 && N <= kDenseMaxExperts && H % 64 == 0 && H % 8 == 0 && k > 0 && T > 0;
}

// workspace: gate matrix [T, N] f32 | coefficients [T, 2N] | transposed down table [H, 2N]
static inline size_t dense_workspace_bytes(int64_t T, int H, int64_t N) {
  return align256((size_t)T * N * 4) + align256((size_t)T * 2 * N * 2) + align256((size_t)H * 2 * N * 2);
}

static int expert_dense_dispatch(const void* x, const void* up, const void* down, const void* gates, const int32_t* ids, void* y,
                                 int64_t T, int H, int k, int64_t N, int dtype, void* workspace, hipStream_t s) {
  if (T == 0) return OMNI_OK;
  if (!dense_covers(T, H, N, k, dtype)) return OMNI_ERR_UNSUPPORTED;
  if (!workspace) return OMNI_ERR_WORKSPACE;
  char* w = (char*)workspace;
  float* gate_matrix = (float*)w;  w += align256((size_t)T * N * 4);
  void* coef = w;                  w += align256((size_t)T * 2 * N * 2);
  uint16_t* vt2 = (uint16_t*)w;
  hipLaunchKernelGGL(dense_gate_rows_kernel, dim3((unsigned)((T + 3) / 4)), dim3(256), (size_t)4 * N * 4, s, gates, ids, gate_matrix, (int)T, k, (int)N, dtype);
  hipLaunchKernelGGL(dense_transpose_kernel, dim3((unsigned)((N + 63) / 64), (unsigned)((H + 63) / 64)), dim3(256), 0, s,
                     (const uint16_t*)down, vt2, (int)N, H);
  if (hipError_t e = hipGetLastError(); e != hipSuccess) return OMNI_ERR_HIP_BASE + (int)e;
  if (int e = omni_gemm_gated(x, up, gate_matrix, coef, T, N, H, dtype, s)) return e;
  return omni_linear_fwd(coef, vt2, nullptr, y, T, (int32_t)(2 * N), H, dtype, s);
}

// What OMNI_EXPERT_ALGO_AUTO runs, from the sizes alone.  The split algorithm gives every XCD a part of each table row, so it pays while that part of the
// tables stays near its caches (its 4 MiB L2 and its part of the memory-side cache) and where what the gather algorithm moves outweighs its second launch.
// Rows up to 1 KiB the gather kernel fetches with half of its lanes or less, so there the number of tokens decides (1024: its waves share a token's slots up to
// there); longer rows go by the bytes that all pairs name ("moved": pairs x row bytes).  A row that is no power of two leaves lanes of a slice idle (`whole`), few
// pairs to a token leave part of a batch of 8 empty, and a table of at most 2 MiB ("little") every L2 holds whole.  More tokens never turn it back to gather.
// Time of split over time of gather, bf16, ids uniform over the experts, tables of 1 to 256 MB each ("table": N x row bytes):
//   rows 512 B    k <= 8: 0.92-1.09 at 1024 tokens, 0.71-0.97 at 1536 to 3000, 0.59-0.88 at 4096, 0.31-0.79 at 32768 and 65536
//                 k 12 to 32 up to 16 MB: 0.80-1.08 at 1536 to 3000, 0.67-0.93 at 4096, 0.51-0.97 beyond; above 16 MB 0.85-1.3
//   rows 1 KiB    k <= 4: 0.71-0.94 at 4096, 0.61-0.91 beyond; k >= 6 up to 64 MB 0.50-0.98, above 0.95-1.13; 1536 to 3000 tokens 0.69-0.98 up to 16 MB, 0.82-1.13 above
//   640 to 896 B  0.65-1.09 up to 16 MB (k 10 1.16); above k 2 0.69-0.92, k 4 0.85-1.11, k 6 and 8 1.04-1.5
//   1.1 to 1.4 KiB  k 2 0.94-1.31; moved >= 64 MB up to 16 MB 0.70-1.0, at 64 MB 1.05-1.3
//   rows 1.5 KiB  moved >= 64 MB: k >= 4 0.49-1.06 up to 64 MB; 32 to 64 MB: k >= 8 0.65-0.95 at 4 and 16 MB, 0.95-1.02 at 64; k 2 0.91-1.26
//   rows 2 KiB    moved >= 64 MB: 0.42-0.95 from 4 to 64 MB, k 4 to 8 over a little table 0.94-1.09, 128 and 256 MB 0.93-1.10; 32 to 64 MB: k 6 0.86-0.94, k 8 0.74-0.95 up to 32 MB
//   rows 2.5 and 3 KiB  k 4 0.93-1.72, k 6 0.71-1.04 from 4 to 64 MB; little tables: k 6 1.06-1.23, k 8 and 12 1.0-1.24 (their backward 0.85-0.92), 16 0.88-1.0, 32 0.83-0.96
//   rows 4 and 8 KiB    moved >= 64 MB: k >= 4 0.34-1.07 from 4 to 64 MB; little tables: k 4 1.2-1.6, k 6 0.93-1.29, k 8 and 12 0.88-1.24, 16 and 32 0.72-1.03; 256 MB: k < 16 0.91-1.16, k >= 16 0.72-1.03
// (the rule's choice takes 0.7 % more than the better of the two on average, over 10 % at 2 % of the 3032 points of these rows)
// A skewed router (few live experts) moves every figure towards the split algorithm; the caller who knows says so.
int resolve_algo(int algo, int64_t T, int H, int64_t N, int k, int dtype) {
  if (algo != OMNI_EXPERT_ALGO_AUTO) return algo;
  // The dense algorithm is never chosen here: it multiplies every token by every table row, so one non-finite value
  // in a row that nobody selected would reach every token (0 * Inf), where the other algorithms and the reference
  // only ever touch selected rows; and where it wins at all it wins little (the reference's group regime, T*k/N > 256
  // with N <= 16 k: 63 us against 67.5 us gather at 16384 tokens, hidden 1024, N = 256, k = 16; 95 against 70 at N = 512).
  const int es = dtype == OMNI_F32 ? 4 : 2;
  // rows beyond 8 KiB do not fit the gather kernel's registers: the split kernels take them in column blocks
  const int64_t row = (int64_t)H * es, table = N * row, pairs = T * (int64_t)k, moved = pairs * row, MiB = 1 << 20;
  if (row > 8192) return OMNI_EXPERT_ALGO_SPLIT;
  if (row < 512 || k > 2 * kWave || split_slices(H, N, es) == 0) return OMNI_EXPERT_ALGO_GATHER;
  const bool whole = (row & (row - 1)) == 0, little = table <= 2 * MiB;
  bool enough, near;
  if (row <= 1024) {
    enough = T >= 4096 || moved >= 64 * MiB || (moved >= 32 * MiB && !little && k >= 16) || (T > 1024 && (table <= (row == 1024 ? 16 : 4) * MiB || (row == 512 && k <= 8)));
    near = table <= (row == 1024 ? 64 : 16) * MiB || k <= (row == 1024 ? 4 : row == 512 ? 8 : 2);
  } else {
    const int least = row <= 2048 || (whole && !little) ? 4 : little ? 8 : 6;
    const bool half = row > 2048 && row < 2560;                  // little more than half of a slice's lanes
    enough = moved >= 64 * MiB ? k >= least : moved >= 32 * MiB && !little && (k >= 16 || (k >= 6 && N <= 16384));
    near = table <= (row < 1536 ? 16 : row < 2048 ? 128 : half ? 32 : k >= 16 ? 256 : 64) * MiB || (row >= 2048 && !half && k >= 16 && pairs >= 262144);
  }
  return enough && near ? OMNI_EXPERT_ALGO_SPLIT : OMNI_EXPERT_ALGO_GATHER;
}

// Whether the whole layer may take its joint launches (layer.hip), whose last kernel gathers the experts and adds, or its stages one by one with what resolve_algo
// says: the joint launches for few pairs, for little tables and for rows that are no power of two or under 1 KiB.  Time of the layer with split by name over its time
// by this rule, bf16, one stream, where the rule gathers and resolve_algo says split:
//   hidden  256   8192 tokens x 8 0.80, 16384 x 16 0.85, 32768 x 32 0.77 over 4096 experts, 4096 x 32 over 1024 0.83
//   hidden  512   4096 x 8 over 1024 0.93          hidden  768   4096 x 8 and 2048 x 16 1.0, 4096 x 32 0.90 over 4096, 4096 x 16 over 65536 1.04
//   hidden 1024   2000 x 16 0.97, 1000 x 32 0.91   hidden 1280   2600 x 16 0.87, 1600 x 32 0.89
//   hidden 2048   1000 x 16 0.90 over 4096, 500 x 32 over 16384 1.01
bool joint_launches_gather(int algo, int64_t T, int H, int64_t N, int k, int dtype) {
  if (algo != OMNI_EXPERT_ALGO_AUTO) return algo == OMNI_EXPERT_ALGO_GATHER;
  const int es = dtype == OMNI_F32 ? 4 : 2;
  const int64_t row = (int64_t)H * es, tables = 2 * N * row, pairs = T * (int64_t)k;
  if (row > 8192) return false;
  const int lanes = split_lanes_per_row(H, es, kSlices);
  if (lanes < 8 || (lanes & (lanes - 1)) || k > 2 * kWave || tables <= (3ll << 20) || pairs < 32768) return true;
  if (lanes == 8) return !(tables <= (32ll << 20) && pairs >= 131072);
  if (lanes == 16) return !(tables <= (128ll << 20) && (pairs >= 65536 || tables >= (16ll << 20)));
  return !((tables <= (256ll << 20) || pairs >= 262144) && 2 * k >= lanes);
}

// OMNI_OK when omni_expert_fwd takes `algo` for these sizes (what the whole-layer call checks before it enqueues anything).
int expert_algo_check(int algo, int64_t T, int H, int64_t N, int k, int dtype) {
  const int es = dtype == OMNI_F32 ? 4 : 2;
  switch (algo) {
    case OMNI_EXPERT_ALGO_AUTO:
      if ((int64_t)H * es <= 8192) return OMNI_OK;
      [[fallthrough]];                                           // wide rows: AUTO is the split algorithm
    case OMNI_EXPERT_ALGO_SPLIT: {
      int lpr = 0;
      return (split_col_blocks(H, es, &lpr) != 0 && k <= 2 * kWave) ? OMNI_OK : OMNI_ERR_UNSUPPORTED;
    }
    case OMNI_EXPERT_ALGO_GATHER: case OMNI_EXPERT_ALGO_SEGMENT: return (int64_t)H * es <= 8192 ? OMNI_OK : OMNI_ERR_UNSUPPORTED;
    case OMNI_EXPERT_ALGO_DENSE: return (k == 0 || T == 0 || dense_covers(T, H, N, k, dtype)) ? OMNI_OK : OMNI_ERR_UNSUPPORTED;
    default: return OMNI_ERR_UNSUPPORTED;
  }
}

}  // namespace omni

extern "C" OMNI_API size_t omni_expert_workspace_bytes(int64_t num_tokens, int32_t hidden_size, int64_t num_experts,
                                                       int32_t num_experts_per_token, int32_t dtype, int32_t algo) {
  if (num_tokens < 0 || num_experts <= 0 || num_experts_per_token < 0) return 0;
  algo = omni::resolve_algo(algo, num_tokens, hidden_size, num_experts, num_experts_per_token, dtype);
  if (algo == OMNI_EXPERT_ALGO_SPLIT) {
    const int col_blocks = omni::split_cut(hidden_size, num_experts, dtype == OMNI_F32 ? 4 : 2).col_blocks;
    return omni::align256((size_t)omni::kSlices * (size_t)(col_blocks ? col_blocks : 1) * (size_t)num_tokens * (size_t)num_experts_per_token * 4);
  }
  if (algo == OMNI_EXPERT_ALGO_DENSE)
    return omni::dense_covers(num_tokens, hidden_size, num_experts, num_experts_per_token, dtype) ? omni::dense_workspace_bytes(num_tokens, hidden_size, num_experts) : 0;
  if (algo != OMNI_EXPERT_ALGO_SEGMENT) return 0;   // the gather algorithm keeps everything in registers
  const size_t P = (size_t)num_tokens * (size_t)num_experts_per_token;
  return omni::align256((size_t)(num_experts + 1) * 4) + 2 * omni::align256(P * 4) +
         omni_schedule_workspace_bytes(num_tokens, num_experts_per_token, num_experts);
}

extern "C" OMNI_API int32_t omni_expert_fwd(const void* x, const void* up_weight, const void* down_weight,
                               const void* routing_weights, const int32_t* indices, void* y,
                               int64_t num_tokens, int32_t hidden_size, int64_t num_experts,
                               int32_t num_experts_per_token, int32_t dtype, int32_t algo,
                               void* workspace, void* stream) {
  return omni_expert_fwd_scores(x, up_weight, down_weight, routing_weights, indices, y, nullptr, num_tokens, hidden_size, num_experts, num_experts_per_token, dtype, algo,
                                workspace, stream);
}

extern "C" OMNI_API int32_t omni_expert_fwd_scores(const void* x, const void* up_weight, const void* down_weight, const void* routing_weights, const int32_t* indices, void* y,
                                                   float* scores, int64_t num_tokens, int32_t hidden_size, int64_t num_experts, int32_t num_experts_per_token, int32_t dtype,
                                                   int32_t algo, void* workspace, void* stream) {
  using namespace omni;
  if (num_tokens < 0 || hidden_size <= 0 || num_experts <= 0 || num_experts_per_token < 0) return OMNI_ERR_SHAPE;
  if (num_tokens > INT32_MAX / 2 || num_experts > UINT32_MAX) return OMNI_ERR_SHAPE;
  if (num_tokens > 0 && (!x || !up_weight || !down_weight || !y)) return OMNI_ERR_NULL;
  if (num_tokens > 0 && num_experts_per_token > 0 && (!routing_weights || !indices)) return OMNI_ERR_NULL;
  hipStream_t s = (hipStream_t)stream;
  int lanes = 0;
  if (algo == OMNI_EXPERT_ALGO_SPLIT && split_col_blocks(hidden_size, dtype == OMNI_F32 ? 4 : 2, &lanes) == 0) return OMNI_ERR_UNSUPPORTED;
  const bool shared = algo == OMNI_EXPERT_ALGO_AUTO;
  algo = resolve_algo(algo, num_tokens, hidden_size, num_experts, num_experts_per_token, dtype);
  if (scores && algo != OMNI_EXPERT_ALGO_GATHER && algo != OMNI_EXPERT_ALGO_SPLIT) return OMNI_ERR_UNSUPPORTED;
  if (algo == OMNI_EXPERT_ALGO_SEGMENT) {
    switch (dtype) {
      case OMNI_BF16: return expert_segment_dispatch<kBF16>(x, up_weight, down_weight, routing_weights, indices, y, num_tokens, hidden_size, num_experts_per_token, num_experts, workspace, s);
      case OMNI_F16: return expert_segment_dispatch<kF16>(x, up_weight, down_weight, routing_weights, indices, y, num_tokens, hidden_size, num_experts_per_token, num_experts, workspace, s);
      case OMNI_F32: return expert_segment_dispatch<kF32>(x, up_weight, down_weight, routing_weights, indices, y, num_tokens, hidden_size, num_experts_per_token, num_experts, workspace, s);
      default: return OMNI_ERR_DTYPE;
    }
  }
  if (algo == OMNI_EXPERT_ALGO_SPLIT) {
    switch (dtype) {
      case OMNI_BF16: return expert_split_dispatch<kBF16>(x, up_weight, down_weight, routing_weights, indices, y, scores, num_tokens, hidden_size, num_experts_per_token, num_experts, workspace, s);
      case OMNI_F16: return expert_split_dispatch<kF16>(x, up_weight, down_weight, routing_weights, indices, y, scores, num_tokens, hidden_size, num_experts_per_token, num_experts, workspace, s);
      case OMNI_F32: return expert_split_dispatch<kF32>(x, up_weight, down_weight, routing_weights, indices, y, scores, num_tokens, hidden_size, num_experts_per_token, num_experts, workspace, s);
      default: return OMNI_ERR_DTYPE;
    }
  }
  if (algo == OMNI_EXPERT_ALGO_DENSE) {
    if (dtype != OMNI_BF16 && dtype != OMNI_F16 && dtype != OMNI_F32) return OMNI_ERR_DTYPE;
    if (num_experts_per_token == 0)   // writes zeros
      return omni_expert_fwd(x, up_weight, down_weight, routing_weights, indices, y, num_tokens, hidden_size, num_experts, 0, dtype, OMNI_EXPERT_ALGO_GATHER, nullptr, stream);
    return expert_dense_dispatch(x, up_weight, down_weight, routing_weights, indices, y, num_tokens, hidden_size, num_experts_per_token,
                                 num_experts, dtype, workspace, s);
  }
  if (algo != OMNI_EXPERT_ALGO_GATHER) return OMNI_ERR_UNSUPPORTED;
  switch (dtype) {
    case OMNI_BF16: return expert_gather_dispatch<kBF16>(x, up_weight, down_weight, routing_weights, indices, y, num_tokens, hidden_size, num_experts_per_token, num_experts, s, scores, shared);
    case OMNI_F16: return expert_gather_dispatch<kF16>(x, up_weight, down_weight, routing_weights, indices, y, num_tokens, hidden_size, num_experts_per_token, num_experts, s, scores, shared);
    case OMNI_F32: return expert_gather_dispatch<kF32>(x, up_weight, down_weight, routing_weights, indices, y, num_tokens, hidden_size, num_experts_per_token, num_experts, s, scores, shared);
    default: return OMNI_ERR_DTYPE;
  }
}
