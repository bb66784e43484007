// The layer (reference omni_moe/modules/omni_moe.py:60-106) for at most 64 tokens, as in decoding: three launches, or two.
//
// What bounds it.  The weights' one trip through memory (25 MB at hidden 1024 x intermediate 4096: 5 us) and, above all, the chain of
// dependent launches: as six kernels -- projection, select, gate/up, experts, down projection, its partial sums -- the stages
// took 5-8 us each although none has work for that long (38 us a call for 1 token, 43 us for 48).  So what does not depend on
// each other shares a launch, by block index:
//   1. the router's projection | gate and up with their SwiGLU product
//   2. the router's selection  | the down projection, K split over the grid, as fp32 partial sums
//   3. the experts, the partial sums and the final add, one block per token; in launch 2 where the host takes longer for a launch than the kernels do (merge_launches).
// 1 token 38.4 -> 18.1 us a call, 48 tokens 42.9 -> 21.9 us, hidden 1024 x intermediate 4096; with the weights through LDS as well 17.2 -> 15.3 and 21.0 -> 20.1
// (three launches in a graph; a program sees the 18 us of host work of a call at 1 token, 15.2 with two launches).
//
// Projections.  There is one row tile, so every weight is used once, and all loads of 1024 K values of a block are in flight at once.  They go through
// each wave's own LDS all the same, because an instruction that reads eight whole 128-byte lines is faster than the one that a matrix fragment asks for,
// 64 bytes from each of 16 rows (kWeightsInLds; straight into registers where two blocks would not fit a CU).
// The eight waves of a block share the K range -- a wave takes 64 of K, a 128-byte line of each row, in turn -- and add up
// through LDS in wave order.  A block has 32 weight rows: 16 gate and the matching 16 up rows, 16 x and 16 y keys, or 32 rows of the
// down projection; with K split up to eight ways the latter fill the chip too.
//
// Experts.  Eight waves share a token's slots, so that all its rows are requested at once, and the block adds their sums in wave order.
#include "few_tokens.h"
#include "omni_moe_hip.h"
#include "rows.h"

#include <type_traits>

namespace omni {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

constexpr int kFewWaves = 8, kFewThreads = kFewWaves * kWave, kUnit = 64 /* of K */, kMostParts = 8;

template <int DT>
__device__ __forceinline__ f32x4_t mfma(const u32x4_t a, const u32x4_t b, f32x4_t c) {
  if constexpr (DT == kBF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}
template <int DT> __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  if constexpr (DT == kBF16) return pack_bf16(lo, hi); else return pack_f16(lo, hi);
}

// A wave's LDS: Q units of R8 times eight rows of activations, and the same units of the block's 32 weight rows.  These stay in registers for more than 48 tokens: with
// them two blocks would not fit a CU (64 tokens 22.1 us; one block to a CU 22.9).
template <int R8, int Q>
struct FewStage {
  static constexpr bool kWeightsInLds = R8 <= 6;
  static constexpr int kRows = Q * R8 * 1024, kPart = kRows + (kWeightsInLds ? Q * 4096 : 0), kBytes = kFewWaves * kPart;
};

// acc[j][i]: rows 16 i + lane % 16 of `a` ([rows of row_bytes], a_bytes in all, K values a row; zeros past the matrix, and beyond 8 R8 rows whatever) times the 16
// rows of weight tile j, columns 4 (lane / 16) .. + 3, over the K units u0 + wave, u0 + wave + 8, .. below u1, Q at a time.
// left[j]: weight rows from b[j] on (at least one; the last one stands in for those past it).  Weights are requested Q units ahead of their use.
// Every block reads all activations, from L2.  Reads of 64 bytes from each of 16 rows -- what a fragment is -- are slow (activations so, 64 tokens, hidden 1024: 15.4 us
// for launch 1, 10.1 us when an instruction reads 1 KiB on end; weights so, a call in a graph, hidden 1024 x intermediate 4096: 1 / 8 / 12 / 32 / 48 tokens 17.2 / 18.5 / 18.7 / 20.0 / 21.0 us, by whole lines 15.3 / 16.7 / 17.0 / 18.3 / 20.1;
// 2048 x 8192, 1 token 35.2 -> 32.5);
// so both take whole 128-byte lines of 8 rows into the wave's own `lds` (position c of row r holds the row's 16-byte piece c ^ (r / 2 % 8), which
// keeps the fragment reads free of bank conflicts).
// kTail: K is no multiple of 64 (but of 8); what is past it reads as zero on both sides.
template <int DT, int R8, int Q, bool kTail>
__device__ __forceinline__ void multiply(f32x4_t (&acc)[2][(R8 + 1) / 2], const uint8_t* a, int row_bytes, int a_bytes, const uint8_t* const (&b)[2], const int (&left)[2], int K,
                                         int u0, int u1, int wave, int lane, uint32_t lds) {
  constexpr int TM = (R8 + 1) / 2;
  using Stage = FewStage<R8, Q>;
  const int r16 = lane & 15, g4 = lane >> 4;
  using Frag = const __attribute__((address_space(3))) u32x4_t*;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int row = lane >> 3;
  // lane's place in the 8 rows that load instruction `part` of unit q brings in, of K step u: r / 2 % 8 = 4 (part % 2) + lane / 16
  auto offset = [&](int u, int q, int part, int at_row) __attribute__((always_inline)) {
    const int piece = (lane & 7) ^ (4 * (part & 1) + (lane >> 4)), v = u + q * kFewWaves, k = v * kUnit + piece * 8;
    return v < u1 && !(kTail && k >= K) ? (uint32_t)(at_row * row_bytes + k * 2) : 0x80000000u;
  };
  u32x4_t w[Q][2][2], next[Q][2][2];                           // [unit][half of it][weight tile]
  auto load_weights = [&](int u) __attribute__((always_inline)) {
    if constexpr (Stage::kWeightsInLds) {
      auto one = [&](auto n_tag) __attribute__((always_inline)) {
        constexpr int n = decltype(n_tag)::value, q = n / 4, part = n % 4, j = part / 2;
        load_to_lds<Stage::kRows + n * 1024>((uint64_t)b[j], min(left[j], 16) * row_bytes, lds, offset(u, q, part, min((part & 1) * 8 + row, left[j] - 1)), 0);
      };
      auto all = [&](auto... n) __attribute__((always_inline)) { (one(n), ...); };
      with_sequence(all, std::make_integer_sequence<int, 4 * Q>{});
    } else {
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int v = u + q * kFewWaves;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const int k = v * kUnit + ks * 32 + g4 * 8;
          const bool inside = v < u1 && !(kTail && k >= K);
#pragma unroll
          for (int j = 0; j < 2; ++j) next[q][ks][j] = inside ? *(const u32x4_t*)(b[j] + (int64_t)min(r16, left[j] - 1) * row_bytes + (int64_t)k * 2) : u32x4_t{0, 0, 0, 0};
        }
      }
    }
  };
  load_weights(u0 + wave);
  for (int u = u0 + wave; u < u1; u += Q * kFewWaves) {
    auto load_rows = [&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value, q = n / R8, part = n % R8;
      load_to_lds<n * 1024>((uint64_t)a, a_bytes, lds, offset(u, q, part, 8 * part + row), 0);
    };
    auto load_all = [&](auto... n) __attribute__((always_inline)) { (load_rows(n), ...); };
    with_sequence(load_all, std::make_integer_sequence<int, Q * R8>{});
    vmcnt<0>();
    __builtin_amdgcn_sched_barrier(0);
    auto fragment = [&](uint32_t at, int ks, int r) __attribute__((always_inline)) { return *(Frag)(uintptr_t)(lds + at + (uint32_t)(r * 128 + ((4 * ks + g4) ^ ((r >> 1) & 7)) * 16)); };
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if constexpr (Stage::kWeightsInLds) w[q][ks][j] = fragment(Stage::kRows + q * 4096 + j * 2048, ks, r16);
          else w[q][ks][j] = next[q][ks][j];
        }
    if (u + Q * kFewWaves < u1) {
      if constexpr (Stage::kWeightsInLds) {
        lds_reads_done();
        __builtin_amdgcn_sched_barrier(0);
      }
      load_weights(u + Q * kFewWaves);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const u32x4_t f = fragment(q * R8 * 1024 + i * 2048, ks, R8 == 1 ? r16 & 7 : r16);
          acc[0][i] = mfma<DT>(w[q][ks][0], f, acc[0][i]);
          acc[1][i] = mfma<DT>(w[q][ks][1], f, acc[1][i]);
        }
    lds_reads_done();                                          // before the next loads overwrite what they read
  }
  vmcnt<0>();                                                  // (a wave without a unit has asked for zeros)
}

// The block's eight sums meet in LDS, each at the start of its wave's own part of it
template <int R8, int Q>
__device__ __forceinline__ void publish(uint8_t* lds, const f32x4_t (&acc)[2][(R8 + 1) / 2], int wave, int lane) {
  constexpr int TM = (R8 + 1) / 2;
  static_assert(FewStage<R8, Q>::kPart >= TM * 2048, "a wave's sums fit its part");
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) *(f32x4_t*)(lds + wave * FewStage<R8, Q>::kPart + ((j * TM + i) * kWave + lane) * 16) = acc[j][i];
  __syncthreads();
}
// columns 4 quad .. + 3 of row `row` of weight tile j, all waves
template <int R8, int Q>
__device__ __forceinline__ f32x4_t gathered(const uint8_t* lds, int j, int row, int quad) {
  constexpr int TM = (R8 + 1) / 2;
  f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < kFewWaves; ++w) {
    const f32x4_t o = *(const f32x4_t*)(lds + w * FewStage<R8, Q>::kPart + ((j * TM + row / 16) * kWave + quad * 16 + row % 16) * 16);
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] += o[q];
  }
  return v;
}

struct FrontArgs {
  const uint8_t *x, *wg, *wu, *wx, *wy;
  uint8_t *h, *z;
  int T, H, I, r, router_blocks;
  uint32_t* tickets;                 // [T][groups], or NULL: cleared for launch 2
  int num_tickets;
};

// Launch 1: blocks below router_blocks project 16 keys of each half, the others 16 columns of gate and of up.
template <int DT, int R8, int Q, bool kTail>
__global__ __launch_bounds__(kFewThreads, Q == 1 || R8 == 1 ? 4 : 2) void few_front_kernel(const FrontArgs g) {
  extern __shared__ __align__(16) uint8_t lds[];               // FewStage
  constexpr int TM = (R8 + 1) / 2;
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t mine = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds + (uint32_t)(wave * FewStage<R8, Q>::kPart);
  const bool router = (int)blockIdx.x < g.router_blocks;
  for (int i = (int)blockIdx.x * kFewThreads + (int)threadIdx.x; i < g.num_tickets; i += (int)gridDim.x * kFewThreads) g.tickets[i] = 0;
  const int n0 = (router ? (int)blockIdx.x : (int)blockIdx.x - g.router_blocks) * 16, rows = router ? g.r : g.I;
  const int64_t b_at = n0 * ((int64_t)g.H * 2);
  f32x4_t acc[2][TM];
  multiply<DT, R8, Q, kTail>(acc, g.x, g.H * 2, g.T * g.H * 2, {(router ? g.wx : g.wg) + b_at, (router ? g.wy : g.wu) + b_at}, {rows - n0, rows - n0}, g.H, 0, (g.H + kUnit - 1) / kUnit,
                             wave, lane, mine);
  publish<R8, Q>(lds, acc, wave, lane);
  for (int i = threadIdx.x; i < TM * 64; i += kFewThreads) {
    const int row = i >> 2, quad = i & 3, n = n0 + quad * 4;
    if (row >= g.T || n >= rows) continue;
    const f32x4_t p = gathered<R8, Q>(lds, 0, row, quad), q = gathered<R8, Q>(lds, 1, row, quad);
    if (router) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < rows) {
          Elem<DT>::store(g.z, (int64_t)row * 2 * g.r + n + e, p[e]);
          Elem<DT>::store(g.z, (int64_t)row * 2 * g.r + g.r + n + e, q[e]);
        }
    } else {
      // gate and up are materialised in the storage dtype, silu(gate) * up is formed in fp32 and rounded once (omni_mlp.py:53-61)
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = silu_fast(Elem<DT>::round(p[e])) * Elem<DT>::round(q[e]);
      *(u32x2_t*)(g.h + ((int64_t)row * g.I + n) * 2) = u32x2_t{pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3])};
    }
  }
}

// ---- launch 2, and for few tokens of a small layer launch 3 with it.
// A call of three launches is 18 us of host work, where the kernels of 1 token, hidden 1024 x intermediate 4096, take 15.  The third one needs every split of the
// down projection and the token's experts; so a block per token selects and sums up its experts, and whoever comes last adds up: a ticket per token and
// group of 32 columns, cleared by launch 1, counts the splits and the token's block, and the one that takes the last number finds all parts there and
// writes y's 32 values.  Nobody waits.  What others read is stored and loaded at agent scope (the XCDs' L2s are not one cache), and a block takes its
// numbers when its stores have been acknowledged.  Three launches / two as a program makes the call, 1 token: 18.3 / 15.2 us.  Replayed from a graph the kernels of two
// take up to 5 % more, of the MLP alone up to 19 %; merge_launches has the figures.
struct MiddleArgs {
  const uint8_t *h, *wd;
  float* parts;                      // [splits][T][H]
  int T, H, I, groups, units, splits;    // groups of 32 output columns; K units to a split
  int select_blocks, select_regs, cells; // the first blocks select, for eight tokens each (merged: for one); keys and candidates per lane
  SelectArgs select;
  // merged
  uint32_t* tickets;                 // [T][groups]
  uint32_t numbers;                  // of a ticket: the splits and, in the layer, the token's block
  uint8_t* experts;                  // the layer: [T][H] the experts' rounded sums
  const uint8_t *x, *up, *down, *residual;   // (residual: the MLP alone, or NULL)
  uint8_t* y;
  uint32_t N;
};
// So two launches are for calls whose kernels take less than the host: up to 16 tokens and 2^23 weights a projection (the MLP alone, whose host work is less: 2^22), up to 48
// tokens and 2^21.  The MLP alone, a call as a program makes it, three / two: 16 tokens 1024 x 4096 12.2 / 11.1 us, 8 tokens 512 x 1024 12.4 / 9.7.
// A graph's replay has no host work, and what is captured takes two launches only where its kernels are no slower for it.  Three / two in a graph, the layer: 1 token 512 x 2048
// 10.7 / 10.7 us, 16 tokens 768 x 3072 12.7 / 12.7, 48 tokens 1024 x 2048 14.1 / 14.2, 512 x 2048 12.8 / 12.5; but 16 tokens 1024 x 4096 13.8 / 14.5.  The MLP alone: 16 tokens 512 x 1024
// 8.4 / 8.3; but 32 tokens 9.0 / 9.3, 16 tokens 512 x 2048 8.5 / 9.1, 1024 x 4096 9.1 / 10.8.  Either form leaves the same bits.
constexpr int kMergedTokens = 48, kMergedRow = 1024;           // (a token's block has a thread for four values of a row)
bool merge_launches(bool layer, int64_t T, int64_t H, int64_t I, bool replayed) {
  const int64_t weights = H * I;
  if (layer && H > kMergedRow) return false;
  if (replayed && !layer) return T <= 16 && weights <= 1 << 19;
  if (T > 16) return T <= kMergedTokens && weights <= 1 << 21;
  return weights <= (replayed ? 3 << 20 : layer ? 1 << 23 : 1 << 22);
}
// Whether the call goes into a graph.  (The null stream is never captured, and asking about it while another stream is being captured is an error.)
bool is_captured(hipStream_t s) {
  if (!s) return false;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &status) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return status != hipStreamCaptureStatusNone;
}
__device__ __forceinline__ void store_agent(void* at, uint32_t a, uint32_t b) {
  __hip_atomic_store((uint64_t*)at, (uint64_t)a | (uint64_t)b << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u32x2_t load_agent(const void* at) {
  const uint64_t v = __hip_atomic_load((const uint64_t*)at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return u32x2_t{(uint32_t)v, (uint32_t)(v >> 32)};
}
__device__ __forceinline__ bool takes_last(const MiddleArgs& g, int t, int group) {
  return __hip_atomic_fetch_add(g.tickets + t * g.groups + group, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g.numbers - 1;
}
__device__ __forceinline__ void stores_acknowledged() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}
// four columns of a token: y = round(round(sum of the parts in split order) + e), or the rounded sum
template <int DT>
__device__ __forceinline__ void add_up(const MiddleArgs& g, int t, int n, const u32x2_t e, bool add = true) {
  u32x2_t part[kMostParts][2];
#pragma unroll
  for (int s = 0; s < kMostParts; ++s)
#pragma unroll
    for (int q = 0; q < 2; ++q) part[s][q] = load_agent(g.parts + ((int64_t)min(s, g.splits - 1) * g.T + t) * g.H + n + 2 * q);
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < kMostParts; ++s)
    if (s < g.splits)
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] += __uint_as_float(part[s][q / 2][q % 2]);
  if (add) {
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = Elem<DT>::round(v[q]) + Elem<DT>::load(&e, q);
  }
  *(u32x2_t*)(g.y + ((int64_t)t * g.H + n) * 2) = u32x2_t{pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3])};
}

template <int DT>
__device__ __forceinline__ void select_tokens(const MiddleArgs& g, int first, int all) {
  auto select = [&](auto cells) {
    constexpr int C = decltype(cells)::value;
    if (g.select_regs <= 1) select_packed<DT, 1, C>(g.select, first, all, g.select.stats);
    else if (g.select_regs <= 2) select_packed<DT, 2, C>(g.select, first, all, g.select.stats);
    else if (g.select_regs <= 4) select_packed<DT, 4, C>(g.select, first, all, g.select.stats);
    else select_packed<DT, 8, C>(g.select, first, all, g.select.stats);
  };
  if (g.cells <= 1) select(std::integral_constant<int, 1>{});
  else select(std::integral_constant<int, 2>{});
}

// The experts of a token by the block's eight waves, which share its slots so that all its rows are requested at once.  Leaves wave w's sums, in fp32, at
// sums + w * stride.  NCH 1-KiB pieces of a row; G slots of a wave at once.  Returns the waves that had any.
struct FewExperts { const uint8_t *x, *up, *down; const void* gates; const int32_t* ids; int H, k; uint32_t N; };
template <int DT, int NCH, int G>
__device__ __forceinline__ int share_experts(const FewExperts& g, int t, int wave, int lane, float* sums, int stride) {
  const int per = (g.k + kFewWaves - 1) / kFewWaves, active = (g.k + per - 1) / per;
  if (wave >= active) return active;
  const int64_t row_bytes = (int64_t)g.H * 2;
  bool live[NCH];
  u32x4_t xr[NCH];
  float acc[NCH][8];
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    live[c] = (c * kWave + lane) * 8 < g.H;
    xr[c] = live[c] ? *(const u32x4_t*)(g.x + t * row_bytes + (c * kWave + lane) * 16) : u32x4_t{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[c][i] = 0.f;
  }
  const int last = min((wave + 1) * per, g.k);
  for (int j0 = wave * per; j0 < last; j0 += G) {
    int64_t at[G];
    float gate[G];
    bool ok[G];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int j = min(j0 + i, last - 1), id = g.ids[(int64_t)t * g.k + j];
      gate[i] = Elem<DT>::load(g.gates, (int64_t)t * g.k + j);
      ok[i] = j0 + i < last && (uint32_t)id < g.N;             // a slot of another wave, or an id outside the table, contributes nothing
      at[i] = ok[i] ? id * row_bytes : 0;
    }
    u32x4_t u[G][NCH], v[G][NCH];
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        u[i][c] = live[c] ? *(const u32x4_t*)(g.up + at[i] + (c * kWave + lane) * 16) : u32x4_t{0, 0, 0, 0};
        v[i][c] = live[c] ? *(const u32x4_t*)(g.down + at[i] + (c * kWave + lane) * 16) : u32x4_t{0, 0, 0, 0};
      }
    float s[G];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      s[i] = 0.f;
#pragma unroll
      for (int c = 0; c < NCH; ++c) s[i] = dot16<DT>(xr[c], u[i][c], s[i]);
    }
#pragma unroll
    for (int i = 0; i < G; ++i) s[i] = wave_sum(s[i]);
#pragma unroll
    for (int i = 0; i < G; ++i) {
      if (!ok[i]) continue;                                    // not even 0 * row: the stand-in row may hold Inf or NaN
      const float coef = silu_f32(s[i]) * gate[i];
#pragma unroll
      for (int c = 0; c < NCH; ++c) axpy16<DT>(coef, v[i][c], acc[c]);
    }
  }
#pragma unroll
  for (int c = 0; c < NCH; ++c)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (live[c])
        *(f32x4_t*)(sums + wave * stride + (c * kWave + lane) * 8 + 4 * h) = f32x4_t{acc[c][4 * h], acc[c][4 * h + 1], acc[c][4 * h + 2], acc[c][4 * h + 3]};
  return active;
}

template <int DT>
__device__ __forceinline__ void token_block(const MiddleArgs& g, int t, uint8_t* lds, int wave, int lane) {
  if (wave == 0) select_tokens<DT>(g, t, g.T);
  __syncthreads();
  float* sums = (float*)lds;                                   // [waves][H]
  const FewExperts f{g.x, g.up, g.down, g.select.gates, g.select.indices, g.H, g.select.k, g.N};
  const int active = share_experts<DT, kMergedRow / 512, 4>(f, t, wave, lane, sums, g.H);
  __syncthreads();
  const int n = (int)threadIdx.x * 4;
  u32x2_t e{0, 0};
  if (n < g.H) {
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < active; ++w) {
      const f32x4_t o = *(const f32x4_t*)(sums + w * g.H + n);
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] += o[q];
    }
    e = u32x2_t{pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3])};
    store_agent(g.experts + ((int64_t)t * g.H + n) * 2, e[0], e[1]);
  }
  stores_acknowledged();
  uint8_t* last = lds;                                         // (the sums have been read)
  if ((int)threadIdx.x < g.groups) last[threadIdx.x] = takes_last(g, t, (int)threadIdx.x);
  __syncthreads();
  if (n < g.H && last[n >> 5]) add_up<DT>(g, t, n, e);
}

// Blocks below select_blocks select (merged: and sum up a token's experts), the others multiply 32 output columns over one of the K splits.
// kTail: as in multiply().  Weights that go through LDS bear it at no cost; on the way into registers it is a branch around every load (down projection of 64 tokens,
// 2048 x 8192, 11.7 us with it, 10.7 without).
template <int DT, int R8, int Q, bool kMerged, bool kTail>
__global__ __launch_bounds__(kFewThreads, Q == 1 ? 4 : 2) void few_middle_kernel(const MiddleArgs g) {
  extern __shared__ __align__(16) uint8_t lds[];               // FewStage
  constexpr int TM = (R8 + 1) / 2;
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  static_assert(FewStage<R8, Q>::kBytes >= kFewWaves * kMergedRow * 4, "a token's block has its waves' sums there");
  if ((int)blockIdx.x < g.select_blocks) {
    if constexpr (kMerged) token_block<DT>(g, (int)blockIdx.x, lds, wave, lane);
    else select_tokens<DT>(g, (int)blockIdx.x * kFewWaves + wave, g.select_blocks * kFewWaves);
    return;
  }
  const uint32_t mine = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds + (uint32_t)(wave * FewStage<R8, Q>::kPart);
  const int block = (int)blockIdx.x - g.select_blocks, split = block / g.groups, group = block - split * g.groups, n0 = group * 32;
  const int64_t row_bytes = (int64_t)g.I * 2;
  const int second = min(n0 + 16, g.H - 1);
  f32x4_t acc[2][TM];
  multiply<DT, R8, Q, kTail>(acc, g.h, g.I * 2, g.T * g.I * 2, {g.wd + n0 * row_bytes, g.wd + second * row_bytes}, {g.H - n0, g.H - second}, g.I, split * g.units,
                            min((split + 1) * g.units, (g.I + kUnit - 1) / kUnit), wave, lane, mine);
  publish<R8, Q>(lds, acc, wave, lane);
  for (int i = threadIdx.x; i < TM * 128; i += kFewThreads) {
    const int row = i >> 3, quad = i & 7, n = n0 + quad * 4;
    if (row >= g.T || n >= g.H) continue;
    const f32x4_t v = gathered<R8, Q>(lds, quad >> 2, row, quad & 3);
    float* out = g.parts + ((int64_t)split * g.T + row) * g.H + n;
    if constexpr (kMerged) {
      store_agent(out, __float_as_uint(v[0]), __float_as_uint(v[1]));
      store_agent(out + 2, __float_as_uint(v[2]), __float_as_uint(v[3]));
    } else {
      *(f32x4_t*)out = v;
    }
  }
  if constexpr (kMerged) {
    stores_acknowledged();
    uint8_t* last = lds;                                       // (the waves' sums have been read)
    if ((int)threadIdx.x < g.T) last[threadIdx.x] = takes_last(g, (int)threadIdx.x, group);
    __syncthreads();
    for (int i = threadIdx.x; i < g.T * 8; i += kFewThreads) {
      const int row = i >> 3, n = n0 + (i & 7) * 4;
      if (n >= g.H || !last[row]) continue;
      const int64_t at = ((int64_t)row * g.H + n) * 2;
      if (g.experts) add_up<DT>(g, row, n, load_agent(g.experts + at));
      else add_up<DT>(g, row, n, g.residual ? *(const u32x2_t*)(g.residual + at) : u32x2_t{0, 0}, g.residual != nullptr);
    }
  }
}

struct BackArgs {
  FewExperts e;
  const uint8_t* residual;
  const float* parts;
  uint8_t* y;
  int T, splits;
};

// Launch 3 where it is one of its own, a block per token: y = round(round(sum of the parts) + round(experts)).  NCH 1-KiB pieces of a row; G slots of a wave at once.
// splits 0: y holds the rounded sums already.
// kExperts false: the MLP alone, residual (or nothing) instead of the experts.
template <int DT, int NCH, int G, bool kExperts>
__global__ __launch_bounds__(kFewThreads, 2) void few_back_kernel(const BackArgs g) {
  extern __shared__ __align__(16) float sums[];                // [waves][NCH * 512]
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t = blockIdx.x, H = g.e.H;
  constexpr int kRow = NCH * 512;
  // this thread's first four columns of every part, requested before anything else
  f32x4_t part[kMostParts];
  const int64_t plane = (int64_t)g.T * H;
  auto request = [&](int n) __attribute__((always_inline)) {
    if (kExperts && g.splits == 0) return;
    const float* at = g.parts + (int64_t)t * H + min(n, H - 4);
#pragma unroll
    for (int s = 0; s < kMostParts; ++s) part[s] = *(const f32x4_t*)(at + min(s, g.splits - 1) * plane);
  };
  request(threadIdx.x * 4);
  int active = 0;
  if constexpr (kExperts) {
    active = share_experts<DT, NCH, G>(g.e, t, wave, lane, sums, kRow);
    __syncthreads();
  }
  for (int n = threadIdx.x * 4; n < H; n += kFewThreads * 4) {
    if (n != (int)threadIdx.x * 4) request(n);
    float v[4] = {0.f, 0.f, 0.f, 0.f}, e[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < kMostParts; ++s)
      if (s < g.splits)
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] += part[s][q];
    const int64_t out = ((int64_t)t * H + n) * 2;
    if (kExperts && g.splits == 0) {
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = Elem<DT>::load(g.y + out, q);
    }
    if (kExperts || g.residual) {
      if constexpr (kExperts) {
        for (int w = 0; w < active; ++w) {
          const f32x4_t o = *(const f32x4_t*)(sums + w * kRow + n);
#pragma unroll
          for (int q = 0; q < 4; ++q) e[q] += o[q];
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) e[q] = Elem<DT>::load(g.residual + out, q);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = Elem<DT>::round(v[q]) + Elem<DT>::round(e[q]);
    }
    *(u32x2_t*)(g.y + out) = u32x2_t{pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3])};
  }
}

// K splits of the down projection: as many as fill 256 CUs with blocks of 32 columns while each of a block's waves still has 64 of K
int few_splits(int64_t H, int64_t I) {
  const int64_t groups = (H + 31) / 32, units = (I + kUnit - 1) / kUnit;
  int64_t n = 256 / groups;
  if (n > units / kFewWaves) n = units / kFewWaves;
  return n < 1 ? 1 : n > kMostParts ? kMostParts : (int)n;
}

template <auto kKernel, int kBytes>
struct FewLds { static inline LdsKernel entry{(const void*)kKernel, kBytes}; };
template <auto kKernel, int kBytes, class Args>
hipError_t start(const Args& a, int64_t blocks, hipStream_t s) {
  if (hipError_t e = FewLds<kKernel, kBytes>::entry.ensure(); e != hipSuccess) return e;
  hipLaunchKernelGGL(kKernel, dim3((unsigned)blocks), dim3(kFewThreads), kBytes, s, a);
  return hipGetLastError();
}

BackArgs back_args(const FewTokens& f, int splits) {
  return BackArgs{FewExperts{(const uint8_t*)f.x, (const uint8_t*)f.up, (const uint8_t*)f.down, f.select.gates, f.select.indices, f.H, f.select.k, (uint32_t)f.N},
                  (const uint8_t*)f.residual, f.parts, (uint8_t*)f.y, f.T, splits};
}
// f.parts: the down projection's parts [splits][T][H], and where launches 2 and 3 are one, the experts' rounded sums [T][H] | tickets [T][groups]
struct FewParts {
  uint8_t* experts;
  uint32_t* tickets;
  size_t bytes;
  FewParts(float* parts, int64_t T, int64_t H, int64_t I) {
    const size_t sums = (size_t)few_splits(H, I) * (size_t)T * (size_t)H * 4, rows = ((size_t)T * (size_t)H * 2 + 15) / 16 * 16;
    experts = (uint8_t*)parts + sums;
    tickets = (uint32_t*)(experts + rows);
    bytes = sums + (merge_launches(true, T, H, I, false) || merge_launches(false, T, H, I, false) ? rows + (size_t)T * (size_t)((H + 31) / 32) * 4 : 0);
  }
};

template <int DT>
hipError_t launch_back(const BackArgs& b, hipStream_t s) {
  const int nch = (b.e.H + 511) / 512;
  if (nch <= 1) return start<few_back_kernel<DT, 1, 4, true>, kFewWaves * 1 * 2048>(b, b.T, s);
  if (nch <= 2) return start<few_back_kernel<DT, 2, 4, true>, kFewWaves * 2 * 2048>(b, b.T, s);
  if (nch <= 4) return start<few_back_kernel<DT, 4, 2, true>, kFewWaves * 4 * 2048>(b, b.T, s);
  return start<few_back_kernel<DT, 8, 1, true>, kFewWaves * 8 * 2048>(b, b.T, s);
}

// What a call takes, from its sizes; r 0: the MLP alone
struct FewPlan {
  int r8;                            // FewStage's
  bool merged;
  int front_units, middle_units;     // K units of a wave in LDS at once
  int splits, units;                 // of the down projection; K units to a split
  int router_blocks, select_blocks;
  int64_t front, middle;             // blocks
};
FewPlan plan_few(int64_t T, int64_t H, int64_t I, int r, bool replayed) {
  FewPlan p;
  p.r8 = T <= 8 ? 1 : T <= 16 ? 2 : T <= 32 ? 4 : T <= 48 ? 6 : 8;
  p.merged = merge_launches(r > 0, T, H, I, replayed);
  p.router_blocks = (r + 15) / 16;
  p.front = p.router_blocks + (I + 15) / 16;
  const int units = (int)((I + kUnit - 1) / kUnit), most = few_splits(H, I);
  p.units = (units + most - 1) / most;
  p.splits = (units + p.units - 1) / p.units;                  // every split has work
  p.select_blocks = (int)(r == 0 ? 0 : p.merged ? T : (T + kFewWaves - 1) / kFewWaves);
  p.middle = p.select_blocks + (H + 31) / 32 * p.splits;
  // Beyond eight tokens two K units of a wave in LDS at once are more than half of a CU's: one block to a CU, and blocks beyond 256 wait for a whole round.
  // One unit at a time then (in turn over three sets of inputs, hidden 1024 x intermediate 4096, weights in registers: 33 tokens 23.5 -> 21.3 us, 48 24.1 -> 21.9, 64
  // 26.2 -> 22.9; 48 tokens, 2048 x 8192 49.9 -> 43.9).  Where a launch has no more blocks than CUs both units stay in flight, if a wave has two.
  p.front_units = (p.r8 > 1 && p.front > 256) || H <= kFewWaves * kUnit ? 1 : 2;
  p.middle_units = (p.r8 > 1 && p.middle > 256) || p.units <= kFewWaves ? 1 : 2;       // (a wave may have one unit only)
  return p;
}

template <int DT, int R8>
hipError_t launch(const FewTokens& f, const FewPlan& plan, hipStream_t s) {
  const bool layer = f.up != nullptr, merged = plan.merged;
  const FewParts p(f.parts, f.T, f.H, f.I);
  const FrontArgs a{(const uint8_t*)f.x, (const uint8_t*)f.wg, (const uint8_t*)f.wu, (const uint8_t*)f.wx, (const uint8_t*)f.wy, (uint8_t*)f.h, (uint8_t*)f.z,
                    f.T, f.H, f.I, f.select.r, plan.router_blocks, merged ? p.tickets : nullptr, merged ? f.T * ((f.H + 31) / 32) : 0};
  auto units_at_once = [&](int units, auto&& go) -> hipError_t {
    if (units == 1) return go(std::integral_constant<int, 1>{});
    return go(std::integral_constant<int, 2>{});
  };
  hipError_t e = units_at_once(plan.front_units, [&](auto q) -> hipError_t {
    constexpr int Q = decltype(q)::value, kBytes = FewStage<R8, Q>::kBytes;
    return f.H % kUnit ? start<few_front_kernel<DT, R8, Q, true>, kBytes>(a, plan.front, s) : start<few_front_kernel<DT, R8, Q, false>, kBytes>(a, plan.front, s);
  });
  if (e != hipSuccess) return e;

  MiddleArgs m{};
  m.h = (const uint8_t*)f.h; m.wd = (const uint8_t*)f.wd; m.parts = f.parts; m.T = f.T; m.H = f.H; m.I = f.I;
  m.groups = (f.H + 31) / 32;
  m.units = plan.units;
  m.splits = plan.splits;
  m.tickets = p.tickets; m.numbers = (uint32_t)(layer ? m.splits + 1 : m.splits); m.experts = layer ? p.experts : nullptr; m.residual = (const uint8_t*)f.residual;
  m.x = (const uint8_t*)f.x; m.up = (const uint8_t*)f.up; m.down = (const uint8_t*)f.down; m.y = (uint8_t*)f.y;
  m.N = (uint32_t)f.N;
  m.select = f.select;
  m.select_regs = (f.select.r + kWave - 1) / kWave;
  m.cells = layer ? prepare_select(m.select) : 0;
  m.select_blocks = plan.select_blocks;
  e = units_at_once(plan.middle_units, [&](auto q) -> hipError_t {
    constexpr int Q = decltype(q)::value, kBytes = FewStage<R8, Q>::kBytes;
    if constexpr (R8 * 8 <= kMergedTokens) {
      if (merged) return start<few_middle_kernel<DT, R8, Q, true, true>, kBytes>(m, plan.middle, s);
    }
    if constexpr (!FewStage<R8, Q>::kWeightsInLds) {
      if (f.I % kUnit == 0) return start<few_middle_kernel<DT, R8, Q, false, false>, kBytes>(m, plan.middle, s);
    }
    return start<few_middle_kernel<DT, R8, Q, false, true>, kBytes>(m, plan.middle, s);
  });
  if (e != hipSuccess || merged) return e;
  const BackArgs b = back_args(f, m.splits);
  if (!layer) return start<few_back_kernel<DT, 1, 1, false>, 0>(b, f.T, s);
  return launch_back<DT>(b, s);
}

}  // namespace

bool few_tokens_covers(int64_t T, int64_t H, int64_t I, int dtype) {
  return T > 0 && T <= kFewTokens && dtype != OMNI_F32 && H % 8 == 0 && I % 8 == 0 && H <= (1 << 20) && I <= (1 << 20);   // (32-bit offsets)
}
bool few_tokens_covers_layer(int64_t T, int64_t H, int64_t I, int r, int k, int dtype) {
  // keys and candidates that the joint launch has registers for; rows that a block holds its waves' sums of
  return few_tokens_covers(T, H, I, dtype) && H <= 4096 && r <= 8 * kWave && k > 0 && num_cells(k, r < k ? r : k) <= 2 * kWave;
}
bool few_tokens_aligned(const FewTokens& f) {
  for (const void* q : {f.x, f.wg, f.wu, f.wd, (const void*)f.h, (const void*)f.y, (const void*)f.parts, f.residual, f.wx, f.wy, (const void*)f.z, f.up, f.down})
    if ((uintptr_t)q % 16) return false;
  return true;
}
size_t few_tokens_parts_bytes(int64_t T, int64_t H, int64_t I) { return FewParts(nullptr, T, H, I).bytes; }

hipError_t launch_few_tokens(int dtype, const FewTokens& f, hipStream_t s) {
  const bool layer = f.up != nullptr;
  const int r = layer ? f.select.r : 0;
  // (asked only where the answer matters)
  const bool replayed = merge_launches(layer, f.T, f.H, f.I, false) && !merge_launches(layer, f.T, f.H, f.I, true) && is_captured(s);
  const FewPlan plan = plan_few(f.T, f.H, f.I, r, replayed);
  auto go = [&](auto dt) -> hipError_t {
    constexpr int DT = decltype(dt)::value;
    if (plan.r8 == 1) return launch<DT, 1>(f, plan, s);
    if (plan.r8 == 2) return launch<DT, 2>(f, plan, s);
    if (plan.r8 == 4) return launch<DT, 4>(f, plan, s);
    if (plan.r8 == 6) return launch<DT, 6>(f, plan, s);
    return launch<DT, 8>(f, plan, s);
  };
  if (dtype == kBF16) return go(std::integral_constant<int, kBF16>{});
  if (dtype == kF16) return go(std::integral_constant<int, kF16>{});
  return hipErrorInvalidValue;
}

hipError_t launch_few_back(int dtype, const FewTokens& f, int splits, hipStream_t s) {
  const BackArgs b = back_args(f, splits);
  if (dtype == kBF16) return launch_back<kBF16>(b, s);
  if (dtype == kF16) return launch_back<kF16>(b, s);
  return hipErrorInvalidValue;
}

}  // namespace omni

extern "C" OMNI_API int32_t omni_probe_few_tokens(int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size, int32_t num_expert_sqrt, int32_t captured, int32_t* plan) {
  using namespace omni;
  if (!few_tokens_covers(num_tokens, hidden_size, intermediate_size, OMNI_BF16) || hidden_size <= 0 || intermediate_size <= 0 || num_expert_sqrt < 0) return OMNI_ERR_SHAPE;
  if (!plan) return OMNI_ERR_NULL;
  const FewPlan p = plan_few(num_tokens, hidden_size, intermediate_size, num_expert_sqrt, captured != 0);
  plan[0] = p.merged ? 2 : 3;
  plan[1] = p.r8 * 8;
  plan[2] = p.front_units;
  plan[3] = p.middle_units;
  plan[4] = p.splits;
  return OMNI_OK;
}
