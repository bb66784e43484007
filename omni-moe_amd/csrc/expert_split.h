// The hidden-split expert algorithm as device functions: the forward's kernels (expert.hip, where the algorithm is described) and the backward's
// token pass (backward.hip) share them.
#pragma once
#include "common.h"
#include "rows.h"

namespace omni {

constexpr int kSlices = 8;

// Sum over the LPR lanes of a group of LPR values per lane, scattered: lane `sub` of the group
// ends up with the total of value `sub`.  Every step halves what a lane keeps (LPR - 1 exchanges
// in all, against LPR * log2(LPR) for one tree per value).
template <int LPR, int N = LPR>
__device__ __forceinline__ float reduce_scatter_group(float (&v)[N], const int lane) {
  if constexpr (N == 1) {
    return v[0];
  } else {
    constexpr int S = N / 2;                   // lane distance of this step = half of what is left
    const bool upper = lane & S;
    float keep[S];
#pragma unroll
    for (int e = 0; e < S; ++e) keep[e] = (upper ? v[e + S] : v[e]) + xor_lane_f<S>(upper ? v[e] : v[e + S], lane);
    return reduce_scatter_group<LPR, S>(keep, lane);
  }
}

// A wave owns GP = 64 / LPR tokens, one per lane group; the group's LPR lanes cover the token's
// row slice, 16 bytes each.  Pairs go in batches of LPR: LPR partial dot products per lane,
// then one reduce-scatter leaves pair `sub` of the batch in lane `sub`.
// SMALL: every table, x, y and the partial sums stay below 4 GiB, ids and row lengths below 2^24 (split_offsets_small):
// a row's byte offset is then one full-rate v_mad_u32_u24 on 32-bit lane offsets instead of a 64-bit multiply-add and two
// 32-bit multiplies at a quarter of the rate -- address arithmetic was more than half of the vector instructions' time here.
template <bool SMALL> struct SplitOff { using type = int64_t; };
template <> struct SplitOff<true> { using type = uint32_t; };
template <bool SMALL>
__device__ __forceinline__ typename SplitOff<SMALL>::type split_mul(uint32_t a, typename SplitOff<SMALL>::type b) {
  if constexpr (SMALL) return __umul24(a, b); else return (int64_t)a * b;
}

// Partial dot products <a[t, slice], table[id, slice]> of the k pairs of a block's tokens -> partial[slice][t][j].  block % 8 is the slice, WAVES the block's
// waves.  (rows wider than 8 slices of 64 lanes go in column blocks of 8 slices, one launch each)
template <int DT, int LPR, bool SMALL, int WAVES>
__device__ __forceinline__ void split_dots_block(const uint8_t* __restrict__ x, const uint8_t* __restrict__ up, const int32_t* __restrict__ ids,
                                                 float* __restrict__ partial, int num_tokens, int hidden, int top_k, uint32_t num_experts, int col_block, int block) {
  using Off = typename SplitOff<SMALL>::type;
  constexpr int E = Row16<DT>::kElems, GP = kWave / LPR;
  constexpr int LD = LPR < 8 ? LPR : 8;                          // row loads in flight at a time
  const int lane = lane_id(), sub = lane % LPR, grp = lane / LPR;
  const int slice = block % kSlices;
  const int t = ((int)(block / kSlices) * WAVES + (threadIdx.x >> 6)) * GP + grp;
  const bool live = t < num_tokens;
  const int tt = live ? t : 0;
  const Off row_bytes = Off(hidden) * (16 / E);
  // this lane's 16 bytes inside a row
  const Off col = (Off(col_block) * kSlices + slice) * LPR * 16 + sub * 16;
  const u32x4_t xr = *(const u32x4_t*)(x + (split_mul<SMALL>((uint32_t)tt, row_bytes) + col));
  const Off base = split_mul<SMALL>((uint32_t)tt, (Off)top_k);
  for (int jb = 0; jb < top_k; jb += LPR) {
    // lane `sub` of a group fetches the id of pair `sub` of the batch; the group reads the ids from its lanes
    const int my_id = ids[base + min(jb + sub, top_k - 1)];
    float d[LPR];
#pragma unroll
    for (int e0 = 0; e0 < LPR; e0 += LD) {
      u32x4_t ur[LD];
#pragma unroll
      for (int e = 0; e < LD; ++e) {
        const int id = __shfl(my_id, grp * LPR + e0 + e, kWave);
        ur[e] = *(const u32x4_t*)(up + (split_mul<SMALL>((uint32_t)id < num_experts ? (uint32_t)id : 0u, row_bytes) + col));
      }
#pragma unroll
      for (int e = 0; e < LD; ++e) d[e0 + e] = dot16<DT>(xr, ur[e], 0.f);
    }
    const float total = reduce_scatter_group<LPR>(d, lane);
    const int j = jb + sub;
    if (live && j < top_k) {
      const bool ok = (uint32_t)my_id < num_experts;
      partial[((Off(col_block) * kSlices + slice) * num_tokens + t) * top_k + j] = ok ? total : 0.f;
    }
  }
}

// Same ownership.  Lane `sub` of a group forms the coefficient of pair `sub` of a batch -- coefficient(token, pair, slot, id inside the table), from the
// sums over the slices -- and the group then walks the batch, every lane fetching its 16 bytes of the pair's row and the coefficient from the lane that
// holds it.  kAll: coefficient() is called for ids outside the table too (its result is then not used).
template <int DT, int LPR, bool SMALL, int WAVES, bool kAll, class Coefficient>
__device__ __forceinline__ void split_accumulate_block(const uint8_t* __restrict__ down, const int32_t* __restrict__ ids, uint8_t* __restrict__ y, int num_tokens,
                                                       int hidden, int top_k, uint32_t num_experts, int col_block, int block, Coefficient&& coefficient) {
  using Off = typename SplitOff<SMALL>::type;
  constexpr int E = Row16<DT>::kElems, GP = kWave / LPR;
  constexpr int LD = LPR < 8 ? LPR : 8;
  const int lane = lane_id(), sub = lane % LPR, grp = lane / LPR;
  const int slice = block % kSlices;
  const int t = ((int)(block / kSlices) * WAVES + (threadIdx.x >> 6)) * GP + grp;
  const bool live = t < num_tokens;
  const int tt = live ? t : 0;
  const Off row_bytes = Off(hidden) * (16 / E);
  const Off col = (Off(col_block) * kSlices + slice) * LPR * 16 + sub * 16;
  const Off base = split_mul<SMALL>((uint32_t)tt, (Off)top_k);
  float acc[E];
#pragma unroll
  for (int i = 0; i < E; ++i) acc[i] = 0.f;
  for (int jb = 0; jb < top_k; jb += LPR) {
    const int j = jb + sub;
    int my_id = -1;                                               // -1: a padded slot or an id outside the table
    if (j < top_k) {
      const int id = ids[base + j];
      if ((uint32_t)id < num_experts) my_id = id;
    }
    // the down rows only need the ids: the first LD of them are requested ahead of the partial sums the coefficients
    // wait for; every row that has been added makes room for the request of a later one (LD row registers in all)
    u32x4_t vr[LD];
    bool used[LD];
    auto request = [&](int slot, int e) {
      const int id = __shfl(my_id, grp * LPR + e, kWave);         // from the lane of this group that holds pair e
      used[slot] = id >= 0;
      vr[slot] = *(const u32x4_t*)(down + (split_mul<SMALL>(used[slot] ? (uint32_t)id : 0u, row_bytes) + col));
    };
#pragma unroll
    for (int e = 0; e < LD; ++e) request(e, e);
    float coef = 0.f;
    if (kAll ? live && j < top_k : my_id >= 0) coef = coefficient(tt, base + j, j, my_id >= 0);
#pragma unroll
    for (int e = 0; e < LPR; ++e) {
      const float cf = __shfl(coef, grp * LPR + e, kWave);
      if (used[e % LD]) axpy16<DT>(cf, vr[e % LD], acc);          // not even 0 * row: the stand-in row may hold Inf or NaN
      if (e + LD < LPR) request(e % LD, e + LD);
    }
  }
  if (live) *(u32x4_t*)(y + (split_mul<SMALL>((uint32_t)t, row_bytes) + col)) = pack16<DT>(acc);
}

// lanes per row slice, or 0 when the row does not cut into 8 slices of 4..64 lanes
static inline int split_lanes_per_row(int hidden, int elem_bytes) {
  const int64_t slice_bytes = (int64_t)hidden * elem_bytes / kSlices;
  if ((int64_t)hidden * elem_bytes % (kSlices * 16) != 0) return 0;
  const int lpr = (int)(slice_bytes / 16);
  return (lpr == 4 || lpr == 8 || lpr == 16 || lpr == 32 || lpr == 64) ? lpr : 0;
}
// Rows beyond 8 KiB (8 slices of 64 lanes): the smallest number of column blocks, each 8 slices of a power-of-two number of
// lanes, that the row cuts into; 0 if there is none (up to 64 blocks: rows of 512 KiB).  1 for rows that split_lanes_per_row takes.
constexpr int kMaxColBlocks = 64;
static inline int split_col_blocks(int hidden, int elem_bytes, int* lanes_per_row) {
  for (int b = 1; b <= kMaxColBlocks; ++b) {
    if (hidden % b != 0) continue;
    const int lpr = split_lanes_per_row(hidden / b, elem_bytes);
    if (lpr) { *lanes_per_row = lpr; return b; }
  }
  return 0;
}

// every byte offset into x, y, the tables and the partial sums fits 32 bits, and the factors of its products 24
static inline bool split_offsets_small(int64_t T, int H, int k, int64_t N, int col_blocks, int elem_bytes) {
  const int64_t row = (int64_t)H * elem_bytes, lim = (int64_t)1 << 32, f24 = (int64_t)1 << 24;
  return row < f24 && N < f24 && T < f24 && k < f24 && N * row < lim && T * row < lim && T * k < lim &&
         (int64_t)kSlices * col_blocks * T * k * 4 < lim;
}

}  // namespace omni
