// The hidden-split expert algorithm as device functions: the forward's kernels (expert.hip, where the algorithm is described) and the backward's
// token pass (backward.hip) share them.
#pragma once
#include "common.h"
#include "rows.h"

namespace omni {

constexpr int kXcds = 8;
constexpr int kSlices = 8;             // at most

// Sum over the LPR lanes of a group of N <= LPR values per lane, scattered: lane `sub` of the group
// ends up with the total of value sub % N.  Every step halves what a lane keeps (N - 1 exchanges
// in all, against N * log2(LPR) for one tree per value); lanes that hold the same value add up last.
template <int LPR, int N>
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
template <int LPR, int N, int D>
__device__ __forceinline__ float fold_group(float v, const int lane) {
  if constexpr (D >= N) return fold_group<LPR, N, D / 2>(v + xor_lane_f<D>(v, lane), lane);
  else return v;
}

// A block's place: which column slice of the rows (block % 8, the XCD that the dispatcher gives it to, names it) and which group of tokens
template <int S>
struct SplitPlace {
  int slice, tokens;
  __device__ __forceinline__ explicit SplitPlace(int block) : slice(block % S), tokens(block / kXcds * (kXcds / S) + block % kXcds / S) {}
};

// A value per lane, handed round inside each group of LPR lanes: get<E>() is lane E's, by register exchanges (__shfl, a ds_bpermute, would be a trip through
// LDS in front of every row's address and sum).
template <int LPR>
struct GroupValues {
  int v[2];
  __device__ __forceinline__ explicit GroupValues(int mine) : v{mine, mine} {
    if constexpr (LPR == 32) {                 // either half of the group in both of its rows of 16 lanes
      const auto s = __builtin_amdgcn_permlane16_swap(mine, mine, false, false);
      v[0] = (int)s[0];
      v[1] = (int)s[1];
    }
  }
  template <int E>
  __device__ __forceinline__ int get() const {
    if constexpr (LPR == 4) return dpp_i<E * 0x55>(v[0]);                       // quad_perm
    else if constexpr (LPR == 8) {                                                                            // row_newbcast, for either half of a row
      const int t = dpp_i<0x150 + E>(v[0]);
      return __builtin_amdgcn_update_dpp(t, v[0], 0x158 + E, 0xf, 0xC, false);
    } else if constexpr (LPR <= 32) return dpp_i<0x150 + E % 16>(v[E / 16]);
    else return __builtin_amdgcn_readlane(v[0], E);
  }
};

// A wave owns GP = 64 / LPR tokens, one per lane group; the group's LPR lanes cover the token's
// row slice, 16 bytes each (RAGGED: its first `lanes` do; the others repeat the first and what they have is dropped).  Pairs go in batches of B = min(LPR, 16): B partial dot products per lane,
// then one reduce-scatter leaves pair `sub % B` of the batch in lane `sub`.
//
// What bounds the passes: vector instructions beside the path into the CU, which takes 16 cycles for 1 KiB of row -- time for 16 vector instructions of the
// CU's four SIMDs, of which the sums alone are 4 (dot products) or 16 (unpacking and adding).  So what goes round a row is kept to an address and a
// coefficient, one instruction each:
// SMALL: every table, x, y and the partial sums stay below 4 GiB, ids and row lengths below 2^24 (split_offsets_small): lane `sub` forms the row offset of its
// pair once, the others add their column to it, and a pair without a row has the table's end for one: buffer loads return zeros there, so nothing is asked
// about it later.  Otherwise 64-bit addresses, one per lane and row.
// What the slices cost is the partial sums' trip over the fabric (split_slices).  16384 tokens x 16 over 4096 experts, hidden 1024, bf16: 27.6 + 34.8 us
// with exchanges through LDS, 64-bit addresses in the second pass and eight slices, 25.4 + 28.5 so; 4096 tokens 9.7 + 12.1 -> 9.2 + 8.5.
template <bool SMALL> struct SplitOff { using type = int64_t; };
template <> struct SplitOff<true> { using type = uint32_t; };
template <bool SMALL>
__device__ __forceinline__ typename SplitOff<SMALL>::type split_mul(uint32_t a, typename SplitOff<SMALL>::type b) {
  if constexpr (SMALL) return __umul24(a, b); else return (int64_t)a * b;
}

// The table rows of a batch: row<E>() is this lane's 16 bytes of pair E's row, zeros where the pair has none.
template <int LPR, bool SMALL> struct SplitRows;
template <int LPR> struct SplitRows<LPR, true> {
  __amdgpu_buffer_rsrc_t table;
  GroupValues<LPR> at;
  uint32_t col;
  __device__ __forceinline__ SplitRows(const uint8_t* base, uint32_t row_bytes, uint32_t num_rows, int id, uint32_t column)
      : table(__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)(num_rows * row_bytes), 0x00020000)),
        at((int)__umul24((uint32_t)id < num_rows ? (uint32_t)id : num_rows, row_bytes)), col(column) {}
  template <int E>
  __device__ __forceinline__ u32x4_t row() const {
    return __builtin_amdgcn_raw_buffer_load_b128(table, (int)((uint32_t)at.template get<E>() + col), 0, 0);
  }
};
template <int LPR> struct SplitRows<LPR, false> {
  const uint8_t* table;
  int64_t bytes, col;
  GroupValues<LPR> at;
  __device__ __forceinline__ SplitRows(const uint8_t* base, int64_t row_bytes, uint32_t num_rows, int id, int64_t column)
      : table(base), bytes(row_bytes), col(column), at((uint32_t)id < num_rows ? id : -1) {}
  template <int E>
  __device__ __forceinline__ u32x4_t row() const {
    const int id = at.template get<E>();
    const u32x4_t v = *(const u32x4_t*)(table + ((id >= 0 ? (int64_t)id * bytes : 0) + col));
    const uint32_t keep = id >= 0 ? ~0u : 0u;                  // not even 0 * row: the stand-in row may hold Inf or NaN
    return u32x4_t{v[0] & keep, v[1] & keep, v[2] & keep, v[3] & keep};
  }
};

// Partial dot products <a[t, slice], table[id, slice]> of the k pairs of a block's tokens -> partial[slice][t][j].  block % 8 names the slice (SplitPlace), WAVES the block's
// waves.  (rows wider than 8 slices of 64 lanes go in column blocks of 8 slices, one launch each)
template <int DT, int LPR, int S, bool RAGGED, bool SMALL, int WAVES>
__device__ __forceinline__ void split_dots_block(const uint8_t* __restrict__ x, const uint8_t* __restrict__ up, const int32_t* __restrict__ ids,
                                                 float* __restrict__ partial, int num_tokens, int hidden, int top_k, uint32_t num_experts, int lanes, int col_block, int block) {
  using Off = typename SplitOff<SMALL>::type;
  constexpr int E = Row16<DT>::kElems, GP = kWave / LPR;
  constexpr int B = LPR < 16 ? LPR : 16, LD = LPR < 8 ? LPR : 8;     // row loads in flight at a time
  const int lane = lane_id(), sub = lane % LPR, grp = lane / LPR;
  const SplitPlace<S> place(block);
  const int t = (place.tokens * WAVES + (int)(threadIdx.x >> 6)) * GP + grp;
  const bool live = t < num_tokens;
  const int tt = live ? t : 0;
  const Off row_bytes = Off(hidden) * (16 / E);
  // this lane's 16 bytes inside a row
  const int width = RAGGED ? lanes : LPR;
  const bool inside = !RAGGED || sub < lanes;
  const Off col = (Off(col_block) * S + place.slice) * width * 16 + (inside ? sub : 0) * 16;
  const u32x4_t xr = *(const u32x4_t*)(x + (split_mul<SMALL>((uint32_t)tt, row_bytes) + col));
  const Off base = split_mul<SMALL>((uint32_t)tt, (Off)top_k);
  for (int jb = 0; jb < top_k; jb += B) {
    // lane `sub` of a group fetches the id of pair `sub % B` of the batch
    const int j = jb + sub % B;
    const SplitRows<LPR, SMALL> rows(up, row_bytes, num_experts, j < top_k ? ids[base + j] : -1, col);
    float d[B];
    auto batch = [&](auto n_tag) __attribute__((always_inline)) {
      constexpr int e0 = decltype(n_tag)::value * LD;
      if (e0 > 0 && jb + e0 >= top_k) {                          // (few pairs to a token: not the whole batch)
#pragma unroll
        for (int e = 0; e < LD; ++e) d[e0 + e] = 0.f;
        return;
      }
      u32x4_t ur[LD];
      auto request = [&](auto... e) __attribute__((always_inline)) { ((ur[decltype(e)::value] = rows.template row<e0 + decltype(e)::value>()), ...); };
      with_sequence(request, std::make_integer_sequence<int, LD>{});
#pragma unroll
      for (int e = 0; e < LD; ++e) d[e0 + e] = inside ? dot16<DT>(xr, ur[e], 0.f) : 0.f;
      if constexpr (!SMALL) __builtin_amdgcn_sched_barrier(0);   // (a batch's 64-bit addresses at a time)
    };
    auto batches = [&](auto... n) __attribute__((always_inline)) { (batch(n), ...); };
    with_sequence(batches, std::make_integer_sequence<int, B / LD>{});
    const float total = fold_group<LPR, B, LPR / 2>(reduce_scatter_group<LPR, B>(d, lane), lane);
    if (live && j < top_k && sub < B) partial[((Off(col_block) * S + place.slice) * num_tokens + t) * top_k + j] = total;
  }
}

// Same ownership.  Lane `sub` of a group forms the coefficient of pair `sub % B` of a batch from the sums over the slices, and the group then walks the batch,
// every lane fetching its 16 bytes of the pair's row and the coefficient from the lane that holds it.  The coefficient comes in two steps so that its
// operands are requested ahead of the rows (loads return in order) and waited for behind the rows' requests: pair.request(token, place of the pair, slot,
// id inside the table), called with `there` for slots below top_k of live tokens, then pair.value().
template <int DT, int LPR, int S, bool RAGGED, bool SMALL, int WAVES, class Pair>
__device__ __forceinline__ void split_accumulate_block(const uint8_t* __restrict__ down, const int32_t* __restrict__ ids, uint8_t* __restrict__ y, int num_tokens,
                                                       int hidden, int top_k, uint32_t num_experts, int lanes, int col_block, int block, Pair&& pair) {
  using Off = typename SplitOff<SMALL>::type;
  constexpr int E = Row16<DT>::kElems, GP = kWave / LPR;
  constexpr int B = LPR < 16 ? LPR : 16, LD = LPR < 8 ? LPR : 8;
  const int lane = lane_id(), sub = lane % LPR, grp = lane / LPR;
  const SplitPlace<S> place(block);
  const int t = (place.tokens * WAVES + (int)(threadIdx.x >> 6)) * GP + grp;
  const bool live = t < num_tokens;
  const int tt = live ? t : 0;
  const Off row_bytes = Off(hidden) * (16 / E);
  const int width = RAGGED ? lanes : LPR;
  const bool inside = !RAGGED || sub < lanes;
  const Off col = (Off(col_block) * S + place.slice) * width * 16 + (inside ? sub : 0) * 16;
  const Off base = split_mul<SMALL>((uint32_t)tt, (Off)top_k);
  float acc[E];
#pragma unroll
  for (int i = 0; i < E; ++i) acc[i] = 0.f;
  for (int jb = 0; jb < top_k; jb += B) {
    const int j = jb + sub % B;
    const bool there = live && j < top_k;
    const int my_id = there ? ids[base + j] : -1;
    pair.request(there, tt, base + min(j, top_k - 1), min(j, top_k - 1), (uint32_t)my_id < num_experts);
    __builtin_amdgcn_sched_barrier(0);
    // every row that has been added makes room for the request of a later one (LD row registers in all)
    const SplitRows<LPR, SMALL> rows(down, row_bytes, num_experts, my_id, col);
    u32x4_t vr[LD];
    auto first = [&](auto... e) __attribute__((always_inline)) { ((vr[decltype(e)::value] = rows.template row<decltype(e)::value>()), ...); };
    with_sequence(first, std::make_integer_sequence<int, LD>{});
    __builtin_amdgcn_sched_barrier(0);
    const GroupValues<LPR> factor(__float_as_int(pair.value()));
    auto add = [&](auto e_tag, auto more) __attribute__((always_inline)) {
      constexpr int e = decltype(e_tag)::value;
      axpy16<DT>(__int_as_float(factor.template get<e>()), vr[e % LD], acc);
      if constexpr (decltype(more)::value && e + LD < B) vr[e % LD] = rows.template row<e + LD>();
      if constexpr (!SMALL) __builtin_amdgcn_sched_barrier(0);
    };
    auto few = [&](auto... e) __attribute__((always_inline)) { (add(e, std::false_type{}), ...); };
    auto every = [&](auto... e) __attribute__((always_inline)) { (add(e, std::true_type{}), ...); };
    if (LD < B && jb + LD >= top_k) with_sequence(few, std::make_integer_sequence<int, LD>{});
    else with_sequence(every, std::make_integer_sequence<int, B>{});
  }
  if (live && inside) *(u32x4_t*)(y + (split_mul<SMALL>((uint32_t)t, row_bytes) + col)) = pack16<DT>(acc);
}

// lanes per row slice, or 0 when the row does not cut into `slices` slices of 4..64 lanes
static inline int split_lanes_per_row(int hidden, int elem_bytes, int slices) {
  const int64_t row = (int64_t)hidden * elem_bytes;
  const int64_t lanes = row / (slices * 16);
  return row % (slices * 16) == 0 && lanes >= 4 && lanes <= 64 ? (int)lanes : 0;
}
// Slices of a row of at most 8 KiB, or 0 where it does not cut: four, each for two XCDs that share out the tokens, or eight.  Fewer slices mean fewer partial
// sums (every slice's blocks read those of all slices: 4 bytes a pair and slice, across the fabric) and longer pieces; more slices mean that an XCD
// keeps a larger part of the table's rows in its 4 MiB L2.  Time with four over eight, bf16, 4096 to 32768 tokens x 16 or 32, ids uniform:
//   rows  512 B, 1 KiB, 1.5 KiB, 2.5 KiB: 0.2-0.6, 0.4-0.9, 0.7-0.9, 0.8-1.0 at tables of 0.5 to 640 MB (2.5 KiB x 40 MB: 1.0-1.07)
//   rows  2 KiB: 0.84-1.04 up to 16 MB, 1.1-1.35 at 32 MB, 0.85-0.99 from 128 MB on
//   rows  4 KiB: 0.88-1.01 up to 16 MB, 1.1-1.5 at 32 and 64 MB, 0.94-1.04 from 256 MB on; 1 GB with the ids of a router that keeps to 3700 rows 1.05-1.1
//   rows  8 KiB: eight slices of 64 lanes
static inline int split_slices(int hidden, int64_t num_experts, int elem_bytes) {
  const int64_t row = (int64_t)hidden * elem_bytes, table = num_experts * row;
  const int four = split_lanes_per_row(hidden, elem_bytes, 4);
  if (four >= 5 && (row < 2048 || table <= (24ll << 20) || (row < 4096 && table >= (128ll << 20)))) return 4;
  return split_lanes_per_row(hidden, elem_bytes, kSlices) ? kSlices : four >= 5 ? 4 : 0;
}
// Rows beyond 8 KiB: the smallest number of column blocks, each 8 slices of a power-of-two number of lanes, that the row cuts into; 0 if there is none (up
// to 64 blocks: rows of 512 KiB).  Shorter rows for which it is 0 are refused where the algorithm is asked for by name.
constexpr int kMaxColBlocks = 64;
static inline int split_col_blocks(int hidden, int elem_bytes, int* lanes_per_row) {
  for (int b = 1; b <= kMaxColBlocks; ++b) {
    if (hidden % b != 0) continue;
    const int lpr = split_lanes_per_row(hidden / b, elem_bytes, kSlices);
    if (lpr && (lpr & (lpr - 1)) == 0) { *lanes_per_row = lpr; return b; }
  }
  return 0;
}
// How a row is cut: the slices of its lanes, in one column block up to 8 KiB
struct SplitCut { int slices, lanes, col_blocks; };
static inline SplitCut split_cut(int hidden, int64_t num_experts, int elem_bytes) {
  if ((int64_t)hidden * elem_bytes <= 8192)
    if (const int s = split_slices(hidden, num_experts, elem_bytes)) return {s, split_lanes_per_row(hidden, elem_bytes, s), 1};
  SplitCut c{kSlices, 0, 0};
  c.col_blocks = split_col_blocks(hidden, elem_bytes, &c.lanes);
  return c;
}

// every byte offset into x, y, the tables (and a row beyond them) and the partial sums fits 32 bits, and the factors of its products 24; the tables lie on
// 16-byte boundaries, which buffer loads of 16 bytes are specified for (views into a flat buffer may lie anywhere)
static inline bool split_offsets_small(const void* up, const void* down, int64_t T, int H, int k, int64_t N, int col_blocks, int elem_bytes) {
  if (((uintptr_t)up | (uintptr_t)down) % 16) return false;
  const int64_t row = (int64_t)H * elem_bytes, lim = (int64_t)1 << 32, f24 = (int64_t)1 << 24;
  return row < f24 && N + 1 < f24 && T < f24 && k < f24 && (N + 1) * row < lim && T * row < lim && T * k < lim &&
         (int64_t)kSlices * col_blocks * T * k * 4 < lim;
}

// blocks of a launch whose blocks own `per_block` tokens each in one of the slices: whole rounds of the eight XCDs
static inline int64_t split_blocks(int64_t T, int per_block, int slices) {
  const int64_t groups = (T + per_block - 1) / per_block, a_round = kXcds / slices;
  return (groups + a_round - 1) / a_round * kXcds;
}
// go(lanes of a group, slices, ragged), all as types: the power of two that `lanes` of a slice take, and whether that is more than they are
template <class Go>
static inline hipError_t split_dispatch(int lanes, int slices, Go&& go) {
  auto by_slices = [&](auto group) -> hipError_t {
    constexpr int LPR = decltype(group)::value;
    auto by_lanes = [&](auto s) -> hipError_t {
      if constexpr (LPR > 4) {                                   // (no slice has fewer lanes: split_lanes_per_row)
        if (lanes != LPR) return go(group, s, std::true_type{});
      }
      return go(group, s, std::false_type{});
    };
    if (slices == 4) {
      if constexpr (LPR >= 8) return by_lanes(std::integral_constant<int, 4>{});
      else return hipErrorInvalidValue;
    }
    return slices == kSlices ? by_lanes(std::integral_constant<int, kSlices>{}) : hipErrorInvalidValue;
  };
  if (lanes < 4 || lanes > 64) return hipErrorInvalidValue;
  if (lanes == 4) return by_slices(std::integral_constant<int, 4>{});
  if (lanes <= 8) return by_slices(std::integral_constant<int, 8>{});
  if (lanes <= 16) return by_slices(std::integral_constant<int, 16>{});
  if (lanes <= 32) return by_slices(std::integral_constant<int, 32>{});
  return by_slices(std::integral_constant<int, 64>{});
}

}  // namespace omni
