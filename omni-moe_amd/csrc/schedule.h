// The passes of the pair schedule as device functions (schedule.hip has what they do and why): its own kernels and the launches of the
// expert backward that sort beside the token pass share them.
#pragma once
#include "common.h"

namespace omni {

constexpr int kSortThreads = 512;
constexpr int kSortWaves = kSortThreads / kWave;
constexpr int kBinSlices = 8;                             // bin slices = XCDs
constexpr int kMaxBins = 4097;                            // 4096 experts (or id slices) + 1 bin for ids outside [0, N)
constexpr int kMaxBinsWide = 16385;                       // ... of a single pass over few pairs: what a block's tables leave room for in LDS
constexpr int kBinChunk = 8;                              // bins per 16-byte load of a histogram row
constexpr int slice_width(int bins) { return ((bins + kBinSlices - 1) / kBinSlices + kBinChunk - 1) / kBinChunk * kBinChunk; }   // bins per slice
constexpr int kMaxSortTiles = 1024;
constexpr int kMaxTile = 63 * 1024;                       // counters are 16 bits wide
constexpr int kRowBatch = 8;                              // histogram rows a thread has in flight
constexpr int kGroup = 8;                                 // steps of 64 items whose loads are issued together
static_assert(kBinSlices == kSortWaves, "the count kernel sums slice w in wave w");

struct SortPass {
  const int32_t* keys_in;   // expert ids, in the order left by the previous pass
  const int32_t* vals_in;   // pair ids travelling with them; NULL = position (first pass)
  int32_t* keys_out;        // NULL: not needed (single pass)
  int32_t* vals_out;
  int32_t* tok_out;         // NULL, or pair id / top_k (last pass)
  int32_t* offsets_out;     // NULL, or [bins]: first output position of every bin (single pass: the segment offsets)
  uint16_t* hist;           // [tiles][stride] bin counts of every tile
  uint32_t* slice_tot;      // [tiles][8] the same counts summed over each slice
  int64_t num_pairs;
  int tile;                 // pairs per tile, a multiple of 512
  int tiles, bins;
  int width, stride;        // bins per slice (a multiple of 8); stride = 8 * width >= bins
  int shift;                // digit = id >> shift ...
  uint32_t mask;            //   ... & mask (0xFFFFFFFF on the last pass)
  int last;                 // last pass: ids outside [0, N) go to bin bins-1; earlier passes: to bin 0
  uint32_t num_experts;
  uint64_t inv_top_k;       // ceil(2^s / top_k) with s = inv_shift = 30 + ceil(log2(top_k)): (v * inv_top_k) >> s == v / top_k for
  int inv_shift;            // every pair id v < 2^30 (the excess v * (inv_top_k * top_k - 2^s) / (top_k * 2^s) stays below
                            // 1 / top_k, and the product below 2^62)
};

__device__ __forceinline__ int sort_digit(const SortPass& a, int32_t key) {
  const bool valid = (uint32_t)key < a.num_experts;
  const int d = (int)(((uint32_t)key >> a.shift) & a.mask);
  return valid ? d : (a.last ? a.bins - 1 : 0);
}

__device__ __forceinline__ int32_t wave_sum_i32(int32_t v) {
#pragma unroll
  for (int m = kWave / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m, kWave);
  return v;
}

// A block of the count kernel: tile `block`.  cnt: [stride] in LDS.
__device__ __forceinline__ void sort_count_block(const SortPass& a, const int block, int32_t* cnt) {
  for (int d = threadIdx.x; d < a.stride; d += kSortThreads) cnt[d] = 0;
  __syncthreads();
  const int64_t t0 = (int64_t)block * a.tile;
  const int64_t t1 = t0 + a.tile < a.num_pairs ? t0 + a.tile : a.num_pairs;
  for (int64_t i0 = t0 + threadIdx.x; i0 < t1; i0 += kGroup * kSortThreads) {
    int32_t key[kGroup];
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      const int64_t i = i0 + u * kSortThreads;
      key[u] = i < t1 ? a.keys_in[i] : 0;
    }
#pragma unroll
    for (int u = 0; u < kGroup; ++u)
      if (i0 + u * kSortThreads < t1) atomicAdd(&cnt[sort_digit(a, key[u])], 1);
  }
  __syncthreads();
  for (int c = threadIdx.x; c < a.stride / kBinChunk; c += kSortThreads) {    // 8 counters per 16-byte store
    const int32_t* v = cnt + c * kBinChunk;
    *(u32x4_t*)(a.hist + (int64_t)block * a.stride + c * kBinChunk) =
        u32x4_t{(uint32_t)v[0] | ((uint32_t)v[1] << 16), (uint32_t)v[2] | ((uint32_t)v[3] << 16),
                (uint32_t)v[4] | ((uint32_t)v[5] << 16), (uint32_t)v[6] | ((uint32_t)v[7] << 16)};
  }
  const int lane = lane_id(), wave = threadIdx.x >> 6;   // wave w sums slice w
  int32_t sum = 0;
  for (int d = lane; d < a.width; d += kWave) sum += cnt[wave * a.width + d];
  sum = wave_sum_i32(sum);
  if (lane == 0) a.slice_tot[(int64_t)block * kBinSlices + wave] = (uint32_t)sum;
}

// A block of the scatter kernel: tile block / 8, slice block % 8.  tables: [(waves + 3) * width] in LDS.
// Of a sort of one tile every block counts all pairs for itself, so no count kernel runs in front of it.
__device__ __forceinline__ void sort_scatter_block(const SortPass& a, const int block, int32_t* tables) {
  int32_t* tbl = tables;                                 // [wave][width]: per wave and bin: count, then running output position
  int32_t *bin_base = tbl + kSortWaves * a.width, *before_s = bin_base + a.width, *total_s = before_s + a.width;
  __shared__ int32_t wave_total_s[kSortWaves];
  __shared__ int32_t below_s;                            // pairs in the slices below this one, all tiles
  const int lane = lane_id(), wave = threadIdx.x >> 6;
  const int tile_idx = block / kBinSlices, slice = block % kBinSlices;
  const int lo = slice * a.width;                        // this block's bins: lo .. lo + width - 1
  // The histogram rows come from other blocks' writes, i.e. from memory.  Thread t sums chunk t % C (8 bins, one
  // 16-byte load per row) of the rows t / C, t / C + G, ..; the first batch of loads flies while the tile is counted.
  const int C = a.width / kBinChunk, G = kSortThreads / C;
  const int chunk = threadIdx.x % C, group = threadIdx.x / C;
  const bool one = a.tiles == 1, summing = group < G && !one;
  auto load_rows = [&](u32x4_t (&row)[kRowBatch], int first) {
#pragma unroll
    for (int j = 0; j < kRowBatch; ++j) {
      const int r = first + j * G;
      row[j] = (summing && r < a.tiles) ? *(const u32x4_t*)(a.hist + (int64_t)r * a.stride + lo + chunk * kBinChunk) : u32x4_t{0, 0, 0, 0};
    }
  };
  u32x4_t early[kRowBatch];
  load_rows(early, group);
  for (int d = threadIdx.x; d < kSortWaves * a.width; d += kSortThreads) tbl[d] = 0;
  for (int d = threadIdx.x; d < a.width; d += kSortThreads) bin_base[d] = before_s[d] = total_s[d] = 0;
  if (threadIdx.x == 0) below_s = 0;
  __syncthreads();

  const int64_t t0 = (int64_t)tile_idx * a.tile;
  const int64_t t1 = t0 + a.tile < a.num_pairs ? t0 + a.tile : a.num_pairs;
  const int per_wave = a.tile / kSortWaves;
  const int64_t w0 = t0 + (int64_t)wave * per_wave < t1 ? t0 + (int64_t)wave * per_wave : t1;   // this wave's eighth, in order
  const int64_t w1 = w0 + per_wave < t1 ? w0 + per_wave : t1;
  int32_t* mine = tbl + wave * a.width;
  int32_t lower = 0;                                     // this lane's pairs in the slices below
  for (int64_t g0 = w0; g0 < w1; g0 += kGroup * kWave) {
    int32_t key[kGroup];
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      const int64_t i = g0 + u * kWave + lane;
      key[u] = i < w1 ? a.keys_in[i] : 0;
    }
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      const int d = sort_digit(a, key[u]) - lo;
      const bool in = g0 + u * kWave + lane < w1;
      if (in && (uint32_t)d < (uint32_t)a.width) atomicAdd(&mine[d], 1);
      lower += in && d < 0 ? 1 : 0;
    }
  }

  // what the slices below this one hold, over all tiles
  {
    int32_t part = lower;
    if (!one) {
      part = 0;
      for (int e = threadIdx.x; e < a.tiles * kBinSlices; e += kSortThreads)
        part += (e % kBinSlices) < slice ? (int32_t)a.slice_tot[e] : 0;
    }
    part = wave_sum_i32(part);
    if (lane == 0 && part) atomicAdd(&below_s, part);
  }
  // this slice of the histogram rows: what earlier tiles put into each bin, and each bin's total
  if (one) {
    __syncthreads();                                       // the waves' counts are complete
    for (int d = threadIdx.x; d < a.width; d += kSortThreads) {
      int32_t sum = 0;
#pragma unroll
      for (int w = 0; w < kSortWaves; ++w) sum += tbl[w * a.width + d];
      total_s[d] = sum;
    }
  } else {
    int32_t before[kBinChunk], rest[kBinChunk];
#pragma unroll
    for (int i = 0; i < kBinChunk; ++i) before[i] = rest[i] = 0;
    auto add_rows = [&](const u32x4_t (&row)[kRowBatch], int first) {
      auto add = [&](int32_t (&acc)[kBinChunk], const u32x4_t& r) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[2 * i] += (int32_t)(r[i] & 0xffffu);
          acc[2 * i + 1] += (int32_t)(r[i] >> 16);
        }
      };
#pragma unroll
      for (int j = 0; j < kRowBatch; ++j) {
        if (first + j * G < tile_idx) add(before, row[j]);
        else add(rest, row[j]);                            // rows past the last tile were loaded as zeros
      }
    };
    add_rows(early, group);
    for (int r0 = group + kRowBatch * G; r0 < a.tiles; r0 += kRowBatch * G) {
      u32x4_t row[kRowBatch];
      load_rows(row, r0);
      add_rows(row, r0);
    }
    if (summing) {
#pragma unroll
      for (int i = 0; i < kBinChunk; ++i) {
        if (before[i]) atomicAdd(&before_s[chunk * kBinChunk + i], before[i]);
        if (before[i] + rest[i]) atomicAdd(&total_s[chunk * kBinChunk + i], before[i] + rest[i]);
      }
    }
  }
  __syncthreads();

  // exclusive scan of the slice's totals (a run of consecutive bins per thread): every bin's first position
  {
    const int per = (a.width + kSortThreads - 1) / kSortThreads, b0 = (int)threadIdx.x * per;
    int32_t sum = 0;
    for (int i = 0; i < per; ++i) sum += b0 + i < a.width ? total_s[b0 + i] : 0;
    int32_t inc = sum;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int32_t o = __shfl_up(inc, d, kWave);
      if (lane >= d) inc += o;
    }
    if (lane == kWave - 1) wave_total_s[wave] = inc;
    __syncthreads();
    int32_t excl = below_s + inc - sum;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) excl += w < wave ? wave_total_s[w] : 0;
    for (int i = 0; i < per; ++i) {
      const int b = b0 + i;
      if (b < a.width) {
        if (a.offsets_out && tile_idx == 0 && lo + b < a.bins) a.offsets_out[lo + b] = excl;
        bin_base[b] = excl + before_s[b];
        excl += total_s[b];
      }
    }
  }
  __syncthreads();
  // per-wave bases: consecutive threads take consecutive bins (no bank conflicts), wave by wave down the table
  for (int d = threadIdx.x; d < a.width; d += kSortThreads) {
    int32_t base = bin_base[d];
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
      const int32_t c = tbl[w * a.width + d];
      tbl[w * a.width + d] = base;
      base += c;
    }
  }
  __syncthreads();

  // Placement, 64 consecutive items at a time and in order; only the items of this block's slice take part.
  // Position = the bin's running base + the number of earlier lanes of the step with the same bin.  Every lane
  // reads the base, then bumps it; a lane that finds the base already bumped shares its bin with another lane of
  // its step, and only then are the lanes of that bin ranked by lane number (whatever order the adds took effect
  // in).  LDS executes a wave's instructions in order, so the reads and adds of all steps of a group are issued
  // back to back (a later step sees the earlier steps' adds) and waited for once.
  const uint64_t below = (1ull << lane) - 1ull;
  for (int64_t g0 = w0; g0 < w1; g0 += kGroup * kWave) {
    int32_t keys[kGroup], vals[kGroup], dig[kGroup], pos[kGroup], bumped[kGroup];
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      const int64_t i = g0 + u * kWave + lane;
      keys[u] = i < w1 ? a.keys_in[i] : 0;
      vals[u] = i < w1 ? (a.vals_in ? a.vals_in[i] : (int32_t)i) : 0;
    }
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      dig[u] = sort_digit(a, keys[u]) - lo;
      const bool active = g0 + u * kWave + lane < w1 && (uint32_t)dig[u] < (uint32_t)a.width;
      pos[u] = bumped[u] = 0;
      if (active) {
        pos[u] = mine[dig[u]];
        bumped[u] = atomicAdd(&mine[dig[u]], 1);
      } else {
        dig[u] = -1;
      }
    }
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      const int d = dig[u];
      const bool active = d >= 0;
      uint64_t shared = __ballot(active && bumped[u] != pos[u]);   // the non-first lanes of shared bins
      while (shared) {
        const int l = __builtin_ctzll(shared);
        const int v = __shfl(d, l, kWave);
        const uint64_t grp = __ballot(d == v);                     // all lanes of that bin; they read the same base
        if (d == v) pos[u] += __popcll(grp & below);
        shared &= ~grp;
      }
      if (active) {
        if (a.keys_out) a.keys_out[pos[u]] = keys[u];
        a.vals_out[pos[u]] = vals[u];
        if (a.tok_out) a.tok_out[pos[u]] = (int32_t)(((uint64_t)(uint32_t)vals[u] * a.inv_top_k) >> a.inv_shift);   // val / top_k
      }
    }
  }
}

// The two kernels' tables in LDS
static inline int count_lds(int stride) { return stride * 4; }
static inline int scatter_lds(int width) { return (kSortWaves + 3) * width * 4; }

// How the sort of P pairs with ids below N is split into passes and tiles.
struct SortPlan {
  int passes, lo_bits, bins[2], width, stride, tile, tiles;
  size_t hist_entries;
};
// The arguments of a schedule that one counting pass does, for a launch of its own or one that it shares: tiles blocks of sort_count_block (none for
// one tile), then tiles * 8 of sort_scatter_block, all of kSortThreads threads.  False where it takes two passes.
bool schedule_single_pass(const int32_t* indices, int32_t* offsets, int32_t* sorted_pair_ids, int32_t* sorted_token_ids, int64_t num_tokens, int num_experts_per_token,
                          int64_t num_experts, void* workspace, SortPass* a);

}  // namespace omni
