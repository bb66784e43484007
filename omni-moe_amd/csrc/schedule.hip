// Expert-centric schedule for gfx950: a stable counting sort of the (token, expert) pairs.
//
// Replaces get_scheduling_info's tail part (omni_moe/ops/triton/omni_scheduler.py:48-101),
// which runs ~12 torch launches including a radix sort and reads two results back to
// the host (:82, :90).  Here the pairs are sorted by expert id with one counting pass (one bin per
// expert) when N <= 4096, or N <= 16384 with few pairs, and two passes (low then high half of the id bits) above that.
// A pass is two kernels:
//   count:   (where there is more than one tile) every block counts the bins of its contiguous tile of the input in LDS and writes
//            them as one row of hist[tile][bin] (16-bit counters: a tile has fewer than 65536
//            pairs), plus the row's sum over each of the 8 bin slices;
//   scatter: the bins are cut into 8 slices and a block places the pairs of ONE tile that fall
//            into ONE slice.  It sums its slice of the hist rows (all rows for the bins' totals,
//            the rows above its tile for its share), the slice sums of the slices below it, scans
//            the totals, and has its output bases; the blocks of tile 0 write them out as the
//            segment offsets.
// Why slices: the scattered 4-byte stores are what the pass costs.  Slice s belongs to the blocks
// with blockIdx % 8 == s, which the dispatcher places on XCD s, so every output line is written
// through ONE L2 (which merges the stores of a line before it goes to memory) and the stores are
// spread over all CUs; and a block's tables cover an eighth of the bins, so zeroing, summing,
// scanning them is an eighth of the work.  The price is that a tile's keys are read by 8 blocks.
// The scatter is order preserving without any global atomic: each of the block's 8 waves owns a
// contiguous eighth of the tile; per-wave bin bases come from an LDS table, and inside a wave 64
// consecutive items rank themselves (an LDS add per item, ballots where two items of a step meet
// in a bin).  So a segment lists its pairs by ascending pair id, and the result is bit-identical
// from run to run.  Offsets are dense over all N experts (an unused expert has an empty segment),
// so no compaction pass is needed, and nothing returns to the host.
#include "common.h"
#include "omni_moe_hip.h"
#include "schedule.h"

#include <algorithm>

namespace omni {

__global__ __launch_bounds__(kSortThreads) void sort_count_kernel(const SortPass a) {
  extern __shared__ int32_t cnt[];                       // [stride]
  sort_count_block(a, (int)blockIdx.x, cnt);
}
__global__ __launch_bounds__(kSortThreads) void sort_scatter_kernel(const SortPass a) {
  extern __shared__ int32_t tables[];
  sort_scatter_block(a, (int)blockIdx.x, tables);
}

// offsets[e] = first position whose (sorted) id is >= e; ids outside [0, N) count as N.  Two-pass sorts only:
// their last pass has a bin per high half of the id, not per expert.
__global__ __launch_bounds__(256) void segment_offsets_kernel(const int32_t* __restrict__ sorted_keys, int32_t* __restrict__ offsets,
                                                              int64_t num_pairs, uint32_t num_experts) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i <= num_pairs; i += gridDim.x * 256ll) {
    const uint32_t n = num_experts;
    int64_t prev = -1, cur = n;
    if (i > 0) { const uint32_t k = (uint32_t)sorted_keys[i - 1]; prev = k < n ? k : n; }
    if (i < num_pairs) { const uint32_t k = (uint32_t)sorted_keys[i]; cur = k < n ? k : n; }
    for (int64_t e = prev + 1; e <= cur; ++e) offsets[e] = (int32_t)i;
  }
}

static inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

static inline int ceil_log2(uint64_t v) { int b = 0; while ((1ull << b) < v) ++b; return b; }

static LdsKernel g_count_kernel{(const void*)sort_count_kernel, slice_width(kMaxBinsWide) * kBinSlices * 4};
static LdsKernel g_scatter_kernel{(const void*)sort_scatter_kernel, (kSortWaves + 3) * slice_width(kMaxBinsWide) * 4};

// Up to so many pairs are one tile: every scatter block counts them all, and the count kernel's launch goes, for longer chains of steps in the scatter
// blocks.  One pass, 512 / 4096 / 8192 pairs over 1024 experts 9.0 / 9.2 / 9.4 -> 5.5 / 6.6 / 9.5 us, 8192 over 16384 15.0 -> 11.9; beside the expert
// backward's token pass (8000 pairs, hidden 512) 3.6 + 8.1 us in two launches -> 11.6 in one.  Two passes: 8000 pairs 22.6 -> 24.5, so half as many.
constexpr int kOneTile = 8192;

static bool make_plan(int64_t P, int64_t N, SortPlan* pl) {
  const int kb = ceil_log2((uint64_t)N);
  // A wave places an eighth of a tile, 64 items a step: tiles of 8192 pairs are 16 steps; at most 256 tiles (a scatter
  // block sums its slice of every tile's row), more only where a tile would outgrow its 16-bit counters
  int64_t tile = 8192;
  if ((P + tile - 1) / tile > 256) tile = ((P + 255) / 256 + 1023) / 1024 * 1024;
  if (tile > kMaxTile) tile = kMaxTile;
  // What the scatter blocks of n tiles read of the histogram in all: n rows each, one block per tile and slice.
  auto rows_read = [&](int64_t of_tile, int64_t bins) { const int64_t n = (P + of_tile - 1) / of_tile; return n * n * slice_width((int)bins) * kBinSlices * 2; };
  // A second pass and the offsets kernel behind it cost about 20 us, as do 64 MB of rows: 32768 pairs over 16384 experts 37 us in two
  // passes, 18 in one.
  const bool wide = N + 1 > kMaxBins && N + 1 <= kMaxBinsWide && rows_read(tile, N + 1) <= (64ll << 20);
  if (N + 1 <= kMaxBins || wide) { pl->passes = 1; pl->lo_bits = 0; pl->bins[0] = (int)N + 1; pl->bins[1] = 0; }
  else {
    pl->passes = 2; pl->lo_bits = kb / 2;
    pl->bins[0] = 1 << pl->lo_bits;
    pl->bins[1] = (int)((N + (1ll << pl->lo_bits) - 1) >> pl->lo_bits) + 1;
  }
  const int maxb = pl->bins[0] > pl->bins[1] ? pl->bins[0] : pl->bins[1];
  if (maxb > (wide ? kMaxBinsWide : kMaxBins)) return false;                       // N > 16 Mi experts
  pl->width = slice_width(maxb);
  pl->stride = pl->width * kBinSlices;
  // Few pairs: smaller tiles, for more blocks with fewer steps each, while the rows stay cheap to read (65536 pairs over 4096 experts:
  // scatter 11.5 -> 8.5 us)
  while (tile > 2048 && tile <= 8192 && rows_read(tile / 2, maxb) <= (16ll << 20)) tile /= 2;
  if ((P + tile - 1) / tile > kMaxSortTiles) return false;   // more than 64 Mi pairs
  pl->tile = (int)tile;
  pl->tiles = (int)((P + tile - 1) / tile);
  if (pl->tiles < 1) pl->tiles = 1;
  pl->hist_entries = (size_t)pl->stride * pl->tiles;
  if (P <= (pl->passes == 1 ? kOneTile : kOneTile / 2)) {
    pl->tile = (int)std::max<int64_t>((P + kSortThreads - 1) / kSortThreads, 1) * kSortThreads;
    pl->tiles = 1;
  }
  return true;
}

// What of a pass's arguments follows from the sizes and the workspace; the arrays it moves are the caller's
static SortPass make_pass(const SortPlan& pl, int pass, int64_t P, int top_k, int64_t N, uint16_t* hist, uint32_t* slice_tot) {
  SortPass a{};
  a.hist = hist;
  a.slice_tot = slice_tot;
  a.num_pairs = P;
  a.tile = pl.tile;
  a.tiles = pl.tiles;
  a.bins = pl.bins[pass];
  a.width = pl.width;
  a.stride = pl.stride;
  a.shift = pass == 0 ? 0 : pl.lo_bits;
  a.mask = (pl.passes == 2 && pass == 0) ? (uint32_t)((1 << pl.lo_bits) - 1) : 0xFFFFFFFFu;
  a.last = pass == pl.passes - 1 ? 1 : 0;
  a.num_experts = (uint32_t)N;
  a.inv_shift = 30;
  while ((1ll << (a.inv_shift - 30)) < (int64_t)top_k) ++a.inv_shift;
  a.inv_top_k = top_k > 0 ? ((1ull << a.inv_shift) + top_k - 1) / (uint64_t)top_k : 0;
  return a;
}

bool schedule_single_pass(const int32_t* indices, int32_t* offsets, int32_t* sorted_pair_ids, int32_t* sorted_token_ids, int64_t num_tokens, int num_experts_per_token,
                          int64_t num_experts, void* workspace, SortPass* a) {
  const int64_t P = num_tokens * (int64_t)num_experts_per_token;
  SortPlan pl;
  if (P > INT32_MAX / 2 || num_experts > INT32_MAX / 2 || !make_plan(P, num_experts, &pl) || pl.passes != 1) return false;
  *a = make_pass(pl, 0, P, num_experts_per_token, num_experts, (uint16_t*)workspace, (uint32_t*)((char*)workspace + align_up(pl.hist_entries * 2, 256)));
  a->keys_in = indices;
  a->vals_out = sorted_pair_ids;
  a->tok_out = sorted_token_ids;
  a->offsets_out = offsets;
  return true;
}

}  // namespace omni

// workspace: hist [tiles][stride] u16 | slice sums [tiles][8] u32 | two-pass sorts only: keys A [P] | keys B [P] | pair ids [P]
extern "C" OMNI_API size_t omni_schedule_workspace_bytes(int64_t num_tokens, int32_t num_experts_per_token, int64_t num_experts) {
  using namespace omni;
  const int64_t P = num_tokens * (int64_t)num_experts_per_token;
  SortPlan pl;
  if (num_tokens < 0 || num_experts_per_token < 0 || num_experts <= 0 || !make_plan(P, num_experts, &pl)) return 0;
  return align_up(pl.hist_entries * 2, 256) + align_up((size_t)pl.tiles * kBinSlices * 4, 256) +
         (pl.passes == 2 ? 3 * align_up((size_t)P * 4 + 4, 256) : 0);
}

extern "C" OMNI_API int32_t omni_schedule(const int32_t* indices, int32_t* offsets, int32_t* sorted_pair_ids,
                                          int32_t* sorted_token_ids, int64_t num_tokens, int32_t num_experts_per_token,
                                          int64_t num_experts, void* workspace, void* stream) {
  using namespace omni;
  const int64_t N = num_experts, P = num_tokens * (int64_t)num_experts_per_token;
  if (num_tokens < 0 || num_experts_per_token < 0 || N <= 0 || P > INT32_MAX / 2 || N > INT32_MAX / 2) return OMNI_ERR_SHAPE;
  SortPlan pl;
  if (!make_plan(P, N, &pl)) return OMNI_ERR_UNSUPPORTED;
  if (!offsets || (P > 0 && (!indices || !sorted_pair_ids))) return OMNI_ERR_NULL;
  if (!workspace) return OMNI_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  char* w = (char*)workspace;
  uint16_t* hist = (uint16_t*)w;     w += align_up(pl.hist_entries * 2, 256);
  uint32_t* slice_tot = (uint32_t*)w; w += align_up((size_t)pl.tiles * kBinSlices * 4, 256);
  int32_t* keys_a = (int32_t*)w;     w += align_up((size_t)P * 4 + 4, 256);      // the three arrays exist for two-pass sorts only
  int32_t* keys_b = (int32_t*)w;     w += align_up((size_t)P * 4 + 4, 256);
  int32_t* vals_a = (int32_t*)w;

  const bool single = pl.passes == 1;
  if (count_lds(pl.stride) > 65536 || scatter_lds(pl.width) > 65536) {
    if (hipError_t e = g_count_kernel.ensure(); e != hipSuccess) return OMNI_ERR_HIP_BASE + (int)e;
    if (hipError_t e = g_scatter_kernel.ensure(); e != hipSuccess) return OMNI_ERR_HIP_BASE + (int)e;
  }
  if (single || P > 0) {
    for (int pass = 0; pass < pl.passes; ++pass) {
      const bool last = pass == pl.passes - 1;
      SortPass a = make_pass(pl, pass, P, num_experts_per_token, N, hist, slice_tot);
      a.keys_in = pass == 0 ? indices : keys_a;
      a.vals_in = pass == 0 ? nullptr : vals_a;
      a.keys_out = single ? nullptr : (last ? keys_b : keys_a);
      a.vals_out = last ? sorted_pair_ids : vals_a;
      a.tok_out = last ? sorted_token_ids : nullptr;
      a.offsets_out = single ? offsets : nullptr;          // one bin per expert: the bins' first positions ARE the offsets
      if (a.tiles > 1) hipLaunchKernelGGL(sort_count_kernel, dim3(a.tiles), dim3(kSortThreads), count_lds(a.stride), s, a);
      hipLaunchKernelGGL(sort_scatter_kernel, dim3(a.tiles * kBinSlices), dim3(kSortThreads), scatter_lds(a.width), s, a);
    }
  }
  if (!single) {
    const int32_t* sorted_keys = P > 0 ? keys_b : indices;  // P == 0: nothing was sorted, every offset is 0
    const unsigned nb = (unsigned)((P + 256) / 256 < 2048 ? (P + 256) / 256 : 2048);
    hipLaunchKernelGGL(segment_offsets_kernel, dim3(nb), dim3(256), 0, s, sorted_keys, offsets, P, (uint32_t)N);
  }
  hipError_t err = hipGetLastError();
  return err == hipSuccess ? OMNI_OK : OMNI_ERR_HIP_BASE + (int)err;
}

// ---- the same schedule for callers that cannot allocate ---------------------------------------
// Code under HIP graph capture, tight serving loops and harnesses that forbid hipMalloc have no
// way to bring a workspace.  For them the sort's workspace is a fixed array in device memory that
// each GPU holds from the moment the library is loaded until the process ends.  In host code the
// array's name is only a handle: its device address is looked up once per device with
// hipGetSymbolAddress and kept; every kernel receives that address as its workspace argument.
namespace omni {

static __device__ __align__(256) unsigned char scratch[OMNI_SCHEDULE_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
static std::atomic<void*> g_scratch_addr[kMaxDevices];

// Device address of `scratch` on the current device (resolved on the first call per device).
static int scratch_address(void** out) {
  int dev = -1;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return OMNI_ERR_HIP_BASE + (int)e;
  if (dev < 0 || dev >= kMaxDevices) return OMNI_ERR_UNSUPPORTED;
  void* p = g_scratch_addr[dev].load(std::memory_order_acquire);
  if (!p) {
    if (hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)); e != hipSuccess) return OMNI_ERR_HIP_BASE + (int)e;
    if (!p) return OMNI_ERR_SCRATCH;
    g_scratch_addr[dev].store(p, std::memory_order_release);   // concurrent first calls store the same address
  }
  *out = p;
  return OMNI_OK;
}

int schedule_scratch_prepare() {
  void* p = nullptr;
  return scratch_address(&p);
}

}  // namespace omni

extern "C" OMNI_API int32_t omni_schedule_noalloc(const int32_t* indices, int32_t* offsets, int32_t* sorted_pair_ids,
                                                  int32_t* sorted_token_ids, int64_t num_tokens, int32_t num_experts_per_token,
                                                  int64_t num_experts, void* stream) {
  using namespace omni;
  const int64_t N = num_experts, P = num_tokens * (int64_t)num_experts_per_token;
  if (num_tokens < 0 || num_experts_per_token < 0 || N <= 0 || P > INT32_MAX / 2 || N > INT32_MAX / 2) return OMNI_ERR_SHAPE;
  SortPlan pl;
  if (!make_plan(P, N, &pl)) return OMNI_ERR_UNSUPPORTED;
  const size_t need = omni_schedule_workspace_bytes(num_tokens, num_experts_per_token, num_experts);
  if (need == 0 || need > (size_t)OMNI_SCHEDULE_NOALLOC_SCRATCH_BYTES) return OMNI_ERR_SCRATCH;
  void* ws = nullptr;
  if (int e = scratch_address(&ws)) return e;
  // every kernel of the sort writes the part of the workspace it later reads (counts, tile sums,
  // keys, pair ids), so nothing of an earlier call's contents has to be cleared
  return omni_schedule(indices, offsets, sorted_pair_ids, sorted_token_ids, num_tokens, num_experts_per_token, num_experts, ws, stream);
}
