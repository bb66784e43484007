// The general tile GEMM for gfx950: 16-bit products of any size and any operand layout, several to a launch, K split where the output
// has fewer tiles than the chip has CUs.  It serves
//   * the training path's gradients, whose operands are not both K-contiguous (the reference leaves them to autograd of torch.matmul,
//     interface.py:23-29):  d(h) = dy Wd,  d(x) = dgate Wg + dup Wu + dz [Wx;Wy],  d(W) = dgate^T x, dup^T x, dy^T h, dz^T x;
//   * the forward projections of a few hundred to a few thousand tokens.
// Nothing is transposed in memory: an operand whose rows run along M or N goes to LDS as it lies there, and its matrix fragments
// come out of LDS through the transposing read ds_read_b64_tr_b16 (within 16 lanes, lane i names 8 bytes, 4 elements, of row i / 4 of
// a 4 x 16 block and receives column i of it; two of them give a lane the 8 consecutive K values of v_mfma_f32_16x16x32).
//
// What bounds it.  The 256 x 256 tile at K = 2048 and more: the matrix pipelines under the board's power limit (gate/up at 32768 x 2 8192 x 2048: busy 74 % of
// the cycles at 1.88 GHz, 1.32 PFLOP/s in the layer, 1.45 in a counter run, which leaves gaps between launches); at K = 1024 the 16 ring steps between its fill and its epilogue
// (4096 x 2 4096 x 1024: 57 % at 1.92 GHz, 1.14 PFLOP/s with a block to a tile, 58 % and 1.16 streamed; d(h) with the SwiGLU backward as epilogue 57 us, 0.60
// PFLOP/s, half of them its 134 MB).  The
// 128 x 128 tile: the path from L2 into LDS, which carries 64 bytes per cycle and CU -- what that tile asks for at full matrix rate --
// and, with one block to a CU, the chain of reads and waits between two barriers.  So a block's waves keep 64 x 64 of the tile each (LDS
// serves 256 bytes a cycle, and smaller wave tiles read more per product) and, alone on its CU, a block has three ring stages in flight (TileRing); the 64 x 64 tile
// has two groups of waves that take every other K tile and add up at the end: one barrier for two K tiles and a second wave to issue while the first waits
// (and the 128 x 128 tile for the gradients' long sums: Shape<9>).
// Splitting K over the grid costs a pass over fp32 partial sums (summed in split order: results do not depend on timing).
#pragma once
#include "common.h"
#include "gemm_tiles.h"
#include "omni_moe_hip.h"
#include "select.h"

#include <type_traits>
#include <utility>

namespace omni {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));

template <int DT>
__device__ __forceinline__ f32x4_t mfma16x16x32(const u32x4_t a, const u32x4_t b, f32x4_t c) {
  if constexpr (DT == kBF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}
template <int DT> __device__ __forceinline__ float lo16(const uint32_t w) {
  if constexpr (DT == kBF16) return bf16_lo(w); else return f16_bits_to_f32((uint16_t)(w & 0xffffu));
}
template <int DT> __device__ __forceinline__ float hi16(const uint32_t w) {
  if constexpr (DT == kBF16) return bf16_hi(w); else return f16_bits_to_f32((uint16_t)(w >> 16));
}
template <int DT> __device__ __forceinline__ uint32_t pack16x2(float lo, float hi) {
  if constexpr (DT == kBF16) return pack_bf16(lo, hi); else return pack_f16(lo, hi);
}

// Where the memory instructions of one K step go among its TM x TN matrix instructions.  A wave issues in order, so a burst of them
// holds up the matrix instructions behind it: fragment reads are dealt out, `cap` behind each one, and the NL loads stand at even
// distances -- the path into LDS takes a load instruction about every 20 cycles a CU, and waves that all issue theirs at once wait for it.
// Fragment reads are for the FOLLOWING step: weight-side fragments (two sets) may be read at once, the fragment of row tile i only
// when row i has issued (one set).
// Codes: 0 none, 1 + n: A read n (row tile n / RA, part n % RA), 65 + n: B read n, 129 + n: load n.
template <int TM, int TN, int RA, int RB, int NL, bool kSync>
struct StepPlan {
  static constexpr int kSlots = TM * TN, kStart = kSync ? TN - 1 : 0, kOps = TM * RA + TN * RB + NL;
  static constexpr int kSpan = kSync ? (kSlots - kStart + 1) / 2 : kSlots;         // those behind the barrier are waited for soonest: they come in its first half
  static constexpr int kCap = (TM * RA + TN * RB + kSlots - kStart - 1) / (kSlots - kStart), kMost = kCap + 2 * RA + NL;
  int op[kSlots][kMost] = {};
  constexpr StepPlan() {
    int na = 0, nb = 0, nl = 0;
    for (int s = kStart; s < kSlots; ++s) {
      const int rows = (s + 1) / TN;                       // row tiles that have issued
      const int cap = s == kSlots - 1 ? kCap + 2 * RA : kCap;
      int u = 0;
      for (; u < cap;) {
        if (nb < TN * RB && nb <= na) op[s][u++] = 65 + nb++;
        else if (na < rows * RA) op[s][u++] = 1 + na++;
        else if (nb < TN * RB) op[s][u++] = 65 + nb++;
        else break;
      }
      while (nl < NL && nl < NL * (s + 1 - kStart) / kSpan) op[s][u++] = 129 + nl++;
    }
  }
  constexpr bool complete() const {
    int n = 0;
    for (int s = 0; s < kSlots; ++s)
      for (int u = 0; u < kMost; ++u) n += op[s][u] != 0;
    return n == kOps;
  }
};

// f(op), with the number as a type: what depends on it is decided at compile time
template <class Plan, int S, class F, int... U>
__device__ __forceinline__ void each_op_of(F&& f, std::integer_sequence<int, U...>) {
  constexpr Plan plan{};
  (f(std::integral_constant<int, plan.op[S][U]>{}), ...);
}
template <class Plan, int S, class F>
__device__ __forceinline__ void each_op(F&& f) { each_op_of<Plan, S>(f, std::make_integer_sequence<int, Plan::kMost>{}); }

__device__ __forceinline__ u32x2_t lds_read_transposed(uint32_t at) {
  return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(uintptr_t)at));
}
// The value, as one that the compiler knows nothing about: what is derived from it is computed where it is needed and not kept in registers
// around the K loop (which must leave room on a SIMD for waves of the kernels that run beside it)
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}
__device__ __forceinline__ u32x4_t row_quads(const uint32_t x0, const uint32_t x1, const uint32_t x2, const uint32_t x3, const int from) {
  return u32x4_t{(uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)x0), (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)x1),
                 (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)x2), (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)x3)};
}
// d(h) word (two values) with its gate and up words -> d(gate), d(up) (omni_mlp.py:232-236)
template <int DT>
__device__ __forceinline__ void swiglu_bwd_word(const uint32_t o, const uint32_t gq, const uint32_t uq, uint32_t& dg, uint32_t& du) {
  float g2[2], u2[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float d = e ? hi16<DT>(o) : lo16<DT>(o), gt = e ? hi16<DT>(gq) : lo16<DT>(gq), upv = e ? hi16<DT>(uq) : lo16<DT>(uq);
    const float sig = sigmoid_f32(gt), silu = gt * sig;
    g2[e] = d * (silu * (1.0f - sig) + sig) * upv;
    u2[e] = d * silu;
  }
  dg = pack16x2<DT>(g2[0], g2[1]);
  du = pack16x2<DT>(u2[0], u2[1]);
}

// Rows of A that a stage holds: as many as the waves' loads bring in (all of them load alike), and a power of two where A's rows run along M
// (the pieces of such a row change places by XOR).
template <int LAY>
constexpr int staged_rows(int rows, int waves) {
  if (LAY != kTN) return (rows + 8 * waves - 1) / (8 * waves) * (8 * waves);
  int up = 1;
  while (up < rows) up *= 2;
  return up;
}

// Stages of the two operands in LDS: NS, and one more for one of them.  That one is requested in step 0 of a K tile, half a tile before the barrier that frees the
// other's: requests are spread over the whole tile, and of two stages the second one's loads have between a half and a whole tile to arrive.  It is the right operand,
// in a forward pass the weights, which come from further away, or the left one where a tile has more rows of it, or where the right one's does not fit.
// Kernels in traces of whole calls, from equal rings of two stages (with half of a step's requests just before the wait for them) to this one, mean of 45 launches each:
// down of 32768 x 2048 x 8192 844 -> 791 us, gate/up there 1668 -> 1662; the five weight gradients of a 4096-token step 102 -> 94, its SwiGLU backward 59.4 -> 57.4, its d(x) 81 -> 75.
// NS is no more than hides memory, for a block requests NS ring steps before its first matrix instruction, at some 20 cycles a load instruction and CU: a stage
// costs every block 0.1 to 0.3 us.  Equal rings of NS + 1 / NS + 1 and one more for the left operand / as it is, us, weights in the caches, and from memory:
//   64 x 64     65 x 1024 x 512   4.62 / 4.82 / 4.55   4.80 / 4.92 / 4.79     256 x 2048 x 4096   12.6 / 11.5 / 11.3   20.0 / 20.6 / 19.6
//   96 x 128    512 x 1024 x 512  6.16 / 6.20 / 6.00   6.11 / 6.33 / 6.02     3000 x 1024 x 4096  28.8 / 27.4 / 26.9   29.6 / 29.1 / 29.1
//   128 x 128   512 x 1024 x 512  6.91 / 6.93 / 6.77   6.93 / 7.08 / 6.79     4096 x 1024 x 4096  34.5 / 33.3 / 33.0   37.1 / 37.2 / 36.4
//   256 x 128   2048 x 4096 x 512 12.2 / 12.3 / 11.4   13.3 / 13.5 / 13.0     2048 x 4096 x 1024  18.7 / 18.8 / 18.1   19.8 / 19.7 / 19.3
//   64 x 128, gate and up   65 x 2 2048 x 512  5.84 / 6.08 / 5.60   7.30 / 7.43 / 7.25     128 x 2 4096 x 1024  7.51 / 7.63 / 6.98   11.2 / 11.3 / 10.9
// (192 x 128 keeps three: with two 3000 x 2048 x 3072 from memory takes 36.8 -> 40.4.)
constexpr int kCuLds = 160 * 1024;
template <int LM, int BN, int KG, int NS>
struct TileRing {
  static constexpr bool kLeadA = LM > 128 ? KG * 128 * (LM * (NS + 1) + BN * NS) <= kCuLds : KG * 128 * (LM * NS + BN * (NS + 1)) > kCuLds;
  static constexpr int kAStages = NS + (kLeadA ? 1 : 0), kBStages = NS + (kLeadA ? 0 : 1);
  static constexpr int kAStage = KG * LM * 128, kBStage = KG * BN * 128, kBFirst = kAStages * kAStage, kBytes = kBFirst + kBStages * kBStage;
  static_assert(kBytes <= kCuLds, "a block's ring fits its CU");
};

// A block is KG groups of WM x WN waves; a wave owns TM x TN matrix tiles of 16 x 16.  The ring advances 64 * KG of K a step through NS stages (TileRing);
// group g multiplies the g-th 64 of each.  kTail: some segment's K is not a multiple of the ring step, and an operand's rows run along K.
//
// kStream (one product, one segment, unsplit): the grid may be smaller than the number of output tiles; a block walks its share, and the ring
// steps of consecutive output tiles form ONE stream through the stages: the next tile's first loads fly while the current one finishes, so
// only a block's first tile waits for memory before its first matrix instruction.  A tile's first wait is for the last one's stores too, which have had half a K tile:
// to let them fly took a branch into the loop, which cost every K tile what this costs one (MI355X, kernels alone, 20 ms of calls: gate/up of 32768 x 2 8192 x 2048
// 1559 -> 1544 us, of 4474 x 2 4096 x 1024 74.7 -> 73.5; down of 32768 x 2048 x 8192 777 -> 756, of 20000 x 1024 x 2048 92.8 -> 89.6).
// (block, blocks): the place in the launch, or in its own part of one that it shares
template <int DT, int LAY, int WM, int WN, int KG, int TM, int TN, int NS, int EPI, bool kTail, bool kStream, class Group>
__device__ __forceinline__ void tiles_block(const Group& g, const int block, const int blocks) {
  constexpr bool AC = LAY == kTN, BC = LAY != kNT;             // the operand's K index is its row
  constexpr int NW = WM * WN * KG, BM = WM * TM * 16, BN = WN * TN * 16, BNO = EPI == kTileSwiglu ? BN / 2 : BN;
  constexpr int LM = staged_rows<LAY>(BM, NW);                 // A's rows in a stage, those behind the tile's unread
  constexpr int kABytes = LM * 128, kBBytes = BN * 128;        // of a group's 64 of K
  using Ring = TileRing<LM, BN, KG, NS>;
  constexpr int PA = LM / 8 / NW, PB = BN / 8 / NW, LPT = KG * (PA + PB);     // 1 KiB load instructions per wave and ring step
  constexpr int kLead = KG * (Ring::kLeadA ? PA : PB);         // ... those of the operand with a stage more
  static_assert(LM % (8 * NW) == 0 && BN % (8 * NW) == 0, "the waves share the loads evenly");
  static_assert(TN % (EPI == kTileSwiglu ? 4 : 2) == 0 && TM % KG == 0, "the epilogue takes column tiles in pairs");
  constexpr int RA = AC ? 2 : 1, RB = BC ? 2 : 1;              // LDS reads per fragment
  using LdsPtr = __attribute__((address_space(3))) void*;
  extern __shared__ __align__(16) uint8_t lds[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / (WM * WN), wm = wave % WM, wn = (wave / WM) % WN;

  // ---- which tile of which product.  Blocks go round-robin over the 8 XCDs: each XCD takes one run of a product's tile order, which
  // walks bands of four tile rows column by column, so that the blocks behind one L2 share operand panels.
  int pi = 0;
  if constexpr (std::is_same<Group, TileGroup>::value) {
#pragma unroll
    for (int i = 1; i < kMaxProducts; ++i)
      if (i < g.count && block >= g.p[i].first) pi = i;
  }
  const TileProduct& p = g.p[pi];
  const int M = p.M, N = p.N;
  const int tm = (M + BM - 1) / BM, tn = (N + BNO - 1) / BNO, nt = tm * tn, all = nt * p.splits;
  auto coords = [&](int l, int& m, int& n) -> int {            // returns the split
    const int x = l & 7, j = l >> 3;
    int t = x * (all >> 3) + min(x, all & 7) + j;
    const int split = kStream ? 0 : t / nt;
    t -= split * nt;
    const int band = t / (4 * tn), w = t - band * 4 * tn, rows = min(4, tm - band * 4);
    m = (band * 4 + w % rows) * BM;
    n = (w / rows) * BNO;
    return split;
  };
  int f_tile = block - p.first, fm0, fn0;            // the output tile that is being fetched
  const int split = coords(f_tile, fm0, fn0);

  // ---- fetch cursor: the next ring step to request
  // Load instruction q of a wave fills KiB q * NW + wave of an operand's 64-wide K tile.  Rows along K: 8 rows of 128 bytes, chunk position
  // c of row r holds chunk c ^ (r / 2 % 8).  Rows along M/N: 512, 256 or 128 bytes a row; the 32-byte piece of 16-wide tile t stands at
  // piece t ^ s(r), s(r) = r % 4 + 4 (r / 8 % 2): the eight rows that 32 lanes of a transposing read take then lie in different
  // banks (rows of 128 bytes, two to the 256 bytes of banks: s(r) = r / 2 % 2 + 2 (r / 8 % 2)).
  auto piece_of = [](int row, int width) -> int { return width >= 128 ? (row & 3) | ((row >> 1) & 4) : ((row >> 1) & 1) | ((row >> 2) & 2); };
  // (rows along K: a lane loads chunk lane % 8 ^ (4 wave + lane / 16) % 8 of its rows, whatever the load -- NW is even)
  constexpr int kOff = kTail ? KG : 1;
  uint32_t a_off[kOff], b_off[kOff];                           // lane offsets, the same for every load of a step (past a segment's K they differ by group)
  // Everything a load takes beside its lane offset is a scalar that moves on once per ring step: the operands' addresses and what is left of
  // their matrices behind them (nothing, once every ring step has been requested: the loads then fetch nothing, which is cheaper than
  // a branch around each -- a scalar branch among the matrix instructions costs a lone wave as much as one of them).
  uint64_t f_a = 0, f_b = 0;
  int f_aleft = 0, f_bleft = 0, f_astep = 0, f_bstep = 0, f_amore = 0, f_bmore = 0;      // ..step: for 64 of K; ..more: from one load of a step to the wave's next
  int f_seg = -1, f_left = 0;                                  // K values of the segment from the cursor on, when its run of steps began
  int f_run = 0, f_until = 0;                                  // ring steps of that run, and what is left of it: the cursor only moves on by f_astep and f_bstep
  int f_half = 0;                                              // kTileTwo: rows of the fetched tile, counted from the wave's first, that are the first matrix's
  constexpr uint32_t kOutside = 0x80000000u;
  auto scalar = [](int v) __attribute__((always_inline)) { return __builtin_amdgcn_readfirstlane(v); };
  auto scalar64 = [](uint64_t v) __attribute__((always_inline)) {
    // (readfirstlane returns a signed value)
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32));
    return (uint64_t)lo | ((uint64_t)hi << 32);
  };
  int f_steps = 0;                                             // ring steps of the fetched tile, when the run began; none: everything has been requested
  // up to the end of the segment or the tile, or to a step of less than 64 * KG
  auto begin_run = [&]() __attribute__((always_inline)) {
    const int n = min(f_steps, (f_left + 64 * KG - 1) / (64 * KG));
    f_run = f_until = scalar(kTail && n > 1 && n * 64 * KG > f_left ? n - 1 : n);
  };
  // rows along K: chunks past the segment's K read as zero (the other operands end with their matrix)
  auto mask_tail = [&]() __attribute__((always_inline)) {
    if constexpr (kTail && (!AC || !BC)) {
      if (f_left < 64 * KG) {
#pragma unroll
        for (int s = 0; s < KG; ++s) {
          const int lane = opaque(tid & 63), row_chunk = (lane & 7) ^ ((4 * wave + (lane >> 4)) & 7);
          const bool outside = row_chunk * 8 + 64 * s >= f_left;
          if (!AC) a_off[s % kOff] = outside ? kOutside : a_off[s % kOff];
          if (!BC) b_off[s % kOff] = outside ? kOutside : b_off[s % kOff];
        }
      }
    }
  };
  auto enter_segment = [&](int skip) {                         // at its ring step `skip`
    const int lane = opaque(tid & 63), row_chunk = (lane & 7) ^ ((4 * wave + (lane >> 4)) & 7);
    const TileSegment& sg = p.seg[f_seg];
    f_left = scalar(sg.K - 64 * KG * skip);
    const int lda = (int)sg.lda, ldb = (int)sg.ldb;
    f_astep = scalar(AC ? 64 * lda : 128);
    f_bstep = scalar(BC ? 64 * ldb : 128);
    const int64_t a_in = (int64_t)KG * skip * f_astep, b_in = (int64_t)KG * skip * f_bstep;
    f_a = scalar64((uint64_t)sg.a + (AC ? (int64_t)fm0 * 2 : (int64_t)fm0 * lda) + a_in);
    f_aleft = scalar((int)((AC ? (int64_t)sg.K * lda - (int64_t)fm0 * 2 : (int64_t)min(M - fm0, BM) * lda) - (AC || M - fm0 <= BM ? sg.a_skip : 0) - a_in));
    f_b = scalar64((uint64_t)sg.b + (BC ? (int64_t)fn0 * 2 : (int64_t)fn0 * ldb) + b_in);
    f_bleft = scalar((int)((BC ? (int64_t)sg.K * ldb - (int64_t)fn0 * 2 : (int64_t)min(N - fn0, BN) * ldb) - b_in));
    if constexpr (EPI == kTileTwo) f_half = scalar(N / 2 - fn0 - wave * 8);
    uint32_t a0, b0;
    if constexpr (AC) {
      constexpr int W = LM / 8;
      const int r = wave * (64 / W) + lane / W, chunk = (lane % W) ^ (piece_of(r, LM) << 1);
      a0 = BM < LM && chunk >= BM / 8 ? kOutside : (uint32_t)(r * lda) + (uint32_t)chunk * 16;
      f_amore = scalar(NW * (64 / W) * lda);
    } else {
      a0 = (uint32_t)((wave * 8 + (lane >> 3)) * lda) + (uint32_t)row_chunk * 16;
      f_amore = scalar(NW * 8 * lda);
    }
    if constexpr (BC) {
      constexpr int W = BN / 8;
      const int r = wave * (64 / W) + lane / W;
      b0 = (uint32_t)(r * ldb) + (uint32_t)((lane % W) ^ (piece_of(r, BN) << 1)) * 16;
      f_bmore = scalar(NW * (64 / W) * ldb);
    } else {
      int r = wave * 8 + (lane >> 3);
      if constexpr (EPI == kTileSwiglu) r = r % (TN * 8);      // a wave's first TN / 2 column tiles are gate rows, the rest the matching up rows
      b0 = (uint32_t)(r * ldb) + (uint32_t)row_chunk * 16;
      f_bmore = scalar((EPI == kTileSwiglu ? TN * 8 : NW * 8) * ldb);
    }
#pragma unroll
    for (int s = 0; s < kOff; ++s) { a_off[s] = a0; b_off[s] = b0; }
    mask_tail();
    begin_run();
  };
  int tiles = p.steps;                                         // ring steps of one output tile in this block
  {
    int skip = split * p.steps, total = 0;
#pragma unroll
    for (int i = 0; i < kMaxSegments; ++i) {
      const int n = i < p.segments ? (p.seg[i].K + 64 * KG - 1) / (64 * KG) : 0;
      if (f_seg < 0 && skip < n) f_seg = i;
      if (f_seg < 0) skip -= n;
      total += n;
    }
    tiles = scalar(min(tiles, total - split * p.steps));
    f_seg = scalar(f_seg);
    f_steps = tiles;
    enter_segment(skip);
  }
  const uint32_t lds_base = (uint32_t)(uintptr_t)(LdsPtr)lds;
  const uint32_t lds_wave = lds_base + (uint32_t)wave * 1024;
  uint32_t f_ato = lds_wave, f_bto = lds_wave + Ring::kBFirst; // the cursor's stages
  // from B's address to the other matrix's: the up weights, or (Two) the upper half of the columns' as if its rows followed on the first's
  uint64_t to_second = 0;
  if constexpr (EPI == kTileSwiglu) to_second = scalar64((uint64_t)p.b_up - (uint64_t)p.seg[0].b);
  if constexpr (EPI == kTileTwo) to_second = scalar64((uint64_t)p.b_up - (uint64_t)p.seg[0].b - (uint64_t)(N / 2) * (uint64_t)p.seg[0].ldb);
  // load q of an operand's part of the cursor's ring step
  auto issue_a = [&](auto q_tag) __attribute__((always_inline)) {
    constexpr int q = decltype(q_tag)::value, s = q / PA, o = q % PA;
    load_to_lds<s * kABytes + o * NW * 1024>(f_a, f_aleft, f_ato, a_off[s % kOff], s * f_astep + o * f_amore);
  };
  auto issue_b = [&](auto q_tag) __attribute__((always_inline)) {
    constexpr int q = decltype(q_tag)::value, s = q / PB, b = q % PB, row = b * NW * 8, nth = EPI == kTileSwiglu ? row / (TN * 16) : b;
    uint64_t base = f_b;
    if constexpr (EPI == kTileSwiglu) base += ((row + wave * 8) / (TN * 8)) & 1 ? to_second : 0;
    if constexpr (EPI == kTileTwo) base += row >= f_half ? to_second : 0;     // (the eight rows of a load are of one matrix)
    load_to_lds<s * kBBytes + b * NW * 1024>(base, f_bleft, f_bto, b_off[s % kOff], s * f_bstep + nth * f_bmore);
  };
  auto issue_lead = [&](auto q_tag) __attribute__((always_inline)) { if constexpr (Ring::kLeadA) issue_a(q_tag); else issue_b(q_tag); };
  auto issue_other = [&](auto q_tag) __attribute__((always_inline)) { if constexpr (Ring::kLeadA) issue_b(q_tag); else issue_a(q_tag); };
  // to the next ring step of a run
  auto move_a = [&]() __attribute__((always_inline)) {
    f_a += KG * (uint32_t)f_astep;
    f_aleft -= KG * f_astep;
    f_ato = f_ato == lds_wave + (Ring::kAStages - 1) * Ring::kAStage ? lds_wave : f_ato + Ring::kAStage;
  };
  auto move_b = [&]() __attribute__((always_inline)) {
    f_b += KG * (uint32_t)f_bstep;
    f_bleft -= KG * f_bstep;
    f_bto = f_bto == lds_wave + Ring::kBFirst + (Ring::kBStages - 1) * Ring::kBStage ? lds_wave + Ring::kBFirst : f_bto + Ring::kBStage;
  };
  auto move_lead = [&]() __attribute__((always_inline)) { if constexpr (Ring::kLeadA) move_a(); else move_b(); };
  auto move_other = [&]() __attribute__((always_inline)) { if constexpr (Ring::kLeadA) move_b(); else move_a(); };
  // where a run has ended
  auto next_run = [&]() __attribute__((always_inline)) {
    f_left -= 64 * KG * f_run;
    f_steps -= f_run;
    if (f_steps > 0) {
      if (f_left <= 0) {
        f_seg = scalar(f_seg + 1);
        enter_segment(0);
      } else {
        mask_tail();
        begin_run();
      }
    } else if (kStream && f_tile + blocks < all) {
      f_tile = scalar(f_tile + blocks);
      f_steps = tiles;
      coords(f_tile, fm0, fn0);
      enter_segment(0);
    } else {                                                   // everything has been requested
      f_aleft = f_bleft = f_astep = f_bstep = 0;
      f_until = INT32_MAX;
    }
  };

  // ---- fragment reads.  Lane (r16 = lane % 16, g4 = lane / 16) takes the K values 32 ks + 8 g4 .. + 7 of row r16 of a 16-row tile.
  const int r16 = lane & 15, g4 = lane >> 4;
  constexpr int kRowA = AC ? LM * 2 : 128, kRowB = BC ? BN * 2 : 128;
  uint32_t a_addr[AC ? TM : 2], b_addr[BC ? TN : 2];
  const uint32_t tr_row = (uint32_t)(8 * g4 + (r16 >> 2)), tr_in = (uint32_t)(r16 & 3) * 8;       // (piece_of() of the row is the same in every K step and part)
  const uint32_t my_a = lds_base + (uint32_t)(kg * kABytes), my_b = lds_base + (uint32_t)(Ring::kBFirst + kg * kBBytes);
  if constexpr (AC) {
#pragma unroll
    for (int i = 0; i < TM; ++i) a_addr[i] = my_a + tr_row * kRowA + (uint32_t)((wm * TM + i) ^ piece_of((int)tr_row, LM)) * 32 + tr_in;
  } else {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) a_addr[ks] = my_a + (uint32_t)(wm * TM * 16 + r16) * 128 + (uint32_t)((4 * ks + g4) ^ (r16 >> 1)) * 16;
  }
  if constexpr (BC) {
#pragma unroll
    for (int j = 0; j < TN; ++j) b_addr[j] = my_b + tr_row * kRowB + (uint32_t)((wn * TN + j) ^ piece_of((int)tr_row, BN)) * 32 + tr_in;
  } else {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) b_addr[ks] = my_b + (uint32_t)(wn * TN * 16 + r16) * 128 + (uint32_t)((4 * ks + g4) ^ (r16 >> 1)) * 16;
  }
  using Frag = const __attribute__((address_space(3))) u32x4_t*;
  u32x4_t af[TM], bf[2][TN];
  // part `n` of the fragments of K step ks in the stage that the addresses stand at
  auto read_a = [&](int ks, int n) __attribute__((always_inline)) {
    if constexpr (AC) {
      const int i = n / 2, h = n % 2;
      const u32x2_t w = lds_read_transposed(a_addr[i] + (32 * ks + 4 * h) * kRowA);
      af[i][2 * h] = w[0]; af[i][2 * h + 1] = w[1];
    } else {
      af[n] = *(Frag)(uintptr_t)(a_addr[ks] + n * 16 * 128);
    }
  };
  auto read_b = [&](int ks, int n) __attribute__((always_inline)) {
    if constexpr (BC) {
      const int j = n / 2, h = n % 2;
      const u32x2_t w = lds_read_transposed(b_addr[j] + (32 * ks + 4 * h) * kRowB);
      bf[ks][j][2 * h] = w[0]; bf[ks][j][2 * h + 1] = w[1];
    } else {
      bf[ks][n] = *(Frag)(uintptr_t)(b_addr[ks] + n * 16 * 128);
    }
  };

  f32x4_t acc[TM][TN];

  // ---- K loop.  Step 0 of a K tile reads the fragments of its step 1 and requests one operand of the ring step NS ahead; then, after the first matrix row of
  // step 1, every wave waits for its own reads and loads and meets the block: the stage is free, the next one is there; step 1 reads the next stage's first
  // fragments and requests the other operand.  Behind the last ring step the reads fetch what nobody uses.
  // The cursor moves between matrix instructions, and where a run of its steps ends, between two K tiles, a branch out of the loop sees to what comes next.
  using Plan0 = StepPlan<TM, TN, RA, RB, kLead, false>;
  using Plan1 = StepPlan<TM, TN, RA, RB, LPT - kLead, true>;
  static_assert(Plan0{}.complete() && Plan1{}.complete(), "a step's memory instructions do not fit");
  auto load_lead = [&](auto... q) __attribute__((always_inline)) { (issue_lead(q), ...); };
  auto load_other = [&](auto... q) __attribute__((always_inline)) { (issue_other(q), ...); };
#pragma unroll
  for (int t = 0; t < NS; ++t) {
    with_sequence(load_lead, std::make_integer_sequence<int, kLead>{});
    with_sequence(load_other, std::make_integer_sequence<int, LPT - kLead>{});
    move_lead();
    move_other();
    if (--f_until == 0) next_run();
  }
  vmcnt<(NS - 1) * LPT>();
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int n = 0; n < TM * RA; ++n) read_a(0, n);
#pragma unroll
  for (int n = 0; n < TN * RB; ++n) read_b(0, n);
  int a_stage = 0, b_stage = 0;                                // those being multiplied
  // Column tiles back and forth, so that one operand of a matrix instruction is always the one before's: under the power limit less that changes is time
  // (gate/up of 32768 x 2 8192 x 2048 1591 -> 1583 us, down of 32768 x 2048 x 8192 787 -> 784, gate/up of 4096 x 2 4096 x 1024 55.6 -> 55.1; five runs of each in turn)
  auto column = [](int s) constexpr { return s / TN % 2 ? TN - 1 - s % TN : s % TN; };
  auto slot0 = [&](auto s_tag) __attribute__((always_inline)) {
    constexpr int s = decltype(s_tag)::value;
    constexpr int i = s / TN, j = column(s);
    acc[i][j] = mfma16x16x32<DT>(bf[0][j], af[i], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
    each_op<Plan0, s>([&](auto op_tag) __attribute__((always_inline)) {
      constexpr int op = decltype(op_tag)::value;
      if constexpr (op >= 129) issue_lead(std::integral_constant<int, op - 129>{});
      else if constexpr (op >= 65) read_b(1, op - 65);
      else if constexpr (op >= 1) read_a(1, op - 1);
    });
    __builtin_amdgcn_sched_barrier(0);
  };
  auto slot1 = [&](auto s_tag) __attribute__((always_inline)) {
    constexpr int s = decltype(s_tag)::value;
    constexpr int i = s / TN, j = column(s);
    acc[i][j] = mfma16x16x32<DT>(bf[1][j], af[i], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (s == TN - 1) {
      lds_reads_done();
      constexpr int kYounger = (NS - 2) * LPT + kLead;
      vmcnt<kYounger>();
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    }
    each_op<Plan1, s>([&](auto op_tag) __attribute__((always_inline)) {
      constexpr int op = decltype(op_tag)::value;
      if constexpr (op >= 129) issue_other(std::integral_constant<int, op - 129>{});
      else if constexpr (op >= 65) read_b(0, op - 65);
      else if constexpr (op >= 1) read_a(0, op - 1);
    });
    if constexpr (s == (TN - 1 + TM * TN - 1) / 2) move_lead();
    if constexpr (s == TM * TN - 1) move_other();
    __builtin_amdgcn_sched_barrier(0);
  };
  auto all0 = [&](auto... s) __attribute__((always_inline)) { (slot0(s), ...); };
  auto all1 = [&](auto... s) __attribute__((always_inline)) { (slot1(s), ...); };
#pragma clang loop unroll(disable)
  for (int tile = block - p.first; tile < all; tile += blocks) {
  int m0, n0;
  coords(tile, m0, n0);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[i][j][q] = 0.f;
  for (int left = tiles; left > 0;) {
    const int run = min(left, f_until);
    // Nothing of the last tile's epilogue and of next_run() is on its way to a register in here, or the compiler makes every K tile's second matrix instruction
    // wait for all reads before it
    if constexpr (kStream) __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
#pragma clang loop unroll(disable)
    for (int i = run; i > 0; --i) {
      with_sequence(all0, std::make_integer_sequence<int, TM * TN>{});
      a_stage = a_stage + 1 == Ring::kAStages ? 0 : a_stage + 1;
      b_stage = b_stage + 1 == Ring::kBStages ? 0 : b_stage + 1;
      const uint32_t a_move = a_stage == 0 ? (uint32_t)(-(Ring::kAStages - 1) * Ring::kAStage) : (uint32_t)Ring::kAStage;
      const uint32_t b_move = b_stage == 0 ? (uint32_t)(-(Ring::kBStages - 1) * Ring::kBStage) : (uint32_t)Ring::kBStage;
#pragma unroll
      for (int i = 0; i < (AC ? TM : 2); ++i) a_addr[i] += a_move;
#pragma unroll
      for (int j = 0; j < (BC ? TN : 2); ++j) b_addr[j] += b_move;
      with_sequence(all1, std::make_integer_sequence<int, TM * TN>{});
    }
    left -= run;
    f_until -= run;
    if (f_until == 0) next_run();
  }
  if constexpr (!kStream) vmcnt<0>();                          // no load may arrive in LDS that the block has given back

  // ---- two groups: each finishes half of the row tiles and hands the other half over through LDS
  if constexpr (KG == 2) {
    constexpr int H = TM / 2;
    lds_reads_done();                                          // the reads behind the last ring step
    __syncthreads();
    f32x4_t* xch = (f32x4_t*)lds + (int64_t)(wave % (WM * WN)) * (2 * H * TN * 64);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        if (i / H != kg) xch[((i / H) * H * TN + (i % H) * TN + j) * 64 + lane] = acc[i][j];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        if (i / H == kg) {
          const f32x4_t o = xch[((i / H) * H * TN + (i % H) * TN + j) * 64 + lane];
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[i][j][q] += o[q];
        }
  }

  // ---- epilogue.  acc[i][j]: row 16 i + r16, columns 16 j + 4 g4 .. + 3.  One bpermute per word puts each row's 64 bytes into four
  // consecutive lanes (the store path wants that: see the streaming GEMM); 16-bit results first trade words between lanes l and
  // l ^ 16, so that a lane holds 8 columns.
  const int lane_e = opaque(lane), tr = lane_e >> 2, tg = lane_e & 3, from = (tr + 16 * tg) * 4;
  const int nb = n0 + wn * (BNO / WN);
  if (p.part) {                                                // partial sums: [split][M][columns] fp32, columns = N (SwiGLU: gate, then up)
    const int64_t cols = EPI == kTileSwiglu ? 2 * (int64_t)N : N;
    float* out = p.part + (int64_t)split * M * cols;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (KG == 2 && i / (TM / 2) != kg) continue;
      const int m = m0 + (wm * TM + i) * 16 + tr;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const u32x4_t w = row_quads(__float_as_uint(acc[i][j][0]), __float_as_uint(acc[i][j][1]), __float_as_uint(acc[i][j][2]), __float_as_uint(acc[i][j][3]), from);
        const bool second = EPI == kTileSwiglu && j >= TN / 2;
        const int n = nb + (second ? j - TN / 2 : j) * 16 + tg * 4;
        if (m < M && n < N) *(u32x4_t*)(out + (int64_t)m * cols + (second ? N : 0) + n) = w;
      }
    }
    return;
  }
  // What the epilogue reads (the residual, or gate and up) is requested one row tile ahead, from inside the matrix whatever the lane: a wait for each
  // piece in turn made the SwiGLU backward of 4096 x 4096 x 1024 take 28 us on top of 32.
  constexpr int kJ = (EPI == kTileSwiglu ? TN / 2 : TN) / 2, kSide = EPI == kTileSwigluBwd ? 2 : EPI == kTileResidual ? 1 : 0;
  u32x4_t side[2][kJ][kSide ? kSide : 1];
  auto place = [&](int i, int jp, int& m, int& n) { m = m0 + (wm * TM + i) * 16 + tr; n = nb + (2 * jp + (tg & 1)) * 16 + (tg & 2) * 4; };
  auto request = [&](int i) {
    if constexpr (kSide > 0) {
#pragma unroll
      for (int jp = 0; jp < kJ; ++jp) {
        int m, n;
        place(i, jp, m, n);
        const int64_t at = (int64_t)min(m, M - 1) * p.ldc + (int64_t)min(n, N - 8) * 2;
        side[i & 1][jp][0] = *(const u32x4_t*)((EPI == kTileResidual ? p.res : p.gate) + at);
        if constexpr (kSide == 2) side[i & 1][jp][kSide - 1] = *(const u32x4_t*)(p.up + at);
      }
    }
  };
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (KG == 2 && i / (TM / 2) != kg) continue;
    if (i == 0 || (KG == 2 && i == TM / 2)) request(i);
    if (i + 1 < TM && (KG == 1 || (i + 1) / (TM / 2) == i / (TM / 2))) request(i + 1);
#pragma unroll
    for (int jp = 0; jp < kJ; ++jp) {
      const int j = 2 * jp;
      uint32_t w[2][2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          v[q] = acc[i][j + t][q];
          // gate and up are materialised in the storage dtype, silu(gate) * up is formed in fp32 and rounded once (omni_mlp.py:53-61)
          if constexpr (EPI == kTileSwiglu) v[q] = silu_fast(Elem<DT>::round(v[q])) * Elem<DT>::round(acc[i][j + t + TN / 2][q]);
        }
        w[t][0] = pack16x2<DT>(v[0], v[1]);
        w[t][1] = pack16x2<DT>(v[2], v[3]);
      }
      const auto s0 = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
      const auto s1 = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
      u32x4_t out = row_quads(s0[0], s1[0], s0[1], s1[1], from);
      int m, n;
      place(i, jp, m, n);
      const int64_t at = (int64_t)m * p.ldc + (int64_t)n * 2;
      const bool inside = m < M && n < N;
      if constexpr (EPI == kTileSwigluBwd) {                   // out is d(h) rounded to the storage type
        u32x4_t dg, du;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t oq = out[q], gq = side[i & 1][jp][0][q], uq = side[i & 1][jp][kSide - 1][q];
          uint32_t a, b;
          swiglu_bwd_word<DT>(oq, gq, uq, a, b);
          dg[q] = a; du[q] = b;
        }
        if (inside) {
          *(u32x4_t*)(p.c + at) = dg;
          *(u32x4_t*)(p.c2 + at) = du;
        }
      } else {
        if constexpr (EPI == kTileResidual) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const uint32_t o = out[q], rq = side[i & 1][jp][0][q];
            out[q] = pack16x2<DT>(lo16<DT>(o) + lo16<DT>(rq), hi16<DT>(o) + hi16<DT>(rq));
          }
        }
        if (inside) *(u32x4_t*)(p.c + at) = out;
        if constexpr (EPI == kTileSwiglu) {
          if (p.c2) {                                          // gate and up, rounded, kept for a backward pass
            uint8_t* keep[2] = {p.c2, p.c3};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              uint32_t k[2][2];
#pragma unroll
              for (int t = 0; t < 2; ++t) {
                const f32x4_t a = acc[i][j + t + h * (TN / 2)];
                k[t][0] = pack16x2<DT>(a[0], a[1]);
                k[t][1] = pack16x2<DT>(a[2], a[3]);
              }
              const auto k0 = __builtin_amdgcn_permlane16_swap(k[0][0], k[1][0], false, false);
              const auto k1 = __builtin_amdgcn_permlane16_swap(k[0][1], k[1][1], false, false);
              const u32x4_t o = row_quads(k0[0], k1[0], k0[1], k1[1], from);
              if (inside) *(u32x4_t*)(keep[h] + at) = o;
            }
          }
        }
      }
    }
  }
  if constexpr (!kStream) return;
  }
  vmcnt<0>();
}

template <int DT, int LAY, int WM, int WN, int KG, int TM, int TN, int NS, int EPI, bool kTail, bool kStream, class Group>
__global__ __launch_bounds__(WM* WN* KG * 64, 2) void gemm_tiles_kernel(const Group g) {
  tiles_block<DT, LAY, WM, WN, KG, TM, TN, NS, EPI, kTail, kStream, Group>(g, (int)blockIdx.x, (int)gridDim.x);
}

// The partial sums of a split product, added in split order and finished like the epilogue above: 8 columns per lane.
template <int DT, int EPI>
__global__ __launch_bounds__(256) void tile_reduce_kernel(const TileProduct p) {
  const int per_row = p.N / 8;
  const int64_t chunks = (int64_t)p.M * per_row, cols = EPI == kTileSwiglu ? 2 * (int64_t)p.N : p.N, plane = (int64_t)p.M * cols;
  for (int64_t c = blockIdx.x * 256ll + threadIdx.x; c < chunks; c += gridDim.x * 256ll) {
    const int64_t m = c / per_row;
    const int n = (int)(c - m * per_row) * 8;
    auto sum8 = [&](const float* at, float (&v)[8]) {
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = 0.f;
      for (int s = 0; s < p.splits; ++s, at += plane) {
        const f32x4_t a = *(const f32x4_t*)at, b = *(const f32x4_t*)(at + 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) { v[q] += a[q]; v[4 + q] += b[q]; }
      }
    };
    float v[8];
    sum8(p.part + m * cols + n, v);
    if constexpr (EPI == kTileSwiglu) {
      float u[8];
      sum8(p.part + m * cols + p.N + n, u);
      if (p.c2) {
        u32x4_t kg, ku;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          kg[q] = pack16x2<DT>(v[2 * q], v[2 * q + 1]);
          ku[q] = pack16x2<DT>(u[2 * q], u[2 * q + 1]);
        }
        *(u32x4_t*)(p.c2 + m * p.ldc + (int64_t)n * 2) = kg;
        *(u32x4_t*)(p.c3 + m * p.ldc + (int64_t)n * 2) = ku;
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = silu_fast(Elem<DT>::round(v[q])) * Elem<DT>::round(u[q]);
    }
    u32x4_t out;
#pragma unroll
    for (int q = 0; q < 4; ++q) out[q] = pack16x2<DT>(v[2 * q], v[2 * q + 1]);
    const int64_t at = m * p.ldc + (int64_t)n * 2;
    if constexpr (EPI == kTileSwigluBwd) {
      const u32x4_t gw = *(const u32x4_t*)(p.gate + at), uw = *(const u32x4_t*)(p.up + at);
      u32x4_t dg, du;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t oq = out[q], gq = gw[q], uq = uw[q];
        uint32_t a, b;
        swiglu_bwd_word<DT>(oq, gq, uq, a, b);
        dg[q] = a; du[q] = b;
      }
      *(u32x4_t*)(p.c + at) = dg;
      *(u32x4_t*)(p.c2 + at) = du;
    } else {
      if constexpr (EPI == kTileResidual) {
        const u32x4_t r = *(const u32x4_t*)(p.res + at);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t o = out[q], rq = r[q];
          out[q] = pack16x2<DT>(lo16<DT>(o) + lo16<DT>(rq), hi16<DT>(o) + hi16<DT>(rq));
        }
      }
      *(u32x4_t*)(p.c + at) = out;
    }
  }
}

// ---- host side -------------------------------------------------------------------------------------
// The tile shapes: waves (rows x columns x K groups), matrix tiles per wave, ring stages.
template <int kId, bool kSwiglu = false> struct Shape;
template <bool kSwiglu> struct Shape<0, kSwiglu> { enum { WM = 2, WN = 4, KG = 1, TM = 8, TN = 4, NS = 2 }; };      // 256 x 256, one block to a CU
template <bool kSwiglu> struct Shape<1, kSwiglu> { enum { WM = 4, WN = 2, KG = 1, TM = 4, TN = 4, NS = 2 }; };      // 256 x 128, one block to a CU
template <bool kSwiglu> struct Shape<2, kSwiglu> { enum { WM = 2, WN = 2, KG = 1, TM = 4, TN = 4, NS = 2 }; };      // 128 x 128, two blocks to a CU
template <bool kSwiglu> struct Shape<3, kSwiglu> { enum { WM = 2, WN = 2, KG = 1, TM = 4, TN = 4, NS = 3 }; };      // 128 x 128, one block to a CU
template <> struct Shape<4, false> { enum { WM = 2, WN = 2, KG = 2, TM = 2, TN = 2, NS = 3 }; };                    // 64 x 64, two K groups, one block to a CU
template <> struct Shape<4, true> { enum { WM = 2, WN = 2, KG = 2, TM = 2, TN = 4, NS = 2 }; };                     // (SwiGLU: 64 x 128, so that a wave holds two column tiles of gate)
template <> struct Shape<10, true> { enum { WM = 2, WN = 2, KG = 2, TM = 2, TN = 4, NS = 3 }; };                    // ... the same for K beyond kShortSum
// Longer sums of few rows wait for memory.  With two stages / three, weights from memory: 128 x 2 5120 x 1280 14.3 / 14.6 us, 90 x 2 6144 x 1536 14.9 / 14.9, 100 x 2 4096 x 2048
// 17.3 / 16.9, 100 x 2 8192 x 4096 33.1 / 32.1.
constexpr int kShortSum = 1536;
// Lower tiles, for row counts that leave the last round of the ones above half empty
template <bool kSwiglu> struct Shape<5, kSwiglu> { enum { WM = 2, WN = 4, KG = 1, TM = 7, TN = 4, NS = 2 }; };      // 224 x 256, one block to a CU
template <bool kSwiglu> struct Shape<6, kSwiglu> { enum { WM = 2, WN = 4, KG = 1, TM = 6, TN = 4, NS = 2 }; };      // 192 x 256, one block to a CU
template <bool kSwiglu> struct Shape<7, kSwiglu> { enum { WM = 4, WN = 2, KG = 1, TM = 3, TN = 4, NS = 3 }; };      // 192 x 128, one block to a CU
template <bool kSwiglu> struct Shape<8, kSwiglu> { enum { WM = 2, WN = 2, KG = 1, TM = 3, TN = 4, NS = 3 }; };      // 96 x 128, one block to a CU
// For long sums of the gradients: a second wave to a SIMD multiplies while the first one's loads are issued, for an exchange of sums at the end.  dy W on 256 tiles,
// K = 8192: 66.2 us against 71.8; 4096: 33.6 against 32.5.  (Not for x W^T: beside the down projection's eight waves the experts' passes find no room, layer of
// 4096 tokens on two streams 119.1 -> 121.7 us, and one stream adds up in the order of two.)
template <bool kSwiglu> struct Shape<9, kSwiglu> { enum { WM = 2, WN = 2, KG = 2, TM = 4, TN = 4, NS = 2 }; };      // 128 x 128, two K groups, one block to a CU
constexpr int kShapes = 10;
constexpr unsigned shapes_of(int layout) { return layout == kNN ? (1u << kShapes) - 1 : (1u << 9) - 1; }
// ... and what a launch of n blocks takes, in microseconds per 64 of K and round of `at_once` blocks: idle + (full - idle) times the share of
// the chip in use.  Measured on 256 x 256 x 4096 (few blocks) and 4096 x 4096 x 4096 (all CUs busy), the lower tiles and the 64 x 64 one over 57 products of
// 300 to 12000 rows, bf16, with equal rings of both operands; about 4 us more for a launch.  The times are lower now, and not all by the same share: over 174 products
// (x W^T, gate/up with SwiGLU, dy W; 64 to 12000 rows, 128 to 8192 columns, K 256 to 8192; weights in the caches) the rule's choice takes 1.9 / 1.1 / 1.2 % more than the
// best shape and split on average.  The most: 150 x 1496 x 6848, 96 x 128 in ten parts 15.6 us where 64 x 64 in three takes 12.9; gate/up of 293 x 2 2840 x 6912 17 %;
// the rest 10 % at most.  Figures fitted to the present kernels would be the way to these.
// The lower tiles took, the best of the others / theirs: gate/up of 3000 x 1024 x 4096 (256 tiles of 256 columns a round) 49.5 / 45.4 us, 613 x 1024 x 4096
// 17.4 / 15.2; down of 3000 x 4096 x 1024 31.9 / 29.4, 12000 x 1536 x 512 23.7 / 19.6; five weight gradients of 4096 tokens x 1024 x 4096 (200 tiles of
// 256 rows, 236 of 224), in a trace of whole steps, 106 / 101.
struct ShapeCost { int bm, bn, kg, at_once; float idle, full, fixed; };
constexpr ShapeCost kCost[kShapes] = {{256, 256, 1, 256, 1.10f, 1.55f, 5.f}, {256, 128, 1, 256, 0.66f, 0.92f, 4.5f}, {128, 128, 1, 512, 0.50f, 1.00f, 4.f},
                                      {128, 128, 1, 256, 0.44f, 0.57f, 4.f}, {64, 64, 2, 256, 0.16f, 0.235f, 4.f}, {224, 256, 1, 256, 1.04f, 1.44f, 5.f},
                                      {192, 256, 1, 256, 0.92f, 1.26f, 5.f}, {192, 128, 1, 256, 0.52f, 0.70f, 4.5f}, {96, 128, 1, 256, 0.36f, 0.47f, 4.f},
                                      {128, 128, 2, 256, 0.41f, 0.535f, 6.5f}};
constexpr ShapeCost kSwigluCost = {64, 128, 2, 256, 0.26f, 0.37f, 4.f};
// A split writes its fp32 sums and a second kernel adds them: its launch, and the two trips
constexpr float kReduceUs = 3.3f, kPartsOut = 8e6f, kPartsIn = 5e6f;      // us, bytes per us
constexpr int kMostSplits = 16;

struct TileChoice { int shape = 0, splits = 1; float us = 1e30f; };
struct TileSize { int64_t M, N; };
template <int DT, int LAY, int kId, int EPI, bool kTail, bool kStream, class Group>
struct TilesLds {
  using S = Shape<kId, EPI == kTileSwiglu>;
  static constexpr int kBytes = TileRing<staged_rows<LAY>(S::WM * S::TM * 16, S::WM * S::WN * S::KG), S::WN * S::TN * 16, S::KG, S::NS>::kBytes;
  static inline LdsKernel entry{(const void*)gemm_tiles_kernel<DT, LAY, S::WM, S::WN, S::KG, S::TM, S::TN, S::NS, EPI, kTail, kStream, Group>, kBytes};
};
template <int DT, int LAY, int kId, int EPI, bool kTail, bool kStream, class Group>
static hipError_t start_tiles(const Group& g, int64_t blocks, hipStream_t s) {
  using S = Shape<kId, EPI == kTileSwiglu>;
  using L = TilesLds<DT, LAY, kId, EPI, kTail, kStream, Group>;
  if (hipError_t e = L::entry.ensure(); e != hipSuccess) return e;
  hipLaunchKernelGGL((gemm_tiles_kernel<DT, LAY, S::WM, S::WN, S::KG, S::TM, S::TN, S::NS, EPI, kTail, kStream, Group>), dim3((unsigned)blocks),
                     dim3(S::WM * S::WN * S::KG * 64), L::kBytes, s, g);
  return hipGetLastError();
}
// ---- launches that two independent stages of the layer share -----------------------------------------
// Up to a few thousand tokens the router's projection and its selection are 6-8 us launches that leave most of the chip idle, and everything waits for
// them.  The projection's tiles go in front of the gate/up projection's (same tile shape), the selection beside the down projection's.
struct TilePair { TileSingle router, mlp; };
template <int DT, int kId, int kMlp, bool kTail>
__global__ __launch_bounds__(Shape<kId>::WM* Shape<kId>::WN* Shape<kId>::KG * 64, 2) void tile_pair_kernel(const TilePair g) {
  using R = Shape<kId>;
  using S = Shape<kMlp, true>;
  if ((int)blockIdx.x < g.mlp.p[0].first)
    tiles_block<DT, kNT, R::WM, R::WN, R::KG, R::TM, R::TN, R::NS, kTileTwo, kTail, false, TileSingle>(g.router, (int)blockIdx.x, (int)gridDim.x);
  else
    tiles_block<DT, kNT, S::WM, S::WN, S::KG, S::TM, S::TN, S::NS, kTileSwiglu, kTail, false, TileSingle>(g.mlp, (int)blockIdx.x, (int)gridDim.x);
}
struct TileSelect {
  TileSingle mlp;
  SelectArgs select;
  int regs, cells;                   // keys and candidates per lane
};
template <int DT, int kId>
__global__ __launch_bounds__(Shape<kId>::WM* Shape<kId>::WN* Shape<kId>::KG * 64, 2) void tile_select_kernel(const TileSelect g) {
  using S = Shape<kId>;
  const int select_blocks = g.mlp.p[0].first;
  if ((int)blockIdx.x < select_blocks) {
    constexpr int kWaves = S::WM * S::WN * S::KG;
    const int first = (int)blockIdx.x * kWaves + (int)(threadIdx.x >> 6), all = select_blocks * kWaves;
    const float* stats = g.select.stats;
    extern __shared__ __align__(16) uint8_t lds[];             // (the ring of the blocks that multiply)
    if (g.select.part_mean) {                                  // batch statistics: the block merges them first
      merge_statistics(g.select, (float*)lds, kWaves * kWave);
      stats = (const float*)lds;
    }
    count_batch(g.select);
    auto select = [&](auto cells) {
      constexpr int C = decltype(cells)::value;
      if (g.regs <= 1) select_packed<DT, 1, C>(g.select, first, all, stats);
      else if (g.regs <= 2) select_packed<DT, 2, C>(g.select, first, all, stats);
      else if (g.regs <= 4) select_packed<DT, 4, C>(g.select, first, all, stats);
      else select_packed<DT, 8, C>(g.select, first, all, stats);
    };
    if (g.cells <= 1) select(std::integral_constant<int, 1>{});
    else select(std::integral_constant<int, 2>{});
    return;
  }
  tiles_block<DT, kNT, S::WM, S::WN, S::KG, S::TM, S::TN, S::NS, kTilePlain, false, false, TileSingle>(g.mlp, (int)blockIdx.x, (int)gridDim.x);
}
template <int kId, bool kSwiglu>
constexpr int tile_lds() {
  using S = Shape<kId, kSwiglu>;
  constexpr int kBytes = TileRing<staged_rows<kNT>(S::WM * S::TM * 16, S::WM * S::WN * S::KG), S::WN * S::TN * 16, S::KG, S::NS>::kBytes;
  static_assert(kBytes >= 4 * merge_lds_floats(kMergeKeys, S::WM * S::WN * S::KG * 64), "a block that selects merges statistics there");
  return kBytes;
}
template <auto kKernel, int kBytes>
struct JointLds { static inline LdsKernel entry{(const void*)kKernel, kBytes}; };

// Tiles of one unsplit product of shape kId
template <int kId, bool kSwiglu>
static int64_t tile_count(const TileProduct& p) {
  using S = Shape<kId, kSwiglu>;
  constexpr int BM = S::WM * S::TM * 16, BN = S::WN * S::TN * 16 / (kSwiglu ? 2 : 1);
  return (int64_t)((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
}
template <int DT, int kId, int kMlp = kId>
static bool start_pair(TilePair& g, hipStream_t s, hipError_t* e) {
  using S = Shape<kId>;
  constexpr int kStep = 64 * S::KG, kBytes = tile_lds<kMlp, true>() > tile_lds<kId, false>() ? tile_lds<kMlp, true>() : tile_lds<kId, false>();
  TileProduct &r = g.router.p[0], &m = g.mlp.p[0];
  const int64_t rb = tile_count<kId, false>(r), mb = tile_count<kMlp, true>(m);
  if (rb + mb > INT32_MAX / 2) return false;
  r.steps = m.steps = (r.seg[0].K + kStep - 1) / kStep;
  m.first = (int)rb;
  auto go = [&](auto tail) {
    constexpr bool kTail = decltype(tail)::value;
    if ((*e = JointLds<tile_pair_kernel<DT, kId, kMlp, kTail>, kBytes>::entry.ensure()) != hipSuccess) return;
    hipLaunchKernelGGL((tile_pair_kernel<DT, kId, kMlp, kTail>), dim3((unsigned)(rb + mb)), dim3(S::WM * S::WN * S::KG * 64), kBytes, s, g);
    *e = hipGetLastError();
  };
  if (r.seg[0].K % kStep) go(std::true_type{});
  else go(std::false_type{});
  return true;
}

template <int DT, int LAY, int kId, int EPI>
static hipError_t launch_tiles(TileGroup& g, float* ws, int splits, bool exclusive, hipStream_t s) {
  using S = Shape<kId, EPI == kTileSwiglu>;
  constexpr int BM = S::WM * S::TM * 16, BN = S::WN * S::TN * 16 / (EPI == kTileSwiglu ? 2 : 1), kStep = 64 * S::KG;
  int64_t blocks = 0;
  bool tail = false;
  for (int i = 0; i < g.count; ++i) {
    TileProduct& p = g.p[i];
    int total = 0;
    for (int q = 0; q < p.segments; ++q) {
      total += (p.seg[q].K + kStep - 1) / kStep;
      tail = tail || p.seg[q].K % kStep != 0;
    }
    p.steps = (total + splits - 1) / splits;
    p.splits = (total + p.steps - 1) / p.steps;                // every split has work
    p.part = p.splits > 1 ? ws : nullptr;
    p.first = (int)blocks;
    blocks += (int64_t)((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN) * p.splits;
  }
  if (blocks > INT32_MAX / 2) return hipErrorInvalidValue;
  hipError_t e;
  if constexpr (LAY == kTN) {                                  // only these come in groups; neither operand's rows run along K
    if (g.count == 1) e = start_tiles<DT, LAY, kId, EPI, false, false>(TileSingle{{g.p[0]}}, blocks, s);
    else e = start_tiles<DT, LAY, kId, EPI, false, false>(g, blocks, s);
  } else {
    if (g.count != 1) return hipErrorInvalidValue;
    const TileSingle one{{g.p[0]}};
    if constexpr (LAY == kNT && (kId == 0 || kId == 5 || kId == 6)) {
      // one stream per CU where there are more tiles than CUs and nothing is meant to run beside the launch; else one block per tile, so
      // that CUs come free for other streams' kernels as blocks retire
      if (exclusive && blocks > 256 && splits == 1 && one.p[0].segments == 1)
        return tail ? start_tiles<DT, LAY, kId, EPI, true, true>(one, 256, s) : start_tiles<DT, LAY, kId, EPI, false, true>(one, 256, s);
    }
    e = tail ? start_tiles<DT, LAY, kId, EPI, true, false>(one, blocks, s) : start_tiles<DT, LAY, kId, EPI, false, false>(one, blocks, s);
  }
  if (e != hipSuccess) return e;
  if (g.p[0].part) {
    const TileProduct& p = g.p[0];
    const int64_t want = ((int64_t)p.M * (p.N / 8) + 255) / 256;
    hipLaunchKernelGGL((tile_reduce_kernel<DT, EPI>), dim3((unsigned)(want < 2048 ? want : 2048)), dim3(256), 0, s, p);
    e = hipGetLastError();
  }
  return e;
}

template <int DT, int LAY, int EPI>
static hipError_t launch_choice(TileGroup& g, const TileChoice& c, float* ws, bool exclusive, hipStream_t s) {
  switch (c.shape) {
    case 0: return launch_tiles<DT, LAY, 0, EPI>(g, ws, c.splits, exclusive, s);
    case 1: return launch_tiles<DT, LAY, 1, EPI>(g, ws, c.splits, exclusive, s);
    case 2: return launch_tiles<DT, LAY, 2, EPI>(g, ws, c.splits, exclusive, s);
    case 3: return launch_tiles<DT, LAY, 3, EPI>(g, ws, c.splits, exclusive, s);
    case 4:
      if constexpr (EPI == kTileSwiglu)
        if (g.p[0].seg[0].K > kShortSum * c.splits) return launch_tiles<DT, LAY, 10, EPI>(g, ws, c.splits, exclusive, s);
      return launch_tiles<DT, LAY, 4, EPI>(g, ws, c.splits, exclusive, s);
    case 5: return launch_tiles<DT, LAY, 5, EPI>(g, ws, c.splits, exclusive, s);
    case 6: return launch_tiles<DT, LAY, 6, EPI>(g, ws, c.splits, exclusive, s);
    case 7: return launch_tiles<DT, LAY, 7, EPI>(g, ws, c.splits, exclusive, s);
    case 9:
      if constexpr (LAY == kNN) return launch_tiles<DT, LAY, 9, EPI>(g, ws, c.splits, exclusive, s);
      else return hipErrorInvalidValue;
    default: return launch_tiles<DT, LAY, 8, EPI>(g, ws, c.splits, exclusive, s);
  }
}

// How the down projection runs on tiles of shape kId: ring steps of a part, parts, tiles of all parts, and the blocks of the selection beside them, if it is
struct DownPlan { int steps, splits; int64_t tiles, blocks; bool selected; };
template <int kId>
static DownPlan plan_down(int64_t M, int64_t N, int K, int splits, int tokens, int regs, int cells) {
  using S = Shape<kId>;
  constexpr int kStep = 64 * S::KG, kWaves = S::WM * S::WN * S::KG, BM = S::WM * S::TM * 16, BN = S::WN * S::TN * 16;
  const int total = (K + kStep - 1) / kStep;
  const int64_t once = kCost[kId].at_once, want = (tokens + kWaves - 1) / kWaves;
  const bool joint = total * kStep == K && regs <= 8 && cells <= 2;
  auto split = [&](int n) {
    DownPlan p;
    p.steps = (total + n - 1) / n;
    p.splits = (total + p.steps - 1) / p.steps;
    p.tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN) * p.splits;
    // the selection takes the places that the last round of tiles leaves free, when they make at most two tokens a wave (of more than 128 keys: one)
    const int64_t free = (p.tiles + once - 1) / once * once - p.tiles;
    p.blocks = want < free ? want : free;
    p.selected = joint && (regs <= 2 ? 2 : 1) * p.blocks * kWaves >= tokens;
    return p;
  };
  // ... for which a product in many splits gives up to a quarter of them (a launch is 5-7 us, a split step 0.2)
  int n = splits;
  DownPlan p = split(n);
  while (!p.selected && n > 1 && n > splits * 3 / 4) p = split(--n);
  return p.selected ? p : split(splits);
}
template <int DT, int kId>
static hipError_t start_down(TileProduct p, const SelectArgs& select, int splits, float* ws, hipStream_t s, bool* selected, int* parts) {
  using S = Shape<kId>;
  constexpr int kStep = 64 * S::KG, kWaves = S::WM * S::WN * S::KG, kBytes = tile_lds<kId, false>();
  TileSelect g{TileSingle{}, select, (select.r + kWave - 1) / kWave, 0};
  g.cells = prepare_select(g.select);
  const DownPlan plan = plan_down<kId>(p.M, p.N, p.seg[0].K, splits, select.num_tokens, g.regs, g.cells);
  p.steps = plan.steps;
  p.splits = plan.splits;
  p.part = p.splits > 1 ? ws : nullptr;
  const int64_t tiles = plan.tiles, blocks = plan.blocks;
  *selected = plan.selected;
  *parts = p.splits;
  if (tiles > INT32_MAX / 2) return hipErrorInvalidValue;
  if (*selected) {
    g.mlp.p[0] = p;
    g.mlp.p[0].first = (int)blocks;
    if (hipError_t e = JointLds<tile_select_kernel<DT, kId>, kBytes>::entry.ensure(); e != hipSuccess) return e;
    hipLaunchKernelGGL((tile_select_kernel<DT, kId>), dim3((unsigned)(blocks + tiles)), dim3(kWaves * 64), kBytes, s, g);
    return hipGetLastError();
  }
  const TileSingle one{{p}};
  return p.seg[0].K % kStep ? start_tiles<DT, kNT, kId, kTilePlain, true, false>(one, tiles, s) : start_tiles<DT, kNT, kId, kTilePlain, false, false>(one, tiles, s);
}

// ---- what gemm_tiles.hip calls, for one storage type
template <int DT>
hipError_t tile_group_of(int layout, int epilogue, TileGroup& g, const TileChoice& c, float* ws, bool exclusive, hipStream_t s) {
  if (layout == kNT && epilogue == kTilePlain) return launch_choice<DT, kNT, kTilePlain>(g, c, ws, exclusive, s);
  if (layout == kNT && epilogue == kTileResidual) return launch_choice<DT, kNT, kTileResidual>(g, c, ws, exclusive, s);
  if (layout == kNT && epilogue == kTileTwo) return launch_choice<DT, kNT, kTileTwo>(g, c, ws, exclusive, s);
  if (layout == kNT && epilogue == kTileSwiglu) return launch_choice<DT, kNT, kTileSwiglu>(g, c, ws, exclusive, s);
  if (layout == kNN && epilogue == kTilePlain) return launch_choice<DT, kNN, kTilePlain>(g, c, ws, exclusive, s);
  if (layout == kNN && epilogue == kTileResidual) return launch_choice<DT, kNN, kTileResidual>(g, c, ws, exclusive, s);
  if (layout == kNN && epilogue == kTileSwigluBwd) return launch_choice<DT, kNN, kTileSwigluBwd>(g, c, ws, exclusive, s);
  if (layout == kTN && epilogue == kTilePlain) return launch_choice<DT, kTN, kTilePlain>(g, c, ws, exclusive, s);
  return hipErrorInvalidValue;
}
template <int DT>
bool tile_pair_of(int shape, TilePair& g, hipStream_t s, hipError_t* e) {
  switch (shape) {
    case 1: return start_pair<DT, 1>(g, s, e);
    case 2: return start_pair<DT, 2>(g, s, e);
    case 3: return start_pair<DT, 3>(g, s, e);
    case 4: return g.mlp.p[0].seg[0].K > kShortSum ? start_pair<DT, 4, 10>(g, s, e) : start_pair<DT, 4>(g, s, e);
    case 7: return start_pair<DT, 7>(g, s, e);
    case 8: return start_pair<DT, 8>(g, s, e);
    default: return false;
  }
}
template <int DT>
hipError_t tile_down_of(const TileProduct& p, const SelectArgs& select, const TileChoice& c, float* ws, hipStream_t s, bool* selected, int* parts) {
  switch (c.shape) {
    case 1: return start_down<DT, 1>(p, select, c.splits, ws, s, selected, parts);
    case 2: return start_down<DT, 2>(p, select, c.splits, ws, s, selected, parts);
    case 3: return start_down<DT, 3>(p, select, c.splits, ws, s, selected, parts);
    case 4: return start_down<DT, 4>(p, select, c.splits, ws, s, selected, parts);
    case 7: return start_down<DT, 7>(p, select, c.splits, ws, s, selected, parts);
    case 8: return start_down<DT, 8>(p, select, c.splits, ws, s, selected, parts);
    default: {                                                 // nothing beside these
      *selected = false;
      *parts = 1;
      TileGroup g;
      g.p[g.count++] = p;
      return launch_choice<DT, kNT, kTilePlain>(g, c, ws, true, s);
    }
  }
}
// (each type's kernels are compiled in a file of their own)
extern template hipError_t tile_group_of<kBF16>(int, int, TileGroup&, const TileChoice&, float*, bool, hipStream_t);
extern template bool tile_pair_of<kBF16>(int, TilePair&, hipStream_t, hipError_t*);
extern template hipError_t tile_down_of<kBF16>(const TileProduct&, const SelectArgs&, const TileChoice&, float*, hipStream_t, bool*, int*);
extern template hipError_t tile_group_of<kF16>(int, int, TileGroup&, const TileChoice&, float*, bool, hipStream_t);
extern template bool tile_pair_of<kF16>(int, TilePair&, hipStream_t, hipError_t*);
extern template hipError_t tile_down_of<kF16>(const TileProduct&, const SelectArgs&, const TileChoice&, float*, hipStream_t, bool*, int*);

}  // namespace omni
