// MFMA GEMMs of the OmniMoE forward path for gfx950 (C = A * B^T, both operands with K
// contiguous, fp32 accumulation on the matrix cores):
//   * router projection   z  = x [Wx;Wy]^T                    (reference omni_moe.py:70-71)
//   * gate/up projection  h  = silu(x Wg^T) * (x Wu^T)         (interface.py:23-29, omni_mlp.py:53-61)
//     - the SwiGLU product is formed in the GEMM epilogue, so gate and up never reach HBM
//   * down projection     y  = h Wd^T (+ expert output)        (interface.py:23-29, omni_moe.py:102)
//
// The 16-bit projections go to the tile GEMM (gemm_tiles.hip) whenever their columns come in eights and every operand is 16-byte aligned.  Here are
//   * `gemm_nt_kernel`: single precision, and 16-bit products whose K is no multiple of 64 or whose operands lie at any other address (global ->
//     registers -> one of two LDS stages with padded rows);
//   * `gemm_nt_dma_kernel` and `gemm_ksplit_kernel`: the 16-bit router projection with column statistics, the gated product of the dense expert
//     algorithm, and aligned products whose columns do not come in eights (global -> LDS directly, ring of stages, swizzled rows).
// Structure: a block of 4 waves (2 x 2) owns a (2*TM*32) x (2*TN*32) tile; each wave owns
// TM x TN MFMA tiles of 32x32 and K advances 64 at a time.  The largest tile, 256 x 256, runs
// on 8 waves (2 x 4, two per SIMD) of 128 x 64 instead.  `gemm_ksplit_kernel` is for fewer 64 x 64 tiles than CUs: a
// block's waves share out the K tiles.
// The weight fragment is the MFMA's first operand, so an accumulator lane holds 4 consecutive
// output columns of one row; two lanes pair up to store 8 columns (16 bytes) each.
#include <algorithm>
#include "common.h"
#include "few_tokens.h"
#include "gemm_tiles.h"
#include "omni_moe_hip.h"
#include "select.h"

#include <type_traits>

namespace omni {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kBK = 64;                       // K elements per LDS stage
constexpr int kRowBytes = kBK * 2 + 16;       // padded LDS row
constexpr int kGemmThreads = 256;

constexpr int ksplit_lds(int tm) { return 4 * (tm == 1 ? 3 : 2) * (32 * tm + 64) * 128; }    // gemm_ksplit_kernel's four rings

enum : int { kEpiPlain = 0, kEpiSwiglu = 1, kEpiResidual = 2, kEpiStats = 3, kEpiGate = 4 };   // kEpiStats: plain + column statistics; kEpiGate: silu(acc) * gate, as a pair of 16-bit values

template <int DT> struct ElemBytes { static constexpr int value = (DT == kF32) ? 4 : 2; };

// One 16-byte fragment per lane of each operand: 8 K-values per lane (32x32x16) for 16-bit
// storage; for fp32 the 4 K-values per lane feed four 32x32x2 steps (lane halves pair up
// k and k+4 -- any pairing works as long as both operands use the same one).
template <int DT>
__device__ __forceinline__ f32x16_t mfma32(const u32x4_t a, const u32x4_t b, f32x16_t c) {
  if constexpr (DT == kBF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  } else if constexpr (DT == kF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t ae = a[e], be = b[e];
      c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(ae), __uint_as_float(be), c, 0, 0, 0);
    }
    return c;
  }
}

template <int DT>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  if constexpr (DT == kBF16) return pack_bf16(lo, hi);
  else if constexpr (DT == kF16) return pack_f16(lo, hi);
  else return 0u;
}

struct GemmArgs {           // all element offsets below are scaled by the element size of DT
  const uint8_t* a;       // [M, K]  activations
  const uint8_t* b0;      // [N, K]  weights (gate weights for SwiGLU)
  const uint8_t* b1;      // [N, K]  up weights (SwiGLU), or the upper half of the columns (plain)
  const uint8_t* res;     // [M, N]  added to the result (residual epilogue only)
  uint8_t* c;             // [M, N]
  int M, N, K;            // N = output columns
  int tiles_m, tiles_n;
  int patch_m, patch_n;   // XCD patch shape (0 = plain order)
  int wide;               // 16-bit output: N % 8 == 0 and C 16-byte aligned, rows are written 16 bytes per lane
  int single;             // N % 4 != 0: rows are not 8-byte aligned, results leave element by element
  float* part_mean;       // kEpiStats only: [ceil(M/32)][N] mean of each column over
  float* part_m2;         //   rows 32s..32s+31 of the ROUNDED result, and the sum of squared deviations
  const float* gate;      // kEpiGate only: [M, N] fp32 factors; C is then [M, 2N]: round(v) in columns 0..N-1, round(v - round(v)) in N..2N-1
};

// Which output tile a block owns.  Blocks go round-robin over the 8 XCDs; each XCD gets
// compact patches of tiles so that the blocks sharing its L2 share operand panels.
__device__ __forceinline__ void tile_coords(const GemmArgs& g, int& tile_m, int& tile_n) {
  const int b = blockIdx.x;
  if (g.patch_m > 0) {
    const int per_patch = g.patch_m * g.patch_n;
    const int xcd = b & 7, idx = b >> 3;
    const int patch = (idx / per_patch) * 8 + xcd, within = idx % per_patch;
    const int patches_m = g.tiles_m / g.patch_m;
    tile_m = (patch % patches_m) * g.patch_m + within % g.patch_m;
    tile_n = (patch / patches_m) * g.patch_n + within / g.patch_m;
  } else {
    tile_m = b % g.tiles_m;
    tile_n = b / g.tiles_m;
  }
}

// Writes a wave's TM x TN accumulator tiles.  acc[i][j][q] is row m = lane%32 and column
// n = (q/4)*8 + (lane/32)*4 + q%4 of MFMA tile (i, j).
template <int DT, int TM, int TN, int EPI>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs& g, f32x16_t (&acc)[TM][TN], const int m0, const int n0,
                                              const int wm, const int wn, const int lane) {
  constexpr int TNO = (EPI == kEpiSwiglu) ? TN / 2 : TN;
  // ---- column statistics of the rounded tile for BatchNorm: every 32-row MFMA tile is one
  // strip.  A column's 32 rows sit in the 32 lanes that share lane/32, one of this lane's 16
  // values each, so the 16 columns of a half-wave are reduced together: a butterfly that halves
  // the values a lane keeps at every step (8 + 4 + 2 + 1 + 1 exchanges) leaves each lane pair
  // with the sum of ONE column; the means travel back the same way (1 + 2 + 4 + 8), the squared
  // deviations are reduced like the sums.  47 register-to-register exchanges per tile.
  if constexpr (EPI == kEpiStats) {
    if (g.part_mean) {
      const bool b16 = lane & 16, b8 = lane & 8, b4 = lane & 4, b2 = lane & 2;
      auto reduce_scatter = [&](const float (&v)[16]) -> float {
        float a8[8], a4[4], a2[2];
#pragma unroll
        for (int e = 0; e < 8; ++e) a8[e] = (b16 ? v[e + 8] : v[e]) + xor_lane_f<16>(b16 ? v[e] : v[e + 8], lane);
#pragma unroll
        for (int e = 0; e < 4; ++e) a4[e] = (b8 ? a8[e + 4] : a8[e]) + xor_lane_f<8>(b8 ? a8[e] : a8[e + 4], lane);
#pragma unroll
        for (int e = 0; e < 2; ++e) a2[e] = (b4 ? a4[e + 2] : a4[e]) + xor_lane_f<4>(b4 ? a4[e] : a4[e + 2], lane);
        const float a1 = (b2 ? a2[1] : a2[0]) + xor_lane_f<2>(b2 ? a2[0] : a2[1], lane);
        return a1 + xor_lane_f<1>(a1, lane);
      };
      // the column this lane ends up with: q = 8*b16 + 4*b8 + 2*b4 + b2
      const int q_mine = (b16 ? 8 : 0) + (b8 ? 4 : 0) + (b4 ? 2 : 0) + (b2 ? 1 : 0);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row0 = m0 + wm * TM * 32 + i * 32;
        const int cnt = min(32, g.M - row0);
        if (cnt <= 0) continue;
        const bool live = (lane & 31) < cnt;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          float v[16];
#pragma unroll
          for (int q = 0; q < 16; ++q) v[q] = live ? Elem<DT>::round(acc[i][j][q]) : 0.f;
          const float mean = reduce_scatter(v) / float(cnt);
          // all-gather of the 16 means, index = column
          float g2[2], g4[4], g8[8], mu[16];
          {
            const float o = xor_lane_f<2>(mean, lane);
            g2[0] = b2 ? o : mean;
            g2[1] = b2 ? mean : o;
          }
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const float o = xor_lane_f<4>(g2[e], lane);
            g4[e] = b4 ? o : g2[e];
            g4[e + 2] = b4 ? g2[e] : o;
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float o = xor_lane_f<8>(g4[e], lane);
            g8[e] = b8 ? o : g4[e];
            g8[e + 4] = b8 ? g4[e] : o;
          }
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float o = xor_lane_f<16>(g8[e], lane);
            mu[e] = b16 ? o : g8[e];
            mu[e + 8] = b16 ? g8[e] : o;
          }
          float d[16];
#pragma unroll
          for (int q = 0; q < 16; ++q) d[q] = live ? (v[q] - mu[q]) * (v[q] - mu[q]) : 0.f;
          const float m2 = reduce_scatter(d);
          const int n = n0 + wn * TN * 32 + j * 32 + (q_mine >> 2) * 8 + (lane >> 5) * 4 + (q_mine & 3);
          if ((lane & 1) == 0 && n < g.N) {
            g.part_mean[(int64_t)(row0 >> 5) * g.N + n] = mean;
            g.part_m2[(int64_t)(row0 >> 5) * g.N + n] = m2;
          }
        }
      }
    }
  }

  // ---- epilogue.  acc[i][j][q]: row m = lane%32, column n = (q/4)*8 + (lane/32)*4 + q%4
  // value q of column group q4 after the element-wise tail, not yet rounded to storage
  auto value = [&](int i, int j, int q4, int q) -> float {
    if constexpr (EPI == kEpiSwiglu) {
      // the reference materialises gate and up in the storage dtype, then forms
      // silu(gate)*up in fp32 and rounds once (omni_mlp.py:53-61)
      const float gt = Elem<DT>::round(acc[i][j][q4 * 4 + q]);
      const float up = Elem<DT>::round(acc[i][j + TNO][q4 * 4 + q]);
      return (DT == kF32) ? silu_f32(gt) * up : silu_fast(gt) * up;
    } else {
      return acc[i][j][q4 * 4 + q];
    }
  };
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + wm * TM * 32 + i * 32 + (lane & 31);
    if (m >= g.M) continue;
#pragma unroll
    for (int j = 0; j < TNO; ++j) {
      const int nt = n0 + wn * TNO * 32 + j * 32;
      if constexpr (DT != kF32) {
        if (g.wide) {
          // lanes l and l+32 hold columns 8*q4+{0..3} and 8*q4+{4..7} of the same row: one
          // v_permlane32_swap per word regroups two column groups into 8 consecutive columns per
          // lane, so a row receives full 32-byte sectors from every store instruction
#pragma unroll
          for (int pr = 0; pr < 2; ++pr) {
            if (nt + pr * 16 >= g.N) continue;             // same answer in both lanes of a pair
            if constexpr (EPI == kEpiGate) {
              // c = silu(acc) * gate in fp32, stored as a 16-bit head and a 16-bit remainder (head + remainder carries 16
              // significant bits), so that a following GEMM over [head | remainder] sums in nearly full precision
              uint32_t hw[2][2], lw[2][2];
#pragma unroll
              for (int e = 0; e < 2; ++e) {
                const int q4 = 2 * pr + e;
                const int n = nt + q4 * 8 + (lane >> 5) * 4;
                f32x4_t gt = {0.f, 0.f, 0.f, 0.f};
                if (n < g.N) gt = *(const f32x4_t*)(g.gate + (int64_t)m * g.N + n);
                float hv[4], lv[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                  const float c = gt[q] != 0.f ? silu_f32(acc[i][j][q4 * 4 + q]) * gt[q] : 0.f;   // an unselected pair contributes exactly 0, whatever its product is
                  hv[q] = Elem<DT>::round(c);
                  lv[q] = c - hv[q];
                }
                hw[e][0] = pack2<DT>(hv[0], hv[1]); hw[e][1] = pack2<DT>(hv[2], hv[3]);
                lw[e][0] = pack2<DT>(lv[0], lv[1]); lw[e][1] = pack2<DT>(lv[2], lv[3]);
              }
              const auto h0 = __builtin_amdgcn_permlane32_swap(hw[0][0], hw[1][0], false, false);
              const auto h1 = __builtin_amdgcn_permlane32_swap(hw[0][1], hw[1][1], false, false);
              const auto l0 = __builtin_amdgcn_permlane32_swap(lw[0][0], lw[1][0], false, false);
              const auto l1 = __builtin_amdgcn_permlane32_swap(lw[0][1], lw[1][1], false, false);
              const int n = nt + pr * 16 + (lane >> 5) * 8;
              if (n < g.N) {
                *(u32x4_t*)(g.c + ((int64_t)m * 2 * g.N + n) * 2) = u32x4_t{h0[0], h1[0], h0[1], h1[1]};
                *(u32x4_t*)(g.c + ((int64_t)m * 2 * g.N + g.N + n) * 2) = u32x4_t{l0[0], l1[0], l0[1], l1[1]};
              }
              continue;
            }
            uint32_t w[2][2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const int q4 = 2 * pr + e;
              float v[4];
#pragma unroll
              for (int q = 0; q < 4; ++q) v[q] = value(i, j, q4, q);
              if constexpr (EPI == kEpiResidual) {
                const int n = nt + q4 * 8 + (lane >> 5) * 4;
                u32x2_t r = {0u, 0u};                      // columns past N are exchanged but never stored
                if (n < g.N) r = *(const u32x2_t*)(g.res + ((int64_t)m * g.N + n) * 2);
                const uint32_t r0 = r[0], r1 = r[1];
                if constexpr (DT == kBF16) {
                  v[0] = Elem<DT>::round(v[0]) + bf16_lo(r0); v[1] = Elem<DT>::round(v[1]) + bf16_hi(r0);
                  v[2] = Elem<DT>::round(v[2]) + bf16_lo(r1); v[3] = Elem<DT>::round(v[3]) + bf16_hi(r1);
                } else {
                  v[0] = Elem<DT>::round(v[0]) + f16_bits_to_f32(r0 & 0xffff); v[1] = Elem<DT>::round(v[1]) + f16_bits_to_f32(r0 >> 16);
                  v[2] = Elem<DT>::round(v[2]) + f16_bits_to_f32(r1 & 0xffff); v[3] = Elem<DT>::round(v[3]) + f16_bits_to_f32(r1 >> 16);
                }
              }
              w[e][0] = pack2<DT>(v[0], v[1]);
              w[e][1] = pack2<DT>(v[2], v[3]);
            }
            const auto s0 = __builtin_amdgcn_permlane32_swap(w[0][0], w[1][0], false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(w[0][1], w[1][1], false, false);
            const int n = nt + pr * 16 + (lane >> 5) * 8;
            if (n < g.N) *(u32x4_t*)(g.c + ((int64_t)m * g.N + n) * 2) = u32x4_t{s0[0], s1[0], s0[1], s1[1]};
          }
          continue;
        }
      }
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int n = nt + q4 * 8 + (lane >> 5) * 4;
        if (n >= g.N) continue;
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = value(i, j, q4, q);
        if (g.single) {                                  // any N: one element at a time
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (n + q >= g.N) continue;
            const int64_t at = (int64_t)m * g.N + n + q;
            float out = v[q];
            if constexpr (EPI == kEpiResidual) out = Elem<DT>::round(out) + Elem<DT>::load(g.res, at);
            Elem<DT>::store(g.c, at, out);
          }
          continue;
        }
        const int64_t o = ((int64_t)m * g.N + n) * ElemBytes<DT>::value;   // N is a multiple of 4 here
        if constexpr (EPI == kEpiResidual) {
          // y = round(h Wd^T) + e, rounded again: the reference adds two stored tensors
          if constexpr (DT == kF32) {
            const f32x4_t r = *(const f32x4_t*)(g.res + o);
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] += r[q];
          } else {
            const u32x2_t r = *(const u32x2_t*)(g.res + o);
            const uint32_t r0 = r[0], r1 = r[1];
            if constexpr (DT == kBF16) {
              v[0] = Elem<DT>::round(v[0]) + bf16_lo(r0); v[1] = Elem<DT>::round(v[1]) + bf16_hi(r0);
              v[2] = Elem<DT>::round(v[2]) + bf16_lo(r1); v[3] = Elem<DT>::round(v[3]) + bf16_hi(r1);
            } else {
              v[0] = Elem<DT>::round(v[0]) + f16_bits_to_f32(r0 & 0xffff); v[1] = Elem<DT>::round(v[1]) + f16_bits_to_f32(r0 >> 16);
              v[2] = Elem<DT>::round(v[2]) + f16_bits_to_f32(r1 & 0xffff); v[3] = Elem<DT>::round(v[3]) + f16_bits_to_f32(r1 >> 16);
            }
          }
        }
        if constexpr (DT == kF32) {
          *(f32x4_t*)(g.c + o) = f32x4_t{v[0], v[1], v[2], v[3]};
        } else {
          u32x2_t w = {pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3])};
          *(u32x2_t*)(g.c + o) = w;
        }
      }
    }
  }
}

// Register-staged kernel, any storage dtype: TM x TN MFMA tiles per wave, K advances by one
// 128-byte row (64 16-bit or 32 fp32 values).  For the SwiGLU epilogue the first TN/2 tiles of
// a wave are gate columns and the last TN/2 the matching up columns.
template <int DT, int TM, int TN, int EPI>
__global__ __launch_bounds__(kGemmThreads, 1) void gemm_nt_kernel(const GemmArgs g) {
  constexpr int BM = 2 * TM * 32;                 // rows of A per block
  constexpr int BR = 2 * TN * 32;                 // rows of the weight tile in LDS per block
  constexpr int BN = (EPI == kEpiSwiglu) ? BR / 2 : BR;   // output columns per block
  constexpr int TNO = (EPI == kEpiSwiglu) ? TN / 2 : TN;  // output tiles per wave along N
  constexpr int kStageBytes = (BM + BR) * kRowBytes;
  extern __shared__ __align__(16) uint8_t lds[];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;

  int tile_m, tile_n;
  tile_coords(g, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  // ---- global -> register staging: thread owns 16-byte chunk (tid%8) of rows tid/8 + 32*p
  constexpr int ES = ElemBytes<DT>::value, CE = 16 / ES, BKE = 128 / ES;   // chunk / tile width in elements
  const int ld_chunk = tid & 7, ld_row = tid >> 3;
  constexpr int PA = BM / 32, PB = BR / 32;
  const uint8_t* a_ptr[PA];
  const uint8_t* b_ptr[PB];
#pragma unroll
  for (int p = 0; p < PA; ++p) {
    int row = m0 + p * 32 + ld_row;
    row = row < g.M ? row : g.M - 1;                     // clamp: tail rows are never stored
    a_ptr[p] = g.a + ((int64_t)row * g.K + ld_chunk * CE) * ES;
  }
#pragma unroll
  for (int p = 0; p < PB; ++p) {
    // LDS weight row p*32+ld_row belongs to wave column p/TN, tile p%TN
    const int pw = p / TN, pj = p % TN;
    const uint8_t* base = g.b0;
    int col;
    if constexpr (EPI == kEpiSwiglu) {
      base = (pj < TNO) ? g.b0 : g.b1;
      col = n0 + pw * (TNO * 32) + (pj % TNO) * 32 + ld_row;
    } else {
      col = n0 + p * 32 + ld_row;
    }
    col = col < g.N ? col : g.N - 1;
    if constexpr (EPI == kEpiPlain || EPI == kEpiStats) {
      // optional second weight matrix supplies the upper half of the output columns
      if (g.b1 && col >= g.N / 2) { base = g.b1; col -= g.N / 2; }
    }
    b_ptr[p] = base + ((int64_t)col * g.K + ld_chunk * CE) * ES;
  }
  const int lds_wr = ld_row * kRowBytes + ld_chunk * 16;

  u32x4_t ra[PA], rb[PB];
  auto load_tile = [&](int k0) {
    const bool ok = k0 + ld_chunk * CE < g.K;            // K is a multiple of the chunk: whole chunks
#pragma unroll
    for (int p = 0; p < PA; ++p) ra[p] = ok ? *(const u32x4_t*)(a_ptr[p] + (int64_t)k0 * ES) : u32x4_t{0, 0, 0, 0};
#pragma unroll
    for (int p = 0; p < PB; ++p) rb[p] = ok ? *(const u32x4_t*)(b_ptr[p] + (int64_t)k0 * ES) : u32x4_t{0, 0, 0, 0};
  };
  auto store_tile = [&](int stage) {
    uint8_t* sa = lds + stage * kStageBytes;
    uint8_t* sb = sa + BM * kRowBytes;
#pragma unroll
    for (int p = 0; p < PA; ++p) *(u32x4_t*)(sa + p * 32 * kRowBytes + lds_wr) = ra[p];
#pragma unroll
    for (int p = 0; p < PB; ++p) *(u32x4_t*)(sb + p * 32 * kRowBytes + lds_wr) = rb[p];
  };

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;

  // fragment read offsets: lane reads row (lane%32), 16-byte chunk (lane/32) of a 32-byte slab
  const int frag_off = (lane & 31) * kRowBytes + (lane >> 5) * 16;
  const int a_frag = (wm * TM * 32) * kRowBytes + frag_off;
  const int b_frag = BM * kRowBytes + (wn * TN * 32) * kRowBytes + frag_off;

  const int num_kt = (g.K + BKE - 1) / BKE;
  load_tile(0);
  store_tile(0);
  __syncthreads();
  for (int kt = 0; kt < num_kt; ++kt) {
    const uint8_t* st = lds + (kt & 1) * kStageBytes;
    if (kt + 1 < num_kt) load_tile((kt + 1) * BKE);
#pragma unroll
    for (int slab = 0; slab < 4; ++slab) {
      u32x4_t af[TM], bf[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = *(const u32x4_t*)(st + a_frag + i * 32 * kRowBytes + slab * 32);
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[j] = *(const u32x4_t*)(st + b_frag + j * 32 * kRowBytes + slab * 32);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mfma32<DT>(bf[j], af[i], acc[i][j]);
    }
    if (kt + 1 < num_kt) store_tile((kt + 1) & 1);
    __syncthreads();
  }

  gemm_epilogue<DT, TM, TN, EPI>(g, acc, m0, n0, wm, wn, lane);
}

// ---- main kernel: global -> LDS without passing through registers ------------------------
// K advances BK (32 or 64) at a time through a ring of NS LDS stages that
// `global_load_lds_dwordx4` fills directly.  Each wave instruction lands 1 KiB of consecutive
// LDS, so rows cannot be padded; instead the 16-byte chunk c of row r is kept at a swizzled
// chunk position (the loading lane applies the swizzle to its GLOBAL address), chosen so that
// the 128-bit fragment reads of 16 consecutive rows cover all 64 banks once.  NS-2 tiles are
// in flight while one is computed.  The K=16 slabs are skewed across the tile boundary: the
// last slab's fragments of a tile are in registers before the barrier that releases its
// stage, so the MFMAs of one slab always cover the LDS reads of the next.  Needs K % BK == 0.
template <int N> __device__ __forceinline__ void wait_vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void wait_lds_reads() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// chunk position of logical 16-byte chunk c in row r of a tile whose rows hold BK elements
template <int BK> __device__ __forceinline__ int swizzle(int r, int c) {
  if constexpr (BK == 32) return c ^ ((r >> 2) & 3);      // 4 chunks per 64-byte row
  else return c ^ ((r >> 1) & 7);                          // 8 chunks per 128-byte row
}

template <int DT, int TM, int TN, int EPI, int BK, int NS, int NW = 4>
__global__ __launch_bounds__(NW * 64, 1) void gemm_nt_dma_kernel(const GemmArgs g) {
  // NW waves as 2 (rows) x NW/2 (columns) wave tiles of TM x TN MFMA tiles
  constexpr int BM = 2 * TM * 32, BR = (NW / 2) * TN * 32;
  constexpr int BN = (EPI == kEpiSwiglu) ? BR / 2 : BR;
  constexpr int TNO = (EPI == kEpiSwiglu) ? TN / 2 : TN;
  constexpr int kRow = BK * 2;                         // bytes per LDS row
  constexpr int kCpr = kRow / 16;                      // chunks per row
  constexpr int kRpi = 64 / kCpr;                      // rows one wave instruction fills
  constexpr int kStageBytes = (BM + BR) * kRow;
  constexpr int PA = BM / (NW * kRpi), PB = BR / (NW * kRpi);   // load instructions per wave per tile
  constexpr int LPT = PA + PB;
  constexpr int S = BK / 16;                           // slabs per tile
  extern __shared__ __align__(16) uint8_t lds[];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  int tile_m, tile_n;
  tile_coords(g, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  // load instruction p of wave w fills tile rows (4p+w)*kRpi ..: lane -> row lane/kCpr, position lane%kCpr
  const uint8_t* a_src[PA];
  const uint8_t* b_src[PB];
#pragma unroll
  for (int p = 0; p < PA; ++p) {
    const int rl = (NW * p + wave) * kRpi + lane / kCpr;
    const int c = swizzle<BK>(rl, lane % kCpr);        // an involution: position -> logical chunk
    int row = m0 + rl;
    row = row < g.M ? row : g.M - 1;                    // clamp: tail rows are never stored
    a_src[p] = g.a + ((int64_t)row * g.K + c * 8) * 2;
  }
#pragma unroll
  for (int p = 0; p < PB; ++p) {
    const int rl = (NW * p + wave) * kRpi + lane / kCpr;   // row of the weight tile in LDS
    const int c = swizzle<BK>(rl, lane % kCpr);
    const uint8_t* base = g.b0;
    int col;
    if constexpr (EPI == kEpiSwiglu) {
      const int pw = rl / (TN * 32), pj = (rl >> 5) % TN;
      base = (pj < TNO) ? g.b0 : g.b1;
      col = n0 + pw * (TNO * 32) + (pj % TNO) * 32 + (rl & 31);
    } else {
      col = n0 + rl;
    }
    col = col < g.N ? col : g.N - 1;
    if constexpr (EPI == kEpiPlain || EPI == kEpiStats) {
      if (g.b1 && col >= g.N / 2) { base = g.b1; col -= g.N / 2; }
    }
    b_src[p] = base + ((int64_t)col * g.K + c * 8) * 2;
  }

  const int wave_s = __builtin_amdgcn_readfirstlane(wave);   // scalar copy: LDS destinations stay in SGPRs
  // load instruction q (0 .. LPT-1) of tile kt: first the PA instructions of the activation tile, then the weights'
  auto issue_one = [&](int kt, int q) __attribute__((always_inline)) {
    uint8_t* st = lds + (kt % NS) * kStageBytes;
    const int koff = kt * kRow;
    if (q < PA)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a_src[q] + koff),
                                       (__attribute__((address_space(3))) void*)(st + (NW * q + wave_s) * 1024), 16, 0, 0);
    else
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(b_src[q - PA] + koff),
                                       (__attribute__((address_space(3))) void*)(st + BM * kRow + (NW * (q - PA) + wave_s) * 1024), 16, 0, 0);
  };
  auto issue_tile = [&](int kt) {
#pragma unroll
    for (int q = 0; q < LPT; ++q) issue_one(kt, q);
  };

  // fragment reads: lane reads row lane%32, logical chunk 2*slab + lane/32, into buffer slab&1
  const int rl = lane & 31;
  int off_slab[S];
#pragma unroll
  for (int sl = 0; sl < S; ++sl) off_slab[sl] = rl * kRow + swizzle<BK>(rl, 2 * sl + (lane >> 5)) * 16;
  const int a_frag = (wm * TM * 32) * kRow, b_frag = BM * kRow + (wn * TN * 32) * kRow;
  u32x4_t af[2][TM], bf[2][TN];
  // fragment f of a slab: 0 .. TM-1 activation rows, TM .. TM+TN-1 weight rows
  auto read_one = [&](int kt, int slab, int f) __attribute__((always_inline)) {
    const uint8_t* st = lds + (kt % NS) * kStageBytes + off_slab[slab];
    if (f < TM) af[slab & 1][f] = *(const u32x4_t*)(st + a_frag + f * 32 * kRow);
    else bf[slab & 1][f - TM] = *(const u32x4_t*)(st + b_frag + (f - TM) * 32 * kRow);
  };

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;

  // One slab = TM*TN MFMAs.  Every MFMA keeps the matrix pipeline busy for 32 cycles, during which
  // this wave may issue other instructions for free -- but a burst of memory instructions takes longer
  // to issue than that and stalls the MFMAs behind it (8 ds_read_b128 in a row cost 9 % of a 16-MFMA
  // slab, one behind each MFMA costs 1 %).  So the memory work of a slab is dealt out behind its MFMAs,
  // a slot each: first the TM + TN fragment reads of the FOLLOWING slab (into the other fragment
  // buffer), then, where a tile is to be fetched, half of that tile's LDS-DMA loads (a tile's loads are
  // issued over two slabs).  The compiler waits for all outstanding LDS reads in front of the next
  // slab's first MFMA; the last read was issued at least TM*TN - (TM+TN) MFMAs earlier.
  constexpr int kMf = TM * TN, kReads = TM + TN, kDmaPerSlab = LPT / 2;
  static_assert(LPT % 2 == 0, "a tile's loads are issued in two halves");
  // kFetch: this slab has slots for loads; they are issued when fetch_kt >= 0 (a scalar branch around
  // each load: control flow around the MFMAs themselves would make the accumulators phi nodes).
  auto slab_step = [&](auto fetch_tag, auto sl_tag, auto next_slab_tag, int next_kt, int fetch_kt, int half) __attribute__((always_inline)) {
    constexpr bool kFetch = decltype(fetch_tag)::value;
    constexpr int sl = decltype(sl_tag)::value, next_slab = decltype(next_slab_tag)::value;
    constexpr int kOps = kReads + (kFetch ? kDmaPerSlab : 0);
    constexpr int kPerSlot = (kOps + kMf - 1) / kMf;
#pragma unroll
    for (int ij = 0; ij < kMf; ++ij) {
      const int i = ij / TN, j = ij % TN;
      acc[i][j] = mfma32<DT>(bf[sl & 1][j], af[sl & 1][i], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < kPerSlot; ++u) {
        const int op = ij * kPerSlot + u;
        if (op < kReads) read_one(next_kt, next_slab, op);
        else if (kFetch && op < kOps) { if (fetch_kt >= 0) issue_one(fetch_kt, half * kDmaPerSlab + (op - kReads)); }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto slab_then_read = [&](auto sl_tag, auto next_slab_tag, int next_kt) __attribute__((always_inline)) {
    slab_step(std::false_type{}, sl_tag, next_slab_tag, next_kt, -1, 0);
  };
  auto slab_then_read_fetch = [&](auto sl_tag, auto next_slab_tag, int next_kt, int fetch_kt, int half) __attribute__((always_inline)) {
    slab_step(std::true_type{}, sl_tag, next_slab_tag, next_kt, fetch_kt, half);
  };
  // slabs 1 .. S-2 of a tile (no loads are issued during them)
  auto middle_slabs = [&](int kt) __attribute__((always_inline)) {
    if constexpr (S >= 3) slab_then_read(std::integral_constant<int, 1>{}, std::integral_constant<int, 2>{}, kt);
    if constexpr (S >= 4) slab_then_read(std::integral_constant<int, 2>{}, std::integral_constant<int, 3>{}, kt);
    static_assert(S <= 4, "at most four slabs per tile");
  };

  const int num_kt = g.K / BK;
#pragma unroll
  for (int t = 0; t < NS; ++t)
    if (t < num_kt) issue_tile(t);
  // before a tile is used, at most NS-2 younger tiles may still be in flight
  auto wait_tile = [&](int younger) {        // younger = tiles issued after the one needed
    if constexpr (NS >= 4) { if (younger >= 2) { wait_vmcnt<2 * LPT>(); return; } }
    if constexpr (NS >= 3) { if (younger >= 1) { wait_vmcnt<LPT>(); return; } }
    wait_vmcnt<0>();
  };
  wait_tile(min(NS, num_kt) - 1 < NS - 2 ? min(NS, num_kt) - 1 : NS - 2);
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int f = 0; f < kReads; ++f) read_one(0, 0, f);
  int fetch = -1;                             // tile whose loads are half issued
  for (int kt = 0; kt < num_kt - 1; ++kt) {
    slab_then_read_fetch(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{}, kt, fetch, 1);   // S >= 2: slab 0 is never the tile's last
    middle_slabs(kt);
    wait_lds_reads();                         // this wave holds every fragment of tile kt
    // tiles kt+1 .. min(kt+NS-1, num_kt-1) are outstanding; tile kt+1 must have landed
    const int younger = num_kt - 2 - kt;
    wait_tile(younger < NS - 2 ? younger : NS - 2);
    __builtin_amdgcn_s_barrier();             // tile kt+1 visible to all; stage of tile kt free
    fetch = (kt + NS < num_kt) ? kt + NS : -1;
    __builtin_amdgcn_sched_barrier(0);
    slab_then_read_fetch(std::integral_constant<int, S - 1>{}, std::integral_constant<int, 0>{}, kt + 1, fetch, 0);
  }
  slab_then_read(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{}, num_kt - 1);   // last tile
  middle_slabs(num_kt - 1);
#pragma unroll
  for (int ij = 0; ij < kMf; ++ij) acc[ij / TN][ij % TN] = mfma32<DT>(bf[(S - 1) & 1][ij % TN], af[(S - 1) & 1][ij / TN], acc[ij / TN][ij % TN]);
  gemm_epilogue<DT, TM, TN, EPI>(g, acc, m0, n0, wm, wn, lane);
}

// ---- few output tiles, long K: the K tiles of one 32 TM x 64 output tile dealt out over the block's four waves ----------
// A product like the router projection at a few thousand tokens (4096 x 128 x 1024) has too few output tiles to fill the
// GPU and its time is the latency of one block's K loop: with the ring kernel above, 16 rounds of wait - barrier - four
// MFMAs.  Here every wave multiplies the whole tile (TM x 2 MFMA tiles) over ITS K tiles (kt = wave, wave + 4,
// ...) through an LDS ring of its own, so the K loop is a quarter as long, has independent accumulators
// to keep the matrix pipeline fed, and meets no block barrier: a wave waits only for its own loads.  The four partial
// tiles then meet in LDS (summed in wave order, so the result does not depend on timing), and wave w finishes MFMA tile
// (w % TM, w / TM) with the common epilogue.  Needs K % 64 == 0; worth it while there are fewer tiles than CUs.
// TM = 1 where that makes at most 256 blocks and nothing runs beside the launch: every CU may have one, which loads three quarters as much, with three
// stages in flight instead of two (router stage of 1000 / 2048 / 4096 tokens, hidden 1024, 64 keys: 16.3 / 16.8 / 19.3 -> 15.6 / 16.3 / 18.5 us).  Beside gate/up,
// whose 256 x 256 tiles take all of a CU's LDS, blocks of both kinds wait for one another: the 4096-token layer on two streams 118 -> 130 us.
template <int DT, int EPI, int TM>
__global__ __launch_bounds__(kGemmThreads, 1) void gemm_ksplit_kernel(const GemmArgs g) {
  constexpr int kRow = 128, kATile = 32 * TM * kRow, kBTile = 64 * kRow, PA = 4 * TM, PB = 8;      // a K tile of each operand, in 1-KiB loads
  constexpr int NS = TM == 1 ? 3 : 2, kStage = kATile + kBTile, kRing = NS * kStage;              // per wave: stages of [activations | weights]
  static_assert(4 * kRing == ksplit_lds(TM), "launch and kernel disagree");
  extern __shared__ __align__(16) uint8_t lds[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile_m = blockIdx.x % g.tiles_m, tile_n = blockIdx.x / g.tiles_m;
  const int m0 = tile_m * 32 * TM, n0 = tile_n * 64;
  uint8_t* ring = lds + wave * kRing;

  // load instruction p fills rows 8p + lane/8 of an operand tile; the lane fetches the logical chunk that belongs at
  // its (swizzled) position
  const uint8_t* a_src[PA];
  const uint8_t* b_src[PB];
#pragma unroll
  for (int p = 0; p < PA; ++p) {
    const int rl = p * 8 + (lane >> 3), row = min(m0 + rl, g.M - 1);      // clamp: tail rows and columns are never stored
    a_src[p] = g.a + ((int64_t)row * g.K + swizzle<64>(rl, lane & 7) * 8) * 2;
  }
#pragma unroll
  for (int p = 0; p < PB; ++p) {
    const int rl = p * 8 + (lane >> 3);
    int col = min(n0 + rl, g.N - 1);
    const uint8_t* base = g.b0;
    if constexpr (EPI == kEpiPlain || EPI == kEpiStats) {
      if (g.b1 && col >= g.N / 2) { base = g.b1; col -= g.N / 2; }
    }
    b_src[p] = base + ((int64_t)col * g.K + swizzle<64>(rl, lane & 7) * 8) * 2;
  }
  auto issue_tile = [&](int kt, int stage) __attribute__((always_inline)) {
    uint8_t* st = ring + stage * kStage;
    const int koff = kt * kRow;
#pragma unroll
    for (int p = 0; p < PA; ++p)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a_src[p] + koff),
                                       (__attribute__((address_space(3))) void*)(st + p * 1024), 16, 0, 0);
#pragma unroll
    for (int p = 0; p < PB; ++p)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(b_src[p] + koff),
                                       (__attribute__((address_space(3))) void*)(st + kATile + p * 1024), 16, 0, 0);
  };

  // fragment reads: lane reads row lane%32 (+32 i), logical chunk 2*slab + lane/32
  const int rl = lane & 31;
  int off_slab[4];
#pragma unroll
  for (int sl = 0; sl < 4; ++sl) off_slab[sl] = rl * kRow + swizzle<64>(rl, 2 * sl + (lane >> 5)) * 16;

  f32x16_t acc[TM][2];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;

  const int num_kt = g.K / 64;
  const int mine = (num_kt - wave + 3) / 4;             // K tiles wave, wave + 4, ...
#pragma unroll
  for (int t = 0; t < NS; ++t)
    if (mine > t) issue_tile(wave + 4 * t, t);
  int stage = 0;
  for (int t = 0; t < mine; ++t) {
    // this tile has landed; the next ones may be in flight
    const int younger = min(mine - 1 - t, NS - 1);
    if (NS > 2 && younger > 1) wait_vmcnt<2 * (PA + PB)>();
    else if (younger > 0) wait_vmcnt<PA + PB>();
    else wait_vmcnt<0>();
    const uint8_t* st = ring + stage * kStage;
    u32x4_t af[2][TM], bf[2][2];
    auto read_slab = [&](int sl) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < TM; ++i) af[sl & 1][i] = *(const u32x4_t*)(st + off_slab[sl] + i * 32 * kRow);
#pragma unroll
      for (int j = 0; j < 2; ++j) bf[sl & 1][j] = *(const u32x4_t*)(st + kATile + off_slab[sl] + j * 32 * kRow);
    };
    read_slab(0);
#pragma unroll
    for (int sl = 0; sl < 4; ++sl) {
      if (sl + 1 < 4) read_slab(sl + 1);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma32<DT>(bf[sl & 1][j], af[sl & 1][i], acc[i][j]);
    }
    if (t + NS < mine) {
      wait_lds_reads();                                  // the stage is read out (by this wave, its only reader)
      issue_tile(wave + 4 * (t + NS), stage);
    }
    stage = stage + 1 == NS ? 0 : stage + 1;
  }

  // ---- the four partial tiles meet in LDS: [wave][MFMA tile][column group][lane] 16 bytes each
  __syncthreads();                                       // every wave is done with its ring
  f32x4_t* xch = (f32x4_t*)lds;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        xch[((wave * 2 * TM + (j * TM + i)) * 4 + q4) * 64 + lane] =
            f32x4_t{acc[i][j][q4 * 4], acc[i][j][q4 * 4 + 1], acc[i][j][q4 * 4 + 2], acc[i][j][q4 * 4 + 3]};
  __syncthreads();
  if (wave >= 2 * TM) return;
  f32x16_t sum[1][1];
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4) {
    f32x4_t v = xch[(wave * 4 + q4) * 64 + lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      const f32x4_t o = xch[((w * 2 * TM + wave) * 4 + q4) * 64 + lane];
      v[0] += o[0]; v[1] += o[1]; v[2] += o[2]; v[3] += o[3];
    }
    sum[0][0][q4 * 4] = v[0]; sum[0][0][q4 * 4 + 1] = v[1]; sum[0][0][q4 * 4 + 2] = v[2]; sum[0][0][q4 * 4 + 3] = v[3];
  }
  gemm_epilogue<DT, 1, 1, EPI>(g, sum, m0, n0, wave % TM, wave / TM, lane);
}

// ---- single precision with few output tiles -----------------------------------------------------------
// What bounds it: v_mfma_f32_32x32x2 takes 64 cycles, so a CU that has a 128 x 128 tile to itself works 4096 cycles on 32 of K, and a launch
// of 32 or 64 such tiles leaves the chip idle (512 tokens, hidden 256 x intermediate 1024: gate/up 22.4 us, down projection 26.8 us on 64 x 64
// tiles, for 4 and 2 us of matrix instructions).  Here a block has 32 x 32 of the output (SwiGLU: of gate and of up) and its four waves deal
// out the K tiles (32 values, 128-byte rows) as in gemm_ksplit_kernel: a ring in LDS per wave, no block barrier, the four sums added in
// wave order: 12.4 and 9.1 us.  Twice the operand traffic of a 64 x 64 tile (32 bytes per cycle and CU), which L2 still carries.
// NS: ring stages.  A K tile's fragments are all read before its matrix instructions, so one stage still has the next tile's loads in flight during them; two
// start a block faster but take 96 KiB (SwiGLU; else 64), one block to a CU: one where the launch has more blocks than fit the CUs that way
// (the layer at 512 x 256 x 1024 29.8 -> 25.9 us, 1000 x 256 x 1024 43.3 -> 38.2, 300 x 1024 x 4096 116 -> 106; the MLP at 512 x 256 x 1024 17.8 -> 16.0).
template <int EPI, int NS>
__device__ __forceinline__ void gemm_f32_small_block(const GemmArgs& g, const int block, uint8_t* lds) {
  constexpr int TB = EPI == kEpiSwiglu ? 2 : 1, kTile = 32 * 128, kStage = (1 + TB) * kTile, kLoads = 4 * (1 + TB);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = block % g.tiles_m * 32, n0 = block / g.tiles_m * 32;
  const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds + (uint32_t)wave * NS * kStage;
  const int row_bytes = g.K * 4;
  const uint64_t a = (uint64_t)g.a + (uint64_t)m0 * (uint32_t)row_bytes;
  const int a_bytes = min(32, g.M - m0) * row_bytes, b_bytes = min(32, g.N - n0) * row_bytes;    // rows past the matrix read as zero
  // a second matrix: the up weights, or the upper half of the columns (whole blocks of it)
  uint64_t b[2] = {(uint64_t)g.b0 + (uint64_t)n0 * (uint32_t)row_bytes, 0};
  if constexpr (EPI == kEpiSwiglu) b[1] = (uint64_t)g.b1 + (uint64_t)n0 * (uint32_t)row_bytes;
  else if (g.b1 && n0 >= g.N / 2) b[0] = (uint64_t)g.b1 + (uint64_t)(n0 - g.N / 2) * (uint32_t)row_bytes;
  auto issue = [&](int kt, int stage) __attribute__((always_inline)) {
    auto one = [&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value, operand = n / 4, part = n % 4;
      const int row = part * 8 + (lane >> 3), k = kt * 32 + swizzle<64>(row, lane & 7) * 4;      // position c of a row holds its piece swizzle(c)
      load_to_lds<n * 1024>(operand == 0 ? a : b[operand == 2], operand == 0 ? a_bytes : b_bytes, ring + (uint32_t)(stage * kStage),
                            k < g.K ? (uint32_t)(row * row_bytes + k * 4) : 0x80000000u, 0);
    };
    auto all = [&](auto... n) __attribute__((always_inline)) { (one(n), ...); };
    with_sequence(all, std::make_integer_sequence<int, kLoads>{});
  };
  f32x16_t acc[TB];
#pragma unroll
  for (int j = 0; j < TB; ++j)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[j][q] = 0.f;

  const int rl = lane & 31, num_kt = (g.K + 31) / 32, mine = (num_kt - wave + 3) / 4;
  if (mine > 0) issue(wave, 0);
  if (NS == 2 && mine > 1) issue(wave + 4, 1);
  for (int t = 0; t < mine; ++t) {
    if (NS == 2 && t + 1 < mine) wait_vmcnt<kLoads>(); else wait_vmcnt<0>();
    const uint32_t st = ring + (uint32_t)(t % NS * kStage + rl * 128);
    using Frag = const __attribute__((address_space(3))) u32x4_t*;
    u32x4_t af[4], bf[4][TB];
#pragma unroll
    for (int sl = 0; sl < 4; ++sl) {
      const uint32_t at = st + (uint32_t)swizzle<64>(rl, 2 * sl + (lane >> 5)) * 16;
      af[sl] = *(Frag)(uintptr_t)at;
#pragma unroll
      for (int j = 0; j < TB; ++j) bf[sl][j] = *(Frag)(uintptr_t)(at + (1 + j) * kTile);
    }
    if (t + NS < mine) {
      wait_lds_reads();                                  // the stage is read out (by this wave, its only reader)
      issue(wave + 4 * (t + NS), t % NS);
    }
#pragma unroll
    for (int sl = 0; sl < 4; ++sl)
#pragma unroll
      for (int j = 0; j < TB; ++j) acc[j] = mfma32<kF32>(bf[sl][j], af[sl], acc[j]);
  }

  __syncthreads();                                       // every wave is done with its ring
  f32x4_t* xch = (f32x4_t*)lds;
#pragma unroll
  for (int j = 0; j < TB; ++j)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4)
      xch[((wave * TB + j) * 4 + q4) * 64 + lane] = f32x4_t{acc[j][q4 * 4], acc[j][q4 * 4 + 1], acc[j][q4 * 4 + 2], acc[j][q4 * 4 + 3]};
  __syncthreads();
  if (wave != 0) return;
  f32x16_t sum[1][TB];
#pragma unroll
  for (int j = 0; j < TB; ++j)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      f32x4_t v = xch[(j * 4 + q4) * 64 + lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) {
        const f32x4_t o = xch[((w * TB + j) * 4 + q4) * 64 + lane];
        v[0] += o[0]; v[1] += o[1]; v[2] += o[2]; v[3] += o[3];
      }
      sum[0][j][q4 * 4] = v[0]; sum[0][j][q4 * 4 + 1] = v[1]; sum[0][j][q4 * 4 + 2] = v[2]; sum[0][j][q4 * 4 + 3] = v[3];
    }
  gemm_epilogue<kF32, 1, TB, EPI>(g, sum, m0, n0, 0, 0, lane);
}
template <int EPI, int NS>
__global__ __launch_bounds__(kGemmThreads, 1) void gemm_f32_small_kernel(const GemmArgs g) {
  extern __shared__ __align__(16) uint8_t lds[];
  gemm_f32_small_block<EPI, NS>(g, (int)blockIdx.x, lds);
}

// A layer of such products in single precision: stages that do not depend on each other share a launch, as in 16 bits (gemm_tiles.hip).  Six dependent launches
// of 4 to 12 us are three: projection | gate/up (the projection's blocks first: half as long), then selection | down projection; the third gathers the experts and adds (expert.hip).
struct F32Front { GemmArgs router, mlp; int router_blocks; };
template <int EPI, int NS>            // of the projection: kEpiStats or kEpiPlain
__global__ __launch_bounds__(kGemmThreads, 1) void gemm_f32_front_kernel(const F32Front g) {
  extern __shared__ __align__(16) uint8_t lds[];
  if ((int)blockIdx.x < g.router_blocks) gemm_f32_small_block<EPI, NS>(g.router, (int)blockIdx.x, lds);
  else gemm_f32_small_block<kEpiSwiglu, NS>(g.mlp, (int)blockIdx.x - g.router_blocks, lds);
}
struct F32Down { GemmArgs down; SelectArgs select; int select_blocks; };
template <int R, int C>
__global__ __launch_bounds__(kGemmThreads, 1) void gemm_f32_select_kernel(const F32Down g) {
  extern __shared__ __align__(16) uint8_t lds[];
  if ((int)blockIdx.x >= g.select_blocks) {
    gemm_f32_small_block<kEpiPlain, 2>(g.down, (int)blockIdx.x - g.select_blocks, lds);
    return;
  }
  const float* stats = g.select.stats;
  if (g.select.part_mean) {                                    // batch statistics: the block merges them first
    merge_statistics(g.select, (float*)lds, kGemmThreads);
    count_batch(g.select);
    stats = (const float*)lds;
  }
  constexpr int kWaves = kGemmThreads / kWave;
  select_pairs<R, C>(g.select, (int)blockIdx.x * kWaves + (int)(threadIdx.x >> 6), g.select_blocks * kWaves, stats);
}

// One list entry per kernel instantiation that launch_gemm can start (the static members come into being
// at library load for every instantiation the dispatch below names).
template <int DT, int TM, int TN, int EPI, int BK, int NS, int NW = 4>
struct DmaKernelLds {
  static inline LdsKernel entry{(const void*)gemm_nt_dma_kernel<DT, TM, TN, EPI, BK, NS, NW>, NS * (2 * TM * 32 + (NW / 2) * TN * 32) * BK * 2};
};
template <int DT, int EPI, int TM>
struct KsplitKernelLds {
  static inline LdsKernel entry{(const void*)gemm_ksplit_kernel<DT, EPI, TM>, ksplit_lds(TM)};
};
template <int EPI, int NS>
struct SmallF32Lds {
  static constexpr int kBytes = 4 * NS * (EPI == kEpiSwiglu ? 3 : 2) * 32 * 128;
  static inline LdsKernel entry{(const void*)gemm_f32_small_kernel<EPI, NS>, kBytes};
};
template <auto kKernel, int kBytes>
struct F32JointLds { static inline LdsKernel entry{(const void*)kKernel, kBytes}; };
template <int DT, int TM, int TN, int EPI>
struct StagedKernelLds {
  static inline LdsKernel entry{(const void*)gemm_nt_kernel<DT, TM, TN, EPI>, 2 * (2 * TM * 32 + 2 * TN * 32) * kRowBytes};
};

// Blocks of gemm_f32_small_kernel where that takes fewer cycles than TM x TN tiles, else 0.
// Cycles of matrix instructions and of what goes round them, per round of 256 blocks: a TM x TN wave tile takes 1024 TM TN for 32 of K, plus
// about 900 with one block to a CU and 450 with more (64 x 64 tiles 1700 and 1490, 128 x 128 tiles 5400); a block of 32 x 32 deals the same K out
// over four waves.  1000 x 1024 x 4096: 106 us on 64 x 64 tiles, 88 us here; 2500 x 768 x 2304: 97 and 102 us.
template <int TM, int TN, int EPI>
static int64_t f32_small_blocks(GemmArgs& g) {
  constexpr int BM = 2 * TM * 32, BN = EPI == kEpiSwiglu ? TN * 32 : 2 * TN * 32, TB = EPI == kEpiSwiglu ? 2 : 1;
  const int64_t blocks = (int64_t)((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
  const int64_t kt = (g.K + 31) / 32, tiles_m = (g.M + 31) / 32, small = tiles_m * ((g.N + 31) / 32);
  const int64_t tiled = (blocks + 255) / 256 * kt * (1024 * TM * TN + (blocks > 256 ? 450 : 900)), dealt = (small + 255) / 256 * ((kt + 3) / 4 * (1024 * TB + 450) + 2500);
  if (dealt >= tiled || small >= INT32_MAX / 4 || (int64_t)g.K * 128 >= INT32_MAX || (EPI != kEpiSwiglu && g.b1 && g.N % 64 != 0)) return 0;
  g.tiles_m = (int)tiles_m;
  g.tiles_n = (g.N + 31) / 32;
  return small;
}
template <int EPI>
static int64_t f32_small_blocks_of(GemmArgs& g) {              // ... against the tiles that gemm_plain and gemm_swiglu choose
  g.single = g.N % 4 != 0;
  if (EPI == kEpiSwiglu) return f32_small_blocks<2, 2, EPI>(g);
  const int64_t big = (int64_t)((g.M + 255) / 256) * ((g.N + 255) / 256), mid = (int64_t)((g.M + 127) / 128) * ((g.N + 127) / 128);
  return big >= 200 ? f32_small_blocks<4, 4, EPI>(g) : mid >= 200 ? f32_small_blocks<2, 2, EPI>(g) : f32_small_blocks<1, 1, EPI>(g);
}

template <int DT, int TM, int TN, int EPI>
static hipError_t launch_gemm(GemmArgs g, hipStream_t s, bool exclusive = false) {
  constexpr int BM = 2 * TM * 32, BR = 2 * TN * 32, BN = (EPI == kEpiSwiglu) ? BR / 2 : BR;
  constexpr int kLds = 2 * (BM + BR) * kRowBytes;
  g.tiles_m = (g.M + BM - 1) / BM;
  g.tiles_n = (g.N + BN - 1) / BN;
  const int blocks = g.tiles_m * g.tiles_n;
  // one XCD runs 32 blocks at a time: give it 4 x 8 patches when the tile grid allows
  g.patch_m = g.patch_n = 0;
  g.wide = (DT != kF32) && g.N % 8 == 0 && ((uintptr_t)g.c % 16 == 0);
  g.single = g.N % 4 != 0;
  if (EPI == kEpiGate && !(g.wide && (uintptr_t)g.gate % 16 == 0)) return hipErrorInvalidValue;   // the gate epilogue has the 16-byte form only
  if (blocks % 256 == 0) {
    if (g.tiles_m % 4 == 0 && g.tiles_n % 8 == 0) { g.patch_m = 4; g.patch_n = 8; }
    else if (g.tiles_m % 8 == 0 && g.tiles_n % 4 == 0) { g.patch_m = 8; g.patch_n = 4; }
  }
  // Loads straight to LDS take 16-byte pieces from 16-byte boundaries; operands that begin anywhere else (views into a flat buffer) are staged
  // through registers.
  const bool aligned = ((uintptr_t)g.a | (uintptr_t)g.b0 | (uintptr_t)g.b1) % 16 == 0;
  // 128-byte LDS rows (64-byte rows halve the fetch rate); as many ring stages as 160 KiB hold, up to 4
  constexpr int kDmaBK = 64;
  constexpr int kFit = (160 * 1024) / ((BM + BR) * kDmaBK * 2);
  constexpr int kDmaStages = kFit > 4 ? 4 : kFit;
  if constexpr (DT != kF32 && EPI != kEpiSwiglu) if (g.K % kDmaBK == 0 && aligned) {
    constexpr int kDmaLds = kDmaStages * (BM + BR) * kDmaBK * 2;
    static_assert(kDmaLds <= 160 * 1024, "LDS ring exceeds 160 KiB");
    if constexpr (TM == 1 && TN == 1 && EPI != kEpiGate) {
      // fewer 64 x 64 tiles than CUs and at least two K tiles per wave: the K tiles dealt out over the waves
      if (blocks <= 256 && g.K >= 512) {
        const int tiles32 = (g.M + 31) / 32, blocks32 = tiles32 * g.tiles_n;
        if (exclusive && blocks32 <= 256) {
          g.tiles_m = tiles32;
          if (hipError_t e = KsplitKernelLds<DT, EPI, 1>::entry.ensure(); e != hipSuccess) return e;
          hipLaunchKernelGGL((gemm_ksplit_kernel<DT, EPI, 1>), dim3(blocks32), dim3(kGemmThreads), ksplit_lds(1), s, g);
          return hipGetLastError();
        }
        if (hipError_t e = KsplitKernelLds<DT, EPI, 2>::entry.ensure(); e != hipSuccess) return e;
        hipLaunchKernelGGL((gemm_ksplit_kernel<DT, EPI, 2>), dim3(blocks), dim3(kGemmThreads), ksplit_lds(2), s, g);
        return hipGetLastError();
      }
    }
    if constexpr (TM == 4 && TN == 4) {
      // the 256 x 256 block tile on 8 waves of 128 x 64, two per SIMD: one wave's barrier and load waits are the other's
      // issue slots (66.7 against 69.1 us for the 4096-token gate/up projection when that ran here), at 6 fragment reads per 8 MFMAs
      auto kern8 = gemm_nt_dma_kernel<DT, 4, 2, EPI, kDmaBK, kDmaStages, 8>;
      if (hipError_t e = DmaKernelLds<DT, 4, 2, EPI, kDmaBK, kDmaStages, 8>::entry.ensure(); e != hipSuccess) return e;
      hipLaunchKernelGGL(kern8, dim3(blocks), dim3(512), kDmaLds, s, g);
      return hipGetLastError();
    } else {
      auto kern = gemm_nt_dma_kernel<DT, TM, TN, EPI, kDmaBK, kDmaStages>;
      static_assert(kDmaLds == kDmaStages * (2 * TM * 32 + 2 * TN * 32) * kDmaBK * 2, "list entry and launch disagree");
      if (hipError_t e = DmaKernelLds<DT, TM, TN, EPI, kDmaBK, kDmaStages>::entry.ensure(); e != hipSuccess) return e;
      hipLaunchKernelGGL(kern, dim3(blocks), dim3(kGemmThreads), kDmaLds, s, g);
      return hipGetLastError();
    }
  }
  if constexpr (DT == kF32 && EPI != kEpiGate) {
    GemmArgs d = g;
    if (const int64_t small = f32_small_blocks<TM, TN, EPI>(d); small && aligned) {
      auto go = [&](auto ns) -> hipError_t {
        constexpr int NS = decltype(ns)::value;
        using L = SmallF32Lds<EPI, NS>;
        if (hipError_t e = L::entry.ensure(); e != hipSuccess) return e;
        hipLaunchKernelGGL((gemm_f32_small_kernel<EPI, NS>), dim3((unsigned)small), dim3(kGemmThreads), L::kBytes, s, d);
        return hipGetLastError();
      };
      if (small > (EPI == kEpiSwiglu ? 256 : 512)) return go(std::integral_constant<int, 1>{});
      return go(std::integral_constant<int, 2>{});
    }
  }
  auto kern = gemm_nt_kernel<DT, TM, TN, EPI>;       // any K % 8 == 0, any address: staged through registers
  if (hipError_t e = StagedKernelLds<DT, TM, TN, EPI>::entry.ensure(); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kGemmThreads), kLds, s, g);
  return hipGetLastError();
}

// Shape rule shared by the entry points: K a multiple of a 16-byte chunk (rows are fetched 16 bytes at a time).
static int check_gemm(int64_t M, int64_t N, int64_t K, int elem_bytes) {
  if (M < 0 || N <= 0 || K <= 0 || M > INT32_MAX / 2 || N > INT32_MAX / 2 || K > INT32_MAX / 2) return OMNI_ERR_SHAPE;
  if (K % (16 / elem_bytes) != 0) return OMNI_ERR_SHAPE;
  return OMNI_OK;
}

static int to_code(hipError_t e) { return e == hipSuccess ? OMNI_OK : OMNI_ERR_HIP_BASE + (int)e; }

// The tile GEMM's terms: columns in eights, 16-byte aligned pointers.  *e is then what its launch returned.
static bool tile_gemm(int dtype, int epilogue, const void* a, const void* b, const void* b2, const void* res, void* c, void* keep_gate, void* keep_up, int64_t M, int64_t N,
                      int64_t K, void* ws, size_t ws_bytes, bool exclusive, hipStream_t s, hipError_t* e) {
  if (dtype == OMNI_F32 || N % 8 != 0) return false;
  for (const void* q : {a, b, b2, res, (const void*)c, (const void*)keep_gate, (const void*)keep_up})
    if ((uintptr_t)q % 16) return false;
  TileGroup g;
  TileProduct& p = g.p[g.count++];
  p.seg[p.segments++] = TileSegment{(const uint8_t*)a, (const uint8_t*)b, K * 2, K * 2, 0, (int)K};
  p.M = (int)M; p.N = (int)N; p.ldc = N * 2; p.c = (uint8_t*)c; p.res = (const uint8_t*)res; p.b_up = (const uint8_t*)b2;
  p.c2 = (uint8_t*)keep_gate; p.c3 = (uint8_t*)keep_up;
  *e = launch_tile_group(dtype, kNT, epilogue, g, ws, ws_bytes, s, exclusive);
  return *e != hipErrorInvalidValue;
}

// C[M,N] = A[M,K] B[N,K]^T (+ res), picking the tile shape from the problem size.  ws: room for a K split (or NULL)
template <int DT>
static int gemm_plain(const void* a, const void* b, const void* b_hi, const void* res, void* c, int64_t M, int64_t N, int64_t K, hipStream_t s,
                      float* part_mean = nullptr, float* part_m2 = nullptr, bool twin = true, bool exclusive = true, void* ws = nullptr, size_t ws_bytes = 0) {
  if (int e = check_gemm(M, N, K, ElemBytes<DT>::value)) return e;
  if (M == 0) return OMNI_OK;
  hipError_t err;
  const int64_t big = ((M + 255) / 256) * ((N + 255) / 256), mid = ((M + 127) / 128) * ((N + 127) / 128);
  // a second weight matrix starts at a multiple of 8 columns there; `twin`: the result is, bit for bit, what two matrices give
  if (!part_mean && (N % 16 == 0 || !twin) &&
      tile_gemm(DT, b_hi ? kTileTwo : res ? kTileResidual : kTilePlain, a, b, b_hi, res, c, nullptr, nullptr, M, N, K, ws, ws_bytes, exclusive, s, &err))
    return to_code(err);
  GemmArgs g{(const uint8_t*)a, (const uint8_t*)b, (const uint8_t*)b_hi, (const uint8_t*)res, (uint8_t*)c, (int)M, (int)N, (int)K, 0, 0, 0, 0, 0, 0, nullptr, nullptr, nullptr};
  g.part_mean = part_mean;
  g.part_m2 = part_m2;
  if (res) {
    if (mid >= 200) err = launch_gemm<DT, 2, 2, kEpiResidual>(g, s);
    else err = launch_gemm<DT, 1, 1, kEpiResidual>(g, s);
  } else if (part_mean) {
    if (big >= 200) err = launch_gemm<DT, 4, 4, kEpiStats>(g, s);
    else if (mid >= 200) err = launch_gemm<DT, 2, 2, kEpiStats>(g, s);
    else err = launch_gemm<DT, 1, 1, kEpiStats>(g, s, exclusive);
  } else {
    if (big >= 200) err = launch_gemm<DT, 4, 4, kEpiPlain>(g, s);
    else if (mid >= 200) err = launch_gemm<DT, 2, 2, kEpiPlain>(g, s);
    else err = launch_gemm<DT, 1, 1, kEpiPlain>(g, s);
  }
  return to_code(err);
}

template <int DT>
static int gemm_swiglu(const void* x, const void* wg, const void* wu, void* h, int64_t M, int64_t I, int64_t K, hipStream_t s,
                       void* save_gate = nullptr, void* save_up = nullptr, bool exclusive = true, void* ws = nullptr, size_t ws_bytes = 0) {
  if (int e = check_gemm(M, I, K, ElemBytes<DT>::value)) return e;
  if (M == 0) return OMNI_OK;
  hipError_t err;
  if (save_gate && (DT == kF32 || I % 8 || ((uintptr_t)h | (uintptr_t)save_gate | (uintptr_t)save_up) % 16)) return OMNI_ERR_UNSUPPORTED;
  const bool tiles = tile_gemm(DT, kTileSwiglu, x, wg, wu, nullptr, h, save_gate, save_up, M, I, K, ws, ws_bytes, exclusive, s, &err);
  if (tiles && (err != hipSuccess || !save_gate || K % 64 == 0)) return to_code(err);
  if (save_gate) {
    // Operands at any other address, or out of the tile GEMM's reach: the two projections by themselves.
    if (!tiles) {
      if (int e = gemm_plain<DT>(x, wg, nullptr, nullptr, save_gate, M, I, K, s)) return e;
      if (int e = gemm_plain<DT>(x, wu, nullptr, nullptr, save_up, M, I, K, s)) return e;
    }
    // Here, and for hidden sizes that are no multiple of 64, the product is the element-wise operator's, which divides: the epilogue's hardware reciprocal is
    // 1 ulp, enough that one in 70 000 products falls on the other side of an f16 rounding, and a differentiable forward of such sizes has always divided.
    // (Dividing in the epilogue instead costs every size: gate/up with the layer around it at 4096 tokens 132 -> 137 us, the MLP at 1024 x 1024 x 16384
    // 108 -> 115 us.)
    return omni_swiglu_fwd(save_gate, save_up, h, M * I, DT, s);
  }
  GemmArgs g{(const uint8_t*)x, (const uint8_t*)wg, (const uint8_t*)wu, nullptr, (uint8_t*)h, (int)M, (int)I, (int)K, 0, 0, 0, 0, 0, 0, nullptr, nullptr, nullptr};
  return to_code(launch_gemm<DT, 2, 2, kEpiSwiglu>(g, s));
}

}  // namespace omni

// c[T, 2N] = [round(v) | round(v - round(v))] with v = silu(x W^T) * gate, gate [T, N] fp32 (16-bit storage types only)
int omni_gemm_gated(const void* x, const void* w, const float* gate, void* c, int64_t T, int64_t N, int64_t K, int dtype, void* stream) {
  using namespace omni;
  if (dtype != OMNI_BF16 && dtype != OMNI_F16) return OMNI_ERR_UNSUPPORTED;
  if (int e = check_gemm(T, N, K, 2)) return e;
  if (T == 0) return OMNI_OK;
  GemmArgs g{(const uint8_t*)x, (const uint8_t*)w, nullptr, nullptr, (uint8_t*)c, (int)T, (int)N, (int)K, 0, 0, 0, 0, 0, 0, nullptr, nullptr, gate};
  hipStream_t s = (hipStream_t)stream;
  const int64_t big = ((T + 255) / 256) * ((N + 255) / 256), mid = ((T + 127) / 128) * ((N + 127) / 128);
  hipError_t err;
  if (dtype == OMNI_BF16) {
    if (big >= 200) err = launch_gemm<kBF16, 4, 4, kEpiGate>(g, s);
    else if (mid >= 200) err = launch_gemm<kBF16, 2, 2, kEpiGate>(g, s);
    else err = launch_gemm<kBF16, 1, 1, kEpiGate>(g, s);
  } else {
    if (big >= 200) err = launch_gemm<kF16, 4, 4, kEpiGate>(g, s);
    else if (mid >= 200) err = launch_gemm<kF16, 2, 2, kEpiGate>(g, s);
    else err = launch_gemm<kF16, 1, 1, kEpiGate>(g, s);
  }
  return to_code(err);
}

int omni_gemm_router_projection(const void* x, const void* wx, const void* wy, void* z, float* part_mean, float* part_m2,
                                int64_t T, int H, int r, int dtype, void* stream, bool exclusive) {
  using namespace omni;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == OMNI_BF16) return gemm_plain<kBF16>(x, wx, wy, nullptr, z, T, 2 * (int64_t)r, H, s, part_mean, part_m2, true, exclusive || !part_mean);
  if (dtype == OMNI_F16) return gemm_plain<kF16>(x, wx, wy, nullptr, z, T, 2 * (int64_t)r, H, s, part_mean, part_m2, true, exclusive || !part_mean);
  if (dtype == OMNI_F32) return gemm_plain<kF32>(x, wx, wy, nullptr, z, T, 2 * (int64_t)r, H, s, part_mean, part_m2);
  return OMNI_ERR_DTYPE;
}

namespace omni {
// Whether the three products of a single-precision layer are all of gemm_f32_small_kernel's kind and the selection fits beside them: from the sizes alone
bool f32_joint_covers(int64_t T, int64_t H, int64_t I, int r, int k) {
  if (check_gemm(T, I, H, 4) || check_gemm(T, H, I, 4) || check_gemm(T, 2 * (int64_t)r, H, 4) || r % 32) return false;       // (r: the halves' weights meet at a tile's border)
  GemmArgs router{}, mlp{}, down{};
  router.M = mlp.M = down.M = (int)T;
  router.N = 2 * r; router.K = mlp.K = (int)H; mlp.N = down.K = (int)I; down.N = (int)H;
  return r <= 4 * kWave && num_cells(k, r < k ? r : k) <= 2 * kWave && f32_small_blocks_of<kEpiPlain>(router) && f32_small_blocks_of<kEpiSwiglu>(mlp) &&
         f32_small_blocks_of<kEpiPlain>(down);
}
// The layer's projection, gate/up, selection and down projection in single precision as two launches (see gemm_f32_front_kernel), y then holding the shared MLP's
// rows: sizes that f32_joint_covers takes, operands 16-byte aligned.
hipError_t launch_f32_joint(const void* x, const void* wx, const void* wy, void* z, const void* wg, const void* wu, const void* wd, void* h, void* y, int64_t T, int64_t H, int64_t I,
                            const SelectArgs& args, bool statistics, hipStream_t s) {
  GemmArgs router{}, mlp{}, down{};
  router.a = mlp.a = (const uint8_t*)x;
  router.b0 = (const uint8_t*)wx; router.b1 = (const uint8_t*)wy; router.c = (uint8_t*)z;
  mlp.b0 = (const uint8_t*)wg; mlp.b1 = (const uint8_t*)wu; mlp.c = (uint8_t*)h;
  down.a = (const uint8_t*)h; down.b0 = (const uint8_t*)wd; down.c = (uint8_t*)y;
  router.M = mlp.M = down.M = (int)T;
  router.N = 2 * args.r; router.K = mlp.K = (int)H; mlp.N = down.K = (int)I; down.N = (int)H;
  if (statistics) { router.part_mean = (float*)args.part_mean; router.part_m2 = (float*)args.part_m2; }
  F32Down d{down, args, 0};
  const int cells = prepare_select(d.select), regs = (args.r + kWave - 1) / kWave;
  const int64_t rb = f32_small_blocks_of<kEpiPlain>(router), mb = f32_small_blocks_of<kEpiSwiglu>(mlp), db = f32_small_blocks_of<kEpiPlain>(d.down);
  if (!rb || !mb || !db || regs > 4 || cells > 2) return hipErrorInvalidValue;
  hipError_t e = hipSuccess;
  const F32Front f{router, mlp, (int)rb};
  constexpr int kDown = SmallF32Lds<kEpiPlain, 2>::kBytes;
  static_assert(kDown >= 4 * merge_lds_floats(kMergeKeys, kGemmThreads), "a block that selects merges statistics there");
  static_assert(kGemmThreads == kF32MergeThreads, "the order of its sums is also the two-stream schedule's");
  auto start = [&](auto kernel, LdsKernel& entry, int bytes, int64_t blocks, const auto& a) {
    if ((e = entry.ensure()) != hipSuccess) return;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kGemmThreads), bytes, s, a);
    e = hipGetLastError();
  };
  auto front = [&](auto ns) {
    constexpr int NS = decltype(ns)::value, kFront = SmallF32Lds<kEpiSwiglu, NS>::kBytes;
    if (statistics) start(gemm_f32_front_kernel<kEpiStats, NS>, F32JointLds<gemm_f32_front_kernel<kEpiStats, NS>, kFront>::entry, kFront, rb + mb, f);
    else start(gemm_f32_front_kernel<kEpiPlain, NS>, F32JointLds<gemm_f32_front_kernel<kEpiPlain, NS>, kFront>::entry, kFront, rb + mb, f);
  };
  if (rb + mb > 256) front(std::integral_constant<int, 1>{});
  else front(std::integral_constant<int, 2>{});
  if (e != hipSuccess) return e;
  constexpr int kWaves = kGemmThreads / kWave;
  d.select_blocks = (int)((T + kWaves - 1) / kWaves < 1024 ? (T + kWaves - 1) / kWaves : 1024);
  auto by_cells = [&](auto r_tag) {
    constexpr int R = decltype(r_tag)::value;
    if (cells <= 1) start(gemm_f32_select_kernel<R, 1>, F32JointLds<gemm_f32_select_kernel<R, 1>, kDown>::entry, kDown, d.select_blocks + db, d);
    else start(gemm_f32_select_kernel<R, 2>, F32JointLds<gemm_f32_select_kernel<R, 2>, kDown>::entry, kDown, d.select_blocks + db, d);
  };
  if (regs <= 1) by_cells(std::integral_constant<int, 1>{});
  else if (regs <= 2) by_cells(std::integral_constant<int, 2>{});
  else by_cells(std::integral_constant<int, 4>{});
  return e;
}
}  // namespace omni

namespace omni {
// partial sums of whichever of the two projections is split along K (they are not alive together)
size_t mlp_sums_bytes(int64_t T, int64_t H, int64_t I, int dtype) {
  if (dtype == OMNI_F32 || I % 8 || H % 8) return 0;
  const size_t few = few_tokens_covers(T, H, I, dtype) ? few_tokens_parts_bytes(T, H, I) : 0;
  return std::max({few, tile_workspace_bytes(kNT, kTileSwiglu, T, I, H), tile_workspace_bytes(kNT, kTileResidual, T, H, I), tile_down_workspace_bytes(T, H, I)});
}
static size_t mlp_h_bytes(int64_t T, int64_t I, int dtype) { return ((size_t)T * (size_t)I * (dtype == OMNI_F32 ? 4 : 2) + 255) / 256 * 256; }

// The two projections of omni_mlp_fwd, each told whether it has the GPU to itself (the whole-layer call on two streams says no, which keeps
// them off the form that holds every CU to the end).  sums: mlp_sums_bytes(); gate, up: NULL, or where the rounded projections go as well (16-bit types).
int mlp_gate_up_impl(const void* x, const void* wg, const void* wu, void* h, void* gate, void* up, int64_t T, int32_t H, int32_t I, int32_t dtype, void* sums, void* stream,
                     bool exclusive) {
  if (!x || !wg || !wu) return OMNI_ERR_NULL;
  hipStream_t s = (hipStream_t)stream;
  const size_t n = mlp_sums_bytes(T, H, I, dtype);
  switch (dtype) {
    case OMNI_BF16: return gemm_swiglu<kBF16>(x, wg, wu, h, T, I, H, s, gate, up, exclusive, sums, n);
    case OMNI_F16: return gemm_swiglu<kF16>(x, wg, wu, h, T, I, H, s, gate, up, exclusive, sums, n);
    case OMNI_F32: return gemm_swiglu<kF32>(x, wg, wu, h, T, I, H, s, gate, up, exclusive, sums, n);
    default: return OMNI_ERR_DTYPE;
  }
}
int mlp_down_impl(const void* h, const void* wd, const void* residual, void* y, int64_t T, int32_t H, int32_t I, int32_t dtype, void* sums, void* stream, bool exclusive) {
  if (!wd || !y) return OMNI_ERR_NULL;
  hipStream_t s = (hipStream_t)stream;
  const size_t n = mlp_sums_bytes(T, H, I, dtype);
  switch (dtype) {
    case OMNI_BF16: return gemm_plain<kBF16>(h, wd, nullptr, residual, y, T, H, I, s, nullptr, nullptr, false, exclusive, sums, n);
    case OMNI_F16: return gemm_plain<kF16>(h, wd, nullptr, residual, y, T, H, I, s, nullptr, nullptr, false, exclusive, sums, n);
    case OMNI_F32: return gemm_plain<kF32>(h, wd, nullptr, residual, y, T, H, I, s, nullptr, nullptr, false, exclusive, sums, n);
    default: return OMNI_ERR_DTYPE;
  }
}
}  // namespace omni

extern "C" OMNI_API size_t omni_mlp_workspace_bytes(int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size, int32_t dtype) {
  if (num_tokens < 0 || intermediate_size < 0) return 0;
  return omni::mlp_h_bytes(num_tokens, intermediate_size, dtype) + omni::mlp_sums_bytes(num_tokens, hidden_size, intermediate_size, dtype);     // h = silu(gate)*up | sums
}

extern "C" OMNI_API int32_t omni_mlp_fwd(const void* x, const void* gate_weight, const void* up_weight, const void* down_weight,
                                         const void* residual, void* y, int64_t num_tokens, int32_t hidden_size,
                                         int32_t intermediate_size, int32_t dtype, void* workspace, void* stream) {
  using namespace omni;
  if (num_tokens < 0 || hidden_size <= 0 || intermediate_size <= 0) return OMNI_ERR_SHAPE;
  if (num_tokens == 0) return OMNI_OK;
  if (!x || !gate_weight || !up_weight || !down_weight || !y) return OMNI_ERR_NULL;
  if (!workspace) return OMNI_ERR_WORKSPACE;
  int e;
  if (dtype != OMNI_BF16 && dtype != OMNI_F16 && dtype != OMNI_F32) return OMNI_ERR_DTYPE;
  // both projections are checked before the first one is enqueued: hidden and intermediate size are each the K of one
  const int es = dtype == OMNI_F32 ? 4 : 2;
  if ((e = check_gemm(num_tokens, intermediate_size, hidden_size, es)) || (e = check_gemm(num_tokens, hidden_size, intermediate_size, es)))
    return e;
  if (few_tokens_covers(num_tokens, hidden_size, intermediate_size, dtype)) {
    const FewTokens f{x, gate_weight, up_weight, down_weight, workspace, y, (float*)((char*)workspace + mlp_h_bytes(num_tokens, intermediate_size, dtype)), residual,
                      (int)num_tokens, hidden_size, intermediate_size};
    if (few_tokens_aligned(f)) {
      const hipError_t he = launch_few_tokens(dtype, f, (hipStream_t)stream);
      return he == hipSuccess ? OMNI_OK : OMNI_ERR_HIP_BASE + (int)he;
    }
  }
  void* const sums = (char*)workspace + mlp_h_bytes(num_tokens, intermediate_size, dtype);
  if ((e = mlp_gate_up_impl(x, gate_weight, up_weight, workspace, nullptr, nullptr, num_tokens, hidden_size, intermediate_size, dtype, sums, stream, true))) return e;
  return mlp_down_impl(workspace, down_weight, residual, y, num_tokens, hidden_size, intermediate_size, dtype, sums, stream, true);
}

namespace omni {
static int swiglu_linear(const void* x, const void* gate_weight, const void* up_weight, void* h, int64_t num_tokens, int32_t hidden_size,
                         int32_t intermediate_size, int32_t dtype, void* stream, bool exclusive) {
  if (num_tokens == 0) return OMNI_OK;
  if (!x || !gate_weight || !up_weight || !h) return OMNI_ERR_NULL;
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case OMNI_BF16: return gemm_swiglu<kBF16>(x, gate_weight, up_weight, h, num_tokens, intermediate_size, hidden_size, s, nullptr, nullptr, exclusive);
    case OMNI_F16: return gemm_swiglu<kF16>(x, gate_weight, up_weight, h, num_tokens, intermediate_size, hidden_size, s, nullptr, nullptr, exclusive);
    case OMNI_F32: return gemm_swiglu<kF32>(x, gate_weight, up_weight, h, num_tokens, intermediate_size, hidden_size, s, nullptr, nullptr, exclusive);
    default: return OMNI_ERR_DTYPE;
  }
}
}  // namespace omni

extern "C" OMNI_API int32_t omni_swiglu_linear_fwd(const void* x, const void* gate_weight, const void* up_weight, void* h,
                                                   int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size,
                                                   int32_t dtype, void* stream) {
  return omni::swiglu_linear(x, gate_weight, up_weight, h, num_tokens, hidden_size, intermediate_size, dtype, stream, true);
}

extern "C" OMNI_API int32_t omni_swiglu_linear_fwd_shared(const void* x, const void* gate_weight, const void* up_weight, void* h,
                                                          int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size,
                                                          int32_t dtype, void* stream) {
  return omni::swiglu_linear(x, gate_weight, up_weight, h, num_tokens, hidden_size, intermediate_size, dtype, stream, false);
}

extern "C" OMNI_API int32_t omni_swiglu_linear_save_fwd(const void* x, const void* gate_weight, const void* up_weight, void* h,
                                                        void* gate_out, void* up_out, int64_t num_tokens, int32_t hidden_size,
                                                        int32_t intermediate_size, int32_t dtype, void* stream) {
  using namespace omni;
  if (num_tokens == 0) return OMNI_OK;
  if (!x || !gate_weight || !up_weight || !h || !gate_out || !up_out) return OMNI_ERR_NULL;
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case OMNI_BF16: return gemm_swiglu<kBF16>(x, gate_weight, up_weight, h, num_tokens, intermediate_size, hidden_size, s, gate_out, up_out);
    case OMNI_F16: return gemm_swiglu<kF16>(x, gate_weight, up_weight, h, num_tokens, intermediate_size, hidden_size, s, gate_out, up_out);
    case OMNI_F32: return OMNI_ERR_UNSUPPORTED;
    default: return OMNI_ERR_DTYPE;
  }
}

extern "C" OMNI_API int32_t omni_linear_fwd(const void* x, const void* weight, const void* residual, void* y, int64_t num_tokens,
                                            int32_t in_features, int32_t out_features, int32_t dtype, void* stream) {
  using namespace omni;
  if (num_tokens == 0) return OMNI_OK;
  if (!x || !weight || !y) return OMNI_ERR_NULL;
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case OMNI_BF16: return gemm_plain<kBF16>(x, weight, nullptr, residual, y, num_tokens, out_features, in_features, s);
    case OMNI_F16: return gemm_plain<kF16>(x, weight, nullptr, residual, y, num_tokens, out_features, in_features, s);
    case OMNI_F32: return gemm_plain<kF32>(x, weight, nullptr, residual, y, num_tokens, out_features, in_features, s);
    default: return OMNI_ERR_DTYPE;
  }
}

extern "C" OMNI_API int32_t omni_linear2_fwd(const void* x, const void* weight_lo, const void* weight_hi, void* y,
                                             int64_t num_tokens, int32_t in_features, int32_t out_features_each,
                                             int32_t dtype, void* stream) {
  using namespace omni;
  if (num_tokens == 0) return OMNI_OK;
  if (!x || !weight_lo || !weight_hi || !y) return OMNI_ERR_NULL;
  hipStream_t s = (hipStream_t)stream;
  const int64_t n = 2 * (int64_t)out_features_each;
  switch (dtype) {
    case OMNI_BF16: return gemm_plain<kBF16>(x, weight_lo, weight_hi, nullptr, y, num_tokens, n, in_features, s);
    case OMNI_F16: return gemm_plain<kF16>(x, weight_lo, weight_hi, nullptr, y, num_tokens, n, in_features, s);
    case OMNI_F32: return gemm_plain<kF32>(x, weight_lo, weight_hi, nullptr, y, num_tokens, n, in_features, s);
    default: return OMNI_ERR_DTYPE;
  }
}

namespace omni {
// y[i] = round(y[i] + e[i]), 8 (16-bit) or 4 (fp32) elements per lane
template <int DT>
__global__ __launch_bounds__(256) void add_inplace_kernel(uint8_t* __restrict__ y, const uint8_t* __restrict__ e, int64_t num_chunks) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < num_chunks; i += gridDim.x * 256ll) {
    const u32x4_t a = *(const u32x4_t*)(y + i * 16), b = *(const u32x4_t*)(e + i * 16);
    u32x4_t o;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t aq = a[q], bq = b[q];
      if constexpr (DT == kBF16) o[q] = pack_bf16(bf16_lo(aq) + bf16_lo(bq), bf16_hi(aq) + bf16_hi(bq));
      else if constexpr (DT == kF16) o[q] = pack_f16(f16_bits_to_f32(aq & 0xffff) + f16_bits_to_f32(bq & 0xffff), f16_bits_to_f32(aq >> 16) + f16_bits_to_f32(bq >> 16));
      else o[q] = __float_as_uint(__uint_as_float(aq) + __uint_as_float(bq));
    }
    *(u32x4_t*)(y + i * 16) = o;
  }
}
}  // namespace omni

extern "C" OMNI_API int32_t omni_add_inplace(void* y, const void* addend, int64_t num_elements, int32_t dtype, void* stream) {
  using namespace omni;
  if (num_elements < 0) return OMNI_ERR_SHAPE;
  if (dtype != OMNI_BF16 && dtype != OMNI_F16 && dtype != OMNI_F32) return OMNI_ERR_DTYPE;
  const int per = dtype == OMNI_F32 ? 4 : 8;
  if (num_elements % per != 0) return OMNI_ERR_SHAPE;
  if (num_elements == 0) return OMNI_OK;
  if (!y || !addend) return OMNI_ERR_NULL;
  const int64_t chunks = num_elements / per;
  const unsigned blocks = (unsigned)((chunks + 255) / 256 < 4096 ? (chunks + 255) / 256 : 4096);
  hipStream_t s = (hipStream_t)stream;
  if (dtype == OMNI_BF16) hipLaunchKernelGGL(add_inplace_kernel<kBF16>, dim3(blocks), dim3(256), 0, s, (uint8_t*)y, (const uint8_t*)addend, chunks);
  else if (dtype == OMNI_F16) hipLaunchKernelGGL(add_inplace_kernel<kF16>, dim3(blocks), dim3(256), 0, s, (uint8_t*)y, (const uint8_t*)addend, chunks);
  else hipLaunchKernelGGL(add_inplace_kernel<kF32>, dim3(blocks), dim3(256), 0, s, (uint8_t*)y, (const uint8_t*)addend, chunks);
  return omni::to_code(hipGetLastError());
}

namespace omni {
template <int DT>
__device__ __forceinline__ f32x4_t mfma16(const u32x4_t a, const u32x4_t b, f32x4_t c) {
  if constexpr (DT == kBF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// Matrix-core rate with nothing else going on: every wave keeps 16 accumulator tiles and issues
// MFMAs on operands it read once (8 KiB of caller data, so that the operand bits are realistic:
// the sustained clock under the board's power limit depends on how many bits toggle).
__global__ __launch_bounds__(kGemmThreads, 1) void mfma_probe_kernel(const u32x4_t* __restrict__ operands, float* __restrict__ sink, int iters) {
  f32x16_t acc[16];
#pragma unroll
  for (int i = 0; i < 16; ++i)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[i][q] = 0.f;
  u32x4_t a[4], b[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[i] = operands[(threadIdx.x * 8 + i) & 511];
    b[i] = operands[(threadIdx.x * 8 + 4 + i) & 511];
  }
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = mfma32<kBF16>(a[i & 3], b[i >> 2], acc[i]);
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) s += acc[i][0] + acc[i][5];
  sink[blockIdx.x * kGemmThreads + threadIdx.x] = s;
}
// The same with v_mfma_f32_16x16x32_bf16, the streaming kernel's instruction: 8 waves per block (two per SIMD, as that
// kernel runs), 8 x 4 independent accumulator tiles per wave.
__global__ __launch_bounds__(512, 1) void mfma_probe16_kernel(const u32x4_t* __restrict__ operands, float* __restrict__ sink, int iters) {
  f32x4_t acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[i][j][q] = 0.f;
  u32x4_t a[8], b[4];
#pragma unroll
  for (int i = 0; i < 8; ++i) a[i] = operands[(threadIdx.x * 12 + i) & 511];
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = operands[(threadIdx.x * 12 + 8 + i) & 511];
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = mfma16<kBF16>(b[j], a[i], acc[i][j]);
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) s += acc[i][j][0] + acc[i][j][3];
  sink[blockIdx.x * 512 + threadIdx.x] = s;
}
}  // namespace omni

extern "C" OMNI_API int32_t omni_probe_mfma16(const void* operands, float* sink, int32_t num_blocks, int32_t iters, void* stream) {
  if (num_blocks <= 0 || iters <= 0) return OMNI_ERR_SHAPE;
  if (!operands || !sink) return OMNI_ERR_NULL;
  hipLaunchKernelGGL(omni::mfma_probe16_kernel, dim3(num_blocks), dim3(512), 0, (hipStream_t)stream, (const omni::u32x4_t*)operands, sink, iters);
  return omni::to_code(hipGetLastError());
}

extern "C" OMNI_API int32_t omni_probe_mfma(const void* operands, float* sink, int32_t num_blocks, int32_t iters, void* stream) {
  if (num_blocks <= 0 || iters <= 0) return OMNI_ERR_SHAPE;
  if (!operands || !sink) return OMNI_ERR_NULL;
  hipLaunchKernelGGL(omni::mfma_probe_kernel, dim3(num_blocks), dim3(omni::kGemmThreads), 0, (hipStream_t)stream,
                     (const omni::u32x4_t*)operands, sink, iters);
  return omni::to_code(hipGetLastError());
}

