// Arguments of the general tile GEMM (gemm_tiles.hip): one launch, several products.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace omni {

// operand layouts.  NT: rows of both run along K (A [M,K], B [N,K]).  NN: A [M,K], B [K,N].  TN: A [K,M], B [K,N].
enum : int { kNT = 0, kNN = 1, kTN = 2 };
// what becomes of a sum.  Plain: rounded.  Residual: rounded, the residual added, rounded again.  Swiglu (NT): B is two matrices, gate and up
// rows; silu(round(gate sum)) * round(up sum).  SwigluBwd: the rounded sum is d(h); out come d(gate) and d(up).  Two (NT): plain, the upper half of
// the columns (N % 16 == 0) from a second B.
enum : int { kTilePlain = 0, kTileResidual = 1, kTileSwiglu = 2, kTileSwigluBwd = 3, kTileTwo = 4 };
constexpr int kMaxSegments = 4, kMaxProducts = 5;

struct TileSegment {       // one K range of a product
  const uint8_t *a, *b;
  int64_t lda, ldb;        // bytes between rows
  int64_t a_skip;          // a's offset in bytes inside the first row of its matrix (a column range of it)
  int K;
};
struct TileProduct {       // C [M, N] = sum over segments of A B; 16-bit storage
  TileSegment seg[kMaxSegments];
  const uint8_t* b_up = nullptr;                   // kTileSwiglu: the up weights (segment 0's b: the gate weights); kTileTwo: the second B
  int segments = 0, M = 0, N = 0;
  int64_t ldc = 0;                                 // bytes between rows of c, c2, res, gate, up
  uint8_t* c = nullptr;
  uint8_t* c2 = nullptr;                           // kTileSwigluBwd: c = d(gate), c2 = d(up)
  uint8_t* c3 = nullptr;                           // kTileSwiglu: c2, c3 = NULL, or where the rounded gate and up sums go as well
  const uint8_t *res = nullptr, *gate = nullptr, *up = nullptr;
  // set by the launch
  int first = 0, splits = 1, steps = 0;            // first block; K split this many ways, `steps` ring steps each
  float* part = nullptr;                           // splits > 1: [splits][M][columns] fp32 partial sums
};
struct TileGroup {
  TileProduct p[kMaxProducts];
  int count = 0;
};
// A launch of one product carries that one only: kernel arguments are read from uncached memory at the start of every block.
struct TileSingle {
  TileProduct p[1];
  int count = 1;
};

// Launches the group on `s`: one product of any layout, or several kTN ones.  M, N, K of any size; N and the rows' lengths in bytes are multiples of
// 8 and 16.  `ws`: room for the partial sums of a product that is split along K (tile_workspace_bytes() bytes; NULL: none is split).
// exclusive: nothing is meant to run beside the launch, which may then hold every CU until it ends.
// hipErrorInvalidValue, and nothing launched, for operands beyond 2 GiB per tile column.
hipError_t launch_tile_group(int dtype, int layout, int epilogue, TileGroup& g, void* ws, size_t ws_bytes, hipStream_t s, bool exclusive = true);
// What launch_tile_group wants for one product; K: the sum of its segments, each rounded up to 64
size_t tile_workspace_bytes(int layout, int epilogue, int64_t M, int64_t N, int64_t K);

// The layer's joint launches.  The router's projection (kTileTwo) in front of the gate/up projection (kTileSwiglu; gate and up kept where c2 and c3 say so), both kNT
// over the same K; false, and nothing launched, where its tiles would cost a round of their own or the operands are out of reach.
bool launch_tile_pair(int dtype, const TileProduct& router, const TileProduct& mlp, hipStream_t s, hipError_t* e);
// The down projection (kTilePlain, kNT) and, beside it, the selection, if there is room (*selected).  *parts > 1: its sums are left in ws, [parts][M][N] fp32.
struct SelectArgs;
constexpr int kMostDownParts = 8;
size_t tile_down_workspace_bytes(int64_t M, int64_t N, int64_t K);               // (what it wants in ws)
hipError_t launch_tile_down(int dtype, const TileProduct& p, const SelectArgs& select, void* ws, size_t ws_bytes, hipStream_t s, bool* selected, int* parts);

}  // namespace omni
