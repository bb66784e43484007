// Backward of the shared SwiGLU MLP, with the router projection's share of the same products (reference: autograd of the matmuls of
// interface.py:23-29 and omni_moe.py:70-71, and omni_mlp.py:180-249 between them).  Three launches of the tile GEMM:
//   d(gate), d(up) [T,I]  from  d(h) = dy Wd, the SwiGLU backward as its epilogue: d(h) itself never reaches memory
//   dWg, dWu, dWd, dWx, dWy  in one launch: each has too few tiles to fill the chip alone
//   d(x) = dgate Wg + dup Wu + dz_x Wx + dz_y Wy  (+ the experts' d(x)) as one sum in fp32
// At 4096 tokens x 1024 x 4096 with 64 keys a half, bf16: 57 + 101 + 76 us of kernels (traced) where the library's nine products, the element-wise SwiGLU
// kernel and the additions took 350.
#include "common.h"
#include "gemm_tiles.h"
#include "omni_moe_hip.h"

namespace omni {
static inline size_t up256(size_t v) { return (v + 255) / 256 * 256; }
static inline int64_t up64(int64_t v) { return (v + 63) / 64 * 64; }
static int to_code(hipError_t e) { return e == hipSuccess ? OMNI_OK : e == hipErrorInvalidValue ? OMNI_ERR_UNSUPPORTED : OMNI_ERR_HIP_BASE + (int)e; }

// partial sums of d(h) or of d(x), whichever is more (they are not alive together)
static size_t sums_bytes(int64_t T, int64_t H, int64_t I, int64_t r) {
  const size_t dh = tile_workspace_bytes(kNN, kTileSwigluBwd, T, I, up64(H)), dx = tile_workspace_bytes(kNN, kTileResidual, T, H, 2 * up64(I) + 2 * up64(r));
  return dh > dx ? dh : dx;
}
}  // namespace omni

extern "C" OMNI_API size_t omni_mlp_bwd_workspace_bytes(int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size, int32_t num_expert_sqrt, int32_t dtype) {
  using namespace omni;
  if (num_tokens <= 0 || hidden_size <= 0 || intermediate_size <= 0 || num_expert_sqrt < 0 || dtype == OMNI_F32) return 0;
  return 2 * up256((size_t)num_tokens * (size_t)intermediate_size * 2) + up256(sums_bytes(num_tokens, hidden_size, intermediate_size, num_expert_sqrt));
}

extern "C" OMNI_API int32_t omni_mlp_bwd(const void* dy, const void* x, const void* gate_weight, const void* up_weight, const void* down_weight, const void* gate,
                                         const void* up, const void* h, const void* dz, const void* router_weight_x, const void* router_weight_y,
                                         const void* dx_addend, void* dx, void* dgate_weight, void* dup_weight, void* ddown_weight, void* drouter_weight_x,
                                         void* drouter_weight_y, int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size, int32_t num_expert_sqrt,
                                         int32_t dtype, void* workspace, void* stream) {
  using namespace omni;
  if (num_tokens <= 0 || hidden_size <= 0 || intermediate_size <= 0 || num_expert_sqrt < 0) return OMNI_ERR_SHAPE;
  if (dtype == OMNI_F32) return OMNI_ERR_UNSUPPORTED;
  if (dtype != OMNI_BF16 && dtype != OMNI_F16) return OMNI_ERR_DTYPE;
  const int64_t most = INT32_MAX / 4, T = num_tokens, H = hidden_size, I = intermediate_size, r = num_expert_sqrt;
  if (H % 8 || I % 8 || T > most || H > most || I > most || r > most / 2) return OMNI_ERR_SHAPE;
  if (!dy || !x || !gate_weight || !up_weight || !down_weight || !gate || !up || !h) return OMNI_ERR_NULL;
  if (dz ? (r == 0 || !router_weight_x || !router_weight_y) : (drouter_weight_x || drouter_weight_y)) return OMNI_ERR_NULL;
  if (!workspace) return OMNI_ERR_WORKSPACE;
  // What the tile GEMM asks of its operands, before anything is enqueued: 16-byte aligned (dy, for one, may be a view that autograd cut out of a flat
  // gradient at any offset), and within reach of 31-bit offsets (2 GiB)
  for (const void* q : {dy, x, gate_weight, up_weight, down_weight, gate, up, h, dz, router_weight_x, router_weight_y, dx_addend, (const void*)dx, (const void*)dgate_weight,
                        (const void*)dup_weight, (const void*)ddown_weight, (const void*)drouter_weight_x, (const void*)drouter_weight_y, (const void*)workspace})
    if ((uintptr_t)q % 16) return OMNI_ERR_UNSUPPORTED;
  if (T * (I > H ? I : H) * 2 > INT32_MAX || H * I * 2 > INT32_MAX || T * 4 * ((r + 7) / 8 * 8) > INT32_MAX) return OMNI_ERR_UNSUPPORTED;
  hipStream_t s = (hipStream_t)stream;
  uint8_t* dgate = (uint8_t*)workspace;
  uint8_t* dup = dgate + up256((size_t)T * I * 2);
  void* sums = dup + up256((size_t)T * I * 2);
  const size_t sums_len = sums_bytes(T, H, I, r);
  const int64_t h2 = H * 2, i2 = I * 2, rp = (r + 7) / 8 * 8, z2 = 4 * rp;
  auto seg = [](const void* a, int64_t lda, const void* b, int64_t ldb, int64_t K, int64_t skip = 0) {
    return TileSegment{(const uint8_t*)a + skip, (const uint8_t*)b, lda, ldb, skip, (int)K};
  };
  hipError_t e;
  if (dx || dgate_weight || dup_weight) {
    TileGroup g;
    TileProduct& p = g.p[g.count++];
    p.seg[p.segments++] = seg(dy, h2, down_weight, i2, H);
    p.M = (int)T; p.N = (int)I; p.ldc = i2; p.c = dgate; p.c2 = dup; p.gate = (const uint8_t*)gate; p.up = (const uint8_t*)up;
    if ((e = launch_tile_group(dtype, kNN, kTileSwigluBwd, g, sums, sums_len, s)) != hipSuccess) return to_code(e);
  }
  {
    TileGroup g;
    auto add = [&](const void* a, int64_t lda, int64_t M, const void* b, int64_t ldb, int64_t N, void* c, int64_t skip = 0) {
      if (!c) return;
      TileProduct& p = g.p[g.count++];
      p.seg[p.segments++] = seg(a, lda, b, ldb, T, skip);
      p.M = (int)M; p.N = (int)N; p.ldc = N * 2; p.c = (uint8_t*)c;
    };
    add(dgate, i2, I, x, h2, H, dgate_weight);
    add(dup, i2, I, x, h2, H, dup_weight);
    add(dy, h2, H, h, i2, I, ddown_weight);
    add(dz, z2, r, x, h2, H, drouter_weight_x);
    add(dz, z2, r, x, h2, H, drouter_weight_y, 2 * rp);
    if ((e = launch_tile_group(dtype, kTN, kTilePlain, g, nullptr, 0, s)) != hipSuccess) return to_code(e);
  }
  if (dx) {
    TileGroup g;
    TileProduct& p = g.p[g.count++];
    p.seg[p.segments++] = seg(dgate, i2, gate_weight, h2, I);
    p.seg[p.segments++] = seg(dup, i2, up_weight, h2, I);
    if (dz) {
      p.seg[p.segments++] = seg(dz, z2, router_weight_x, h2, r);
      p.seg[p.segments++] = seg(dz, z2, router_weight_y, h2, r, 2 * rp);
    }
    p.M = (int)T; p.N = (int)H; p.ldc = h2; p.c = (uint8_t*)dx; p.res = (const uint8_t*)dx_addend;
    if ((e = launch_tile_group(dtype, kNN, dx_addend ? kTileResidual : kTilePlain, g, sums, sums_len, s)) != hipSuccess) return to_code(e);
  }
  return OMNI_OK;
}
