// The tile GEMM's host side: which tile shape and K split a product takes, and the launches.  The kernels: gemm_tiles_kernels.h.
#include "gemm_tiles_kernels.h"

namespace omni {

// (joint: those that share their launch with the layer's router)
constexpr unsigned kForwardShapes = shapes_of(kNT), kJointShapes = 1u << 1 | 1u << 2 | 1u << 3 | 1u << 4 | 1u << 7 | 1u << 8;

constexpr float kJoinedSumUs = 1.8f;

// Microseconds that a launch of n blocks of one shape takes for 64 of K.  Where two blocks share a CU, the CUs with two set the time however few they are
// (gate/up of 613 x 1024 x 4096 on 128 x 128 tiles, 320 blocks: 19.7 us; 450 rows, 256 blocks: 16.4; 1000 rows, 512 blocks: 21.4).
static float step_us(const ShapeCost& c, int64_t n) {
  constexpr int kCus = 256;
  const int64_t rounds = (n + c.at_once - 1) / c.at_once;
  const float used = n >= c.at_once ? 1.f : n > kCus ? 0.86f + 0.14f * (float)(n - kCus) / (c.at_once - kCus) : (float)n / c.at_once;
  return (float)rounds * (c.idle + (c.full - c.idle) * used);
}
// The fastest shape and K split by those figures.  K is split for a product on its own only, where every part keeps 256 of K, and the shapes
// whose two groups also split K (64 x 64; for dy W 128 x 128) are for K >= 512: shorter sums stay in one order whatever the shape.
// joined: the layer's down projection, whose parts the experts' kernel adds up if they are of a shape that the selection runs beside.  A split costs that kernel's
// longer wait then instead of a launch (kJoinedSumUs).  Layers in a graph, with a launch's 3.3 us / with 1.8: 197 x 512 x 1536 18.4 / 16.1 us, 221 x 1024 x 2048 23.8 / 21.0,
// 251 x 1536 x 3072 30.4 / 26.9, 613 x 1024 x 4096 40.0 / 37.8, 2475 x 512 x 2048 48.2 / 45.5, 85 x 256 x 1024 15.6 / 14.2, 714 x 1280 x 5120 55.6 / 55.1; of 20 none is slower by more
// than 0.3 %.  With 1.0 391 x 1024 x 2048 gains (26.0 -> 25.3) and 583 x 1280 x 3840 (43.1 -> 42.6), but 800 x 768 x 3072 leaves the selection no place, 33.7 -> 37.1.
static TileChoice choose_of(int epilogue, const TileSize* sizes, int count, int64_t K, bool may_split, unsigned shapes, bool joined) {
  TileChoice best;
  for (int i = 0; i < kShapes; ++i) {
    if (!(shapes >> i & 1)) continue;
    const ShapeCost& c = i == 4 && epilogue == kTileSwiglu ? kSwigluCost : kCost[i];
    if (c.kg > 1 && K < 512) continue;
    const int bn = epilogue == kTileSwiglu ? c.bn / 2 : c.bn;
    int64_t tiles = 0;
    for (int q = 0; q < count; ++q) tiles += ((sizes[q].M + c.bm - 1) / c.bm) * ((sizes[q].N + bn - 1) / bn);
    const int64_t kt = (K + 63) / 64;
    const float sum_us = joined && (kJointShapes >> i & 1) ? kJoinedSumUs : kReduceUs;
    for (int s = 1; s <= (!may_split || count != 1 ? 1 : joined ? kMostDownParts : kMostSplits); ++s) {
      if (s > 1 && kt / s < 4) break;
      float us = c.fixed + (float)((kt + s - 1) / s) * step_us(c, tiles * s);
      if (s > 1) us += sum_us + (float)s * (float)sizes[0].M * (float)(epilogue == kTileSwiglu ? 2 * sizes[0].N : sizes[0].N) * 4.f * (1.f / kPartsOut + 1.f / kPartsIn);
      if (us < best.us) best = TileChoice{i, s, us};
    }
  }
  return best;
}
// A call asks for its workspace and then for its launches, a program for the same sizes over and over, and a choice takes 0.6 us: a layer of one token,
// bound by the host, asked eight times.  Each thread keeps the last few products' choices, which nothing but the sizes goes into.
static TileChoice choose_tiles(int epilogue, const TileSize* sizes, int count, int64_t K, bool may_split, unsigned shapes = kForwardShapes, bool joined = false) {
  if (count != 1) return choose_of(epilogue, sizes, count, K, may_split, shapes, joined);
  struct Kept { int64_t M, N, K; uint64_t how; TileChoice choice; };
  constexpr int kKept = 16;
  static thread_local Kept kept[kKept];                        // (M = 0: none)
  static thread_local int oldest = 0;
  const uint64_t how = (uint64_t)shapes << 8 | (uint64_t)joined << 7 | (uint64_t)epilogue << 1 | (may_split ? 1 : 0);
  for (const Kept& k : kept)
    if (k.M == sizes->M && k.N == sizes->N && k.K == K && k.how == how) return k.choice;
  Kept& k = kept[oldest];
  oldest = (oldest + 1) % kKept;
  k = Kept{sizes->M, sizes->N, K, how, choose_of(epilogue, sizes, count, K, may_split, shapes, joined)};
  return k.choice;
}

// The layer's down projection: a shape that takes the selection beside it, unless another one gains more than the selection's own launch costs.  (That seldom decides: over the
// 56 layers below, 0 us for that launch or any price makes none faster, and two slower by 2 %.)
static TileChoice choose_down(const TileSize& size, int64_t K, bool may_split) {
  constexpr float kSelectUs = 6.f;
  const TileChoice any = choose_tiles(kTilePlain, &size, 1, K, may_split, kForwardShapes, true),
                   joint = choose_tiles(kTilePlain, &size, 1, K, may_split, kJointShapes, true);
  return joint.us <= any.us + kSelectUs ? joint : any;
}
// The shape that both products' tiles take least time in, by the figures above, if that is less than a launch for each; -1: it is not.
// Over 56 layers in a graph (65 to 3000 tokens, hidden 256 to 2048, 24 to 128 keys) a launch for each instead is slower by more than 1.5 % in 47 and faster in none (130 x 1536 x 3072
// 23.8 / 31.2 us); one launch always is faster in none.
static int choose_pair(const TileSize& router, const TileSize& mlp, int64_t K) {
  const TileSize sizes[2] = {router, mlp};
  const int64_t kt = (K + 63) / 64;
  int shape = -1;
  float best = choose_tiles(kTileTwo, sizes, 1, K, false).us + choose_tiles(kTileSwiglu, sizes + 1, 1, K, true).us;
  for (int i = 0; i < kShapes; ++i) {
    if (!(kJointShapes >> i & 1)) continue;                    // (256 x 256: 30.6 us at 1024 tokens, where the two launches take 25.8)
    const ShapeCost &r = kCost[i], &m = i == 4 ? kSwigluCost : kCost[i];
    if (r.kg > 1 && K < 512) continue;
    const int64_t n = ((router.M + r.bm - 1) / r.bm) * ((router.N + r.bn - 1) / r.bn) + ((mlp.M + m.bm - 1) / m.bm) * ((mlp.N + m.bn / 2 - 1) / (m.bn / 2));
    const float us = m.fixed + (float)kt * step_us(m, n);
    if (us < best) { best = us; shape = i; }
  }
  return shape;
}
static size_t parts_bytes(const TileChoice& c, int64_t M, int64_t columns) { return c.splits > 1 ? (size_t)c.splits * (size_t)M * (size_t)columns * 4 : 0; }

size_t tile_workspace_bytes(int layout, int epilogue, int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const TileSize size{M, N};
  const TileChoice c = choose_tiles(epilogue, &size, 1, K, true, shapes_of(layout));
  return parts_bytes(c, M, epilogue == kTileSwiglu ? 2 * N : N);
}
size_t tile_down_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return parts_bytes(choose_down(TileSize{M, N}, K, true), M, N);
}

hipError_t launch_tile_group(int dtype, int layout, int epilogue, TileGroup& g, void* ws, size_t ws_bytes, hipStream_t s, bool exclusive) {
  if (g.count <= 0) return hipSuccess;
  TileSize sizes[kMaxProducts];
  int64_t K = 0;
  for (int i = 0; i < g.count; ++i) {
    sizes[i] = TileSize{g.p[i].M, g.p[i].N};
    int64_t k = 0;
    for (int q = 0; q < g.p[i].segments; ++q) {
      const TileSegment& sg = g.p[i].seg[q];
      k += (sg.K + 63) / 64 * 64;
      // offsets inside a block's share of an operand are 31-bit
      const int64_t a_span = layout == kTN ? (int64_t)sg.K * sg.lda : 256 * sg.lda, b_span = layout == kNT ? 256 * sg.ldb : (int64_t)sg.K * sg.ldb;
      if (a_span > INT32_MAX || b_span > INT32_MAX || 128 * sg.lda > INT32_MAX || 128 * sg.ldb > INT32_MAX) return hipErrorInvalidValue;
    }
    K = k > K ? k : K;
  }
  TileChoice c = choose_tiles(epilogue, sizes, g.count, K, ws != nullptr, shapes_of(layout));
  if (parts_bytes(c, g.p[0].M, epilogue == kTileSwiglu ? 2 * (int64_t)g.p[0].N : g.p[0].N) > ws_bytes)
    c = choose_tiles(epilogue, sizes, g.count, K, false, shapes_of(layout));
  if (dtype == kBF16) return tile_group_of<kBF16>(layout, epilogue, g, c, (float*)ws, exclusive, s);
  if (dtype == kF16) return tile_group_of<kF16>(layout, epilogue, g, c, (float*)ws, exclusive, s);
  return hipErrorInvalidValue;
}

static bool in_reach(const TileProduct& p) { return 256 * p.seg[0].lda <= INT32_MAX && 256 * p.seg[0].ldb <= INT32_MAX; }     // as launch_tile_group has it

bool launch_tile_pair(int dtype, const TileProduct& router, const TileProduct& mlp, hipStream_t s, hipError_t* e) {
  if ((dtype != kBF16 && dtype != kF16) || !in_reach(router) || !in_reach(mlp)) return false;
  TilePair g;
  g.router.p[0] = router;
  g.mlp.p[0] = mlp;
  const int shape = choose_pair(TileSize{router.M, router.N}, TileSize{mlp.M, mlp.N}, mlp.seg[0].K);
  return dtype == kBF16 ? tile_pair_of<kBF16>(shape, g, s, e) : tile_pair_of<kF16>(shape, g, s, e);
}

hipError_t launch_tile_down(int dtype, const TileProduct& p, const SelectArgs& select, void* ws, size_t ws_bytes, hipStream_t s, bool* selected, int* parts) {
  if ((dtype != kBF16 && dtype != kF16) || !in_reach(p)) return hipErrorInvalidValue;
  const TileSize size{p.M, p.N};
  TileChoice c = choose_down(size, p.seg[0].K, ws != nullptr);
  if (parts_bytes(c, p.M, p.N) > ws_bytes) c = choose_down(size, p.seg[0].K, false);
  return dtype == kBF16 ? tile_down_of<kBF16>(p, select, c, (float*)ws, s, selected, parts) : tile_down_of<kF16>(p, select, c, (float*)ws, s, selected, parts);
}
}  // namespace omni

extern "C" OMNI_API int32_t omni_probe_joint_tiles(int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size, int32_t num_expert_sqrt, int32_t num_experts_per_token,
                                                   int32_t* pair, int32_t* down) {
  using namespace omni;
  if (num_tokens <= 0 || num_tokens > INT32_MAX / 256 || hidden_size <= 0 || intermediate_size <= 0 || num_expert_sqrt <= 0 || num_experts_per_token <= 0) return OMNI_ERR_SHAPE;
  if (num_experts_per_token > 128) return OMNI_ERR_TOPK;
  if (!pair || !down) return OMNI_ERR_NULL;
  const int shape = choose_pair(TileSize{num_tokens, 2 * (int64_t)num_expert_sqrt}, TileSize{num_tokens, intermediate_size}, hidden_size);
  const TileChoice c = choose_down(TileSize{num_tokens, hidden_size}, intermediate_size, true);
  SelectArgs select{};
  select.r = num_expert_sqrt; select.k = num_experts_per_token;
  const int cells = prepare_select(select), regs = (num_expert_sqrt + kWave - 1) / kWave;
  auto plan = [&](auto id) { return plan_down<decltype(id)::value>(num_tokens, hidden_size, intermediate_size, c.splits, (int)num_tokens, regs, cells); };
  DownPlan p{0, c.splits, 0, 0, false};                          // (the other shapes: nothing beside them)
  if (c.shape == 1) p = plan(std::integral_constant<int, 1>{});
  else if (c.shape == 2) p = plan(std::integral_constant<int, 2>{});
  else if (c.shape == 3) p = plan(std::integral_constant<int, 3>{});
  else if (c.shape == 4) p = plan(std::integral_constant<int, 4>{});
  else if (c.shape == 7) p = plan(std::integral_constant<int, 7>{});
  else if (c.shape == 8) p = plan(std::integral_constant<int, 8>{});
  pair[0] = shape < 0 ? 0 : kCost[shape].bm;
  pair[1] = shape < 0 ? 0 : kCost[shape].bn;
  down[0] = kCost[c.shape].bm;
  down[1] = kCost[c.shape].bn;
  down[2] = p.splits;
  down[3] = p.selected ? 1 : 0;
  return OMNI_OK;
}
extern "C" OMNI_API int32_t omni_probe_tile_choice(int32_t layout, int32_t epilogue, int64_t rows, int64_t columns, int64_t k, int32_t* choice) {
  using namespace omni;
  if (layout < kNT || layout > kTN || epilogue < kTilePlain || epilogue > kTileSwigluBwd || rows <= 0 || columns <= 0 || k <= 0) return OMNI_ERR_SHAPE;
  if (!choice) return OMNI_ERR_NULL;
  const TileSize size{rows, columns};
  const TileChoice c = choose_tiles(epilogue, &size, 1, k, layout != kTN, shapes_of(layout));
  choice[0] = kCost[c.shape].bm;
  choice[1] = kCost[c.shape].bn;
  choice[2] = kCost[c.shape].kg;
  choice[3] = c.splits;
  return OMNI_OK;
}
