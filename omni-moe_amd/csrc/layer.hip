// The whole OmniMoE forward (reference omni_moe/modules/omni_moe.py:60-106) as one call:
// router -> fused experts on one branch, gate/up projection -> down projection on the other,
// joined by the final add.  With a second stream the two branches are enqueued side by side
// (the expert kernel lives on cache bandwidth and no LDS, the down projection on LDS and the
// matrix cores, so they share CUs); the fork and the join are two events the caller owns.
#include "common.h"
#include "few_tokens.h"
#include "gemm_tiles.h"
#include "omni_moe_hip.h"

// defined beside the GEMM kernels: z = x [Wx;Wy]^T
int omni_gemm_router_projection(const void* x, const void* wx, const void* wy, void* z, float* part_mean, float* part_m2, int64_t T, int H, int r, int dtype, void* stream, bool exclusive = true);

namespace omni {
static inline size_t up256(size_t v) { return (v + 255) / 256 * 256; }
static inline size_t elem_bytes(int dtype) { return dtype == OMNI_F32 ? 4 : 2; }
// defined beside the expert kernels: OMNI_OK when omni_expert_fwd takes `algo` at this shape (decided from the sizes alone)
int expert_algo_check(int algo, int64_t num_tokens, int hidden_size, int64_t num_experts, int top_k, int dtype);
// ... and whether the joint launches may gather the experts there
bool joint_launches_gather(int algo, int64_t T, int H, int64_t N, int k, int dtype);
// defined beside the select kernels: whether they take num_expert_sqrt keys per half with top_k and this dtype
bool select_covers(int r, int k, int dtype);
int launch_router_select(const SelectArgs& g, hipStream_t s);
// defined there: omni_router_fwd, with the caller's word on whether the call has the GPU to itself, and (0: none) the block size of the joint launches whose order
// the batch statistics' sums take
int router_fwd(const void* x, const void* weight_x, const void* weight_y,
               void* running_mean_x, void* running_var_x, int64_t* num_batches_tracked_x,
               void* running_mean_y, void* running_var_y, int64_t* num_batches_tracked_y,
               int32_t training, float momentum, float eps, void* gates, int32_t* indices,
               void* scores, int64_t num_tokens, int32_t hidden_size, int32_t num_expert_sqrt,
               int32_t num_experts_per_token, int32_t dtype, int32_t stats_dtype,
               void* workspace, void* stream, bool exclusive, int order_threads);
// defined beside the expert kernels: the gather algorithm with the final add (shared: AUTO's, whose waves may share a token's slots)
hipError_t launch_gather_add(const void* x, const void* up, const void* down, const void* gates, const int32_t* ids, void* y, const float* parts, int splits, bool shared, int64_t T,
                             int H, int k, int64_t N, int dtype, hipStream_t s);
// ... and alone
int expert_gather_f32(const void* x, const void* up, const void* down, const void* gates, const int32_t* ids, void* y, bool shared, int64_t T, int H, int k, int64_t N,
                      hipStream_t s);
// defined beside the GEMM kernels: a small single-precision layer up to the experts, as two launches, and whether they cover its sizes
bool f32_joint_covers(int64_t T, int64_t H, int64_t I, int r, int k);
hipError_t launch_f32_joint(const void* x, const void* wx, const void* wy, void* z, const void* wg, const void* wu, const void* wd, void* h, void* y, int64_t T, int64_t H, int64_t I,
                            const SelectArgs& args, bool statistics, hipStream_t s);
// defined beside the GEMM kernels: the two projections of omni_mlp_fwd with the caller's word on whether the launch has the GPU to itself
// (then a GEMM of more tiles than CUs may take the form that holds every CU until it ends).  gate, up: NULL, or where the rounded projections go as well;
// sums: mlp_sums_bytes()
int mlp_gate_up_impl(const void* x, const void* wg, const void* wu, void* h, void* gate, void* up, int64_t T, int32_t H, int32_t I, int32_t dtype, void* sums, void* stream, bool exclusive);
int mlp_down_impl(const void* h, const void* wd, const void* residual, void* y, int64_t T, int32_t H, int32_t I, int32_t dtype, void* sums, void* stream, bool exclusive);
size_t mlp_sums_bytes(int64_t T, int64_t H, int64_t I, int dtype);
// What a differentiable forward leaves for its backward pass: the router's workspace (z and the statistics), gates and ids, the pair scores (or NULL), the
// rounded gate and up projections, their SwiGLU product
struct Kept { void *router, *gates; int32_t* ids; float* scores; void *gate, *up, *h; };
// The experts with a block of eight waves per token up to here, with one to four waves per token (gather_waves) beyond.  The whole layer, block against waves, at
// 65 / 128 / 256 / 320 / 384 tokens, bf16:
//   hidden  256, top-16   20 / 20     20 / 20     20 / 20     20 / 20     20 / 20 us
//   hidden 1024, top-2    20 / 25     21 / 25     25 / 27     29 / 28     29 / 28
//   hidden 1024, top-16   21 / 26     22 / 26     27 / 28     31 / 30     32 / 30
//   hidden 1024, top-32   23 / 27     25 / 29     28 / 30     33 / 32     34 / 33
//   hidden 2048, top-16   27 / 30     28 / 31     40 / 41     45 / 44     46 / 45
//   hidden 4096, top-4    51 / 67     55 / 70     87 / 92
constexpr int kBlockPerToken = 256;
// Projection | gate/up, selection | down projection, experts and add; where two stages do not fit one launch, each is its own.
// shared: launch_gather_add's (a block per token always shares its slots).  statistics (training): projects z and leaves its column statistics, which f.select
// merges or reads.
// kept: NULL, or where gate and up stay.
template <class Statistics>
static int joint_forward(const FewTokens& f, const Kept* kept, int dtype, size_t parts_bytes, hipStream_t s, bool shared, bool training, Statistics&& statistics) {
  auto code = [](hipError_t e) { return e == hipSuccess ? OMNI_OK : OMNI_ERR_HIP_BASE + (int)e; };
  const int64_t H2 = (int64_t)f.H * 2, I2 = (int64_t)f.I * 2;
  TileProduct router, mlp, down;
  router.seg[0] = TileSegment{(const uint8_t*)f.x, (const uint8_t*)f.wx, H2, H2, 0, f.H};
  router.b_up = (const uint8_t*)f.wy;
  router.segments = mlp.segments = down.segments = 1;
  router.M = mlp.M = down.M = f.T;
  router.N = 2 * f.select.r; router.ldc = 2 * (int64_t)router.N; router.c = (uint8_t*)f.z;
  mlp.seg[0] = TileSegment{(const uint8_t*)f.x, (const uint8_t*)f.wg, H2, H2, 0, f.H};
  mlp.b_up = (const uint8_t*)f.wu;
  mlp.N = f.I; mlp.ldc = I2; mlp.c = (uint8_t*)f.h;
  void *const gate = kept ? kept->gate : nullptr, *const up = kept ? kept->up : nullptr;
  mlp.c2 = (uint8_t*)gate; mlp.c3 = (uint8_t*)up;
  down.seg[0] = TileSegment{(const uint8_t*)f.h, (const uint8_t*)f.wd, I2, I2, 0, f.I};
  down.N = f.H; down.ldc = H2; down.c = (uint8_t*)f.y;
  hipError_t he = hipSuccess;
  if (training) {
    if (int e = statistics()) return e;
    if (int e = mlp_gate_up_impl(f.x, f.wg, f.wu, f.h, gate, up, f.T, f.H, f.I, dtype, f.parts, s, true)) return e;
  } else if ((!kept || f.H % 64 == 0) && launch_tile_pair(dtype, router, mlp, s, &he)) {     // (other sizes' kept products divide: mlp_gate_up_impl)
    if (he != hipSuccess) return code(he);
  } else {
    if (int e = omni_gemm_router_projection(f.x, f.wx, f.wy, f.z, nullptr, nullptr, f.T, f.H, f.select.r, dtype, s)) return e;
    if (int e = mlp_gate_up_impl(f.x, f.wg, f.wu, f.h, gate, up, f.T, f.H, f.I, dtype, f.parts, s, true)) return e;
  }
  bool selected = false;
  int parts = 1;
  if ((he = launch_tile_down(dtype, down, f.select, parts_bytes ? f.parts : nullptr, parts_bytes, s, &selected, &parts)) != hipSuccess) return code(he);
  if (!selected)
    if (int e = launch_router_select(f.select, s)) return e;
  if (f.T <= kBlockPerToken) return code(launch_few_back(dtype, f, parts > 1 ? parts : 0, s));
  return code(launch_gather_add(f.x, f.up, f.down, f.select.gates, f.select.indices, f.y, parts > 1 ? f.parts : nullptr, parts, shared, f.T, f.H, f.select.k, f.N, dtype, s));
}
}  // namespace omni

// workspace: router workspace | gates [T,k] | ids [T,k] | expert output [T,H] | expert workspace | MLP workspace
extern "C" OMNI_API size_t omni_moe_workspace_bytes(int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size,
                                                    int64_t num_experts, int32_t num_expert_sqrt, int32_t num_experts_per_token,
                                                    int32_t dtype) {
  return omni_moe_workspace_bytes_algo(num_tokens, hidden_size, intermediate_size, num_experts, num_expert_sqrt, num_experts_per_token,
                                       dtype, OMNI_EXPERT_ALGO_AUTO);
}

extern "C" OMNI_API size_t omni_moe_workspace_bytes_algo(int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size,
                                                         int64_t num_experts, int32_t num_expert_sqrt, int32_t num_experts_per_token,
                                                         int32_t dtype, int32_t expert_algo) {
  using namespace omni;
  if (num_tokens < 0 || hidden_size <= 0 || intermediate_size <= 0 || num_expert_sqrt <= 0 || num_experts_per_token < 0) return 0;
  const size_t es = elem_bytes(dtype), T = (size_t)num_tokens, k = (size_t)num_experts_per_token;
  return up256(omni_router_workspace_bytes(num_tokens, num_expert_sqrt, dtype)) + up256(T * k * es) + up256(T * k * 4) +
         up256(T * (size_t)hidden_size * es) +
         up256(omni_expert_workspace_bytes(num_tokens, hidden_size, num_experts, num_experts_per_token, dtype, expert_algo)) +
         up256(omni_mlp_workspace_bytes(num_tokens, hidden_size, intermediate_size, dtype));
}

extern "C" OMNI_API int32_t omni_moe_fwd(const void* x, const void* gate_weight, const void* up_weight, const void* down_weight,
                                         const void* router_weight_x, const void* router_weight_y,
                                         void* running_mean_x, void* running_var_x, int64_t* num_batches_tracked_x,
                                         void* running_mean_y, void* running_var_y, int64_t* num_batches_tracked_y,
                                         const void* up_embed, const void* down_embed, void* y,
                                         int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size, int64_t num_experts,
                                         int32_t num_expert_sqrt, int32_t num_experts_per_token, int32_t dtype, int32_t stats_dtype,
                                         int32_t training, float momentum, float eps, void* workspace, void* stream,
                                         void* side_stream, void* fork_event, void* join_event) {
  return omni_moe_fwd_algo(x, gate_weight, up_weight, down_weight, router_weight_x, router_weight_y, running_mean_x, running_var_x,
                           num_batches_tracked_x, running_mean_y, running_var_y, num_batches_tracked_y, up_embed, down_embed, y,
                           num_tokens, hidden_size, intermediate_size, num_experts, num_expert_sqrt, num_experts_per_token, dtype,
                           stats_dtype, training, momentum, eps, workspace, stream, side_stream, fork_event, join_event,
                           OMNI_EXPERT_ALGO_AUTO);
}

namespace omni {
static int moe_fwd(const void* x, const void* gate_weight, const void* up_weight, const void* down_weight, const void* router_weight_x, const void* router_weight_y,
                   void* running_mean_x, void* running_var_x, int64_t* num_batches_tracked_x, void* running_mean_y, void* running_var_y, int64_t* num_batches_tracked_y,
                   const void* up_embed, const void* down_embed, void* y, int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size, int64_t num_experts,
                   int32_t num_expert_sqrt, int32_t num_experts_per_token, int32_t dtype, int32_t stats_dtype, int32_t training, float momentum, float eps,
                   void* workspace, void* stream, void* side_stream, void* fork_event, void* join_event, int32_t expert_algo, const Kept* kept) {
  if (num_tokens < 0 || hidden_size <= 0 || intermediate_size <= 0 || num_experts <= 0 || num_expert_sqrt <= 0) return OMNI_ERR_SHAPE;
  if (dtype != OMNI_BF16 && dtype != OMNI_F16 && dtype != OMNI_F32) return OMNI_ERR_DTYPE;
  // every stage's shape rule, before the first kernel is enqueued
  {
    const int64_t esz = (int64_t)elem_bytes(dtype), r = num_expert_sqrt, k = num_experts_per_token;
    if ((hidden_size * esz) % 16 != 0 || (intermediate_size * esz) % 16 != 0) return OMNI_ERR_SHAPE;   // rows are fetched 16 bytes at a time
    if (k < 0 || k > r * r || k > 128 || k % 2 != 0) return OMNI_ERR_TOPK;
    // (a differentiable call is as permissive as the operators it is made of: no selection needs no kernel, and ids beyond the table add nothing)
    if ((k > 0 || !kept) && !select_covers((int)r, (int)k, dtype)) return OMNI_ERR_UNSUPPORTED;
    if (r * r > num_experts && !kept) return OMNI_ERR_SHAPE;                                          // ids reach r*r - 1
    if (int e = expert_algo_check(expert_algo, num_tokens, hidden_size, num_experts, num_experts_per_token, dtype)) return e;
  }
  if (num_tokens == 0) return OMNI_OK;
  if (training && num_tokens == 1) return OMNI_ERR_SHAPE;   // batch statistics of one sample: nn.BatchNorm1d raises
  if (!x || !y || !up_embed || !down_embed) return OMNI_ERR_NULL;
  if (!workspace) return OMNI_ERR_WORKSPACE;
  if (side_stream && (!fork_event || !join_event)) return OMNI_ERR_NULL;
  const size_t es = elem_bytes(dtype), T = (size_t)num_tokens, k = (size_t)num_experts_per_token;
  char* w = (char*)workspace;
  auto take = [&](void* own, size_t n) -> void* {               // a part of the workspace, unless the caller keeps it
    if (own) return own;
    void* const at = w;
    w += up256(n);
    return at;
  };
  void* router_ws = take(kept ? kept->router : nullptr, omni_router_workspace_bytes(num_tokens, num_expert_sqrt, dtype));
  void* gates = take(kept ? kept->gates : nullptr, T * k * es);
  int32_t* ids = (int32_t*)take(kept ? kept->ids : nullptr, T * k * 4);
  void* experts = take(nullptr, T * (size_t)hidden_size * es);
  void* expert_ws = take(nullptr, omni_expert_workspace_bytes(num_tokens, hidden_size, num_experts, num_experts_per_token, dtype, expert_algo));
  void* h = take(kept ? kept->h : nullptr, T * (size_t)intermediate_size * es);
  float* const sums = (float*)w;
  const size_t sums_bytes = mlp_sums_bytes(num_tokens, hidden_size, intermediate_size, dtype);

  hipStream_t main_s = (hipStream_t)stream;
  // Up to a certain size the layer is joint launches on the caller's stream: stages that do not depend on each other share one.
  //   * at most 64 tokens in eval mode (four row tiles, what a wave has registers and LDS for): few_tokens.hip, two or three launches; 64 tokens 44 -> 27 us (hidden 1024, bf16).
  //   * up to 2^33 token x hidden x intermediate (2048 tokens at 1024 x 4096), beyond which gate/up fills the chip for several rounds and two streams are the
  //     better overlap: projection | gate/up, selection | down projection, experts and add.  The bound is this rule's own: a side stream that is given
  //     does not move it (OmniMoE.overlap_min_work, the least work that OmniMoE gives one for, is the same number so that the two schedules meet).
  //     Key counts in eights: the projection's tiles take the two halves' weights eight rows at a time.  Others keep the six launches below (100 x 100 keys
  //     against 104 x 104, hidden 1024 x 4096: 43 / 27 us at 65 tokens, 59 / 44 at 613, 63 / 64 at 1024, 94 / 93 at 2000).
  const bool few = !kept && few_tokens_covers_layer(num_tokens, hidden_size, intermediate_size, num_expert_sqrt, num_experts_per_token, dtype);
  //     (rows within reach of the tile kernels' 31-bit offsets, as few_tokens_covers bounds them; the two launches of the general path have no such bound)
  const bool joint = dtype != OMNI_F32 && num_experts_per_token > 0 && num_expert_sqrt % 8 == 0 && hidden_size % 8 == 0 && intermediate_size % 8 == 0 &&
                     intermediate_size <= (1 << 20) && (double)num_tokens * hidden_size * intermediate_size <= 8589934592.0;
  // (batch statistics: the projection is a launch of its own, and the selecting blocks merge them up to where merge_here says, else a launch in front; a
  // cumulative average, momentum < 0, takes the general path)
  //   * single precision where every product has few output tiles (f32_joint_covers): the same bound.  A side stream that is given is used, and the two
  //     schedules give the same bits: the sizes alone say how the experts' sums run, on either.
  const bool gathers = joint_launches_gather(expert_algo, num_tokens, hidden_size, num_experts, num_experts_per_token, dtype) && num_experts <= UINT32_MAX;
  const bool shared = expert_algo == OMNI_EXPERT_ALGO_AUTO;
  const bool f32_sizes = dtype == OMNI_F32 && !kept && gathers && num_experts_per_token > 0 && (double)num_tokens * hidden_size * intermediate_size <= 8589934592.0 &&
                         num_tokens <= INT32_MAX / 256 && (!training || (momentum >= 0.f && merge_here(num_tokens, num_expert_sqrt))) &&
                         f32_joint_covers(num_tokens, hidden_size, intermediate_size, num_expert_sqrt, num_experts_per_token);
  const bool joint_f32 = f32_sizes && !side_stream;
  // (kept pair scores come from the split algorithm, which the joint launches do not have)
  if (joint_f32 || (gathers && !(kept && kept->scores) && (training ? joint && momentum >= 0.f : few || joint))) {
    if (stats_dtype != OMNI_BF16 && stats_dtype != OMNI_F16 && stats_dtype != OMNI_F32) return OMNI_ERR_DTYPE;
    if (!gate_weight || !up_weight || !down_weight || !router_weight_x || !router_weight_y || !running_mean_x || !running_var_x || !running_mean_y || !running_var_y)
      return OMNI_ERR_NULL;
    FewTokens f{x, gate_weight, up_weight, down_weight, h, y, sums, nullptr,
                (int)num_tokens, hidden_size, intermediate_size, router_weight_x, router_weight_y, router_ws};
    SelectArgs& g = f.select;
    g.lx = router_ws; g.ly = (const char*)router_ws + (size_t)num_expert_sqrt * es; g.row_stride = 2 * num_expert_sqrt;
    const bool merge = training && merge_here(num_tokens, num_expert_sqrt);
    const size_t strips = ((size_t)num_tokens + kBnRows - 1) / kBnRows;
    float* const stats = (float*)((char*)router_ws + omni_router_workspace_stats_offset(num_tokens, num_expert_sqrt, dtype));
    float* const part_mean = (float*)((char*)stats + up256((size_t)4 * num_expert_sqrt * 4));       // as omni_router_fwd lays its workspace out
    float* const part_m2 = (float*)((char*)part_mean + up256(strips * 2 * num_expert_sqrt * 4));
    if (merge) {
      g.part_mean = part_mean; g.part_m2 = part_m2; g.strips = (int)strips; g.momentum = momentum; g.stats_out = stats;
      g.count_batch[0] = num_batches_tracked_x; g.count_batch[1] = num_batches_tracked_y;
    }
    if (training && !merge) {
      g.stats = stats;
    } else {
      g.run_mean[0] = running_mean_x; g.run_mean[1] = running_mean_y;
      g.run_var[0] = running_var_x; g.run_var[1] = running_var_y;
      g.stat_dt = stats_dtype; g.eps = eps;
      if (kept) g.stats_out = stats;
    }
    g.gates = gates; g.indices = ids;
    g.num_tokens = (int)num_tokens; g.r = num_expert_sqrt; g.k = num_experts_per_token; g.dt = dtype;
    f.up = up_embed; f.down = down_embed; f.N = num_experts;
    const bool aligned = few_tokens_aligned(f) && !(kept && ((uintptr_t)kept->gate | (uintptr_t)kept->up) % 16);
    if (aligned && num_tokens <= INT32_MAX / 256) {
      if (dtype == OMNI_F32) {
        hipError_t he = launch_f32_joint(x, router_weight_x, router_weight_y, router_ws, gate_weight, up_weight, down_weight, h, y, num_tokens, hidden_size, intermediate_size, g,
                                         training != 0, main_s);
        if (he == hipSuccess) he = launch_gather_add(x, up_embed, down_embed, gates, ids, y, nullptr, 0, shared, num_tokens, hidden_size, num_experts_per_token, num_experts, dtype, main_s);
        return he == hipSuccess ? OMNI_OK : OMNI_ERR_HIP_BASE + (int)he;
      } else if (few && !training) {
        const hipError_t he = launch_few_tokens(dtype, f, main_s);
        return he == hipSuccess ? OMNI_OK : OMNI_ERR_HIP_BASE + (int)he;
      }
      return joint_forward(f, kept, dtype, sums_bytes, main_s, shared, training != 0, [&]() -> int {
        if (merge) return omni_gemm_router_projection(x, router_weight_x, router_weight_y, router_ws, part_mean, part_m2, num_tokens, hidden_size, num_expert_sqrt, dtype, main_s);
        // without a selection (k = 0) omni_router_fwd projects, merges the statistics, moves the running buffers and counts the batch
        return omni_router_fwd(x, router_weight_x, router_weight_y, running_mean_x, running_var_x, num_batches_tracked_x, running_mean_y, running_var_y,
                               num_batches_tracked_y, 1, momentum, eps, nullptr, nullptr, nullptr, num_tokens, hidden_size, num_expert_sqrt, 0, dtype, stats_dtype,
                               router_ws, main_s);
      });
    }
  }
  hipStream_t branch = side_stream ? (hipStream_t)side_stream : main_s;
  hipError_t he;
  if (side_stream) {
    if ((he = hipEventRecord((hipEvent_t)fork_event, main_s)) != hipSuccess) return OMNI_ERR_HIP_BASE + (int)he;
    if ((he = hipStreamWaitEvent(branch, (hipEvent_t)fork_event, 0)) != hipSuccess) return OMNI_ERR_HIP_BASE + (int)he;
  }
  // From here on the side stream may hold work: whatever happens, the caller's stream is made to wait
  // for it before this call returns, so that an error leaves no work behind that the caller cannot order.
  const bool alone = side_stream == nullptr;            // one stream: every kernel runs by itself
  int e = router_fwd(x, router_weight_x, router_weight_y, running_mean_x, running_var_x, num_batches_tracked_x, running_mean_y, running_var_y, num_batches_tracked_y,
                     training, momentum, eps, gates, ids, nullptr, num_tokens, hidden_size, num_expert_sqrt, num_experts_per_token, dtype, stats_dtype, router_ws, branch, alone,
                     f32_sizes ? kF32MergeThreads : 0);
  // Beside the side branch the gate/up projection keeps its one-block-per-tile grid while that is at most two rounds of 256 tiles
  // (CUs come free between the rounds); with more tiles the streaming form wins although it holds every CU (hidden 1024 x
  // intermediate 4096, two streams: 4096 tokens 125.7 against 128.0 us, 6144 tokens 188.9 against 178.5, 8192 tokens 243.5 against 228.7)
  const int64_t gate_up_tiles = ((num_tokens + 255) / 256) * (((int64_t)intermediate_size + 127) / 128);
  const bool exclusive = alone || gate_up_tiles > 512;
  if (e) {
  } else if (kept && dtype == OMNI_F32) {
    if (!(e = omni_linear_fwd(x, gate_weight, nullptr, kept->gate, num_tokens, hidden_size, intermediate_size, dtype, main_s)) &&
        !(e = omni_linear_fwd(x, up_weight, nullptr, kept->up, num_tokens, hidden_size, intermediate_size, dtype, main_s)))
      e = omni_swiglu_fwd(kept->gate, kept->up, h, num_tokens * intermediate_size, dtype, main_s);
  } else {
    e = mlp_gate_up_impl(x, gate_weight, up_weight, h, kept ? kept->gate : nullptr, kept ? kept->up : nullptr, num_tokens, hidden_size, intermediate_size, dtype, sums, main_s, exclusive);
  }
  if (!e) e = f32_sizes ? expert_gather_f32(x, up_embed, down_embed, gates, ids, experts, shared, num_tokens, hidden_size, num_experts_per_token, num_experts, branch)
                        : omni_expert_fwd_scores(x, up_embed, down_embed, gates, ids, experts, kept ? kept->scores : nullptr, num_tokens, hidden_size, num_experts,
                                                 num_experts_per_token, dtype, expert_algo, expert_ws, branch);
  if (!side_stream) {   // one stream: the add is the down projection's epilogue
    if (!e) e = mlp_down_impl(h, down_weight, experts, y, num_tokens, hidden_size, intermediate_size, dtype, sums, main_s, true);
    return e;
  }
  if (!e) e = mlp_down_impl(h, down_weight, nullptr, y, num_tokens, hidden_size, intermediate_size, dtype, sums, main_s, false);
  if ((he = hipEventRecord((hipEvent_t)join_event, branch)) != hipSuccess) return e ? e : OMNI_ERR_HIP_BASE + (int)he;
  if ((he = hipStreamWaitEvent(main_s, (hipEvent_t)join_event, 0)) != hipSuccess) return e ? e : OMNI_ERR_HIP_BASE + (int)he;
  if (e) return e;
  return omni_add_inplace(y, experts, (int64_t)T * hidden_size, dtype, main_s);
}
}  // namespace omni

extern "C" OMNI_API int32_t omni_moe_fwd_algo(const void* x, const void* gate_weight, const void* up_weight, const void* down_weight,
                                              const void* router_weight_x, const void* router_weight_y,
                                              void* running_mean_x, void* running_var_x, int64_t* num_batches_tracked_x,
                                              void* running_mean_y, void* running_var_y, int64_t* num_batches_tracked_y,
                                              const void* up_embed, const void* down_embed, void* y,
                                              int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size, int64_t num_experts,
                                              int32_t num_expert_sqrt, int32_t num_experts_per_token, int32_t dtype, int32_t stats_dtype,
                                              int32_t training, float momentum, float eps, void* workspace, void* stream,
                                              void* side_stream, void* fork_event, void* join_event, int32_t expert_algo) {
  return omni::moe_fwd(x, gate_weight, up_weight, down_weight, router_weight_x, router_weight_y, running_mean_x, running_var_x, num_batches_tracked_x, running_mean_y, running_var_y,
                       num_batches_tracked_y, up_embed, down_embed, y, num_tokens, hidden_size, intermediate_size, num_experts, num_expert_sqrt, num_experts_per_token, dtype,
                       stats_dtype, training, momentum, eps, workspace, stream, side_stream, fork_event, join_event, expert_algo, nullptr);
}

// workspace: expert output [T,H] | expert workspace | partial sums of the MLP
extern "C" OMNI_API size_t omni_moe_save_workspace_bytes(int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size, int64_t num_experts, int32_t num_experts_per_token,
                                                         int32_t dtype) {
  using namespace omni;
  if (num_tokens < 0 || hidden_size <= 0 || intermediate_size <= 0 || num_experts_per_token < 0) return 0;
  return up256((size_t)num_tokens * (size_t)hidden_size * elem_bytes(dtype)) +
         up256(omni_expert_workspace_bytes(num_tokens, hidden_size, num_experts, num_experts_per_token, dtype, OMNI_EXPERT_ALGO_AUTO)) +
         up256(mlp_sums_bytes(num_tokens, hidden_size, intermediate_size, dtype));
}

extern "C" OMNI_API int32_t omni_moe_save_fwd(const void* x, const void* gate_weight, const void* up_weight, const void* down_weight,
                                              const void* router_weight_x, const void* router_weight_y,
                                              void* running_mean_x, void* running_var_x, int64_t* num_batches_tracked_x,
                                              void* running_mean_y, void* running_var_y, int64_t* num_batches_tracked_y,
                                              const void* up_embed, const void* down_embed, void* y,
                                              void* router_workspace, void* gates, int32_t* indices, float* scores, void* gate, void* up, void* h,
                                              int64_t num_tokens, int32_t hidden_size, int32_t intermediate_size, int64_t num_experts,
                                              int32_t num_expert_sqrt, int32_t num_experts_per_token, int32_t dtype, int32_t stats_dtype,
                                              int32_t training, float momentum, float eps, void* workspace, void* stream,
                                              void* side_stream, void* fork_event, void* join_event) {
  if (num_tokens > 0 && (!router_workspace || !gates || !indices || !gate || !up || !h)) return OMNI_ERR_NULL;
  const omni::Kept kept{router_workspace, gates, indices, scores, gate, up, h};
  return omni::moe_fwd(x, gate_weight, up_weight, down_weight, router_weight_x, router_weight_y, running_mean_x, running_var_x, num_batches_tracked_x, running_mean_y, running_var_y,
                       num_batches_tracked_y, up_embed, down_embed, y, num_tokens, hidden_size, intermediate_size, num_experts, num_expert_sqrt, num_experts_per_token, dtype,
                       stats_dtype, training, momentum, eps, workspace, stream, side_stream, fork_event, join_event, OMNI_EXPERT_ALGO_AUTO, &kept);
}
