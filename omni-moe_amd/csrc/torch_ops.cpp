// Host path of the operators for PyTorch: argument checks, allocation of outputs and workspaces, and the autograd nodes, in
// front of the C ABI of include/omni_moe_hip.h.  No kernel is launched from here except through that ABI.
//
// Why it is native: at a few hundred tokens the layer's kernels take 20-60 us, and the same work in Python -- attribute look-ups
// of a dozen parameters, shape checks, torch.empty, ctypes conversion -- took 47 us a call (a differentiable step, whose
// operators were Python autograd functions: 660 us for 246 us of kernels).
//
// Each entry takes the case that a program meets call after call: tensors on one GPU, contiguous, of one dtype, of matching
// shapes.  For anything else it returns None and the Python function in front of it goes on: it makes tensors contiguous, and
// it raises the errors that the operator contract names.
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/extension.h>

#include <algorithm>
#include <atomic>
#include <cmath>

#include "omni_moe_hip.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;

namespace {

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return OMNI_BF16;
    case at::kHalf: return OMNI_F16;
    case at::kFloat: return OMNI_F32;
    default: return -1;
  }
}

// on the GPU of `like`, contiguous, of its dtype
bool same(const Tensor& t, const Tensor& like) {
  return t.defined() && t.layout() == at::kStrided && t.scalar_type() == like.scalar_type() && t.device() == like.device() && t.is_contiguous();
}
bool is(const Tensor& t, std::initializer_list<int64_t> shape) { return t.sizes() == at::IntArrayRef(shape.begin(), shape.size()); }
bool on_gpu(const Tensor& t) { return t.defined() && t.layout() == at::kStrided && t.is_cuda() && t.is_contiguous() && dtype_code(t.scalar_type()) >= 0; }

// omni_init() once per device, before anything is launched there
bool prepare(const at::Device& dev) {
  static std::atomic<uint64_t> done{0};
  const uint64_t bit = 1ull << (dev.index() & 63);
  if (done.load(std::memory_order_acquire) & bit) return true;
  const c10::DeviceGuard guard(dev);
  if (omni_init() != OMNI_OK) return false;       // the Python path reports it
  done.fetch_or(bit, std::memory_order_release);
  return true;
}

void* stream_of(const at::Device& dev) { return (void*)c10::hip::getCurrentHIPStream(dev.index()).stream(); }
void* ptr(const Tensor& t) { return t.defined() && t.numel() ? t.data_ptr() : nullptr; }
Tensor bytes(size_t n, const at::Device& dev) { return at::empty({(int64_t)(n ? n : 1)}, at::TensorOptions().dtype(at::kByte).device(dev)); }

// A HIP error keeps the type that the Python path raises for it, from the autograd engine's threads too: torch translates what derives from PyTorchError.
PyObject* hip_error_type = nullptr;               // OmniHipError, handed over at load
struct HipError : torch::PyTorchError {
  using PyTorchError::PyTorchError;
  PyObject* python_type() override { return hip_error_type ? hip_error_type : PyExc_RuntimeError; }
};
struct TopkError : torch::PyTorchError {
  using PyTorchError::PyTorchError;
  PyObject* python_type() override { return PyExc_AssertionError; }      // the reference asserts (utils.py:81-104)
};

[[noreturn]] void raise(int32_t code, const char* what) {
  const std::string text = std::string(what) + ": " + omni_error_string(code), full = text + " (code " + std::to_string(code) + ")";
  if (code == OMNI_ERR_TOPK) throw TopkError(text);
  if (code >= 0) throw HipError(full);
  C10_THROW_ERROR(ValueError, full);
}
inline void check(int32_t code, const char* what) {
  if (code != OMNI_OK) raise(code, what);
}

bool records(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

// ---- expert op -------------------------------------------------------------------------------------
// x: T rows; gates, ids: [T, k]; scores: NULL, or where the pair scores that a backward pass takes over are put
Tensor expert_forward(const Tensor& x, int64_t T, const Tensor& up, const Tensor& down, const void* gates, const void* ids, int64_t k, int algo, void* scores) {
  const int64_t H = up.size(1), N = up.size(0);
  const int dt = dtype_code(x.scalar_type());
  Tensor y = at::empty_like(x);
  const size_t need = omni_expert_workspace_bytes(T, (int32_t)H, N, (int32_t)k, dt, algo);
  Tensor ws = need ? bytes(need, x.device()) : Tensor();
  check(omni_expert_fwd_scores(ptr(x), ptr(up), ptr(down), gates, (const int32_t*)ids, ptr(y), (float*)scores, T, (int32_t)H, N, (int32_t)k,
                               dt, algo, ptr(ws), stream_of(x.device())), "omni_expert_fwd");
  return y;
}

struct ExpertFn : public torch::autograd::Function<ExpertFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& up, const Tensor& down, const Tensor& gates, const Tensor& ids) {
    Tensor scores;                                 // kept where the backward pass reads them
    if (omni_expert_bwd_reads_scores(x.size(0), (int32_t)x.size(1), up.size(0), (int32_t)ids.size(1), dtype_code(x.scalar_type())))
      scores = at::empty(ids.sizes(), x.options().dtype(at::kFloat));
    Tensor y = expert_forward(x, x.size(0), up, down, ptr(gates), ptr(ids), ids.size(1), OMNI_EXPERT_ALGO_AUTO, ptr(scores));
    variable_list kept{x, up, down, gates, ids};
    if (scores.defined()) kept.push_back(scores);
    ctx->save_for_backward(kept);
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &up = s[1], &down = s[2], &gates = s[3], &ids = s[4];
    if (!grads[0].defined()) return {Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    const c10::DeviceGuard guard(x.device());
    const Tensor dy = grads[0].contiguous();
    const int64_t T = x.size(0), H = x.size(1), N = up.size(0), k = ids.size(1);
    const int dt = dtype_code(x.scalar_type());
    Tensor dx = at::empty_like(x), dup = at::empty_like(up), ddown = at::empty_like(down), dg = at::empty_like(gates);
    Tensor ws = bytes(omni_expert_bwd_workspace_bytes(T, (int32_t)H, N, (int32_t)k, dt), x.device());
    check(omni_expert_bwd_scores(ptr(dy), ptr(x), ptr(up), ptr(down), ptr(gates), (const int32_t*)ptr(ids), s.size() > 5 ? (const float*)ptr(s[5]) : nullptr, ptr(dx), ptr(dup), ptr(ddown), ptr(dg), T,
                                 (int32_t)H, N, (int32_t)k, dt, ptr(ws), stream_of(x.device())), "omni_expert_bwd");
    return {dx, dup, ddown, dg, Tensor()};
  }
};

py::object expert(const Tensor& x, const Tensor& up, const Tensor& down, const Tensor& gates, const Tensor& ids, int algo) {
  if (!on_gpu(x) || x.dim() != 2 || !same(up, x) || !same(down, x) || !same(gates, x) || up.dim() != 2 || gates.dim() != 2) return py::none();
  if (ids.scalar_type() != at::kInt || ids.device() != x.device() || !ids.is_contiguous() || ids.sizes() != gates.sizes()) return py::none();
  if (gates.size(0) != x.size(0) || down.sizes() != up.sizes() || up.size(1) != x.size(1) || !prepare(x.device())) return py::none();
  const bool grad = records({&x, &up, &down, &gates});
  if (grad && algo > OMNI_EXPERT_ALGO_GATHER) return py::none();
  Tensor y;
  {
    py::gil_scoped_release nogil;
    const c10::DeviceGuard guard(x.device());
    y = grad ? ExpertFn::apply(x, up, down, gates, ids) : expert_forward(x, x.size(0), up, down, ptr(gates), ptr(ids), ids.size(1), algo, nullptr);
  }
  return py::cast(y);
}

// ---- router ----------------------------------------------------------------------------------------
py::object router_select(const Tensor& lx, const Tensor& ly, int64_t r, int64_t k) {
  if (!on_gpu(lx) || lx.dim() != 2 || lx.size(1) != r || !same(ly, lx) || ly.sizes() != lx.sizes()) return py::none();
  if (k < 0 || k > r * r || k > 128 || k % 2 || records({&lx, &ly}) || !prepare(lx.device())) return py::none();
  py::gil_scoped_release nogil;
  const c10::DeviceGuard guard(lx.device());
  const int64_t T = lx.size(0);
  Tensor scores = at::empty({T, k}, lx.options()), ids = at::empty({T, k}, lx.options().dtype(at::kInt));
  check(omni_router_select(ptr(lx), ptr(ly), ptr(scores), (int32_t*)ptr(ids), T, (int32_t)r, (int32_t)k, dtype_code(lx.scalar_type()), stream_of(lx.device())),
        "omni_router_select");
  py::gil_scoped_acquire gil;
  return py::make_tuple(scores, ids);
}

// The running statistics of the two norms as the library takes them: six pointers, one dtype.
struct Norms {
  Tensor rmx, rvx, nbx, rmy, rvy, nby;
  bool training = false;
  double momentum = 0.1, eps = 1e-5;
  // what the operator contract asks of them, for r keys and T tokens beside x
  bool fits(const Tensor& x, int64_t r, int64_t T) const {
    const int64_t shape[1] = {r};
    for (const Tensor* t : {&rmx, &rvx, &rmy, &rvy})
      if (!t->defined() || t->sizes() != at::IntArrayRef(shape, 1) || t->scalar_type() != rmx.scalar_type() || t->device() != x.device() || !t->is_contiguous()) return false;
    for (const Tensor* t : {&nbx, &nby})
      if (t->defined() && (t->scalar_type() != at::kLong || t->numel() != 1 || t->device() != x.device())) return false;
    return dtype_code(rmx.scalar_type()) >= 0 && !(training && T == 1);
  }
};

void router_forward(const Tensor& x, int64_t T, int64_t H, const Tensor& wx, const Tensor& wy, const Norms& n, int64_t k, void* gates, void* ids, void* ws) {
  const int64_t r = wx.size(0);
  check(omni_router_fwd(ptr(x), ptr(wx), ptr(wy), ptr(n.rmx), ptr(n.rvx), (int64_t*)ptr(n.nbx), ptr(n.rmy), ptr(n.rvy), (int64_t*)ptr(n.nby), n.training ? 1 : 0,
                        (float)n.momentum, (float)n.eps, gates, (int32_t*)ids, nullptr, T, (int32_t)H, (int32_t)r, (int32_t)k, dtype_code(x.scalar_type()),
                        dtype_code(n.rmx.scalar_type()), ws, stream_of(x.device())), "omni_router_fwd");
}

py::object router_stage(const Tensor& x, const Tensor& wx, const Tensor& wy, const Tensor& rmx, const Tensor& rvx, const c10::optional<Tensor>& nbx,
                        const Tensor& rmy, const Tensor& rvy, const c10::optional<Tensor>& nby, int64_t k, bool training, double momentum, double eps) {
  if (!on_gpu(x) || x.dim() != 2 || !same(wx, x) || !same(wy, x) || wx.dim() != 2 || wx.sizes() != wy.sizes() || wx.size(1) != x.size(1)) return py::none();
  const Norms n{rmx, rvx, nbx.value_or(Tensor()), rmy, rvy, nby.value_or(Tensor()), training, momentum, eps};
  const int64_t r = wx.size(0);
  if (k < 0 || k > r * r || k > 128 || k % 2 || !n.fits(x, r, x.size(0)) || records({&x, &wx, &wy}) || !prepare(x.device())) return py::none();
  py::gil_scoped_release nogil;
  const c10::DeviceGuard guard(x.device());
  const int64_t T = x.size(0);
  Tensor gates = at::empty({T, k}, x.options()), ids = at::empty({T, k}, x.options().dtype(at::kInt));
  Tensor ws = bytes(omni_router_workspace_bytes(T, (int32_t)r, dtype_code(x.scalar_type())), x.device());
  router_forward(x, T, x.size(1), wx, wy, n, k, ptr(gates), ptr(ids), ptr(ws));
  py::gil_scoped_acquire gil;
  return py::make_tuple(gates, ids);
}

// ---- shared MLP ------------------------------------------------------------------------------------
py::object mlp(const Tensor& x, const Tensor& wg, const Tensor& wu, const Tensor& wd, const c10::optional<Tensor>& residual) {
  if (!on_gpu(x) || x.dim() != 2 || !same(wg, x) || !same(wu, x) || !same(wd, x) || wg.dim() != 2) return py::none();
  const int64_t T = x.size(0), H = x.size(1), I = wg.size(0);
  const Tensor res = residual.value_or(Tensor());
  if (!is(wg, {I, H}) || !is(wu, {I, H}) || !is(wd, {H, I}) || (res.defined() && (!same(res, x) || res.sizes() != x.sizes()))) return py::none();
  if (records({&x, &wg, &wu, &wd, &res}) || !prepare(x.device())) return py::none();
  Tensor y;
  {
    py::gil_scoped_release nogil;
    const c10::DeviceGuard guard(x.device());
    const int dt = dtype_code(x.scalar_type());
    y = at::empty_like(x);
    Tensor ws = bytes(omni_mlp_workspace_bytes(T, (int32_t)H, (int32_t)I, dt), x.device());
    check(omni_mlp_fwd(ptr(x), ptr(wg), ptr(wu), ptr(wd), ptr(res), ptr(y), T, (int32_t)H, (int32_t)I, dt, ptr(ws), stream_of(x.device())), "omni_mlp_fwd");
  }
  return py::cast(y);
}

// ---- the layer -------------------------------------------------------------------------------------
struct Layer {
  Tensor wg, wu, wd, rx, ry, up, down;
  Norms norms;
  int64_t H = 0, I = 0, N = 0, r = 0, k = 0;
  void *side = nullptr, *fork = nullptr, *join = nullptr;      // the second stream and its events, where the call takes one
};

// What the forward pass leaves for the backward one, in ONE allocation (as are the backward pass's temporaries): a step of 1000 tokens with
// hidden 512 is bound by the host, and two dozen allocations and fifteen saved tensors cost it a fifth of its time (195-205 -> 160-168 us).
struct Slab {
  size_t size = 0;
  size_t add(size_t n) {
    const size_t at = size;
    size += (n + 255) / 256 * 256;
    return at;
  }
};
struct Kept {     // gates and ids, the router's workspace (z and the statistics), pair scores where the backward pass reads them, rounded gate and up projections, their SwiGLU product
  Slab s;
  size_t gates, ids, router, scores, gate, up, h;
  bool scored;
  Kept(int64_t T, int64_t H, int64_t I, int64_t N, int64_t r, int64_t k, int dt) : scored(omni_expert_bwd_reads_scores(T, (int32_t)H, N, (int32_t)k, dt) != 0) {
    const size_t es = dt == OMNI_F32 ? 4 : 2, pairs = (size_t)(T * k), wide = (size_t)(T * I) * es;
    gates = s.add(pairs * es); ids = s.add(pairs * 4); router = s.add(omni_router_workspace_bytes(T, (int32_t)r, dt)); scores = s.add(scored ? pairs * 4 : 0);
    gate = s.add(wide); up = s.add(wide); h = s.add(wide);
  }
};
// [rows, cols] of dtype `like`, `at` bytes into the slab
Tensor part(const Tensor& slab, size_t at, int64_t rows, int64_t cols, const Tensor& like) {
  return slab.narrow(0, (int64_t)at, rows * cols * like.element_size()).view(like.scalar_type()).view({rows, cols});
}

// One differentiable node for the whole layer (reference omni_moe.py:64-104).
struct LayerFn : public torch::autograd::Function<LayerFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& wg, const Tensor& wu, const Tensor& wd, const Tensor& rx, const Tensor& ry,
                        const Tensor& up, const Tensor& down, const Layer& l) {
    const int64_t T = x.numel() / l.H;
    const int dt = dtype_code(x.scalar_type());
    const Kept at(T, l.H, l.I, l.N, l.r, l.k, dt);
    const Tensor kept = bytes(at.s.size, x.device());
    uint8_t* k = (uint8_t*)ptr(kept);
    // given back at the end of the call: the current stream waits for a side branch, as below
    const Tensor ws = bytes(omni_moe_save_workspace_bytes(T, (int32_t)l.H, (int32_t)l.I, l.N, (int32_t)l.k, dt), x.device());
    Tensor y = at::empty(x.sizes(), x.options());
    const Norms& b = l.norms;
    check(omni_moe_save_fwd(ptr(x), ptr(wg), ptr(wu), ptr(wd), ptr(rx), ptr(ry), ptr(b.rmx), ptr(b.rvx), (int64_t*)ptr(b.nbx), ptr(b.rmy), ptr(b.rvy), (int64_t*)ptr(b.nby), ptr(up),
                            ptr(down), ptr(y), k + at.router, k + at.gates, (int32_t*)(k + at.ids), at.scored ? (float*)(k + at.scores) : nullptr, k + at.gate, k + at.up, k + at.h, T,
                            (int32_t)l.H, (int32_t)l.I, l.N, (int32_t)l.r, (int32_t)l.k, dt, dtype_code(b.rmx.scalar_type()), b.training ? 1 : 0, (float)b.momentum, (float)b.eps,
                            ptr(ws), stream_of(x.device()), l.side, l.fork, l.join), "omni_moe_save_fwd");
    ctx->save_for_backward({x, wg, wu, wd, rx, ry, up, down, kept});
    ctx->saved_data["training"] = l.norms.training;
    ctx->saved_data["top_k"] = l.k;
    return y;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x3 = s[0], &wg = s[1], &wu = s[2], &wd = s[3], &rx = s[4], &ry = s[5], &up = s[6], &down = s[7], &kept = s[8];
    if (!grads[0].defined()) return variable_list(9);
    const c10::DeviceGuard guard(x3.device());
    const int64_t H = wg.size(1), I = wg.size(0), N = up.size(0), r = rx.size(0), k = ctx->saved_data["top_k"].toInt(), T = x3.numel() / H;
    const bool training = ctx->saved_data["training"].toBool();
    const int dt = dtype_code(x3.scalar_type());
    void* st = stream_of(x3.device());
    const Tensor dy = grads[0].contiguous();
    bool need[8];
    for (int i = 0; i < 8; ++i) need[i] = ctx->needs_input_grad(i);
    variable_list out(9);
    const bool own = dt != OMNI_F32, router = need[0] || need[4] || need[5];        // 16-bit products are the library's own
    const int64_t rp = own ? (r + 7) / 8 * 8 : r;
    const Kept at(T, H, I, N, r, k, dt);
    const uint8_t* saved = (const uint8_t*)ptr(kept);
    // temporaries: the experts' d(x), d(gates), d(z), and one workspace for two stages that follow one another on the stream
    Slab t;
    const size_t es = own ? 2 : 4, dx_at = t.add((size_t)(T * H) * es), dg_at = t.add((size_t)(T * k) * es), dz_at = t.add(router ? (size_t)(T * 2 * rp) * es : 0);
    const size_t ws_at = t.add(std::max(router ? omni_expert_router_bwd_workspace_bytes(T, (int32_t)H, N, (int32_t)r, (int32_t)k, dt)
                                               : omni_expert_bwd_workspace_bytes(T, (int32_t)H, N, (int32_t)k, dt),
                                        own ? omni_mlp_bwd_workspace_bytes(T, (int32_t)H, (int32_t)I, (int32_t)r, dt) : 0));
    const Tensor temp = bytes(t.size, x3.device());
    uint8_t* w = (uint8_t*)ptr(temp);
    // experts, and the router stage behind their gates' gradient
    Tensor dup = at::empty_like(up), ddown = at::empty_like(down);
    const float* scores = at.scored ? (const float*)(saved + at.scores) : nullptr;
    const int32_t* ids = (const int32_t*)(saved + at.ids);
    if (router) {
      const uint8_t* z = saved + at.router;
      check(omni_expert_router_bwd(ptr(dy), ptr(x3), ptr(up), ptr(down), saved + at.gates, ids, scores, z, (const float*)(z + omni_router_workspace_stats_offset(T, (int32_t)r, dt)),
                                   w + dx_at, ptr(dup), ptr(ddown), w + dg_at, w + dz_at, T, (int32_t)H, N, (int32_t)r, (int32_t)k, dt, training ? 1 : 0, own ? 1 : 0, w + ws_at, st),
            "omni_expert_router_bwd");
    } else {
      check(omni_expert_bwd_scores(ptr(dy), ptr(x3), ptr(up), ptr(down), saved + at.gates, ids, scores, w + dx_at, ptr(dup), ptr(ddown), w + dg_at, T, (int32_t)H, N, (int32_t)k, dt,
                                   w + ws_at, st), "omni_expert_bwd");
    }
    if (need[6]) out[6] = dup;
    if (need[7]) out[7] = ddown;
    if (own) {
      const Tensor* like[6] = {&x3, &wg, &wu, &wd, &rx, &ry};
      for (int i = 0; i < 6; ++i)
        if (need[i]) out[i] = at::empty_like(*like[i]);
      const int32_t code = omni_mlp_bwd(ptr(dy), ptr(x3), ptr(wg), ptr(wu), ptr(wd), saved + at.gate, saved + at.up, saved + at.h, router ? w + dz_at : nullptr, ptr(rx),
                                        ptr(ry), w + dx_at, ptr(out[0]), ptr(out[1]), ptr(out[2]), ptr(out[3]), ptr(out[4]), ptr(out[5]), T, (int32_t)H, (int32_t)I,
                                        (int32_t)r, dt, w + ws_at, st);
      if (code != OMNI_ERR_UNSUPPORTED) {
        check(code, "omni_mlp_bwd");
        return out;
      }
    }
    // single precision, operands off a 16-byte boundary, and operands of 2 GiB and more: library products
    const Tensor x = x3.view({T, H}), dy2 = dy.view({T, H}), gate = part(kept, at.gate, T, I, x3), upp = part(kept, at.up, T, I, x3);
    Tensor dx = part(temp, dx_at, T, H, x3);
    if (router) {
      const Tensor dz = part(temp, dz_at, T, 2 * rp, x3), zx = dz.narrow(1, 0, r), zy = dz.narrow(1, rp, r);
      if (need[4]) out[4] = at::mm(zx.t(), x);
      if (need[5]) out[5] = at::mm(zy.t(), x);
      if (need[0]) dx = at::addmm(dx, zx, rx).addmm_(zy, ry);                       // (a tensor of its own)
    }
    if (need[3]) out[3] = at::mm(dy2.t(), part(kept, at.h, T, I, x3));
    if (need[0] || need[1] || need[2]) {
      const Tensor dh = at::mm(dy2, wd);
      Tensor dgate = at::empty_like(gate), dupp = at::empty_like(upp);
      check(omni_swiglu_bwd(ptr(dh), ptr(gate), ptr(upp), ptr(dgate), ptr(dupp), T * I, dt, st), "omni_swiglu_bwd");
      if (need[1]) out[1] = at::mm(dgate.t(), x);
      if (need[2]) out[2] = at::mm(dupp.t(), x);
      if (need[0]) dx.addmm_(dgate, wg).addmm_(dupp, wu);
    }
    if (need[0]) out[0] = dx.view(x3.sizes());
    return out;
  }
};

// Attribute names, interned once.
struct Names {
  PyObject *modules, *parameters, *buffers, *weight, *training, *momentum, *eps, *running_mean, *running_var, *tracked, *norm_x, *norm_y, *overlap, *min_work, *max_work,
      *algo, *resources, *top_k, *hidden, *cuda_stream, *cuda_event;
  PyObject* layers[7];
  Names() {
    auto in = [](const char* s) { return PyUnicode_InternFromString(s); };
    modules = in("_modules"); parameters = in("_parameters"); buffers = in("_buffers"); weight = in("weight"); training = in("training"); momentum = in("momentum");
    eps = in("eps"); running_mean = in("running_mean"); running_var = in("running_var"); tracked = in("num_batches_tracked"); norm_x = in("router_norm_x");
    norm_y = in("router_norm_y"); overlap = in("overlap_branches"); min_work = in("overlap_min_work"); max_work = in("overlap_max_work"); algo = in("expert_algo");
    resources = in("_branch_resources"); top_k = in("top_k"); hidden = in("hidden_size"); cuda_stream = in("cuda_stream"); cuda_event = in("cuda_event");
    const char* l[7] = {"gate_proj", "up_proj", "down_proj", "router_gate_x", "router_gate_y", "up_embed", "down_embed"};
    for (int i = 0; i < 7; ++i) layers[i] = in(l[i]);
  }
};

// The entry of a module's own dictionaries, as a borrowed reference (or NULL): what nn.Module.__getattr__ would find, without its search
PyObject* item(PyObject* dict, PyObject* name) { return dict && PyDict_Check(dict) ? PyDict_GetItemWithError(dict, name) : nullptr; }
PyObject* dict_of(PyObject* o) {
  PyObject** d = o ? _PyObject_GetDictPtr(o) : nullptr;
  return d ? *d : nullptr;
}
bool tensor_at(PyObject* module, PyObject* group, PyObject* name, Tensor& out, bool may_be_none = false) {
  PyObject* t = item(item(dict_of(module), group), name);
  if (t && t == Py_None && may_be_none) return true;
  if (!t || !THPVariable_Check(t)) return false;
  out = THPVariable_Unpack(t);
  return true;
}

// OmniMoE.forward of the plain module.  `algos`: expert_algo name -> code.
py::object layer_forward(py::handle self, const Tensor& x, const py::dict& algos) {
  static const Names n;
  PyObject* own = dict_of(self.ptr());
  PyObject* modules = item(own, n.modules);
  if (!modules || !on_gpu(x) || x.dim() != 3) return py::none();
  Layer l;
  Tensor* w[7] = {&l.wg, &l.wu, &l.wd, &l.rx, &l.ry, &l.up, &l.down};
  for (int i = 0; i < 7; ++i)
    if (!tensor_at(item(modules, n.layers[i]), n.parameters, n.weight, *w[i]) || !same(*w[i], x) || w[i]->dim() != 2) return py::none();
  PyObject *nx = item(modules, n.norm_x), *ny = item(modules, n.norm_y);
  Norms& b = l.norms;
  if (!tensor_at(nx, n.buffers, n.running_mean, b.rmx) || !tensor_at(nx, n.buffers, n.running_var, b.rvx) || !tensor_at(nx, n.buffers, n.tracked, b.nbx, true) ||
      !tensor_at(ny, n.buffers, n.running_mean, b.rmy) || !tensor_at(ny, n.buffers, n.running_var, b.rvy) || !tensor_at(ny, n.buffers, n.tracked, b.nby, true))
    return py::none();
  auto number = [](PyObject* o, double& v) { return o && (PyFloat_Check(o) || PyLong_Check(o)) && ((v = PyFloat_AsDouble(o)), !PyErr_Occurred()); };
  double mx, my, ex, ey, hidden, top_k;
  if (!number(item(dict_of(nx), n.momentum), mx) || !number(item(dict_of(ny), n.momentum), my) || !number(item(dict_of(nx), n.eps), ex) ||
      !number(item(dict_of(ny), n.eps), ey) || mx != my || ex != ey || !number(item(own, n.hidden), hidden) || !number(item(own, n.top_k), top_k)) {
    PyErr_Clear();
    return py::none();
  }
  b.training = item(own, n.training) == Py_True;
  b.momentum = mx;
  b.eps = ex;
  const int64_t T = x.size(0) * x.size(1);
  l.H = (int64_t)hidden; l.I = l.wg.size(0); l.N = l.up.size(0); l.r = l.rx.size(0); l.k = (int64_t)top_k;
  if (x.size(2) != l.H || T == 0 || !is(l.wg, {l.I, l.H}) || !is(l.wu, {l.I, l.H}) || !is(l.wd, {l.H, l.I}) || !is(l.rx, {l.r, l.H}) || !is(l.ry, {l.r, l.H}) ||
      !is(l.up, {l.N, l.H}) || !is(l.down, {l.N, l.H}) || l.k < 0 || l.k > l.r * l.r || l.k > 128 || l.k % 2 || !b.fits(x, l.r, T) || !prepare(x.device()))
    return py::none();
  const py::object overlap = py::reinterpret_steal<py::object>(PyObject_GetAttr(self.ptr(), n.overlap)), low = py::reinterpret_steal<py::object>(PyObject_GetAttr(self.ptr(), n.min_work)),
                   high = py::reinterpret_steal<py::object>(PyObject_GetAttr(self.ptr(), n.max_work)), name = py::reinterpret_steal<py::object>(PyObject_GetAttr(self.ptr(), n.algo));
  if (!overlap || !low || !high || !name) throw py::error_already_set();
  const double work = (double)T * (double)l.H * (double)l.I;
  if (PyObject_IsTrue(overlap.ptr()) == 1 && low.cast<double>() < work && work < high.cast<double>()) {
    const py::tuple res = self.attr(py::handle(n.resources))(py::cast(x.device()));
    auto handle = [](py::handle o, PyObject* attr) { return (void*)(uintptr_t)o.attr(py::handle(attr)).cast<uint64_t>(); };
    l.side = handle(res[0], n.cuda_stream); l.fork = handle(res[1], n.cuda_event); l.join = handle(res[2], n.cuda_event);
  }
  if (records({&x, &l.wg, &l.wu, &l.wd, &l.rx, &l.ry, &l.up, &l.down})) {
    Tensor y;
    {
      py::gil_scoped_release nogil;
      const c10::DeviceGuard guard(x.device());
      y = LayerFn::apply(x, l.wg, l.wu, l.wd, l.rx, l.ry, l.up, l.down, l);
    }
    return py::cast(y);
  }
  PyObject* algo_code = PyDict_GetItemWithError(algos.ptr(), name.ptr());
  if (!algo_code) { PyErr_Clear(); return py::none(); }
  const int algo = (int)PyLong_AsLong(algo_code);
  Tensor y;
  {
    py::gil_scoped_release nogil;
    const c10::DeviceGuard guard(x.device());
    const at::AutoDispatchBelowADInplaceOrView below;
    const int dt = dtype_code(x.scalar_type());
    y = at::empty(x.sizes(), x.options());
    // given back at the end of the call: the current stream has been made to wait for the side branch, so every later use of
    // that memory (allocated from this stream's pool) is ordered after both branches
    Tensor ws = bytes(omni_moe_workspace_bytes_algo(T, (int32_t)l.H, (int32_t)l.I, l.N, (int32_t)l.r, (int32_t)l.k, dt, algo), x.device());
    check(omni_moe_fwd_algo(ptr(x), ptr(l.wg), ptr(l.wu), ptr(l.wd), ptr(l.rx), ptr(l.ry), ptr(b.rmx), ptr(b.rvx), (int64_t*)ptr(b.nbx), ptr(b.rmy), ptr(b.rvy),
                            (int64_t*)ptr(b.nby), ptr(l.up), ptr(l.down), ptr(y), T, (int32_t)l.H, (int32_t)l.I, l.N, (int32_t)l.r, (int32_t)l.k, dt,
                            dtype_code(b.rmx.scalar_type()), b.training ? 1 : 0, (float)b.momentum, (float)b.eps, ptr(ws), stream_of(x.device()), l.side, l.fork, l.join, algo),
          "omni_moe_fwd_algo");
  }
  return py::cast(y);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("hip_error_type", [](py::object type) { hip_error_type = type.release().ptr(); });
  m.def("check", [](int32_t code, const std::string& what) { check(code, what.c_str()); });
  m.def("expert", &expert);
  m.def("router_select", &router_select);
  m.def("router_stage", &router_stage);
  m.def("mlp", &mlp);
  m.def("layer_forward", &layer_forward);
}
