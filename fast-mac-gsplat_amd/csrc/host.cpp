// host.cpp -- the host path of the per-step calls in C++: argument checks,
// buffers, the launches' C-ABI calls, the wait for the binning's report and
// the autograd nodes of the rasterizer and the projection.
//
// A training step of a small scene is host bound: 30 us of kernels took 200 us
// of Python calls, ctypes conversions, tensor allocations and autograd nodes
// run under the interpreter lock.  Here one call from Python does the forward,
// and the backward nodes run without the interpreter.
//
// What is not the plain case returns None from Plan.run / project, and the
// Python path takes it, with its messages: inputs that fail a check, tensors
// that are not plain ones (subclasses, functorch and dispatch-mode wrappers,
// forward-mode duals), batches to be split, the first binning of a shape,
// images above the two-launch depth order, dense scenes to be sliced, staged
// timing.
#include <ATen/SavedTensorHooks.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/PythonDispatcherTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <memory>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "../../include/gsplat_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The C ABI, from the library that the Python layer has loaded.
#define GS_API(F)                       \
  F(last_error)                         \
  F(bin_workspace_bytes)                \
  F(render_workspace_bytes)             \
  F(bin_render_forward)                 \
  F(render_forward_long)                \
  F(render_backward)                    \
  F(direct_workspace_bytes)             \
  F(direct_pairs)                       \
  F(direct_render)                      \
  F(tile_workspace_bytes)               \
  F(tile_render)                        \
  F(project_forward)                    \
  F(project_backward)                   \
  F(project_backward_workspace_bytes)
struct Api {
#define GS_POINTER(name) decltype(&gsplat_hip_##name) name = nullptr;
  GS_API(GS_POINTER)
#undef GS_POINTER
} api;

void bind(const std::string& path) {
  void* h = dlopen(path.c_str(), RTLD_NOW | RTLD_NOLOAD);
  TORCH_CHECK(h != nullptr, "libgsplat_hip.so is not loaded: ", dlerror());
#define GS_RESOLVE(name)                                                  \
  api.name = reinterpret_cast<decltype(&gsplat_hip_##name)>(              \
      dlsym(h, "gsplat_hip_" #name));                                     \
  TORCH_CHECK(api.name != nullptr, "gsplat_hip_" #name " is not exported");
  GS_API(GS_RESOLVE)
#undef GS_RESOLVE
}

void check(int rc, const char* what) {
  if (rc == 0) return;
  const char* msg = api.last_error();
  TORCH_CHECK(false, what, " failed (status ", rc, "): ", msg ? msg : "");
}

hipStream_t stream_of(const Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

constexpr int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }

const float* f32(const Tensor& t) { return t.data_ptr<float>(); }

// A tensor the C++ path takes: an ordinary strided float32 tensor in device
// memory, of a type whose operations nothing intercepts.
bool plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return false;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.scalar_type() != at::kFloat ||
      t.layout() != at::kStrided || !t.has_storage())
    return false;
  const auto ks = t.key_set();
  if (ks.has_any(c10::DispatchKeySet(
          {c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
           c10::DispatchKey::FuncTorchGradWrapper,
           c10::DispatchKey::Functionalize})) ||
      t.is_conj() || t.is_neg())
    return false;
  return !t._fw_grad(0).defined();
}

// Nothing that intercepts operations is active (modes, functorch, tracing).
bool plain_context() {
  return !c10::impl::dispatch_mode_enabled() &&
         c10::impl::PythonDispatcherTLS::get_state() == nullptr &&
         !c10::impl::tls_is_dispatch_key_included(
             c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !torch::jit::tracer::isTracing();
}

// Timing of a backward call by the Python layer (_ops.set_timing): the
// context manager _ops._timed, entered around the C-ABI call.
std::atomic<bool> g_timed{false};
struct Timed {
  PyObject* cm = nullptr;
  explicit Timed(const char* name) {
    if (!g_timed.load(std::memory_order_relaxed)) return;
    py::gil_scoped_acquire gil;
    py::object ops = py::module_::import("torch_gsplat_bridge_fast._ops");
    py::object c = ops.attr("_timed")(name);
    c.attr("__enter__")();
    cm = c.release().ptr();
  }
  ~Timed() {
    if (cm == nullptr) return;
    py::gil_scoped_acquire gil;
    try {
      py::object c = py::reinterpret_steal<py::object>(cm);
      c.attr("__exit__")(py::none(), py::none(), py::none());
    } catch (py::error_already_set& e) {
      e.discard_as_unraisable("gsplat timing");
    }
  }
};

// Pinned words for the binnings' reports: 1024 rows of {N, status, long-range
// flag, ready} per device, one per call.
struct Rows {
  static constexpr int kRows = 1024;
  Tensor words;
  std::atomic<uint32_t> calls{0};
  int32_t* next() {
    return words.data_ptr<int32_t>() + 4 * (calls.fetch_add(1) % kRows);
  }
};
Rows& rows_of(int device) {
  static std::mutex mu;
  static std::unordered_map<int, std::unique_ptr<Rows>> all;
  std::lock_guard<std::mutex> lock(mu);
  auto& r = all[device];
  if (!r) {
    r = std::make_unique<Rows>();
    r->words = at::zeros({Rows::kRows, 4}, at::dtype(at::kInt).pinned_memory(true));
  }
  return *r;
}

// Waits for a report's ready word without the interpreter lock.  After a
// second it synchronises the device (which fails if the device did) and
// requires the word to be set then.
void wait_report(const int32_t* row) {
  auto ready = [row] {
    return __atomic_load_n(row + 3, __ATOMIC_ACQUIRE) != 0;
  };
  const auto limit = std::chrono::steady_clock::now() + std::chrono::seconds(1);
  for (int spins = 1; !ready(); ++spins) {
    if ((spins & 1023) != 0) {
      __builtin_ia32_pause();
      continue;
    }
    if (std::chrono::steady_clock::now() < limit) continue;
    const hipError_t e = hipDeviceSynchronize();
    TORCH_CHECK(e == hipSuccess, "binning: ", hipGetErrorString(e));
    TORCH_CHECK(ready(), "binning: the device did not write its report to the host words");
  }
}

// ---- rasterizer

// Byte offsets of a call's buffers: kept for the backward {packed, pairs,
// tile offsets, tile stops, render workspace, end}, used by the forward only
// {perm, splat offsets, binning workspace, end}.
struct Sizes {
  std::array<int64_t, 6> keep;
  std::array<int64_t, 4> use;
};

// What a backward needs beside its tensors.
struct Saved : torch::CustomClassHolder {
  gsplat_raster_meta meta;
  std::array<int64_t, 6> keep;
  int64_t n_pairs = 0;
  std::array<std::vector<int64_t>, 5> shapes;  // of the inputs
  bool depth_grad = true;
};

enum class Mode { kDirect, kTiled, kBinned };

struct Call {
  gsplat_raster_meta meta;
  Sizes sizes;
  int64_t n_pairs = 0;  // pair capacity (direct: gsplat_hip_direct_pairs)
  Mode mode = Mode::kBinned;
  bool batched = false, depth_grad = true;
};

struct Result {
  Tensor img, final_T, last, kept;
  int32_t n = 0;  // N of a binned call
  bool skewed = false;  // a tiled call that is to be done by kBinned
};

Tensor bytes(int64_t n, const Tensor& like) {
  return at::empty({n}, like.options().dtype(at::kByte).requires_grad(false));
}

std::vector<int64_t> image_shape(const Call& c, bool rgb) {
  std::vector<int64_t> s;
  if (c.batched) s.push_back(c.meta.batch);
  s.push_back(c.meta.height);
  s.push_back(c.meta.width);
  if (rgb) s.push_back(3);
  return s;
}

// Binning and forward; with GIL held or not.  N above the capacity is left to
// the caller (the image is then incomplete).
Result render(const Call& c, const std::array<Tensor, 5>& in, bool train) {
  const Tensor& like = in[0];
  const auto opt = like.options().requires_grad(false);
  std::array<Tensor, 5> t;
  for (int k = 0; k < 5; ++k) t[k] = in[k].contiguous();
  Result r;
  r.kept = bytes(c.sizes.keep[5], like);
  Tensor used = bytes(c.sizes.use[3], like);
  r.img = at::empty(image_shape(c, true), opt);
  if (train) {
    r.final_T = at::empty(image_shape(c, false), opt);
    r.last = at::empty(image_shape(c, false), opt.dtype(at::kInt));
  }
  char* k = static_cast<char*>(r.kept.data_ptr());
  char* u = static_cast<char*>(used.data_ptr());
  const auto& ko = c.sizes.keep;
  const auto& uo = c.sizes.use;
  float* T = train ? r.final_T.data_ptr<float>() : nullptr;
  int32_t* last = train ? r.last.data_ptr<int32_t>() : nullptr;
  int32_t* stop = train ? reinterpret_cast<int32_t*>(k + ko[3]) : nullptr;
  auto* packed = reinterpret_cast<float*>(k + ko[0]);
  auto* pairs = reinterpret_cast<int32_t*>(k + ko[1]);
  auto* offsets = reinterpret_cast<int32_t*>(k + ko[2]);
  void* rws = k + ko[4];
  const size_t rws_bytes = (size_t)(ko[5] - ko[4]);
  hipStream_t s = stream_of(like);
  if (c.mode == Mode::kDirect) {
    check(api.direct_render(&c.meta, f32(t[0]), f32(t[1]), f32(t[2]), f32(t[3]),
                            f32(t[4]), packed, offsets, pairs,
                            r.img.data_ptr<float>(), T, last, stop, u + uo[2],
                            (size_t)(uo[3] - uo[2]), rws, rws_bytes, s),
          "gsplat_hip_direct_render");
    return r;
  }
  int32_t* row = rows_of(like.device().index()).next();
  if (c.mode == Mode::kTiled)
    check(api.tile_render(&c.meta, f32(t[0]), f32(t[1]), f32(t[2]), f32(t[3]),
                          f32(t[4]), c.n_pairs, packed, offsets, pairs, row,
                          r.img.data_ptr<float>(), T, last, stop, u + uo[2],
                          (size_t)(uo[3] - uo[2]), rws, rws_bytes, s),
          "gsplat_hip_tile_render");
  else
    check(api.bin_render_forward(
            &c.meta, f32(t[0]), f32(t[1]), f32(t[2]), f32(t[3]), f32(t[4]),
            c.n_pairs, reinterpret_cast<int32_t*>(u + uo[0]), packed,
            reinterpret_cast<int32_t*>(u + uo[1]), pairs, offsets, row,
            u + uo[2], (size_t)(uo[3] - uo[2]), r.img.data_ptr<float>(), T, last,
            stop, rws, rws_bytes, s, nullptr, nullptr, nullptr, nullptr),
        "gsplat_hip_bin_render_forward");
  if (PyGILState_Check()) {
    py::gil_scoped_release nogil;
    wait_report(row);
  } else {
    wait_report(row);
  }
  const int32_t status = row[1];
  TORCH_CHECK(!(status & GSPLAT_STATUS_LOOKBACK_TIMEOUT),
              "binning failed: a decoupled look-back wait gave up (a predecessor "
              "workgroup did not make progress for ~1 s); the results of this call "
              "are invalid");
  TORCH_CHECK(status == 0, "binning failed with device status ", status);
  r.n = row[0];
  TORCH_CHECK(r.n >= 0, "pair count overflowed int32");
  r.skewed = c.mode == Mode::kTiled && (row[2] & GSPLAT_TILE_SKEWED) != 0;
  if (r.n <= c.n_pairs && !r.skewed && row[2] != 0)
    check(api.render_forward_long(&c.meta, packed, offsets, pairs,
                                  r.img.data_ptr<float>(), T, last, stop,
                                  c.n_pairs, rws, rws_bytes, s),
          "gsplat_hip_render_forward_long");
  return r;
}

class Plan;
Call grown(Plan& plan, const Call& c, const Tensor& like, int32_t n, bool train);
Call unskewed(Plan& plan, const Call& c, const Tensor&, bool train);

// The forward with the pairs it found room for: binned again, once, when N was
// above the capacity of the shape's earlier calls.
Result render_all(Plan& plan, Call& c, const std::array<Tensor, 5>& in, bool train) {
  Result r = render(c, in, train);
  if (c.mode == Mode::kDirect) return r;
  if (r.skewed) {
    c = unskewed(plan, c, in[0], train);
    r = render(c, in, train);
  }
  const int32_t n = r.n;
  Call next = grown(plan, c, in[0], n, train);
  if (n <= c.n_pairs) return r;
  c = next;
  r = render(c, in, train);
  TORCH_CHECK(r.n <= c.n_pairs,
              "binning: pair count changed between two binnings of the same inputs");
  return r;
}

struct Rasterize : torch::autograd::Function<Rasterize> {
  static Tensor forward(AutogradContext* ctx, const Tensor& means2d,
                        const Tensor& conics, const Tensor& colors,
                        const Tensor& opacities, const Tensor& depths,
                        Plan* plan, Call* call) {
    const std::array<Tensor, 5> in{means2d, conics, colors, opacities, depths};
    Result r = render_all(*plan, *call, in, true);
    auto saved = c10::make_intrusive<Saved>();
    saved->meta = call->meta;
    saved->keep = call->sizes.keep;
    saved->n_pairs = call->n_pairs;
    saved->depth_grad = call->depth_grad;
    for (int k = 0; k < 5; ++k) saved->shapes[k] = in[k].sizes().vec();
    ctx->save_for_backward({r.final_T, r.last, r.kept});
    ctx->saved_data["call"] = c10::IValue::make_capsule(saved);
    return r.img;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const auto capsule = ctx->saved_data["call"].toCapsule();
    const Saved& c = *static_cast<const Saved*>(capsule.get());
    const Tensor grad = grads[0].contiguous();
    const auto opt = grad.options().requires_grad(false);
    std::array<Tensor, 4> g;
    for (int k = 0; k < 4; ++k) g[k] = at::empty(c.shapes[k], opt);
    char* k = static_cast<char*>(saved[2].data_ptr());
    const c10::DeviceGuard device(grad.device());
    {
      const Timed timed("render_backward");
      check(api.render_backward(
                &c.meta, reinterpret_cast<const float*>(k + c.keep[0]),
                reinterpret_cast<const int32_t*>(k + c.keep[2]),
                reinterpret_cast<const int32_t*>(k + c.keep[1]), f32(saved[0]),
                saved[1].data_ptr<int32_t>(),
                reinterpret_cast<const int32_t*>(k + c.keep[3]), f32(grad),
                g[0].data_ptr<float>(), g[1].data_ptr<float>(),
                g[2].data_ptr<float>(), g[3].data_ptr<float>(), c.n_pairs,
                k + c.keep[4], (size_t)(c.keep[5] - c.keep[4]), stream_of(grad)),
            "gsplat_hip_render_backward");
    }
    variable_list out(7);
    for (int i = 0; i < 4; ++i)
      if (ctx->needs_input_grad(i)) out[i] = g[i];
    // The depth gradient is zero; for depths computed by the projection it is
    // left undefined.
    if (c.depth_grad && ctx->needs_input_grad(4)) out[4] = at::zeros(c.shapes[4], opt);
    return out;
  }
};

// A validated RasterConfig: Plan.run is rasterize_projected_gaussians for the
// plain cases.
class Plan {
 public:
  Plan(int height, int width, float alpha_threshold, float transmittance_threshold,
       std::array<float, 3> background, float eps, float max_alpha, int strategy,
       int64_t limit_tiles, int64_t limit_gaussians, bool split_pairs, py::dict capacity,
       py::function note_pairs, int64_t sliced_pairs, int64_t sliced_pairs_per_tile)
      : strategy_(strategy), limit_tiles_(limit_tiles), limit_gaussians_(limit_gaussians),
        split_pairs_(split_pairs), sliced_pairs_(sliced_pairs),
        sliced_pairs_per_tile_(sliced_pairs_per_tile), capacity_(std::move(capacity)),
        note_pairs_(std::move(note_pairs)) {
    meta_ = gsplat_raster_meta{};
    meta_.height = height;
    meta_.width = width;
    meta_.tile_size = GSPLAT_TILE_SIZE;
    meta_.alpha_threshold = alpha_threshold;
    meta_.transmittance_threshold = transmittance_threshold;
    for (int k = 0; k < 3; ++k) meta_.background[k] = background[k];
    meta_.eps = eps;
    meta_.max_alpha = max_alpha;
    tiles_ = (int64_t)((height + 15) / 16) * ((width + 15) / 16);
  }

  py::object run(py::handle means2d, py::handle conics, py::handle colors,
                 py::handle opacities, py::handle depths, bool depth_grad) {
    const std::array<PyObject*, 5> o{means2d.ptr(), conics.ptr(), colors.ptr(),
                                     opacities.ptr(), depths.ptr()};
    for (PyObject* p : o)
      if (!plain(p)) return py::none();
    if (!plain_context()) return py::none();
    std::array<Tensor, 5> t;
    for (int k = 0; k < 5; ++k) t[k] = THPVariable_Unpack(o[k]);
    const Tensor& m = t[0];
    const int64_t nd = m.dim();
    if (nd != 2 && nd != 3) return py::none();
    const int64_t B = nd == 3 ? m.size(0) : 1, G = m.size(nd - 2);
    const int64_t width[5] = {2, 3, 3, 0, 0};
    for (int k = 0; k < 5; ++k) {
      const Tensor& x = t[k];
      if (x.device() != m.device() || x.dim() != (width[k] ? nd : nd - 1)) return py::none();
      if (nd == 3 && x.size(0) != B) return py::none();
      if (x.size(nd - 2) != G || (width[k] && x.size(nd - 1) != width[k])) return py::none();
    }
    if (B <= 0 || G <= 0 || B > (1 << 20) || G > (1 << 28)) return py::none();
    if (!one_launch(B, G)) return py::none();
    Call c;
    c.meta = meta_;
    c.meta.batch = (int32_t)B;
    c.meta.gaussians_per_batch = (int32_t)G;
    c.batched = nd == 3;
    c.depth_grad = depth_grad;
    bool grad = false;
    for (int k = 0; k < 4; ++k) grad |= t[k].requires_grad();
    const bool train = at::GradMode::is_enabled() && grad;
    const c10::DeviceGuard device(m.device());
    if (!choose(c, m, train)) return py::none();
    Tensor img;
    if (train) {
      img = Rasterize::apply(t[0], t[1], t[2], t[3], t[4], this, &c);
    } else {
      at::NoGradGuard no_grad;
      for (auto& x : t) x = x.detach();
      img = render_all(*this, c, t, false).img;
    }
    return py::reinterpret_steal<py::object>(THPVariable_Wrap(img));
  }

  // The capacity after a binning of n pairs (the policy of BinState.confirm,
  // in Python), and the call with room for them.  Takes the interpreter lock.
  Call after(const Call& c, const Tensor& like, int32_t n, bool train) {
    const int64_t head = (int64_t)n + n / 4 + 4096;
    if (n <= c.n_pairs && 2 * head >= c.n_pairs) return c;
    py::gil_scoped_acquire gil;
    const int64_t cap = note_pairs_(key(c, like), n).cast<int64_t>();
    Call next = c;
    if (n > c.n_pairs) {
      next.mode = Mode::kBinned;
      next.n_pairs = cap;
      next.sizes = sizes_of(c.meta, Mode::kBinned, cap, train);
    }
    return next;
  }

  // The call of a skewed scene by the one-call binning; the shape's next
  // calls go there at once: kSkewedCalls of them, twice as many each time it
  // turns out skewed again (a try costs a tile-sorted binning and a forward).
  Call binned(const Call& c, bool train) {
    {
      std::lock_guard<std::mutex> lock(mu_);
      Skewed* e = skewed(c);
      if (e == nullptr) {
        if (skewed_.size() >= 64) skewed_.erase(skewed_.begin());
        skewed_.push_back({c.meta.batch, c.meta.gaussians_per_batch, kSkewedCalls / 2, 0});
        e = &skewed_.back();
      }
      e->calls = std::min(2 * e->calls, 1 << 20);
      e->left = e->calls;
    }
    Call next = c;
    next.mode = Mode::kBinned;
    next.sizes = sizes_of(c.meta, Mode::kBinned, c.n_pairs, train);
    return next;
  }

 private:
  // A shape with skewed scenes: calls it is to be binned for, and those left.
  struct Skewed {
    int32_t B, G;
    int calls, left;
  };
  static constexpr int kSkewedCalls = 1024;
  Skewed* skewed(const Call& c) {  // with mu_ held
    for (auto& e : skewed_)
      if (e.B == c.meta.batch && e.G == c.meta.gaussians_per_batch) return &e;
    return nullptr;
  }

  // Whether the batch goes in one launch (the chunking of the Python layer).
  bool one_launch(int64_t B, int64_t G) const {
    if (split_pairs_ && B > 1) return false;
    if (strategy_ == 1) return true;  // flatten
    if (strategy_ == 2) return B == 1;  // serial
    const int64_t by_tiles = std::max<int64_t>(1, limit_tiles_ / std::max<int64_t>(tiles_, 1));
    const int64_t by_g = std::max<int64_t>(1, limit_gaussians_ / G);
    return B <= by_tiles && B <= by_g;
  }

  static py::tuple key(const Call& c, const Tensor& like) {
    return py::make_tuple((int)like.device().index(), c.meta.batch, c.meta.gaussians_per_batch,
                          c.meta.height, c.meta.width);
  }

  bool choose(Call& c, const Tensor& like, bool train) {
    const int64_t B = c.meta.batch, G = c.meta.gaussians_per_batch;
    if (G <= 4096) {
      const Sizes& s = sizes_of(c.meta, Mode::kDirect, tiles_ * B * G, train);
      if (s.keep[5] > 0) {
        c.mode = Mode::kDirect;
        c.n_pairs = api.direct_pairs(&c.meta);
        c.sizes = s;
        return true;
      }
    }
    // above: the count on a second stream, in the Python layer
    if (G > 131072 || B * G > 524288) return false;
    py::object cap = py::reinterpret_borrow<py::object>(
        PyDict_GetItem(capacity_.ptr(), key(c, like).ptr()));
    if (!cap) return false;
    c.n_pairs = cap.cast<int64_t>();
    if (c.n_pairs <= 0 || c.n_pairs > 0x7fffffff ||
        4 * c.n_pairs >= 5 * (sliced_pairs_ + sliced_pairs_per_tile_ * tiles_ * B))
      return false;
    bool binned = false;
    {
      std::lock_guard<std::mutex> lock(mu_);
      Skewed* e = skewed(c);
      if (e != nullptr && e->left > 0) {
        binned = true;
        --e->left;
      }
    }
    if (!binned) {
      c.mode = Mode::kTiled;
      c.sizes = sizes_of(c.meta, Mode::kTiled, c.n_pairs, train);
      if (c.sizes.keep[5] > 0) return true;
    }
    c.mode = Mode::kBinned;
    c.sizes = sizes_of(c.meta, Mode::kBinned, c.n_pairs, train);
    return true;
  }

  // Kept per shape, capacity and kind (keep[5] = 0: no such path).
  Sizes sizes_of(const gsplat_raster_meta& m, Mode mode, int64_t n, bool train) {
    const std::array<int64_t, 5> k{m.batch, m.gaussians_per_batch, (int64_t)mode, n, train};
    std::lock_guard<std::mutex> lock(mu_);
    for (const auto& e : sizes_)
      if (e.first == k) return e.second;
    Sizes s{};
    const int64_t BG = (int64_t)m.batch * m.gaussians_per_batch, T = tiles_ * m.batch;
    const int64_t work = mode == Mode::kDirect  ? (int64_t)api.direct_workspace_bytes(&m)
                         : mode == Mode::kTiled ? (int64_t)api.tile_workspace_bytes(&m, n)
                                                : (int64_t)api.bin_workspace_bytes(&m, n);
    if (work > 0) {
      const int64_t walked = mode == Mode::kDirect ? api.direct_pairs(&m) : n;
      const int64_t part[5] = {BG * GSPLAT_RECORD_FLOATS * 4, n * 4, (T + 1) * 4, train ? T * 4 : 0,
                               (int64_t)api.render_workspace_bytes(&m, train ? walked : 0)};
      for (int i = 0; i < 5; ++i) s.keep[i + 1] = s.keep[i] + align256(part[i]);
      const bool direct = mode != Mode::kBinned;  // (no depth order or offsets)
      s.use[1] = direct ? 0 : align256(BG * 4);
      s.use[2] = s.use[1] + (direct ? 0 : align256((BG + 1) * 4));
      s.use[3] = s.use[2] + align256(work);
    }
    if (sizes_.size() >= 16) sizes_.erase(sizes_.begin());
    sizes_.emplace_back(k, s);
    return s;
  }

  gsplat_raster_meta meta_;
  int64_t tiles_;
  int strategy_;
  int64_t limit_tiles_, limit_gaussians_;
  bool split_pairs_;
  int64_t sliced_pairs_, sliced_pairs_per_tile_;
  py::dict capacity_;
  py::function note_pairs_;
  std::mutex mu_;
  std::vector<std::pair<std::array<int64_t, 5>, Sizes>> sizes_;
  std::vector<Skewed> skewed_;
};

Call grown(Plan& plan, const Call& c, const Tensor& like, int32_t n, bool train) {
  return plan.after(c, like, n, train);
}

Call unskewed(Plan& plan, const Call& c, const Tensor&, bool train) {
  return plan.binned(c, train);
}

// ---- projection

struct Project : torch::autograd::Function<Project> {
  static variable_list forward(AutogradContext* ctx, const Tensor& means3d,
                               const Tensor& scales, const Tensor& quats,
                               const Tensor& opacities, const Tensor& c2w,
                               const Tensor& cam, double near_plane, bool batched) {
    ctx->set_materialize_grads(false);
    const int64_t B = batched ? means3d.size(0) : 1, G = means3d.size(-2);
    const Tensor t[6] = {means3d.contiguous(), scales.contiguous(), quats.contiguous(),
                         opacities.contiguous(), c2w.contiguous(), cam.contiguous()};
    const auto opt = t[0].options().requires_grad(false);
    auto shape = [&](int64_t width) {
      std::vector<int64_t> s;
      if (batched) s.push_back(B);
      s.push_back(G);
      if (width > 0) s.push_back(width);
      return s;
    };
    Tensor m2 = at::empty(shape(2), opt), cq = at::empty(shape(3), opt);
    Tensor op = at::empty(shape(0), opt), dp = at::empty(shape(0), opt);
    gsplat_project_meta meta{};
    meta.batch = (int32_t)B;
    meta.gaussians_per_batch = (int32_t)G;
    meta.near_plane = (float)near_plane;
    check(api.project_forward(&meta, f32(t[0]), f32(t[1]), f32(t[2]), f32(t[3]), f32(t[4]),
                              f32(t[5]), m2.data_ptr<float>(), cq.data_ptr<float>(),
                              op.data_ptr<float>(), dp.data_ptr<float>(), stream_of(t[0])),
          "gsplat_hip_project_forward");
    ctx->save_for_backward({t[0], t[1], t[2], t[3], t[4], t[5]});
    ctx->saved_data["near"] = near_plane;
    ctx->saved_data["B"] = B;
    ctx->saved_data["G"] = G;
    ctx->saved_data["opac"] = opacities.sizes().vec();
    return {m2, cq, op, dp};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto t = ctx->get_saved_variables();
    const int64_t B = ctx->saved_data["B"].toInt(), G = ctx->saved_data["G"].toInt();
    variable_list out(8);
    bool any = false;
    for (int k = 0; k < 6; ++k) any |= ctx->needs_input_grad(k);
    if (!any) return out;
    const auto opt = t[0].options().requires_grad(false);
    const c10::DeviceGuard device(t[0].device());
    // a depth gradient that is not there is zero: the C ABI takes a null pointer
    auto in = [&](int k, int64_t w) {
      return grads[k].defined() ? grads[k].contiguous() : at::zeros({B * G * w}, opt);
    };
    const Tensor g_m2 = in(0, 2), g_cq = in(1, 3), g_op = in(2, 1);
    const Tensor g_dp = grads[3].defined() ? grads[3].contiguous() : Tensor();
    Tensor g[6];
    for (int k = 0; k < 4; ++k) g[k] = at::empty(t[k].sizes(), opt);
    g[4] = at::empty({B, 4, 4}, opt);
    g[5] = at::empty({B, 4}, opt);
    gsplat_project_meta meta{};
    meta.batch = (int32_t)B;
    meta.gaussians_per_batch = (int32_t)G;
    meta.near_plane = (float)ctx->saved_data["near"].toDouble();
    const int64_t bytes_n = (int64_t)api.project_backward_workspace_bytes(&meta);
    const Tensor ws = bytes(std::max<int64_t>(bytes_n, 1), t[0]);
    {
      const Timed timed("project_backward");
      check(api.project_backward(
                &meta, f32(g_m2), f32(g_cq), f32(g_op), g_dp.defined() ? f32(g_dp) : nullptr,
                f32(t[0]), f32(t[1]), f32(t[2]), f32(t[3]), f32(t[4]), f32(t[5]),
                g[0].data_ptr<float>(), g[1].data_ptr<float>(), g[2].data_ptr<float>(),
                g[3].data_ptr<float>(), g[4].data_ptr<float>(), g[5].data_ptr<float>(),
                ws.data_ptr(), (size_t)bytes_n, stream_of(t[0])),
            "gsplat_hip_project_backward");
    }
    for (int k = 0; k < 6; ++k)
      if (ctx->needs_input_grad(k)) out[k] = g[k].view(k == 3 ? ctx->saved_data["opac"].toIntVector()
                                                              : g[k].sizes().vec());
    return out;
  }
};

// The number of images of plain [G,..] or [B,G,..] projection inputs of
// matching shapes, 0 for others.
int64_t project_images(py::handle means3d, py::handle scales, py::handle quats,
                       py::handle opacities) {
  const std::array<PyObject*, 4> o{means3d.ptr(), scales.ptr(), quats.ptr(), opacities.ptr()};
  for (PyObject* p : o)
    if (!plain(p)) return 0;
  if (!plain_context() || g_timed.load(std::memory_order_relaxed)) return 0;
  const Tensor& m = THPVariable_Unpack(o[0]);
  const int64_t nd = m.dim();
  if (nd != 2 && nd != 3) return 0;
  const int64_t B = nd == 3 ? m.size(0) : 1, G = m.size(nd - 2);
  if (m.size(nd - 1) != 3 || B <= 0 || G <= 0 || B > (1 << 20) || B * G > (int64_t(1) << 28))
    return 0;
  const Tensor &q = THPVariable_Unpack(o[2]), &op = THPVariable_Unpack(o[3]);
  if (THPVariable_Unpack(o[1]).sizes() != m.sizes()) return 0;
  if (q.dim() != nd || q.size(nd - 1) != 4 || q.sizes().slice(0, nd - 1) != m.sizes().slice(0, nd - 1))
    return 0;
  if (op.dim() == nd && op.size(nd - 1) != 1) return 0;
  if (op.dim() != nd && op.dim() != nd - 1) return 0;
  if (op.sizes().slice(0, nd - 1) != m.sizes().slice(0, nd - 1)) return 0;
  for (PyObject* p : o)
    if (THPVariable_Unpack(p).device() != m.device()) return 0;
  return B;
}

// The projection of inputs that project_images accepted, with c2w [B,4,4] and
// cam [B,4]; None where those are not plain.
py::object project(py::handle means3d, py::handle scales, py::handle quats,
                   py::handle opacities, py::handle c2w, py::handle cam, double near_plane) {
  const std::array<PyObject*, 6> o{means3d.ptr(), scales.ptr(), quats.ptr(),
                                   opacities.ptr(), c2w.ptr(), cam.ptr()};
  for (PyObject* p : o)
    if (!plain(p)) return py::none();
  const Tensor& m = THPVariable_Unpack(o[0]);
  const bool batched = m.dim() == 3;
  const int64_t B = batched ? m.size(0) : 1;
  const Tensor &w = THPVariable_Unpack(o[4]), &c = THPVariable_Unpack(o[5]);
  if (w.dim() != 3 || w.size(0) != B || c.dim() != 2 || c.size(0) != B) return py::none();
  for (PyObject* p : o)
    if (THPVariable_Unpack(p).device() != m.device()) return py::none();
  const c10::DeviceGuard device(m.device());
  const auto r = Project::apply(m, THPVariable_Unpack(o[1]), THPVariable_Unpack(o[2]),
                                THPVariable_Unpack(o[3]), w, c, near_plane, batched);
  py::tuple out(4);
  for (int k = 0; k < 4; ++k)
    out[k] = py::reinterpret_steal<py::object>(THPVariable_Wrap(r[k]));
  return out;
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.def("bind", &bind);
  m.def("set_timed", [](bool on) { g_timed.store(on); });
  // Whether saved tensors go through hooks of the caller's (checkpointing,
  // offloading).
  m.def("saved_tensor_hooks",
        [] { return at::SavedTensorDefaultHooks::get_hooks(true).has_value(); });
  m.def("project_images", &project_images);
  m.def("project", &project);
  py::class_<Plan>(m, "Plan")
      .def(py::init<int, int, float, float, std::array<float, 3>, float, float, int, int64_t,
                    int64_t, bool, py::dict, py::function, int64_t, int64_t>())
      .def("run", &Plan::run);
}
