// The calls of cumm_amd/torch_bridge.py in native code: a layer's forward pass, its node in torch's autograd
// graph, and the construction of a geometry.  What these do is the bridge's own sequence of calls of the
// C entry points; what they save is Python around launches of a few microseconds.  Forward of a layer on
// 2 k voxels 10.9 us of host time -> 4.8; forward and backward 67 - 120 us (Python in autograd's thread,
// with the interpreter's lock between the two threads) -> 46 - 50; two geometries and two layers with
// gradients 335 - 420 -> 235.
//
// A call is made here when its kind - pass, types, channels, kernel volume, epilogue, size class of the
// positions - has been validated and tuned by the bridge before (remember()); the argument block of that
// call then gets this geometry's tables and this call's tensors.  Everything else - first calls of a kind,
// tensors that are not plain ones of the tables' device, tracing, dispatch modes, forward-mode
// derivatives - is left to the bridge's Python function, whose results are the same.
#include <ATen/SavedTensorHooks.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/util/Exception.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/dynamo/compiled_autograd.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <atomic>
#include <cstring>
#include <mutex>
#include <tuple>
#include <unordered_map>

#include "../../include/cumm_hip.h"

namespace py = pybind11;
using at::Tensor;

namespace {

// ---- the C entry points, by the addresses that the bridge has of them
struct Api {
#define CUMM_API(name) decltype(&::cumm_hip_##name) name = nullptr
  CUMM_API(sparse_conv_more);
  CUMM_API(last_error);
  CUMM_API(relu_backward);
  CUMM_API(gate_sums);
  CUMM_API(column_sum_workspace);
  CUMM_API(query_conv_workspace);
  CUMM_API(query_wgrad_ordered_workspace);
  CUMM_API(wgrad_pairs_sums);
  CUMM_API(wgrad_pairs_workspace);
  CUMM_API(subm_pairs);
  CUMM_API(subm_pairs_workspace);
  CUMM_API(conv_pairs_workspace);
  CUMM_API(conv_pairs_sites);
  CUMM_API(conv_pairs_fill);
  CUMM_API(order_pairs_coarse);
  CUMM_API(order_pairs_coarse_workspace);
#undef CUMM_API
} api;

void bind(const py::dict &addresses) {
#define CUMM_API(name) api.name = reinterpret_cast<decltype(api.name)>(addresses["cumm_hip_" #name].cast<uintptr_t>())
  CUMM_API(sparse_conv_more);
  CUMM_API(last_error);
  CUMM_API(relu_backward);
  CUMM_API(gate_sums);
  CUMM_API(column_sum_workspace);
  CUMM_API(query_conv_workspace);
  CUMM_API(query_wgrad_ordered_workspace);
  CUMM_API(wgrad_pairs_sums);
  CUMM_API(wgrad_pairs_workspace);
  CUMM_API(subm_pairs);
  CUMM_API(subm_pairs_workspace);
  CUMM_API(conv_pairs_workspace);
  CUMM_API(conv_pairs_sites);
  CUMM_API(conv_pairs_fill);
  CUMM_API(order_pairs_coarse);
  CUMM_API(order_pairs_coarse_workspace);
#undef CUMM_API
}

// (the exception classes of _capi.check)
void check(int status) {
  if (status == CUMM_HIP_OK) return;
  const char *text = api.last_error();
  const std::string message = text ? text : "";
  if (status == CUMM_HIP_EINVAL) C10_THROW_ERROR(ValueError, message);
  C10_THROW_ERROR(Error, message);
}

c10::hip::HIPStreamMasqueradingAsCUDA current_stream() { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(); }

Tensor bytes(int64_t n, const c10::Device &device) {
  return at::empty({n > 256 ? n : 256}, at::TensorOptions().dtype(at::kByte).device(device));
}

// tv's number of an element type; -1 for those without kernels
int tv_type(at::ScalarType t) { return t == at::kHalf ? CUMM_HIP_F16 : (t == at::kBFloat16 ? CUMM_HIP_BF16 : -1); }

int size_class(int64_t n) {      // (the tuner's bucket of the position count)
  int bits = 0;
  for (int64_t v = n > 1 ? n - 1 : 0; v > 0; v >>= 1) ++bits;
  return bits;
}

// ---- validated calls by kind
struct Kind {
  CummHipConvDesc desc;
  CummHipSparseConvArgs args;
  int tile_m;
};
// pass, types of features / weight / bias (-1: none), K, C, kernel volume, submanifold, size class, device, ReLU,
// tile height (backward-weight) and determinism
using Key = std::tuple<int, int, int, int, int64_t, int64_t, int, bool, int, int, bool, int, bool>;
struct KeyHash {
  size_t operator()(const Key &k) const {
    size_t h = 0;
    std::apply([&](auto... v) { ((h = (h ^ (size_t)v) * 0x9E3779B97F4A7C15ull), ...); }, k);
    return h ^ (h >> 29);
  }
};
std::mutex kinds_mutex;
std::unordered_map<Key, Kind, KeyHash> kinds;      // (entries are added and never change)

const Kind *find_kind(const Key &key) {
  std::lock_guard<std::mutex> lock(kinds_mutex);
  const auto it = kinds.find(key);
  return it == kinds.end() ? nullptr : &it->second;
}

bool remember(int op, at::ScalarType x, at::ScalarType w, std::optional<at::ScalarType> bias, int64_t k_out, int64_t c_in, int kv, bool subm, int cls, int device,
              bool relu, int tile_m, bool deterministic, const std::string &desc, const std::string &args, int launch_tile_m) {
  Kind kind;
  if (desc.size() != sizeof(kind.desc) || args.size() != sizeof(kind.args)) throw py::value_error("argument blocks of another layout");
  std::memcpy(&kind.desc, desc.data(), desc.size());
  std::memcpy(&kind.args, args.data(), args.size());
  kind.tile_m = launch_tile_m;
  std::lock_guard<std::mutex> lock(kinds_mutex);
  return kinds.emplace(Key(op, (int)x, (int)w, bias.has_value() ? (int)*bias : -1, k_out, c_in, kv, subm, cls, device, relu, tile_m, deterministic), kind).second;
}

// ---- a geometry
struct Geometry {
  Tensor block, lists;      // (lists: several mask words only)
  std::vector<int32_t> counts;
  c10::Device device = c10::Device(c10::kCPU);
  void *stream = nullptr;
  int64_t n_in = 0, n_out = 0;
  int kv = 0, words = 1;
  bool subm = false;
  // as torch_bridge.SparseConvGeometry._lay_out
  int32_t *indices_fwd, *indices_bwd, *indices_fwd_pos, *indices_bwd_pos, *order_fwd, *order_bwd;
  uint32_t *mask_fwd, *mask_bwd, *reduced_64, *reduced_128;
  std::atomic<bool> written_64{false}, written_128{false};
  std::atomic<bool> made[3] = {};      // passes made here: forward, backward-input, backward-weight

  void allocate() {
    const int64_t pos_words = words;
    int64_t at = 0;
    const auto take = [&](int64_t count) { const int64_t here = at; at += (4 * count + 255) / 256 * 256; return here; };
    const int64_t fwd = take((int64_t)kv * n_out), bwd = take((int64_t)kv * n_in), fwd_pos = take((int64_t)kv * n_out),
                  bwd_pos = take((int64_t)kv * n_in), mf = take(n_out * pos_words), of = take(n_out);
    const int64_t mb = subm ? mf : take(n_in * pos_words), ob = subm ? of : take(n_in);
    const int64_t r64 = at, r128 = at + (n_out / 64 + 64) / 64 * 256;
    if (words == 1) at = r128 + (n_out / 128 + 64) / 64 * 256;
    block = bytes(at, device);
    char *base = static_cast<char *>(block.data_ptr());
    const auto i32 = [&](int64_t o) { return reinterpret_cast<int32_t *>(base + o); };
    const auto u32 = [&](int64_t o) { return reinterpret_cast<uint32_t *>(base + o); };
    indices_fwd = i32(fwd); indices_bwd = i32(bwd); indices_fwd_pos = i32(fwd_pos); indices_bwd_pos = i32(bwd_pos);
    mask_fwd = u32(mf); order_fwd = i32(of); mask_bwd = u32(mb); order_bwd = i32(ob);
    reduced_64 = u32(r64); reduced_128 = u32(r128);
  }
  // tell torch's allocator that the current stream reads the tables
  void used_on(const c10::hip::HIPStreamMasqueradingAsCUDA &s) const {
    if ((void *)s.stream() == stream) return;
    block.record_stream(s.unwrap());
    if (lists.defined()) lists.record_stream(s.unwrap());
  }
};
using GeometryPtr = std::shared_ptr<Geometry>;
using Three = std::array<int32_t, 3>;

// tables, order and tables by position -> (geometry, out_coords, out_shape, ordered): large tables are left to be
// ordered by the caller
py::tuple build(const Tensor &coords, const Three &shape, const Three &ksize, const std::optional<Three> &stride, const Three &padding,
                const Three &dilation, int batch) {
  GeometryPtr g = std::make_shared<Geometry>();
  Tensor out_coords;
  Three out_shape = shape;
  bool ordered = false;
  {
    py::gil_scoped_release release;
    const auto s = current_stream().stream();
    g->device = coords.device();
    g->stream = s;
    g->subm = !stride.has_value();
    g->n_in = coords.size(0);
    g->kv = ksize[0] * ksize[1] * ksize[2];
    g->words = (g->kv + 31) / 32;
    const int n_in = (int)g->n_in;
    const int32_t *at = coords.data_ptr<int32_t>();
    if (g->subm) {
      g->n_out = g->n_in;
      out_coords = coords;
      g->allocate();
      const Tensor ws = bytes((int64_t)api.subm_pairs_workspace(n_in), g->device);
      check(api.subm_pairs(at, n_in, shape.data(), ksize.data(), dilation.data(), g->indices_fwd, g->indices_bwd, nullptr, nullptr,
                           ws.data_ptr(), (size_t)ws.numel(), s));
    } else {
      const size_t need = api.conv_pairs_workspace(n_in, batch, shape.data(), ksize.data(), stride->data(), padding.data(), dilation.data());
      if (need == 0) C10_THROW_ERROR(ValueError, "bad geometry (kernel volume 1..128, non-empty output grid) or too many voxels");
      const Tensor ws = bytes((int64_t)need, g->device);
      int32_t found = 0;
      check(api.conv_pairs_sites(at, n_in, batch, shape.data(), ksize.data(), stride->data(), padding.data(), dilation.data(),
                                 out_shape.data(), &found, ws.data_ptr(), (size_t)ws.numel(), s));
      g->n_out = found;
      out_coords = at::empty({found, 4}, coords.options());
      g->allocate();
      check(api.conv_pairs_fill(at, n_in, batch, shape.data(), ksize.data(), stride->data(), padding.data(), dilation.data(), found,
                                out_coords.data_ptr<int32_t>(), g->indices_fwd, g->indices_bwd, nullptr, nullptr, ws.data_ptr(),
                                (size_t)ws.numel(), s));
    }
    // masks, an order of the positions by them, and the pair tables once more in that order
    if (4 * (int64_t)g->kv * std::max(g->n_in, g->n_out) < (int64_t)1 << 31) {
      ordered = true;
      CummHipOrderSide sides[2] = {};
      sides[0] = {g->indices_fwd, (int32_t)g->n_out, g->mask_fwd, g->order_fwd, g->indices_fwd_pos, nullptr};
      sides[1] = {g->indices_bwd, (int32_t)g->n_in, g->mask_bwd, g->order_bwd, g->indices_bwd_pos, nullptr};
      int count = 2;
      if (g->subm) {      // (one order serves both; the backward table is the forward one with its offsets reversed)
        sides[0].by_position_reversed = g->indices_bwd_pos;
        count = 1;
      }
      const Tensor ws = bytes((int64_t)api.order_pairs_coarse_workspace(sides, count, g->kv), g->device);
      check(api.order_pairs_coarse(sides, count, ksize.data(), ws.data_ptr(), (size_t)ws.numel(), s));
    }
  }
  return py::make_tuple(g, out_coords, py::make_tuple(out_shape[0], out_shape[1], out_shape[2]), ordered);
}

// ---- a layer
// Output channels from which the gate of a fused ReLU goes over the gradient in the order of the positions, in which
// the forward pass leaves its bits - also where there are none (first calls, saved-tensor hooks, compiled autograd: the output
// is what they have), so that a bias gradient has the same bits whoever computes it.  Rows of 128 bytes (32 channels:
// 15.2 -> 15.6 us, and 1.6 for the bits; 64: 11.6 -> 10.2 at 120 k rows, 50 -> 46 at 798 k).  torch_bridge.py has the same.
constexpr int64_t kGateFrom = 64;
// backward in Python, for calls that are not known here: (geometry, features, weight, out or None, gradient, needed
// gradients, relu, has_bias, tile_m) -> three gradients
PyObject *python_backward = nullptr;

Key key_of(const Geometry &g, int op, const Tensor &x, const Tensor &w, int bias, int64_t positions, bool relu, int tile_m, bool det) {
  return Key(op, (int)x.scalar_type(), (int)w.scalar_type(), bias, w.size(0), w.size(2), g.kv, g.subm, size_class(positions),
             g.device.index(), relu, tile_m, det);
}

CummHipSparseConvArgs moved(const Kind &kind, const Geometry &g, int64_t positions, const int32_t *indices, const uint32_t *mask,
                            const int32_t *order, uint32_t *mask_out) {
  CummHipSparseConvArgs a = kind.args;
  a.N = (int32_t)positions; a.rows_in = (int32_t)g.n_in; a.rows_out = (int32_t)g.n_out;
  a.indice_ptr = indices; a.mask_ptr = mask; a.mask_argsort_ptr = order; a.mask_out_ptr = mask_out;
  return a;
}

uint32_t *reduced_at(Geometry &g, int width) { return width == 64 ? g.reduced_64 : (width == 128 ? g.reduced_128 : nullptr); }

bool plain(const Tensor &t, const Geometry &g) {
  return t.defined() && t.device() == g.device && t.layout() == at::kStrided && !t.is_conj() && !t.is_neg() && t.numel() > 0 &&
         !t.key_set().has(c10::DispatchKey::Python) && !t._fw_grad(0).defined();
}

struct SparseConvBackward;

// Nodes that torch's compiled autograd has met, by the number that its graph has of them: a graph is used again
// for other nodes, so that it takes the number - a tensor, one of its inputs - and not the node.
struct Met {
  std::mutex mutex;
  std::unordered_map<int64_t, std::weak_ptr<torch::autograd::Node>> nodes;
  int64_t next = 0;
};
Met &met() {
  static Met *all = new Met();      // (nodes may outlive the statics)
  return *all;
}
torch::autograd::variable_list run_met(const torch::autograd::variable_list &grads, const std::vector<c10::IValue> &args);

struct SparseConvBackward : public torch::autograd::Node {
  GeometryPtr g;
  py::object owner;      // the bridge's geometry (for the Python path)
  torch::autograd::SavedVariable features, weight, out;
  Tensor gate;      // a bit per element of out, is it positive; undefined where the backward pass is to look at out itself
  std::vector<int64_t> sizes;
  at::TensorOptions options;
  bool relu = false, has_bias = false;
  int tile_m = 0;
  mutable Tensor number;      // in met()

  std::string name() const override { return "_SparseConvFunctionBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);      // (another thread may be in apply)
    features.reset_data();
    weight.reset_data();
    out.reset_data();
    gate = Tensor();
  }
  ~SparseConvBackward() override {
    if (number.defined()) {
      std::lock_guard<std::mutex> lock(met().mutex);
      met().nodes.erase(*number.data_ptr<int64_t>());
    }
    if (!Py_IsInitialized()) {
      owner.release();
    } else {
      py::gil_scoped_acquire gil;
      owner = py::object();
    }
  }

  torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    const Tensor x = features.unpack(), w = weight.unpack(), y = relu ? out.unpack(getptr()) : Tensor();
    const bool need[3] = {task_should_compute_output(0), task_should_compute_output(1), has_bias && task_should_compute_output(2)};
    return gradients(x, w, y, gate, grads[0], need);
  }

  torch::autograd::variable_list gradients(const Tensor &x, const Tensor &w, const Tensor &y, const Tensor &bits, const Tensor &grad,
                                           const bool (&need)[3]) {
    at::AutoGradMode no_grad(false);
    Tensor gy = grad.defined() ? grad.contiguous() : at::zeros(sizes, options);
    torch::autograd::variable_list result(3);
    if (!native(x, w, y, bits, gy, need, result)) python(x, w, y, gy, need, result);
    return result;
  }

  // ---- compiled autograd: what of the node is an input of its graph, and the call that the graph makes (opaque to
  // it: it takes addresses)
  void compiled_args(torch::dynamo::autograd::CompiledNodeArgs &args) const override {
    if (!number.defined()) {
      std::lock_guard<std::mutex> lock(met().mutex);
      number = at::full({1}, met().next, at::kLong);
      met().nodes[met().next++] = const_cast<SparseConvBackward *>(this)->weak_from_this();
    }
    args.collect(features, false);
    args.collect(weight, false);
    args.collect(relu);
    if (relu) args.collect(out, true);
    args.collect(has_bias);
    args.collect(number);
  }

  torch::autograd::variable_list apply_with_saved(const torch::autograd::variable_list &grads,
                                                  torch::dynamo::autograd::SwapSavedVariables &saved) override {
    namespace ca = torch::dynamo::autograd;
    saved.before(features);
    saved.before(weight);
    if (relu) saved.before(out);
    saved.before(number);
    std::vector<c10::IValue> args = {number, task_should_compute_output(0), task_should_compute_output(1),
                                     has_bias && task_should_compute_output(2), features.unpack(), weight.unpack()};
    if (relu) args.emplace_back(out.unpack(getptr()));
    std::vector<at::TypePtr> types;
    for (const c10::IValue &a : args) types.push_back(a.isTensor() ? at::TypePtr(at::TensorType::get()) : a.type());
    const auto &compiler = ca::getPyCompilerInterface();
    const std::string call = compiler->bind_function(saved.get_py_compiler(), "sparse_conv_backward", run_met, types,
                                                     /*is_custom_function=*/true, /*is_traceable=*/false);
    auto result = compiler->call_function(
        saved.get_py_compiler(), "apply_functional", call, grads, args,
        ca::IValuePacker<std::vector<std::optional<torch::autograd::InputMetadata>>>::pack(ca::get_input_metadata(next_edges())));
    saved.after(features);
    saved.after(weight);
    if (relu) saved.after(out);
    saved.after(number);
    return result;
  }

  bool native(const Tensor &x, const Tensor &w, const Tensor &y, const Tensor &bits, const Tensor &gy, const bool (&need)[3],
              torch::autograd::variable_list &result) {
    const int dtype = tv_type(x.scalar_type());
    const auto expected = [&](const Tensor &t) { return plain(t, *g) && t.is_contiguous() && t.scalar_type() == x.scalar_type(); };
    if (dtype < 0 || c10::impl::TorchDispatchModeTLS::any_modes_set() || !expected(x) || !expected(w) || !expected(gy) ||
        (relu && !expected(y)))
      return false;
    const bool deterministic = at::globalContext().deterministicAlgorithms();
    const Kind *dgrad = nullptr, *wgrad = nullptr;
    int64_t list_bytes = 0;
    const int64_t k_out = w.size(0), c_in = w.size(2);
    if (need[0] && !(dgrad = find_kind(key_of(*g, CUMM_HIP_OP_BACKWARD_INPUT, x, w, -1, g->n_in, false, 0, deterministic)))) return false;
    if (need[1] && g->words == 1 &&
        (!reduced_at(*g, tile_m) ||
         !(wgrad = find_kind(key_of(*g, CUMM_HIP_OP_BACKWARD_WEIGHT, x, w, -1, g->n_out, false, tile_m, deterministic)))))
      return false;
    if (need[1] && g->words > 1) {
      if (g->counts.empty()) return false;
      list_bytes = api.wgrad_pairs_workspace(g->counts.data(), g->kv, (int)k_out, (int)c_in);
      if (list_bytes < 0) return false;
    }
    const auto stream = current_stream();
    const auto s = stream.stream();
    g->used_on(stream);
    // the gradient passes where the fused ReLU let the output through; its column sums are the bias gradient.
    // With a weight gradient behind them its launches make both.
    const int64_t rows = gy.size(0);
    Tensor sums_ws;
    CummHipGateSums sums = {};
    if (need[2]) {
      result[2] = at::empty({k_out}, gy.options());
      sums_ws = bytes((int64_t)api.column_sum_workspace(rows, (int)k_out), g->device);
      sums.sums = result[2].data_ptr(); sums.grad = gy.data_ptr();
      sums.rows = rows; sums.channels = (int32_t)k_out;
      sums.workspace = sums_ws.data_ptr(); sums.workspace_bytes = (size_t)sums_ws.numel();
    }
    Tensor gated = gy;
    if (relu) {
      gated = at::empty_like(gy);
      sums.gated = gated.data_ptr();
      if (bits.defined()) sums.gate = bits.data_ptr();
      else sums.out = y.data_ptr();
      if (k_out >= kGateFrom) sums.order = g->order_fwd;
    }
    if (need[2] && !need[1]) check(api.gate_sums(&sums, dtype, s));
    if (!need[2] && relu) check(api.relu_backward(gated.data_ptr(), gy.data_ptr(), y.data_ptr(), (size_t)gy.numel(), dtype, s));
    if (need[1] && wgrad) {
      result[1] = at::empty_like(w);
      int64_t size = api.query_conv_workspace(&wgrad->desc, (int)k_out, (int)(g->kv * c_in), (int)rows, wgrad->args.split_k_slices, g->kv);
      if (deterministic) size = std::max(size, api.query_wgrad_ordered_workspace((int)rows, (int)c_in, (int)k_out, g->kv, tile_m));
      size = std::max(size, (int64_t)256);
      const Tensor ws = bytes(size, g->device);
      CummHipSparseConvArgs a = moved(*wgrad, *g, rows, g->indices_fwd, reduced_at(*g, tile_m), g->order_fwd, nullptr);
      a.ptr_A = gated.data_ptr(); a.ptr_B = x.data_ptr();
      a.ptr_C = result[1].data_ptr(); a.ptr_D = a.ptr_C;
      a.workspace = ws.data_ptr(); a.workspace_bytes = (size_t)size;
      CummHipSparseConvMore more = {};
      more.sums = need[2] ? &sums : nullptr;
      more.by_position = g->indices_fwd_pos;
      check(api.sparse_conv_more(&wgrad->desc, &a, &more, s));
      g->made[2] = true;
    } else if (need[1]) {
      // the products of all kernel offsets over their pair lists (an offset without pairs writes zeros)
      result[1] = at::empty_like(w);
      const Tensor ws = bytes(list_bytes, g->device);
      const int32_t *pair_in = g->lists.data_ptr<int32_t>(), *pair_out = pair_in + (int64_t)g->kv * g->n_out;
      check(api.wgrad_pairs_sums(result[1].data_ptr(), gated.data_ptr(), x.data_ptr(), pair_out, pair_in, g->counts.data(), g->kv, g->n_out,
                                 (int)g->n_out, (int)g->n_in, (int)k_out, (int)c_in, dtype, need[2] ? &sums : nullptr, ws.data_ptr(),
                                 (size_t)list_bytes, s));
      g->made[2] = true;
    }
    if (need[0]) {
      // inputs that feed no output site lie in tiles of mask 0: the kernel writes their zeros
      result[0] = at::empty_like(x);
      CummHipSparseConvMore more = {};
      more.write_empty = 1;
      CummHipSparseConvArgs a = moved(*dgrad, *g, g->n_in, g->indices_bwd_pos, g->mask_bwd, g->order_bwd, nullptr);
      a.ptr_A = gated.data_ptr(); a.ptr_B = w.data_ptr();
      a.ptr_C = result[0].data_ptr(); a.ptr_D = a.ptr_C;
      check(api.sparse_conv_more(&dgrad->desc, &a, &more, s));
      g->made[1] = true;
    }
    return true;
  }

  void python(const Tensor &x, const Tensor &w, const Tensor &y, const Tensor &gy, const bool (&need)[3], torch::autograd::variable_list &result) {
    py::gil_scoped_acquire gil;
    try {
      const py::tuple all = py::reinterpret_borrow<py::object>(python_backward)(
          owner, x, w, relu ? py::cast(y) : py::none(), gy, py::make_tuple(need[0], need[1], need[2]), relu, has_bias, tile_m);
      for (int i = 0; i < 3; ++i)
        if (!all[i].is_none()) result[i] = all[i].cast<Tensor>();
    } catch (py::error_already_set &e) {
      python_error error;
      e.restore();
      error.persist();
      throw error;
    }
  }
};

torch::autograd::variable_list run_met(const torch::autograd::variable_list &grads, const std::vector<c10::IValue> &args) {
  std::shared_ptr<torch::autograd::Node> node;
  {
    std::lock_guard<std::mutex> lock(met().mutex);
    const auto it = met().nodes.find(args[0].toTensor().item<int64_t>());
    if (it != met().nodes.end()) node = it->second.lock();
  }
  TORCH_CHECK(node != nullptr, "a compiled backward pass of a sparse convolution that is no longer there");
  const bool need[3] = {args[1].toBool(), args[2].toBool(), args[3].toBool()};
  return static_cast<SparseConvBackward &>(*node).gradients(args[4].toTensor(), args[5].toTensor(), args.size() > 6 ? args[6].toTensor() : Tensor(),
                                                            Tensor(), grads[0], need);
}

// the forward pass, or an undefined tensor where the call is the bridge's own
Tensor run_forward(const Tensor &features, const Tensor &weight, const std::optional<Tensor> &bias, const py::object &owner, Geometry &g,
                   const GeometryPtr &shared, bool relu) {
  if (!plain(features, g) || !plain(weight, g) || (bias.has_value() && !plain(*bias, g)) || features.dim() != 2 || weight.dim() != 3 ||
      features.size(0) != g.n_in || weight.size(1) != g.kv || weight.size(2) != features.size(1) ||
      (bias.has_value() && (bias->dim() != 1 || bias->size(0) != weight.size(0))) || g.n_out == 0 ||
      c10::impl::TorchDispatchModeTLS::any_modes_set() || torch::jit::tracer::isTracing())
    return Tensor();
  const Kind *kind = find_kind(key_of(g, CUMM_HIP_OP_FORWARD, features, weight, bias.has_value() ? (int)bias->scalar_type() : -1, g.n_out,
                                      relu, 0, at::globalContext().deterministicAlgorithms()));
  if (kind == nullptr || (g.words == 1 && reduced_at(g, kind->tile_m) == nullptr)) return Tensor();
  const bool differentiable =
      at::GradMode::is_enabled() && (features.requires_grad() || weight.requires_grad() || (bias.has_value() && bias->requires_grad()));
  // The gate of the backward pass as bits, which a pass over the gradient reads instead of the output.  Saved-tensor
  // hooks may hand back another output, which then is what counts.
  const bool gated = differentiable && relu && weight.size(0) >= kGateFrom && bias.has_value() && bias->requires_grad() &&
                     !at::SavedTensorDefaultHooks::get_hooks().has_value();
  Tensor x, w, y, gate;
  {
    at::AutoGradMode no_grad(false);
    x = features.contiguous();
    w = weight.contiguous();
    y = at::empty({g.n_out, w.size(0)}, x.options());
    const auto stream = current_stream();
    g.used_on(stream);
    CummHipSparseConvArgs a = moved(*kind, g, g.n_out, g.indices_fwd_pos, g.mask_fwd, g.order_fwd,
                                    g.words == 1 ? reduced_at(g, kind->tile_m) : nullptr);
    a.ptr_A = x.data_ptr(); a.ptr_B = w.data_ptr();
    a.ptr_C = y.data_ptr(); a.ptr_D = a.ptr_C;
    Tensor b;
    if (bias.has_value()) {
      b = bias->contiguous();
      a.ptr_D = a.bias_pointer = b.data_ptr();
    }
    CummHipSparseConvMore more = {};
    if (gated) {
      gate = bytes((w.size(0) + 63) / 64 * g.n_out * 8, g.device);
      more.gate = gate.data_ptr();
    }
    check(api.sparse_conv_more(&kind->desc, &a, &more, stream.stream()));
    g.made[0] = true;
    if (g.words == 1) (kind->tile_m == 64 ? g.written_64 : g.written_128) = true;
  }
  if (differentiable) {
    auto node = std::shared_ptr<SparseConvBackward>(new SparseConvBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(features, weight, bias.has_value() ? *bias : Tensor()));
    node->g = shared;
    node->relu = relu;
    node->has_bias = bias.has_value();
    node->tile_m = kind->tile_m;
    node->gate = gate;
    node->sizes = y.sizes().vec();
    node->options = y.options();
    node->features = torch::autograd::SavedVariable(x, false);
    node->weight = torch::autograd::SavedVariable(w, false);
    {
      py::gil_scoped_acquire gil;
      node->owner = owner;
    }
    torch::autograd::set_history(y, node);
    if (relu) node->out = torch::autograd::SavedVariable(y, true);
  }
  return y;
}

py::object forward(const Tensor &features, const Tensor &weight, const std::optional<Tensor> &bias, const py::object &owner,
                   const GeometryPtr &g, bool relu) {
  Tensor result;
  {
    py::gil_scoped_release release;
    result = run_forward(features, weight, bias, owner, *g, g, relu);
  }
  return result.defined() ? py::cast(result) : py::none();
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.attr("stamp") = "cumm_torch_native:" CUMM_STAMP;      // (build.py looks for it in the file)
  py::class_<Geometry, GeometryPtr>(m, "Geometry")
      .def_readonly("block", &Geometry::block)
      .def_readonly("n_in", &Geometry::n_in)
      .def_readonly("n_out", &Geometry::n_out)
      .def("made", [](const Geometry &g, int pass) { return g.made[pass].load(); })
      .def("written", [](const Geometry &g, int width) { return width == 64 ? g.written_64.load() : (width == 128 && g.written_128.load()); })
      .def("set_lists",
           [](Geometry &g, const Tensor &lists, std::vector<int32_t> counts) {
             g.lists = lists;
             g.counts = std::move(counts);
           })
      .def("tables", [](const Geometry &g) {
        const auto at = [](const void *p) { return (uintptr_t)p; };
        py::dict d;
        d["indices_fwd"] = at(g.indices_fwd); d["indices_bwd"] = at(g.indices_bwd);
        d["indices_fwd_pos"] = at(g.indices_fwd_pos); d["indices_bwd_pos"] = at(g.indices_bwd_pos);
        d["mask_fwd"] = at(g.mask_fwd); d["order_fwd"] = at(g.order_fwd); d["mask_bwd"] = at(g.mask_bwd); d["order_bwd"] = at(g.order_bwd);
        if (g.words == 1) { d["reduced_64"] = at(g.reduced_64); d["reduced_128"] = at(g.reduced_128); }
        return d;
      });
  m.def("bind", &bind);
  m.def("set_backward", [](py::object f) {
    Py_XDECREF(python_backward);
    python_backward = f.release().ptr();
  });
  m.def("remember", &remember);
  m.def("build", &build);
  m.def("forward", &forward);
}
