// Python binding of libdlt_hip.so for torch tensors: argument checks, output allocation, the autograd nodes and the
// calls into the C ABI, compiled.  The Python modules next to it only name the entry points.
//
// A training step of one attention layer is three kernel launches of 10 ... 20 us each on the sizes most layers have.
// Through torch.autograd.Function and ctypes the host needed 146 us for that step (two Python frames per direction,
// descriptor and stride arrays built object by object, a device guard object, three to seven torch.empty calls from
// Python), so every such step waited for the host.  Here the same work is done on the tensor structs themselves.
//
// Nothing is kept from one call for the next and nothing is launched that the Python version did not launch.  The Python
// classes (torch.autograd.Function) stay the general path: a compiled entry point answers NotImplemented to every call that is
// not a plain eager one (see plain() below), and apply() of its class then goes on through the class.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/VariableTypeUtils.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <array>
#include <mutex>
#include <string>

#include "../../include/dlt.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

PyObject* g_dlt_error = nullptr;   // dl_templates_amd._lib.DltError

// ---- errors ---------------------------------------------------------------------------------
// Python exceptions that can also leave an engine thread: the error is kept inside the C++ exception.
[[noreturn]] void raise_py(PyObject* type, const std::string& msg) {
  pybind11::gil_scoped_acquire gil;
  PyErr_SetString(type, msg.c_str());
  python_error e;
  e.persist();
  throw std::move(e);
}

void require(bool ok, PyObject* type, const char* msg) {
  if (C10_UNLIKELY(!ok)) raise_py(type, msg);
}
void check_assert(bool ok, const char* msg) { require(ok, PyExc_AssertionError, msg); }

void check_rc(int rc) {
  if (C10_LIKELY(rc == DLT_OK)) return;
  const std::string msg = dlt_last_error();
  pybind11::gil_scoped_acquire gil;
  PyObject* exc = PyObject_CallFunction(g_dlt_error, "is", rc, msg.c_str());
  if (exc != nullptr) {
    PyErr_SetObject(g_dlt_error, exc);
    Py_DECREF(exc);
  }
  python_error e;
  e.persist();
  throw std::move(e);
}

std::string shown(const at::Device& d) { return d.str(); }

// every tensor on one ROCm device
template <typename... T>
void require_gpu(const Tensor& first, const T&... rest) {
  const at::Device dev = first.device();
  auto one = [&](const Tensor& t) {
    if (C10_UNLIKELY(!t.is_cuda()))
      raise_py(PyExc_RuntimeError, "dl_templates_amd runs on a ROCm GPU only: got a tensor on " + shown(t.device()));
    if (C10_UNLIKELY(t.device() != dev))
      raise_py(PyExc_RuntimeError, "all tensors must be on one device, got " + shown(dev) + " and " + shown(t.device()));
  };
  one(first);
  (one(rest), ...);
}

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return DLT_BF16;
    case at::kHalf: return DLT_FP16;
    case at::kFloat: return DLT_FP32;
    default: break;
  }
  raise_py(PyExc_TypeError, std::string("unsupported dtype ") + c10::toString(t.scalar_type()) + "; expected bfloat16, float16 or float32");
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor empty(at::IntArrayRef size, at::ScalarType st, const Tensor& like) {
  return Tensor(at::detail::empty_cuda(size, st, like.device(), std::nullopt));
}
// torch.empty_like: the strides of a dense tensor are kept
Tensor grad_like(const Tensor& t) { return t.is_contiguous() ? empty(t.sizes(), t.scalar_type(), t) : at::empty_like(t); }

const int64_t* st(const Tensor& t) { return t.strides().data(); }

// ---- which calls the compiled nodes take -----------------------------------------------------------
// Plain eager calls: no trace, transform (torch.func) or dispatch mode is active, the tensors are ordinary strided ones and
// none carries a forward-mode tangent.  Everything else (and its errors) belongs to the autograd.Function classes: a node made
// here would drop the tangent, be missing from the trace, or hide from the mode.
bool plain_keys(c10::DispatchKeySet ks, c10::DispatchKeySet allowed) {
  return (ks.raw_repr() & ~allowed.raw_repr() & ~c10::full_backend_mask) == 0;
}
template <typename... T>
bool plain(const T&... ts) {
  using K = c10::DispatchKey;
  constexpr c10::DispatchKeySet MODES = c10::DispatchKeySet({K::BackendSelect, K::ADInplaceOrView}) | c10::autocast_dispatch_keyset;
  constexpr c10::DispatchKeySet TENSOR = c10::DispatchKeySet({K::Dense, K::ADInplaceOrView, K::AutogradFunctionality}) | c10::autocast_dispatch_keyset;
  auto one = [&](const Tensor& t) { return plain_keys(t.key_set(), TENSOR) && !t._fw_grad(/*level=*/0).defined(); };
  return plain_keys(c10::impl::tls_local_dispatch_key_set().included_, MODES) && (one(ts) && ...);
}

// ---- rotary operands --------------------------------------------------------------------------
struct Rope {
  Tensor idx, row, col;   // row, col: fp32 [len, R, 2] with a contiguous [R, 2] tail
  dlt_rope_t d;
};

Rope make_rope(const Tensor& idx, const Tensor& row, const Tensor& col) {
  require(idx.scalar_type() == at::kInt && idx.dim() == 1 && idx.is_contiguous(), PyExc_TypeError, "idx must be a contiguous 1-D int32 tensor");
  Rope r;
  r.idx = idx;
  auto table = [](const Tensor& t) {
    require(t.dim() == 3 && t.size(2) == 2, PyExc_ValueError, "cos/sin table must have shape [len, R, 2]");
    if (t.scalar_type() == at::kFloat && t.stride(2) == 1 && t.stride(1) == 2) return t;
    return t.to(at::kFloat).contiguous();
  };
  r.row = table(row);
  r.col = table(col);
  r.d.idx = idx.const_data_ptr<int32_t>();
  r.d.row_cs = r.row.const_data_ptr<float>();
  r.d.col_cs = r.col.const_data_ptr<float>();
  r.d.row_cs_stride0 = r.row.stride(0);
  r.d.col_cs_stride0 = r.col.stride(0);
  r.d.n_rdim = (int32_t)r.row.size(1);
  r.d.row_len = (int32_t)r.row.size(0);
  r.d.col_len = (int32_t)r.col.size(0);
  return r;
}

Rope make_rope_for(const Tensor& idx, const Tensor& row, const Tensor& col, const Tensor& like, int64_t n_tokens) {
  if (C10_UNLIKELY(idx.dim() != 1 || idx.size(0) != n_tokens))
    raise_py(PyExc_ValueError, "idx has " + std::to_string(idx.dim() > 0 ? idx.size(0) : 0) + " entries for " + std::to_string(n_tokens) + " tokens");
  require_gpu(like, idx, row, col);
  return make_rope(idx, row, col);
}

// ---- the attention operators --------------------------------------------------------------------
enum class Op { Swa, Image, Flash };

struct Spec {
  Op op = Op::Swa;
  dlt_swa_shape_t swa{};
  dlt_swa_tile_t tile{};
  dlt_flash_shape_t flash{};
  bool narrow = false;   // Swa: see small_tiles
};

Spec swa_spec(const Tensor& q, const Tensor& k, const Tensor& v, const int64_t* dims /* b_size, th, tw, row, col */, double scale) {
  check_assert(q.dim() == 4, "q must have shape [B, H, N, D]");
  const int64_t B = q.size(0), H = q.size(1), N = q.size(2), dk = q.size(3);
  check_assert(N == dims[0] * dims[1] * dims[2], "seqlen should match image size");
  check_assert(k.sizes() == q.sizes() && v.dim() == 4 && v.size(0) == B && v.size(1) == H && v.size(2) == N, "k and v must match q");
  check_assert(q.scalar_type() == k.scalar_type() && k.scalar_type() == v.scalar_type(), "q, k and v must have one dtype");
  Spec s;
  s.op = Op::Swa;
  s.swa = {(int32_t)B, (int32_t)H, (int32_t)dims[0], (int32_t)dims[1], (int32_t)dims[2], (int32_t)dims[3], (int32_t)dims[4],
           (int32_t)dk, (int32_t)v.size(3), (float)scale, dtype_code(q)};
  return s;
}

Spec image_spec(const Tensor& q, const Tensor& k, const Tensor& v, const int64_t* dims /* bh, bw, row, col */, double scale) {
  check_assert(q.dim() == 5, "q must have shape [B, IH, IW, heads, D]");
  const int64_t IH = q.size(1), IW = q.size(2), bh = dims[0], bw = dims[1];
  require(bh != 0 && bw != 0, PyExc_ZeroDivisionError, "tile of zero pixels");
  check_assert(IH % bh == 0 && IW % bw == 0, "image size should be a multiple of the tile size");
  check_assert(k.sizes() == q.sizes() && v.dim() == 5 && v.sizes().slice(0, 4) == q.sizes().slice(0, 4), "k and v must match q");
  check_assert(q.scalar_type() == k.scalar_type() && k.scalar_type() == v.scalar_type(), "q, k and v must have one dtype");
  Spec s;
  s.op = Op::Image;
  s.swa = {(int32_t)q.size(0), (int32_t)q.size(3), (int32_t)(bh * bw), (int32_t)(IH / bh), (int32_t)(IW / bw), (int32_t)dims[2], (int32_t)dims[3],
           (int32_t)q.size(4), (int32_t)v.size(4), (float)scale, dtype_code(q)};
  s.tile = {(int32_t)bh, (int32_t)bw};
  return s;
}

Spec flash_spec(const Tensor& q, const Tensor& k, const Tensor& v, bool causal, double scale) {
  check_assert(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "q, k and v must have shape [B, H, L, D]");
  check_assert(q.size(3) == k.size(3), "q and k must have one head dim");
  check_assert(q.sizes().slice(0, 2) == k.sizes().slice(0, 2) && q.sizes().slice(0, 2) == v.sizes().slice(0, 2) && k.size(2) == v.size(2),
               "k and v must match q");
  check_assert(q.scalar_type() == k.scalar_type() && k.scalar_type() == v.scalar_type(), "q, k and v must have one dtype");
  Spec s;
  s.op = Op::Flash;
  s.flash = {(int32_t)q.size(0), (int32_t)q.size(1), (int32_t)q.size(2), (int32_t)k.size(2), (int32_t)q.size(3), (int32_t)v.size(3),
             (float)scale, causal ? 1 : 0, dtype_code(q)};
  return s;
}

// Partial results of a flash pass that splits its other side: from the caching allocator, on the call's stream, for the call alone.
struct Workspace {
  Tensor t;
  void* ptr = nullptr;
  int64_t bytes = 0;
};
Workspace flash_workspace(const dlt_flash_shape_t& shape, int backward, const Tensor& like) {
  Workspace w;
  check_rc(dlt_flash_workspace(&shape, backward, &w.bytes));
  if (w.bytes > 0) {
    w.t = empty({w.bytes / 4}, at::kFloat, like);
    w.ptr = w.t.mutable_data_ptr();
  }
  return w;
}

struct Forward { Tensor o, lse, q_rot, k_rot; };

// keep_rot: the rotated q and k are stored as well (for the backward pass)
Forward run_forward(const Spec& s, const Tensor& q, const Tensor& k, const Tensor& v, const Rope* rope, bool keep_rot) {
  require_gpu(q, k, v);
  c10::DeviceGuard guard(q.device());
  Forward f;
  const at::ScalarType dt = q.scalar_type();
  void* stream = stream_of(q);
  if (s.op == Op::Flash) {
    f.o = empty({q.size(0), q.size(1), q.size(2), v.size(3)}, dt, q);
    f.lse = empty({q.size(0), q.size(1), q.size(2)}, at::kFloat, q);
    const Workspace ws = flash_workspace(s.flash, 0, q);
    check_rc(dlt_flash_fwd_ws(q.const_data_ptr(), st(q), k.const_data_ptr(), st(k), v.const_data_ptr(), st(v), f.o.mutable_data_ptr(), st(f.o),
                              (float*)f.lse.mutable_data_ptr(), st(f.lse), &s.flash, ws.ptr, ws.bytes, stream));
    return f;
  }
  if (s.op == Op::Image) {
    f.o = empty({q.size(0), q.size(1), q.size(2), q.size(3), v.size(4)}, dt, q);
    f.lse = empty({q.size(0), q.size(3), q.size(1) * q.size(2)}, at::kFloat, q);
    check_rc(dlt_swa_fwd_image(q.const_data_ptr(), st(q), k.const_data_ptr(), st(k), v.const_data_ptr(), st(v), f.o.mutable_data_ptr(), st(f.o),
                               (float*)f.lse.mutable_data_ptr(), st(f.lse), &s.swa, &s.tile, nullptr, stream));
    return f;
  }
  f.o = empty({q.size(0), q.size(1), q.size(2), v.size(3)}, dt, q);
  f.lse = empty({q.size(0), q.size(1), q.size(2)}, at::kFloat, q);
  if (keep_rot) {
    f.q_rot = empty(q.sizes(), dt, q);
    f.k_rot = empty(k.sizes(), dt, q);
    check_rc(dlt_swa_fwd_rot(q.const_data_ptr(), st(q), k.const_data_ptr(), st(k), v.const_data_ptr(), st(v), f.o.mutable_data_ptr(), st(f.o),
                             (float*)f.lse.mutable_data_ptr(), st(f.lse), f.q_rot.mutable_data_ptr(), st(f.q_rot), f.k_rot.mutable_data_ptr(),
                             st(f.k_rot), &s.swa, &rope->d, stream));
  } else {
    if (s.narrow)
      check_rc(dlt_swa_fwd_narrow(q.const_data_ptr(), st(q), k.const_data_ptr(), st(k), v.const_data_ptr(), st(v), f.o.mutable_data_ptr(), st(f.o),
                                  (float*)f.lse.mutable_data_ptr(), st(f.lse), &s.swa, stream));
    else
      check_rc(dlt_swa_fwd(q.const_data_ptr(), st(q), k.const_data_ptr(), st(k), v.const_data_ptr(), st(v), f.o.mutable_data_ptr(), st(f.o),
                           (float*)f.lse.mutable_data_ptr(), st(f.lse), &s.swa, rope ? &rope->d : nullptr, stream));
  }
  return f;
}

// rotated: q and k are the rotated tensors that the forward pass kept
std::array<Tensor, 3> run_backward(const Spec& s, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse,
                                   const Tensor& d_o, const Rope* rope, bool rotated) {
  require_gpu(q, k, v, o, lse, d_o);
  c10::DeviceGuard guard(q.device());
  Tensor dq = grad_like(q), dk = grad_like(k), dv = grad_like(v), delta = grad_like(lse);
  void* stream = stream_of(q);
  auto call = [&](auto fn, auto... shape) {
    check_rc(fn(q.const_data_ptr(), st(q), k.const_data_ptr(), st(k), v.const_data_ptr(), st(v), o.const_data_ptr(), st(o), d_o.const_data_ptr(),
                st(d_o), (const float*)lse.const_data_ptr(), (float*)delta.mutable_data_ptr(), st(lse), dq.mutable_data_ptr(), st(dq),
                dk.mutable_data_ptr(), st(dk), dv.mutable_data_ptr(), st(dv), shape..., stream));
  };
  const dlt_rope_t* none = nullptr;
  if (s.op == Op::Flash) {
    const Workspace ws = flash_workspace(s.flash, 1, q);
    call(dlt_flash_bwd_ws, &s.flash, ws.ptr, ws.bytes);
  }
  else if (s.op == Op::Image) call(dlt_swa_bwd_image, &s.swa, &s.tile, none);
  else if (rotated) call(dlt_swa_bwd_rot, &s.swa, (const dlt_rope_t*)&rope->d);
  else if (s.narrow) call(dlt_swa_bwd_narrow, &s.swa);
  else call(dlt_swa_bwd, &s.swa, rope ? (const dlt_rope_t*)&rope->d : none);
  return {dq, dk, dv};
}

// ---- head dims outside the tuned shapes -----------------------------------------------------------
// {dk, dv} to pad q / k and v to before the launch.  Zero columns appended to q, k, v (and to dO) change no score and no
// output column; the copies cost a few percent of what the generic kernels would.
struct Pad { int64_t dk, dv; };

// The token-grid kernels (b_size == 1) take head dims that are multiples of 32 with both in one class (both <= 64, or
// both in 65 ... 128): anything else runs 6 to 9 times slower on the generic kernels.  Tiles of 2 ... 15 tokens run on the
// streaming kernels at head dim 64 or 128 exactly (2 to 4 times).  Tiles of 16 k tokens are padded inside their kernels.
Pad swa_pad(int64_t dk, int64_t dv, at::ScalarType dt, int64_t b_size) {
  const int64_t big = std::max(dk, dv);
  if ((dt != at::kBFloat16 && dt != at::kHalf) || big > 128) return {dk, dv};
  if (2 <= b_size && b_size <= 15) return big <= 64 ? Pad{64, 64} : Pad{128, 128};
  if (b_size != 1) return {dk, dv};
  auto up = [](int64_t d) { return (d + 31) / 32 * 32; };
  return big <= 64 ? Pad{up(dk), up(dv)} : Pad{std::max<int64_t>(96, up(dk)), std::max<int64_t>(96, up(dv))};
}

// Tiles of 2 ... 15 tokens at smaller head dims whose rows can be read in 16-byte pieces as they lie run there without padding (d = 32, 16 heads of 20 x 6
// tiles of 4: the copies around the kernels were 22 of 35 us of host time in the forward pass).
bool rows_of_pieces(const Tensor& x) {
  return x.dim() == 4 && x.size(3) % 8 == 0 && x.stride(3) == 1 && (uintptr_t)x.const_data_ptr() % 16 == 0 && x.stride(0) % 8 == 0 && x.stride(1) % 8 == 0 &&
         x.stride(2) % 8 == 0 && x.stride(2) >= 0 && (x.size(2) + 64) * std::max<int64_t>(x.stride(2), 64) < ((int64_t)1 << 30);
}
bool small_tiles(const Tensor& q, const Tensor& k, const Tensor& v, int64_t b_size, double scale) {
  const at::ScalarType dt = q.scalar_type();
  return 2 <= b_size && b_size <= 15 && (dt == at::kBFloat16 || dt == at::kHalf) && scale > 0 && q.size(-1) <= 64 && v.size(-1) <= 64 &&
         rows_of_pieces(q) && rows_of_pieces(k) && rows_of_pieces(v);
}

// The flash kernels read 16-byte row pieces: head dims that are not multiples of 8 run 3 to 6 times slower on the generic ones.
Pad flash_pad(int64_t dk, int64_t dv, at::ScalarType dt) {
  if ((dt != at::kBFloat16 && dt != at::kHalf) || std::max(dk, dv) > 128) return {dk, dv};
  return {(dk + 7) / 8 * 8, (dv + 7) / 8 * 8};
}

Tensor pad_last(const Tensor& x, int64_t d) { return x.size(-1) == d ? x : at::constant_pad_nd(x, {0, d - x.size(-1)}); }
Tensor cut_last(const Tensor& x, int64_t d) { return x.size(-1) == d ? x : x.narrow(-1, 0, d).contiguous(); }

// ---- autograd ---------------------------------------------------------------------------------------
struct AttnBackward : public Node {
  Spec spec;
  bool has_rope = false, rotated = false;
  int64_t dk = 0, dv = 0;   // head dims of the caller's tensors
  SavedVariable q, k, v, o, lse, idx, row, col;

  std::string name() const override { return "DltAttentionBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (SavedVariable* s : {&q, &k, &v, &o, &lse, &idx, &row, &col}) s->reset_data();
  }
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    if (!grads[0].defined()) grads[0] = input_metadata(0).zeros_like();   // as torch.autograd.Function does
    // Unpacked with autograd as it is: an unpack hook may run the forward pass again (activation checkpointing), and what it runs
    // has to be recorded.
    const Tensor q_ = q.unpack(), k_ = k.unpack(), v_ = v.unpack(), o_ = o.unpack(shared_from_this()), lse_ = lse.unpack();
    Tensor idx_, row_, col_;
    if (has_rope) {
      idx_ = idx.unpack();
      row_ = row.unpack();
      col_ = col.unpack();
    }
    at::AutoDispatchBelowADInplaceOrView below;
    Rope rope;
    if (has_rope) rope = make_rope_for(idx_, row_, col_, q_, q_.size(2));
    Tensor d_o = pad_last(grads[0], v_.size(-1));
    if (spec.narrow && !rows_of_pieces(d_o)) d_o = d_o.contiguous();
    auto g = run_backward(spec, q_, k_, v_, o_, lse_, d_o, has_rope ? &rope : nullptr, rotated);
    return {cut_last(g[0], dk), cut_last(g[1], dk), cut_last(g[2], dv)};
  }
};

struct RopeBackward : public Node {
  SavedVariable idx, row, col;
  std::string name() const override { return "DltRotaryPE2DBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    idx.reset_data();
    row.reset_data();
    col.reset_data();
  }
  variable_list apply(variable_list&& grads) override;
};

template <typename N>
std::shared_ptr<N> make_node() { return std::shared_ptr<N>(new N(), torch::autograd::deleteNode); }

// Forward pass with the graph recorded when q, k or v asks for it (graph == false: never).
Tensor attention(Op op, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor* rope_t, const int64_t* dims, bool causal, double scale,
                 bool keep_rot, bool graph) {
  std::shared_ptr<AttnBackward> node;
  const bool grad = graph && torch::autograd::compute_requires_grad(q, k, v);
  if (grad) {
    node = make_node<AttnBackward>();
    node->set_next_edges(torch::autograd::collect_next_edges(q, k, v));
  }
  pybind11::gil_scoped_release nogil;
  Tensor out, pq = q, pk = k, pv = v;
  Forward f;
  Spec spec;
  check_assert(q.dim() >= 2 && k.dim() == q.dim() && v.dim() == q.dim(), "q, k and v must have the same number of dims");
  const int64_t dk = q.size(-1), dv = v.size(-1);
  {
    at::AutoDispatchBelowADInplaceOrView below;
    const bool narrow = op == Op::Swa && rope_t == nullptr && small_tiles(q, k, v, dims[0], scale);
    const Pad pad = narrow ? Pad{dk, dv} : op == Op::Flash ? flash_pad(dk, dv, q.scalar_type()) : op == Op::Swa ? swa_pad(dk, dv, q.scalar_type(), dims[0]) : Pad{dk, dv};
    if (C10_UNLIKELY(pad.dk != dk || pad.dv != dv)) {
      pq = pad_last(q, pad.dk);
      pk = pad_last(k, pad.dk);
      pv = pad_last(v, pad.dv);
    }
    spec = op == Op::Flash ? flash_spec(pq, pk, pv, causal, scale) : op == Op::Image ? image_spec(pq, pk, pv, dims, scale) : swa_spec(pq, pk, pv, dims, scale);
    spec.narrow = narrow;
    Rope rope;
    if (rope_t != nullptr) {
      check_assert(rope_t[1].dim() == 3 && rope_t[2].dim() == 3 && rope_t[1].size(1) == rope_t[2].size(1), "row and column table must have one R");
      check_assert(rope_t[0].dim() == 1 && rope_t[0].size(0) == pq.size(2), "idx must have one entry per token");
      require_gpu(pq, pk, pv);
      rope = make_rope_for(rope_t[0], rope_t[1], rope_t[2], pq, pq.size(2));
    }
    f = run_forward(spec, pq, pk, pv, rope_t ? &rope : nullptr, keep_rot);
    out = cut_last(f.o, dv);
  }
  // saved with autograd as it is: pack hooks are the caller's code
  if (grad) {
    node->spec = spec;
    node->dk = dk;
    node->dv = dv;
    node->q = SavedVariable(keep_rot ? f.q_rot : pq, false);
    node->k = SavedVariable(keep_rot ? f.k_rot : pk, false);
    node->v = SavedVariable(pv, false);
    node->lse = SavedVariable(f.lse, false);
    if (rope_t != nullptr) {
      node->has_rope = true;
      node->rotated = keep_rot;
      node->idx = SavedVariable(rope_t[0], false);
      node->row = SavedVariable(rope_t[1], false);
      node->col = SavedVariable(rope_t[2], false);
    }
    const bool whole = out.is_same(f.o);
    if (!whole) node->o = SavedVariable(f.o, false);
    torch::autograd::set_history(out, node);
    if (whole) node->o = SavedVariable(out, true);
  }
  return out;
}

// ---- rotation -----------------------------------------------------------------------------------------
// {batch stride, token stride, element stride} and batch rows of x[..., N, C] when the leading dims are one run
struct Rows { int64_t s[3], nb; };
bool rows_of(const Tensor& x, Rows& r) {
  const int64_t nd = x.dim();
  r.nb = 1;
  r.s[0] = 0;
  for (int64_t i = nd - 3; i >= 0; i--) {
    if (x.size(i) == 1) continue;
    if (r.nb == 1) r.s[0] = x.stride(i);
    else if (x.stride(i) != r.nb * r.s[0]) return false;
    r.nb *= x.size(i);
  }
  r.s[1] = x.stride(nd - 2);
  r.s[2] = x.stride(nd - 1);
  return true;
}

void rotate_inplace(const Tensor& x, const Rows& r, const Rope& rope, bool inverse) {
  c10::DeviceGuard guard(x.device());
  check_rc(dlt_rope2d(x.mutable_data_ptr(), r.s, r.nb, x.size(-2), x.size(-1), &rope.d, inverse, dtype_code(x), stream_of(x)));
}

variable_list RopeBackward::apply(variable_list&& grads) {
  std::lock_guard<std::mutex> lock(mutex_);
  if (!grads[0].defined()) grads[0] = input_metadata(0).zeros_like();
  const Tensor idx_ = idx.unpack(), row_ = row.unpack(), col_ = col.unpack();   // before the guard: see AttnBackward
  Tensor dy = grads[0], dx;
  {
    at::AutoDispatchBelowADInplaceOrView below;
    const Rope rope = make_rope(idx_, row_, col_);
    require_gpu(dy, rope.idx, rope.row, rope.col);
    Rows rs, rd;
    if (!rows_of(dy, rs)) {
      dy = dy.contiguous();
      rows_of(dy, rs);
    }
    c10::DeviceGuard guard(dy.device());
    dx = empty(dy.sizes(), dy.scalar_type(), dy);
    rows_of(dx, rd);
    check_rc(dlt_rope2d_copy(dy.const_data_ptr(), rs.s, dx.mutable_data_ptr(), rd.s, rd.nb, dy.size(-2), dy.size(-1), &rope.d, 1, dtype_code(dy),
                             stream_of(dy)));
  }
  // differentiable once: a second derivative raises where it is asked for (without a graph it would be dropped in silence)
  if (C10_UNLIKELY(at::GradMode::is_enabled() && grads[0].requires_grad())) {
    std::shared_ptr<torch::autograd::DelayedError> once(
        new torch::autograd::DelayedError("trying to differentiate twice a function that was marked with @once_differentiable", 1), torch::autograd::deleteNode);
    return (*once)({dx.detach().requires_grad_(true)});
  }
  return {dx};
}

// x[..., N, C] is rotated in place; the graph sees an in-place operation on x
void rope_apply(const Tensor& x, const Rows& r, const Tensor& idx, const Tensor& row, const Tensor& col) {
  check_assert(row.dim() == 3 && col.dim() == 3 && row.size(1) == col.size(1), "row and column table must have one R");
  check_assert(idx.dim() == 1 && idx.size(0) == x.size(-2), "idx must have one entry per token");
  require_gpu(x, idx, row, col);
  const bool grad = torch::autograd::compute_requires_grad(x);
  torch::autograd::check_inplace(x, grad);
  std::shared_ptr<RopeBackward> node;
  if (grad) {
    node = make_node<RopeBackward>();
    node->set_next_edges(torch::autograd::collect_next_edges(x));
    node->idx = SavedVariable(idx, false);
    node->row = SavedVariable(row, false);
    node->col = SavedVariable(col, false);
  }
  {
    at::AutoDispatchBelowADInplaceOrView below;
    rotate_inplace(x, r, make_rope(idx, row, col), false);
  }
  torch::autograd::increment_version(x);
  if (grad) torch::autograd::rebase_history(x, node);
}

// ---- arguments --------------------------------------------------------------------------------------------
const Tensor& tensor_arg(PyObject* o) {
  if (C10_UNLIKELY(!THPVariable_Check(o))) raise_py(PyExc_TypeError, std::string("expected a tensor, got ") + Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}

int64_t int_arg(PyObject* o) {
  const int64_t v = PyLong_Check(o) ? PyLong_AsLongLong(o) : [&] {
    PyObject* i = PyNumber_Index(o);
    if (i == nullptr) throw python_error();
    const int64_t r = PyLong_AsLongLong(i);
    Py_DECREF(i);
    return r;
  }();
  if (C10_UNLIKELY(v == -1 && PyErr_Occurred())) throw python_error();
  if (C10_UNLIKELY(v < INT32_MIN || v > INT32_MAX)) raise_py(PyExc_OverflowError, "argument does not fit 32 bits");
  return v;
}

double float_arg(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (C10_UNLIKELY(v == -1.0 && PyErr_Occurred())) throw python_error();
  return v;
}

bool bool_arg(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (C10_UNLIKELY(v < 0)) throw python_error();
  return v != 0;
}

void count(Py_ssize_t n, Py_ssize_t lo, Py_ssize_t hi) {
  if (C10_UNLIKELY(n < lo || n > hi)) raise_py(PyExc_TypeError, "takes " + std::to_string(hi) + " positional arguments, got " + std::to_string(n));
}

// ---- entry points: see the Python modules for what they do ----------------------------------------------------
PyObject* py_tiled_swa(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 9, 9);
  int64_t dims[5];
  for (int i = 0; i < 5; i++) dims[i] = int_arg(a[3 + i]);
  if (!plain(tensor_arg(a[0]), tensor_arg(a[1]), tensor_arg(a[2]))) Py_RETURN_NOTIMPLEMENTED;
  return THPVariable_Wrap(attention(Op::Swa, tensor_arg(a[0]), tensor_arg(a[1]), tensor_arg(a[2]), nullptr, dims, false, float_arg(a[8]), false, true));
  END_HANDLE_TH_ERRORS
}

PyObject* py_tiled_swa_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 9, 9);
  int64_t dims[5];
  for (int i = 0; i < 5; i++) dims[i] = int_arg(a[3 + i]);
  return THPVariable_Wrap(attention(Op::Swa, tensor_arg(a[0]), tensor_arg(a[1]), tensor_arg(a[2]), nullptr, dims, false, float_arg(a[8]), false, false));
  END_HANDLE_TH_ERRORS
}

PyObject* py_tiled_swa_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 12, 13);
  int64_t dims[5];
  for (int i = 0; i < 5; i++) dims[i] = int_arg(a[6 + i]);
  const Tensor rope[3] = {tensor_arg(a[3]), tensor_arg(a[4]), tensor_arg(a[5])};
  if (!plain(tensor_arg(a[0]), tensor_arg(a[1]), tensor_arg(a[2]), rope[0], rope[1], rope[2])) Py_RETURN_NOTIMPLEMENTED;
  const bool keep = n < 13 || a[12] == Py_None || bool_arg(a[12]);
  return THPVariable_Wrap(attention(Op::Swa, tensor_arg(a[0]), tensor_arg(a[1]), tensor_arg(a[2]), rope, dims, false, float_arg(a[11]), keep, true));
  END_HANDLE_TH_ERRORS
}

PyObject* py_tiled_swa_image(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 8, 8);
  int64_t dims[4];
  for (int i = 0; i < 4; i++) dims[i] = int_arg(a[3 + i]);
  if (!plain(tensor_arg(a[0]), tensor_arg(a[1]), tensor_arg(a[2]))) Py_RETURN_NOTIMPLEMENTED;
  return THPVariable_Wrap(attention(Op::Image, tensor_arg(a[0]), tensor_arg(a[1]), tensor_arg(a[2]), nullptr, dims, false, float_arg(a[7]), false, true));
  END_HANDLE_TH_ERRORS
}

PyObject* py_flash(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 5, 5);
  if (!plain(tensor_arg(a[0]), tensor_arg(a[1]), tensor_arg(a[2]))) Py_RETURN_NOTIMPLEMENTED;
  return THPVariable_Wrap(attention(Op::Flash, tensor_arg(a[0]), tensor_arg(a[1]), tensor_arg(a[2]), nullptr, nullptr, bool_arg(a[3]), float_arg(a[4]),
                                    false, true));
  END_HANDLE_TH_ERRORS
}

// (q, k, v, rope or None, keep_rot, B, H, b_size, th, tw, row, col, dk, dv, scale, dtype) -> (o, lse2[, q_rot, k_rot])
// and (q, k, v, o, lse2, do, rope or None, rotated, <the same 11 numbers>) -> (dq, dk, dv): one direction without a graph
Spec swa_spec_from(PyObject* const* a) {
  Spec s;
  s.op = Op::Swa;
  s.swa = {(int32_t)int_arg(a[0]), (int32_t)int_arg(a[1]), (int32_t)int_arg(a[2]), (int32_t)int_arg(a[3]), (int32_t)int_arg(a[4]), (int32_t)int_arg(a[5]),
           (int32_t)int_arg(a[6]), (int32_t)int_arg(a[7]), (int32_t)int_arg(a[8]), (float)float_arg(a[9]), (int32_t)int_arg(a[10])};
  return s;
}

bool rope_arg(PyObject* o, const Tensor& like, Rope& r) {
  if (o == Py_None) return false;
  require(PyTuple_Check(o) && PyTuple_GET_SIZE(o) == 3, PyExc_TypeError, "rope must be (idx, row table, column table)");
  r = make_rope_for(tensor_arg(PyTuple_GET_ITEM(o, 0)), tensor_arg(PyTuple_GET_ITEM(o, 1)), tensor_arg(PyTuple_GET_ITEM(o, 2)), like, like.size(2));
  return true;
}

PyObject* py_swa_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 16, 16);
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor &q = tensor_arg(a[0]), &k = tensor_arg(a[1]), &v = tensor_arg(a[2]);
  require_gpu(q, k, v);
  Rope r;
  const bool rope = rope_arg(a[3], q, r), keep = bool_arg(a[4]);
  const Forward f = run_forward(swa_spec_from(a + 5), q, k, v, rope ? &r : nullptr, keep);
  if (keep) return Py_BuildValue("(NNNN)", THPVariable_Wrap(f.o), THPVariable_Wrap(f.lse), THPVariable_Wrap(f.q_rot), THPVariable_Wrap(f.k_rot));
  return Py_BuildValue("(NN)", THPVariable_Wrap(f.o), THPVariable_Wrap(f.lse));
  END_HANDLE_TH_ERRORS
}

PyObject* py_swa_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 19, 19);
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor &q = tensor_arg(a[0]), &k = tensor_arg(a[1]), &v = tensor_arg(a[2]), &o = tensor_arg(a[3]), &lse = tensor_arg(a[4]), &d_o = tensor_arg(a[5]);
  Rope r;
  const bool rope = rope_arg(a[6], v, r), rotated = bool_arg(a[7]);
  auto g = run_backward(swa_spec_from(a + 8), q, k, v, o, lse, d_o, rope ? &r : nullptr, rotated);
  return Py_BuildValue("(NNN)", THPVariable_Wrap(g[0]), THPVariable_Wrap(g[1]), THPVariable_Wrap(g[2]));
  END_HANDLE_TH_ERRORS
}

// (q, k, v, bh, bw, row, col, scale) -> (o, lse2) and (q, k, v, o, lse2, do, the same 5 numbers) -> (dq, dk, dv): no graph
PyObject* py_image_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 8, 8);
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor &q = tensor_arg(a[0]), &k = tensor_arg(a[1]), &v = tensor_arg(a[2]);
  const int64_t dims[4] = {int_arg(a[3]), int_arg(a[4]), int_arg(a[5]), int_arg(a[6])};
  const Forward f = run_forward(image_spec(q, k, v, dims, float_arg(a[7])), q, k, v, nullptr, false);
  return Py_BuildValue("(NN)", THPVariable_Wrap(f.o), THPVariable_Wrap(f.lse));
  END_HANDLE_TH_ERRORS
}

PyObject* py_image_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 11, 11);
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor &q = tensor_arg(a[0]), &k = tensor_arg(a[1]), &v = tensor_arg(a[2]), &o = tensor_arg(a[3]), &lse = tensor_arg(a[4]), &d_o = tensor_arg(a[5]);
  const int64_t dims[4] = {int_arg(a[6]), int_arg(a[7]), int_arg(a[8]), int_arg(a[9])};
  auto g = run_backward(image_spec(q, k, v, dims, float_arg(a[10])), q, k, v, o, lse, d_o, nullptr, false);
  return Py_BuildValue("(NNN)", THPVariable_Wrap(g[0]), THPVariable_Wrap(g[1]), THPVariable_Wrap(g[2]));
  END_HANDLE_TH_ERRORS
}

// (q, k, v, o, M, do, causal, scale) -> (dq, dk, dv) without a graph and without padding
PyObject* py_flash_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 8, 8);
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor &q = tensor_arg(a[0]), &k = tensor_arg(a[1]), &v = tensor_arg(a[2]), &o = tensor_arg(a[3]), &lse = tensor_arg(a[4]), &d_o = tensor_arg(a[5]);
  auto g = run_backward(flash_spec(q, k, v, bool_arg(a[6]), float_arg(a[7])), q, k, v, o, lse, d_o, nullptr, false);
  return Py_BuildValue("(NNN)", THPVariable_Wrap(g[0]), THPVariable_Wrap(g[1]), THPVariable_Wrap(g[2]));
  END_HANDLE_TH_ERRORS
}

// (q, k, v, causal, scale) -> (o, M) without a graph and without padding
PyObject* py_flash_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 5, 5);
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor &q = tensor_arg(a[0]), &k = tensor_arg(a[1]), &v = tensor_arg(a[2]);
  const Forward f = run_forward(flash_spec(q, k, v, bool_arg(a[3]), float_arg(a[4])), q, k, v, nullptr, false);
  return Py_BuildValue("(NN)", THPVariable_Wrap(f.o), THPVariable_Wrap(f.lse));
  END_HANDLE_TH_ERRORS
}

// (x[B', N, C], idx, row, col): rotated in place, returned
PyObject* py_rope_apply(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 4, 4);
  const Tensor& x = tensor_arg(a[0]);
  if (!plain(x, tensor_arg(a[1]), tensor_arg(a[2]), tensor_arg(a[3]))) Py_RETURN_NOTIMPLEMENTED;
  if (x.dim() != 3) raise_py(PyExc_ValueError, "x must have shape [B', N, C]");
  Rows r;
  rows_of(x, r);
  rope_apply(x, r, tensor_arg(a[1]), tensor_arg(a[2]), tensor_arg(a[3]));
  Py_INCREF(a[0]);
  return a[0];
  END_HANDLE_TH_ERRORS
}

// (x[B, H, N, C], idx, row, col): rotated in place where B and H are one run of rows, else a rotated copy
PyObject* py_rope_heads(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 4, 4);
  const Tensor& x = tensor_arg(a[0]);
  if (!plain(x, tensor_arg(a[1]), tensor_arg(a[2]), tensor_arg(a[3]))) Py_RETURN_NOTIMPLEMENTED;
  if (x.dim() != 4) raise_py(PyExc_ValueError, "x must have shape [B, H, N, C]");
  Rows r;
  if (C10_LIKELY(rows_of(x, r))) {
    rope_apply(x, r, tensor_arg(a[1]), tensor_arg(a[2]), tensor_arg(a[3]));
    Py_INCREF(a[0]);
    return a[0];
  }
  Tensor y = x.reshape({-1, x.size(2), x.size(3)});
  rows_of(y, r);
  rope_apply(y, r, tensor_arg(a[1]), tensor_arg(a[2]), tensor_arg(a[3]));
  return THPVariable_Wrap(y.reshape(x.sizes()));
  END_HANDLE_TH_ERRORS
}

// (x[B', N, C], idx, row, col, inverse): in place, no graph
PyObject* py_rope_inplace(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 5, 5);
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor &x = tensor_arg(a[0]), &idx = tensor_arg(a[1]), &row = tensor_arg(a[2]), &col = tensor_arg(a[3]);
  require_gpu(x, idx, row, col);
  if (x.dim() != 3) raise_py(PyExc_ValueError, "x must have shape [B', N, C]");
  Rows r;
  rows_of(x, r);
  rotate_inplace(x, r, make_rope(idx, row, col), bool_arg(a[4]));
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// (q, k, idx, row, col, inverse): both in place with one launch, no graph
PyObject* py_rope_pair(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 6, 6);
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor &q = tensor_arg(a[0]), &k = tensor_arg(a[1]), &idx = tensor_arg(a[2]), &row = tensor_arg(a[3]), &col = tensor_arg(a[4]);
  require_gpu(q, k, idx, row, col);
  check_assert(q.dim() >= 2 && k.dim() >= 2 && q.size(-2) == k.size(-2) && q.size(-1) == k.size(-1) && q.scalar_type() == k.scalar_type(),
               "q and k must have one token count, head dim and dtype");
  check_assert(idx.dim() != 1 || idx.size(0) >= q.size(-2), "idx must have an entry for every token");
  Rows rq, rk;
  require(rows_of(q, rq) && rows_of(k, rk), PyExc_RuntimeError, "q and k must be viewable as [rows, N, C] (batch and head dims in one run)");
  const Rope rope = make_rope(idx, row, col);
  c10::DeviceGuard guard(q.device());
  check_rc(dlt_rope2d_pair(q.mutable_data_ptr(), rq.s, rq.nb, k.mutable_data_ptr(), rk.s, rk.nb, q.size(-2), q.size(-1), &rope.d, bool_arg(a[5]),
                           dtype_code(q), stream_of(q)));
  return PyTuple_Pack(2, a[0], a[1]);
  END_HANDLE_TH_ERRORS
}

// (dk, dv, dtype-carrying tensor, b_size) -> None or (dk, dv) to pad to; b_size -1: flash
PyObject* py_pad_plan(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  count(n, 4, 4);
  const int64_t dk = int_arg(a[0]), dv = int_arg(a[1]), b = int_arg(a[3]);
  const at::ScalarType dt = tensor_arg(a[2]).scalar_type();
  const Pad p = b < 0 ? flash_pad(dk, dv, dt) : swa_pad(dk, dv, dt, b);
  if (p.dk == dk && p.dv == dv) Py_RETURN_NONE;
  return Py_BuildValue("(LL)", (long long)p.dk, (long long)p.dv);
  END_HANDLE_TH_ERRORS
}

#define DLT_FN(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr}
PyMethodDef METHODS[] = {DLT_FN(tiled_swa), DLT_FN(tiled_swa_fwd), DLT_FN(tiled_swa_rope), DLT_FN(tiled_swa_image), DLT_FN(flash), DLT_FN(swa_forward),
                         DLT_FN(swa_backward), DLT_FN(image_forward), DLT_FN(image_backward), DLT_FN(flash_forward), DLT_FN(flash_backward), DLT_FN(rope_apply), DLT_FN(rope_heads), DLT_FN(rope_inplace), DLT_FN(rope_pair),
                         DLT_FN(pad_plan), {nullptr, nullptr, 0, nullptr}};
#undef DLT_FN

PyModuleDef MODULE = {PyModuleDef_HEAD_INIT, "_dlt_torch", "torch binding of libdlt_hip.so", -1, METHODS, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dlt_torch() {
  PyObject* lib = PyImport_ImportModule("dl_templates_amd._lib");
  if (lib == nullptr) return nullptr;
  g_dlt_error = PyObject_GetAttrString(lib, "DltError");
  Py_DECREF(lib);
  if (g_dlt_error == nullptr) return nullptr;
  return PyModule_Create(&MODULE);
}
