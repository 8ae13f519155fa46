// Native call path of the operator and of the decode step (module atomic_gdn2._bind).
//
// Small calls are bound by the host: through Python and ctypes a gradient evaluation costs about
// 200 us and a decode step 23 us (36 with reset flags to cast) before the GPU matters.  The functions here do the same work from
// C++ (the segment loop, the autograd node, allocation, the C-ABI calls of include/gdn2.h) for plain
// calls: CUDA tensors of one device, the shapes and dtypes the kernels take as they are, no
// dispatch modes, functorch wrappers or forward-mode tangents.  For anything else, and for whatever
// the library refuses, they return None and the caller goes on in Python, which casts, validates
// and raises.  MI355X, per pass: B1 H2 L256 gradient evaluation 209 -> 135 us, B1 H6 decode step
// 23.0 -> 6.4 us, B8 H16 with raw inputs and reset flags 36.4 -> 7.7 us.
//
// Nothing is kept between calls but the configuration a caller passed to op().
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "../../include/gdn2.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The C ABI, by address: the library that atomic_gdn2._lib has loaded.
struct Abi {
  decltype(&gdn2_residual_layout) residual_layout;
  decltype(&gdn2_fwd_workspace_bytes) fwd_ws;
  decltype(&gdn2_bwd_workspace_bytes) bwd_ws;
  decltype(&gdn2_fwd) fwd;
  decltype(&gdn2_fwd_bf16) fwd_bf16;
  decltype(&gdn2_bwd) bwd;
  decltype(&gdn2_decode_flags) decode;
  decltype(&gdn2_default_state_ckpt) default_ckpt;
  decltype(&gdn2_last_error) last_error;
} abi{};

// The library refused the call: the Python path raises what belongs to it.
struct Refused {};

const c10::DispatchKeySet kUnplain{c10::DispatchKey::Python,          c10::DispatchKey::PythonTLSSnapshot,
                                   c10::DispatchKey::Functionalize,   c10::DispatchKey::FuncTorchBatched,
                                   c10::DispatchKey::Batched,         c10::DispatchKey::FuncTorchGradWrapper,
                                   c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::VmapMode,
                                   c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                   c10::DispatchKey::FuncTorchDynamicLayerBackMode,
                                   c10::DispatchKey::Negative,        c10::DispatchKey::Conjugate,
                                   c10::DispatchKey::ZeroTensor};

bool plain_mode() {
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  return !tls.included_.has_any(kUnplain);
}
bool plain(const Tensor& t, const c10::Device& dev) {
  return t.defined() && t.layout() == c10::kStrided && t.device() == dev && !t.key_set().has_any(kUnplain) &&
         !t._fw_grad(0).defined();
}

void* stream_of(const c10::Device& dev) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream();
}
Tensor empty_on(const Tensor& like, at::IntArrayRef size, at::ScalarType dt) {
  return at::empty(size, at::TensorOptions().dtype(dt).device(like.device()));
}
float* f32_at(const Tensor& t, int64_t off = 0) { return t.defined() ? static_cast<float*>(t.data_ptr()) + off : nullptr; }

// One operator configuration: the descriptor without its shape (trivially copyable).
struct Op {
  gdn2_desc base;
  int64_t segment;     // tokens per segment (max_chunks_per_call * bt)

  // base.state_ckpt < 0: the library's choice for the shape
  gdn2_desc training_desc(int64_t B, int64_t H, int64_t L, int64_t D, int64_t seq_ld) const {
    gdn2_desc d = desc(B, H, L, D, seq_ld, base.state_ckpt);
    if (d.state_ckpt < 0) d.state_ckpt = abi.default_ckpt(&d);
    return d;
  }
  gdn2_desc desc(int64_t B, int64_t H, int64_t L, int64_t D, int64_t seq_ld, int ckpt) const {
    gdn2_desc d = base;
    d.B = (int32_t)B;
    d.H = (int32_t)H;
    d.L = (int32_t)L;
    d.D = (int32_t)D;
    d.seq_ld = (int32_t)seq_ld;
    d.state_ckpt = ckpt;
    return d;
  }
};

// A saved tensor as the backward takes it: saved-tensor hooks may give back other dtypes, strides or
// devices (brought back here) or another shape (refused).
Tensor restored(const Tensor& t, at::IntArrayRef size, at::ScalarType dt, const c10::Device& dev) {
  TORCH_CHECK(t.defined() && t.sizes() == size, "saved-tensor hooks gave back another shape than was saved");
  return t.to(dev, dt).contiguous();
}

// The identity on the gradients of a Sequence, as functions of what they were formed from; raises when
// they are differentiated.
struct Once : torch::autograd::Function<Once> {
  static variable_list forward(AutogradContext*, at::TensorList, const variable_list& grads) { return grads; }
  static variable_list backward(AutogradContext*, variable_list) {
    TORCH_CHECK(false, "the GDN-2 operator is once differentiable: its gradients cannot be differentiated");
  }
};

// The whole call as one autograd node: forward and backward run the segment loop over views of the
// full tensors (gdn2_desc.seq_ld), the state carried through h0 / h_final and dh0 / dh_final.
// float32 inputs and clip <= 1e4 (then the reference's final cast of the gradients is the identity).
struct Sequence : torch::autograd::Function<Sequence> {
  // (the node keeps a copy of the configuration: it may outlive the caller's)
  static variable_list forward(AutogradContext* ctx, const Op* op, const Tensor& q, const Tensor& k, const Tensor& v,
                               const Tensor& w, const Tensor& b, const Tensor& g, const std::optional<Tensor>& h0) {
    Tensor xs[6] = {q.contiguous(), k.contiguous(), v.contiguous(), w.contiguous(), b.contiguous(), g.contiguous()};
    Tensor h = h0 ? h0->contiguous() : Tensor();
    const int64_t B = q.size(0), H = q.size(1), L = q.size(2), D = q.size(3);
    c10::DeviceGuard guard(q.device());
    void* stream = stream_of(q.device());
    Tensor o = empty_on(q, {B, H, L, D}, at::kFloat);
    variable_list saved(xs, xs + 6);
    for (int64_t t0 = 0; t0 < L; t0 += op->segment) {
      const gdn2_desc d = op->training_desc(B, H, std::min(L - t0, op->segment), D, L);
      size_t off[GDN2_RES_COUNT], total = 0;
      if (abi.residual_layout(&d, off, &total)) throw Refused();
      Tensor res = empty_on(q, {(int64_t)total}, at::kByte);
      Tensor ws = empty_on(q, {(int64_t)abi.fwd_ws(&d, 1)}, at::kByte);
      Tensor hf = empty_on(q, {B, H, D, D}, at::kFloat);
      const int64_t x = t0 * D;
      if (abi.fwd(&d, f32_at(xs[0], x), f32_at(xs[1], x), f32_at(xs[2], x), f32_at(xs[3], x), f32_at(xs[4], x),
                  f32_at(xs[5], x), f32_at(h), f32_at(o, x), f32_at(hf), res.data_ptr(), ws.data_ptr(), stream))
        throw Refused();
      saved.push_back(res);
      h = hf;
    }
    ctx->save_for_backward(saved);
    ctx->saved_data["op"] = std::string(reinterpret_cast<const char*>(op), sizeof(Op));
    ctx->saved_data["h0"] = h0.has_value() && h0->requires_grad();
    ctx->saved_data["shape"] = std::vector<int64_t>{B, H, L, D};
    ctx->saved_data["device"] = q.device();
    return {o, h};
  }

  static variable_list backward(AutogradContext* ctx, variable_list gs) {
    const variable_list saved = ctx->get_saved_variables();
    Op conf;
    std::memcpy(&conf, ctx->saved_data["op"].toStringRef().data(), sizeof(Op));
    const Op* op = &conf;
    const std::vector<int64_t> shape = ctx->saved_data["shape"].toIntVector();
    const int64_t B = shape[0], H = shape[1], L = shape[2], D = shape[3];
    const c10::Device dev = ctx->saved_data["device"].toDevice();
    c10::DeviceGuard guard(dev);
    void* stream = stream_of(dev);
    Tensor xs[6];
    for (int i = 0; i < 6; ++i) xs[i] = restored(saved[i], shape, at::kFloat, dev);
    Tensor dout = gs[0].to(at::kFloat).contiguous(), dh = gs[1].to(at::kFloat).contiguous();
    Tensor gr[6];
    for (Tensor& t : gr) t = empty_on(xs[0], {B, H, L, D}, at::kFloat);
    const int64_t n_seg = (L + op->segment - 1) / op->segment;
    for (int64_t s = n_seg - 1; s >= 0; --s) {
      const int64_t t0 = s * op->segment, x = t0 * D;
      const gdn2_desc d = op->training_desc(B, H, std::min(L - t0, op->segment), D, L);
      size_t off[GDN2_RES_COUNT], total = 0;
      TORCH_CHECK(abi.residual_layout(&d, off, &total) == 0, "gdn2_bwd: ", abi.last_error());
      const Tensor res = restored(saved[6 + s], {(int64_t)total}, at::kByte, dev);
      Tensor ws = empty_on(xs[0], {(int64_t)abi.bwd_ws(&d)}, at::kByte);
      Tensor dh0 = empty_on(xs[0], {B, H, D, D}, at::kFloat);
      const int st = abi.bwd(&d, f32_at(xs[0], x), f32_at(xs[1], x), f32_at(xs[2], x), f32_at(xs[3], x),
                             f32_at(xs[4], x), f32_at(xs[5], x), res.data_ptr(), f32_at(dout, x), f32_at(dh),
                             f32_at(gr[0], x), f32_at(gr[1], x), f32_at(gr[2], x), f32_at(gr[3], x), f32_at(gr[4], x),
                             f32_at(gr[5], x), f32_at(dh0), ws.data_ptr(), stream);
      TORCH_CHECK(st == 0, "gdn2_bwd: ", abi.last_error());
      dh = dh0;
    }
    variable_list out{gr[0], gr[1], gr[2], gr[3], gr[4], gr[5], ctx->saved_data["h0"].toBool() ? dh : Tensor()};
    if (at::GradMode::is_enabled()) {
      // a backward that keeps its graph: the kernels' gradients have no derivative, and say so when asked
      if (!out.back().defined()) out.pop_back();
      variable_list from(gs);
      from.insert(from.end(), saved.begin(), saved.begin() + 6);
      // (copies made of strided inputs have no history: a leaf of its own keeps the node in the graph)
      from.push_back(at::empty({0}).requires_grad_(true));
      out = Once::apply(at::TensorList(from), out);
      out.resize(7);
    }
    out.insert(out.begin(), Tensor());
    return out;
  }
};

// No gradient: one kernel sequence over all L, float32 or bfloat16 inputs.
variable_list forward_only(const Op* op, const Tensor* in, const Tensor& h0) {
  const bool bf16 = in[0].scalar_type() == at::kBFloat16;
  Tensor xs[6];
  for (int i = 0; i < 6; ++i) xs[i] = in[i].contiguous();
  const Tensor h = h0.defined() ? h0.contiguous() : Tensor();
  const int64_t B = xs[0].size(0), H = xs[0].size(1), L = xs[0].size(2), D = xs[0].size(3);
  c10::DeviceGuard guard(xs[0].device());
  const gdn2_desc d = op->desc(B, H, L, D, 0, 0);
  Tensor o = empty_on(xs[0], {B, H, L, D}, at::kFloat), hf = empty_on(xs[0], {B, H, D, D}, at::kFloat);
  Tensor ws = empty_on(xs[0], {(int64_t)abi.fwd_ws(&d, 0)}, at::kByte);
  void* stream = stream_of(xs[0].device());
  int st;
  if (bf16) {
    auto p = [&](int i) { return static_cast<const uint16_t*>(xs[i].data_ptr()); };
    st = abi.fwd_bf16(&d, p(0), p(1), p(2), p(3), p(4), p(5), f32_at(h), f32_at(o), f32_at(hf), nullptr, ws.data_ptr(), stream);
  } else {
    st = abi.fwd(&d, f32_at(xs[0]), f32_at(xs[1]), f32_at(xs[2]), f32_at(xs[3]), f32_at(xs[4]), f32_at(xs[5]), f32_at(h),
                 f32_at(o), f32_at(hf), nullptr, ws.data_ptr(), stream);
  }
  if (st) throw Refused();
  return {o, hf};
}

// Runs f without the interpreter lock (a launch can block while the device's queue is full).
template <class F>
auto unlocked(F&& f) {
  struct Lock {
    PyThreadState* s = PyEval_SaveThread();
    ~Lock() { PyEval_RestoreThread(s); }
  } lock;
  return f();
}
PyObject* pair(const Tensor& a, const Tensor& b) {
  PyObject* x = THPVariable_Wrap(a);
  PyObject* y = x ? THPVariable_Wrap(b) : nullptr;
  PyObject* t = y ? PyTuple_Pack(2, x, y) : nullptr;
  Py_XDECREF(x);
  Py_XDECREF(y);
  return t;
}
PyObject* none() { Py_RETURN_NONE; }

// bind(addresses): the C ABI's entry points in the order of struct Abi
PyObject* py_bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  constexpr Py_ssize_t kN = sizeof(Abi) / sizeof(void*);
  if (n != kN) return PyErr_Format(PyExc_TypeError, "bind takes %zd addresses", kN);
  void* p[kN];
  for (Py_ssize_t i = 0; i < kN; ++i) {
    p[i] = PyLong_AsVoidPtr(args[i]);
    if (PyErr_Occurred()) return nullptr;
  }
  std::memcpy(static_cast<void*>(&abi), p, sizeof(abi));
  return none();
}

const char* const kOpName = "atomic_gdn2._bind.op";
void free_op(PyObject* cap) { delete static_cast<Op*>(PyCapsule_GetPointer(cap, kOpName)); }

// op(descriptor bytes, segment tokens): a configuration for sequence()
PyObject* py_op(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 2 || !PyBytes_Check(args[0]) || PyBytes_GET_SIZE(args[0]) != (Py_ssize_t)sizeof(gdn2_desc))
    return PyErr_Format(PyExc_TypeError, "op takes the bytes of a gdn2_desc and a token count");
  Op op;
  std::memcpy(&op.base, PyBytes_AS_STRING(args[0]), sizeof(gdn2_desc));
  op.segment = PyLong_AsLongLong(args[1]);
  if (PyErr_Occurred()) return nullptr;
  if (op.segment < 1) return PyErr_Format(PyExc_ValueError, "segment must be positive");
  return PyCapsule_New(new Op(op), kOpName, free_op);
}

// sequence(op, q, k, v, w, b, g, h0 or None) -> (o, h_final), or None: not a plain call
PyObject* py_sequence(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) return PyErr_Format(PyExc_TypeError, "sequence takes 8 arguments");
  const auto* held = static_cast<const Op*>(PyCapsule_GetPointer(args[0], kOpName));
  if (!held) return nullptr;
  const Op op = *held;
  for (int i = 1; i < 7; ++i)
    if (!THPVariable_Check(args[i])) return none();
  if (args[7] != Py_None && !THPVariable_Check(args[7])) return none();
  Tensor x[6], h0;
  for (int i = 0; i < 6; ++i) x[i] = THPVariable_Unpack(args[1 + i]);
  if (args[7] != Py_None) h0 = THPVariable_Unpack(args[7]);
  if (!plain_mode() || !x[0].is_cuda() || x[0].dim() != 4 || x[0].numel() == 0) return none();
  const c10::Device dev = x[0].device();
  const at::ScalarType dt = x[0].scalar_type();
  bool grad = false;
  for (const Tensor& t : x) {
    if (!plain(t, dev) || t.scalar_type() != dt || t.sizes() != x[0].sizes()) return none();
    grad = grad || t.requires_grad();
  }
  const int64_t L = x[0].size(2), D = x[0].size(3);
  for (int i = 0; i < 4; ++i)
    if (x[0].size(i) > INT32_MAX) return none();
  if (L % op.base.bt) return none();
  if (h0.defined()) {
    if (!plain(h0, dev) || h0.scalar_type() != at::kFloat || h0.dim() != 4 || h0.size(0) != x[0].size(0) ||
        h0.size(1) != x[0].size(1) || h0.size(2) != D || h0.size(3) != D)
      return none();
    grad = grad || h0.requires_grad();
  }
  grad = grad && at::GradMode::is_enabled();
  if (dt != at::kFloat && (grad || dt != at::kBFloat16)) return none();
  if (grad && !(op.base.clip <= 1e4)) return none();
  variable_list out;
  bool refused = false;
  unlocked([&] {
    try {
      if (grad)
        out = Sequence::apply(&op, x[0], x[1], x[2], x[3], x[4], x[5], h0.defined() ? std::optional<Tensor>(h0) : std::nullopt);
      else
        out = forward_only(&op, x, h0);
    } catch (const Refused&) {
      refused = true;
    }
  });
  return refused ? none() : pair(out[0], out[1]);
  END_HANDLE_TH_ERRORS
}

// decode(q, k, v, w, b, g, state, scale, reset or None, state is bf16, tau or None, fuse, a_log or
// None, dt_bias or None) -> (o, new state), or None: not a plain call
PyObject* py_decode(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 14) return PyErr_Format(PyExc_TypeError, "decode takes 14 arguments");
  for (int i = 0; i < 7; ++i)
    if (!THPVariable_Check(args[i])) return none();
  for (int i : {8, 12, 13})
    if (args[i] != Py_None && !THPVariable_Check(args[i])) return none();
  if (!PyFloat_Check(args[7]) || (args[10] != Py_None && !PyFloat_Check(args[10]))) return none();
  Tensor x[7], reset, a_log, dt_bias;
  for (int i = 0; i < 7; ++i) x[i] = THPVariable_Unpack(args[i]);
  if (args[8] != Py_None) reset = THPVariable_Unpack(args[8]);
  const bool sbf = PyObject_IsTrue(args[9]) == 1, fuse = PyObject_IsTrue(args[11]) == 1;
  if (args[12] != Py_None) a_log = THPVariable_Unpack(args[12]);
  if (args[13] != Py_None) dt_bias = THPVariable_Unpack(args[13]);
  if (!plain_mode() || !x[0].is_cuda() || x[0].dim() != 3 || x[0].numel() == 0) return none();
  const c10::Device dev = x[0].device();
  const int64_t B = x[0].size(0), H = x[0].size(1), D = x[0].size(2);
  const at::ScalarType dt = x[0].scalar_type(), sdt = sbf ? at::kBFloat16 : at::kFloat;
  if ((dt != at::kFloat && dt != at::kBFloat16) || (D != 64 && D != 128) || B * H > (int64_t(1) << 22)) return none();
  auto ready = [&](const Tensor& t, at::ScalarType ty) {
    return plain(t, dev) && t.scalar_type() == ty && t.is_contiguous() && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
  };
  for (int i = 0; i < 6; ++i)
    if (!ready(x[i], dt) || x[i].sizes() != x[0].sizes()) return none();
  if (!ready(x[6], sdt) || x[6].dim() != 4 || x[6].size(0) != B || x[6].size(1) != H || x[6].size(2) != D || x[6].size(3) != D)
    return none();
  int kind = 0;
  if (reset.defined()) {
    if (!plain(reset, dev) || !reset.is_contiguous() || reset.numel() != B) return none();
    switch (reset.scalar_type()) {
      case at::kBool: case at::kByte: kind = GDN2_FLAG_BYTE; break;
      case at::kInt: kind = GDN2_FLAG_INT32; break;
      case at::kLong: kind = GDN2_FLAG_INT64; break;
      default: return none();
    }
  }
  if (fuse && !(a_log.defined() && dt_bias.defined() && ready(a_log, at::kFloat) && ready(dt_bias, at::kFloat) &&
                a_log.numel() == H && dt_bias.numel() == D))
    return none();
  gdn2_decode_desc d{};
  d.B = (int32_t)B; d.H = (int32_t)H; d.D = (int32_t)D;
  d.n_tok = d.seq_ld = 1;
  d.in_dtype = d.out_dtype = dt == at::kBFloat16;
  d.state_dtype = sbf;
  d.fuse_prologue = fuse;
  d.cap = args[10] != Py_None;
  d.scale = PyFloat_AS_DOUBLE(args[7]);
  d.stability_tau = d.cap ? PyFloat_AS_DOUBLE(args[10]) : 0.0;
  Tensor o, st;
  int status = 0;
  unlocked([&] {
    c10::DeviceGuard guard(dev);
    o = empty_on(x[0], {B, H, D}, dt);
    st = empty_on(x[0], {B, H, D, D}, sdt);
    auto p = [&](const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; };
    status = abi.decode(&d, kind, p(x[0]), p(x[1]), p(x[2]), p(x[3]), p(x[4]), p(x[5]),
                        fuse ? f32_at(a_log) : nullptr, fuse ? f32_at(dt_bias) : nullptr, p(reset), p(x[6]), p(o), p(st),
                        stream_of(dev));
  });
  return status ? none() : pair(o, st);
  END_HANDLE_TH_ERRORS
}

// What a saved tensor looked like (lm_kernels.py): forty of them a block, looked over in Python at 1.5 us
// each, would be a fifth of a small block's host time.
struct Form {
  std::vector<int64_t> sizes;
  at::ScalarType dtype;
  c10::Device device;
};
const char* const kFormsName = "atomic_gdn2._bind.forms";
void free_forms(PyObject* cap) { delete static_cast<std::vector<Form>*>(PyCapsule_GetPointer(cap, kFormsName)); }
bool tensors_of(PyObject* t) {
  if (!PyTuple_Check(t)) return false;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(t); ++i)
    if (!THPVariable_Check(PyTuple_GET_ITEM(t, i))) return false;
  return true;
}

// forms(tensors): their sizes, dtypes and devices
PyObject* py_forms(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 1 || !tensors_of(args[0])) return PyErr_Format(PyExc_TypeError, "forms takes a tuple of tensors");
  auto f = std::make_unique<std::vector<Form>>();
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args[0]); ++i) {
    const Tensor& t = THPVariable_Unpack(PyTuple_GET_ITEM(args[0], i));
    f->push_back(Form{t.sizes().vec(), t.scalar_type(), t.device()});
  }
  PyObject* cap = PyCapsule_New(f.get(), kFormsName, free_forms);
  if (cap) f.release();
  return cap;
  END_HANDLE_TH_ERRORS
}

// differ(forms, tensors) -> None when every tensor has its form, contiguous and 16-byte aligned; else
// a list with (sizes, dtype, device) for those that do not, None for the others
PyObject* py_differ(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !tensors_of(args[1])) return PyErr_Format(PyExc_TypeError, "differ takes forms and a tuple of tensors");
  const auto* f = static_cast<const std::vector<Form>*>(PyCapsule_GetPointer(args[0], kFormsName));
  if (!f) return nullptr;
  if ((Py_ssize_t)f->size() != PyTuple_GET_SIZE(args[1])) return PyErr_Format(PyExc_ValueError, "another number of tensors");
  auto same = [&](const Tensor& t, const Form& o) {
    return t.layout() == c10::kStrided && t.sizes() == at::IntArrayRef(o.sizes) && t.scalar_type() == o.dtype &&
           t.device() == o.device && t.is_contiguous() && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
  };
  bool all = true;
  for (size_t i = 0; i < f->size() && all; ++i) all = same(THPVariable_Unpack(PyTuple_GET_ITEM(args[1], i)), (*f)[i]);
  if (all) return none();
  PyObject* out = PyList_New((Py_ssize_t)f->size());
  for (size_t i = 0; out && i < f->size(); ++i) {
    const Form& o = (*f)[i];
    PyObject* x = Py_None;
    if (same(THPVariable_Unpack(PyTuple_GET_ITEM(args[1], i)), o)) {
      Py_INCREF(x);
    } else {
      PyObject *sz = PyTuple_New((Py_ssize_t)o.sizes.size()), *dev = THPDevice_New(o.device);
      for (size_t k = 0; sz && k < o.sizes.size(); ++k) PyTuple_SET_ITEM(sz, (Py_ssize_t)k, PyLong_FromLongLong(o.sizes[k]));
      PyObject* dt = reinterpret_cast<PyObject*>(torch::getTHPDtype(o.dtype));
      x = sz && dev ? PyTuple_Pack(3, sz, dt, dev) : nullptr;
      Py_XDECREF(sz);
      Py_XDECREF(dev);
      if (!x) {
        Py_DECREF(out);
        return nullptr;
      }
    }
    PyList_SET_ITEM(out, (Py_ssize_t)i, x);
  }
  return out;
  END_HANDLE_TH_ERRORS
}

// dense(tensors, x) -> whether each is as the kernels read it: float32, on x's device, contiguous,
// 16-byte aligned, not empty
PyObject* py_dense(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !tensors_of(args[0]) || !THPVariable_Check(args[1])) return PyErr_Format(PyExc_TypeError, "dense takes a tuple of tensors and a tensor");
  const c10::Device dev = THPVariable_Unpack(args[1]).device();
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args[0]); ++i) {
    const Tensor& t = THPVariable_Unpack(PyTuple_GET_ITEM(args[0], i));
    if (t.layout() != c10::kStrided || t.device() != dev || t.scalar_type() != at::kFloat || t.numel() == 0 || !t.is_contiguous() ||
        (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) != 0)
      Py_RETURN_FALSE;
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)())py_bind, METH_FASTCALL, "bind(*addresses)"},
    {"op", (PyCFunction)(void (*)())py_op, METH_FASTCALL, "op(desc, segment)"},
    {"sequence", (PyCFunction)(void (*)())py_sequence, METH_FASTCALL, "sequence(op, q, k, v, w, b, g, h0)"},
    {"forms", (PyCFunction)(void (*)())py_forms, METH_FASTCALL, "forms(tensors)"},
    {"differ", (PyCFunction)(void (*)())py_differ, METH_FASTCALL, "differ(forms, tensors)"},
    {"dense", (PyCFunction)(void (*)())py_dense, METH_FASTCALL, "dense(tensors, x)"},
    {"decode", (PyCFunction)(void (*)())py_decode, METH_FASTCALL, "decode(...)"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module{PyModuleDef_HEAD_INIT, "_bind", "native call path of the operator", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__bind(void) { return PyModule_Create(&module); }
