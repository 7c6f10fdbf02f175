// The host path of the Python ops: argument checks, layout conversions, output allocation, autograd nodes and the C-ABI
// call of every op, as one CPython module (_host) over ATen.  The kernels of a decode token or of a small training
// step take 2-10 us each; driving them from Python (attribute look-ups, a ctypes structure per call, a Python autograd
// node with its saved tensors) took 14-17 us per forward op and more in the backward, so a program that calls six ops
// per layer and token waited for the interpreter.  Here a call is one METH_FASTCALL function and the graph nodes are
// torch::autograd::Function in C++, which the engine runs without taking the interpreter lock.
//
// Everything below works on tensors of one GPU and on torch's current stream; it keeps no state between calls.
#include <torch/extension.h>

#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <c10/hip/HIPStream.h>

#include <atomic>
#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/linearnexus_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;
typedef std::optional<Tensor> OptT;

PyObject* g_kernel_error = nullptr;  // linearnexus_amd._lib.HipKernelError

// A negative status of a C-ABI call; reaches Python as HipKernelError.
struct KernelError : std::runtime_error {
  using std::runtime_error::runtime_error;
};

void check_status(int status, const char* what) {
  if (status == 0) return;
  throw KernelError(std::string(what) + " failed (status " + std::to_string(status) + "): " + lnx_last_error());
}

// ---------------------------------------------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------------------------------------------

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

bool capturing(const Tensor& t) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  TORCH_CHECK(hipStreamIsCapturing(c10::hip::getCurrentHIPStream(t.get_device()).stream(), &status) == hipSuccess, "hipStreamIsCapturing failed");
  return status != hipStreamCaptureStatusNone;
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return static_cast<float*>(ptr(t)); }
OptT opt(const Tensor& t) { return t.defined() ? OptT(t) : OptT(); }
Tensor undef(const OptT& t) { return t.has_value() ? *t : Tensor(); }

bool known_dtype(at::ScalarType t) { return t == at::kFloat || t == at::kBFloat16; }
int code_of(at::ScalarType t) { return t == at::kBFloat16 ? LNX_BF16 : LNX_F32; }
at::ScalarType type_of(int64_t code) { return code == LNX_BF16 ? at::kBFloat16 : at::kFloat; }

Tensor f32(const Tensor& t) { return t.defined() ? t.to(at::kFloat).contiguous() : t; }

bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

// The kernels read values only: an input that carries a tangent would give a result without one, so it is refused, whether a gradient
// is wanted or not.
void refuse_tangents(const char* op, std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    TORCH_CHECK_NOT_IMPLEMENTED(!t->defined() || !t->_fw_grad(/*level=*/0).defined(), op, " has no forward-mode derivative (jvp)");
}

void refuse_tangents(const char* op, const variable_list& ts) {
  for (const Tensor& t : ts) refuse_tangents(op, {&t});
}

std::string shape_text(const Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + (t.dim() == 1 ? ",)" : ")");
}

// Memory layout of the token tensors.  The ops take the reference's head-first [B, H, T, .] shapes; a caller whose data
// lives token-first -- [B, T, H, .], what the reference's blocks hold before they transpose (delta_net.py:645-647) --
// passes x.transpose(1, 2) views, and the kernels then read and write that memory in place (`token_first` in the
// argument block) instead of working on contiguous copies.
bool is_token_first(const Tensor& x) {
  if (x.dim() < 3 || x.is_contiguous()) return false;
  int64_t want = 1;
  for (int64_t d = x.dim() - 1; d >= 0; --d) {
    const int64_t e = d == 2 ? 1 : d == 1 ? 2 : d;  // dimension d of the transposed tensor
    if (x.size(e) == 1) continue;
    if (x.stride(e) != want) return false;
    want *= x.size(e);
  }
  return true;
}

// `x` (logical [B, H, T, ...]) with dense memory in the chosen layout; no copy when it already has it.
Tensor as_layout(Tensor x, bool token_first) {
  if (!x.defined()) return x;
  if (reinterpret_cast<uintptr_t>(x.data_ptr()) % 16)  // a dense view that starts inside a 16-byte vector of its storage
    x = x.clone(at::MemoryFormat::Preserve);
  if (token_first) return is_token_first(x) ? x : x.transpose(1, 2).contiguous().transpose(1, 2);
  return x.contiguous();
}

Tensor empty_layout(int64_t B, int64_t H, int64_t T, int64_t d, const at::TensorOptions& o, bool token_first) {
  return token_first ? at::empty({B, T, H, d}, o).transpose(1, 2) : at::empty({B, H, T, d}, o);
}

void check_inputs(const Tensor& q, const Tensor& k, const Tensor& v) {
  const char* names = "qkv";
  const Tensor* ts[3] = {&q, &k, &v};
  for (int i = 0; i < 3; ++i)
    TORCH_CHECK(ts[i]->is_cuda(), names[i], " is on ", ts[i]->device().str(), "; the delta-rule ops run on the GPU only");
  TORCH_CHECK(known_dtype(q.scalar_type()), "unsupported dtype ", q.scalar_type(), ": use float32 or bfloat16");
  TORCH_CHECK(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type(), "q, k, v must share one dtype, got ",
              q.scalar_type(), ", ", k.scalar_type(), ", ", v.scalar_type());
  bool same = q.sizes() == k.sizes() && q.dim() == v.dim() && q.dim() > 0;
  for (int64_t i = 0; same && i + 1 < q.dim(); ++i) same = q.size(i) == v.size(i);
  TORCH_CHECK(same, "shape mismatch: q ", shape_text(q), " k ", shape_text(k), " v ", shape_text(v));
}

// LNX_GATE_NONE / SCALAR / VECTOR from g's shape over `lead` leading dimensions of q
int gate_kind(const Tensor& g, const Tensor& q) {
  if (!g.defined()) return LNX_GATE_NONE;
  const int64_t lead = q.dim() - 1;
  bool ok = g.dim() == lead || g.dim() == lead + 1;
  for (int64_t i = 0; ok && i < lead; ++i) ok = g.size(i) == q.size(i);
  if (ok && g.dim() == lead) return LNX_GATE_SCALAR;
  if (ok && g.size(lead) == q.size(lead)) return LNX_GATE_VECTOR;
  TORCH_CHECK(false, "gate shape ", shape_text(g), " matches neither the leading dimensions of q ", shape_text(q), " nor q's shape");
}

// ---------------------------------------------------------------------------------------------------------------
// arguments of a METH_FASTCALL function
// ---------------------------------------------------------------------------------------------------------------

struct Args {
  PyObject* const* a;
  Py_ssize_t n;
  Args(PyObject* const* args, Py_ssize_t nargs, Py_ssize_t want, const char* name) : a(args), n(nargs) {
    TORCH_CHECK(n == want, name, ": ", n, " arguments given, ", want, " expected");
  }
  bool is_tensor(int i) const { return THPVariable_Check(a[i]); }
  bool is_none(int i) const { return a[i] == Py_None; }
  Tensor tensor(int i, const char* name) const {
    if (!is_tensor(i)) C10_THROW_ERROR(TypeError, std::string(name) + " must be a torch.Tensor on an AMD GPU, got " + Py_TYPE(a[i])->tp_name);
    return THPVariable_Unpack(a[i]);
  }
  Tensor maybe(int i, const char* name) const { return is_none(i) ? Tensor() : tensor(i, name); }
  double number(int i) const {
    const double x = PyFloat_AsDouble(a[i]);
    if (x == -1.0 && PyErr_Occurred()) throw python_error();
    return x;
  }
  int64_t integer(int i) const {
    const int64_t x = PyLong_AsLongLong(a[i]);
    if (x == -1 && PyErr_Occurred()) throw python_error();
    return x;
  }
  bool flag(int i) const {
    const int x = PyObject_IsTrue(a[i]);
    if (x < 0) throw python_error();
    return x != 0;
  }
};

PyObject* pack(const Tensor& x, const Tensor& y) {
  PyObject* t = PyTuple_New(2);
  if (!t) throw python_error();
  auto wrap = [](const Tensor& z) -> PyObject* {
    if (z.defined()) return THPVariable_Wrap(z);
    Py_INCREF(Py_None);
    return Py_None;
  };
  PyTuple_SET_ITEM(t, 0, wrap(x));
  PyTuple_SET_ITEM(t, 1, wrap(y));
  return t;
}

// What an op does between reading its arguments and wrapping its results: allocations and launches, which can wait for the driver or for
// a full queue.  Other Python threads run meanwhile.  0.1 us a call.
struct NoLock {
  PyThreadState* state = PyEval_SaveThread();
  NoLock() = default;
  NoLock(const NoLock&) = delete;
  ~NoLock() { PyEval_RestoreThread(state); }
};
template <typename F> auto without_lock(F&& f) {
  const NoLock released;
  return f();
}

// Every entry point: C++ exceptions become Python ones (a failed C-ABI call: HipKernelError).
#define LNX_BEGIN HANDLE_TH_ERRORS try {
#define LNX_END                                      \
  }                                                  \
  catch (const KernelError& e) {                     \
    PyErr_SetString(g_kernel_error, e.what());       \
    return nullptr;                                  \
  }                                                  \
  END_HANDLE_TH_ERRORS

// ---------------------------------------------------------------------------------------------------------------
// decode step and token-by-token scan
// ---------------------------------------------------------------------------------------------------------------

lnx_scan_args base_args(int64_t B, int64_t H, int64_t T, int64_t dk, int64_t dv, int dtype, int o_dtype, int gate, bool l2norm, double scale) {
  lnx_scan_args a{};
  a.B = (int32_t)B, a.H = (int32_t)H, a.T = (int32_t)T, a.dk = (int32_t)dk, a.dv = (int32_t)dv;
  a.chunk = 64;
  a.dtype = dtype, a.o_dtype = o_dtype, a.gate = gate;
  a.use_qk_l2norm = l2norm;
  a.scale = (float)scale;
  return a;
}

// step(q, k, v, g, beta, state, scale or None, l2norm, output in the state's dtype, inplace): (o, state), or None where the
// inputs are not plain -- one dtype of the kernels, contiguous, fp32 beta, g and state, no gradient wanted -- and the caller
// has to convert them or to report what is wrong with them.
PyObject* py_step(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  LNX_BEGIN
  Args in(args, nargs, 10, "step");
  for (int i = 0; i < 6; ++i)
    if (!in.is_tensor(i) && !(i == 3 && in.is_none(i))) Py_RETURN_NONE;
  const Tensor q = THPVariable_Unpack(args[0]), k = THPVariable_Unpack(args[1]), v = THPVariable_Unpack(args[2]);
  const Tensor g = in.is_none(3) ? Tensor() : THPVariable_Unpack(args[3]);
  const Tensor beta = THPVariable_Unpack(args[4]), state = THPVariable_Unpack(args[5]);
  const auto dt = q.scalar_type();
  if (q.dim() != 3 || v.dim() != 3 || !q.is_cuda() || !k.is_cuda() || !v.is_cuda() || !known_dtype(dt) || k.scalar_type() != dt || v.scalar_type() != dt) Py_RETURN_NONE;
  const int64_t B = q.size(0), H = q.size(1), dk = q.size(2), dv = v.size(2);
  auto plain_f32 = [&](const Tensor& t) { return t.is_cuda() && t.scalar_type() == at::kFloat && t.is_contiguous(); };
  if (k.sizes() != q.sizes() || v.size(0) != B || v.size(1) != H || !q.is_contiguous() || !k.is_contiguous() || !v.is_contiguous() || !plain_f32(beta) ||
      !plain_f32(state) || state.sizes() != at::IntArrayRef({B, H, dk, dv}))
    Py_RETURN_NONE;
  if (!(beta.dim() == 2 || (beta.dim() == 3 && beta.size(2) == 1)) || beta.size(0) != B || beta.size(1) != H) Py_RETURN_NONE;
  int gate = LNX_GATE_NONE;
  if (g.defined()) {
    if (!plain_f32(g) || g.dim() < 2 || g.size(0) != B || g.size(1) != H) Py_RETURN_NONE;
    if (g.dim() == 2) gate = LNX_GATE_SCALAR;
    else if (g.dim() == 3 && g.size(2) == dk) gate = LNX_GATE_VECTOR;
    else Py_RETURN_NONE;
  }
  if (wants_grad({&q, &k, &v, &g, &beta, &state})) Py_RETURN_NONE;
  refuse_tangents("step", {&q, &k, &v, &g, &beta, &state});
  const bool l2norm = in.flag(7), o_f32 = in.flag(8), inplace = in.flag(9);
  const double scale = in.is_none(6) ? 1.0 / std::sqrt((double)dk) : in.number(6);
  const auto r = without_lock([&] {
    const Tensor s_out = inplace ? state : at::empty_like(state);
    const Tensor o = at::empty({B, H, dv}, q.options().dtype(o_f32 ? at::kFloat : dt));
    lnx_scan_args a = base_args(B, H, 1, dk, dv, code_of(dt), code_of(o.scalar_type()), gate, l2norm, scale);
    a.q = ptr(q), a.k = ptr(k), a.v = ptr(v), a.beta = fptr(beta), a.g = fptr(g);
    a.initial_state = fptr(state), a.final_state = fptr(s_out), a.o = ptr(o);
    check_status(lnx_decode_step(&a, stream_of(q)), "lnx_decode_step");
    return std::make_pair(o, s_out);
  });
  return pack(r.first, r.second);
  LNX_END
}

struct SeqShape {
  int64_t B, H, T, dk, dv, nseq, nstate;
  int gate;
};

// Shapes of a scan over [B, H, T, d] tensors.  cu: a device int32 table (or undefined), already checked by the caller.
SeqShape seq_shape(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, const Tensor& beta, const Tensor& cu) {
  check_inputs(q, k, v);
  TORCH_CHECK(q.dim() == 4, "scan ops take [B, H, T, d] tensors, got q ", shape_text(q));
  SeqShape s{q.size(0), q.size(1), q.size(2), q.size(3), v.size(3), 0, 0, 0};
  TORCH_CHECK(beta.dim() == 3 && beta.size(0) == s.B && beta.size(1) == s.H && beta.size(2) == s.T, "beta shape ", shape_text(beta),
              " != (", s.B, ", ", s.H, ", ", s.T, ")");
  s.gate = gate_kind(g, q);
  if (cu.defined()) {
    TORCH_CHECK(s.B == 1, "cu_seqlens needs a packed batch with B == 1");
    s.nseq = cu.numel() - 1;
  }
  s.nstate = s.nseq ? s.nseq : s.B;
  return s;
}

void check_state(const Tensor& s0, const SeqShape& s, int64_t dv) {
  if (!s0.defined()) return;
  TORCH_CHECK(s0.sizes() == at::IntArrayRef({s.nstate, s.H, s.dk, dv}), "initial_state shape ", shape_text(s0), " != (", s.nstate, ", ", s.H,
              ", ", s.dk, ", ", dv, ")");
}

// A trailing singleton of beta is accepted (delta_net.py:166-167, :257-258, :378-379).
Tensor squeeze_beta(const Tensor& beta, int64_t ndim) { return beta.dim() == ndim ? beta.squeeze(-1) : beta; }

// recurrent(q, k, v, g, beta, initial_state, scale, l2norm, cu)
PyObject* py_recurrent(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  LNX_BEGIN
  Args in(args, nargs, 9, "recurrent");
  const Tensor q0 = in.tensor(0, "q"), k0 = in.tensor(1, "k"), v0 = in.tensor(2, "v"), g0 = in.maybe(3, "g"), s0 = in.maybe(5, "initial_state"),
               cu = in.maybe(8, "cu_seqlens");
  const Tensor b0 = squeeze_beta(in.tensor(4, "beta"), 4);
  refuse_tangents("recurrent", {&q0, &k0, &v0, &g0, &b0, &s0});
  const SeqShape s = seq_shape(q0, k0, v0, g0, b0, cu);
  check_state(s0, s, s.dv);
  const bool l2norm = in.flag(7);
  const double scale = in.is_none(6) ? 1.0 / std::sqrt((double)s.dk) : in.number(6);
  const auto r = without_lock([&] {
    const bool tf = is_token_first(q0) && is_token_first(k0) && is_token_first(v0);
    const Tensor q = as_layout(q0, tf), k = as_layout(k0, tf), v = as_layout(v0, tf), beta = as_layout(b0.to(at::kFloat), tf);
    const Tensor g = g0.defined() ? as_layout(g0.to(at::kFloat), tf) : g0, si = f32(s0);
    const Tensor o = empty_layout(s.B, s.H, s.T, s.dv, q.options(), tf);
    const Tensor sT = at::empty({s.nstate, s.H, s.dk, s.dv}, q.options().dtype(at::kFloat));
    const int dt = code_of(q.scalar_type());
    lnx_scan_args a = base_args(s.B, s.H, s.T, s.dk, s.dv, dt, dt, s.gate, l2norm, scale);
    a.nseq = (int32_t)s.nseq;
    a.token_first = tf;
    a.q = ptr(q), a.k = ptr(k), a.v = ptr(v), a.beta = fptr(beta), a.g = fptr(g);
    a.initial_state = fptr(si), a.final_state = fptr(sT), a.o = ptr(o), a.cu_seqlens = static_cast<const int32_t*>(ptr(cu));
    check_status(lnx_recurrent_fwd(&a, stream_of(q)), "lnx_recurrent_fwd");
    return std::make_pair(o, sT);
  });
  return pack(r.first, r.second);
  LNX_END
}

// ---------------------------------------------------------------------------------------------------------------
// row normalisation
// ---------------------------------------------------------------------------------------------------------------

// A dense tensor over x's memory (or a copy); `turned`: its dimensions 1 and 2 are exchanged.
Tensor dense(const Tensor& x, bool& turned) {
  turned = !x.is_contiguous() && x.dim() >= 4 && is_token_first(x);  // with fewer dimensions it would move the last axis itself
  return turned ? x.transpose(1, 2) : x.contiguous();
}

Tensor l2norm_fwd(const Tensor& x0) {
  bool turned;
  const Tensor x = dense(x0, turned);
  Tensor y = at::empty_like(x);
  const int64_t d = x.size(-1);
  check_status(lnx_l2norm_fwd(ptr(x), ptr(y), d ? x.numel() / d : 0, (int32_t)d, code_of(x.scalar_type()), stream_of(x)), "lnx_l2norm_fwd");
  return turned ? y.transpose(1, 2) : y;
}

Tensor l2norm_bwd(const Tensor& x0, const Tensor& dy0) {
  bool turned;
  const Tensor x = dense(x0, turned), dy = (turned ? dy0.transpose(1, 2) : dy0).contiguous();
  Tensor dx = at::empty_like(x);
  const int64_t d = x.size(-1);
  check_status(lnx_l2norm_bwd(ptr(x), ptr(dy), ptr(dx), d ? x.numel() / d : 0, (int32_t)d, code_of(x.scalar_type()), stream_of(x)), "lnx_l2norm_bwd");
  return turned ? dx.transpose(1, 2) : dx;
}

// q and k of a chunk call (one shape, dense in the call's layout), one launch for both
std::pair<Tensor, Tensor> l2norm_pair_fwd(const Tensor& q0, const Tensor& k0) {
  bool turned_q, turned_k;
  const Tensor q = dense(q0, turned_q), k = dense(k0, turned_k);
  Tensor qn = at::empty_like(q), kn = at::empty_like(k);
  const int64_t d = q.size(-1);
  check_status(lnx_l2norm_pair_fwd(ptr(q), ptr(k), ptr(qn), ptr(kn), d ? q.numel() / d : 0, (int32_t)d, code_of(q.scalar_type()), stream_of(q)), "lnx_l2norm_pair_fwd");
  return {turned_q ? qn.transpose(1, 2) : qn, turned_k ? kn.transpose(1, 2) : kn};
}
std::pair<Tensor, Tensor> l2norm_pair_bwd(const Tensor& q0, const Tensor& k0, const Tensor& dq0, const Tensor& dk0) {
  bool turned_q, turned_k;
  const Tensor q = dense(q0, turned_q), k = dense(k0, turned_k);
  const Tensor gq = (turned_q ? dq0.transpose(1, 2) : dq0).contiguous(), gk = (turned_k ? dk0.transpose(1, 2) : dk0).contiguous();
  Tensor dq = at::empty_like(q), dk = at::empty_like(k);
  const int64_t d = q.size(-1);
  check_status(lnx_l2norm_pair_bwd(ptr(q), ptr(k), ptr(gq), ptr(gk), ptr(dq), ptr(dk), d ? q.numel() / d : 0, (int32_t)d, code_of(q.scalar_type()), stream_of(q)),
               "lnx_l2norm_pair_bwd");
  return {turned_q ? dq.transpose(1, 2) : dq, turned_k ? dk.transpose(1, 2) : dk};
}

struct L2NormFn : Function<L2NormFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x) {
    ctx->save_for_backward({x});
    return l2norm_fwd(x);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    refuse_tangents("the gradient of l2norm_rows", grads);
    const Tensor x = ctx->get_saved_variables()[0];
    return {l2norm_bwd(x, grads[0].to(x.scalar_type()))};
  }
};

PyObject* py_l2norm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  LNX_BEGIN
  Args in(args, nargs, 1, "l2norm");
  const Tensor x = in.tensor(0, "x");
  TORCH_CHECK(x.is_cuda() && x.dim() > 0 && known_dtype(x.scalar_type()), "l2norm_rows takes float32 or bfloat16 rows on the GPU, got ", shape_text(x), " ",
              x.scalar_type(), " on ", x.device().str());
  refuse_tangents("l2norm_rows", {&x});
  return THPVariable_Wrap(without_lock([&] { return wants_grad({&x}) ? L2NormFn::apply(x) : l2norm_fwd(x); }));
  LNX_END
}

// l2norm_bwd(x, dy): the vector-Jacobian product on its own
PyObject* py_l2norm_bwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  LNX_BEGIN
  Args in(args, nargs, 2, "l2norm_bwd");
  const Tensor x = in.tensor(0, "x"), dy = in.tensor(1, "dy");
  return THPVariable_Wrap(without_lock([&] { return l2norm_bwd(x, dy); }));
  LNX_END
}

// ---------------------------------------------------------------------------------------------------------------
// chunked scan
// ---------------------------------------------------------------------------------------------------------------

// What one chunk call is given besides its tensors.
struct ChunkOptions {
  double scale = 1.0, threshold = 0.0;
  bool l2norm = false, forward_only = false;
  int64_t o_dtype = 0;
  int64_t scan_slab = 0, out_slabs = 0;  // test hooks of lnx_scan_args
  Tensor cu;                             // sequence table of a packed batch, or undefined
};

// The call in the form the kernels take, kept for the backward pass.
struct ChunkCall {
  Tensor q_in, k_in;  // as given, in the call's layout (the gradient goes through the normalisation of these)
  Tensor qn, kn;      // what the kernels read: q_in and k_in, or their normalised copies
  Tensor v, beta, g, s0, cu, ws, A, bias;
  lnx_scan_args a{};
  bool norm_outside = false;
};

void set_gate(lnx_scan_args& a, const ChunkCall& c, double threshold) {
  if (!c.A.defined()) return;
  a.g = nullptr;
  a.gate_raw = ptr(c.g), a.gate_A_log = fptr(c.A), a.gate_bias = fptr(c.bias), a.gate_threshold = (float)threshold;
}

std::pair<Tensor, Tensor> chunk_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, const Tensor& beta, const Tensor& s0,
                                        const Tensor& A_log, const Tensor& g_bias, const ChunkOptions& opt_, ChunkCall& c) {
  const Tensor& cu = opt_.cu;
  const SeqShape s = seq_shape(q, k, v, g, beta, cu);
  check_state(s0, s, s.dv);
  const bool tf = is_token_first(q) && is_token_first(k) && is_token_first(v);
  c.q_in = as_layout(q, tf), c.k_in = as_layout(k, tf), c.v = as_layout(v, tf);
  c.beta = as_layout(beta.to(at::kFloat), tf);
  c.g = !g.defined() ? g : as_layout(A_log.defined() ? g : g.to(at::kFloat), tf);
  c.s0 = f32(s0), c.cu = cu;
  c.A = f32(A_log), c.bias = f32(g_bias);
  const auto o_t = type_of(opt_.o_dtype);
  const Tensor o = empty_layout(s.B, s.H, s.T, s.dv, q.options().dtype(o_t), tf);
  const Tensor sT = at::empty({s.nstate, s.H, s.dk, s.dv}, q.options().dtype(at::kFloat));
  lnx_scan_args a = base_args(s.B, s.H, s.T, s.dk, s.dv, code_of(q.scalar_type()), (int)opt_.o_dtype, s.gate, false, opt_.scale);
  a.test_scan_slab = (int32_t)opt_.scan_slab, a.test_out_slabs = (int32_t)opt_.out_slabs;
  // The reference's chunk path normalises in the input dtype before anything else (gated_deltanet.py:273-275,
  // kda.py:379-381).  Where the kernels scale the rows themselves (no normalised copies, gradients carried through the
  // normalisation inside lnx_chunk_bwd) they get the raw q and k; otherwise the rows are normalised first.
  const bool fused = opt_.l2norm && lnx_chunk_normalises_qk(&a);
  a.use_qk_l2norm = fused;
  c.norm_outside = opt_.l2norm && !fused;
  if (c.norm_outside) std::tie(c.qn, c.kn) = l2norm_pair_fwd(c.q_in, c.k_in);
  else c.qn = c.q_in, c.kn = c.k_in;
  a.nseq = (int32_t)s.nseq;
  a.token_first = tf;
  a.forward_only = opt_.forward_only;
  a.q = ptr(c.qn), a.k = ptr(c.kn), a.v = ptr(c.v), a.beta = fptr(c.beta), a.g = fptr(c.g);
  a.initial_state = fptr(c.s0), a.final_state = fptr(sT), a.o = ptr(o), a.cu_seqlens = static_cast<const int32_t*>(ptr(cu));
  set_gate(a, c, opt_.threshold);
  const uint64_t nbytes = lnx_chunk_workspace_bytes(&a);
  if (nbytes == 0 && s.T > 0 && s.B > 0) check_status(-2, "lnx_chunk_workspace_bytes");
  c.ws = at::empty({(int64_t)std::max<uint64_t>(nbytes, 1)}, q.options().dtype(at::kByte));
  a.workspace = ptr(c.ws), a.workspace_bytes = nbytes;
  check_status(lnx_chunk_fwd(&a, stream_of(q)), "lnx_chunk_fwd");
  c.a = a;
  return {o, sT};
}

// Pairs lnx_chunk_fwd with lnx_chunk_bwd (the role jax.custom_vjp plays for a JAX caller).
struct ChunkFn : Function<ChunkFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const OptT& g, const Tensor& beta, const OptT& s0,
                               const OptT& A_log, const OptT& g_bias, const ChunkOptions& opt_) {
    ChunkCall c;
    auto [o, sT] = chunk_forward(q, k, v, undef(g), beta, undef(s0), undef(A_log), undef(g_bias), opt_, c);
    ctx->save_for_backward({c.q_in, c.k_in, c.norm_outside ? c.qn : Tensor(), c.norm_outside ? c.kn : Tensor(), c.v, c.beta, c.g, c.s0, c.cu, c.ws, c.A, c.bias});
    const lnx_scan_args& a = c.a;
    auto kind = [](const OptT& t) { return (int64_t)(t.has_value() ? t->scalar_type() : at::kFloat); };
    ctx->saved_data["i"] = std::vector<int64_t>{a.B, a.H, a.T, a.dk, a.dv, a.dtype, a.o_dtype, a.gate, a.use_qk_l2norm, a.nseq, a.token_first, a.test_scan_slab,
                                                a.test_out_slabs, (int64_t)beta.scalar_type(), kind(g), kind(s0), kind(A_log), kind(g_bias)};
    ctx->saved_data["d"] = std::vector<double>{opt_.scale, opt_.threshold};
    // an output that takes no part in the loss arrives in backward() undefined, not as a tensor of zeros that a fill kernel
    // wrote and lnx_chunk_bwd would read: a null d_final_state is the kernels' "no gradient"
    ctx->set_materialize_grads(false);
    return {o, sT};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    refuse_tangents("the gradient of chunkwise", grads);
    const variable_list s = ctx->get_saved_variables();
    const std::vector<int64_t> m = ctx->saved_data["i"].toIntVector();
    const std::vector<double> d = ctx->saved_data["d"].toDoubleVector();
    ChunkCall c;
    c.q_in = s[0], c.k_in = s[1];
    c.norm_outside = s[2].defined();
    c.qn = c.norm_outside ? s[2] : s[0], c.kn = c.norm_outside ? s[3] : s[1];
    c.v = s[4], c.beta = s[5], c.g = s[6], c.s0 = s[7], c.cu = s[8], c.ws = s[9], c.A = s[10], c.bias = s[11];
    lnx_scan_args a = base_args(m[0], m[1], m[2], m[3], m[4], (int)m[5], (int)m[6], (int)m[7], m[8] != 0, d[0]);
    a.nseq = (int32_t)m[9], a.token_first = (int32_t)m[10];
    a.test_scan_slab = (int32_t)m[11], a.test_out_slabs = (int32_t)m[12];
    const bool tf = m[10] != 0;
    const auto o = c.qn.options();
    // in fp32 as the kernels can take it: rounded there, into a scratch tensor
    const Tensor given = grads[0];
    const bool rounds = given.defined() && given.scalar_type() == at::kFloat && given.numel() > 0 && !given.is_neg() && lnx_chunk_rounds_d_o(&a) &&
                        reinterpret_cast<uintptr_t>(given.data_ptr()) % 16 == 0 && (tf ? is_token_first(given) : given.is_contiguous());
    const Tensor d_o = rounds ? empty_layout(m[0], m[1], m[2], m[4], o, tf)
                              : as_layout(given.defined() ? given.to(c.qn.scalar_type()) : at::zeros({m[0], m[1], m[2], m[4]}, o), tf);
    const Tensor d_sT = f32(grads[1]);
    Tensor dq = at::empty_like(c.qn), dk = at::empty_like(c.kn), dv = at::empty_like(c.v), dbeta = at::empty_like(c.beta);
    Tensor dg = c.g.defined() ? at::empty_like(c.g) : Tensor(), ds0, dA, dbias;
    if (c.s0.defined()) ds0 = at::empty_like(c.s0);
    a.q = ptr(c.qn), a.k = ptr(c.kn), a.v = ptr(c.v), a.beta = fptr(c.beta), a.g = fptr(c.g);
    a.initial_state = fptr(c.s0), a.cu_seqlens = static_cast<const int32_t*>(ptr(c.cu));
    a.d_o = ptr(d_o), a.d_final_state = fptr(d_sT);
    a.d_q = ptr(dq), a.d_k = ptr(dk), a.d_v = ptr(dv), a.d_beta = fptr(dbeta), a.d_g = fptr(dg), a.d_initial_state = fptr(ds0);
    a.workspace = ptr(c.ws), a.workspace_bytes = (uint64_t)c.ws.numel();
    if (c.A.defined()) {  // g is the raw gate projection: its gradient and the activation's parameter gradients
      dA = at::empty_like(c.A);
      if (c.bias.defined()) dbias = at::empty_like(c.bias);
      set_gate(a, c, d[1]);
      a.d_g = nullptr;
      a.d_gate_raw = ptr(dg), a.d_gate_A_log = fptr(dA), a.d_gate_bias = fptr(dbias);
    }
    if (rounds) check_status(lnx_chunk_bwd_d_o32(&a, fptr(given), stream_of(c.qn)), "lnx_chunk_bwd_d_o32");
    else check_status(lnx_chunk_bwd(&a, stream_of(c.qn)), "lnx_chunk_bwd");
    if (c.norm_outside) std::tie(dq, dk) = l2norm_pair_bwd(c.q_in, c.k_in, dq, dk);
    auto to = [](const Tensor& t, int64_t type) { return t.defined() ? t.to((at::ScalarType)type) : t; };
    return {dq, dk, dv, to(dg, m[14]), to(dbeta, m[13]), to(ds0, m[15]), to(dA, m[16]), to(dbias, m[17]), Tensor()};
  }
};

std::pair<Tensor, Tensor> chunk_segmented(const Tensor& q0, const Tensor& k0, const Tensor& v0, const Tensor& g0, const Tensor& beta0, const Tensor& s00, double scale,
                                          bool l2norm, int64_t o_dtype, int64_t wanted) {
  at::NoGradGuard no_grad;
  const SeqShape s = seq_shape(q0, k0, v0, g0, beta0, Tensor());
  check_state(s00, s, s.dv);
  const int64_t rows = s.B * s.H, chunks = (s.T + 63) / 64, per = (chunks + wanted - 1) / wanted, nseg = (chunks + per - 1) / per;
  auto fold = [&](const Tensor& t) {
    if (!t.defined() || s.B == 1) return t;
    std::vector<int64_t> sizes = t.sizes().vec();
    sizes[0] = 1, sizes[1] = rows;
    return t.reshape(sizes);
  };
  const Tensor q1 = fold(q0), k1 = fold(k0), v1 = fold(v0);
  const bool tf = is_token_first(q1) && is_token_first(k1) && is_token_first(v1);
  Tensor q = as_layout(q1, tf), k = as_layout(k1, tf);
  const Tensor v = as_layout(v1, tf), beta = as_layout(fold(beta0).to(at::kFloat), tf), g = g0.defined() ? as_layout(fold(g0).to(at::kFloat), tf) : g0, s0 = f32(s00);
  const Tensor o = empty_layout(1, rows, s.T, s.dv, q.options().dtype(type_of(o_dtype)), tf);
  const Tensor sT = at::empty({s.B, s.H, s.dk, s.dv}, q.options().dtype(at::kFloat));
  lnx_scan_args a = base_args(1, rows, s.T, s.dk, s.dv, code_of(q.scalar_type()), (int)o_dtype, s.gate, false, scale);
  a.use_qk_l2norm = l2norm && lnx_chunk_normalises_qk(&a);
  if (l2norm && !a.use_qk_l2norm) std::tie(q, k) = l2norm_pair_fwd(q, k);
  a.token_first = tf, a.forward_only = 1;
  a.q = ptr(q), a.k = ptr(k), a.v = ptr(v), a.beta = fptr(beta), a.g = fptr(g);
  a.initial_state = fptr(s0), a.final_state = fptr(sT), a.o = ptr(o);
  const uint64_t nbytes = lnx_chunk_fwd_segmented_bytes(&a, (int32_t)nseg);
  const Tensor ws = at::empty({(int64_t)std::max<uint64_t>(nbytes, 1)}, q.options().dtype(at::kByte));
  a.workspace = ptr(ws), a.workspace_bytes = nbytes;
  check_status(lnx_chunk_fwd_segmented_final(&a, (int32_t)nseg, stream_of(q)), "lnx_chunk_fwd_segmented_final");
  return {s.B == 1 ? o : o.reshape({s.B, s.H, s.T, s.dv}), sT};
}

// chunk_segmented(q, k, v, g, beta, initial_state, scale, l2norm, o_dtype, nseg): (o, final state) of a forward-only call on dense
// sequences, cut into about nseg segments that run in parallel (lnx_chunk_fwd_segmented_final); batch rows become heads.
PyObject* py_chunk_segmented(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  LNX_BEGIN
  Args in(args, nargs, 10, "chunk_segmented");
  const Tensor q = in.tensor(0, "q"), k = in.tensor(1, "k"), v = in.tensor(2, "v"), g = in.maybe(3, "g"), s0 = in.maybe(5, "initial_state");
  const Tensor beta = squeeze_beta(in.tensor(4, "beta"), 4);
  refuse_tangents("chunkwise", {&q, &k, &v, &g, &beta, &s0});
  const double scale = in.number(6);
  const bool l2norm = in.flag(7);
  const int64_t o_dtype = in.integer(8), nseg = in.integer(9);
  const auto r = without_lock([&] { return chunk_segmented(q, k, v, g, beta, s0, scale, l2norm, o_dtype, nseg); });
  return pack(r.first, r.second);
  LNX_END
}

// chunk(q, k, v, g, beta, initial_state, scale, l2norm, o_dtype, cu, forward_only, A_log, g_bias, threshold,
//       scan_slab, out_slabs): (o or None, final state), in the graph unless forward_only
PyObject* py_chunk(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  LNX_BEGIN
  Args in(args, nargs, 16, "chunk");
  const Tensor q = in.tensor(0, "q"), k = in.tensor(1, "k"), v = in.tensor(2, "v"), g = in.maybe(3, "g"), s0 = in.maybe(5, "initial_state"),
               A_log = in.maybe(11, "A_log"), g_bias = in.maybe(12, "g_bias");
  const Tensor beta = squeeze_beta(in.tensor(4, "beta"), 4);
  refuse_tangents("chunkwise", {&q, &k, &v, &g, &beta, &s0, &A_log, &g_bias});
  ChunkOptions o;
  o.cu = in.maybe(9, "cu_seqlens");
  o.scale = in.number(6), o.l2norm = in.flag(7), o.o_dtype = in.integer(8), o.forward_only = in.flag(10);
  o.threshold = in.number(13), o.scan_slab = in.integer(14), o.out_slabs = in.integer(15);
  const auto r = without_lock([&]() -> std::pair<Tensor, Tensor> {
    if (!o.forward_only) {
      const variable_list r = ChunkFn::apply(q, k, v, opt(g), beta, opt(s0), opt(A_log), opt(g_bias), o);
      return {r[0], r[1]};
    }
    at::NoGradGuard no_grad;
    ChunkCall c;
    return chunk_forward(q, k, v, g, beta, s0, A_log, g_bias, o, c);
  });
  return pack(r.first, r.second);
  LNX_END
}

// ---------------------------------------------------------------------------------------------------------------
// short convolution
// ---------------------------------------------------------------------------------------------------------------

// What the kernels take besides the parameters: the inputs (contiguous), the cache before and after the call and the
// sequence table of a packed batch (each of the last three may be undefined).
struct ConvSide {
  Tensor x, cin, cout, cu;
};

// A buffer that the forward kernel has cleared, for the first backward pass of its node.  Only between eager passes: a captured
// backward pass is replayed and would find its own sums, and a captured forward pass clears the buffer at every replay, when it has long
// been somebody's gradient.
struct Cleared : torch::CustomClassHolder {
  Tensor buffer;
  std::atomic<bool> taken{false};
};

// zeroed: cleared by the kernel on its way, or undefined
Tensor conv_forward(const Tensor& w, const Tensor& bias, const ConvSide& side, int64_t act, const Tensor& zeroed = Tensor()) {
  const Tensor &x = side.x, &cin = side.cin, &cout = side.cout, &cu = side.cu;
  const int32_t B = (int32_t)x.size(0), T = (int32_t)x.size(1), D = (int32_t)x.size(2), K = (int32_t)w.size(0), dt = code_of(x.scalar_type());
  Tensor y = at::empty_like(x);
  if (zeroed.defined())
    check_status(lnx_conv1d_fwd_zero(ptr(x), fptr(w), fptr(bias), ptr(cin), static_cast<const int32_t*>(ptr(cu)), cu.defined() ? (int32_t)cu.numel() - 1 : 0, ptr(y),
                                     ptr(cout), fptr(zeroed), zeroed.numel(), B, T, D, K, dt, (int32_t)act, stream_of(x)), "lnx_conv1d_fwd_zero");
  else if (cu.defined())
    check_status(lnx_conv1d_packed_fwd(ptr(x), fptr(w), fptr(bias), static_cast<const int32_t*>(ptr(cu)), (int32_t)cu.numel() - 1, ptr(y), ptr(cout), T, D, K,
                                       dt, (int32_t)act, stream_of(x)), "lnx_conv1d_packed_fwd");
  else
    check_status(lnx_conv1d_fwd(ptr(x), fptr(w), fptr(bias), ptr(cin), ptr(y), ptr(cout), B, T, D, K, dt, (int32_t)act, stream_of(x)), "lnx_conv1d_fwd");
  return y;
}

// The cache after the call is filled on the side: it takes no part in the graph.
struct ConvFn : Function<ConvFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const OptT& bias, const OptT& cache, const ConvSide& side,
                        int64_t act, bool lost_cache) {
    const Tensor w = f32(weight), b = f32(undef(bias));
    // the parameters' gradients are sums that start from zero: this kernel clears them, the backward pass saves a launch
    auto cleared = c10::make_intrusive<Cleared>();
    if (capturing(x)) cleared->taken = true;
    else cleared->buffer = at::empty({w.size(0) + (b.defined() ? 1 : 0), w.size(1)}, w.options());
    Tensor y = conv_forward(w, b, side, act, cleared->buffer);
    ctx->saved_data["cleared"] = c10::IValue::make_capsule(cleared);
    ctx->save_for_backward({x.is_contiguous() ? x : side.x, w, b, lost_cache ? Tensor() : side.cin, side.cu});
    ctx->saved_data["i"] = std::vector<int64_t>{act, (int64_t)weight.scalar_type(), (int64_t)(bias.has_value() ? bias->scalar_type() : at::kFloat),
                                                (int64_t)(cache.has_value() ? cache->scalar_type() : at::kFloat), lost_cache,
                                                cache.has_value() && cache->requires_grad()};
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    refuse_tangents("the gradient of depthwise_conv1d_causal", grads);
    const variable_list s = ctx->get_saved_variables();
    const std::vector<int64_t> m = ctx->saved_data["i"].toIntVector();
    TORCH_CHECK(!m[4], "cannot differentiate through a convolution whose cache was updated in place");
    const Tensor &x = s[0], &w = s[1], &b = s[2], &cin = s[3], &cu = s[4];
    const int32_t B = (int32_t)x.size(0), T = (int32_t)x.size(1), D = (int32_t)x.size(2), K = (int32_t)w.size(0), dt = code_of(x.scalar_type()), act = (int32_t)m[0];
    const Tensor dy = grads[0].to(x.scalar_type()).contiguous();
    Tensor dx = at::empty_like(x), dw, db, dc;
    auto cleared = c10::static_intrusive_pointer_cast<Cleared>(ctx->saved_data["cleared"].toCapsule());
    if (!capturing(x) && !cleared->taken.exchange(true)) {
      const Tensor buffer = std::move(cleared->buffer);
      dw = b.defined() ? buffer.narrow(0, 0, K) : buffer;
      if (b.defined()) db = buffer.select(0, K);
      check_status(lnx_conv1d_bwd_add(ptr(x), fptr(w), fptr(b), ptr(cin), static_cast<const int32_t*>(ptr(cu)), cu.defined() ? (int32_t)cu.numel() - 1 : 0, ptr(dy),
                                      ptr(dx), fptr(dw), fptr(db), B, T, D, K, dt, act, stream_of(x)), "lnx_conv1d_bwd_add");
    } else if (dw = at::empty_like(w), db = b.defined() ? at::empty_like(b) : Tensor(); cu.defined())
      check_status(lnx_conv1d_packed_bwd(ptr(x), fptr(w), fptr(b), static_cast<const int32_t*>(ptr(cu)), (int32_t)cu.numel() - 1, ptr(dy), ptr(dx), fptr(dw),
                                         fptr(db), T, D, K, dt, act, stream_of(x)), "lnx_conv1d_packed_bwd");
    else
      check_status(lnx_conv1d_bwd(ptr(x), fptr(w), fptr(b), ptr(cin), ptr(dy), ptr(dx), fptr(dw), fptr(db), B, T, D, K, dt, act, stream_of(x)), "lnx_conv1d_bwd");
    if (cin.defined() && m[5] && K > 1) {
      dc = at::empty_like(cin);
      check_status(lnx_conv1d_cache_bwd(ptr(x), fptr(w), fptr(b), ptr(cin), ptr(dy), ptr(dc), B, T, D, K, dt, act, stream_of(x)), "lnx_conv1d_cache_bwd");
      dc = dc.to((at::ScalarType)m[3]);
    }
    return {dx, dw.to((at::ScalarType)m[1]), db.defined() ? db.to((at::ScalarType)m[2]) : db, dc, Tensor(), Tensor(), Tensor()};
  }
};

// conv1d(inputs, weight, bias, cache, activation code, inplace_cache, cu): (output, cache after the call)
PyObject* py_conv1d(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  LNX_BEGIN
  Args in(args, nargs, 7, "conv1d");
  TORCH_CHECK(in.is_tensor(0) && THPVariable_Unpack(args[0]).is_cuda(), "inputs must be a torch.Tensor on the GPU; the convolution runs on the GPU only");
  const Tensor x = in.tensor(0, "inputs"), weight = in.tensor(1, "weight"), bias = in.maybe(2, "bias"), cache = in.maybe(3, "cache"), cu = in.maybe(6, "cu_seqlens");
  refuse_tangents("depthwise_conv1d_causal", {&x, &weight, &bias, &cache});
  const int64_t act = in.integer(4);
  const bool inplace = in.flag(5);
  TORCH_CHECK(x.dim() == 3, "inputs must be [batch, seq, channels], got ", shape_text(x));
  TORCH_CHECK(known_dtype(x.scalar_type()), "unsupported dtype ", x.scalar_type(), ": use float32 or bfloat16");
  const int64_t B = x.size(0), D = x.size(2);
  TORCH_CHECK(weight.dim() == 2 && weight.size(1) == D, "weight must be [kernel, ", D, "], got ", shape_text(weight));
  const int64_t K = weight.size(0);
  TORCH_CHECK_VALUE(K >= 1, "kernel_size must be >= 1");  // conv.py:36-37
  TORCH_CHECK(K <= 4, "kernel_size ", K, " is not supported (1..4)");
  TORCH_CHECK(!bias.defined() || (bias.dim() == 1 && bias.size(0) == D), "bias must be [", D, "], got ", bias.defined() ? shape_text(bias) : "");
  TORCH_CHECK_VALUE(!cache.defined() || K == 1 || cache.sizes() == at::IntArrayRef({B, K - 1, D}),  // conv.py:49-53
                    "cache shape must be (batch, kernel-1, channels); got ", cache.defined() ? shape_text(cache) : "", " for kernel_size=", K);
  if (cu.defined()) {
    TORCH_CHECK(B == 1, "cu_seqlens needs a packed batch with B == 1");
    TORCH_CHECK(!cache.defined(), "a packed batch starts every sequence from a zero cache: pass cache=None");
  }
  Tensor cin, cout;  // cache before and after
  const bool kept = cache.defined() && K > 1, own = kept && inplace;
  TORCH_CHECK(!own || (cache.scalar_type() == x.scalar_type() && cache.is_contiguous()), "inplace_cache=True needs a contiguous cache of the inputs' dtype");
  const Tensor y = without_lock([&] {
    const Tensor xc = x.is_contiguous() ? x : x.detach().contiguous();
    if (own) {
      cin = cout = cache.detach();
    } else if (kept) {
      cin = cache.detach().to(x.scalar_type()).contiguous();
      cout = at::empty_like(cin);
    } else {
      cout = at::empty({B, K - 1, D}, x.options());
    }
    const ConvSide side{xc, cin, cout, cu};
    return wants_grad({&x, &weight, &bias, &cache}) ? ConvFn::apply(x, weight, opt(bias), opt(cache), side, act, own)
                                                    : conv_forward(f32(weight), f32(bias), side, act);
  });
  return pack(y, own ? cache : cout);
  LNX_END
}

// ---------------------------------------------------------------------------------------------------------------
// gated RMSNorm
// ---------------------------------------------------------------------------------------------------------------

Tensor rms_forward(const Tensor& x, const Tensor& gate, const Tensor& w, double eps) {
  Tensor y = at::empty_like(x);
  const int64_t d = x.size(-1);
  check_status(lnx_rmsnorm_gated_fwd(ptr(x), ptr(gate), fptr(w), ptr(y), d ? x.numel() / d : 0, (int32_t)d, (float)eps, code_of(x.scalar_type()), stream_of(x)),
               "lnx_rmsnorm_gated_fwd");
  return y;
}

struct RmsFn : Function<RmsFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x0, const OptT& gate0, const Tensor& weight, double eps) {
    const Tensor x = x0.contiguous(), gate = gate0.has_value() ? gate0->to(x.scalar_type()).contiguous() : Tensor(), w = f32(weight);
    ctx->save_for_backward({x, gate, w});
    ctx->saved_data["i"] = std::vector<int64_t>{(int64_t)weight.scalar_type(), (int64_t)(gate0.has_value() ? gate0->scalar_type() : at::kFloat)};
    ctx->saved_data["d"] = eps;
    return rms_forward(x, gate, w, eps);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    refuse_tangents("the gradient of rmsnorm_gated", grads);
    const variable_list s = ctx->get_saved_variables();
    const std::vector<int64_t> m = ctx->saved_data["i"].toIntVector();
    const Tensor &x = s[0], &gate = s[1], &w = s[2];
    const int64_t d = x.size(-1), rows = d ? x.numel() / d : 0;
    const int dt = code_of(x.scalar_type());
    const Tensor dy = grads[0].to(x.scalar_type()).contiguous();
    Tensor dx = at::empty_like(x), dg = gate.defined() ? at::empty_like(gate) : Tensor(), dw = at::empty_like(w);
    const uint64_t nws = lnx_rmsnorm_gated_bwd_workspace_bytes(rows, (int32_t)d, dt);
    const Tensor ws = at::empty({(int64_t)std::max<uint64_t>(nws, 1)}, x.options().dtype(at::kByte));
    check_status(lnx_rmsnorm_gated_bwd(ptr(x), ptr(gate), fptr(w), ptr(dy), ptr(dx), ptr(dg), fptr(dw), rows, (int32_t)d, (float)ctx->saved_data["d"].toDouble(), dt,
                                       ptr(ws), nws, stream_of(x)), "lnx_rmsnorm_gated_bwd");
    return {dx, dg.defined() ? dg.to((at::ScalarType)m[1]) : dg, dw.to((at::ScalarType)m[0]), Tensor()};
  }
};

// rmsnorm_gated(x, gate, weight, eps)
PyObject* py_rmsnorm_gated(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  LNX_BEGIN
  Args in(args, nargs, 4, "rmsnorm_gated");
  TORCH_CHECK(in.is_tensor(0) && THPVariable_Unpack(args[0]).is_cuda(), "x must be a torch.Tensor on the GPU; the op runs on the GPU only");
  const Tensor x = in.tensor(0, "x"), gate = in.maybe(1, "gate"), weight = in.tensor(2, "weight");
  const double eps = in.number(3);
  TORCH_CHECK(known_dtype(x.scalar_type()), "unsupported dtype ", x.scalar_type(), ": use float32 or bfloat16");
  TORCH_CHECK(!gate.defined() || gate.sizes() == x.sizes(), "gate shape ", gate.defined() ? shape_text(gate) : "", " != x shape ", shape_text(x));
  TORCH_CHECK(x.dim() > 0 && weight.dim() == 1 && weight.size(0) == x.size(-1), "weight must be [", x.dim() ? x.size(-1) : 0, "], got ", shape_text(weight));
  refuse_tangents("rmsnorm_gated", {&x, &gate, &weight});
  return THPVariable_Wrap(without_lock([&] {
    if (wants_grad({&x, &gate, &weight})) return RmsFn::apply(x, opt(gate), weight, eps);
    return rms_forward(x.contiguous(), gate.defined() ? gate.to(x.scalar_type()).contiguous() : gate, f32(weight), eps);
  }));
  LNX_END
}

// ---------------------------------------------------------------------------------------------------------------
// gate activations
// ---------------------------------------------------------------------------------------------------------------

std::pair<Tensor, Tensor> gdn_forward(const Tensor& a, const Tensor& b, const Tensor& A, const Tensor& bias, double beta_scale) {
  const int64_t H = A.size(0);
  const auto o = a.options().dtype(at::kFloat);
  const Tensor g = at::empty(a.sizes(), o), beta = b.defined() ? at::empty(a.sizes(), o) : Tensor();
  check_status(lnx_gdn_gate_fwd(ptr(a), ptr(b), fptr(A), fptr(bias), fptr(g), fptr(beta), H ? a.numel() / H : 0, (int32_t)H, (float)beta_scale,
                                code_of(a.scalar_type()), stream_of(a)), "lnx_gdn_gate_fwd");
  return {g, beta};
}

struct GdnGateFn : Function<GdnGateFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& a0, const OptT& b0, const Tensor& A_log, const OptT& dt_bias, double beta_scale) {
    const Tensor a = a0.contiguous(), b = b0.has_value() ? b0->to(a.scalar_type()).contiguous() : Tensor(), A = f32(A_log), bias = f32(undef(dt_bias));
    auto [g, beta] = gdn_forward(a, b, A, bias, beta_scale);
    ctx->save_for_backward({a, b, A, bias});
    auto kind = [](const OptT& t) { return (int64_t)(t.has_value() ? t->scalar_type() : at::kFloat); };
    ctx->saved_data["i"] = std::vector<int64_t>{(int64_t)A_log.scalar_type(), kind(dt_bias), kind(b0)};
    ctx->saved_data["d"] = beta_scale;
    ctx->set_materialize_grads(false);
    if (!beta.defined()) return {g};
    return {g, beta};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    refuse_tangents("the gradient of gated_deltanet_gate", grads);
    const variable_list s = ctx->get_saved_variables();
    const std::vector<int64_t> m = ctx->saved_data["i"].toIntVector();
    const Tensor &a = s[0], &b = s[1], &A = s[2], &bias = s[3];
    const int64_t H = A.size(0), rows = H ? a.numel() / H : 0;
    const Tensor d_g = f32(grads[0]), d_beta = b.defined() && grads.size() > 1 ? f32(grads[1]) : Tensor();
    Tensor d_a = at::empty_like(a), d_b = b.defined() ? at::empty_like(b) : Tensor(), d_A = at::empty_like(A), d_bias = bias.defined() ? at::empty_like(bias) : Tensor();
    const uint64_t nws = lnx_gdn_gate_bwd_workspace_bytes(rows, (int32_t)H);
    const Tensor ws = at::empty({(int64_t)std::max<uint64_t>(nws, 1)}, a.options().dtype(at::kByte));
    check_status(lnx_gdn_gate_bwd(ptr(a), ptr(b), fptr(A), fptr(bias), fptr(d_g), fptr(d_beta), ptr(d_a), ptr(d_b), fptr(d_A), fptr(d_bias), rows, (int32_t)H,
                                  (float)ctx->saved_data["d"].toDouble(), code_of(a.scalar_type()), ptr(ws), nws, stream_of(a)), "lnx_gdn_gate_bwd");
    auto to = [](const Tensor& t, int64_t type) { return t.defined() ? t.to((at::ScalarType)type) : t; };
    return {d_a, to(d_b, m[2]), to(d_A, m[0]), to(d_bias, m[1]), Tensor()};
  }
};

// gdn_gate(a, A_log, dt_bias, b, beta_scale): (g, beta or None)
PyObject* py_gdn_gate(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  LNX_BEGIN
  Args in(args, nargs, 5, "gdn_gate");
  TORCH_CHECK(in.is_tensor(0) && THPVariable_Unpack(args[0]).is_cuda(), "a must be a torch.Tensor on the GPU; the op runs on the GPU only");
  const Tensor a = in.tensor(0, "a"), A_log = in.tensor(1, "A_log"), dt_bias = in.maybe(2, "dt_bias"), b = in.maybe(3, "b");
  const double beta_scale = in.number(4);
  TORCH_CHECK(known_dtype(a.scalar_type()), "unsupported dtype ", a.scalar_type(), ": use float32 or bfloat16");
  TORCH_CHECK(A_log.dim() == 1 && a.dim() >= 1 && a.size(-1) == A_log.size(0), "a ", shape_text(a), " must end in the heads of A_log ", shape_text(A_log));
  TORCH_CHECK(!dt_bias.defined() || dt_bias.sizes() == A_log.sizes(), "dt_bias must be [", A_log.size(0), "], got ", dt_bias.defined() ? shape_text(dt_bias) : "");
  TORCH_CHECK(!b.defined() || b.sizes() == a.sizes(), "b ", b.defined() ? shape_text(b) : "", " must have a's shape ", shape_text(a));
  refuse_tangents("gated_deltanet_gate", {&a, &A_log, &dt_bias, &b});
  const auto r = without_lock([&]() -> std::pair<Tensor, Tensor> {
    if (wants_grad({&a, &A_log, &dt_bias, &b})) {
      const variable_list r = GdnGateFn::apply(a, opt(b), A_log, opt(dt_bias), beta_scale);
      return {r[0], r.size() > 1 ? r[1] : Tensor()};
    }
    return gdn_forward(a.contiguous(), b.defined() ? b.to(a.scalar_type()).contiguous() : b, f32(A_log), f32(dt_bias), beta_scale);
  });
  return pack(r.first, r.second);
  LNX_END
}

Tensor kda_gate_forward(const Tensor& g, const Tensor& A, const Tensor& bias, int64_t dk, double threshold, int64_t out_dtype) {
  const int64_t B = g.size(0), T = g.size(1), H = A.size(0);
  const Tensor out = at::empty({B, T, H, dk}, g.options().dtype(type_of(out_dtype)));
  check_status(lnx_kda_gate_fwd(ptr(g), fptr(A), fptr(bias), ptr(out), B * T, (int32_t)H, (int32_t)dk, (float)threshold, code_of(g.scalar_type()), (int32_t)out_dtype,
                                stream_of(g)), "lnx_kda_gate_fwd");
  return out;
}

struct KdaGateFn : Function<KdaGateFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& g0, const Tensor& A_log, const OptT& g_bias, int64_t dk, double threshold, int64_t out_dtype) {
    const Tensor g = g0.contiguous(), A = f32(A_log), bias = f32(undef(g_bias));
    ctx->save_for_backward({g, A, bias});
    ctx->saved_data["i"] = std::vector<int64_t>{dk, out_dtype, (int64_t)A_log.scalar_type(), (int64_t)(g_bias.has_value() ? g_bias->scalar_type() : at::kFloat)};
    ctx->saved_data["d"] = threshold;
    return kda_gate_forward(g, A, bias, dk, threshold, out_dtype);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    refuse_tangents("the gradient of kda_gate", grads);
    const variable_list s = ctx->get_saved_variables();
    const std::vector<int64_t> m = ctx->saved_data["i"].toIntVector();
    const Tensor &g = s[0], &A = s[1], &bias = s[2];
    const int64_t rows = g.size(0) * g.size(1), H = A.size(0), dk = m[0];
    const Tensor d_out = grads[0].to(type_of(m[1])).contiguous();
    Tensor d_g = at::empty_like(g), d_A = at::empty_like(A), d_b = bias.defined() ? at::empty_like(bias) : Tensor();
    const uint64_t nws = lnx_kda_gate_bwd_workspace_bytes(rows, (int32_t)H, (int32_t)dk);
    const Tensor ws = at::empty({(int64_t)std::max<uint64_t>(nws, 1)}, g.options().dtype(at::kByte));
    check_status(lnx_kda_gate_bwd(ptr(g), fptr(A), fptr(bias), ptr(d_out), ptr(d_g), fptr(d_A), fptr(d_b), rows, (int32_t)H, (int32_t)dk,
                                  (float)ctx->saved_data["d"].toDouble(), code_of(g.scalar_type()), (int32_t)m[1], ptr(ws), nws, stream_of(g)), "lnx_kda_gate_bwd");
    return {d_g, d_A.to((at::ScalarType)m[2]), d_b.defined() ? d_b.to((at::ScalarType)m[3]) : d_b, Tensor(), Tensor(), Tensor()};
  }
};

Tensor sigmoid_forward(const Tensor& x) {
  Tensor y = at::empty_like(x);
  check_status(lnx_sigmoid_fwd(fptr(x), fptr(y), x.numel(), stream_of(x)), "lnx_sigmoid_fwd");
  return y;
}

struct SigmoidFn : Function<SigmoidFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x) {
    const Tensor y = sigmoid_forward(f32(x));
    ctx->save_for_backward({y});
    ctx->saved_data["i"] = (int64_t)x.scalar_type();
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    refuse_tangents("the gradient of kda_gate", grads);
    const Tensor y = ctx->get_saved_variables()[0], dy = f32(grads[0]);
    Tensor dx = at::empty_like(y);
    check_status(lnx_sigmoid_bwd(fptr(y), fptr(dy), fptr(dx), y.numel(), stream_of(y)), "lnx_sigmoid_bwd");
    return {dx.to((at::ScalarType)ctx->saved_data["i"].toInt())};
  }
};

// kda_gate(g, A_log, head_k_dim, g_bias, beta, threshold, out_dtype): (activated gate, sigmoid(beta) or None)
PyObject* py_kda_gate(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  LNX_BEGIN
  Args in(args, nargs, 7, "kda_gate");
  TORCH_CHECK(in.is_tensor(0) && THPVariable_Unpack(args[0]).is_cuda(), "g must be a torch.Tensor on the GPU; the op runs on the GPU only");
  const Tensor g = in.tensor(0, "g"), A_log = in.tensor(1, "A_log"), g_bias = in.maybe(3, "g_bias"), beta = in.maybe(4, "beta");
  const int64_t dk = in.integer(2);
  const double threshold = in.number(5);
  TORCH_CHECK(known_dtype(g.scalar_type()), "unsupported dtype ", g.scalar_type(), ": use float32 or bfloat16");
  TORCH_CHECK(g.dim() == 3 && A_log.dim() == 1 && g.size(2) == A_log.size(0) * dk, "g ", shape_text(g), " must be [batch, seq, heads of A_log ", shape_text(A_log),
              " * ", dk, "]");
  TORCH_CHECK(!g_bias.defined() || (g_bias.dim() == 1 && g_bias.size(0) == g.size(2)), "g_bias must be [", g.size(2), "], got ", g_bias.defined() ? shape_text(g_bias) : "");
  refuse_tangents("kda_gate", {&g, &A_log, &g_bias, &beta});
  const int64_t out_dtype = in.is_none(6) ? code_of(g.scalar_type()) : in.integer(6);
  TORCH_CHECK(!beta.defined() || beta.is_cuda(), "beta is on ", beta.defined() ? beta.device().str() : "", "; the op runs on the GPU only");
  const auto r = without_lock([&]() -> std::pair<Tensor, Tensor> {
    const Tensor out = wants_grad({&g, &A_log, &g_bias}) ? KdaGateFn::apply(g, A_log, opt(g_bias), dk, threshold, out_dtype)
                                                         : kda_gate_forward(g.contiguous(), f32(A_log), f32(g_bias), dk, threshold, out_dtype);
    if (!beta.defined()) return {out, Tensor()};
    return {out, wants_grad({&beta}) ? SigmoidFn::apply(beta) : sigmoid_forward(f32(beta))};
  });
  return pack(r.first, r.second);
  LNX_END
}

// ---------------------------------------------------------------------------------------------------------------
// RWKV-7's diagonal-plus-low-rank rule
// ---------------------------------------------------------------------------------------------------------------

void check_dplr(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& a, const Tensor& b, const Tensor& gk, int64_t dims) {
  check_inputs(q, k, v);
  TORCH_CHECK(q.dim() == dims, "expected ", dims, "-dimensional q, got ", shape_text(q));
  const char* names[3] = {"a", "b", "gk"};
  const Tensor* ts[3] = {&a, &b, &gk};
  for (int i = 0; i < 3; ++i) {
    TORCH_CHECK(ts[i]->is_cuda(), names[i], " is on ", ts[i]->device().str(), "; the delta-rule ops run on the GPU only");
    TORCH_CHECK(ts[i]->sizes() == q.sizes(), names[i], " shape ", shape_text(*ts[i]), " != q shape ", shape_text(q));
  }
  TORCH_CHECK(a.scalar_type() == q.scalar_type() && b.scalar_type() == q.scalar_type(), "a and b must have q's dtype ", q.scalar_type(), ", got ", a.scalar_type(),
              ", ", b.scalar_type());
}

lnx_dplr_args dplr_args(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& a, const Tensor& b, const Tensor& gk, const Tensor& s_in, double scale, bool step) {
  lnx_dplr_args r{};
  r.B = (int32_t)q.size(0), r.H = (int32_t)q.size(1), r.T = step ? 1 : (int32_t)q.size(2);
  r.dk = (int32_t)q.size(-1), r.dv = (int32_t)v.size(-1);
  r.dtype = r.o_dtype = code_of(q.scalar_type());
  r.scale = (float)scale;
  r.q = ptr(q), r.k = ptr(k), r.v = ptr(v), r.a = ptr(a), r.b = ptr(b), r.gk = fptr(gk);
  r.initial_state = fptr(s_in);
  return r;
}

// q, k, v, a, b contiguous, gk and the states contiguous fp32
Tensor dplr_call(bool step, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& a, const Tensor& b, const Tensor& gk, const Tensor& s_in, const Tensor& s_out,
                 double scale) {
  Tensor o = at::empty_like(v);
  lnx_dplr_args r = dplr_args(q, k, v, a, b, gk, s_in, scale, step);
  r.o = ptr(o), r.final_state = fptr(s_out);
  if (step) check_status(lnx_dplr_step(&r, stream_of(q)), "lnx_dplr_step");
  else check_status(lnx_dplr_recurrent_fwd(&r, stream_of(q)), "lnx_dplr_recurrent_fwd");
  return o;
}

Tensor work_area(const Tensor& like, uint64_t bytes) { return at::empty({(int64_t)std::max<uint64_t>(bytes, 1)}, like.options().dtype(at::kByte)); }

// Whether the chunked kernels take a scan (lnx_dplr_chunk_fits, and tensors that start on 16-byte boundaries)
bool dplr_chunked(std::initializer_list<const Tensor*> ts, const Tensor& v) {
  const Tensor& q = **ts.begin();
  if (!lnx_dplr_chunk_fits((int32_t)q.size(0), (int32_t)q.size(1), (int32_t)q.size(2), (int32_t)q.size(3), (int32_t)v.size(3))) return false;
  for (const Tensor* t : ts)
    if (reinterpret_cast<uintptr_t>(t->data_ptr()) % 16) return false;
  return true;
}

// The scan; `kept`: receives the chunked kernels' tensors for the backward pass (undefined where the token kernels ran)
Tensor dplr_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& a, const Tensor& b, const Tensor& gk, const Tensor& s_in, const Tensor& s_out, double scale,
                    Tensor* kept) {
  if (!dplr_chunked({&q, &k, &v, &a, &b, &gk}, v)) return dplr_call(false, q, k, v, a, b, gk, s_in, s_out, scale);
  lnx_dplr_args r = dplr_args(q, k, v, a, b, gk, s_in, scale, false);
  Tensor o = at::empty_like(v);
  r.o = ptr(o), r.final_state = fptr(s_out);
  if (kept) *kept = work_area(q, lnx_dplr_chunk_bytes(r.B, r.H, r.T, LNX_DPLR_KEPT));
  const Tensor ws = work_area(q, lnx_dplr_chunk_bytes(r.B, r.H, r.T, kept ? LNX_DPLR_FWD_SCRATCH : LNX_DPLR_ONLY_SCRATCH));
  check_status(lnx_dplr_chunk_fwd(&r, kept ? ptr(*kept) : nullptr, ptr(ws), stream_of(q)), "lnx_dplr_chunk_fwd");
  return o;
}

Tensor dplr_state(const Tensor& q, const Tensor& v) { return at::empty({q.size(0), q.size(1), q.size(-1), v.size(-1)}, q.options().dtype(at::kFloat)); }

struct DplrFn : Function<DplrFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q0, const Tensor& k0, const Tensor& v0, const Tensor& a0, const Tensor& b0, const Tensor& gk0, const OptT& s0,
                               double scale) {
    const Tensor q = q0.contiguous(), k = k0.contiguous(), v = v0.contiguous(), a = a0.contiguous(), b = b0.contiguous(), gk = f32(gk0), s_in = f32(undef(s0));
    Tensor kept;
    const Tensor s_out = dplr_state(q, v), o = dplr_forward(q, k, v, a, b, gk, s_in, s_out, scale, &kept);
    ctx->save_for_backward({q, k, v, a, b, gk, s_in, kept});
    ctx->saved_data["i"] = std::vector<int64_t>{(int64_t)gk0.scalar_type(), (int64_t)(s0.has_value() ? s0->scalar_type() : at::kFloat), s0.has_value() && s0->requires_grad()};
    ctx->saved_data["d"] = scale;
    ctx->set_materialize_grads(false);
    return {o, s_out};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    refuse_tangents("the gradient of dplr_delta_rule_recurrent", grads);
    const variable_list s = ctx->get_saved_variables();
    const std::vector<int64_t> m = ctx->saved_data["i"].toIntVector();
    const Tensor &q = s[0], &k = s[1], &v = s[2], &a = s[3], &b = s[4], &gk = s[5], &s_in = s[6];
    const int64_t B = q.size(0), H = q.size(1), T = q.size(2), dk = q.size(3), dv = v.size(3);
    const auto dt = q.scalar_type();
    const auto fo = q.options().dtype(at::kFloat);
    const lnx_dplr_args args = dplr_args(q, k, v, a, b, gk, s_in, ctx->saved_data["d"].toDouble(), false);
    const Tensor d_o = grads[0].defined() ? as_layout(grads[0].to(dt), false) : at::zeros_like(v), d_s = f32(grads[1]);
    if (const Tensor& kept = s[7]; kept.defined()) {
      Tensor r[5] = {at::empty_like(q), at::empty_like(k), at::empty_like(v), at::empty_like(a), at::empty_like(b)}, dgk = at::empty_like(gk), d0;
      if (s_in.defined() && m[2]) d0 = at::empty_like(s_in);
      const Tensor ws = work_area(q, lnx_dplr_chunk_bytes(args.B, args.H, args.T, LNX_DPLR_BWD_SCRATCH));
      const lnx_dplr_chunk_grads cg{ptr(d_o), fptr(d_s), ptr(r[0]), ptr(r[1]), ptr(r[2]), ptr(r[3]), ptr(r[4]), fptr(dgk), fptr(d0)};
      check_status(lnx_dplr_chunk_bwd(&args, &cg, ptr(kept), ptr(ws), stream_of(q)), "lnx_dplr_chunk_bwd");
      return {r[0], r[1], r[2], r[3], r[4], dgk.to((at::ScalarType)m[0]), d0.defined() ? d0.to((at::ScalarType)m[1]) : d0, Tensor()};
    }
    lnx_dplr_bwd_args g{};
    g.fwd = args;
    Tensor tok = at::empty({5, B, H, T, dk}, fo), dvv = at::empty({B, H, T, dv}, fo), ds0;
    if (s_in.defined() && m[2]) ds0 = at::empty_like(s_in);
    const uint64_t nws = lnx_dplr_recurrent_bwd_workspace_bytes((int32_t)B, (int32_t)H, (int32_t)T, (int32_t)dk, (int32_t)dv);
    const Tensor ws = at::empty({(int64_t)std::max<uint64_t>(nws, 1)}, q.options().dtype(at::kByte));
    g.d_o = ptr(d_o), g.d_final_state = fptr(d_s);
    Tensor r[5];
    for (int i = 0; i < 5; ++i) r[i] = tok[i];
    g.dq = fptr(r[0]), g.dk = fptr(r[1]), g.dv = fptr(dvv), g.da = fptr(r[2]), g.db = fptr(r[3]), g.dgk = fptr(r[4]);
    g.d_initial_state = fptr(ds0), g.workspace = ptr(ws), g.workspace_bytes = nws;
    check_status(lnx_dplr_recurrent_bwd(&g, stream_of(q)), "lnx_dplr_recurrent_bwd");
    return {r[0].to(dt), r[1].to(dt), dvv.to(dt), r[2].to(dt), r[3].to(dt), r[4].to((at::ScalarType)m[0]), ds0.defined() ? ds0.to((at::ScalarType)m[1]) : ds0, Tensor()};
  }
};

std::pair<Tensor, Tensor> dplr_scan(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& a, const Tensor& b, const Tensor& gk, const Tensor& s0, double scale) {
  if (wants_grad({&q, &k, &v, &a, &b, &gk, &s0})) {
    TORCH_CHECK(v.size(-1) <= 256, "the DPLR backward kernel takes dv <= 256, got ", v.size(-1));
    const variable_list r = DplrFn::apply(q, k, v, a, b, gk, opt(s0), scale);
    return {r[0], r[1]};
  }
  const Tensor s_out = dplr_state(q, v);
  return {dplr_forward(q.contiguous(), k.contiguous(), v.contiguous(), a.contiguous(), b.contiguous(), f32(gk), f32(s0), s_out, scale, nullptr), s_out};
}

// dplr(q, k, v, a, b, gk, scale, initial_state)
PyObject* py_dplr(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  LNX_BEGIN
  Args in(args, nargs, 8, "dplr");
  const Tensor q = in.tensor(0, "q"), k = in.tensor(1, "k"), v = in.tensor(2, "v"), a = in.tensor(3, "a"), b = in.tensor(4, "b"), gk = in.tensor(5, "gk"),
               s0 = in.maybe(7, "initial_state");
  refuse_tangents("dplr_delta_rule_recurrent", {&q, &k, &v, &a, &b, &gk, &s0});
  check_dplr(q, k, v, a, b, gk, 4);
  TORCH_CHECK(!s0.defined() || s0.sizes() == at::IntArrayRef({q.size(0), q.size(1), q.size(3), v.size(3)}), "initial_state shape ",
              s0.defined() ? shape_text(s0) : "", " != (", q.size(0), ", ", q.size(1), ", ", q.size(3), ", ", v.size(3), ")");
  const double scale = in.number(6);
  const auto r = without_lock([&] { return dplr_scan(q, k, v, a, b, gk, s0, scale); });
  return pack(r.first, r.second);
  LNX_END
}

// dplr_step(q, k, v, a, b, gk, state, scale, inplace)
PyObject* py_dplr_step(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  LNX_BEGIN
  Args in(args, nargs, 9, "dplr_step");
  const Tensor q = in.tensor(0, "q"), k = in.tensor(1, "k"), v = in.tensor(2, "v"), a = in.tensor(3, "a"), b = in.tensor(4, "b"), gk = in.tensor(5, "gk"),
               state = in.tensor(6, "state");
  const double scale = in.number(7);
  const bool inplace = in.flag(8);
  refuse_tangents("dplr_delta_rule_step", {&q, &k, &v, &a, &b, &gk, &state});
  check_dplr(q, k, v, a, b, gk, 3);
  TORCH_CHECK(state.sizes() == at::IntArrayRef({q.size(0), q.size(1), q.size(2), v.size(2)}), "state shape ", shape_text(state), " != (", q.size(0), ", ", q.size(1), ", ",
              q.size(2), ", ", v.size(2), ")");
  const bool grad = wants_grad({&q, &k, &v, &a, &b, &gk, &state});
  TORCH_CHECK(!grad || !inplace, "cannot differentiate through a step that updates its state in place");
  TORCH_CHECK(!inplace || (state.scalar_type() == at::kFloat && state.is_contiguous()), "inplace=True needs a contiguous float32 state");
  const auto r = without_lock([&]() -> std::pair<Tensor, Tensor> {
    if (grad) {
      const auto r = dplr_scan(q.unsqueeze(2), k.unsqueeze(2), v.unsqueeze(2), a.unsqueeze(2), b.unsqueeze(2), gk.unsqueeze(2), state, scale);
      return {r.first.squeeze(2), r.second};
    }
    const Tensor s_in = f32(state), s_out = inplace ? state : at::empty_like(s_in);
    return {dplr_call(true, q.contiguous(), k.contiguous(), v.contiguous(), a.contiguous(), b.contiguous(), f32(gk), s_in, s_out, scale), s_out};
  });
  return pack(r.first, r.second);
  LNX_END
}

// set_kernel_error(class): the exception a failed C-ABI call raises
PyObject* py_set_kernel_error(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 1 || !PyExceptionClass_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "set_kernel_error takes an exception class");
    return nullptr;
  }
  Py_INCREF(args[0]);
  Py_XSETREF(g_kernel_error, args[0]);
  Py_RETURN_NONE;
}

#define LNX_FN(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {LNX_FN(step),     LNX_FN(recurrent), LNX_FN(l2norm), LNX_FN(l2norm_bwd), LNX_FN(chunk), LNX_FN(chunk_segmented),     LNX_FN(conv1d),           LNX_FN(rmsnorm_gated), LNX_FN(gdn_gate),
                         LNX_FN(kda_gate), LNX_FN(dplr),      LNX_FN(dplr_step), LNX_FN(set_kernel_error), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", "Host path of the linearnexus_amd ops.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  Py_INCREF(PyExc_RuntimeError);
  g_kernel_error = PyExc_RuntimeError;
  return PyModule_Create(&module_def);
}
