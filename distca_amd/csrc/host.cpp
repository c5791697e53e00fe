// The host side of the calls a training step makes on its critical path, as native code: argument checks, allocation of results and
// workspace, the current stream, the C ABI call, and for core attention the autograd node.
//
// What bounds it: for a step of few tokens the host is slower than the device.  Written in Python (ctypes, torch.autograd.Function) core
// attention over 389 tokens cost 82 us of host time forward and backward, most of it interpreting, and the backward half ran in
// autograd's device thread, which had to take the interpreter's lock from the caller's: 96 us a step where the two threads shared
// a cache, 190 to 215 us where they did not.  Here the backward takes no lock and runs no bytecode.
//
// Everything is computed through libdistca_ca.so; nothing here touches device memory.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/Functions.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <cmath>
#include <optional>
#include <stdexcept>
#include <string>

#include "../../include/distca_ca.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

constexpr int64_t kHeadDim = 128;   // what the kernels are built for; smaller head dimensions are zero-padded to it on the way in

[[noreturn]] void fail(const std::string &what) { throw std::runtime_error(what); }
[[noreturn]] void type_error(const std::string &what) {
  PyErr_SetString(PyExc_TypeError, what.c_str());
  throw python_error();
}

void check_rc(int64_t rc, const char *what) {
  if (rc != 0) {
    const char *msg = distca_last_error();
    fail(std::string(what) + " failed (" + std::to_string(rc) + "): " + (msg ? msg : ""));
  }
}

// The device of a tensor made current for a scope, where it is not already, and its current stream.
struct OnDevice {
  c10::OptionalDeviceGuard guard;
  void *stream;
  explicit OnDevice(c10::Device d) {
    if (d.index() != c10::hip::current_device()) guard.reset_device(d);
    stream = c10::hip::getCurrentHIPStream(d.index()).stream();
  }
};

bool elem_code(const Tensor &t, int32_t *code) {
  switch (t.scalar_type()) {
    case at::kHalf: *code = DISTCA_DTYPE_F16; return true;
    case at::kBFloat16: *code = DISTCA_DTYPE_BF16; return true;
    default: return false;
  }
}

// One batch of tasks, as ca_varlen_fwd and ca_varlen_bwd take it.
struct Batch {
  Tensor q, k, v, cu_q, cu_k;
  OptTensor kv_off;
  int64_t max_q, max_k;
  std::optional<double> scale;
  bool causal;

  void check() const {
    int32_t code;
    const struct { const char *name; const Tensor &t; } rows[] = {{"q", q}, {"k", k}, {"v", v}};
    for (const auto &r : rows) {
      if (r.t.dim() != 3) fail(std::string(r.name) + " must have shape [tokens, heads, head_dim]");
      if (!r.t.is_cuda()) fail(std::string(r.name) + " must be on CUDA");
      if (!elem_code(r.t, &code) || r.t.scalar_type() != q.scalar_type())
        fail(std::string(r.name) + " must be bfloat16 or float16, the same for q, k and v (got " + c10::toString(r.t.scalar_type()) + ")");
      if (!r.t.is_contiguous()) fail(std::string(r.name) + " must be contiguous");
    }
    if (k.sizes() != v.sizes()) fail("k and v must have the same shape");
    if (q.size(2) != k.size(2)) fail("q and k must have the same head_dim");
    const struct { const char *name; const Tensor &t; } lens[] = {{"cu_seqlens_q", cu_q}, {"cu_seqlens_k", cu_k}};
    for (const auto &r : lens)
      if (r.t.scalar_type() != at::kInt || !r.t.is_cuda() || r.t.dim() != 1 || !r.t.is_contiguous())
        fail(std::string(r.name) + " must be a contiguous 1-D int32 CUDA tensor");
    if (cu_q.size(0) != cu_k.size(0)) fail("cu_seqlens_q and cu_seqlens_k must have the same shape");
    if (kv_off && (kv_off->scalar_type() != at::kInt || !kv_off->is_cuda() || kv_off->dim() < 1 || kv_off->size(0) != cu_q.size(0) - 1))
      fail("kv_task_offsets must be an int32 CUDA tensor of shape [num_tasks]");
  }

  double scale_or_default() const { return scale ? *scale : std::pow((double)q.size(2), -0.5); }

  distca_ca_params params(bool deterministic) const {
    distca_ca_params p{};
    p.num_tasks = (int32_t)cu_q.size(0) - 1;
    p.total_q = (int32_t)q.size(0);
    p.total_k = (int32_t)k.size(0);
    p.num_heads_q = (int32_t)q.size(1);
    p.num_heads_kv = (int32_t)k.size(1);
    p.head_dim = (int32_t)q.size(2);
    p.max_seqlen_q = (int32_t)max_q;
    p.max_seqlen_k = (int32_t)max_k;
    p.softmax_scale = (float)scale_or_default();
    p.causal = causal;
    p.deterministic = deterministic;
    elem_code(q, &p.dtype);
    return p;
  }

  const int32_t *offsets() const { return kv_off ? kv_off->const_data_ptr<int32_t>() : nullptr; }

  // [T, H, d] -> [T, H, 128] with zeros behind the d values of every head
  static Tensor pad(const Tensor &t) {
    const int64_t d = t.size(-1);
    if (d == kHeadDim) return t;
    if (d > kHeadDim || d % 8) fail("head_dim=" + std::to_string(d) + ": must be a multiple of 8 and at most " + std::to_string(kHeadDim));
    return at::constant_pad_nd(t, {0, kHeadDim - d});
  }
  Batch padded() const { return {pad(q), pad(k), pad(v), cu_q, cu_k, kv_off, max_q, max_k, scale_or_default(), causal}; }
};

// The caller's workspace, of at least `least` bytes, or one of `size`, or of `least` where the device has no memory left for that.
Tensor workspace_of(const OptTensor &given, int64_t least, int64_t size, c10::Device device, const char *what) {
  if (least < 0) check_rc(least, what);
  if (given) {
    if (given->scalar_type() != at::kByte || !given->is_cuda() || !given->is_contiguous() || given->numel() < least)
      fail("workspace must be a contiguous uint8 CUDA tensor of at least " + std::to_string(least) + " bytes");
    return *given;
  }
  auto empty = [&](int64_t n) { return at::empty({n > 16 ? n : 16}, at::TensorOptions().dtype(at::kByte).device(device)); };
  if (size > least) {
    try {
      return empty(size);
    } catch (const c10::OutOfMemoryError &) {
    }
  }
  return empty(least);
}

std::pair<Tensor, Tensor> varlen_fwd(const Batch &b, const OptTensor &workspace) {
  b.check();
  const int64_t d = b.q.size(2);
  if (d != kHeadDim) {
    auto [out, lse] = varlen_fwd(b.padded(), workspace);
    return {out.narrow(2, 0, d).contiguous(), lse};
  }
  const distca_ca_params p = b.params(false);
  const Tensor ws = workspace_of(workspace, distca_ca_fwd_workspace_bytes(&p), distca_ca_fwd_workspace_preferred_bytes(&p), b.q.device(), "ca_varlen_fwd");
  Tensor out = at::empty_like(b.q);
  Tensor lse = at::empty({b.q.size(1), b.q.size(0)}, b.q.options().dtype(at::kFloat));
  const OnDevice on(b.q.device());
  check_rc(distca_ca_fwd(b.q.data_ptr(), b.k.data_ptr(), b.v.data_ptr(), out.data_ptr(), lse.data_ptr<float>(),
                         b.cu_q.const_data_ptr<int32_t>(), b.cu_k.const_data_ptr<int32_t>(), b.offsets(), &p, ws.data_ptr(), ws.numel(), on.stream),
           "ca_varlen_fwd");
  return {std::move(out), std::move(lse)};
}

struct Grads {
  OptTensor dq, dk, dv;
};

std::array<Tensor, 3> varlen_bwd(const Batch &b, Tensor dout, Tensor out, Tensor lse, bool deterministic, const Grads &given,
                                 const OptTensor &workspace) {
  b.check();
  const struct { const char *name; const Tensor &t; } rows[] = {{"dout", dout}, {"out", out}};
  for (const auto &r : rows)
    if (r.t.sizes() != b.q.sizes() || r.t.scalar_type() != b.q.scalar_type() || !r.t.is_cuda())
      fail(std::string(r.name) + " must be a CUDA tensor with the shape and type of q");
  const int64_t d = b.q.size(2);
  if (d != kHeadDim) {
    auto grads = varlen_bwd(b.padded(), Batch::pad(dout), Batch::pad(out), lse, deterministic, {}, workspace);
    const OptTensor *to[] = {&given.dq, &given.dk, &given.dv};
    for (int i = 0; i < 3; ++i) {
      const Tensor g = grads[i].narrow(2, 0, d);
      if (*to[i]) {
        Tensor t = **to[i];
        t.copy_(g);
        grads[i] = t;
      } else {
        grads[i] = g.contiguous();
      }
    }
    return grads;
  }
  dout = dout.contiguous();
  out = out.contiguous();
  if (lse.dim() != 2 || lse.size(0) != b.q.size(1) || lse.size(1) != b.q.size(0) || lse.scalar_type() != at::kFloat)
    fail("softmax_lse must be fp32 of shape [Hq, Tq] = (" + std::to_string(b.q.size(1)) + ", " + std::to_string(b.q.size(0)) + ")");
  lse = lse.contiguous();
  const distca_ca_params p = b.params(deterministic);
  // (A call over shared K/V rows brings what distca_ca_bwd_workspace_bytes asks for: the same bits as the C ABI's other forms give with
  // it; the server's tick takes the preferred size.  A small batch, for which more is asked without the deterministic switch than
  // with it, is cut into pieces either way, and brings room for all of them.)
  const int64_t least = distca_ca_bwd_workspace_bytes(&p);
  bool whole = b.kv_off.has_value();
  if (whole && !deterministic) {
    const distca_ca_params smallest = b.params(true);
    whole = least == distca_ca_bwd_workspace_bytes(&smallest);
  }
  const Tensor ws = workspace_of(workspace, least, whole ? least : distca_ca_bwd_workspace_preferred_bytes(&p), b.q.device(), "ca_varlen_bwd");
  std::array<Tensor, 3> grads{given.dq ? *given.dq : at::empty_like(b.q), given.dk ? *given.dk : at::empty_like(b.k),
                              given.dv ? *given.dv : at::empty_like(b.v)};
  const struct { const char *name; const Tensor &of; } like[] = {{"dq", b.q}, {"dk", b.k}, {"dv", b.v}};
  for (int i = 0; i < 3; ++i)
    if (grads[i].sizes() != like[i].of.sizes() || grads[i].scalar_type() != b.q.scalar_type() || !grads[i].is_contiguous() || !grads[i].is_cuda())
      fail(std::string(like[i].name) + " must be a contiguous CUDA tensor with the shape and type of its input");
  const OnDevice on(b.q.device());
  check_rc(distca_ca_bwd(dout.data_ptr(), b.q.data_ptr(), b.k.data_ptr(), b.v.data_ptr(), out.data_ptr(), lse.data_ptr<float>(),
                         grads[0].data_ptr(), grads[1].data_ptr(), grads[2].data_ptr(), b.cu_q.const_data_ptr<int32_t>(),
                         b.cu_k.const_data_ptr<int32_t>(), b.offsets(), &p, ws.data_ptr(), ws.numel(), on.stream),
           "ca_varlen_bwd");
  return grads;
}

// Differentiable core attention; what is not a tensor travels beside the saved tensors.
struct CoreAttention : torch::autograd::Function<CoreAttention> {
  static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &cu_q,
                        const Tensor &cu_k, const OptTensor &kv_off, int64_t max_q, int64_t max_k, std::optional<double> scale, bool causal,
                        bool deterministic) {
    auto [out, lse] = varlen_fwd({q, k, v, cu_q, cu_k, kv_off, max_q, max_k, scale, causal}, std::nullopt);
    ctx->save_for_backward({q, k, v, out, lse, cu_q, cu_k});
    auto &data = ctx->saved_data;
    data["kv_off"] = kv_off;   // (beside the saved tensors: a caller may write the offsets of one layer into the buffer of the last)
    data["max_q"] = max_q;
    data["max_k"] = max_k;
    data["scale"] = scale;
    data["flags"] = (int64_t)causal | (int64_t)deterministic << 1;
    return out;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grad) {
    const auto s = ctx->get_saved_variables();
    auto &data = ctx->saved_data;
    const int64_t flags = data["flags"].toInt();
    const Batch b{s[0], s[1], s[2], s[5], s[6], data["kv_off"].toOptional<Tensor>(), data["max_q"].toInt(), data["max_k"].toInt(),
                  data["scale"].toOptional<double>(), (flags & 1) != 0};
    auto g = varlen_bwd(b, grad[0], s[3], s[4], (flags & 2) != 0, {}, std::nullopt);
    torch::autograd::variable_list res(11);
    for (int i = 0; i < 3; ++i) res[i] = std::move(g[i]);
    return res;
  }
};

// ---------------------------------------------------------------------------------------
// Arguments from Python, by position
// ---------------------------------------------------------------------------------------
const Tensor &tensor_arg(PyObject *o, const char *name) {
  if (!THPVariable_Check(o)) type_error(std::string(name) + " must be a tensor, not " + Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
OptTensor optional_arg(PyObject *o, const char *name) { return o == Py_None ? OptTensor() : OptTensor(tensor_arg(o, name)); }
int64_t int_arg(PyObject *o) {
  if (PyLong_Check(o)) {
    const int64_t n = PyLong_AsLongLong(o);
    if (n == -1 && PyErr_Occurred()) throw python_error();
    return n;
  }
  PyObject *as_int = PyNumber_Long(o);
  if (!as_int) throw python_error();
  const int64_t n = PyLong_AsLongLong(as_int);
  Py_DECREF(as_int);
  if (n == -1 && PyErr_Occurred()) throw python_error();
  return n;
}
std::optional<double> optional_float(PyObject *o) {
  if (o == Py_None) return std::nullopt;
  if (PyFloat_Check(o)) return PyFloat_AS_DOUBLE(o);
  PyObject *as_float = PyNumber_Float(o);   // (what float() takes, strings among them)
  if (!as_float) throw python_error();
  const double x = PyFloat_AS_DOUBLE(as_float);
  Py_DECREF(as_float);
  return x;
}
bool bool_arg(PyObject *o) {
  const int r = PyObject_IsTrue(o);
  if (r < 0) throw python_error();
  return r != 0;
}
void expect(Py_ssize_t given, Py_ssize_t takes, const char *name) {
  if (given != takes) type_error(std::string(name) + " takes " + std::to_string(takes) + " arguments, " + std::to_string(given) + " given");
}
// The interpreter's lock is not held while memory is allocated and kernels are launched (a full queue makes a launch wait).
struct Unlocked {
  PyThreadState *state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

Batch batch_args(PyObject *const *a) {   // q, k, v, cu_q, cu_k, max_q, max_k, scale, causal, kv_off
  return {tensor_arg(a[0], "q"), tensor_arg(a[1], "k"), tensor_arg(a[2], "v"), tensor_arg(a[3], "cu_seqlens_q"), tensor_arg(a[4], "cu_seqlens_k"),
          optional_arg(a[9], "kv_task_offsets"), int_arg(a[5]), int_arg(a[6]), optional_float(a[7]), bool_arg(a[8])};
}

PyObject *py_varlen_fwd(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 11, "varlen_fwd");
  const Batch b = batch_args(a);
  const OptTensor ws = optional_arg(a[10], "workspace");
  std::pair<Tensor, Tensor> r;
  {
    const Unlocked u;
    r = varlen_fwd(b, ws);
  }
  PyObject *t = PyTuple_New(2);
  if (!t) throw python_error();
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(std::move(r.first)));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(std::move(r.second)));
  return t;
  END_HANDLE_TH_ERRORS
}

PyObject *py_varlen_bwd(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 18, "varlen_bwd");
  const Batch b = batch_args(a);
  const Tensor dout = tensor_arg(a[10], "dout"), out = tensor_arg(a[11], "out"), lse = tensor_arg(a[12], "softmax_lse");
  const bool deterministic = bool_arg(a[13]);
  const Grads given{optional_arg(a[14], "dq"), optional_arg(a[15], "dk"), optional_arg(a[16], "dv")};
  const OptTensor ws = optional_arg(a[17], "workspace");
  std::array<Tensor, 3> g;
  {
    const Unlocked u;
    g = varlen_bwd(b, dout, out, lse, deterministic, given, ws);
  }
  PyObject *t = PyTuple_New(3);
  if (!t) throw python_error();
  for (int i = 0; i < 3; ++i) PyTuple_SET_ITEM(t, i, THPVariable_Wrap(std::move(g[i])));
  return t;
  END_HANDLE_TH_ERRORS
}

PyObject *py_core_attention(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 11, "core_attention");
  const Batch b = batch_args(a);
  const bool deterministic = bool_arg(a[10]);
  Tensor out;
  {
    const Unlocked u;
    out = CoreAttention::apply(b.q, b.k, b.v, b.cu_q, b.cu_k, b.kv_off, b.max_q, b.max_k, b.scale, b.causal, deterministic);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------------------------------
// Jobs of one exchange launch.  A job from Python is a tuple (kind, parts, offset, tokens, mask, token_bytes, num_copies, copy_start),
// None for what it has not; the tuple keeps its tensors alive until the launch.
// ---------------------------------------------------------------------------------------
void check_tensor(const Tensor &t, int64_t ndim, const char *name) {
  if (t.dim() != ndim) fail(std::string("tensor ") + name + " must have " + std::to_string(ndim) + " dimensions");
  if (!t.is_cuda()) fail(std::string("tensor ") + name + " must be on CUDA");
  if (!t.is_contiguous()) fail(std::string("tensor ") + name + " must be contiguous");
}
template <typename T>
const T *data_of(const Tensor &t, const char *name) {
  if (t.scalar_type() != c10::CppTypeToScalarType<T>::value)
    fail(std::string("expected scalar type ") + c10::toString(c10::CppTypeToScalarType<T>::value) + " but found " + c10::toString(t.scalar_type()) +
         " for " + name);
  return t.const_data_ptr<T>();
}

// The parts a job's token is made of.
void set_parts(distca_exchange_job &j, const Tensor *const *parts, int64_t n) {
  const bool plain = j.kind == DISTCA_JOB_PLAIN, sums = j.kind == DISTCA_JOB_COPY_SUM || j.kind == DISTCA_JOB_REPLICA_SUM;
  int64_t row = 0;
  for (int64_t i = 0; i < n; ++i) {
    const Tensor &t = *parts[i];
    if (!plain) check_tensor(t, 2, "tensor");
    if (t.dim() != 2) fail("tensor must have 2 dimensions");
    if (!t.is_cuda()) fail("tensor must be on CUDA");
    if (t.size(1) > 1 && t.stride(1) != 1) fail("tensor must have contiguous rows");
    const int64_t esz = (int64_t)t.element_size(), bytes = t.size(1) * esz;
    if (i == 0) j.num_tokens = t.size(0);
    else if (t.size(0) != j.num_tokens) fail("token parts disagree on the token count");
    j.part[i] = {t.data_ptr(), t.size(0) > 1 ? t.stride(0) * esz : bytes, bytes};
    row += bytes;
    switch (t.scalar_type()) {
      case at::kFloat: j.dtype = DISTCA_DTYPE_F32; break;
      case at::kHalf: j.dtype = DISTCA_DTYPE_F16; break;
      case at::kBFloat16: j.dtype = DISTCA_DTYPE_BF16; break;
      default:
        if (sums) fail("Only fp32, fp16 and bf16 inputs are supported");
    }
  }
  j.num_parts = n;
  j.token_bytes = row;
}
// Its shards: places, lengths, and which are sent (mask, may be null) or which replicas there are.
void set_shards(distca_exchange_job &j, const Tensor &offset, const Tensor &tokens, const Tensor *mask) {
  if (j.kind == DISTCA_JOB_REPLICAS || j.kind == DISTCA_JOB_REPLICA_SUM) {
    check_tensor(offset, 2, "seq_nvshmem_offset");
    check_tensor(tokens, 1, "seq_tokens");
    check_tensor(*mask, 2, "do_shard");
    j.max_cp = offset.size(0);
    j.num_seq = offset.size(1);
    if (tokens.size(0) != j.num_seq) fail("seq_tokens must be of dimension (num_sequence)");
    if (mask->size(0) != j.num_seq || mask->size(1) != j.max_cp) fail("do_shard must be of dimension (num_sequence, cp_degree)");
    j.mask = data_of<int8_t>(*mask, "do_shard");
  } else {
    check_tensor(offset, 1, "seq_nvshmem_offset");
    check_tensor(tokens, tokens.dim(), "seq_tokens");   // (of any shape that begins with a length per shard)
    j.max_cp = 1;
    j.num_seq = offset.size(0);
    if (tokens.numel() < j.num_seq) fail("seq_tokens must be of shape (num_sequence,)");
    if (mask) {
      check_tensor(*mask, 1, "copy_seq_mask");
      j.mask = data_of<int8_t>(*mask, "copy_seq_mask");
      if (mask->size(0) != j.num_seq) fail("copy_seq_mask must be of shape (num_sequence,)");
    }
  }
  j.seq_offset = data_of<int64_t>(offset, "seq_nvshmem_offset");
  j.seq_tokens = data_of<int64_t>(tokens, "seq_tokens");
}
distca_exchange_job make_job(int64_t kind, std::initializer_list<const Tensor *> parts, const Tensor &offset, const Tensor &tokens, const Tensor *mask = nullptr) {
  distca_exchange_job j{};
  j.kind = kind;
  set_parts(j, parts.begin(), (int64_t)parts.size());
  set_shards(j, offset, tokens, mask);
  return j;
}

// Fills in the job and returns the device of its first tensor.
c10::Device read_job(PyObject *o, distca_exchange_job &j) {
  if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != 8) type_error("a job is a tuple of eight");
  PyObject *const *f = &PyTuple_GET_ITEM(o, 0);
  j = distca_exchange_job{};
  j.kind = int_arg(f[0]);
  const bool replicas = j.kind == DISTCA_JOB_REPLICAS || j.kind == DISTCA_JOB_REPLICA_SUM;
  const Tensor &offset = tensor_arg(f[2], "seq_nvshmem_offset"), &tokens = tensor_arg(f[3], "seq_tokens");

  PyObject *list = f[1];
  if (!PyList_Check(list) && !PyTuple_Check(list)) type_error(std::string("the parts of a token are a list or a tuple of tensors, not ") + Py_TYPE(list)->tp_name);
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(list);
  if (n < 1 || n > DISTCA_TOKEN_MAX_PARTS) fail("a token has one to " + std::to_string(DISTCA_TOKEN_MAX_PARTS) + " parts");
  const Tensor *parts[DISTCA_TOKEN_MAX_PARTS];
  for (Py_ssize_t i = 0; i < n; ++i) parts[i] = &tensor_arg(PySequence_Fast_GET_ITEM(list, i), "tensor");
  set_parts(j, parts, n);
  if (f[5] != Py_None) j.token_bytes = int_arg(f[5]);
  const Tensor *mask = replicas || f[4] != Py_None ? &tensor_arg(f[4], replicas ? "do_shard" : "copy_seq_mask") : nullptr;
  set_shards(j, offset, tokens, mask);
  if (j.kind == DISTCA_JOB_COPY_SUM) {
    const Tensor &num_copies = tensor_arg(f[6], "num_copies"), &start = tensor_arg(f[7], "copy_start_id");
    check_tensor(num_copies, 1, "num_copies");
    check_tensor(start, 2, "copy_start_id");
    if (num_copies.size(0) != j.num_seq || tokens.dim() != 1 || tokens.size(0) != j.num_seq) fail("seq_lens must be of shape (num_sequence,)");
    if (start.size(0) != j.num_seq) fail("copy_start_id must be of shape (num_sequence, max_num_copies)");
    j.num_copies = data_of<int32_t>(num_copies, "num_copies");
    j.copy_start = data_of<int64_t>(start, "copy_start_id");
    j.max_copies = start.size(1);
  }
  return parts[0]->device();
}

// The launch goes to the device, and its stream, that made the tensors: the buffer may be another device's memory
void run_exchange(const distca_exchange_job *jobs, int32_t n, const Tensor &buffer, bool to_buffer, c10::Device device) {
  if (!buffer.is_cuda()) fail("tensor buffer must be on CUDA");
  const Unlocked u;
  const OnDevice on(device);
  check_rc(distca_exchange(jobs, n, buffer.data_ptr(), to_buffer, on.stream), "exchange");
}

PyObject *py_exchange(PyObject *, PyObject *const *a, Py_ssize_t n) {   // jobs, buffer, to_buffer
  HANDLE_TH_ERRORS
  expect(n, 3, "exchange");
  const Tensor &buffer = tensor_arg(a[1], "buffer");
  const bool to_buffer = bool_arg(a[2]);
  if (!PyList_Check(a[0]) && !PyTuple_Check(a[0])) type_error("jobs must be a list");
  const Py_ssize_t num = PySequence_Fast_GET_SIZE(a[0]);
  if (num > DISTCA_EXCHANGE_MAX_JOBS) fail("at most " + std::to_string(DISTCA_EXCHANGE_MAX_JOBS) + " jobs per launch");
  distca_exchange_job jobs[DISTCA_EXCHANGE_MAX_JOBS];
  std::optional<c10::Device> device;
  for (Py_ssize_t i = 0; i < num; ++i) {
    const c10::Device d = read_job(PySequence_Fast_GET_ITEM(a[0], i), jobs[i]);
    if (!device) device = d;
  }
  run_exchange(jobs, (int32_t)num, buffer, to_buffer, device ? *device : buffer.device());
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// The two halves of the linear side's forward in one call each: with the jobs made and the results allocated in Python the host took longer
// over them than the device (1021 tokens, 8/2 heads, a pass among others: 14.7 us, by these two 11.8; the kernels take 8.5).
// q shards as they are, every k / v shard once per destination: (q, k, v, do_shard, q_tokens, k_tokens, q_offset, k_offset, v_offset, buffer)
PyObject *py_pack_qkv(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 10, "pack_qkv");
  const Tensor q = tensor_arg(a[0], "tensor").contiguous(), k = tensor_arg(a[1], "tensor").contiguous(), v = tensor_arg(a[2], "tensor").contiguous();
  const Tensor &mask = tensor_arg(a[3], "do_shard"), &q_tokens = tensor_arg(a[4], "seq_tokens"), &k_tokens = tensor_arg(a[5], "seq_tokens");
  const char *off = "seq_nvshmem_offset";
  const distca_exchange_job jobs[3] = {make_job(DISTCA_JOB_PLAIN, {&q}, tensor_arg(a[6], off), q_tokens),
                                       make_job(DISTCA_JOB_REPLICAS, {&k}, tensor_arg(a[7], off), k_tokens, &mask),
                                       make_job(DISTCA_JOB_REPLICAS, {&v}, tensor_arg(a[8], off), k_tokens, &mask)};
  run_exchange(jobs, 3, tensor_arg(a[9], "buffer"), true, q.device());
  PyObject *t = PyTuple_New(3);
  if (!t) throw python_error();
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(q));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(k));
  PyTuple_SET_ITEM(t, 2, THPVariable_Wrap(v));
  return t;
  END_HANDLE_TH_ERRORS
}

// The [out | lse | pad] tokens of a reply taken apart: (buffer, tensor on the device of the results, dtype of out, tokens, elements of out,
// bytes of lse, bytes of a token, offset, lengths) -> out [tokens, 1, elements], lse [tokens, bytes]
PyObject *py_unpack_reply(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 9, "unpack_reply");
  if (!THPDtype_Check(a[2])) type_error(std::string("dtype must be a torch.dtype, not ") + Py_TYPE(a[2])->tp_name);
  const auto dtype = reinterpret_cast<THPDtype *>(a[2])->scalar_type;
  const int64_t rows = int_arg(a[3]), elements = int_arg(a[4]), lse_bytes = int_arg(a[5]);
  const auto on_device = at::TensorOptions().device(tensor_arg(a[1], "q").device());
  const Tensor out = at::empty({rows, 1, elements}, on_device.dtype(dtype)), lse = at::empty({rows, lse_bytes}, on_device.dtype(at::kByte));
  const Tensor out_rows = out.view({rows, elements});
  distca_exchange_job j = make_job(DISTCA_JOB_PLAIN, {&out_rows, &lse}, tensor_arg(a[7], "seq_nvshmem_offset"), tensor_arg(a[8], "seq_tokens"));
  j.token_bytes = int_arg(a[6]);
  run_exchange(&j, 1, tensor_arg(a[0], "buffer"), false, out.device());
  PyObject *t = PyTuple_New(2);
  if (!t) throw python_error();
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(out));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(lse));
  return t;
  END_HANDLE_TH_ERRORS
}

// (the current device, the current stream of device `index`, or of the current one for -1, as a raw handle)
PyObject *py_current_stream(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 1, "current_stream");
  const int here = c10::hip::current_device();
  const int64_t index = int_arg(a[0]);
  void *const stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)(index < 0 ? here : index)).stream();
  return Py_BuildValue("iK", here, (unsigned long long)reinterpret_cast<uintptr_t>(stream));
  END_HANDLE_TH_ERRORS
}

template <typename F>
constexpr PyCFunction fast(F *f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }

PyMethodDef methods[] = {
    {"varlen_fwd", fast(py_varlen_fwd), METH_FASTCALL, nullptr},
    {"varlen_bwd", fast(py_varlen_bwd), METH_FASTCALL, nullptr},
    {"core_attention", fast(py_core_attention), METH_FASTCALL, nullptr},
    {"exchange", fast(py_exchange), METH_FASTCALL, nullptr},
    {"pack_qkv", fast(py_pack_qkv), METH_FASTCALL, nullptr},
    {"unpack_reply", fast(py_unpack_reply), METH_FASTCALL, nullptr},
    {"current_stream", fast(py_current_stream), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Native host side of the attention and exchange calls.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
