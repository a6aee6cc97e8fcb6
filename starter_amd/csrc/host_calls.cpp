// The kernel wrappers' ordinary calls as one native call each.
//
// A decode or prompt call of a few microseconds on the GPU spent ~10 us on the
// host in Python: operand checks attribute by attribute, the output
// allocation, the stream lookup and a ctypes call of 8-23 converted
// arguments.  Each function here does the same for the ordinary case - plain
// contiguous tensors of one GPU - in about half of that (rms_norm [8, 2560] 10.3 ->
// 5.8 us a call, its launch included), and returns NotImplemented, having
// done nothing, for every other one: the Python wrapper then runs its own
// checks and raises or launches as before.  Nothing is decided here that the
// wrapper decides differently, so what is refused, and how, stays there.
//
// "Plain" excludes tensor subclasses and functorch wrappers, and any call
// under a torch function or dispatch mode (tracing, fake tensors): those take
// the wrapper's path, whose torch calls such modes see.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/core/grad_mode.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

#include "qwen_fused.h"

namespace {

constexpr int64_t kHead = 128;
constexpr int64_t kMaxBlock = 8192;  // widest row of the norms

// Arguments of one call: reading one that does not qualify clears `ok`, and
// every later step is skipped.
struct Call {
  PyObject* const* args;
  Py_ssize_t count;
  bool ok;
  c10::DeviceIndex device = -1;

  Call(PyObject* const* a, Py_ssize_t n, Py_ssize_t expected)
      : args(a), count(n),
        ok(n == expected && !at::impl::torch_function_mode_enabled() &&
           !c10::impl::dispatch_mode_enabled()) {}

  bool need(bool condition) { return ok = ok && condition; }

  // Contiguous plain GPU tensor of `type`, on the device of the call's first one.
  const at::Tensor* tensor(int i, at::ScalarType type, int64_t dims = -1) {
    if (!ok) return nullptr;
    if (!THPVariable_CheckExact(args[i])) return ok = false, nullptr;
    const at::Tensor& t = THPVariable_Unpack(args[i]);
    if (!t.defined() || !t.is_cuda() || at::isTensorSubclassLike(t) || t.scalar_type() != type ||
        t.layout() != at::kStrided || !t.is_contiguous() || (dims >= 0 && t.dim() != dims))
      return ok = false, nullptr;
    if (device < 0) device = t.get_device();
    return need(t.get_device() == device) ? &t : nullptr;
  }
  const at::Tensor* bf16(int i, int64_t dims = -1) { return tensor(i, at::kBFloat16, dims); }
  // A bf16 vector of n elements.
  const at::Tensor* vec(int i, int64_t n) {
    const at::Tensor* t = bf16(i, 1);
    return ok && need(t->size(0) == n) ? t : nullptr;
  }
  // Split-K partials [S, ...] (f32, 3-D): S; or a bf16 matrix: 0.  Both of the given trailing shape.
  const at::Tensor* branch(int i, int64_t rows, int64_t cols, int32_t* splits) {
    if (!ok || !need(THPVariable_CheckExact(args[i]))) return nullptr;
    const at::Tensor& probe = THPVariable_Unpack(args[i]);
    const bool parts = probe.scalar_type() == at::kFloat;
    const at::Tensor* t = parts ? tensor(i, at::kFloat, 3) : bf16(i, 2);
    if (!ok) return nullptr;
    *splits = parts ? (int32_t)t->size(0) : 0;
    return need((!parts || *splits >= 1) && t->size(parts) == rows && t->size(parts + 1) == cols)
               ? t : nullptr;
  }
  double number(int i) {
    if (!ok || !need(PyFloat_CheckExact(args[i]) || PyLong_CheckExact(args[i]))) return 0;
    const double v = PyFloat_AsDouble(args[i]);
    if (v == -1.0 && PyErr_Occurred()) return PyErr_Clear(), ok = false, 0;
    return v;
  }
  int64_t integer(int i) {
    if (!ok || !need(PyLong_CheckExact(args[i]))) return 0;
    const int64_t v = PyLong_AsLongLong(args[i]);
    if (v == -1 && PyErr_Occurred()) return PyErr_Clear(), ok = false, 0;
    return v;
  }
  void* stream() const { return c10::hip::getCurrentHIPStream(device).stream(); }
  at::Tensor empty(at::IntArrayRef shape, at::ScalarType type) const {
    return at::empty(shape, at::TensorOptions().dtype(type).device(at::kCUDA, device));
  }
};

bool aligned(const at::Tensor* t) { return (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15u) == 0; }
void* ptr(const at::Tensor& t) { return t.data_ptr(); }
void* ptr(const at::Tensor* t) { return t->data_ptr(); }

PyObject* not_taken() {
  Py_INCREF(Py_NotImplemented);
  return Py_NotImplemented;
}

// The error the wrappers' own calls raise for a status.
bool failed(const char* name, int status) {
  if (status == 0) return false;
  PyErr_Format(PyExc_RuntimeError, "%s failed: %s (status %d)", name, qf_error_string(status), status);
  return true;
}

// Allocation and launch run without the interpreter's lock, as torch's and
// ctypes' calls do.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

PyObject* rms_norm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c(args, n, 3);
  const at::Tensor* x = c.bf16(0);
  if (!c.ok || !c.need(x->dim() >= 1 && x->numel() > 0)) return not_taken();
  const int64_t cols = x->size(-1), rows = x->numel() / cols;
  const at::Tensor* weight = c.vec(1, cols);
  const float eps = (float)c.number(2);
  if (!c.need(cols <= kMaxBlock)) return not_taken();
  at::Tensor out;
  int status;
  {
    Unlocked unlocked;
    out = c.empty(x->sizes(), at::kBFloat16);
    status = qf_rms_norm(ptr(x), rows, cols, rows, 0, rows > 1 ? cols : 0, ptr(weight), eps, ptr(out), c.stream());
  }
  return failed("qf_rms_norm", status) ? nullptr : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyObject* add_rms_norm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c(args, n, 4);
  const at::Tensor* residual = c.bf16(0, 2);
  if (!c.ok) return not_taken();
  const int64_t rows = residual->size(0), cols = residual->size(1);
  int32_t splits = 0;
  const at::Tensor* branch = c.branch(1, rows, cols, &splits);
  const at::Tensor* weight = c.vec(2, cols);
  const float eps = (float)c.number(3);
  if (!c.need(rows > 0 && cols > 0 && cols <= kMaxBlock)) return not_taken();
  at::Tensor total, normed;
  int status;
  {
    Unlocked unlocked;
    total = at::empty_like(*residual);
    normed = at::empty_like(*residual);
    status = qf_add_rms_norm(ptr(residual), ptr(branch), splits, ptr(weight), rows, cols, eps, ptr(total), ptr(normed),
                             c.stream());
  }
  if (failed("qf_add_rms_norm", status)) return nullptr;
  PyObject* pair = PyTuple_New(2);
  if (!pair) return nullptr;
  PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(total)));
  PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(normed)));
  return pair;
  END_HANDLE_TH_ERRORS
}

PyObject* silu_mul(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c(args, n, 1);
  const at::Tensor* x = c.bf16(0, 2);
  if (!c.ok || !c.need(x->numel() > 0 && x->size(1) % 2 == 0)) return not_taken();
  const int64_t rows = x->size(0), cols = x->size(1) / 2;
  at::Tensor out;
  int status;
  {
    Unlocked unlocked;
    out = c.empty({rows, cols}, at::kBFloat16);
    status = qf_silu_mul(ptr(x), rows, cols, ptr(out), c.stream());
  }
  return failed("qf_silu_mul", status) ? nullptr : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyObject* embedding(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c(args, n, 2);
  const at::Tensor* ids = c.tensor(0, at::kLong);
  const at::Tensor* weight = c.bf16(1, 2);
  if (!c.ok || !c.need(ids->numel() > 0 && weight->size(1) > 0)) return not_taken();
  c10::SmallVector<int64_t, 5> shape(ids->sizes().begin(), ids->sizes().end());
  shape.push_back(weight->size(1));
  at::Tensor out;
  int status;
  {
    Unlocked unlocked;
    out = c.empty(shape, at::kBFloat16);
    status = qf_embedding(ids->const_data_ptr<int64_t>(), ids->numel(), ptr(weight), weight->size(0), weight->size(1),
                          ptr(out), c.stream());
  }
  return failed("qf_embedding", status) ? nullptr : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// x [M, K] and W [N, K] as the decode projections take them (N a multiple of `columns`).
bool projection(Call& c, const at::Tensor*& x, const at::Tensor*& w, int64_t columns) {
  x = c.bf16(0, 2);
  w = c.bf16(1, 2);
  return c.ok && c.need(x->size(1) == w->size(1) && x->size(0) >= 1 && x->size(0) <= 64 && x->size(1) > 0 &&
                        x->size(1) % 64 == 0 && w->size(0) > 0 && w->size(0) % columns == 0 && aligned(x) && aligned(w));
}

PyObject* linear_partials(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c(args, n, 2);
  const at::Tensor *x, *w;
  if (!projection(c, x, w, 32)) return not_taken();
  const int64_t m = x->size(0), k = x->size(1), cols = w->size(0);
  const int splits = qf_linear_splits(m, k, cols);
  if (splits < 1) return not_taken();
  at::Tensor out;
  int status;
  {
    Unlocked unlocked;
    out = c.empty({splits, m, cols}, at::kFloat);
    status = qf_linear_partials(ptr(x), m, k, ptr(w), cols, splits, ptr(out), c.stream());
  }
  return failed("qf_linear_partials", status) ? nullptr : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyObject* linear_silu_mul(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c(args, n, 2);
  const at::Tensor *x, *w;
  if (!projection(c, x, w, 64)) return not_taken();
  const int64_t m = x->size(0), k = x->size(1), cols = w->size(0) / 2;
  at::Tensor out;
  int status;
  {
    Unlocked unlocked;
    out = c.empty({m, cols}, at::kBFloat16);
    status = qf_linear_silu_mul(ptr(x), m, k, ptr(w), cols, ptr(out), c.stream());
  }
  return failed("qf_linear_silu_mul", status) ? nullptr : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// (x, weight, logits: bool) -> tokens, or (tokens, logits).
PyObject* lm_head_argmax(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c(args, n, 3);
  const at::Tensor *x, *w;
  if (!projection(c, x, w, 16) || !c.need(PyBool_Check(args[2]))) return not_taken();
  const bool keep = args[2] == Py_True;
  const int64_t m = x->size(0), k = x->size(1), vocab = w->size(0);
  at::Tensor tokens, logits;
  int status;
  {
    Unlocked unlocked;
    const at::Tensor candidates = c.empty({m, qf_lm_head_blocks(vocab), 2}, at::kInt);
    tokens = c.empty({m}, at::kLong);
    if (keep) logits = c.empty({m, vocab}, at::kBFloat16);
    status = qf_lm_head_argmax(ptr(x), m, k, ptr(w), vocab, ptr(candidates), tokens.mutable_data_ptr<int64_t>(),
                               keep ? ptr(logits) : nullptr, c.stream());
  }
  if (failed("qf_lm_head_argmax", status)) return nullptr;
  if (!keep) return THPVariable_Wrap(std::move(tokens));
  PyObject* pair = PyTuple_New(2);
  if (!pair) return nullptr;
  PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(tokens)));
  PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(logits)));
  return pair;
  END_HANDLE_TH_ERRORS
}

// (qkv, qw, kw, qeps, keps, cos, sin, keys, values, length)
PyObject* prefill_qkv(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c(args, n, 10);
  const at::Tensor* qkv = c.bf16(0, 2);
  const at::Tensor *qw = c.vec(1, kHead), *kw = c.vec(2, kHead);
  const float qeps = (float)c.number(3), keps = (float)c.number(4);
  const at::Tensor *cos = c.bf16(5, 2), *sin = c.bf16(6, 2), *keys = c.bf16(7, 4), *values = c.bf16(8, 4);
  const int64_t length = c.integer(9);
  if (!c.ok) return not_taken();
  const int64_t batch = keys->size(0), nk = keys->size(1), capacity = keys->size(2);
  const int64_t nq = qkv->size(1) / kHead - 2 * nk;
  if (!c.need(values->sizes() == keys->sizes() && batch >= 1 && nk >= 1 && keys->size(3) == kHead && length >= 1 &&
              length <= capacity && qkv->size(0) == batch * length && nq >= 1 && nq % nk == 0 &&
              qkv->size(1) == (nq + 2 * nk) * kHead && cos->size(0) == capacity && cos->size(1) == kHead &&
              sin->sizes() == cos->sizes()))
    return not_taken();
  at::Tensor q;
  int status;
  {
    Unlocked unlocked;
    q = c.empty({batch, length, nq, kHead}, at::kBFloat16);
    status = qf_prefill_qkv(ptr(qkv), batch, length, (int32_t)nq, (int32_t)nk, ptr(qw), ptr(kw), qeps, keps, ptr(cos),
                            ptr(sin), capacity, ptr(q), ptr(keys), ptr(values), c.stream());
  }
  return failed("qf_prefill_qkv", status) ? nullptr : THPVariable_Wrap(std::move(q));
  END_HANDLE_TH_ERRORS
}

// (q, keys, values, length, scale)
PyObject* prefill_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c(args, n, 5);
  const at::Tensor *q = c.bf16(0, 4), *keys = c.bf16(1, 4), *values = c.bf16(2, 4);
  const int64_t length = c.integer(3);
  const double scale = c.number(4);
  if (!c.ok) return not_taken();
  const int64_t batch = keys->size(0), nk = keys->size(1), capacity = keys->size(2), nq = q->size(2);
  if (!c.need(values->sizes() == keys->sizes() && keys->size(3) == kHead && q->size(3) == kHead && nk >= 1 &&
              q->size(0) == batch && q->size(1) == length && batch >= 1 && length >= 1 && length <= capacity &&
              nq >= 1 && nq % nk == 0 && std::isfinite(scale)))
    return not_taken();
  const int64_t groups = nq / nk;
  if (groups != 1 && groups != 2 && groups != 4 && groups != 8) return not_taken();
  at::Tensor out;
  int status;
  {
    Unlocked unlocked;
    out = at::empty_like(*q);
    status = qf_prefill_attention(ptr(q), ptr(keys), ptr(values), batch, length, (int32_t)nq, (int32_t)nk, capacity,
                                  (float)scale, ptr(out), c.stream());
  }
  return failed("qf_prefill_attention", status) ? nullptr : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// (qkv, qw, kw, qeps, keps, cos, sin, position, keys, values): the operands
// qkv_norm_rope_cache and the fused decode attention share.
struct DecodeQkv {
  const at::Tensor *qkv, *qw, *kw, *cos, *sin, *position, *keys, *values;
  float qeps, keps;
  int32_t splits = 0;
  int64_t batch, nq, nk, capacity;

  bool read(Call& c) {
    keys = c.bf16(8, 4);
    values = c.bf16(9, 4);
    qw = c.vec(1, kHead);
    kw = c.vec(2, kHead);
    qeps = (float)c.number(3);
    keps = (float)c.number(4);
    cos = c.bf16(5, 2);
    sin = c.bf16(6, 2);
    position = c.tensor(7, at::kLong, 1);
    if (!c.ok || !c.need(THPVariable_CheckExact(c.args[0]))) return false;
    batch = keys->size(0);
    nk = keys->size(1);
    capacity = keys->size(2);
    const at::Tensor& packed = THPVariable_Unpack(c.args[0]);
    if (!c.need(packed.dim() >= 2)) return false;
    const int64_t width = packed.size(-1);
    nq = width / kHead - 2 * nk;
    qkv = c.branch(0, batch, width, &splits);
    return c.need(batch >= 1 && nk >= 1 && capacity >= 1 && keys->size(3) == kHead &&
                  values->sizes() == keys->sizes() && nq >= 1 && width == (nq + 2 * nk) * kHead &&
                  cos->size(0) == capacity && cos->size(1) == kHead && sin->sizes() == cos->sizes() &&
                  position->size(0) == 1);
  }
};

PyObject* qkv_norm_rope_cache(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c(args, n, 10);
  DecodeQkv d;
  if (!c.ok || !d.read(c)) return not_taken();
  at::Tensor q;
  int status;
  {
    Unlocked unlocked;
    q = c.empty({d.batch, d.nq, 1, kHead}, at::kBFloat16);
    status = qf_qkv_norm_rope_cache(ptr(d.qkv), d.splits, d.batch, (int32_t)d.nq, (int32_t)d.nk, ptr(d.qw), ptr(d.kw),
                                    d.qeps, d.keps, ptr(d.cos), ptr(d.sin), d.position->const_data_ptr<int64_t>(),
                                    d.capacity, ptr(q), ptr(d.keys), ptr(d.values), c.stream());
  }
  return failed("qf_qkv_norm_rope_cache", status) ? nullptr : THPVariable_Wrap(std::move(q));
  END_HANDLE_TH_ERRORS
}

// The operands above, then (used, scale, partials, stats, batch, hq, hk,
// capacity, splits, span) of a SmallQueryAttention, then whether to merge.
PyObject* attention_qkv(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c(args, n, 21);
  DecodeQkv d;
  if (!c.ok || at::GradMode::is_enabled() || !d.read(c)) return not_taken();
  const at::Tensor* used = c.tensor(10, at::kInt, 1);
  const double scale = c.number(11);
  const at::Tensor *partials = c.tensor(12, at::kFloat), *stats = c.tensor(13, at::kFloat);
  const int64_t batch = c.integer(14), hq = c.integer(15), hk = c.integer(16), capacity = c.integer(17);
  const int64_t splits = c.integer(18), span = c.integer(19);
  if (!c.ok || !c.need(batch == d.batch && hq == d.nq && hk == d.nk && capacity == d.capacity && std::isfinite(scale) &&
                       used->size(0) == batch * hk && PyBool_Check(args[20])))
    return not_taken();
  const bool merge = args[20] == Py_True;
  at::Tensor out;
  int status;
  {
    Unlocked unlocked;
    if (merge) out = c.empty({batch, 1, hq, kHead}, at::kBFloat16);
    status = qf_decode_attention_qkv(
        ptr(d.qkv), d.splits, ptr(d.qw), ptr(d.kw), d.qeps, d.keps, ptr(d.cos), ptr(d.sin),
        d.position->const_data_ptr<int64_t>(), ptr(d.keys), ptr(d.values), used->const_data_ptr<int32_t>(), batch,
        (int32_t)hq, (int32_t)hk, capacity, (float)scale, (int32_t)splits, span, partials->mutable_data_ptr<float>(),
        stats->mutable_data_ptr<float>(), merge ? ptr(out) : nullptr, c.stream());
  }
  if (failed("qf_decode_attention_qkv", status)) return nullptr;
  if (merge) return THPVariable_Wrap(std::move(out));
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

#define QF_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    QF_METHOD(rms_norm),        QF_METHOD(add_rms_norm),      QF_METHOD(silu_mul),
    QF_METHOD(embedding),       QF_METHOD(linear_partials),   QF_METHOD(linear_silu_mul),
    QF_METHOD(lm_head_argmax),  QF_METHOD(prefill_qkv),       QF_METHOD(prefill_attention),
    QF_METHOD(attention_qkv),   QF_METHOD(qkv_norm_rope_cache), {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_calls", "Native forms of the kernel wrappers' ordinary calls.",
                      -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_calls() {
  // Everything above reads torch's C++ objects as the headers of one torch
  // build lay them out, so the import fails under any other (the file's name
  // carries the interpreter's ABI); the wrappers then go their own way.
  PyObject* torch = PyImport_ImportModule("torch.version");
  PyObject* version = torch ? PyObject_GetAttrString(torch, "__version__") : nullptr;
  PyObject* revision = version ? PyObject_GetAttrString(torch, "git_version") : nullptr;
  PyObject* running = revision ? PyUnicode_FromFormat("%S %S", version, revision) : nullptr;
  PyObject* made = nullptr;
  if (running && PyUnicode_CompareWithASCIIString(running, QF_TORCH_BUILD) == 0) {
    made = PyModule_Create(&module);
  } else if (running) {
    PyErr_Format(PyExc_ImportError, "built for torch %s, this is %U", QF_TORCH_BUILD, running);
  } else {
    PyErr_Clear();
    PyErr_Format(PyExc_ImportError, "built for torch %s, this one names no version", QF_TORCH_BUILD);
  }
  Py_XDECREF(running);
  Py_XDECREF(revision);
  Py_XDECREF(version);
  Py_XDECREF(torch);
  return made;
}
