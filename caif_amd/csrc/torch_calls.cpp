// Native side of caif_amd/torch_ops.py: the per-call work around an entry point of the C ABI (argument checks, result and
// workspace allocation, current stream) for torch tensors.  In Python that work took 8.5 us of a call whose launch costs
// the host 3 to 4 us: a one-row linear of 1408 x 2048 (2.9 MB of weight) took 12.1 us a call, bound by the host; from here
// it takes 6.5 (host 5.1).
//
// The entry points are the ones the ctypes layer has loaded (caif_amd/capi.py hands their addresses to bind()), so there
// is one copy of libcaifx.so in the process and no state here besides those addresses.  A non-zero status is returned as a
// Python int; the caller turns it into the exception.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <stdexcept>

#include "caifx.h"

namespace {

// ------------------------------------------------------------------ entry points
#define ENTRIES(X)                                                                                                      \
  X(caifx_qlinear_forward) X(caifx_qlinear_forward_add) X(caifx_qlinear_backward_input)                                  \
  X(caifx_qlinear_backward_input_add) X(caifx_qlinear_workspace_bytes) X(caifx_qlinear_grouped_forward)                  \
  X(caifx_qlinear_grouped_backward_input) X(caifx_qlinear_grouped_backward_input_add)                                    \
  X(caifx_qlinear_grouped_workspace_bytes) X(caifx_qlinear_grouped_fresh) X(caifx_silu) X(caifx_silu_backward) X(caifx_multiply) X(caifx_add)           \
  X(caifx_silu_multiply) X(caifx_swiglu_backward) X(caifx_moe_dispatch_map_workspace_bytes)                              \
  X(caifx_moe_build_dispatch_map) X(caifx_moe_dispatch) X(caifx_moe_combine) X(caifx_moe_combine_backward_grad_expert)   \
  X(caifx_moe_combine_backward_grad_weights) X(caifx_moe_dispatch_backward) X(caifx_moe_dispatch_fresh)                  \
  X(caifx_moe_combine_backward_grad_expert_fresh) X(caifx_quantize_int8_per_channel)           \
  X(caifx_quantize_int8_per_tensor) X(caifx_quantize_to_int4)

struct Api {
#define X(name) decltype(&::name) name = nullptr;
  ENTRIES(X)
#undef X
} api;

PyObject *bind(PyObject *, PyObject *table)
{
  // every address is looked up before any is taken
  Api fresh;
#define X(name)                                                                                   \
  {                                                                                               \
    PyObject *v = PyDict_GetItemString(table, #name);                                             \
    const unsigned long long p = v ? PyLong_AsUnsignedLongLong(v) : 0;                            \
    if (p == 0 || PyErr_Occurred()) {                                                             \
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "missing entry point " #name);   \
      return nullptr;                                                                             \
    }                                                                                             \
    fresh.name = reinterpret_cast<decltype(&::name)>(p);                                          \
  }
  ENTRIES(X)
#undef X
  api = fresh;
  Py_RETURN_NONE;
}

// ------------------------------------------------------------------ arguments
struct Error {
  PyObject *type;
  const char *what;
};

const at::Tensor &tensor(PyObject *o)
{
  if (!THPVariable_Check(o)) throw Error{PyExc_TypeError, "expected a torch tensor"};
  return THPVariable_Unpack(o);
}

// device memory, contiguous: the C ABI sees raw pointers
const at::Tensor &device_tensor(PyObject *o)
{
  const at::Tensor &t = tensor(o);
  if (!t.is_cuda()) throw Error{PyExc_RuntimeError, "host backend not supported"};
  if (!t.is_contiguous()) throw Error{PyExc_RuntimeError, "tensor must be contiguous"};
  return t;
}

int64_t integer(PyObject *o)
{
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw Error{nullptr, nullptr};
  return v;
}

int code_of(at::ScalarType t)
{
  switch (t) {
    case at::kFloat: return CAIFX_F32;
    case at::kHalf: return CAIFX_F16;
    case at::kBFloat16: return CAIFX_BF16;
    default: throw Error{PyExc_KeyError, "tensor must be fp32, fp16 or bf16"};
  }
}

at::ScalarType type_of(int64_t code)
{
  switch (code) {
    case CAIFX_F32: return at::kFloat;
    case CAIFX_F16: return at::kHalf;
    case CAIFX_BF16: return at::kBFloat16;
    default: throw Error{PyExc_KeyError, "unknown dtype code"};
  }
}

// an attribute of a Python weight object; names are interned once
struct Attr {
  PyObject *name;
  explicit Attr(const char *s) : name(PyUnicode_InternFromString(s)) {}
};

struct Owned {
  PyObject *p;
  explicit Owned(PyObject *q) : p(q)
  {
    if (!p) throw Error{nullptr, nullptr};
  }
  ~Owned() { Py_DECREF(p); }
  Owned(const Owned &) = delete;
  Owned &operator=(const Owned &) = delete;
};

int64_t int_attr(PyObject *o, const Attr &a) { return integer(Owned(PyObject_GetAttr(o, a.name)).p); }

// data pointer of a tensor attribute, null for None (the weight object keeps the tensor alive)
void *ptr_attr(PyObject *o, const Attr &a)
{
  Owned v(PyObject_GetAttr(o, a.name));
  return v.p == Py_None ? nullptr : tensor(v.p).data_ptr();
}

struct WeightAttrs {
  Attr wq{"wq"}, scales{"scales"}, wq_ptrs{"wq_ptrs"}, scales_ptrs{"scales_ptrs"}, weights{"weights"}, n{"N"}, k{"K"},
      kind{"w_kind"}, period{"scale_period"}, group{"group_size"};
};
const WeightAttrs &attrs()
{
  static const WeightAttrs a;
  return a;
}

// the launch itself without the interpreter lock: it can wait for room in the queue.  It takes the entry point and its
// arguments, so whatever can throw (sizes, data pointers, the stream) is evaluated while the lock is held.
struct Unlocked {
  PyThreadState *state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename... P, typename... A> int launch(int (*entry)(P...), A... args)
{
  const Unlocked without_lock;
  return entry(args...);
}

void *stream() { return static_cast<void *>(c10::hip::getCurrentHIPStream().stream()); }

at::Tensor bytes_like(const at::Tensor &x, size_t n)
{
  return at::empty({static_cast<int64_t>(n)}, x.options().dtype(at::kByte));
}

// the caller's workspace, or one of the size the library asks for (none for zero bytes)
struct Workspace {
  at::Tensor held;
  void *p = nullptr;
  size_t bytes = 0;
  template <typename Query> Workspace(PyObject *given, const at::Tensor &x, Query query)
  {
    if (given != Py_None) {
      const at::Tensor &t = tensor(given);
      p = t.data_ptr();
      bytes = static_cast<size_t>(t.numel());
    } else if ((bytes = query()) > 0) {
      // the workspace is optional: on a card that is full up to the result the calls run without it, as those kernels do that
      // never asked for one
      try {
        held = bytes_like(x, bytes);
        p = held.data_ptr();
      } catch (const c10::OutOfMemoryError &) {
        bytes = 0;
      }
    }
  }
};

PyObject *result(int status, const at::Tensor &t)
{
  if (status != CAIFX_OK) return PyLong_FromLong(status);
  return THPVariable_Wrap(t);
}

// argument count, C++ and Python errors
template <typename F> PyObject *guarded(Py_ssize_t have, Py_ssize_t want, F f)
{
  if (have != want) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, have);
    return nullptr;
  }
  try {
    return f();
  } catch (const Error &e) {
    if (e.type) PyErr_SetString(e.type, e.what);
    return nullptr;
  } catch (const c10::Error &e) {
    // torch's own out-of-memory type where there is one
    PyObject *type = PyExc_RuntimeError;
    if (std::strstr(e.what_without_backtrace(), "out of memory")) {
      PyObject *torch = PyImport_ImportModule("torch");
      PyObject *oom = torch ? PyObject_GetAttrString(torch, "OutOfMemoryError") : nullptr;
      Py_XDECREF(torch);
      PyErr_Clear();
      if (oom) {
        PyErr_SetString(oom, e.what_without_backtrace());
        Py_DECREF(oom);
        return nullptr;
      }
    }
    PyErr_SetString(type, e.what_without_backtrace());
    return nullptr;
  } catch (const std::exception &e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// ------------------------------------------------------------------ frozen linear
// qlinear(backward, x, weight, compute_dtype, out_dtype, out, workspace, addend) -> result or status
PyObject *qlinear(PyObject *, PyObject *const *a, Py_ssize_t n)
{
  return guarded(n, 8, [&]() -> PyObject * {
    const bool backward = integer(a[0]) != 0;
    const at::Tensor &x = device_tensor(a[1]);
    PyObject *w = a[2];
    const WeightAttrs &at_ = attrs();
    const int64_t N = int_attr(w, at_.n), K = int_attr(w, at_.k);
    const int64_t in = backward ? N : K, out_dim = backward ? K : N;
    if (in <= 0) throw Error{PyExc_ValueError, "the weight has no elements"};
    const int64_t M = x.numel() / in;
    const int compute = static_cast<int>(integer(a[3])), od = static_cast<int>(integer(a[4]));
    const int xd = code_of(x.scalar_type());
    const int kind = static_cast<int>(int_attr(w, at_.kind));
    const int64_t period = int_attr(w, at_.period);
    const int group = static_cast<int>(int_attr(w, at_.group));
    const void *wq = ptr_attr(w, at_.wq), *scales = ptr_attr(w, at_.scales);
    const at::Tensor y = a[5] != Py_None ? tensor(a[5]) : at::empty({M, out_dim}, x.options().dtype(type_of(od)));
    const Workspace ws(a[6], x, [&] { return api.caifx_qlinear_workspace_bytes(M, N, K, xd, compute, kind, backward ? 1 : 0); });
    if (a[7] != Py_None) {
      const at::Tensor &add = tensor(a[7]);
      if (add.scalar_type() != y.scalar_type() || add.numel() != y.numel())
        throw Error{PyExc_AssertionError, "the addend must have the result's dtype and size"};
      const auto fn = backward ? api.caifx_qlinear_backward_input_add : api.caifx_qlinear_forward_add;
      return result(launch(fn, M, N, K, x.data_ptr(), xd, compute, wq, kind, scales, period, group, y.data_ptr(), od, add.data_ptr(), ws.p, ws.bytes, stream()), y);
    }
    const auto fn = backward ? api.caifx_qlinear_backward_input : api.caifx_qlinear_forward;
    return result(launch(fn, M, N, K, x.data_ptr(), xd, compute, wq, kind, scales, period, group, y.data_ptr(), od, ws.p, ws.bytes, stream()), y);
  });
}

// grouped(backward, x, offsets, weights, compute_dtype, out_dtype, out, workspace, addend) -> result or status
PyObject *grouped(PyObject *, PyObject *const *a, Py_ssize_t n)
{
  return guarded(n, 9, [&]() -> PyObject * {
    const bool backward = integer(a[0]) != 0;
    const at::Tensor &x = device_tensor(a[1]);
    const at::Tensor &offsets = device_tensor(a[2]);
    PyObject *w = a[3];
    const WeightAttrs &at_ = attrs();
    const int64_t N = int_attr(w, at_.n), K = int_attr(w, at_.k);
    const int64_t in = backward ? N : K, out_dim = backward ? K : N;
    if (in <= 0) throw Error{PyExc_ValueError, "the weight has no elements"};
    const int64_t rows = x.numel() / in;
    const int compute = static_cast<int>(integer(a[4])), od = static_cast<int>(integer(a[5]));
    const int xd = code_of(x.scalar_type());
    const int kind = static_cast<int>(int_attr(w, at_.kind));
    Owned list(PyObject_GetAttr(w, at_.weights.name));
    const Py_ssize_t E = PySequence_Size(list.p);
    if (E < 0) throw Error{nullptr, nullptr};
    // sizes and dtypes are checked here, before anything is launched
    if (x.numel() != rows * in) throw Error{PyExc_ValueError, "the input's size is not a multiple of the reduction length"};
    if (offsets.scalar_type() != at::kInt || offsets.numel() != E + 1) throw Error{PyExc_ValueError, "offsets must be int32 [experts + 1]"};
    if (a[6] != Py_None) {
      const at::Tensor &o = device_tensor(a[6]);
      if (o.scalar_type() != type_of(od) || o.numel() != rows * out_dim)
        throw Error{PyExc_ValueError, "the result tensor must have the result's dtype and rows x columns elements"};
    }
    const at::Tensor y = a[6] != Py_None ? tensor(a[6]) : at::empty({rows, out_dim}, x.options().dtype(type_of(od)));
    const int64_t period = int_attr(w, at_.period);
    const int group = static_cast<int>(int_attr(w, at_.group));
    const auto wq = static_cast<const void *const *>(ptr_attr(w, at_.wq_ptrs));
    const auto scales = static_cast<const void *const *>(ptr_attr(w, at_.scales_ptrs));
    const Workspace ws(a[7], x, [&] {
      return api.caifx_qlinear_grouped_workspace_bytes(static_cast<int>(E), rows, N, K, xd, compute, kind, backward ? 1 : 0);
    });
    const auto off = static_cast<const int32_t *>(offsets.data_ptr());
    const void *addend = nullptr;
    if (a[8] != Py_None) {
      if (!backward) throw Error{PyExc_AssertionError, "the forward takes no addend"};
      const at::Tensor &add = tensor(a[8]);
      if (add.scalar_type() != y.scalar_type() || add.numel() != y.numel())
        throw Error{PyExc_AssertionError, "the addend must have the result's dtype and size"};
      addend = add.data_ptr();
    }
    // a fresh result's rows outside the segments are zero
    if (a[6] == Py_None)
      return result(launch(api.caifx_qlinear_grouped_fresh, backward ? 1 : 0, static_cast<int>(E), off, rows, N, K, x.data_ptr(), xd, compute, wq, kind, scales,
                           period, group, y.data_ptr(), od, addend, ws.p, ws.bytes, stream()), y);
    if (addend) {
      return result(launch(api.caifx_qlinear_grouped_backward_input_add, static_cast<int>(E), off, rows, N, K, x.data_ptr(), xd, compute, wq, kind, scales,
                                                                 period, group, y.data_ptr(), od, addend, ws.p, ws.bytes, stream()), y);
    }
    const auto fn = backward ? api.caifx_qlinear_grouped_backward_input : api.caifx_qlinear_grouped_forward;
    return result(launch(fn, static_cast<int>(E), off, rows, N, K, x.data_ptr(), xd, compute, wq, kind, scales, period, group, y.data_ptr(), od, ws.p,
                     ws.bytes, stream()), y);
  });
}

PyObject *pair(int status, const at::Tensor &x, const at::Tensor &y)
{
  if (status != CAIFX_OK) return PyLong_FromLong(status);
  Owned p(THPVariable_Wrap(x)), q(THPVariable_Wrap(y));
  return PyTuple_Pack(2, p.p, q.p);
}

// ------------------------------------------------------------------ quantise
// quantize_int8(x, per_channel) -> (codes, scales) or status
PyObject *quantize_int8(PyObject *, PyObject *const *a, Py_ssize_t n)
{
  return guarded(n, 2, [&]() -> PyObject * {
    const at::Tensor &x = device_tensor(a[0]);
    if (x.scalar_type() != at::kFloat) throw Error{PyExc_RuntimeError, "QuantizeInt8: input must be fp32"};
    const int per_channel = PyObject_IsTrue(a[1]);
    if (per_channel < 0) throw Error{nullptr, nullptr};
    if (per_channel && x.dim() != 2) throw Error{PyExc_RuntimeError, "QuantizeInt8 PerChannel: input must be 2D"};
    const at::Tensor q = at::empty(x.sizes(), x.options().dtype(at::kChar));
    const at::Tensor s = at::empty({per_channel ? x.size(1) : 1}, x.options());
    const auto in = static_cast<const float *>(x.data_ptr());
    if (!per_channel) return pair(launch(api.caifx_quantize_int8_per_tensor, in, q.data_ptr(), s.data_ptr(), x.numel(), stream()), q, s);
    const int64_t rows = x.size(0), cols = x.size(1);
    if (rows > INT32_MAX || cols > INT32_MAX) throw Error{PyExc_OverflowError, "QuantizeInt8 PerChannel: too many rows or columns"};
    return pair(launch(api.caifx_quantize_int8_per_channel, in, q.data_ptr(), s.data_ptr(), static_cast<int>(rows), static_cast<int>(cols), stream()), q, s);
  });
}

// quantize_int4(x, group_size) -> (packed, fp16 scales) or status
PyObject *quantize_int4(PyObject *, PyObject *const *a, Py_ssize_t n)
{
  return guarded(n, 2, [&]() -> PyObject * {
    const at::Tensor &x = device_tensor(a[0]);
    if (x.scalar_type() != at::kFloat) throw Error{PyExc_RuntimeError, "QuantizeInt4PerGroup: input must be fp32"};
    const int64_t group = integer(a[1]), count = x.numel();
    if (group == 0) throw Error{PyExc_RuntimeError, "QuantizeInt4PerGroup: group_size must be > 0"};
    if (group > INT32_MAX || group < INT32_MIN) throw Error{PyExc_OverflowError, "QuantizeInt4PerGroup: group_size out of range"};
    const int64_t groups = group > 0 ? (count + group - 1) / group : 0;      // a negative size is the library's error
    const at::Tensor packed = at::empty({(count + 1) / 2}, x.options().dtype(at::kByte));
    const at::Tensor s = at::empty({groups}, x.options().dtype(at::kHalf));
    return pair(launch(api.caifx_quantize_to_int4, static_cast<const float *>(x.data_ptr()), packed.data_ptr(), s.data_ptr(), count, static_cast<int>(group), stream()), packed, s);
  });
}

// ------------------------------------------------------------------ element-wise
// elementwise(op, a, b or None, out or None): 0 silu, 1 silu_backward, 2 multiply, 3 add, 4 silu_multiply
PyObject *elementwise(PyObject *, PyObject *const *a, Py_ssize_t n)
{
  return guarded(n, 4, [&]() -> PyObject * {
    const at::Tensor &x = device_tensor(a[1]);
    const void *b = a[2] == Py_None ? nullptr : device_tensor(a[2]).data_ptr();
    if (a[3] != Py_None) {
      const at::Tensor &o = tensor(a[3]);
      if (!o.is_cuda()) throw Error{PyExc_RuntimeError, "host backend not supported"};
      if (o.scalar_type() != x.scalar_type() || o.numel() != x.numel() || !o.is_contiguous())
        throw Error{o.is_contiguous() ? PyExc_ValueError : PyExc_RuntimeError,
                    o.is_contiguous() ? "out must be a contiguous tensor of the input's dtype and size" : "tensor must be contiguous"};
    }
    const at::Tensor y = a[3] != Py_None ? tensor(a[3]) : at::empty_like(x);
    const int dt = code_of(x.scalar_type());
    const int64_t op = integer(a[0]);
    if (op == 0) return result(launch(api.caifx_silu, x.data_ptr(), y.data_ptr(), x.numel(), dt, stream()), y);
    const auto fn = op == 1 ? api.caifx_silu_backward : op == 2 ? api.caifx_multiply : op == 3 ? api.caifx_add : api.caifx_silu_multiply;
    return result(launch(fn, x.data_ptr(), b, y.data_ptr(), x.numel(), dt, stream()), y);
  });
}

// swiglu_backward(gate, up, grad_hidden, out_gate, out_up) -> (grad_gate, grad_up) or status
PyObject *swiglu_backward(PyObject *, PyObject *const *a, Py_ssize_t n)
{
  return guarded(n, 5, [&]() -> PyObject * {
    const at::Tensor &gate = device_tensor(a[0]), &up = device_tensor(a[1]), &gh = device_tensor(a[2]);
    if (gate.sizes() != up.sizes() || gate.sizes() != gh.sizes() || gate.scalar_type() != up.scalar_type() || gate.scalar_type() != gh.scalar_type())
      throw Error{PyExc_AssertionError, "gate, up and grad_hidden must have one shape and dtype"};
    const at::Tensor gg = a[3] != Py_None ? tensor(a[3]) : at::empty_like(gate);
    const at::Tensor gu = a[4] != Py_None ? tensor(a[4]) : at::empty_like(gate);
    const int dt = code_of(gate.scalar_type());
    const int st = launch(api.caifx_swiglu_backward, gate.data_ptr(), up.data_ptr(), gh.data_ptr(), gg.data_ptr(), gu.data_ptr(), gate.numel(), dt, stream());
    if (st != CAIFX_OK) return PyLong_FromLong(st);
    Owned p(THPVariable_Wrap(gg)), q(THPVariable_Wrap(gu));
    return PyTuple_Pack(2, p.p, q.p);
  });
}

// ------------------------------------------------------------------ MoE token routing
// moe_build_dispatch_map(expert_indices, num_experts, capacity) -> (map, offsets) or status
PyObject *moe_build_dispatch_map(PyObject *, PyObject *const *a, Py_ssize_t n)
{
  return guarded(n, 3, [&]() -> PyObject * {
    const at::Tensor &ids = device_tensor(a[0]);
    if (ids.scalar_type() != at::kInt || ids.dim() != 2) throw Error{PyExc_AssertionError, "expert_indices must be int32 [tokens, top_k]"};
    const int64_t tokens = ids.size(0);
    const int top_k = static_cast<int>(ids.size(1)), E = static_cast<int>(integer(a[1]));
    const at::Tensor map = at::empty_like(ids);
    const at::Tensor offsets = at::empty({E + 1}, ids.options());
    size_t nb = api.caifx_moe_dispatch_map_workspace_bytes(tokens, top_k, E);
    if (nb < 4 * static_cast<size_t>(E)) nb = 4 * static_cast<size_t>(E);
    const at::Tensor ws = bytes_like(ids, nb);
    const int capacity = static_cast<int>(integer(a[2]));
    return pair(launch(api.caifx_moe_build_dispatch_map, static_cast<const int32_t *>(ids.data_ptr()), tokens, top_k, E, capacity,
                                                 static_cast<int32_t *>(map.data_ptr()), static_cast<int32_t *>(offsets.data_ptr()), ws.data_ptr(),
                                                 nb, stream()), map, offsets);
  });
}

// rows x columns: the tensor that gives the number of tokens has no other rank
const at::Tensor &matrix(const at::Tensor &t)
{
  if (t.dim() != 2) throw Error{PyExc_ValueError, "expected a two-dimensional tensor"};
  return t;
}

// the second extent of a tensor of two dimensions or more
int64_t columns(const at::Tensor &t)
{
  if (t.dim() < 2) throw Error{PyExc_IndexError, "expected a tensor of at least two dimensions"};
  return t.size(1);
}

const int32_t *ints(PyObject *o) { return static_cast<const int32_t *>(device_tensor(o).data_ptr()); }

// moe_dispatch(x, ids, map, offsets, total_rows, out)
PyObject *moe_dispatch(PyObject *, PyObject *const *a, Py_ssize_t n)
{
  return guarded(n, 6, [&]() -> PyObject * {
    const at::Tensor &x = device_tensor(a[0]), &ids = device_tensor(a[1]), &offsets = device_tensor(a[3]);
    const int64_t tokens = matrix(x).size(0), dim = x.size(1), top_k = columns(ids);
    const bool fresh = a[5] == Py_None;
    const at::Tensor buf = fresh ? at::empty({integer(a[4]), dim}, x.options()) : tensor(a[5]);
    const int32_t *i1 = ints(a[1]); const int32_t *i2 = ints(a[2]); const int32_t *i3 = ints(a[3]); const int dt = code_of(x.scalar_type());
    if (fresh)
      return result(launch(api.caifx_moe_dispatch_fresh, x.data_ptr(), i1, i2, i3, buf.data_ptr(), buf.size(0), tokens, dim,
                                               static_cast<int>(top_k), static_cast<int>(offsets.numel() - 1), dt, stream()), buf);
    return result(launch(api.caifx_moe_dispatch, x.data_ptr(), i1, i2, i3, buf.data_ptr(), tokens, dim,
                                         static_cast<int>(top_k), static_cast<int>(offsets.numel() - 1), dt, stream()), buf);
  });
}

// moe_combine(expert_buffer, ids, weights, map, offsets, out)
PyObject *moe_combine(PyObject *, PyObject *const *a, Py_ssize_t n)
{
  return guarded(n, 6, [&]() -> PyObject * {
    const at::Tensor &buf = device_tensor(a[0]), &ids = device_tensor(a[1]), &w = device_tensor(a[2]), &offsets = device_tensor(a[4]);
    const int64_t tokens = matrix(ids).size(0), dim = columns(buf), top_k = ids.size(1);
    const at::Tensor y = a[5] != Py_None ? tensor(a[5]) : at::empty({tokens, dim}, buf.options());
    const int32_t *i1 = ints(a[1]); const int32_t *i3 = ints(a[3]); const int32_t *i4 = ints(a[4]); const int dt = code_of(buf.scalar_type());
    return result(launch(api.caifx_moe_combine, buf.data_ptr(), i1, w.data_ptr(), i3, i4, y.data_ptr(), tokens, dim,
                                        static_cast<int>(top_k), static_cast<int>(offsets.numel() - 1), dt, stream()), y);
  });
}

// moe_combine_backward_grad_expert(grad_output, ids, weights, map, offsets, total_rows, out)
PyObject *moe_combine_backward_grad_expert(PyObject *, PyObject *const *a, Py_ssize_t n)
{
  return guarded(n, 7, [&]() -> PyObject * {
    const at::Tensor &g = device_tensor(a[0]), &ids = device_tensor(a[1]), &w = device_tensor(a[2]), &offsets = device_tensor(a[4]);
    const int64_t tokens = matrix(g).size(0), dim = g.size(1), top_k = columns(ids);
    const bool fresh = a[6] == Py_None;
    const at::Tensor buf = fresh ? at::empty({integer(a[5]), dim}, g.options()) : tensor(a[6]);
    const int32_t *i1 = ints(a[1]); const int32_t *i3 = ints(a[3]); const int32_t *i4 = ints(a[4]); const int dt = code_of(g.scalar_type());
    if (fresh)
      return result(launch(api.caifx_moe_combine_backward_grad_expert_fresh, g.data_ptr(), i1, w.data_ptr(), i3, i4, buf.data_ptr(), buf.size(0), tokens,
                                                                   dim, static_cast<int>(top_k), static_cast<int>(offsets.numel() - 1), dt, stream()), buf);
    return result(launch(api.caifx_moe_combine_backward_grad_expert, g.data_ptr(), i1, w.data_ptr(), i3, i4, buf.data_ptr(), tokens, dim,
                                                             static_cast<int>(top_k), static_cast<int>(offsets.numel() - 1),
                                                             dt, stream()), buf);
  });
}

// moe_dispatch_backward(grad_expert_buffer, ids, map, offsets, out)
PyObject *moe_dispatch_backward(PyObject *, PyObject *const *a, Py_ssize_t n)
{
  return guarded(n, 5, [&]() -> PyObject * {
    const at::Tensor &g = device_tensor(a[0]), &ids = device_tensor(a[1]), &offsets = device_tensor(a[3]);
    const int64_t tokens = matrix(ids).size(0), dim = columns(g), top_k = ids.size(1);
    const at::Tensor y = a[4] != Py_None ? tensor(a[4]) : at::empty({tokens, dim}, g.options());
    const int32_t *i1 = ints(a[1]); const int32_t *i2 = ints(a[2]); const int32_t *i3 = ints(a[3]); const int dt = code_of(g.scalar_type());
    return result(launch(api.caifx_moe_dispatch_backward, g.data_ptr(), i1, i2, i3, y.data_ptr(), tokens, dim,
                                                  static_cast<int>(top_k), static_cast<int>(offsets.numel() - 1), dt,
                                                  stream()), y);
  });
}

// moe_combine_backward_grad_weights(grad_output, expert_buffer, ids, map, offsets)
PyObject *moe_combine_backward_grad_weights(PyObject *, PyObject *const *a, Py_ssize_t n)
{
  return guarded(n, 5, [&]() -> PyObject * {
    const at::Tensor &g = device_tensor(a[0]), &buf = device_tensor(a[1]), &ids = device_tensor(a[2]), &offsets = device_tensor(a[4]);
    const int64_t tokens = matrix(ids).size(0), top_k = ids.size(1), dim = columns(g);
    const at::Tensor y = at::empty({tokens, top_k}, g.options());
    const int32_t *i2 = ints(a[2]); const int32_t *i3 = ints(a[3]); const int32_t *i4 = ints(a[4]); const int dt = code_of(g.scalar_type());
    return result(launch(api.caifx_moe_combine_backward_grad_weights, g.data_ptr(), buf.data_ptr(), i2, i3, i4, y.data_ptr(), tokens, dim,
                                                              static_cast<int>(top_k), static_cast<int>(offsets.numel() - 1),
                                                              dt, stream()), y);
  });
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
#define M(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr},
    M(qlinear) M(grouped) M(quantize_int8) M(quantize_int4) M(elementwise) M(swiglu_backward) M(moe_build_dispatch_map) M(moe_dispatch) M(moe_combine)
    M(moe_combine_backward_grad_expert) M(moe_dispatch_backward) M(moe_combine_backward_grad_weights)
#undef M
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "caifx_torch_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject *PyInit_caifx_torch_calls() { return PyModule_Create(&module); }
