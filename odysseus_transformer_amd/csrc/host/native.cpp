// The ops of ops.py in their plain form -- checks, allocations and the call of the C ABI -- without a trip through Python and ctypes
// for each of them.
//
// Bound by the interpreter: the wrappers in ops.py take 9 to 15 us per op, of which the launch is 2; a decoding step, a short sequence
// or a small layer is a row of ops whose kernels take no longer.  A decoding step of hidden 4096 behind 8191 tokens (8 ops of 110 us of
// kernels): 176 us a pass through Python, 110 through here; attention of 4 x 331 tokens, forward and backward: 88 us of host work, now 65 (without the graph).
//
// A function here answers None for whatever is not the plain form of its op: a tensor that is not a dense CUDA tensor of the current
// device (subclasses, wrappers of function transforms, conjugate or negative views included), a shape or stride that needs a copy or an
// error message, a workspace that does not fit.  Its caller then goes on with the checks and copies written in Python, which stay the
// definition of what an op accepts and of the error it raises.
//
// No state but what bind() is given once: the addresses of the library's entry points, so that this module uses the library that
// Python loaded, and six Python objects.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <c10/util/Exception.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstring>

#include "odysseus_hip.h"

namespace {

// ------------------------------------------------------------------------------------------------ the library and Python's side
#define ODY_ENTRY_POINTS(X)                                                                                                       \
  X(ody_rmsnorm_fwd) X(ody_rmsnorm_bwd_partials) X(ody_rmsnorm_bwd) X(ody_gemm_workspace_bytes) X(ody_gemm) X(ody_linear_residual_ws) \
  X(ody_linear_rope_ws) X(ody_linear_swiglu) X(ody_linear_swiglu_h_fused) X(ody_linear_swiglu_h)                                  \
  X(ody_linear_dgrad_swiglu_workspace_bytes) X(ody_linear_dgrad_swiglu) X(ody_attn_fwd_workspace_bytes) X(ody_attn_fwd)           \
  X(ody_attn_bwd_workspace_bytes) X(ody_attn_bwd) X(ody_attn_bwd_rope) X(ody_rope) X(ody_rope_table)           \
  X(ody_norm_linear_rope) X(ody_norm_linear_swiglu_h)

struct Library {
#define X(name) decltype(&::name) name = nullptr;
  ODY_ENTRY_POINTS(X)
#undef X
} lib;
PyObject* arena_holder = nullptr;   // class whose attribute `instance` is the scratch arena, or None
PyObject* scratch_fn = nullptr;     // scratch(nbytes, name, device) of ops.py
PyObject* raise_fn = nullptr;       // raises for (name, status)
PyObject* no_memory = nullptr;      // torch.OutOfMemoryError
PyObject* never_keeps_ds = nullptr; // _never_keeps_ds() of ops.py
PyObject* attn_bwd_fn = nullptr;    // attn_bwd(q, k, v, out, lse, dout, causal, scale) of ops.py

struct NotPlain {};      // the caller answers None
struct PythonError {};   // a Python exception is set

// ------------------------------------------------------------------------------------------------ arguments
constexpr c10::DispatchKeySet special{c10::DispatchKey::Python,          c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
                                      c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize, c10::DispatchKey::Batched,
                                      c10::DispatchKey::Conjugate,       c10::DispatchKey::Negative,          c10::DispatchKey::ZeroTensor};

void need(bool plain) {
  if (!plain) throw NotPlain{};
}

bool plain_tensor(const at::Tensor& t) {
  return t.defined() && t.is_cuda() && t.layout() == c10::Layout::Strided && !t.unsafeGetTensorImpl()->key_set().has_any(special) && t.numel() > 0;
}

// The arguments of one call; `like` (the first tensor) sets device and dtype.
struct Call {
  PyObject* const* args;
  Py_ssize_t n;
  c10::DeviceIndex device;
  hipStream_t stream;

  Call(PyObject* const* a, Py_ssize_t count, Py_ssize_t expected) : args(a), n(count), device(-1), stream(nullptr) { need(count == expected); }

  // any strided tensor of the current device
  const at::Tensor& any(Py_ssize_t i) {
    PyObject* o = args[i];
    need(THPVariable_CheckExact(o));
    const at::Tensor& t = THPVariable_Unpack(o);
    need(plain_tensor(t));
    if (device < 0) {
      device = c10::hip::current_device();
      stream = c10::hip::getCurrentHIPStream(device).stream();
    }
    need(t.get_device() == device);
    return t;
  }
  // ... that the kernels compute with
  const at::Tensor& values(Py_ssize_t i) {
    const at::Tensor& t = any(i);
    need(t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat);
    return t;
  }
  const at::Tensor& like(Py_ssize_t i, const at::Tensor& ref) {
    const at::Tensor& t = any(i);
    need(t.scalar_type() == ref.scalar_type());
    return t;
  }
  // row-major, rows any distance apart
  const at::Tensor& matrix(Py_ssize_t i, const at::Tensor* ref) {
    const at::Tensor& t = ref ? like(i, *ref) : values(i);
    need(t.dim() == 2 && t.stride(1) == 1 && t.size(0) < INT32_MAX && t.size(1) < INT32_MAX);
    return t;
  }
  // (B, L, H, D)
  const at::Tensor& heads(Py_ssize_t i, const at::Tensor* ref) {
    const at::Tensor& t = ref ? like(i, *ref) : values(i);
    need(t.dim() == 4 && t.stride(3) == 1);
    for (int d = 0; d < 4; d++) need(t.size(d) < INT32_MAX);
    return t;
  }
  bool none(Py_ssize_t i) const { return args[i] == Py_None; }
  bool flag(Py_ssize_t i) const {
    need(PyBool_Check(args[i]));
    return args[i] == Py_True;
  }
  int64_t whole(Py_ssize_t i) const {
    need(PyLong_CheckExact(args[i]));
    const int64_t v = PyLong_AsLongLong(args[i]);
    if (v == -1 && PyErr_Occurred()) throw PythonError{};
    return v;
  }
  double real(Py_ssize_t i) const {
    need(PyFloat_Check(args[i]) || PyLong_CheckExact(args[i]));
    const double v = PyFloat_AsDouble(args[i]);
    if (v == -1 && PyErr_Occurred()) throw PythonError{};
    return v;
  }
};

int dt(const at::Tensor& t) { return t.scalar_type() == at::kBFloat16 ? ODY_BF16 : ODY_F32; }
int64_t pitch(const at::Tensor& t) { return t.size(0) > 1 ? t.stride(0) : std::max(t.stride(0), t.size(1)); }
at::Tensor make(at::IntArrayRef shape, const at::Tensor& like) { return at::empty(shape, like.options().requires_grad(false)); }
at::Tensor make_f32(at::IntArrayRef shape, const at::Tensor& like) { return at::empty(shape, like.options().dtype(at::kFloat).requires_grad(false)); }

// Kernel scratch, from the arena where one is set up.  Nothing: no such memory; the caller of the op has other ways.
struct Scratch {
  at::Tensor t;
  size_t bytes;
  Scratch(size_t nbytes, const char* name, const at::Tensor& like) : bytes(nbytes) {
    if (nbytes == 0) return;
    PyObject* arena = PyObject_GetAttrString(arena_holder, "instance");
    if (!arena) throw PythonError{};
    const bool have = arena != Py_None;
    Py_DECREF(arena);
    if (have) {
      PyObject* device = THPDevice_New_(like);
      PyObject* r = PyObject_CallFunction(scratch_fn, "nsO", (Py_ssize_t)nbytes, name, device);
      Py_XDECREF(device);
      if (!r) {
        if (!PyErr_ExceptionMatches(no_memory)) throw PythonError{};
        PyErr_Clear();
        throw NotPlain{};
      }
      t = THPVariable_Unpack(r);
      Py_DECREF(r);
      return;
    }
    try {
      t = at::empty({(int64_t)nbytes}, like.options().dtype(at::kByte).requires_grad(false));
    } catch (const c10::OutOfMemoryError&) {
      throw NotPlain{};
    }
  }
  void* ptr() const { return t.defined() ? t.data_ptr() : nullptr; }

 private:
  static PyObject* THPDevice_New_(const at::Tensor& like) {
    PyObject* o = THPVariable_Wrap(like);
    PyObject* d = o ? PyObject_GetAttrString(o, "device") : nullptr;
    Py_XDECREF(o);
    if (!d) throw PythonError{};
    return d;
  }
};

// an entry point's answer; the interpreter is free meanwhile (a launch waits where the queue is full)
template <typename F, typename... A>
void call(const char* name, F fn, A... a) {
  int rc;
  {
    PyThreadState* save = PyEval_SaveThread();
    rc = fn(a...);
    PyEval_RestoreThread(save);
  }
  if (rc == 0) return;
  PyObject* r = PyObject_CallFunction(raise_fn, "si", name, rc);
  Py_XDECREF(r);
  if (r) PyErr_Format(PyExc_RuntimeError, "%s failed with status %d", name, rc);
  throw PythonError{};
}
#define CALL(name, ...) call(#name, lib.name, __VA_ARGS__)

PyObject* wrap(const at::Tensor& t) {
  PyObject* o = THPVariable_Wrap(t);
  if (!o) throw PythonError{};
  return o;
}
template <typename... T>
PyObject* tuple(const T&... t) {
  PyObject* r = PyTuple_New(sizeof...(T));
  if (!r) throw PythonError{};
  Py_ssize_t i = 0;
  (PyTuple_SET_ITEM(r, i++, wrap(t)), ...);
  return r;
}

// ------------------------------------------------------------------------------------------------ the ops
// (x, weight, eps) -> (y, rstd)
PyObject* rmsnorm_fwd(Call c) {
  const at::Tensor &x = c.values(0), &w = c.like(1, x);
  need(x.dim() >= 1 && x.is_contiguous() && w.dim() == 1 && w.is_contiguous() && w.size(0) == x.size(-1));
  const int64_t d = x.size(-1), T = x.numel() / d;
  need(T < INT32_MAX && d < INT32_MAX);
  const float eps = (float)c.real(2);
  at::Tensor y = make(x.sizes(), x), rstd = make_f32({T}, x);
  CALL(ody_rmsnorm_fwd, x.data_ptr(), w.data_ptr(), y.data_ptr(), rstd.data_ptr<float>(), (int)T, (int)d, eps, dt(x), (void*)c.stream);
  return tuple(y, rstd);
}

// (x, weight, rstd, dy, dx_add or None) -> (dx, dw)
PyObject* rmsnorm_bwd(Call c) {
  const at::Tensor &x = c.values(0), &w = c.like(1, x), &rstd = c.any(2), &dy = c.like(3, x);
  need(x.dim() >= 1 && x.is_contiguous() && w.dim() == 1 && w.is_contiguous() && w.size(0) == x.size(-1));
  const int64_t d = x.size(-1), T = x.numel() / d;
  need(T < INT32_MAX && d < INT32_MAX && rstd.scalar_type() == at::kFloat && rstd.is_contiguous() && rstd.numel() == T);
  need(dy.sizes() == x.sizes() && dy.is_contiguous());
  const at::Tensor* add = c.none(4) ? nullptr : &c.like(4, x);
  need(!add || (add->sizes() == x.sizes() && add->is_contiguous()));
  at::Tensor dx = make(x.sizes(), x), dw = make(w.sizes(), w);
  Scratch part((size_t)lib.ody_rmsnorm_bwd_partials((int)T) * d * 4, "rmsnorm_dw_partials", x);
  CALL(ody_rmsnorm_bwd, x.data_ptr(), w.data_ptr(), rstd.data_ptr<float>(), dy.data_ptr(), add ? add->data_ptr() : nullptr, dx.data_ptr(),
       (float*)part.ptr(), dw.data_ptr(), (int)T, (int)d, dt(x), (void*)c.stream);
  return tuple(dx, dw);
}

// (op, a, b) -> out
PyObject* gemm(Call c) {
  const int64_t op = c.whole(0);
  const at::Tensor &a = c.matrix(1, nullptr), &b = c.matrix(2, &a);
  need(op == ODY_GEMM_NT || op == ODY_GEMM_NN || op == ODY_GEMM_TN);
  const int64_t M = a.size(op == ODY_GEMM_TN ? 1 : 0), K = a.size(op == ODY_GEMM_TN ? 0 : 1), N = b.size(op == ODY_GEMM_NT ? 0 : 1);
  need(b.size(op == ODY_GEMM_NT ? 1 : 0) == K);
  at::Tensor out = make({M, N}, a);
  Scratch ws(lib.ody_gemm_workspace_bytes((int)op, (int)M, (int)N, (int)K, dt(a)), "gemm_workspace", a);
  CALL(ody_gemm, (int)op, a.data_ptr(), b.data_ptr(), out.data_ptr(), nullptr, (int)M, (int)N, (int)K, pitch(a), pitch(b), pitch(out), 0, dt(a),
       ws.ptr(), ws.bytes, (void*)c.stream);
  return wrap(out);
}

// (x, weight, residual) -> y
PyObject* linear_residual(Call c) {
  const at::Tensor &x = c.matrix(0, nullptr), &w = c.matrix(1, &x), &r = c.matrix(2, &x);
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  need(w.size(1) == K && r.size(0) == M && r.size(1) == N);
  at::Tensor y = make({M, N}, x);
  Scratch ws(lib.ody_gemm_workspace_bytes(ODY_GEMM_NT, (int)M, (int)N, (int)K, dt(x)), "gemm_workspace", x);
  CALL(ody_linear_residual_ws, x.data_ptr(), w.data_ptr(), r.data_ptr(), y.data_ptr(), (int)M, (int)N, (int)K, pitch(x), pitch(w), pitch(r),
       y.stride(0), dt(x), ws.ptr(), ws.bytes, (void*)c.stream);
  return wrap(y);
}

// (x, weight, table, n_rot, head_dim) -> y
PyObject* linear_rope(Call c) {
  const at::Tensor &x = c.matrix(0, nullptr), &w = c.matrix(1, &x), &table = c.matrix(2, &x);
  const int64_t n_rot = c.whole(3), D = c.whole(4), M = x.size(0), K = x.size(1), N = w.size(0);
  need(x.scalar_type() == at::kBFloat16 && D == 128 && w.size(1) == K && N % D == 0 && n_rot >= 0 && n_rot <= N / D);
  need(table.is_contiguous() && table.size(0) == M && table.size(1) == D);
  at::Tensor y = make({M, N}, x);
  Scratch ws(lib.ody_gemm_workspace_bytes(ODY_GEMM_NT, (int)M, (int)N, (int)K, dt(x)), "gemm_workspace", x);
  CALL(ody_linear_rope_ws, x.data_ptr(), w.data_ptr(), table.data_ptr(), y.data_ptr(), (int)M, (int)N, (int)K, (int)n_rot, (int)D, pitch(x),
       pitch(w), table.stride(0), y.stride(0), dt(x), ws.ptr(), ws.bytes, (void*)c.stream);
  return wrap(y);
}

// (x, w_gate_up) -> (gate_up, h)
PyObject* linear_swiglu(Call c) {
  const at::Tensor &x = c.matrix(0, nullptr), &w = c.matrix(1, &x);
  const int64_t T = x.size(0), K = x.size(1), I2 = w.size(0);
  need(w.size(1) == K && I2 % 2 == 0);
  at::Tensor gu = make({T, I2}, x), h = make({T, I2 / 2}, x);
  CALL(ody_linear_swiglu, x.data_ptr(), w.data_ptr(), gu.data_ptr(), h.data_ptr(), (int)T, (int)(I2 / 2), (int)K, pitch(x), pitch(w), gu.stride(0),
       h.stride(0), dt(x), (void*)c.stream);
  return tuple(gu, h);
}

// (x, w_gate_up) -> h, where one kernel does it
PyObject* linear_swiglu_h(Call c) {
  const at::Tensor &x = c.matrix(0, nullptr), &w = c.matrix(1, &x);
  const int64_t T = x.size(0), K = x.size(1), I2 = w.size(0);
  need(w.size(1) == K && I2 % 2 == 0 &&
       lib.ody_linear_swiglu_h_fused(x.data_ptr(), w.data_ptr(), (int)T, (int)(I2 / 2), (int)K, pitch(x), pitch(w), dt(x)) != 0);
  at::Tensor h = make({T, I2 / 2}, x);
  CALL(ody_linear_swiglu_h, x.data_ptr(), w.data_ptr(), h.data_ptr(), (int)T, (int)(I2 / 2), (int)K, pitch(x), pitch(w), h.stride(0), dt(x),
       (void*)c.stream);
  return wrap(h);
}

// (dy, w_down, gate_up) -> d_gate_up
PyObject* linear_dgrad_swiglu(Call c) {
  const at::Tensor &dy = c.matrix(0, nullptr), &w = c.matrix(1, &dy), &gu = c.matrix(2, &dy);
  const int64_t T = dy.size(0), K = dy.size(1), I = w.size(1);
  need(w.size(0) == K && gu.size(0) == T && gu.size(1) == 2 * I);
  for (const at::Tensor* t : {&dy, &w, &gu})   // what one kernel wants where the size query goes by the shape alone
    need(reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0 && t->stride(0) % 8 == 0);
  need(pitch(dy) < (1 << 22) && pitch(w) < (1 << 24));
  at::Tensor dgu = make({T, 2 * I}, dy);
  Scratch ws(lib.ody_linear_dgrad_swiglu_workspace_bytes((int)T, (int)I, (int)K, dt(dy)), "dgrad_swiglu_workspace", dy);
  CALL(ody_linear_dgrad_swiglu, dy.data_ptr(), w.data_ptr(), gu.data_ptr(), dgu.data_ptr(), (int)T, (int)I, (int)K, pitch(dy), pitch(w), pitch(gu),
       dgu.stride(0), dt(dy), ws.ptr(), ws.bytes, (void*)c.stream);
  return wrap(dgu);
}

#define STRIDES(t) (t).stride(0), (t).stride(1), (t).stride(2)

void check_kv(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  need(k.sizes() == v.sizes() && k.size(0) == q.size(0) && k.size(3) == q.size(3));
}

struct OutLse { at::Tensor out, lse; };
OutLse run_attn_fwd(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, bool causal, float scale, hipStream_t stream) {
  const int B = q.size(0), Lq = q.size(1), Hq = q.size(2), D = q.size(3), Lk = k.size(1), Hkv = k.size(2);
  at::Tensor out = make({B, Lq, Hq, D}, q), lse = make_f32({B, Hq, Lq}, q);
  Scratch ws(lib.ody_attn_fwd_workspace_bytes(B, Lq, Lk, Hq, Hkv, D, dt(q)), "attn_fwd_workspace", q);
  CALL(ody_attn_fwd, q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr<float>(), B, Lq, Lk, Hq, Hkv, D, STRIDES(q), STRIDES(k),
       STRIDES(v), STRIDES(out), scale, (int)causal, dt(q), ws.ptr(), ws.bytes, (void*)stream);
  return {out, lse};
}

// (q, k, v, causal, scale) -> (out, lse)
PyObject* attn_fwd(Call c) {
  const at::Tensor &q = c.heads(0, nullptr), &k = c.heads(1, &q), &v = c.heads(2, &q);
  check_kv(q, k, v);
  const OutLse r = run_attn_fwd(q, k, v, c.flag(3), (float)c.real(4), c.stream);
  return tuple(r.out, r.lse);
}

// (q, k, v, out, lse, dout, causal, scale, dq or None, dk or None, dv or None, table_q or None, table_k or None) -> (dq, dk, dv)
void run_attn_bwd(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& out, const at::Tensor& lse, const at::Tensor& dout,
                  bool causal, float scale, at::Tensor (&g)[3], const at::Tensor* const (&table)[2], hipStream_t stream) {
  const int B = q.size(0), Lq = q.size(1), Hq = q.size(2), D = q.size(3), Lk = k.size(1), Hkv = k.size(2);
  Scratch ws(lib.ody_attn_bwd_workspace_bytes(B, Lq, Lk, Hq, Hkv, D, dt(q)), "attn_bwd_workspace", q);
#define BWD_ARGS                                                                                                                   \
  q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr<float>(), dout.data_ptr(), g[0].data_ptr(), g[1].data_ptr(), \
      g[2].data_ptr(), B, Lq, Lk, Hq, Hkv, D, STRIDES(q), STRIDES(k), STRIDES(v), STRIDES(out), STRIDES(dout), STRIDES(g[0]),       \
      STRIDES(g[1]), STRIDES(g[2]), scale, (int)causal, 0, dt(q), ws.ptr(), ws.bytes, (void*)stream
  if (table[0]) CALL(ody_attn_bwd_rope, BWD_ARGS, table[0]->data_ptr(), table[1]->data_ptr());
  else CALL(ody_attn_bwd, BWD_ARGS);
}
void check_bwd(const at::Tensor& q, const at::Tensor& out, const at::Tensor& lse, const at::Tensor& dout) {
  need(out.sizes() == q.sizes() && dout.sizes() == q.sizes());
  need(lse.scalar_type() == at::kFloat && lse.is_contiguous() && lse.dim() == 3 && lse.size(0) == q.size(0) && lse.size(1) == q.size(2) &&
       lse.size(2) == q.size(1));
}
at::Tensor gradient_of(const at::Tensor& t) { return at::empty_like(t, t.options().requires_grad(false)); }

PyObject* attn_bwd(Call c) {
  const at::Tensor &q = c.heads(0, nullptr), &k = c.heads(1, &q), &v = c.heads(2, &q), &out = c.heads(3, &q), &lse = c.any(4), &dout = c.heads(5, &q);
  check_kv(q, k, v);
  const bool causal = c.flag(6);
  const float scale = (float)c.real(7);
  const int64_t B = q.size(0), Lq = q.size(1), D = q.size(3), Lk = k.size(1);
  check_bwd(q, out, lse, dout);
  at::Tensor g[3];
  const at::Tensor* of[3] = {&q, &k, &v};
  for (int i = 0; i < 3; i++) {
    g[i] = c.none(8 + i) ? gradient_of(*of[i]) : c.heads(8 + i, &q);
    need(g[i].sizes() == of[i]->sizes() && g[i].stride(3) == 1);
  }
  need(c.none(11) == c.none(12));
  const at::Tensor* table[2] = {nullptr, nullptr};
  if (!c.none(11))
    for (int i = 0; i < 2; i++) {
      table[i] = &c.matrix(11 + i, &q);
      need(q.scalar_type() == at::kBFloat16 && table[i]->is_contiguous() && table[i]->size(0) == B * (i ? Lk : Lq) && table[i]->size(1) == D);
    }
  run_attn_bwd(q, k, v, out, lse, dout, causal, scale, g, table, c.stream);
  return tuple(g[0], g[1], g[2]);
}

// ------------------------------------------------------------------------------------------------ the attention routine as a node of the graph
// What FlashAttnFunc of ops.py is, without dropout.  Forward and backward of 4 x 331 tokens, 8 heads on 2, 49 us of kernels, in a loop: 99 us of host work
// a pass through autograd's Python function, 80 through this one, of which an empty graph and the clearing of gradients take 35.  Its backward holds the
// interpreter, as the scratch arena and the budget of kept dS are Python's, and where the plain form of attn_bwd is not the one to be taken it calls
// that function.  Transforms, forward mode and tracing are left to the Python function (ops.transformed).
struct Interpreter {
  PyGILState_STATE state = PyGILState_Ensure();
  ~Interpreter() { PyGILState_Release(state); }
};
[[noreturn]] void throw_python_error() {
  python_error e;
  e.persist();
  throw e;
}

struct FlashNode : torch::autograd::Function<FlashNode> {
  using Tensors = torch::autograd::variable_list;

  static Tensors forward(torch::autograd::AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, bool causal, double scale,
                         void* stream) {
    OutLse r = run_attn_fwd(q, k, v, causal, (float)scale, (hipStream_t)stream);
    ctx->save_for_backward({q, k, v, r.out, r.lse});
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["scale"] = scale;
    ctx->mark_non_differentiable({r.lse});
    ctx->set_materialize_grads(false);
    return {r.out, r.lse};
  }

  static Tensors backward(torch::autograd::AutogradContext* ctx, const Tensors& grads) {
    const Tensors saved = ctx->get_saved_variables();
    const at::Tensor &q = saved[0], &k = saved[1], &v = saved[2], &out = saved[3], &lse = saved[4];
    at::Tensor dout = grads[0].defined() ? grads[0] : at::zeros_like(out);
    if (dout.dim() == 4 && dout.stride(3) != 1) dout = dout.contiguous();
    const bool causal = ctx->saved_data["causal"].toBool();
    const double scale = ctx->saved_data["scale"].toDouble();
    Interpreter held;
    try {
      if (PyObject* never = PyObject_CallNoArgs(never_keeps_ds)) {
        const bool plain = never == Py_True;
        Py_DECREF(never);
        if (plain) {
          try {
            const c10::DeviceIndex device = c10::hip::current_device();
            for (const at::Tensor* t : {&q, &k, &v, &out, &lse, (const at::Tensor*)&dout}) need(plain_tensor(*t) && t->get_device() == device);
            for (const at::Tensor* t : {&k, &v, &out, (const at::Tensor*)&dout}) need(t->scalar_type() == q.scalar_type());
            for (const at::Tensor* t : {&q, &k, &v, &out, (const at::Tensor*)&dout}) need(t->dim() == 4 && t->stride(3) == 1);
            check_bwd(q, out, lse, dout);
            at::Tensor g[3] = {gradient_of(q), gradient_of(k), gradient_of(v)};
            for (const at::Tensor& t : g) need(t.stride(3) == 1);
            const at::Tensor* const table[2] = {nullptr, nullptr};
            run_attn_bwd(q, k, v, out, lse, dout, causal, (float)scale, g, table, c10::hip::getCurrentHIPStream(device).stream());
            return {g[0], g[1], g[2], at::Tensor(), at::Tensor(), at::Tensor()};
          } catch (const NotPlain&) {
          }
        }
        const at::Tensor args[6] = {q, k, v, out, lse, dout};
        PyObject* a = PyTuple_New(8);
        if (!a) throw PythonError{};
        for (int i = 0; i < 6; i++) PyTuple_SET_ITEM(a, i, THPVariable_Wrap(args[i]));
        PyTuple_SET_ITEM(a, 6, PyBool_FromLong(causal));
        PyTuple_SET_ITEM(a, 7, PyFloat_FromDouble(scale));
        PyObject* r = PyErr_Occurred() ? nullptr : PyObject_CallObject(attn_bwd_fn, a);
        Py_DECREF(a);
        if (!r) throw PythonError{};
        Tensors g;
        for (int i = 0; i < 3; i++) g.push_back(THPVariable_Unpack(PyTuple_GET_ITEM(r, i)));
        Py_DECREF(r);
        g.resize(6);
        return g;
      }
      throw PythonError{};
    } catch (const PythonError&) {
      throw_python_error();
    }
  }
};

// (q, k, v, causal, scale) -> (out, lse), recorded where one of them requires a gradient
PyObject* flash(Call c) {
  const at::Tensor &q = c.heads(0, nullptr), &k = c.heads(1, &q), &v = c.heads(2, &q);
  check_kv(q, k, v);
  const auto r = FlashNode::apply(q, k, v, c.flag(3), c.real(4), (void*)c.stream);
  return tuple(r[0], r[1]);
}

const int64_t* positions(Call& c, Py_ssize_t i, int64_t rows) {
  if (c.none(i)) return nullptr;
  const at::Tensor& p = c.any(i);
  need(p.scalar_type() == at::kLong && p.is_contiguous() && p.numel() == rows);
  return p.data_ptr<int64_t>();
}
const at::Tensor& frequencies(Call& c, Py_ssize_t i, int64_t D) {
  const at::Tensor& f = c.any(i);
  need(D % 2 == 0 && f.scalar_type() == at::kFloat && f.is_contiguous() && f.numel() == D / 2);
  return f;
}

// (x, n_rot, position_ids or None, inv_freq, base, inverse) -> True: x (B, L, H, D) is rotated in place
PyObject* rope(Call c) {
  const at::Tensor& x = c.heads(0, nullptr);
  const int64_t n_rot = c.whole(1);
  const int B = x.size(0), L = x.size(1), D = x.size(3);
  need(n_rot >= 0 && n_rot <= x.size(2));
  if (!c.none(2)) {   // (B, L), or (L) of a batch of one
    const at::Tensor& given = c.any(2);
    need((given.dim() == 2 || (given.dim() == 1 && B == 1)) && given.size(-1) == L);
  }
  const int64_t* pos = positions(c, 2, (int64_t)B * L);
  const at::Tensor& f = frequencies(c, 3, D);
  need(f.dim() == 1);
  CALL(ody_rope, x.data_ptr(), pos, f.data_ptr<float>(), B, L, (int)n_rot, D, STRIDES(x), (float)c.real(4), (int)c.flag(5), dt(x), (void*)c.stream);
  Py_RETURN_TRUE;
}

// (position_ids or None, rows, head_dim, inv_freq, base) -> table
PyObject* rope_table(Call c) {
  const int64_t rows = c.whole(1), D = c.whole(2);
  const at::Tensor& f = frequencies(c, 3, D);
  need(rows > 0);
  const int64_t* pos = positions(c, 0, rows);
  at::Tensor table = at::empty({rows, D}, f.options().dtype(at::kBFloat16).requires_grad(false));
  CALL(ody_rope_table, pos, f.data_ptr<float>(), rows, (int)D, (float)c.real(4), table.data_ptr(), (void*)c.stream);
  return wrap(table);
}

// What ody_norm_linear_* take: bf16 rows of x and of the weight on 16-byte boundaries, few of x.
void check_norm_linear(const at::Tensor& x, const at::Tensor& norm, const at::Tensor& w) {
  need(x.scalar_type() == at::kBFloat16 && x.size(0) <= 4 && x.size(0) * (x.size(1) + 8) * 2 <= 64 * 1024 && x.size(1) % 8 == 0 && w.size(1) == x.size(1));
  need(norm.dim() == 1 && norm.is_contiguous() && norm.size(0) == x.size(1));
  for (const at::Tensor* t : {&x, &norm, &w}) need(reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0);
  need(pitch(x) % 8 == 0 && pitch(w) % 8 == 0);
}

// (x, norm_weight, eps, weight, n_rot, head_dim, position_ids, inv_freq) -> y
PyObject* norm_linear_rope(Call c) {
  const at::Tensor &x = c.matrix(0, nullptr), &norm = c.like(1, x), &w = c.matrix(3, &x);
  check_norm_linear(x, norm, w);
  const int64_t n_rot = c.whole(4), D = c.whole(5), M = x.size(0), K = x.size(1), N = w.size(0);
  need(D == 128 && N % D == 0 && n_rot >= 0 && n_rot <= N / D && !c.none(6));
  const float eps = (float)c.real(2);
  const int64_t* pos = positions(c, 6, M);
  const at::Tensor& f = frequencies(c, 7, D);
  at::Tensor y = make({M, N}, x);
  CALL(ody_norm_linear_rope, x.data_ptr(), norm.data_ptr(), eps, w.data_ptr(), pos, f.data_ptr<float>(), y.data_ptr(), (int)M, (int)N, (int)K,
       (int)n_rot, (int)D, pitch(x), pitch(w), y.stride(0), dt(x), (void*)c.stream);
  return wrap(y);
}

// (x, norm_weight, eps, w_gate_up) -> h
PyObject* norm_linear_swiglu_h(Call c) {
  const at::Tensor &x = c.matrix(0, nullptr), &norm = c.like(1, x), &w = c.matrix(3, &x);
  check_norm_linear(x, norm, w);
  const int64_t T = x.size(0), K = x.size(1), I = w.size(0) / 2;
  need(w.size(0) % 32 == 0);
  const float eps = (float)c.real(2);
  at::Tensor h = make({T, I}, x);
  CALL(ody_norm_linear_swiglu_h, x.data_ptr(), norm.data_ptr(), eps, w.data_ptr(), h.data_ptr(), (int)T, (int)I, (int)K, pitch(x), pitch(w),
       h.stride(0), dt(x), (void*)c.stream);
  return wrap(h);
}

// the raw stream that the ops above launch on
PyObject* current_stream(Call) {
  return PyLong_FromVoidPtr((void*)c10::hip::getCurrentHIPStream(c10::hip::current_device()).stream());
}

template <PyObject* (*OP)(Call), int N>
PyObject* method(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  try {
    return OP(Call(args, n, N));
  } catch (const NotPlain&) {
    Py_RETURN_NONE;
  } catch (const PythonError&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// (addresses by name, arena holder, scratch, raise, torch.OutOfMemoryError, _never_keeps_ds, attn_bwd)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 7 || !PyDict_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "bind(addresses, arena_holder, scratch, raise, no_memory, never_keeps_ds, attn_bwd)");
    return nullptr;
  }
#define X(name)                                                                      \
  {                                                                                  \
    PyObject* a = PyDict_GetItemString(args[0], #name);                              \
    void* p = a ? PyLong_AsVoidPtr(a) : nullptr;                                     \
    if (!p) {                                                                        \
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, #name);                 \
      return nullptr;                                                                \
    }                                                                                \
    lib.name = reinterpret_cast<decltype(lib.name)>(p);                              \
  }
  ODY_ENTRY_POINTS(X)
#undef X
  PyObject** to[6] = {&arena_holder, &scratch_fn, &raise_fn, &no_memory, &never_keeps_ds, &attn_bwd_fn};
  for (int i = 0; i < 6; i++) {
    Py_INCREF(args[1 + i]);
    Py_XSETREF(*to[i], args[1 + i]);
  }
  Py_RETURN_NONE;
}

#define METHOD(name, n) {#name, (PyCFunction)(void (*)(void))method<name, n>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
    METHOD(rmsnorm_fwd, 3), METHOD(rmsnorm_bwd, 5), METHOD(gemm, 3), METHOD(linear_residual, 3), METHOD(linear_rope, 5), METHOD(linear_swiglu, 2),
    METHOD(linear_swiglu_h, 2), METHOD(linear_dgrad_swiglu, 3), METHOD(attn_fwd, 5), METHOD(attn_bwd, 13), METHOD(flash, 5), METHOD(rope, 6), METHOD(rope_table, 5),
    METHOD(norm_linear_rope, 8), METHOD(norm_linear_swiglu_h, 4),
    METHOD(current_stream, 0), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_odysseus_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__odysseus_native() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "TORCH_VERSION", ODY_TORCH_VERSION) != 0) Py_CLEAR(m);
  return m;
}
