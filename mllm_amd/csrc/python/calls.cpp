// The short calls of mllm_amd/qlinear.py in native code: argument checks, output tensors and the call into the C ABI.  A decode-size launch
// takes the host 2.5 us; the same checks in Python and a ctypes call took another 2.3 (one projection of a token: 4.8 us, 3.3 now), a torch.empty
// 1.7 of which the allocator needs a third.  The Linear over many rows is two launches, which short prompts are done with before
// Python had queued them: 139 x 2176 x 1248 Q4_0 8.7 -> 7.7 us, 79 x 4384 x 2016 9.3 -> 8.7.  Same checks, results and streams as the Python code had, and the same exceptions but
// one: an argument that is no tensor is a TypeError (AttributeError before).  The interpreter's lock is released for the call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "mllm_hip_qlinear.h"

namespace {

PyObject *g_error, *g_check;                  // HipQLinearError, _lib.check
PyObject *g_stream, *g_device;                // torch._C._cuda_getCurrentRawStream, _cuda_getDevice
PyObject *s_wtype, *s_buf, *s_N, *s_K, *s_layout;

// an error is set: unwinds to the entry point, which returns it
struct Raised {};
[[noreturn]] void raise(PyObject* type, const char* what = nullptr) {
  if (what) PyErr_SetString(type, what);
  else PyErr_SetNone(type);
  throw Raised();
}
void require(bool ok) {
  if (!ok) raise(PyExc_AssertionError);
}
const at::Tensor& tensor(PyObject* o) {
  if (!THPVariable_Check(o)) raise(PyExc_TypeError, "a torch.Tensor is needed");
  return THPVariable_Unpack(o);
}
void* pointer(PyObject* o) { return o == Py_None ? nullptr : tensor(o).data_ptr(); }
int64_t integer(PyObject* o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw Raised();
  return v;
}
int truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw Raised();
  return v;
}
struct Owned {  // a new reference
  PyObject* o;
  explicit Owned(PyObject* p) : o(p) {
    if (!p) throw Raised();
  }
  ~Owned() { Py_DECREF(o); }
  Owned(const Owned&) = delete;
};
int64_t number(PyObject* o) { return integer(Owned(PyNumber_Long(o)).o); }  // int(o): flags that are no whole numbers (numpy's booleans)
int64_t attribute(PyObject* o, PyObject* name) { return integer(Owned(PyObject_GetAttr(o, name)).o); }
void* stream() {  // the current stream of the current device
  Owned device(PyObject_CallNoArgs(g_device));
  Owned handle(PyObject_CallOneArg(g_stream, device.o));
  void* p = PyLong_AsVoidPtr(handle.o);
  if (!p && PyErr_Occurred()) throw Raised();
  return p;
}
int xdtype(const at::Tensor& x) {
  if (x.scalar_type() == at::kFloat) return MLLM_HIP_F32;
  if (x.scalar_type() == at::kBFloat16) return MLLM_HIP_BF16;
  raise(PyExc_TypeError, "activations must be float32 or bfloat16");
}
at::Tensor empty(at::IntArrayRef sizes, at::ScalarType type) { return at::empty(sizes, at::TensorOptions().dtype(type).device(at::kCUDA)); }
// the caller's workspace, which has to hold what the call writes (the C ABI takes its size on trust), or a new one
void* workspace(PyObject* o, size_t bytes, at::Tensor& made) {
  if (o == Py_None) return (made = empty({(int64_t)bytes}, at::kByte)).data_ptr();
  const at::Tensor& t = tensor(o);
  if (t.nbytes() < bytes) {
    PyErr_Format(g_error, "a workspace of %zu bytes, %zu needed", (size_t)t.nbytes(), bytes);
    throw Raised();
  }
  return t.data_ptr();
}
void need_rank(const at::Tensor& t, int64_t dims) {
  if (t.dim() < dims) raise(PyExc_IndexError, "tuple index out of range");
}
PyObject* given(PyObject* o) {
  Py_INCREF(o);
  return o;
}
template <typename F>
void run(const char* what, F f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS rc = f();
  Py_END_ALLOW_THREADS
  if (rc != 0) {
    PyObject* r = PyObject_CallFunction(g_check, "is", rc, what);
    Py_XDECREF(r);
    if (!PyErr_Occurred()) PyErr_SetString(g_error, what);
    throw Raised();
  }
}

typedef PyObject* const* Args;

// (wtype, buf, N, K, x, bias, act_scale_mode, out)
PyObject* linear_q_gemv(Args a) {
  const int64_t N = integer(a[2]), K = integer(a[3]);
  const at::Tensor& x = tensor(a[4]);
  require(x.is_cuda() && x.is_contiguous() && x.dim() == 2 && x.size(1) == K);
  const int64_t M = x.size(0);
  at::Tensor made;
  if (a[7] == Py_None) made = empty({M, N}, at::kFloat);
  float* y = static_cast<float*>(a[7] == Py_None ? made.data_ptr() : pointer(a[7]));
  const int wtype = (int)integer(a[0]), xt = xdtype(x), mode = (int)integer(a[6]);
  const void *w = pointer(a[1]), *xp = x.data_ptr();
  const float* bias = static_cast<const float*>(pointer(a[5]));
  void* st = stream();
  run("mllm_hip_linear_q_gemv", [&] { return mllm_hip_linear_q_gemv(wtype, w, xp, xt, bias, y, M, N, K, mode, st); });
  return a[7] == Py_None ? THPVariable_Wrap(made) : given(a[7]);
}

// (ws, x, biases, act_scale_mode, outs, workspace)
PyObject* linear_q_gemv_multi(Args a) {
  Owned ws(PySequence_Fast(a[0], "a list of weights is needed"));
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(ws.o);
  const at::Tensor& x = tensor(a[1]);
  require(n >= 1 && n <= 4 && x.is_cuda() && x.is_contiguous() && x.dim() == 2);
  const int64_t M = x.size(0), K = x.size(1);
  mllm_hip_gemv_part parts[4];
  int wtype = 0;
  Owned outs(a[4] == Py_None ? PyList_New(n) : given(a[4]));
  for (Py_ssize_t i = 0; i < n; i++) {
    PyObject* w = PySequence_Fast_GET_ITEM(ws.o, i);
    const int type = (int)attribute(w, s_wtype);
    if (i == 0) wtype = type;
    require(attribute(w, s_K) == K && type == wtype);
    const int64_t N = attribute(w, s_N);
    if (a[4] == Py_None) {
      PyObject* y = THPVariable_Wrap(empty({M, N}, at::kFloat));
      if (!y) throw Raised();
      PyList_SET_ITEM(outs.o, i, y);
    }
    Owned y(PySequence_GetItem(outs.o, i)), buf(PyObject_GetAttr(w, s_buf));
    const void* bias = nullptr;
    if (a[2] != Py_None) bias = pointer(Owned(PySequence_GetItem(a[2], i)).o);
    parts[i] = mllm_hip_gemv_part{pointer(buf.o), static_cast<const float*>(bias), static_cast<float*>(tensor(y.o).data_ptr()), N};
  }
  const int xt = xdtype(x), mode = (int)integer(a[3]);
  void *xp = x.data_ptr(), *work = pointer(a[5]), *st = stream();
  const size_t room = a[5] == Py_None ? 0 : (size_t)tensor(a[5]).numel();
  run("mllm_hip_linear_q_gemv_multi_wsn", [&] { return mllm_hip_linear_q_gemv_multi_wsn(wtype, (int)n, parts, xp, xt, M, K, mode, work, room, st); });
  return given(outs.o);
}

// (x)
PyObject* softmax(Args a) {
  const at::Tensor& x = tensor(a[0]);
  require(x.is_cuda() && x.is_contiguous() && x.scalar_type() == at::kFloat);
  need_rank(x, 1);
  const int64_t n = x.size(-1);
  at::Tensor y = at::empty_like(x), work;
  if (n == 0) raise(PyExc_ZeroDivisionError, "integer division or modulo by zero");
  const int64_t rows = x.numel() / n;
  const size_t need = mllm_hip_softmax_workspace_bytes(rows, n);
  if (need) work = empty({(int64_t)need}, at::kByte);
  const float* xp = static_cast<const float*>(x.data_ptr());
  float* yp = static_cast<float*>(y.data_ptr());
  void *wp = need ? work.data_ptr() : nullptr, *st = stream();
  run("mllm_hip_softmax_ws", [&] { return mllm_hip_softmax_ws(xp, yp, rows, n, wp, st); });
  return THPVariable_Wrap(y);
}

// (x, k, largest, sorted)
PyObject* topk(Args a) {
  const at::Tensor& x = tensor(a[0]);
  require(x.is_cuda() && x.is_contiguous() && x.scalar_type() == at::kFloat);
  need_rank(x, 1);
  const int64_t n = x.size(-1), k = integer(a[1]);
  const int largest = (int)number(a[2]), sorted = (int)number(a[3]);
  at::DimVector shape(x.sizes().begin(), x.sizes().end());
  shape.back() = k;
  at::Tensor v = empty(shape, at::kFloat), i = empty(shape, at::kInt), work;
  if (n == 0) raise(PyExc_ZeroDivisionError, "integer division or modulo by zero");
  const int64_t rows = x.numel() / n;
  const size_t need = mllm_hip_topk_workspace_bytes(rows, n, (int)k);
  if (need) work = empty({(int64_t)need}, at::kByte);
  const float* xp = static_cast<const float*>(x.data_ptr());
  float* vp = static_cast<float*>(v.data_ptr());
  int32_t* ip = static_cast<int32_t*>(i.data_ptr());
  void *wp = need ? work.data_ptr() : nullptr, *st = stream();
  run("mllm_hip_topk_ws", [&] { return mllm_hip_topk_ws(xp, vp, ip, rows, n, (int)k, largest, sorted, wp, st); });
  Owned vo(THPVariable_Wrap(v)), io(THPVariable_Wrap(i));
  return PyTuple_Pack(2, vo.o, io.o);
}

// (a, b, transpose_a, transpose_b, out)
PyObject* matmul(Args p) {
  const at::Tensor &a = tensor(p[0]), &b = tensor(p[1]);
  const at::ScalarType type = a.scalar_type();
  require(type == b.scalar_type() && (type == at::kFloat || type == at::kBFloat16 || type == at::kHalf) && a.is_contiguous() && b.is_contiguous());
  need_rank(a, 2);
  need_rank(b, 2);
  const int ta = truth(p[2]), tb = truth(p[3]);
  const int64_t M = a.size(ta ? -1 : -2), K = a.size(ta ? -2 : -1), N = b.size(tb ? -2 : -1);
  require(K == b.size(tb ? -1 : -2));
  int64_t batch = 1, bbatch = 1;
  for (int64_t d = 0; d < a.dim() - 2; d++) batch *= a.size(d);
  for (int64_t d = 0; d < b.dim() - 2; d++) bbatch *= b.size(d);
  require(bbatch == 1 || bbatch == batch);
  at::Tensor made;
  if (p[4] == Py_None) {
    at::DimVector shape(a.sizes().begin(), a.sizes().end());
    shape[shape.size() - 2] = M, shape.back() = N;
    made = empty(shape, type);
  }
  void *ap = a.data_ptr(), *bp = b.data_ptr(), *cp = p[4] == Py_None ? made.data_ptr() : pointer(p[4]), *st = stream();
  const int dtype = type == at::kFloat ? (int)MLLM_HIP_F32 : type == at::kBFloat16 ? (int)MLLM_HIP_BF16 : (int)MLLM_HIP_F16;
  run("mllm_hip_matmul_batched", [&] {
    return mllm_hip_matmul_batched(ap, bp, cp, dtype, batch, M, N, K, M * K, bbatch == batch && batch > 1 ? N * K : 0, M * N, ta, tb, st);
  });
  return p[4] == Py_None ? THPVariable_Wrap(made) : given(p[4]);
}

void two_dimensional(const at::Tensor& x) {
  if (x.dim() != 2) raise(PyExc_ValueError, "a matrix is needed");
}

// (x, W_packed, N, w_scale, bias, workspace, out)
PyObject* w8a8_linear_packed(Args a) {
  const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]);
  two_dimensional(x);
  const int64_t M = x.size(0), K = x.size(1), N = integer(a[2]);
  require(w.numel() == (int64_t)mllm_hip_w8a8_packed_bytes(N, K));
  at::Tensor work, made;
  void* sp = workspace(a[5], mllm_hip_w8a8_workspace_bytes(M, K), work);
  if (a[6] == Py_None) made = empty({M, N}, at::kBFloat16);
  const int xt = xdtype(x);
  void *xp = x.data_ptr(), *wp = w.data_ptr(), *yp = a[6] == Py_None ? made.data_ptr() : pointer(a[6]);
  const float *scale = static_cast<const float*>(tensor(a[3]).data_ptr()), *bias = static_cast<const float*>(pointer(a[4]));
  void* st = stream();
  run("mllm_hip_w8a8_linear_packed", [&] { return mllm_hip_w8a8_linear_packed(xp, xt, wp, scale, bias, yp, M, N, K, sp, st); });
  return a[6] == Py_None ? THPVariable_Wrap(made) : given(a[6]);
}

// (a, packed, N, bias, group, out)
PyObject* w4a16_gemm_packed(Args a) {
  const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]);
  require(x.scalar_type() == at::kBFloat16 && x.is_contiguous());
  two_dimensional(x);
  const int64_t M = x.size(0), K = x.size(1), N = integer(a[2]);
  const int group = (int)integer(a[4]);
  require(w.numel() == (int64_t)mllm_hip_w4a16_packed_bytes(N, K, group));
  at::Tensor made;
  if (a[5] == Py_None) made = empty({M, N}, at::kBFloat16);
  void *xp = x.data_ptr(), *wp = w.data_ptr(), *bp = pointer(a[3]), *yp = a[5] == Py_None ? made.data_ptr() : pointer(a[5]), *st = stream();
  run("mllm_hip_w4a16_gemm_packed", [&] { return mllm_hip_w4a16_gemm_packed(xp, wp, bp, yp, M, N, K, group, st); });
  return a[5] == Py_None ? THPVariable_Wrap(made) : given(a[5]);
}

// a Linear over many rows: w, x, bias, workspace, out, short of both kinds of block formats
template <typename Bytes, typename ShortBytes, typename Call>
PyObject* linear_gemm(const char* what, PyObject* w, PyObject* xo, PyObject* bias, PyObject* room, PyObject* out, Bytes bytes, ShortBytes short_bytes,
                      bool shorter, Call call) {
  const at::Tensor& x = tensor(xo);
  require(x.is_cuda() && x.is_contiguous() && x.dim() == 2 && x.size(1) == attribute(w, s_K));
  Owned layout(PyObject_GetAttr(w, s_layout)), buf(PyObject_GetAttr(w, s_buf));
  require(PyUnicode_Check(layout.o) && PyUnicode_CompareWithASCIIString(layout.o, "gemm") == 0);
  const int64_t M = x.size(0), K = x.size(1), N = attribute(w, s_N);
  const int wtype = (int)attribute(w, s_wtype), xt = xdtype(x);
  at::Tensor work, made;
  void* sp = workspace(room, shorter ? short_bytes(M, N, K) : bytes(M, K), work);
  if (out == Py_None) made = empty({M, N}, at::kFloat);
  const void *wp = pointer(buf.o), *xp = x.data_ptr();
  const float* bp = static_cast<const float*>(pointer(bias));
  float* yp = static_cast<float*>(out == Py_None ? made.data_ptr() : pointer(out));
  void* st = stream();
  run(what, [&] { return call(wtype, wp, xp, xt, bp, yp, M, N, K, sp, st); });
  return out == Py_None ? THPVariable_Wrap(made) : given(out);
}

// (w, x, bias, act_scale_mode, workspace, out, short)
PyObject* linear_q_gemm(Args a) {
  const bool shorter = truth(a[6]);
  const int mode = (int)integer(a[3]);
  return linear_gemm("mllm_hip_linear_q_gemm", a[0], a[1], a[2], a[4], a[5], mllm_hip_linear_q_gemm_workspace_bytes, mllm_hip_linear_q_gemm_short_workspace_bytes, shorter,
                     [&](int wtype, const void* w, const void* x, int xt, const float* bias, float* y, int64_t M, int64_t N, int64_t K, void* work, void* st) {
                       return (shorter ? mllm_hip_linear_q_gemm_short : mllm_hip_linear_q_gemm)(wtype, w, x, xt, bias, y, M, N, K, mode, work, st);
                     });
}

// (w, x, bias, workspace, out, short)
PyObject* linear_kq_gemm(Args a) {
  const bool shorter = truth(a[5]);
  return linear_gemm("mllm_hip_linear_kq_gemm", a[0], a[1], a[2], a[3], a[4], mllm_hip_linear_kq_gemm_workspace_bytes, mllm_hip_linear_kq_gemm_short_workspace_bytes, shorter,
                     shorter ? mllm_hip_linear_kq_gemm_short : mllm_hip_linear_kq_gemm);
}

template <PyObject* (*F)(Args), int N>
PyObject* entry(PyObject*, Args args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "%d arguments are needed", N);
    return nullptr;
  }
  try {
    return F(args);
  } catch (const Raised&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}
#define CALL(name, n) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(entry<name, n>)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {CALL(linear_q_gemv, 8), CALL(linear_q_gemv_multi, 6), CALL(softmax, 1), CALL(topk, 4), CALL(matmul, 5),
                           CALL(w8a8_linear_packed, 7), CALL(w4a16_gemm_packed, 6), CALL(linear_q_gemm, 7), CALL(linear_kq_gemm, 6), {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "mllm_calls", nullptr, -1, g_methods};

}  // namespace

PyMODINIT_FUNC PyInit_mllm_calls() {
  PyObject* m = PyModule_Create(&g_module);
  PyObject *lib = PyImport_ImportModule("mllm_amd._lib"), *torch = PyImport_ImportModule("torch._C");
  if (!m || !lib || !torch) return nullptr;
  g_error = PyObject_GetAttrString(lib, "HipQLinearError");
  g_check = PyObject_GetAttrString(lib, "check");
  g_stream = PyObject_GetAttrString(torch, "_cuda_getCurrentRawStream");
  g_device = PyObject_GetAttrString(torch, "_cuda_getDevice");
  s_wtype = PyUnicode_InternFromString("wtype");
  s_buf = PyUnicode_InternFromString("buf");
  s_N = PyUnicode_InternFromString("N");
  s_K = PyUnicode_InternFromString("K");
  s_layout = PyUnicode_InternFromString("layout");
  if (!g_error || !g_check || !g_stream || !g_device || !s_wtype || !s_buf || !s_N || !s_K || !s_layout) return nullptr;
  return m;
}
