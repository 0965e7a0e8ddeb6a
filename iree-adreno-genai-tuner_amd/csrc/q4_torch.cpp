// CPython module _q4torch: the ordinary calls of the tensor-level wrappers (q4llm/ops.py, QLinear.forward)
// in native code.
//
// A decode projection or a decode attention call takes 4 to 8 us on the GPU, and the Python wrapper took 11
// to 17 us of host time: checks, attribute reads, torch.empty, the current stream and the ctypes
// conversions. Each function here does the same for the usual operands (plain contiguous device tensors of
// the documented types and shapes) in one step and returns the result. For anything else, and whenever
// the library returns a status other than Q4_OK, it returns None without having launched anything, and
// the Python wrapper runs its own checks and raises its own error. Nothing is kept between calls.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>

#include "q4llm.h"

namespace {

using at::Tensor;

// A plain strided device tensor that the library may read through its address.
bool plain(const Tensor& t) {
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.is_neg() && !t.is_conj() &&
         !at::isTensorSubclassLike(t);
}
bool plain_as(const Tensor& t, at::ScalarType dt) { return plain(t) && t.scalar_type() == dt && t.is_contiguous(); }
bool same_device(const Tensor& a, const Tensor& b) { return a.get_device() == b.get_device(); }

// A tensor argument: false when it is neither a tensor nor (if `optional`) None.
bool arg(PyObject* o, Tensor* t, bool optional = false) {
  if (optional && o == Py_None) return true;
  if (!THPVariable_Check(o)) return false;
  *t = THPVariable_Unpack(o);
  return t->defined();
}

bool arg(PyObject* o, int64_t* v) {
  if (!PyLong_Check(o)) return false;
  *v = PyLong_AsLongLong(o);
  if (*v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// An int4 weight pair [N, K/8] int32, [N, K/group] fp16 on one device.
bool weights(const Tensor& qw, const Tensor& sc, int64_t group, int64_t* n, int64_t* k) {
  if (group <= 0 || group > INT32_MAX || !plain_as(qw, at::kInt) || !plain_as(sc, at::kHalf) || qw.dim() != 2 ||
      sc.dim() != 2 || !same_device(qw, sc))
    return false;
  *n = qw.size(0);
  *k = qw.size(1) * 8;
  return *n > 0 && *k > 0 && *k % group == 0 && sc.size(0) == *n && sc.size(1) == *k / group;
}

template <typename T>
T* data(const Tensor& t) {
  return t.defined() ? static_cast<T*>(t.data_ptr()) : nullptr;
}

// Runs `f` without the interpreter lock, as ctypes does.
template <typename F>
int unlocked(F f) {
  PyThreadState* s = PyEval_SaveThread();
  const int st = f();
  PyEval_RestoreThread(s);
  return st;
}

// Every entry: a C++ exception (an allocation that fails, say) means "not here".
template <typename F>
PyObject* guarded(F f) {
  try {
    return f();
  } catch (...) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// gemv(qweight, scales, x, group, out dtype code or -1, residual, out): y [N]
PyObject* gemv(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    Tensor qw, sc, x, res, out;
    int64_t group, code, n, k;
    if (nargs != 7 || !arg(a[0], &qw) || !arg(a[1], &sc) || !arg(a[2], &x) || !arg(a[3], &group) || !arg(a[4], &code) ||
        !arg(a[5], &res, true) || !arg(a[6], &out, true) || !weights(qw, sc, group, &n, &k))
      Py_RETURN_NONE;
    const bool f16x = x.scalar_type() == at::kHalf;
    if (!plain_as(x, f16x ? at::kHalf : at::kFloat) || x.numel() != k || !same_device(x, qw)) Py_RETURN_NONE;
    if (res.defined() && (!plain_as(res, at::kFloat) || res.dim() != 1 || res.size(0) != n || !same_device(res, qw)))
      Py_RETURN_NONE;
    if (out.defined()) {
      const bool f16 = out.scalar_type() == at::kHalf;
      if (!plain_as(out, f16 ? at::kHalf : at::kFloat) || out.dim() != 1 || out.size(0) != n || !same_device(out, qw) ||
          (f16 && res.defined()))
        Py_RETURN_NONE;
      code = f16 ? Q4_F16 : Q4_F32;
    } else {
      if ((code != Q4_F16 && code != Q4_F32) || (code == Q4_F16 && res.defined())) Py_RETURN_NONE;
      out = at::empty({n}, x.options().dtype(code == Q4_F16 ? at::kHalf : at::kFloat));
    }
    void* st = stream_of(x);
    const int rc = unlocked([&] {
      return q4_gemv(data<int32_t>(qw), data<uint16_t>(sc), x.data_ptr(), f16x ? Q4_F16 : Q4_F32, out.data_ptr(),
                     static_cast<int>(code), data<float>(res), n, k, static_cast<int>(group), st);
    });
    if (rc != Q4_OK) Py_RETURN_NONE;
    return a[6] != Py_None ? (Py_INCREF(a[6]), a[6]) : THPVariable_Wrap(out);
  });
}

// y [M, N] = residual + x [M, K] W^T; M == 1 with `gemv_row` set: the decode GEMV
PyObject* linear_impl(const Tensor& qw, const Tensor& sc, const Tensor& x, int64_t group, const Tensor& res,
                      bool gemv_row) {
  int64_t n, k;
  if (!weights(qw, sc, group, &n, &k) || !plain_as(x, at::kFloat) || x.dim() != 2 || x.size(1) != k || x.size(0) < 1 ||
      !same_device(x, qw))
    Py_RETURN_NONE;
  const int64_t m = x.size(0);
  if (res.defined() && (!plain_as(res, at::kFloat) || !same_device(res, qw) || res.dim() != 2 || res.size(0) != m ||
                        res.size(1) != n))
    Py_RETURN_NONE;
  const bool one = m == 1 && gemv_row;
  // the sizes q4_linear's tiled path takes through a workspace (ops._linear_workspace)
  const bool ws_path = !one && m > 16 && k % 64 == 0 && group % 32 == 0 && (group & (group - 1)) == 0 &&
                       m * k < (int64_t{1} << 29);
  Tensor out = at::empty({m, n}, x.options()), ws;
  size_t ws_bytes = 0;
  if (ws_path) {
    if (q4_linear_ws_split_bytes(m, n, k, static_cast<int>(group), &ws_bytes) != Q4_OK) Py_RETURN_NONE;
    ws = at::empty({static_cast<int64_t>(ws_bytes)}, x.options().dtype(at::kByte));
  }
  void* st = stream_of(x);
  const int rc = unlocked([&] {
    const int g = static_cast<int>(group);
    if (one)
      return q4_gemv(data<int32_t>(qw), data<uint16_t>(sc), x.data_ptr(), Q4_F32, out.data_ptr(), Q4_F32,
                     data<float>(res), n, k, g, st);
    if (ws_path)
      return q4_linear_ws(data<float>(x), m, data<int32_t>(qw), data<uint16_t>(sc), data<float>(out), data<float>(res),
                          n, k, g, ws.data_ptr(), ws_bytes, st);
    return q4_linear(data<float>(x), m, data<int32_t>(qw), data<uint16_t>(sc), data<float>(out), data<float>(res), n, k,
                     g, st);
  });
  if (rc != Q4_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(out);
}

// linear(qweight, scales, x, group, residual, decode row as GEMV: bool)
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    Tensor qw, sc, x, res;
    int64_t group;
    if (nargs != 6 || !arg(a[0], &qw) || !arg(a[1], &sc) || !arg(a[2], &x) || !arg(a[3], &group) ||
        !arg(a[4], &res, true))
      Py_RETURN_NONE;
    return linear_impl(qw, sc, x, group, res, a[5] == Py_True);
  });
}

// attn_bucket(q, k_cache, v_cache, L, start, scale, workspace): out [C, n_q * hd]
PyObject* attn(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    Tensor q, kc, vc, start, ws;
    int64_t L;
    if (nargs != 7 || !arg(a[0], &q) || !arg(a[1], &kc) || !arg(a[2], &vc) || !arg(a[3], &L) || !arg(a[4], &start) ||
        !PyFloat_Check(a[5]) || !arg(a[6], &ws, true))
      Py_RETURN_NONE;
    if (!plain(q) || q.scalar_type() != at::kFloat || q.dim() != 3 || q.stride(2) != 1 || q.stride(1) != q.size(2) ||
        !plain_as(kc, at::kHalf) || !plain_as(vc, at::kHalf) || kc.dim() != 3 || !plain_as(start, at::kInt) ||
        start.numel() < 1 || !same_device(kc, q) || !same_device(vc, q) || !same_device(start, q))
      Py_RETURN_NONE;
    const int64_t c = q.size(0), nq = q.size(1), hd = q.size(2), nkv = kc.size(1);
    if (c > INT32_MAX || nq > INT32_MAX || L > INT32_MAX || L < INT32_MIN || q.stride(0) > INT32_MAX || c < 1)
      Py_RETURN_NONE;
    if (ws.defined()) {
      if (!plain_as(ws, at::kByte) || !same_device(ws, q)) Py_RETURN_NONE;
    } else {
      size_t b = 0;
      if (attn_workspace_bytes(c, nq, nkv, hd, L, &b) != Q4_OK) Py_RETURN_NONE;
      ws = at::empty({static_cast<int64_t>(b > 0 ? b : 1)}, q.options().dtype(at::kByte));
    }
    Tensor out = at::empty({c, nq * hd}, q.options());
    void* st = stream_of(q);
    const float scale = static_cast<float>(PyFloat_AS_DOUBLE(a[5]));
    const int rc = unlocked([&] {
      return attn_bucket(data<float>(q), static_cast<int>(q.stride(0)), data<uint16_t>(kc), data<uint16_t>(vc),
                         data<float>(out), c, nq, nkv, hd, L, data<int32_t>(start), scale, ws.data_ptr(), ws.numel(), st);
    });
    if (rc != Q4_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(out);
  });
}

// gemm(a, b, workspace): C [M, N] fp16 (gemm_f16_nt_ws with a workspace, gemm_f16_nt with None)
PyObject* gemm(PyObject*, PyObject* const* o, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    Tensor a, b, ws;
    if (nargs != 3 || !arg(o[0], &a) || !arg(o[1], &b) || !arg(o[2], &ws, true) || !plain(a) || !plain(b) ||
        a.scalar_type() != at::kHalf || b.scalar_type() != at::kHalf || a.dim() != 2 || b.dim() != 2 ||
        a.stride(1) != 1 || b.stride(1) != 1 || a.size(1) != b.size(1) || !same_device(a, b))
      Py_RETURN_NONE;
    if (ws.defined() && (!plain_as(ws, at::kByte) || !same_device(ws, a))) Py_RETURN_NONE;
    const int64_t m = a.size(0), n = b.size(0), k = a.size(1);
    if (m < 1 || n < 1 || k < 1) Py_RETURN_NONE;
    Tensor c = at::empty({m, n}, a.options());
    void* st = stream_of(a);
    const int rc = unlocked([&] {
      if (ws.defined())
        return gemm_f16_nt_ws(data<uint16_t>(a), data<uint16_t>(b), data<uint16_t>(c), m, n, k, a.stride(0), b.stride(0),
                              n, ws.data_ptr(), ws.numel(), st);
      return gemm_f16_nt(data<uint16_t>(a), data<uint16_t>(b), data<uint16_t>(c), m, n, k, a.stride(0), b.stride(0), n,
                         st);
    });
    if (rc != Q4_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(c);
  });
}

PyMethodDef kMethods[] = {
    {"gemv", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(gemv)), METH_FASTCALL, nullptr},
    {"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(linear)), METH_FASTCALL, nullptr},
    {"attn", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(attn)), METH_FASTCALL, nullptr},
    {"gemm", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(gemm)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_q4torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__q4torch() { return PyModule_Create(&kModule); }
