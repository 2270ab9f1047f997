// The calls of cigemm.py that a program issues by the thousand, from tensors to the C ABI in native code.
// Every small product takes as long as the host does: 5.0 to 5.7 us a call with shapes, strides, addresses
// and the foreign call in Python, 2.8 to 3.1 here, nearly all of it the launch.
//
// Each function returns the library's status, or -1 with nothing done where an argument is not a plain
// tensor (a subclass, a traced or wrapped one): the caller then asks it in Python.  Wrong shapes and types raise
// AssertionError, as the Python code does.
#include <torch/csrc/autograd/python_variable.h>

#include "cigemm.h"

namespace {

struct Mat {
  int64_t rows, cols, ld;
  void* data;
};

bool fail(const char* what) {
  PyErr_SetString(PyExc_AssertionError, what);
  return false;
}

bool plain(PyObject* o) { return THPVariable_CheckExact(o); }

// Rows, columns, leading dimension and address of a matrix whose rows are contiguous.
bool matrix(PyObject* o, Mat* m) {
  const at::Tensor& t = THPVariable_Unpack(o);
  if (t.dim() != 2) return fail("two dimensions expected");
  m->rows = t.size(0);
  m->cols = t.size(1);
  const int64_t step = t.stride(0);
  if (m->cols > 1 && t.stride(1) != 1) return fail("rows must be contiguous");
  m->ld = m->rows > 1 ? step : std::max(std::max(m->cols, step), (int64_t)1);
  m->data = t.data_ptr();
  return true;
}

// An output with room for rows x cols elements of `bytes`: more of any of them was always taken.
bool output(PyObject* o, Mat* m, int64_t rows, int64_t cols, int64_t bytes) {
  if (!matrix(o, m)) return false;
  return (m->rows >= rows && m->cols >= cols && (int64_t)THPVariable_Unpack(o).element_size() >= bytes) ||
         fail("the output is too small");
}

// A bias or the scales: the kernels read (write) numel elements in a row.
bool dense(PyObject* o) { return THPVariable_Unpack(o).is_contiguous() || fail("contiguous vectors expected"); }

// int8, or its bits in another type
bool bytes(PyObject* o) { return THPVariable_Unpack(o).element_size() == 1 || fail("unexpected dtype"); }

bool typed(PyObject* o, at::ScalarType type) {
  return THPVariable_Unpack(o).scalar_type() == type || fail("unexpected dtype");
}

template <typename F>
F function(PyObject* address) {
  return reinterpret_cast<F>(PyLong_AsVoidPtr(address));
}
cigemmHandle_t handle(PyObject* o) { return static_cast<cigemmHandle_t>(PyLong_AsVoidPtr(o)); }

// The library call, without the interpreter's lock (a launch may wait for room in its queue), its status.
template <typename Call>
PyObject* run(Call call) {
  cigemmStatus_t st;
  Py_BEGIN_ALLOW_THREADS;
  st = call();
  Py_END_ALLOW_THREADS;
  return PyLong_FromLong(st);
}

// Nothing thrown by an accessor (a tensor without storage ...) may leave through the C entry.
template <typename Body>
PyObject* guarded(Body body) {
  try {
    return body();
  } catch (const std::exception& e) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

bool counted(Py_ssize_t n, Py_ssize_t want) {
  if (n == want) return true;
  PyErr_Format(PyExc_TypeError, "%zd arguments expected, got %zd", want, n);
  return false;
}

typedef cigemmStatus_t (*gemm_f32_fn)(cigemmHandle_t, int64_t, int64_t, int64_t, const float*, int64_t,
                                      const float*, int64_t, float*, int64_t);

// gemm(function, handle, dtype, A, B, out): the entry points of one element type (their pointers differ in
// that type only); dtype: 0 fp32, 1 fp16, 2 bf16.
PyObject* gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!counted(n, 6)) return nullptr;
  return guarded([&]() -> PyObject* {
    if (!plain(a[3]) || !plain(a[4]) || !plain(a[5])) return PyLong_FromLong(-1);
    const long code = PyLong_AsLong(a[2]);
    const at::ScalarType type = code == 0 ? at::kFloat : code == 1 ? at::kHalf : at::kBFloat16;
    Mat A, B, C;
    if (!typed(a[3], type) || !typed(a[4], type) || !matrix(a[3], &A) || !matrix(a[4], &B)) return nullptr;
    if (A.cols != B.rows) return fail("inner dimensions differ"), nullptr;
    if (!output(a[5], &C, A.rows, B.cols, code == 0 ? 4 : 2)) return nullptr;
    const auto fn = function<gemm_f32_fn>(a[0]);
    const cigemmHandle_t h = handle(a[1]);
    if (PyErr_Occurred()) return nullptr;
    return run([&] {
      return fn(h, A.rows, B.cols, A.cols, static_cast<const float*>(A.data), A.ld,
                static_cast<const float*>(B.data), B.ld, static_cast<float*>(C.data), C.ld);
    });
  });
}

// linear_f32(function, handle, X, W, bias or None, act, out)
PyObject* linear_f32(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!counted(n, 7)) return nullptr;
  return guarded([&]() -> PyObject* {
    const bool has_bias = a[4] != Py_None;
    if (!plain(a[2]) || !plain(a[3]) || (has_bias && !plain(a[4])) || !plain(a[6])) return PyLong_FromLong(-1);
    Mat X, W, C;
    if (!typed(a[2], at::kFloat) || !typed(a[3], at::kFloat) || !matrix(a[2], &X) || !matrix(a[3], &W)) return nullptr;
    if (X.cols != W.rows) return fail("inner dimensions differ"), nullptr;
    const float* bias = nullptr;
    if (has_bias) {
      const at::Tensor& b = THPVariable_Unpack(a[4]);
      if (!typed(a[4], at::kFloat) || !dense(a[4])) return nullptr;
      if (b.numel() != W.cols) return fail("one bias for each column expected"), nullptr;
      bias = static_cast<const float*>(b.data_ptr());
    }
    if (!output(a[6], &C, X.rows, W.cols, 4)) return nullptr;
    const auto fn = function<decltype(&cigemm_linear_f32)>(a[0]);
    const cigemmHandle_t h = handle(a[1]);
    const long act = PyLong_AsLong(a[5]);
    if (PyErr_Occurred()) return nullptr;
    return run([&] {
      return fn(h, X.rows, W.cols, X.cols, static_cast<const float*>(X.data), X.ld,
                static_cast<const float*>(W.data), W.ld, bias, (cigemmActivation_t)act,
                static_cast<float*>(C.data), C.ld);
    });
  });
}

// gemm_i8_i32(function, handle, A, B, layout, out)
PyObject* gemm_i8_i32(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!counted(n, 6)) return nullptr;
  return guarded([&]() -> PyObject* {
    if (!plain(a[2]) || !plain(a[3]) || !plain(a[5])) return PyLong_FromLong(-1);
    Mat A, B, C;
    if (!typed(a[2], at::kChar) || !typed(a[3], at::kChar) || !matrix(a[2], &A) || !matrix(a[3], &B)) return nullptr;
    const long layout = PyLong_AsLong(a[4]);
    const bool nk = layout == CIGEMM_B_NK;
    if (A.cols != (nk ? B.cols : B.rows)) return fail("inner dimensions differ"), nullptr;
    if (!output(a[5], &C, A.rows, nk ? B.rows : B.cols, 4)) return nullptr;
    const auto fn = function<decltype(&cigemm_gemm_i8_i32)>(a[0]);
    const cigemmHandle_t h = handle(a[1]);
    if (PyErr_Occurred()) return nullptr;
    return run([&] {
      return fn(h, A.rows, nk ? B.rows : B.cols, A.cols, static_cast<const int8_t*>(A.data), A.ld,
                static_cast<const int8_t*>(B.data), B.ld, (cigemmBLayout_t)layout, static_cast<int32_t*>(C.data),
                C.ld);
    });
  });
}

// gemm_i8_dequant(function, handle, A, B, scale_a, scale_b, layout, out type, out)
PyObject* gemm_i8_dequant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!counted(n, 9)) return nullptr;
  return guarded([&]() -> PyObject* {
    if (!plain(a[2]) || !plain(a[3]) || !plain(a[4]) || !plain(a[5]) || !plain(a[8])) return PyLong_FromLong(-1);
    Mat A, B, C;
    if (!bytes(a[2]) || !bytes(a[3]) || !matrix(a[2], &A) || !matrix(a[3], &B)) return nullptr;
    const long layout = PyLong_AsLong(a[6]), out_type = PyLong_AsLong(a[7]);
    const bool nk = layout == CIGEMM_B_NK;
    const int64_t N = nk ? B.rows : B.cols;
    if (A.cols != (nk ? B.cols : B.rows)) return fail("inner dimensions differ"), nullptr;
    if (!typed(a[4], at::kFloat) || !typed(a[5], at::kFloat) || !dense(a[4]) || !dense(a[5])) return nullptr;
    const at::Tensor &sa = THPVariable_Unpack(a[4]), &sb = THPVariable_Unpack(a[5]);
    const int64_t na = sa.numel(), nb = sb.numel();
    if ((na != 1 && na != A.rows) || (nb != 1 && nb != N))
      return fail("one scale, or one for each row of A / column of C, expected"), nullptr;
    if (!output(a[8], &C, A.rows, N, out_type == CIGEMM_OUT_BF16 ? 2 : 4)) return nullptr;
    const auto fn = function<decltype(&cigemm_gemm_i8_dequant)>(a[0]);
    const cigemmHandle_t h = handle(a[1]);
    if (PyErr_Occurred()) return nullptr;
    const float *pa = static_cast<const float*>(sa.data_ptr()), *pb = static_cast<const float*>(sb.data_ptr());
    return run([&] {
      return fn(h, A.rows, N, A.cols, static_cast<const int8_t*>(A.data), A.ld,
                static_cast<const int8_t*>(B.data), B.ld, (cigemmBLayout_t)layout, pa,
                na > 1 ? CIGEMM_SCALE_VECTOR : CIGEMM_SCALE_TENSOR, pb,
                nb > 1 ? CIGEMM_SCALE_VECTOR : CIGEMM_SCALE_TENSOR, C.data, (cigemmOutType_t)out_type, C.ld, nullptr,
                0);
    });
  });
}

// quantize_rows_i8(function, handle, x, q, scales)
PyObject* quantize_rows_i8(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!counted(n, 5)) return nullptr;
  return guarded([&]() -> PyObject* {
    if (!plain(a[2]) || !plain(a[3]) || !plain(a[4])) return PyLong_FromLong(-1);
    Mat x, q;
    if (!typed(a[2], at::kFloat) || !matrix(a[2], &x) || !typed(a[3], at::kChar) || !matrix(a[3], &q) ||
        !typed(a[4], at::kFloat) || !dense(a[4]))
      return nullptr;
    if (q.rows != x.rows || q.cols != x.cols || THPVariable_Unpack(a[4]).numel() < x.rows)
      return fail("shapes differ"), nullptr;
    const auto fn = function<decltype(&cigemm_quantize_rows_i8)>(a[0]);
    const cigemmHandle_t h = handle(a[1]);
    if (PyErr_Occurred()) return nullptr;
    float* scales = static_cast<float*>(THPVariable_Unpack(a[4]).data_ptr());
    return run([&] {
      return fn(h, x.rows, x.cols, static_cast<const float*>(x.data), x.ld, static_cast<int8_t*>(q.data), q.ld,
                scales);
    });
  });
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyMethodDef method(const char* name) {
  return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)), METH_FASTCALL, nullptr};
}

PyMethodDef methods[] = {method<gemm>("gemm"),
                         method<linear_f32>("linear_f32"),
                         method<gemm_i8_i32>("gemm_i8_i32"),
                         method<gemm_i8_dequant>("gemm_i8_dequant"),
                         method<quantize_rows_i8>("quantize_rows_i8"),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding() { return PyModule_Create(&module); }
