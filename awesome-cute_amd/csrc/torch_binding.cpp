// The calls of marlin.py and streamk.py on tensors, in C++: checks, sizes,
// pointers, the current stream, the output's allocation and the library call.
//
// Bound: host time.  A product of a few rows takes the GPU 3 to 10 us; the same
// steps in Python through ctypes took the host 5.8 us for `mul` and 12.5 us for
// a layer, so a decoder's linear layers ran at the host's pace.  Here they take
// 3.3 and 5.0 us (of which the output's allocation 1.2), the launch itself
// about 2.5: one row through the sixteen layers of four blocks of a 7B model
// 206 -> 122 us on one box, 189 -> 135 on another.
//
// Tensors are allocated and the library is entered with the interpreter lock
// released, as torch's own calls and ctypes do: a launch may wait for room in
// the stream's queue, a stream's first call allocates, and an allocation may
// wait for another thread's.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>

#include "../../include/marlin_amd.h"
#include "../../include/streamk_amd.h"

namespace {

const at::Tensor* tensor(PyObject* o, const char* name) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "%s must be a torch.Tensor", name);
    return nullptr;
  }
  return &THPVariable_Unpack(o);
}

bool to_int(PyObject* o, int* v) {
  const long x = PyLong_AsLong(o);
  if (x == -1 && PyErr_Occurred()) return false;
  if (x != (int)x) {
    PyErr_SetString(PyExc_OverflowError, "argument does not fit into a C int");
    return false;
  }
  *v = (int)x;
  return true;
}

void* current_stream(int dev) { return (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream(); }

constexpr int kMulTensors = 5;
const char* const kMulNames[kMulTensors] = {"A", "B", "C", "s", "workspace"};

bool check_mul(const at::Tensor* const* t) {
  for (int i = 0; i < kMulTensors; i++)
    if (!t[i]->is_cuda()) {
      PyErr_Format(PyExc_RuntimeError, "%s must be a GPU tensor", kMulNames[i]);
      return false;
    }
  for (int i = 0; i < kMulTensors; i++)
    if (!t[i]->is_contiguous()) {
      PyErr_Format(PyExc_RuntimeError, "%s must be contiguous", kMulNames[i]);
      return false;
    }
  return true;
}

struct Hints {
  int thread_k = -1, thread_n = -1, sms = -1, max_par = 16, cute = 1;
};

// C (m, n) = A (m, k) * dequantised B; false with an exception set
bool enqueue_mul(const at::Tensor& A, const at::Tensor& B, const at::Tensor& C, const at::Tensor& s,
                 const at::Tensor& workspace, int64_t m, int64_t n, int64_t k, const Hints& h) {
  const int dev = A.get_device();
  char err[512];
  int rc;
  void* const st = current_stream(dev);
  const void *pa = A.data_ptr(), *pb = B.data_ptr(), *ps = s.data_ptr();
  void *pc = C.data_ptr(), *pw = workspace.data_ptr();
  const int s_rows = (int)s.size(0);
  const long long ws = workspace.numel();
  Py_BEGIN_ALLOW_THREADS
  rc = marlin_mul(pa, pb, pc, ps, (int)m, (int)n, (int)k, s_rows, pw, ws, dev, st, h.thread_k,
                  h.thread_n, h.sms, h.max_par, h.cute, err, sizeof(err));
  Py_END_ALLOW_THREADS
  if (rc == 0) return true;
  if (err[0])
    PyErr_SetString(PyExc_RuntimeError, err);
  else
    PyErr_Format(PyExc_RuntimeError, "marlin_mul failed with code %d", rc);
  return false;
}

// mul(A, B, C, s, workspace, thread_k, thread_n, sms, max_par, cute_version)
PyObject* py_mul(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 10) {
    PyErr_SetString(PyExc_TypeError, "mul takes 10 arguments");
    return nullptr;
  }
  const at::Tensor* t[kMulTensors];
  for (int i = 0; i < kMulTensors; i++)
    if (!(t[i] = tensor(args[i], kMulNames[i]))) return nullptr;
  Hints h;
  if (!to_int(args[5], &h.thread_k) || !to_int(args[6], &h.thread_n) || !to_int(args[7], &h.sms) ||
      !to_int(args[8], &h.max_par))
    return nullptr;
  h.cute = PyObject_IsTrue(args[9]);
  if (h.cute < 0 || !check_mul(t)) return nullptr;
  if (!enqueue_mul(*t[0], *t[1], *t[2], *t[3], *t[4], t[0]->size(0), t[2]->size(1), t[0]->size(1), h))
    return nullptr;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// linear(A, B, s, workspace, cute_version) -> C: the last dimension of A times
// the weight, rows of any shape
PyObject* py_linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 5) {
    PyErr_SetString(PyExc_TypeError, "linear takes 5 arguments");
    return nullptr;
  }
  const at::Tensor *A = tensor(args[0], "A"), *B = tensor(args[1], "B"), *s = tensor(args[2], "s"),
                   *workspace = tensor(args[3], "workspace");
  if (!A || !B || !s || !workspace) return nullptr;
  Hints h;
  h.cute = PyObject_IsTrue(args[4]);
  if (h.cute < 0) return nullptr;
  if (A->dim() < 1 || s->dim() < 2) {
    PyErr_SetString(PyExc_IndexError, "A needs a last dimension and s two");
    return nullptr;
  }
  const int64_t n = s->size(1), k = A->size(-1);
  c10::SmallVector<int64_t, 6> shape(A->sizes().begin(), A->sizes().end());
  shape.back() = n;
  at::Tensor C, rows;
  {
    pybind11::gil_scoped_release unlocked;
    C = at::empty(shape, A->options().requires_grad(false).memory_format(c10::nullopt));
    // (a copy where the leading dimensions do not fold into one)
    if (!A->is_contiguous() || k == 0) rows = A->reshape({-1, k});
  }
  if (rows.defined()) A = &rows;
  const at::Tensor* const t[kMulTensors] = {A, B, &C, s, workspace};
  if (!check_mul(t)) return nullptr;
  if (!enqueue_mul(*A, *B, C, *s, *workspace, A->numel() / k, n, k, h)) return nullptr;
  return THPVariable_Wrap(std::move(C));
  END_HANDLE_TH_ERRORS
}

// dense(A, B, C or None) -> C (m, n) = A (m, k) * B (n, k)^T
PyObject* py_dense(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 3) {
    PyErr_SetString(PyExc_TypeError, "dense takes 3 arguments");
    return nullptr;
  }
  const at::Tensor* in[2];
  for (int i = 0; i < 2; i++) {
    const char* const name = i ? "B" : "A";
    if (!(in[i] = tensor(args[i], name))) return nullptr;
    if (in[i]->scalar_type() != at::kHalf || !in[i]->is_cuda() || !in[i]->is_contiguous() ||
        in[i]->dim() != 2) {
      PyErr_Format(PyExc_ValueError, "%s must be a contiguous 2-d torch.half tensor on the GPU", name);
      return nullptr;
    }
  }
  const at::Tensor &A = *in[0], &B = *in[1];
  const int64_t m = A.size(0), k = A.size(1), n = B.size(0);
  if (B.size(1) != k) {
    PyErr_SetString(PyExc_ValueError, "A and B must have the same k");
    return nullptr;
  }
  at::Tensor C;
  if (args[2] == Py_None) {
    pybind11::gil_scoped_release unlocked;
    C = at::empty({m, n}, A.options().requires_grad(false));
  } else {
    const at::Tensor* c = tensor(args[2], "C");
    if (!c) return nullptr;
    if (c->dim() != 2 || c->size(0) != m || c->size(1) != n || c->scalar_type() != at::kHalf ||
        !c->is_contiguous() || c->device() != A.device()) {
      PyErr_SetString(PyExc_ValueError, "C must be a contiguous (m, n) torch.half tensor on A's device");
      return nullptr;
    }
    C = *c;
  }
  const int dev = A.get_device();
  void* const st = current_stream(dev);
  const void *pa = A.data_ptr(), *pb = B.data_ptr();
  void* pc = C.data_ptr();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = streamk_gemm_tn(pa, pb, pc, (int)m, (int)n, (int)k, dev, st);
  Py_END_ALLOW_THREADS
  if (rc == STREAMK_ERR_SHAPE) {
    PyErr_Format(PyExc_ValueError,
                 "shape (m=%lld, n=%lld, k=%lld) not supported: n must be a multiple of 256, k of 64",
                 (long long)m, (long long)n, (long long)k);
    return nullptr;
  }
  if (rc != STREAMK_OK) {
    PyErr_Format(PyExc_RuntimeError, "streamk_gemm_tn: %s", streamk_amd_last_error());
    return nullptr;
  }
  if (args[2] == Py_None) return THPVariable_Wrap(std::move(C));
  Py_INCREF(args[2]);
  return args[2];
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"mul", (PyCFunction)(void (*)(void))py_mul, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void (*)(void))py_linear, METH_FASTCALL, nullptr},
    {"dense", (PyCFunction)(void (*)(void))py_dense, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_marlin_torch", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__marlin_torch(void) { return PyModule_Create(&module); }
