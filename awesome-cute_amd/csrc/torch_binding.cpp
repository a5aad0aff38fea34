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
#include <c10/core/GradMode.h>
#include <c10/core/InferenceMode.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>

#include "../../include/marlin_amd.h"
#include "../../include/marlin_amd_convert.h"
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

// What the conversion kernels may take: plain tensors on one GPU, 16-byte aligned,
// without gradients.  (That nothing looks on is the caller's to know.)
//
// Bound: host time for layers up to about 3000 x 3000; the two kernels of a
// 1024 x 1024 one take 12 us, the same checks in Python and two calls through
// ctypes took 32 for quantising and packing, here 17 (4096 x 4096: 38.8 -> 33.3).
const at::Tensor* plain(PyObject* o) {
  return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}
bool convertible(const at::Tensor& t, const at::Device& dev) {
  return t.device() == dev && !t.is_neg() && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0 &&
         !(t.requires_grad() && c10::GradMode::is_enabled());
}
// 1 launched, 0 not a problem for the kernels, -1 with an exception set
int converted(int rc) {
  if (rc == MARLIN_OK) return 1;
  if (rc == MARLIN_ERR_PROB_SHAPE) return 0;
  PyErr_Format(PyExc_RuntimeError, "weight conversion failed with code %d: %s", rc,
               marlin_amd_convert_last_error());
  return -1;
}

// quantize(w, groupsize) -> (fake, q, s), or None where the tensor operations have to do it
PyObject* py_quantize(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  int gs;
  if (nargs != 2) {
    PyErr_SetString(PyExc_TypeError, "quantize takes 2 arguments");
    return nullptr;
  }
  const at::Tensor* const pw = plain(args[0]);
  if (!to_int(args[1], &gs)) {  // what else a group size may be, the tensor operations say
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  if (!pw || pw->dim() != 2 || pw->scalar_type() != at::kHalf || !pw->is_cuda() || pw->numel() == 0)
    Py_RETURN_NONE;
  const at::Tensor& w = *pw;
  const int64_t k = w.size(0), n = w.size(1);
  if (gs == -1 && k == (int)k) gs = (int)k;
  const bool by_column = !w.is_contiguous();
  if (gs <= 0 || k % gs != 0 || k != (int)k || n != (int)n || !convertible(w, w.device()) ||
      (by_column ? !(w.stride(0) == 1 && w.stride(1) == k && gs % 4 == 0) : n % 4 != 0))
    Py_RETURN_NONE;
  const int dev = w.get_device();
  void* const st = current_stream(dev);
  at::Tensor fake, q, s;
  int rc;
  {
    pybind11::gil_scoped_release unlocked;
    const auto plain_options = w.options().requires_grad(false);
    fake = at::empty_like(w, plain_options, at::MemoryFormat::Preserve);
    q = at::empty_like(fake, plain_options.dtype(at::kInt), at::MemoryFormat::Preserve);
    s = at::empty({k / gs, n}, plain_options);
    rc = marlin_amd_quantize(w.data_ptr(), (int)k, (int)n, gs, by_column, fake.data_ptr(), q.data_ptr(),
                             s.data_ptr(), dev, st);
  }
  const int done = converted(rc);
  if (done < 0) return nullptr;
  if (done == 0) Py_RETURN_NONE;
  PyObject* const out[3] = {THPVariable_Wrap(std::move(fake)), THPVariable_Wrap(std::move(q)),
                            THPVariable_Wrap(std::move(s))};
  PyObject* const tuple = PyTuple_New(3);
  if (!tuple) return nullptr;
  for (int i = 0; i < 3; i++) PyTuple_SET_ITEM(tuple, i, out[i]);
  return tuple;
  END_HANDLE_TH_ERRORS
}

// whether `read` has no bytes between the first and the last of the contiguous `written`: a
// kernel would read what it is overwriting, the tensor operations read everything first
bool apart(const at::Tensor& written, const at::Tensor& read) {
  const char* const lo = (const char*)written.data_ptr();
  const char* const hi = lo + written.numel() * written.element_size();
  int64_t last = 0;
  for (int64_t d = 0; d < read.dim(); d++) last += (read.size(d) - 1) * read.stride(d);
  const char* const at = (const char*)read.data_ptr();
  return at >= hi || at + (last + 1) * read.element_size() <= lo;
}

// pack(w (k, n), s (groups, n), B, packed, k, n, groupsize or -1) -> whether B and the packed
// scales have been written; False where the tensor operations have to do it
PyObject* py_pack(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  int k, n, gs;
  if (nargs != 7) {
    PyErr_SetString(PyExc_TypeError, "pack takes 7 arguments");
    return nullptr;
  }
  const at::Tensor *pw = plain(args[0]), *ps = plain(args[1]), *pb = plain(args[2]), *pp = plain(args[3]);
  if (!to_int(args[4], &k) || !to_int(args[5], &n) || !to_int(args[6], &gs)) {
    PyErr_Clear();
    Py_RETURN_FALSE;
  }
  if (!pw || !ps || !pb || !pp || !pw->is_cuda() || (gs <= 0 && gs != -1)) Py_RETURN_FALSE;
  const at::Tensor &w = *pw, &s = *ps, &B = *pb, &packed = *pp;
  const auto is = [](const at::Tensor& t, at::ScalarType type, int64_t rows, int64_t columns) {
    return t.scalar_type() == type && t.dim() == 2 && t.size(0) == rows && t.size(1) == columns;
  };
  const int64_t groups = gs == -1 ? 1 : k / gs;
  const bool by_column = !w.is_contiguous();
  const at::Device on = w.device();
  if (!is(w, at::kHalf, k, n) || !is(s, at::kHalf, groups, n) || !is(packed, at::kHalf, groups, n) ||
      !is(B, at::kInt, k / 16, 2 * (int64_t)n) || (by_column && !(w.stride(0) == 1 && w.stride(1) == k)) ||
      !B.is_contiguous() || !packed.is_contiguous() || !convertible(w, on) || !convertible(B, on) ||
      !convertible(packed, on) || s.device() != on || s.requires_grad() || s.is_neg() ||
      // (writes to inference tensors elsewhere are refused by the tensor operations)
      (!c10::InferenceMode::is_enabled() && (B.is_inference() || packed.is_inference())) ||
      !apart(B, w) || !apart(B, s) || !apart(B, packed) || !apart(packed, w) || !apart(packed, s))
    Py_RETURN_FALSE;
  const int dev = w.get_device();
  void* const st = current_stream(dev);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = marlin_amd_pack(w.data_ptr(), k, n, gs, by_column, s.data_ptr(), s.stride(0), s.stride(1),
                       B.data_ptr(), packed.data_ptr(), dev, st);
  Py_END_ALLOW_THREADS
  const int done = converted(rc);
  if (done < 0) return nullptr;
  if (done == 0) Py_RETURN_FALSE;
  // written in place, as an assignment to them would be
  for (const at::Tensor* t : {&B, &packed})
    if (!t->is_inference()) t->unsafeGetTensorImpl()->bump_version();
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"mul", (PyCFunction)(void (*)(void))py_mul, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void (*)(void))py_linear, METH_FASTCALL, nullptr},
    {"quantize", (PyCFunction)(void (*)(void))py_quantize, METH_FASTCALL, nullptr},
    {"pack", (PyCFunction)(void (*)(void))py_pack, METH_FASTCALL, nullptr},
    {"dense", (PyCFunction)(void (*)(void))py_dense, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_marlin_torch", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__marlin_torch(void) { return PyModule_Create(&module); }
