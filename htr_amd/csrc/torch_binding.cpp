// htr_amd._fast: the host side of a packed linear and of a routed-expert layer on torch tensors, in C++.
//
// A decode launch takes the GPU 6 microseconds and took the interpreter 16 (a dozen attribute reads, shape checks, two
// dictionary look-ups, a 19-argument foreign call), so small calls ran at the interpreter's pace; collecting the 512
// tensors of a 64-expert layer took it half a millisecond.  Here the same checks read the tensors' fields directly.  Every
// function returns None where something is not as expected: the caller's Python path then handles the call, or says
// what is wrong with it.  Only torch's C++ interface is used; the kernels stay behind the C ABI of libhtr_gfx950.so, whose
// entry points bind() takes as addresses.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <chrono>
#include <cstdint>
#include <cstring>
#include <vector>
#include "../../include/htr_gfx950.h"

namespace {

// the library's entry points, with the types that its header declares
decltype(&htr_linear) f_linear = nullptr;
decltype(&htr_stream_capture_id) f_capture = nullptr;
decltype(&htr_moe_scratch_bytes) f_moe_bytes = nullptr;
decltype(&htr_moe_experts) f_moe = nullptr;
decltype(&htr_linear_route) f_route = nullptr;
decltype(&htr_dequant_w) f_dequant = nullptr;

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return 0;
    case at::kHalf: return 1;
    case at::kFloat: return 2;
    default: return -1;
  }
}

struct Owned {      // one reference, given back at the end of the scope
  PyObject* p;
  ~Owned() { Py_XDECREF(p); }
};

const at::Tensor* tensor_of(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// Memory of its own (not the wrapper of a function transform such as torch.func.grad)
bool raw_ok(const at::Tensor& t) { return t.has_storage(); }
// Whether torch follows derivatives through t now, backward or forward
bool differentiable(const at::Tensor& t) { return (c10::GradMode::is_enabled() && t.requires_grad()) || t._fw_grad(0).defined(); }

struct Shape { int64_t m = 0, n = 0, K = 0; };

// One HTR-W1 tensor set (qweight int32 [m/16, n/16, 8K], scales float16 [m], su uint8 [n/8], sv uint8 [m/8], all contiguous on
// device `dev`): its shape, or false.
bool weight_ok(const at::Tensor& qw, const at::Tensor& sc, const at::Tensor& su, const at::Tensor& sv, c10::Device dev, Shape& s) {
  if (qw.dim() != 3 || qw.scalar_type() != at::kInt || sc.scalar_type() != at::kHalf || su.scalar_type() != at::kByte || sv.scalar_type() != at::kByte)
    return false;
  const int64_t W = qw.size(2);
  s.m = qw.size(0) * 16; s.n = qw.size(1) * 16; s.K = W / 8;
  if (W % 8 || s.K < 2 || s.K > 8 || s.m % 128 || s.n % 128 || s.m == 0 || s.n == 0) return false;
  if (sc.numel() != s.m || su.numel() * 8 != s.n || sv.numel() * 8 != s.m) return false;
  for (const at::Tensor* t : {&qw, &sc, &su, &sv})
    if (t->device() != dev || !t->is_contiguous()) return false;
  return true;
}

// linear(x, qweight, scales, su, sv, bias, workspace address, its bytes, address of its failure word (0: none), stream, rows)
// -> tensor or None; None also while the stream is being captured (a capture has workspaces of its own), after a launch
// on the workspace gave up, and for more activation rows than `rows` (128 if not given).  Beyond 128 rows the call goes where
// htr_linear_route says, as in ops._linear_impl: one launch, or the weight dequantized and multiplied by torch, for which the workspace may
// be missing (address 0).
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs < 10 || nargs > 11 || f_linear == nullptr || !THPVariable_CheckExact(args[0])) Py_RETURN_NONE;
  const at::Tensor* t[6];
  for (int i = 0; i < 6; ++i) t[i] = args[i] == Py_None ? nullptr : tensor_of(args[i]);
  for (int i = 0; i < 5; ++i) if (t[i] == nullptr) Py_RETURN_NONE;
  if (args[5] != Py_None && t[5] == nullptr) Py_RETURN_NONE;
  const at::Tensor& x = *t[0];
  Shape s;
  const int code = dtype_code(x.scalar_type());
  if (code < 0 || !x.is_cuda() || x.dim() < 1 || !x.is_contiguous() || !weight_ok(*t[1], *t[2], *t[3], *t[4], x.device(), s)) Py_RETURN_NONE;
  if (x.size(-1) != s.n) Py_RETURN_NONE;
  const int64_t M = x.numel() / s.n;
  if (t[5] != nullptr && (t[5]->scalar_type() != x.scalar_type() || t[5]->numel() != s.m || t[5]->device() != x.device() || !t[5]->is_contiguous()))
    Py_RETURN_NONE;
  void* ws = PyLong_AsVoidPtr(args[6]);
  const size_t bytes = PyLong_AsSize_t(args[7]);
  const volatile int* failed = (const volatile int*)PyLong_AsVoidPtr(args[8]);
  void* stream = PyLong_AsVoidPtr(args[9]);
  const long rows = nargs > 10 && f_route != nullptr && f_dequant != nullptr ? PyLong_AsLong(args[10]) : HTR_MAX_ROWS_PER_TILE;
  if (PyErr_Occurred()) return nullptr;
  if (M < 1 || M > rows) Py_RETURN_NONE;
  int route = 0;
  if (M > HTR_MAX_ROWS_PER_TILE) {
    // torch's product can be differentiated and transformed, a launch on raw pointers cannot: the general path tells them apart
    if (M > HTR_MAX_BATCH || !raw_ok(x) || differentiable(x) || (t[5] != nullptr && (!raw_ok(*t[5]) || differentiable(*t[5])))) Py_RETURN_NONE;
    route = f_route((int)s.m, (int)s.n, (int)s.K, (int)M, code, 1);
    if (route < HTR_ROUTE_DEQUANTIZE) Py_RETURN_NONE;
  }
  if ((failed != nullptr && *failed != 0) || f_capture(stream) != 0) Py_RETURN_NONE;
  at::Tensor y;
  int rc;
  {
    // other threads run meanwhile: a launch waits where the stream's queue is full.  The caller's frame holds the tensors.
    pybind11::gil_scoped_release no_lock;
    c10::DeviceGuard guard(x.device());
    at::DimVector shape(x.sizes().begin(), x.sizes().end());
    shape.back() = s.m;
    if (route == HTR_ROUTE_DEQUANTIZE) {
      at::Tensor w = at::empty({s.m, s.n}, x.options().dtype(at::kBFloat16));
      rc = f_dequant(t[1]->const_data_ptr(), t[2]->const_data_ptr(), t[3]->const_data_ptr(), t[4]->const_data_ptr(), w.mutable_data_ptr(),
                     (int)s.m, (int)s.n, (int)s.K, stream);
      if (rc == HTR_OK) {
        // rows and columns only: with more dimensions, and an outer one of size 1 whose stride is not the inner ones' product (a prompt cut
        // from a longer buffer), torch takes a batched product with a transposed view of the weight
        y = at::linear(x.view({M, s.n}), code == 0 ? w : w.to(x.scalar_type()),
                       t[5] == nullptr ? std::optional<at::Tensor>() : std::optional<at::Tensor>(*t[5])).view(shape);
        if (y.scalar_type() != x.scalar_type()) y = y.to(x.scalar_type());      // autocast
      }
    } else {
      y = at::empty(shape, x.options());
      rc = f_linear(t[1]->const_data_ptr(), t[2]->const_data_ptr(), t[3]->const_data_ptr(), t[4]->const_data_ptr(), x.const_data_ptr(),
                  t[5] == nullptr ? nullptr : t[5]->const_data_ptr(), y.mutable_data_ptr(), (int)s.m, (int)s.n, (int)s.K, (int)M, code, code, route,
                  ws, bytes, stream);
    }
  }
  if (rc != HTR_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// The tensor addresses of one tuple of HTR-W1 tuples into every eighth slot group of `ptrs`; false where one is not like the first.
// The tensors of an expert given as a list, which another thread may change, go to `keep`.
bool collect(PyObject* experts, int offset, c10::Device dev, Shape& shape, std::vector<const void*>& ptrs, std::vector<at::Tensor>& keep) {
  const Py_ssize_t E = PyTuple_GET_SIZE(experts);
  for (Py_ssize_t e = 0; e < E; ++e) {
    PyObject* tup = PyTuple_GET_ITEM(experts, e);
    if (!(PyTuple_Check(tup) || PyList_Check(tup)) || PySequence_Fast_GET_SIZE(tup) != 4) return false;
    const at::Tensor* t[4];
    for (int k = 0; k < 4; ++k) { t[k] = tensor_of(PySequence_Fast_GET_ITEM(tup, k)); if (t[k] == nullptr) return false; }
    Shape s;
    if (!weight_ok(*t[0], *t[1], *t[2], *t[3], dev, s)) return false;
    if (e == 0) shape = s;
    else if (s.m != shape.m || s.n != shape.n || s.K != shape.K) return false;
    for (int k = 0; k < 4; ++k) ptrs[8 * e + offset + k] = t[k]->const_data_ptr();
    if (PyList_Check(tup)) for (int k = 0; k < 4; ++k) keep.push_back(*t[k]);
  }
  return true;
}

// moe(x, ids, weights, gate_up, down, host word address (0: none), ticket, stream) -> float32 [tokens, hidden], None, or the status of
// a launch that the runtime refused
PyObject* moe(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 8 || f_moe == nullptr) Py_RETURN_NONE;
  const at::Tensor *xt = tensor_of(args[0]), *it = tensor_of(args[1]), *wt = tensor_of(args[2]);
  if (xt == nullptr || it == nullptr || wt == nullptr || !xt->is_cuda() || xt->dim() != 2 || it->dim() != 2 || wt->dim() != 2) Py_RETURN_NONE;
  const int64_t T = xt->size(0), H = xt->size(1), top = it->size(1);
  const int code = dtype_code(xt->scalar_type());
  if (code < 0 || it->size(0) != T || wt->size(0) != T || wt->size(1) != top || it->device() != xt->device() || wt->device() != xt->device()) Py_RETURN_NONE;
  if ((it->scalar_type() != at::kLong && it->scalar_type() != at::kInt) || !wt->is_floating_point()) Py_RETURN_NONE;
  // the result is differentiable in the routing weights only where torch adds it up: not behind a raw pointer
  if (!raw_ok(*xt) || !raw_ok(*it) || !raw_ok(*wt) || differentiable(*wt)) Py_RETURN_NONE;
  // plain lists and tuples only: another kind of collection may load an expert when it is asked for, and is asked for the chosen ones
  for (int i = 3; i < 5; ++i) if (!PyTuple_CheckExact(args[i]) && !PyList_CheckExact(args[i])) Py_RETURN_NONE;
  Owned gu{PySequence_Tuple(args[3])}, dn{PySequence_Tuple(args[4])};      // own references to the experts: no other thread can drop one
  if (gu.p == nullptr || dn.p == nullptr) return nullptr;
  const Py_ssize_t E = PyTuple_GET_SIZE(gu.p);
  if (E < 1 || PyTuple_GET_SIZE(dn.p) != E) Py_RETURN_NONE;
  std::vector<const void*> ptrs((size_t)E * 8);
  std::vector<at::Tensor> keep;
  Shape s1, s2;
  if (!collect(gu.p, 0, xt->device(), s1, ptrs, keep) || !collect(dn.p, 4, xt->device(), s2, ptrs, keep)) Py_RETURN_NONE;
  const int64_t F = s1.m / 2;
  if (s1.n != H || s2.m != H || s2.n != F || T < 1 || top < 1 || T > (1 << 24) || E > (1 << 20)) Py_RETURN_NONE;
  unsigned int* word = (unsigned int*)PyLong_AsVoidPtr(args[5]);
  const unsigned int ticket = (unsigned int)PyLong_AsUnsignedLong(args[6]);
  void* stream = PyLong_AsVoidPtr(args[7]);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor y;
  int rc;
  {
    pybind11::gil_scoped_release no_lock;      // as in linear()
    c10::DeviceGuard guard(xt->device());
    at::Tensor x = xt->contiguous(), ids = it->contiguous(), w = wt->to(at::kFloat).contiguous();
    if ((uintptr_t)x.const_data_ptr() & 15) x = x.clone();
    const size_t need = f_moe_bytes((int)T, (int)top, (int)E, (int)H, (int)F);
    if (need == 0) {
      rc = HTR_ERR_SHAPE;
    } else {
      at::Tensor scratch = at::empty({(int64_t)need}, x.options().dtype(at::kByte));
      y = at::empty({T, H}, x.options().dtype(at::kFloat));
      rc = f_moe(x.const_data_ptr(), code, ids.const_data_ptr(), ids.scalar_type() == at::kLong ? 1 : 0, (const float*)w.const_data_ptr(), (int)T,
                 (int)top, ptrs.data(), (int)E, (int)H, (int)F, (int)s1.K, (int)s2.K, (float*)y.mutable_data_ptr(), scratch.mutable_data_ptr(),
                 need, word, ticket, stream);
    }
  }
  if (rc == HTR_ERR_LAUNCH) return PyLong_FromLong(rc);      // part of the layer may be queued: an error, not another way to run it
  if (rc != HTR_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// wait_word(address, ticket, seconds) -> the word's low bit once its upper bits are the ticket, or None after that time
PyObject* wait_word(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 3) Py_RETURN_NONE;
  const volatile unsigned int* word = (const volatile unsigned int*)PyLong_AsVoidPtr(args[0]);
  const unsigned int ticket = (unsigned int)PyLong_AsUnsignedLong(args[1]) & 0x7FFFFFFFu;
  const double seconds = PyFloat_AsDouble(args[2]);
  if (PyErr_Occurred()) return nullptr;
  unsigned int v = 0;
  bool done = false;
  Py_BEGIN_ALLOW_THREADS
  const auto until = std::chrono::steady_clock::now() + std::chrono::duration<double>(seconds);
  for (;;) {
    for (int i = 0; i < 256 && !done; ++i) { v = *word; done = (v >> 1) == ticket; __builtin_ia32_pause(); }
    if (done || std::chrono::steady_clock::now() > until) break;
  }
  Py_END_ALLOW_THREADS
  if (!done) Py_RETURN_NONE;
  return PyLong_FromLong((long)(v & 1u));
  END_HANDLE_TH_ERRORS
}

// bind(version of the library's C ABI, version of the running torch, addresses of htr_linear, htr_stream_capture_id,
// htr_moe_scratch_bytes, htr_moe_experts and, for linear() beyond 128 rows, htr_linear_route and htr_dequant_w); ImportError where either
// version is not the one that this file was compiled with
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 6 && nargs != 8) { PyErr_SetString(PyExc_TypeError, "bind wants two versions and four or six addresses"); return nullptr; }
  const long abi = PyLong_AsLong(args[0]);
  const char* torch_version = PyUnicode_AsUTF8(args[1]);
  void* p[6] = {};
  for (int i = 0; i < nargs - 2; ++i) p[i] = PyLong_AsVoidPtr(args[2 + i]);
  if (PyErr_Occurred()) return nullptr;
  if (abi != HTR_ABI_VERSION) return PyErr_Format(PyExc_ImportError, "compiled for version %d of the library's C ABI, not %ld", HTR_ABI_VERSION, abi);
  if (strcmp(torch_version, HTR_BUILD_TORCH) != 0) return PyErr_Format(PyExc_ImportError, "compiled for torch %s, not %s", HTR_BUILD_TORCH, torch_version);
  f_linear = (decltype(f_linear))p[0]; f_capture = (decltype(f_capture))p[1];
  f_moe_bytes = (decltype(f_moe_bytes))p[2]; f_moe = (decltype(f_moe))p[3];
  f_route = (decltype(f_route))p[4]; f_dequant = (decltype(f_dequant))p[5];
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"bind", (PyCFunction)(void*)bind, METH_FASTCALL, nullptr},
                         {"linear", (PyCFunction)(void*)linear, METH_FASTCALL, nullptr},
                         {"moe", (PyCFunction)(void*)moe, METH_FASTCALL, nullptr},
                         {"wait_word", (PyCFunction)(void*)wait_word, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast(void) { return PyModule_Create(&module); }
