// Host side of the calls that a decode step makes most, in one native function each: checks, allocation, stream and launch.
//
// One token through a small linear is bound by the host: its two kernels take 2.3 and 5.3 us, the Python of the two calls (shape
// and type checks, two or three tensor constructions, six data_ptr() and stride() calls each, the marshalling of 21 arguments)
// took 9.8 us a call, of which the launch itself is 2.5.
//
// Each function serves the plain case -- torch.Tensor or Parameter, matrices, unit column strides, one GPU that is the current one, no tensor
// subclass, no functorch level, no Python key -- and returns None for anything else and for whatever is wrong: the Python code of the
// operator then does what it does, error messages included.  No error is raised here but those of the allocation and of the
// launch.
//
// Links torch's libraries, nothing of libflaggems_amd.so: the addresses of the C functions come in from Python.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <ATen/ops/empty.h>
#include <c10/core/impl/VirtualGuardImpl.h>

#include <algorithm>
#include <cstdint>

namespace {

using at::ScalarType;
using at::Tensor;

typedef int (*block_gemm_fn)(const void*, int64_t, const void*, int64_t, const float*, int64_t, int64_t, const float*, int64_t, int64_t, void*,
                             int64_t, int, int64_t, int64_t, int64_t, int64_t, int64_t, void*, size_t, void*);
typedef size_t (*workspace_fn)(int64_t, int64_t, int64_t);
typedef int (*group_quant_fn)(const void*, int, int64_t, int64_t, int64_t, void*, int, int64_t, float*, int64_t, int64_t, int64_t, float, float,
                              float, float, int, int, int, void*);

block_gemm_fn gemm_any = nullptr, gemm_pow2 = nullptr;
workspace_fn gemm_workspace = nullptr;
group_quant_fn group_quant_call = nullptr;
PyObject* get_workspace = nullptr;  // _lib.workspace(device, bytes, stream)
PyObject* check_status = nullptr;   // _lib.check(status, what)
PyObject* raw_stream = nullptr;     // device index -> address of torch's current stream

// A tensor whose memory is what its sizes and strides say, on a GPU: nothing wraps it or waits to be applied to it.
bool plain(const Tensor& t) {
  constexpr c10::DispatchKeySet usual({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView,
                                       c10::DispatchKey::AutocastCUDA});
  return t.defined() && t.layout() == at::kStrided && (t.key_set().raw_repr() & ~usual.raw_repr()) == 0 && t.is_cuda();
}
const Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  return plain(t) ? &t : nullptr;
}

int type_code(ScalarType t) {  // FG_BF16, FG_F16, FG_F32
  return t == ScalarType::BFloat16 ? 0 : t == ScalarType::Half ? 1 : t == ScalarType::Float ? 2 : -1;
}

bool is_128(PyObject* o) {
  int beyond = 0;  // (a number that fits no long is no error here: the Python code refuses it)
  return PyLong_CheckExact(o) && PyLong_AsLongAndOverflow(o, &beyond) == 128;
}

// The workspace a problem asks for depends on its sizes and on the current device's compute units alone; the last ones asked are
// remembered (under the GIL).
size_t workspace_bytes(int64_t m, int64_t n, int64_t k, int device) {
  static struct { int64_t m, n, k; int device; size_t bytes; } seen[64] = {};
  auto& e = seen[(uint64_t)(m * 31 + n * 7 + (k >> 7)) % 64];
  if (e.m != m || e.n != n || e.k != k || e.device != device) {
    e.bytes = gemm_workspace(m, n, k);
    e.m = m; e.n = n; e.k = k;
    e.device = device;
  }
  return e.bytes;
}

// Whether `device` is the current one; torch's current stream there then (null with a Python error set: the stream could not be asked).
bool current_stream(const c10::Device& device, THPObjectPtr& stream) {
  const c10::impl::VirtualGuardImpl guard(c10::DeviceType::CUDA);
  if (guard.getDevice() != device) return false;
  THPObjectPtr index(PyLong_FromLong(device.index()));
  stream = index ? PyObject_CallFunctionObjArgs(raw_stream, index.get(), nullptr) : nullptr;
  return true;
}

// block_matmul(A, B, As, Bs, block_n, block_k, output_dtype, powers_of_two) -> C or None
PyObject* block_matmul(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 8 || gemm_any == nullptr || !is_128(args[4]) || !is_128(args[5]) || !THPDtype_Check(args[6])) Py_RETURN_NONE;
  const Tensor *a = plain(args[0]), *b = plain(args[1]), *as = plain(args[2]), *bs = plain(args[3]);
  if (!a || !b || !as || !bs || a->dim() != 2 || b->dim() != 2 || as->dim() != 2 || bs->dim() != 2) Py_RETURN_NONE;
  const ScalarType out = reinterpret_cast<THPDtype*>(args[6])->scalar_type;
  const int code = type_code(out);
  const int64_t m = a->size(0), k = a->size(1), n = b->size(0), kb = (k + 127) / 128;
  if (code < 0 || m < 1 || n < 1 || k < 1 || b->size(1) != k || !a->is_contiguous() || b->stride(1) != 1) Py_RETURN_NONE;
  if (a->scalar_type() != ScalarType::Float8_e4m3fn || b->scalar_type() != ScalarType::Float8_e4m3fn || as->scalar_type() != ScalarType::Float ||
      bs->scalar_type() != ScalarType::Float)
    Py_RETURN_NONE;
  if (as->size(0) != m || as->size(1) != kb || bs->size(0) != (n + 127) / 128 || bs->size(1) != kb) Py_RETURN_NONE;
  const c10::Device device = a->device();
  THPObjectPtr stream;
  if (b->device() != device || as->device() != device || bs->device() != device || !current_stream(device, stream)) Py_RETURN_NONE;
  if (!stream) return nullptr;
  const int pow2 = PyObject_IsTrue(args[7]);
  if (pow2 < 0) return nullptr;
  Tensor c = at::empty({m, n}, a->options().dtype(out));
  if (!plain(c)) Py_RETURN_NONE;  // (a mode that makes other tensors)
  const size_t bytes = workspace_bytes(m, n, k, device.index());
  void* ws = nullptr;
  size_t ws_len = 0;
  THPObjectPtr ws_tensor;
  if (bytes) {
    THPObjectPtr dev(THPDevice_New(device));
    THPObjectPtr size(PyLong_FromSize_t(bytes));
    if (!dev || !size) return nullptr;
    ws_tensor = PyObject_CallFunctionObjArgs(get_workspace, dev.get(), size.get(), stream.get(), nullptr);
    if (!ws_tensor) return nullptr;
    const Tensor& w = THPVariable_Unpack(ws_tensor.get());
    ws = w.data_ptr();
    ws_len = (size_t)w.numel();
  }
  const int64_t lda = m > 1 ? a->stride(0) : std::max(k, a->stride(0)), ldb = n > 1 ? b->stride(0) : std::max(k, b->stride(0));
  const int status = (pow2 ? gemm_pow2 : gemm_any)(a->data_ptr(), lda, b->data_ptr(), ldb, static_cast<const float*>(as->data_ptr()), as->stride(0),
                                                   as->stride(1), static_cast<const float*>(bs->data_ptr()), bs->stride(0), bs->stride(1),
                                                   c.data_ptr(), n, code, m, n, k, 128, 128, ws, ws_len, PyLong_AsVoidPtr(stream.get()));
  if (status != 0) {
    THPObjectPtr r(PyObject_CallFunction(check_status, "is", status, "fg_block_fp8_gemm"));
    if (!r) return nullptr;
  }
  return THPVariable_Wrap(std::move(c));
  END_HANDLE_TH_ERRORS
}

// group_quant(x, group_size, column_major_scales, floor, scale_rule, quotient_rule, pow2_rule) -> (codes, scales) or None
PyObject* group_quant(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 7 || group_quant_call == nullptr || !PyLong_CheckExact(args[1])) Py_RETURN_NONE;
  const Tensor* x = plain(args[0]);
  if (!x || x->dim() != 2) Py_RETURN_NONE;
  const int code = type_code(x->scalar_type());
  const int64_t rows = x->size(0), cols = x->size(1), group = PyLong_AsLongLong(args[1]);
  if (group < 1) { PyErr_Clear(); Py_RETURN_NONE; }
  if (code < 0 || rows < 1 || cols < 1 || cols % group != 0 || x->stride(1) != 1) Py_RETURN_NONE;
  const int columns = PyObject_IsTrue(args[2]);
  const double floor_value = PyFloat_AsDouble(args[3]);
  const long scale_rule = PyLong_AsLong(args[4]), quotient_rule = PyLong_AsLong(args[5]), pow2_rule = PyLong_AsLong(args[6]);
  if (columns < 0 || PyErr_Occurred()) return nullptr;
  const c10::Device device = x->device();
  THPObjectPtr stream;
  if (!current_stream(device, stream)) Py_RETURN_NONE;
  if (!stream) return nullptr;
  const int64_t groups = cols / group;
  Tensor q = at::empty({rows, cols}, x->options().dtype(ScalarType::Float8_e4m3fn));
  Tensor s = columns ? at::empty({groups, rows}, x->options().dtype(ScalarType::Float)).t() : at::empty({rows, groups}, x->options().dtype(ScalarType::Float));
  if (!plain(q) || !plain(s)) Py_RETURN_NONE;  // (a mode that makes other tensors)
  const int64_t x_rs = rows > 1 ? x->stride(0) : std::max(cols, x->stride(0));
  const int status = group_quant_call(x->data_ptr(), code, rows, cols, x_rs, q.data_ptr(), 3 /* FG_FP8_E4M3FN */, cols,
                                      static_cast<float*>(s.data_ptr()), s.stride(0), s.stride(1), group, (float)floor_value, -448.f, 448.f,
                                      (float)(1.0 / 448.0), (int)scale_rule, (int)quotient_rule, (int)pow2_rule, PyLong_AsVoidPtr(stream.get()));
  if (status != 0) {
    THPObjectPtr r(PyObject_CallFunction(check_status, "is", status, "fg_group_quant_fp8"));
    if (!r) return nullptr;
  }
  THPObjectPtr pq(THPVariable_Wrap(std::move(q))), ps(THPVariable_Wrap(std::move(s)));
  if (!pq || !ps) return nullptr;
  return PyTuple_Pack(2, pq.get(), ps.get());
  END_HANDLE_TH_ERRORS
}

// connect(block gemm, block gemm with power-of-two scales, its workspace size, group quantizer: addresses; workspace, check, raw stream: callables)
PyObject* connect(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 7) {
    PyErr_SetString(PyExc_TypeError, "connect: seven arguments");
    return nullptr;
  }
  void* p[4];
  for (int i = 0; i < 4; ++i) {
    p[i] = PyLong_AsVoidPtr(args[i]);
    if (PyErr_Occurred()) return nullptr;
  }
  PyObject** const held[3] = {&get_workspace, &check_status, &raw_stream};
  for (int i = 0; i < 3; ++i) {
    Py_INCREF(args[4 + i]);
    PyObject* const before = *held[i];
    *held[i] = args[4 + i];
    Py_XDECREF(before);
  }
  gemm_any = reinterpret_cast<block_gemm_fn>(p[0]);
  gemm_pow2 = reinterpret_cast<block_gemm_fn>(p[1]);
  gemm_workspace = reinterpret_cast<workspace_fn>(p[2]);
  group_quant_call = reinterpret_cast<group_quant_fn>(p[3]);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"block_matmul", (PyCFunction)(void (*)(void))block_matmul, METH_FASTCALL,
     "block_matmul(A, B, As, Bs, block_n, block_k, output_dtype, powers_of_two) -> C, or None where the general path has to look"},
    {"group_quant", (PyCFunction)(void (*)(void))group_quant, METH_FASTCALL,
     "group_quant(x, group_size, column_major_scales, floor, scale_rule, quotient_rule, pow2_rule) -> (codes, scales) or None"},
    {"connect", (PyCFunction)(void (*)(void))connect, METH_FASTCALL, "connect(four addresses, workspace, check, raw stream)"},
    {nullptr, nullptr, 0, nullptr}};

struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fg_hostcalls", "native host side of the decode-critical flaggems_amd calls", -1, methods,
                             nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fg_hostcalls(void) { return PyModule_Create(&module); }
