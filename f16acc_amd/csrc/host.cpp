// Native call path of mm and of the patched F.linear: the checks, the output
// allocation and the launch of a call that needs nothing else, in one C++
// call.  In Python the same steps (strides, layout rules, ctypes' 20 argument
// conversions) took 11 us for mm and 15.5 us for a biased F.linear, more than
// the kernels of short calls run.  Measured per pass, back to back: F.linear of
// the Qwen2.5-1.5B k/v layer (256 x 1536, biased) 15.6 -> 7.6 us on 128 rows and
// 15.5 -> 8.8 on 2048, where the kernel now sets the pace.
//
// Every function returns None for a call it does not take, and its caller then
// runs the general path in kernel.py / patch.py, which decides everything
// again: wrong arguments (it raises), tensor subclasses, batched or otherwise
// wrapped tensors, active function or dispatch modes, tracing, another current
// device, operands to be packed, plans with a workspace.  So the rules below
// only have to name calls that the general path would launch directly, with the
// same arguments.  Nothing is kept between calls.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/version.h>

#include "f16acc.h"

namespace {

decltype(&f16acc_gemm) gemm = nullptr;
decltype(&f16acc_gemm_bias) gemm_bias = nullptr;
decltype(&f16acc_workspace_size) workspace_size = nullptr;
decltype(&f16acc_tile_config) tile_config = nullptr;
decltype(&f16acc_strerror) strerror_of = nullptr;
PyObject* raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream
int64_t pack_min_macs = 0;

// A torch.Tensor or Parameter that is nothing but a strided fp16 GPU tensor.
const at::Tensor* plain_fp16(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.scalar_type() != at::kHalf || !t.is_cuda() || t.layout() != at::kStrided) return nullptr;
  static const uint64_t allowed =
      c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::HIP, c10::DispatchKey::ADInplaceOrView,
                           c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutogradHIP,
                           c10::DispatchKey::AutocastCUDA})
          .raw_repr();
  return (t.key_set().raw_repr() & ~allowed) == 0 ? &t : nullptr;
}

// Whether anything may want to see the calls the general path makes.
bool observed() {
  return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
         torch::jit::tracer::isTracing() ||
         c10::impl::tls_local_dispatch_key_set().included_.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

int64_t up8(int64_t v) { return (v + 7) / 8 * 8; }

// kernel.py's _pack_plan: whether the GEMM reads a [M, K] and b [K, N] as they are.
bool read_as_they_are(const void* a, const void* b, int64_t M, int64_t N, int64_t K, int64_t sam, int64_t sak,
                      int64_t sbk, int64_t sbn) {
  // _fast_a, _fast_b
  const int64_t fam = M > 1 ? sam : up8(K), fbk = K > 1 ? sbk : up8(N), fbn = N > 1 ? sbn : up8(K);
  const bool ok_a = K % 8 == 0 && (sak == 1 || K <= 1) && fam % 8 == 0 && fam >= K && (uintptr_t)a % 16 == 0;
  const bool ok_b = (uintptr_t)b % 16 == 0 &&
                    ((K % 8 == 0 && (fbk == 1 || K <= 1) && fbn % 8 == 0 && fbn >= K) ||
                     (N % 8 == 0 && (fbn == 1 || N <= 1) && fbk % 8 == 0 && fbk >= N));
  if (ok_a && ok_b) return true;
  const double macs = (double)M * N * K;
  if (macs < (double)pack_min_macs) return true;
  // _reg_beats_pack, and a loader that reads these operands
  if (!(0.4 * 2.0 * macs / 500e12 < 4.0 * (double)(M + N) * K / 6e12 + 5e-6)) return false;
  int family = -1;
  return tile_config(M, N, K, sam, sak, sbk, sbn, a, b, -1, nullptr, nullptr, nullptr, nullptr, nullptr, &family,
                     nullptr) == 0 &&
         family == F16ACC_FAMILY_REG;
}

// a @ b (+ bias) into a new tensor of the given sizes, or None.
PyObject* launch(const at::Tensor& a, const at::Tensor& b, const at::Tensor* bias, int64_t M, int64_t N, int64_t K,
                 int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, at::IntArrayRef sizes, bool out32, bool chunked) {
  if (M == 0 || N == 0 || K == 0) Py_RETURN_NONE;
  const c10::Device dev = a.device();
  if (b.device() != dev || (bias && bias->device() != dev) ||
      c10::impl::VirtualGuardImpl(dev.type()).getDevice() != dev)
    Py_RETURN_NONE;
  const void *pa = a.const_data_ptr(), *pb = b.const_data_ptr();
  if (!read_as_they_are(pa, pb, M, N, K, sam, sak, sbk, sbn)) Py_RETURN_NONE;
  size_t ws = 0;
  if (workspace_size(M, N, K, sam, sak, sbk, sbn, pa, pb, &ws) != 0 || ws != 0) Py_RETURN_NONE;
  PyObject* index = PyLong_FromLong(dev.index());
  if (!index) return nullptr;
  PyObject* s = PyObject_CallOneArg(raw_stream, index);
  Py_DECREF(index);
  if (!s) return nullptr;
  void* stream = PyLong_AsVoidPtr(s);
  Py_DECREF(s);
  if (!stream && PyErr_Occurred()) return nullptr;
  at::Tensor c = at::empty(sizes, a.options().dtype(out32 ? at::kFloat : at::kHalf).requires_grad(false));
  const int out = out32 ? F16ACC_OUT_F32 : F16ACC_OUT_F16;
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  if (bias)
    rc = gemm_bias(pa, pb, bias->const_data_ptr(), c.mutable_data_ptr(), nullptr, M, N, K, sam, sak, sbk, sbn, N, 1,
                   out, chunked, stream);
  else
    rc = gemm(pa, pb, c.mutable_data_ptr(), nullptr, M, N, K, sam, sak, sbk, sbn, N, 1, out, chunked, stream);
  Py_END_ALLOW_THREADS;
  if (rc != 0) {
    PyErr_SetString(PyExc_RuntimeError, strerror_of(rc));
    return nullptr;
  }
  return THPVariable_Wrap(std::move(c));
}

template <class F>
PyObject* guarded(F f) {
  try {
    return f();
  } catch (python_error& e) {
    e.restore();
  } catch (const std::exception& e) {
    // (an allocation's out-of-memory error among them: the general path raises it in its own type)
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  return nullptr;
}

// mm(a, b, bias or None, out32, chunked)
PyObject* host_mm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 5) Py_RETURN_NONE;
    const at::Tensor *a = plain_fp16(args[0]), *b = plain_fp16(args[1]);
    const at::Tensor* bias = args[2] == Py_None ? nullptr : plain_fp16(args[2]);
    if (!a || !b || (args[2] != Py_None && !bias) || a->dim() != 2 || b->dim() != 2 || a->size(1) != b->size(0) ||
        observed())
      Py_RETURN_NONE;
    const int64_t M = a->size(0), K = a->size(1), N = b->size(1);
    if (bias && (bias->dim() != 1 || bias->size(0) != N || !bias->is_contiguous())) Py_RETURN_NONE;
    return launch(*a, *b, bias, M, N, K, a->stride(0), a->stride(1), b->stride(0), b->stride(1), {M, N},
                  args[3] == Py_True, args[4] == Py_True);
  });
}

// linear(x, w, bias or None, min_rows): x @ w.T (+ bias) under no_grad.
PyObject* host_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 4 || c10::GradMode::is_enabled()) Py_RETURN_NONE;
    const at::Tensor *x = plain_fp16(args[0]), *w = plain_fp16(args[1]);
    const at::Tensor* bias = args[2] == Py_None ? nullptr : plain_fp16(args[2]);
    if (!x || !w || (args[2] != Py_None && !bias) || x->dim() < 1 || w->dim() != 2) Py_RETURN_NONE;
    const int64_t K = x->size(-1), N = w->size(0);
    if (w->size(1) != K || K == 0 || observed()) Py_RETURN_NONE;
    const int64_t rows = x->numel() / K;
    const long long min_rows = PyLong_AsLongLong(args[3]);
    if (min_rows == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    if (rows < min_rows) Py_RETURN_NONE;
    // x as [rows, K]: as it is, or contiguous (a view then, as reshape makes it)
    const bool two = x->dim() == 2;
    if (!two && !x->is_contiguous()) Py_RETURN_NONE;
    if (bias && (bias->dim() != 1 || bias->size(0) != N || !bias->is_contiguous())) Py_RETURN_NONE;
    c10::SmallVector<int64_t, 6> sizes(x->sizes().begin(), x->sizes().end());
    sizes.back() = N;
    return launch(*x, *w, bias, rows, N, K, two ? x->stride(0) : K, two ? x->stride(1) : 1, w->stride(1),
                  w->stride(0), sizes, false, true);
  });
}

// setup(raw_stream, pack_min_macs, addresses of gemm, gemm_bias, workspace_size, tile_config, strerror)
PyObject* host_setup(PyObject*, PyObject* args) {
  PyObject* stream_fn;
  long long macs;
  Py_ssize_t g, gb, ws, tc, se;
  if (!PyArg_ParseTuple(args, "OLnnnnn", &stream_fn, &macs, &g, &gb, &ws, &tc, &se)) return nullptr;
  Py_INCREF(stream_fn);
  Py_XDECREF(raw_stream);
  raw_stream = stream_fn;
  pack_min_macs = macs;
  gemm = (decltype(gemm))g;
  gemm_bias = (decltype(gemm_bias))gb;
  workspace_size = (decltype(workspace_size))ws;
  tile_config = (decltype(tile_config))tc;
  strerror_of = (decltype(strerror_of))se;
  Py_RETURN_NONE;
}

// reads(M, N, K, sam, sak, sbk, sbn, address of a, of b): read_as_they_are, for
// its comparison with kernel.py's rules
PyObject* host_reads(PyObject*, PyObject* args) {
  long long M, N, K, sam, sak, sbk, sbn;
  Py_ssize_t a, b;
  if (!PyArg_ParseTuple(args, "LLLLLLLnn", &M, &N, &K, &sam, &sak, &sbk, &sbn, &a, &b)) return nullptr;
  return PyBool_FromLong(read_as_they_are((const void*)a, (const void*)b, M, N, K, sam, sak, sbk, sbn));
}

PyMethodDef methods[] = {
    {"mm", (PyCFunction)(void (*)(void))host_mm, METH_FASTCALL, "mm(a, b, bias, out32, chunked) -> Tensor or None"},
    {"linear", (PyCFunction)(void (*)(void))host_linear, METH_FASTCALL,
     "linear(x, w, bias, min_rows) -> Tensor or None"},
    {"reads", host_reads, METH_VARARGS, "reads(M, N, K, sam, sak, sbk, sbn, a, b) -> bool"},
    {"setup", host_setup, METH_VARARGS, "setup(raw_stream, pack_min_macs, 5 function addresses)"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "f16acc_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_f16acc_host() {
  PyObject* m = PyModule_Create(&module);
  // the module uses torch's C++ types, which change between versions: _lib.py checks it
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
