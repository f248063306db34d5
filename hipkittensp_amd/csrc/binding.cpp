// Python binding of the operator's hot calls (module hipkittensp_amd._native): torch tensors in, one call of the C ABI
// (include/mxfp6_gemm.h) out.
//
// What bounds small calls is host work: a decode projection of a few MB runs in 5 - 10 us on the GPU, and reading the
// metadata of five tensors from Python and marshalling twenty arguments through ctypes took 5.3 us for a GEMM, 8 us for a
// quantisation and 30 us for a linear layer (quantise + torch.library operator + GEMM, three allocations).  Here a call reads
// the tensors' fields directly and makes one C call; a linear layer is one such call (mxfp6_linear: quantiser and GEMM,
// the packed input in the stream's workspace, so the output is the only allocation).
// These functions recognise the usual call -- torch.Tensor arguments of the right types, shapes and device, contiguous, on the
// current device -- and return None for anything else: the Python code behind them (tk_kernel.py, torch_op.py) then takes the
// general cases and raises the errors of the reference's binding (include/pyutils/pyutils.cuh:15-48).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/mxfp6_gemm.h"

namespace {

constexpr int64_t kMaxDim = 0x7fffffff;

const at::Tensor* tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.has_storage() ? &t : nullptr;  // wrappers of function transforms have none
}
bool plain(const at::Tensor& t, at::ScalarType dtype, int dev) {
  return t.scalar_type() == dtype && t.is_cuda() && t.get_device() == dev && t.is_contiguous() && t.layout() == at::kStrided;
}
bool plain2d(const at::Tensor& t, at::ScalarType dtype, int dev, int64_t rows, int64_t cols) {
  return t.dim() == 2 && t.size(0) == rows && t.size(1) == cols && plain(t, dtype, dev);
}
int small_int(PyObject* o) {  // -1: not an int of the codes used here
  if (!PyLong_CheckExact(o)) return -1;
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) PyErr_Clear();
  return v >= 0 && v < 16 ? (int)v : -1;
}
int64_t scale_width(int64_t K, int layout) { return layout == MXFP6_LAYOUT_ROW ? K / 32 : (K + 511) / 512 * 16; }
bool rows_fit(int64_t rows, int64_t K, int layout) { return layout == MXFP6_LAYOUT_ROW || (rows % 32 == 0 && K % 128 == 0); }
bool known(int fmt, int layout) { return (fmt == 2 || fmt == 3) && (layout == 0 || layout == 1); }
hipStream_t stream_of(int dev) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream(); }

// The GIL released for a scope.  What may throw (data_ptr() of a tensor without memory, sizes of a nested one) is read before.
struct NoGil {
  PyThreadState* const state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

PyObject* done(int rc, const char* what) {
  if (rc) {
    PyErr_Format(PyExc_RuntimeError, "%s: %s (code %d)", what, mxfp6_strerror(rc), rc);
    return nullptr;
  }
  Py_RETURN_TRUE;
}

// An optional vector of the fused epilogue: false = not the plain case
bool vector(PyObject* o, int dev, int64_t n, bool bf16_too, const void** p, int* bf16) {
  *p = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* t = tensor(o);
  if (!t || t->dim() != 1 || t->size(0) != n) return false;
  if (plain(*t, at::kFloat, dev)) {
    *p = t->data_ptr();
    return true;
  }
  if (!bf16_too || !plain(*t, at::kBFloat16, dev)) return false;
  *p = t->data_ptr(), *bf16 = 1;
  return true;
}

// gemm(A, B, A_scale, B_scale, C, fmt_a, fmt_b, layout_a, layout_b, bias, row_scale, col_scale, act, C_scale, fmt_c)
PyObject* gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 15) Py_RETURN_NONE;
  const at::Tensor *A = tensor(a[0]), *B = tensor(a[1]), *As = tensor(a[2]), *Bs = tensor(a[3]), *C = tensor(a[4]);
  if (!A || !B || !As || !Bs || !C || A->dim() != 2 || B->dim() != 2 || C->dim() != 2 || !C->is_cuda()) Py_RETURN_NONE;
  const int fa = small_int(a[5]), fb = small_int(a[6]), la = small_int(a[7]), lb = small_int(a[8]), act = small_int(a[12]);
  if (!known(fa, la) || !known(fb, lb) || act < 0 || act > 3) Py_RETURN_NONE;
  const int dev = C->get_device();
  if (dev != c10::hip::current_device()) Py_RETURN_NONE;
  const int64_t M = A->size(0), N = B->size(0), w = A->size(1), K = w / 3 * 4;
  if (w % 24 || M > kMaxDim || N > kMaxDim || K > kMaxDim || !rows_fit(M, K, la) || !rows_fit(N, K, lb)) Py_RETURN_NONE;
  if (!plain(*A, at::kByte, dev) || !plain2d(*B, at::kByte, dev, N, w) || !plain2d(*As, at::kByte, dev, M, scale_width(K, la)) ||
      !plain2d(*Bs, at::kByte, dev, N, scale_width(K, lb)))
    Py_RETURN_NONE;
  const void *bias, *row, *col;
  int bias_bf16 = 0, none = 0;
  if (!vector(a[9], dev, N, true, &bias, &bias_bf16) || !vector(a[10], dev, M, false, &row, &none) || !vector(a[11], dev, N, false, &col, &none)) Py_RETURN_NONE;
  const void *const pa = A->data_ptr(), *const pb = B->data_ptr(), *const pas = As->data_ptr(), *const pbs = Bs->data_ptr();
  void* const pc = C->data_ptr();
  const hipStream_t s = stream_of(dev);
  int rc;
  if (a[13] != Py_None) {
    const at::Tensor* Cs = tensor(a[13]);
    const int fc = small_int(a[14]);
    if (!Cs || !known(fc, 0) || N % 32 || !plain2d(*C, at::kByte, dev, M, N / 4 * 3) || !plain2d(*Cs, at::kByte, dev, M, N / 32)) Py_RETURN_NONE;
    void* const scales = Cs->data_ptr();
    {
      NoGil released;
      rc = mxfp6_gemm_fused_fp6(pa, pb, pas, pbs, pc, scales, (int)M, (int)N, (int)K, fa, fb, la, lb, fc, bias, bias_bf16, (const float*)row, (const float*)col, act, s);
    }
    return done(rc, "dispatch_micro");
  }
  const bool f32 = C->scalar_type() == at::kFloat;
  if (!plain2d(*C, f32 ? at::kFloat : at::kBFloat16, dev, M, N)) Py_RETURN_NONE;
  {
    NoGil released;
    rc = mxfp6_gemm_fused(pa, pb, pas, pbs, pc, (int)M, (int)N, (int)K, fa, fb, la, lb, f32, bias, bias_bf16, (const float*)row, (const float*)col, act, s);
  }
  return done(rc, "dispatch_micro");
}

// quantize(X, fmt, layout) -> (packed, scales)
PyObject* quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const at::Tensor* X = n == 3 ? tensor(a[0]) : nullptr;
  if (!X || X->dim() != 2 || !X->is_cuda()) Py_RETURN_NONE;
  const int fmt = small_int(a[1]), layout = small_int(a[2]), dev = X->get_device();
  const int64_t rows = X->size(0), K = X->size(1);
  const bool bf16 = X->scalar_type() == at::kBFloat16;
  if (!known(fmt, layout) || dev != c10::hip::current_device() || !plain(*X, bf16 ? at::kBFloat16 : at::kFloat, dev) || K % 32 || rows > kMaxDim ||
      K > kMaxDim || !rows_fit(rows, K, layout))
    Py_RETURN_NONE;
  const auto opt = X->options().dtype(at::kByte).requires_grad(false);
  at::Tensor packed = at::empty({rows, K / 4 * 3}, opt), scales = at::empty({rows, scale_width(K, layout)}, opt);
  const void* const px = X->data_ptr();
  void *const pp = packed.data_ptr(), *const ps = scales.data_ptr();
  const hipStream_t s = stream_of(dev);
  int rc;
  {
    NoGil released;
    rc = bf16 ? mxfp6_quantize_bf16(px, pp, ps, (int)rows, (int)K, fmt, layout, s) : mxfp6_quantize_ex((const float*)px, pp, ps, (int)rows, (int)K, fmt, layout, s);
  }
  if (rc) return done(rc, "quantize");
  PyObject* p = THPVariable_Wrap(std::move(packed));
  PyObject* q = p ? THPVariable_Wrap(std::move(scales)) : nullptr;
  PyObject* r = q ? PyTuple_Pack(2, p, q) : nullptr;
  Py_XDECREF(p), Py_XDECREF(q);
  return r;
}

// linear(x, weight, weight_scale, bias, fmt_x, fmt_w, layout_w, act) -> y
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  // tracers and dispatch modes see the torch.library operator
  if (n != 8 || c10::impl::TorchDispatchModeTLS::any_modes_set() || torch::jit::tracer::isTracing()) Py_RETURN_NONE;
  const at::Tensor *X = tensor(a[0]), *W = tensor(a[1]), *Ws = tensor(a[2]);
  if (!X || !W || !Ws || X->dim() < 1 || W->dim() != 2 || !X->is_cuda()) Py_RETURN_NONE;
  const int fx = small_int(a[4]), fw = small_int(a[5]), lw = small_int(a[6]), act = small_int(a[7]), dev = X->get_device();
  const int64_t N = W->size(0), w = W->size(1), K = w / 3 * 4, rows = K ? X->numel() / K : 0;
  const bool bf16 = X->scalar_type() == at::kBFloat16;
  if (!known(fx, 0) || !known(fw, lw) || act < 0 || act > 3 || dev != c10::hip::current_device() || w % 24 || K == 0 || X->size(-1) != K || rows == 0 ||
      rows > kMaxDim || N > kMaxDim || K > kMaxDim || !rows_fit(N, K, lw) || !plain(*X, bf16 ? at::kBFloat16 : at::kFloat, dev) ||
      !plain(*W, at::kByte, dev) || !plain2d(*Ws, at::kByte, dev, N, scale_width(K, lw)) || ((uintptr_t)X->data_ptr() & 15))
    Py_RETURN_NONE;
  const void* bias;
  int bias_bf16 = 0;
  if (!vector(a[3], dev, N, true, &bias, &bias_bf16)) Py_RETURN_NONE;
  const auto opt = X->options().dtype(at::kBFloat16).requires_grad(false);
  at::Tensor C;
  if (X->dim() == 2) {
    C = at::empty({rows, N}, opt);
  } else {
    auto shape = X->sizes().vec();
    shape.back() = N;
    C = at::empty(shape, opt);
  }
  const void *const px = X->data_ptr(), *const pw = W->data_ptr(), *const pws = Ws->data_ptr();
  void* const pc = C.data_ptr();
  const hipStream_t s = stream_of(dev);
  int rc;
  {
    NoGil released;
    rc = mxfp6_linear(px, bf16, pw, pws, pc, (int)rows, (int)N, (int)K, fx, fw, lw, bias, bias_bf16, act, s);
  }
  // no workspace (a stream under capture, whose graph owns its activations; the allocator's refusal): the two steps with tensors of the caller's allocator
  if (rc == MXFP6_EWORKSPACE) Py_RETURN_NONE;
  if (rc) return done(rc, "linear");
  return THPVariable_Wrap(std::move(C));
}

// What throws in torch's code (a nested tensor's sizes, a tensor without memory, a HIP error, an allocation) is not the usual call:
// the Python code takes it and raises its error.  THPVariable_Wrap reports its own failures as python_error.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  try {
    return F(self, a, n);
  } catch (python_error& e) {
    e.restore();
    return nullptr;
  } catch (const std::exception&) {
    Py_RETURN_NONE;
  }
}

PyMethodDef methods[] = {{"gemm", (PyCFunction)(void (*)(void))guarded<gemm>, METH_FASTCALL, nullptr},
                         {"quantize", (PyCFunction)(void (*)(void))guarded<quantize>, METH_FASTCALL, nullptr},
                         {"linear", (PyCFunction)(void (*)(void))guarded<linear>, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
