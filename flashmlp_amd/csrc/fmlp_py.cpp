// _fmlp_fast: the per-call fast path of flashmlp_fwd / flashmlp_bwd (flashmlp_amd/flashmlp.py).
//
// A CPython module (METH_FASTCALL) over the C ABI of libflashmlp.so for the common case:
// inputs on one GPU, a shape with kernels of its own (views that they do not read in place are copied
// to dense tensors first). It allocates the
// outputs and the workspace with ATen on the inputs' device, launches on torch's current HIP
// stream of that device and returns the C ABI status with the outputs; for any other input it
// returns None and the Python wrapper takes its general path (which also raises the reference's
// errors). Same entry points, same results as the ctypes calls of the general path; only the
// host work per call is smaller (no ctypes argument conversion, allocations from C++).
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <c10/util/Exception.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "flashmlp.h"

namespace {

int io_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return FMLP_DTYPE_F16;
    case at::kBFloat16: return FMLP_DTYPE_BF16;
    case at::kFloat: return FMLP_DTYPE_F32;
    default: return -1;
  }
}

bool dense16(const at::Tensor& t) {
  return t.dim() == 3 && t.is_contiguous() && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0;
}

// x and dout: dense 16-byte aligned rows, heads any multiple of 16 bytes apart (0: one matrix
// expanded to every head)
bool rows16(const at::Tensor& t) {
  return t.dim() == 3 && t.stride(2) == 1 && t.stride(1) == t.size(2) &&
         (t.stride(0) * (int64_t)t.element_size()) % 16 == 0 && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0;
}

// the tensors of a call that those kernels take, as they are or (bit i of *copy) as a dense copy: one GPU,
// one dtype, strided; sets the io dtype code
bool eligible(PyObject* const* args, int n, const at::Tensor** ts, int* code, unsigned* copy) {
  for (int i = 0; i < n; ++i) {
    if (!THPVariable_Check(args[i])) return false;
    ts[i] = &THPVariable_Unpack(args[i]);
  }
  const at::Tensor& x = *ts[0];
  if (!x.is_cuda()) return false;
  const int c = io_code(x);
  if (c < 0) return false;
  *copy = 0;
  for (int i = 0; i < n; ++i) {
    const at::Tensor& t = *ts[i];
    if (t.scalar_type() != x.scalar_type() || t.device() != x.device() || t.layout() != at::kStrided || t.dim() != 3)
      return false;
    if (!dense16(t) && !((i == 0 || i == 3) && rows16(t))) {
      if (t.is_neg() || t.is_conj()) return false;  // (a lazily negated view: its copy has to apply the sign)
      *copy |= 1u << i;
    }
  }
  *code = c;
  return true;
}

// A call's inputs as the kernels take them: the caller's tensors, or dense copies held here.
struct Inputs {
  const void* p[4];
  int64_t st[4][3];
  at::Tensor held[4];
};

at::Tensor bytes_on(const at::Tensor& like, size_t n) {
  return at::empty({(int64_t)n}, like.options().dtype(at::kByte));
}

// Elements up to which a call's copies are one launch (fmlp_copy_dense); above, ATen copies each view by
// itself, which streams rows of large ones faster (bf16 padded rows, this launch / ATen: 2^20 elements 4.4 /
// 6.2 us, 2^21 4.8 / 6.1, 2^22 7.1 / 6.1, 2^24 19.3 / 13.1).
constexpr int64_t kFusedElems = (int64_t)1 << 21;

// status of the copies (FMLP_OK); throws c10::OutOfMemoryError when they do not fit
int take_inputs(const at::Tensor* const* ts, int n, unsigned copy, hipStream_t stream, Inputs* in) {
  int64_t total = 0;
  for (int i = 0; i < n; ++i) {
    const at::Tensor& t = *ts[i];
    if (copy >> i & 1u) total += t.numel();
    in->p[i] = t.data_ptr();
    for (int k = 0; k < 3; ++k) in->st[i][k] = t.stride(k);
  }
  if (copy == 0) return FMLP_OK;
  const bool fused = total <= kFusedElems;
  const int64_t es = ts[0]->element_size();
  if (fused) in->held[0] = bytes_on(*ts[0], (size_t)(total * es + 4 * 256));
  char* next = fused ? (char*)in->held[0].data_ptr() : nullptr;
  const void* src[4];
  void* dst[4];
  int64_t sizes[12], strides[12];
  int m = 0;
  for (int i = 0; i < n; ++i) {
    if (!(copy >> i & 1u)) continue;
    const at::Tensor& t = *ts[i];
    if (fused) {
      src[m] = t.data_ptr();
      dst[m] = next;
      for (int k = 0; k < 3; ++k) {
        sizes[3 * m + k] = t.size(k);
        strides[3 * m + k] = t.stride(k);
      }
      ++m;
      in->p[i] = next;
      next += (t.numel() * es + 255) / 256 * 256;
    } else {
      in->held[i] = t.is_contiguous() ? t.clone(at::MemoryFormat::Contiguous) : t.contiguous();
      in->p[i] = in->held[i].data_ptr();
    }
    in->st[i][0] = t.size(1) * t.size(2);
    in->st[i][1] = t.size(2);
    in->st[i][2] = 1;
  }
  return m ? fmlp_copy_dense(m, src, dst, sizes, strides, (int)es, stream) : FMLP_OK;
}

// a dense output of t's shape
at::Tensor empty_dense(const at::Tensor& t) {
  return t.is_contiguous() ? at::empty_like(t) : at::empty(t.sizes(), t.options());
}

PyObject* wrap_or_none(const at::Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}

// fwd(x, w1, w2, act) -> (status, o) or None
PyObject* fast_fwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 4) {
    PyErr_SetString(PyExc_TypeError, "fwd(x, w1, w2, act)");
    return nullptr;
  }
  const at::Tensor* ts[3];
  int code = 0;
  unsigned copy = 0;
  if (!eligible(args, 3, ts, &code, &copy)) Py_RETURN_NONE;
  const at::Tensor &x = *ts[0], &w1 = *ts[1];
  const int act = (int)PyLong_AsLong(args[3]);
  if (act == -1 && PyErr_Occurred()) return nullptr;
  const int64_t H = x.size(0), B = x.size(1), D = x.size(2), E = w1.size(2);
  if (!fmlp_shape_dense(D, E, code)) Py_RETURN_NONE;
  c10::DeviceGuard guard(x.device());
  const hipStream_t stream = c10::hip::getCurrentHIPStream(x.device().index()).stream();
  Inputs in;
  try {
    const int st = take_inputs(ts, 3, copy, stream, &in);
    if (st != FMLP_OK) return Py_BuildValue("(iO)", st, Py_None);
  } catch (const c10::OutOfMemoryError&) {
    if (copy == 0) throw;
    Py_RETURN_NONE;
  }
  at::Tensor o = empty_dense(x);
  size_t n = fmlp_fwd_workspace_bytes(H, B, D, E, code);
  at::Tensor ws;
  if (n) {
    try {
      ws = bytes_on(x, n);
    } catch (const c10::OutOfMemoryError&) {  // the kernels then run every tile whole
      n = 0;
    }
  }
  const int st = fmlp_fwd_strided_ws(in.p[0], in.p[1], in.p[2], o.data_ptr(), H, B, D, E, in.st[0], in.st[1], in.st[2],
                                     code, act, n ? ws.data_ptr() : nullptr, n, stream);
  return Py_BuildValue("(iN)", st, THPVariable_Wrap(o));
  END_HANDLE_TH_ERRORS
}

// bwd(x, w1, w2, do, act, flags) -> (status, dx, dw1, dw2) or None; flags: the backward's flag
// bits (FMLP_DW_HILO, FMLP_BWD_RECOMPUTE, FMLP_BWD_NO_DX, FMLP_BWD_NO_DW), the io dtype is added
PyObject* fast_bwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 6) {
    PyErr_SetString(PyExc_TypeError, "bwd(x, w1, w2, do, act, flags)");
    return nullptr;
  }
  const at::Tensor* ts[4];
  int code = 0;
  unsigned copy = 0;
  if (!eligible(args, 4, ts, &code, &copy)) Py_RETURN_NONE;
  const at::Tensor &x = *ts[0], &w1 = *ts[1], &w2 = *ts[2];
  const int act = (int)PyLong_AsLong(args[4]);
  if (act == -1 && PyErr_Occurred()) return nullptr;
  int flags = (int)PyLong_AsLong(args[5]);
  if (flags == -1 && PyErr_Occurred()) return nullptr;
  const int64_t H = x.size(0), B = x.size(1), D = x.size(2), E = w1.size(2);
  if (!fmlp_shape_dense(D, E, code)) Py_RETURN_NONE;
  flags |= code;
  const bool need_dx = (flags & FMLP_BWD_NO_DX) == 0, need_dw = (flags & FMLP_BWD_NO_DW) == 0;
  c10::DeviceGuard guard(x.device());
  const hipStream_t stream = c10::hip::getCurrentHIPStream(x.device().index()).stream();
  Inputs in;
  try {
    const int st = take_inputs(ts, 4, copy, stream, &in);
    if (st != FMLP_OK) return Py_BuildValue("(iOOO)", st, Py_None, Py_None, Py_None);
  } catch (const c10::OutOfMemoryError&) {
    if (copy == 0) throw;
    Py_RETURN_NONE;
  }
  at::Tensor dx, dw1, dw2, ws;
  if (need_dx) dx = empty_dense(x);
  if (need_dw) {
    dw1 = empty_dense(w1);
    dw2 = empty_dense(w2);
  }
  // the workspace this call's plan needs (one plan lookup, for its own activation)
  auto ws_need = [&](int f) -> size_t {
    int64_t info[9];
    if (fmlp_bwd_plan(H, B, D, E, f, act, info, 9) == FMLP_OK) return (size_t)info[8];
    return fmlp_bwd_workspace_bytes(H, B, D, E, f);
  };
  size_t n = ws_need(flags);
  if (n) {
    try {
      ws = bytes_on(x, n);
    } catch (const c10::OutOfMemoryError&) {
      // the stored-dZ form's workspace does not fit: the recompute form needs at most the fp32
      // dW partials (as the general path does)
      const bool any_ws = !fmlp_shape_tuned(D, E, code);  // such calls accept any workspace
      if ((flags & FMLP_BWD_RECOMPUTE) && !any_ws) throw;
      flags |= FMLP_BWD_RECOMPUTE;
      n = ws_need(flags);
      try {
        if (n) ws = bytes_on(x, n);
      } catch (const c10::OutOfMemoryError&) {
        if (!any_ws) throw;
        n = 0;
      }
    }
  }
  const int st = fmlp_bwd_strided(in.p[0], in.p[1], in.p[2], in.p[3], need_dx ? dx.data_ptr() : nullptr,
                                  need_dw ? dw1.data_ptr() : nullptr, need_dw ? dw2.data_ptr() : nullptr, H, B, D, E,
                                  in.st[0], in.st[1], in.st[2], in.st[3], flags, act, n ? ws.data_ptr() : nullptr, n,
                                  stream);
  return Py_BuildValue("(iNNN)", st, wrap_or_none(dx), wrap_or_none(dw1), wrap_or_none(dw2));
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"fwd", (PyCFunction)(void (*)(void))fast_fwd, METH_FASTCALL, "fwd(x, w1, w2, act) -> (status, o) or None"},
    {"bwd", (PyCFunction)(void (*)(void))fast_bwd, METH_FASTCALL,
     "bwd(x, w1, w2, do, act, flags) -> (status, dx, dw1, dw2) or None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fmlp_fast", "fast path of flashmlp_fwd / flashmlp_bwd", -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__fmlp_fast() { return PyModule_Create(&kModule); }
