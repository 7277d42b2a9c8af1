// Native host path of the Python operators (module cutile_amd._mxhost).
//
// A decode-sized product keeps the GPU busy for less than 10 us, while building five ctypes descriptors, asking torch
// for the stream and switching device contexts took about 19 us of Python per operator.  The functions here do the same
// work -- read the tensors, fill in the descriptors, allocate the results from torch's caching allocator, call the C
// ABI of libmxgemm.so -- in one or two microseconds.  They handle the ordinary calls only: anything unusual (another
// device, a dtype or layout that needs a message or the general kernel's rules) returns None before anything is
// enqueued, and ops.py then runs its own path, which validates like the reference and raises its errors.
//
// Scratch comes from the caching allocator on every call and goes back to it when the call returns: blocks are reused
// in stream order, so calls from several threads and streams, and graph captures, need no rule of their own.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/Context.h>
#include <ATen/Functions.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>

#include <vector>

#include "mxgemm.h"

namespace {

#define MX_FN(name) decltype(&name) p_##name = nullptr
struct Lib {
  MX_FN(mx_gemm);
  MX_FN(mx_gemm_add);
  MX_FN(mx_gemm_workspace_bytes);
  MX_FN(mx_packed_scale_bytes);
  MX_FN(mx_gemm_list);
  MX_FN(mx_gemm_list_workspace_bytes);
  MX_FN(mx_quantize);
  MX_FN(mx_silu_mul_quantize);
  MX_FN(mx_moe_forward);
  MX_FN(mx_moe_forward_workspace_bytes);
} lib;
#undef MX_FN
PyObject* packed_type = nullptr;   // ops.PackedScales
PyObject *s_data, *s_rows, *s_K, *s_operand, *s_layout, *s_batch;

struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// MX element format of a tensor given the caller's format argument (None or a str); -1: not for the native path
int elem_format(const at::Tensor& t, PyObject* fmt) {
  const auto dt = t.scalar_type();
  int from_dtype = -1;
  if (dt == at::kFloat8_e4m3fn) from_dtype = MX_E4M3;
  else if (dt == at::kFloat8_e5m2) from_dtype = MX_E5M2;
  else if (dt == at::kFloat4_e2m1fn_x2) from_dtype = MX_E2M1;
  if (fmt == Py_None) return from_dtype;
  if (!PyUnicode_Check(fmt)) return -1;
  int want = -1;
  if (PyUnicode_CompareWithASCIIString(fmt, "e4m3") == 0) want = MX_E4M3;
  else if (PyUnicode_CompareWithASCIIString(fmt, "e5m2") == 0) want = MX_E5M2;
  else if (PyUnicode_CompareWithASCIIString(fmt, "e2m1") == 0) want = MX_E2M1;
  return (want >= 0 && (dt == at::kByte || from_dtype == want)) ? want : -1;
}

inline bool is_e8m0(const at::Tensor& t) {
  return t.scalar_type() == at::kFloat8_e8m0fnu || t.scalar_type() == at::kByte;
}

// descriptor of a tensor of up to 4 dimensions; the extent of `packed` (an FP4 tensor's K axis) counts elements
inline mx_tensor desc(const at::Tensor& t, int dtype, int packed = -1) {
  mx_tensor d;
  d.ptr = t.data_ptr();
  d.dtype = dtype;
  d.ndim = (int32_t)t.dim();
  const auto sz = t.sizes(), st = t.strides();
  for (int i = 0; i < d.ndim; ++i) { d.shape[i] = sz[i]; d.stride[i] = st[i]; }
  if (packed >= 0) d.shape[packed] *= 2;
  d.packed_dim = packed;
  d.reserved = 0;
  return d;
}

inline bool on_current_device(const at::Tensor& t) {
  return t.is_cuda() && t.device().index() == c10::hip::current_device();
}

// a scale argument as descriptor + layout: a 2-D / 3-D / swizzled 4-D E8M0 tensor or a PackedScales made for this
// operand; false: leave it to ops.py
bool scale_desc(PyObject* o, int64_t rows, int64_t K, bool is_b, const at::Device& dev, mx_tensor* d, int32_t* layout) {
  if (THPVariable_Check(o)) {
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!is_e8m0(t) || t.device() != dev || t.dim() < 2 || t.dim() > 4) return false;
    *d = desc(t, MX_E8M0);
    *layout = t.dim() == 4 ? MX_SCALE_SWIZZLE_32_4_4 : MX_SCALE_2D;
    return true;
  }
  if ((PyObject*)Py_TYPE(o) != packed_type) return false;
  PyObject* data = PyObject_GetAttr(o, s_data);
  PyObject* prow = PyObject_GetAttr(o, s_rows);
  PyObject* pk = PyObject_GetAttr(o, s_K);
  PyObject* pop = PyObject_GetAttr(o, s_operand);
  PyObject* pl = PyObject_GetAttr(o, s_layout);
  bool ok = data && prow && pk && pop && pl && THPVariable_Check(data) && PyUnicode_Check(pop);
  if (ok) {
    const at::Tensor& t = THPVariable_Unpack(data);   // kept alive by the PackedScales object
    ok = PyLong_AsLongLong(prow) == rows && PyLong_AsLongLong(pk) == K && t.device() == dev &&
         PyUnicode_CompareWithASCIIString(pop, is_b ? "b" : "a") == 0;
    *d = mx_tensor{t.data_ptr(), MX_E8M0, 2, {rows, K / 32, 0, 0}, {K / 32, 1, 0, 0}, -1, 0};
    *layout = (int32_t)PyLong_AsLong(pl);
  }
  Py_XDECREF(data); Py_XDECREF(prow); Py_XDECREF(pk); Py_XDECREF(pop); Py_XDECREF(pl);
  if (PyErr_Occurred()) { PyErr_Clear(); return false; }
  return ok;
}

// at::empty without the dispatcher (0.47 instead of 0.72 us; a call allocates up to three tensors, a list one per problem),
// unless something has asked to see factory calls (dispatch modes, functorch) or to have new memory filled.
inline at::Tensor device_empty(at::IntArrayRef shape, at::ScalarType t, const at::Device& dev) {
  const c10::impl::LocalDispatchKeySet tls = c10::impl::tls_local_dispatch_key_set();
  if ((tls.included_ - c10::default_included_set).empty() && !at::globalContext().deterministicAlgorithms())
    return at::detail::empty_cuda(shape, t, dev, std::nullopt);
  return at::empty(shape, at::TensorOptions().dtype(t).device(dev));
}

inline void* stream_of(const at::Device& dev) { return (void*)c10::hip::getCurrentHIPStream(dev.index()).stream(); }

inline PyObject* rc_or(int rc, const at::Tensor& t) { return rc == MX_OK ? THPVariable_Wrap(t) : PyLong_FromLong(rc); }

int out_code(at::ScalarType t) { return t == at::kFloat ? MX_F32 : t == at::kBFloat16 ? MX_BF16 : -1; }

// operands of one 2-D product; false: not for the native path
struct Product {
  mx_tensor A, As, B, Bs;
  int32_t la, lb;
  int64_t M, N, K;
};
bool product(PyObject* pa, PyObject* pas, PyObject* pb, PyObject* pbs, PyObject* af, PyObject* bf, Product* p,
             at::Device* dev) {
  if (!THPVariable_Check(pa) || !THPVariable_Check(pb)) return false;
  const at::Tensor &A = THPVariable_Unpack(pa), &B = THPVariable_Unpack(pb);
  if (A.dim() != 2 || B.dim() != 2 || !on_current_device(A) || B.device() != A.device()) return false;
  const int fa = elem_format(A, af), fb = elem_format(B, bf);
  if (fa < 0 || fb < 0) return false;
  if ((fa == MX_E2M1 && A.stride(1) != 1) || (fb == MX_E2M1 && B.stride(0) != 1)) return false;
  p->A = desc(A, fa, fa == MX_E2M1 ? 1 : -1);
  p->B = desc(B, fb, fb == MX_E2M1 ? 0 : -1);
  p->M = p->A.shape[0]; p->K = p->A.shape[1]; p->N = p->B.shape[1];
  if (p->B.shape[0] != p->K) return false;
  *dev = A.device();
  return scale_desc(pas, p->M, p->K, false, *dev, &p->As, &p->la) && scale_desc(pbs, p->N, p->K, true, *dev, &p->Bs, &p->lb);
}

// gemm(A, A_scale, B, B_scale, C | None, out_dtype, a_format, b_format, accumulate, kernel, split_k)
//   -> result tensor, a negative MX_ERR_* code, or None
PyObject* py_gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 11) { PyErr_SetString(PyExc_TypeError, "gemm takes 11 arguments"); return nullptr; }
  Product p;
  at::Device dev(at::kCUDA);
  if (!product(a[0], a[1], a[2], a[3], a[6], a[7], &p, &dev)) Py_RETURN_NONE;
  const int accumulate = PyObject_IsTrue(a[8]);
  at::Tensor C;
  if (a[4] != Py_None) {
    if (!THPVariable_Check(a[4])) Py_RETURN_NONE;
    C = THPVariable_Unpack(a[4]);
    if (C.dim() != 2 || C.size(0) != p.M || C.size(1) != p.N || out_code(C.scalar_type()) < 0 || C.device() != dev)
      Py_RETURN_NONE;
  } else {
    if (accumulate || !THPDtype_Check(a[5])) Py_RETURN_NONE;
    const auto t = ((THPDtype*)a[5])->scalar_type;
    if (out_code(t) < 0) Py_RETURN_NONE;
    C = device_empty({p.M, p.N}, t, dev);
  }
  mx_tensor dC = desc(C, out_code(C.scalar_type()));
  mx_gemm_opts o = {sizeof(mx_gemm_opts), accumulate, p.la, p.lb, (int32_t)PyLong_AsLong(a[9]), 32,
                    (int32_t)PyLong_AsLong(a[10]), 0};
  if (PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
  const int64_t need = lib.p_mx_gemm_workspace_bytes(p.M, p.N, p.K, &o);
  at::Tensor ws;
  if (need > 0) ws = device_empty({need}, at::kByte, dev);
  int rc;
  {
    NoGil nogil;
    rc = lib.p_mx_gemm(&p.A, &p.As, &p.B, &p.Bs, &dC, &o, need > 0 ? ws.data_ptr() : nullptr, need, stream_of(dev));
  }
  if (rc == MX_OK && a[4] != Py_None) { Py_INCREF(a[4]); return a[4]; }
  return rc_or(rc, C);
}

// gemm_list(As, A_scales, Bs, B_scales, Cs | None, out_dtype, kernel) -> list of results, error code, or None
PyObject* py_gemm_list(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 7) { PyErr_SetString(PyExc_TypeError, "gemm_list takes 7 arguments"); return nullptr; }
  auto seq = [](PyObject* o) { return PyList_Check(o) || PyTuple_Check(o); };
  if (!seq(a[0]) || !seq(a[1]) || !seq(a[2]) || !seq(a[3]) || (a[4] != Py_None && !seq(a[4])) || !THPDtype_Check(a[5]))
    Py_RETURN_NONE;
  const Py_ssize_t cnt = PySequence_Fast_GET_SIZE(a[0]);
  for (int i = 1; i < 5; ++i)
    if (a[i] != Py_None && PySequence_Fast_GET_SIZE(a[i]) != cnt) Py_RETURN_NONE;
  const auto out_t = ((THPDtype*)a[5])->scalar_type;
  if (cnt == 0 || out_code(out_t) < 0) Py_RETURN_NONE;
  std::vector<mx_tensor> A(cnt), As(cnt), B(cnt), Bs(cnt), C(cnt);
  std::vector<at::Tensor> outs(cnt), keep;   // keep: the lists may change while the GIL is released
  keep.reserve(4 * cnt);
  at::Device dev(at::kCUDA);
  int32_t la = 0, lb = 0;
  for (Py_ssize_t i = 0; i < cnt; ++i) {
    auto item = [&](int k) { return PySequence_Fast_GET_ITEM(a[k], i); };
    Product p;
    at::Device d(at::kCUDA);
    if (!product(item(0), item(1), item(2), item(3), Py_None, Py_None, &p, &d)) Py_RETURN_NONE;
    if (i > 0 && (p.la != la || p.lb != lb || d != dev)) Py_RETURN_NONE;
    la = p.la; lb = p.lb; dev = d;
    for (int k = 0; k < 4; ++k) {
      if (THPVariable_Check(item(k))) { keep.push_back(THPVariable_Unpack(item(k))); continue; }
      PyObject* data = PyObject_GetAttr(item(k), s_data);   // PackedScales: product() has seen a tensor here
      if (!data) return nullptr;
      if (THPVariable_Check(data)) keep.push_back(THPVariable_Unpack(data));
      Py_DECREF(data);
    }
    if (a[4] != Py_None) {
      if (!THPVariable_Check(item(4))) Py_RETURN_NONE;
      outs[i] = THPVariable_Unpack(item(4));
      if (outs[i].dim() != 2 || outs[i].size(0) != p.M || outs[i].size(1) != p.N ||
          out_code(outs[i].scalar_type()) < 0 || outs[i].device() != dev)
        Py_RETURN_NONE;
    } else {
      outs[i] = device_empty({p.M, p.N}, out_t, dev);
    }
    A[i] = p.A; As[i] = p.As; B[i] = p.B; Bs[i] = p.Bs;
    C[i] = desc(outs[i], out_code(outs[i].scalar_type()));
  }
  mx_gemm_opts o = {sizeof(mx_gemm_opts), 0, la, lb, (int32_t)PyLong_AsLong(a[6]), 32, 0, 0};
  if (PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
  const int64_t need = lib.p_mx_gemm_list_workspace_bytes((int32_t)cnt, A.data(), B.data(), &o);
  at::Tensor ws;
  if (need > 0) ws = device_empty({need}, at::kByte, dev);
  int rc;
  {
    NoGil nogil;
    rc = lib.p_mx_gemm_list((int32_t)cnt, A.data(), As.data(), B.data(), Bs.data(), C.data(), &o,
                            need > 0 ? ws.data_ptr() : nullptr, need, stream_of(dev));
  }
  if (rc != MX_OK) return PyLong_FromLong(rc);
  PyObject* res = PyList_New(cnt);
  if (!res) return nullptr;
  for (Py_ssize_t i = 0; i < cnt; ++i) {
    PyList_SET_ITEM(res, i, THPVariable_Wrap(outs[i]));   // (a tensor of Cs is the same Python object again)
  }
  return res;
}

// mma(x, x_scale, y, y_scale, acc, x_format, y_format, allow_mixed) -> acc + x @ y (a new tensor), error code, or None.
// Every rule of mma_scaled that could fail is a condition here: what is not the plain block-32 case is left to ops.py.
PyObject* py_mma(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 8) { PyErr_SetString(PyExc_TypeError, "mma takes 8 arguments"); return nullptr; }
  for (int i = 0; i < 5; ++i)
    if (!THPVariable_Check(a[i])) Py_RETURN_NONE;
  const at::Tensor &x = THPVariable_Unpack(a[0]), &xs = THPVariable_Unpack(a[1]), &y = THPVariable_Unpack(a[2]),
                   &ys = THPVariable_Unpack(a[3]), &acc = THPVariable_Unpack(a[4]);
  const int xd = (int)x.dim(), yd = (int)y.dim();
  if ((xd != 2 && xd != 3) || (yd != 2 && yd != 3) || xs.dim() != xd || ys.dim() != yd || !on_current_device(x)) Py_RETURN_NONE;
  const at::Device dev = x.device();
  if (xs.device() != dev || y.device() != dev || ys.device() != dev || acc.device() != dev) Py_RETURN_NONE;
  const int fx = elem_format(x, a[5]), fy = elem_format(y, a[6]);
  if (fx < 0 || fy < 0 || (fx != fy && !PyObject_IsTrue(a[7])) || !is_e8m0(xs) || !is_e8m0(ys)) Py_RETURN_NONE;
  if ((fx == MX_E2M1 && x.stride(-1) != 1) || (fy == MX_E2M1 && y.stride(-2) != 1)) Py_RETURN_NONE;
  mx_tensor dx = desc(x, fx, fx == MX_E2M1 ? xd - 1 : -1), dy = desc(y, fy, fy == MX_E2M1 ? yd - 2 : -1),
            dxs = desc(xs, MX_E8M0), dys = desc(ys, MX_E8M0);
  const int64_t M = dx.shape[xd - 2], K = dx.shape[xd - 1], N = dy.shape[yd - 1];
  const int64_t bx = xd == 3 ? x.size(0) : 1, by = yd == 3 ? y.size(0) : 1, batch = bx > by ? bx : by;
  if (dy.shape[yd - 2] != K || K == 0 || K % 32 != 0 || M == 0 || N == 0 || (bx != by && bx != 1 && by != 1) || bx == 0 || by == 0 ||
      dxs.shape[xd - 2] != M || dxs.shape[xd - 1] != K / 32 || dys.shape[yd - 2] != K / 32 || dys.shape[yd - 1] != N ||
      (xd == 3 && dxs.shape[0] != bx) || (yd == 3 && dys.shape[0] != by))
    Py_RETURN_NONE;
  const bool batched = xd == 3 || yd == 3;
  if (acc.scalar_type() != at::kFloat || !acc.is_contiguous() || acc.dim() != (batched ? 3 : 2) || acc.size(-2) != M ||
      acc.size(-1) != N || (batched && acc.size(0) != batch) || acc.requires_grad())   // (there the result is a clone of acc)
    Py_RETURN_NONE;
  at::Tensor out = device_empty(acc.sizes(), at::kFloat, dev);
  mx_tensor dD = desc(acc, MX_F32), dC = desc(out, MX_F32);
  mx_gemm_opts o = {sizeof(mx_gemm_opts), 0, MX_SCALE_2D, MX_SCALE_2D, MX_KERNEL_AUTO, 32, 0, 0};
  // one product at a time needs its workspace once, a batch in one launch all re-laid scales at once
  const int64_t one = lib.p_mx_gemm_workspace_bytes(M, N, K, &o),
                all = (lib.p_mx_packed_scale_bytes(M, K) + lib.p_mx_packed_scale_bytes(N, K)) * batch, need = one > all ? one : all;
  at::Tensor ws;
  if (need > 0) ws = device_empty({need}, at::kByte, dev);
  int rc;
  {
    NoGil nogil;
    rc = lib.p_mx_gemm_add(&dx, &dxs, &dy, &dys, &dD, &dC, &o, need > 0 ? ws.data_ptr() : nullptr, need, stream_of(dev));
  }
  return rc_or(rc, out);
}

// quantize(x, dtype | str, mode, silu) -> (elements, scales), error code, or None.
// mode: 0 "ceil", 1 "floor"; silu: x is gate | up and silu(gate) * up is what is quantised
PyObject* py_quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 4) { PyErr_SetString(PyExc_TypeError, "quantize takes 4 arguments"); return nullptr; }
  if (!THPVariable_Check(a[0])) Py_RETURN_NONE;
  const at::Tensor& x = THPVariable_Unpack(a[0]);
  const auto xt = x.scalar_type();
  const int xc = xt == at::kFloat ? MX_F32 : xt == at::kBFloat16 ? MX_BF16 : xt == at::kHalf ? MX_F16 : -1;
  int fmt = -1;
  if (THPDtype_Check(a[1])) {
    const auto t = ((THPDtype*)a[1])->scalar_type;
    fmt = t == at::kFloat8_e4m3fn ? MX_E4M3 : t == at::kFloat8_e5m2 ? MX_E5M2 : t == at::kFloat4_e2m1fn_x2 ? MX_E2M1 : -1;
  } else if (PyUnicode_Check(a[1])) {
    if (PyUnicode_CompareWithASCIIString(a[1], "e2m1") == 0) fmt = MX_E2M1;
    else if (PyUnicode_CompareWithASCIIString(a[1], "e4m3") == 0) fmt = MX_E4M3;
    else if (PyUnicode_CompareWithASCIIString(a[1], "e5m2") == 0) fmt = MX_E5M2;
  }
  const int silu = PyObject_IsTrue(a[3]);
  if (fmt < 0 || xc < 0 || x.dim() < 1 || x.dim() > 4 || !on_current_device(x)) Py_RETURN_NONE;
  const int64_t cols = x.size(-1), K = silu ? cols / 2 : cols;
  if (cols == 0 || K % 32 != 0 || K < 32 || (silu && cols % 64 != 0) || x.numel() == 0) Py_RETURN_NONE;
  if (!(x.is_contiguous() || (x.dim() == 2 && x.stride(1) == 1))) Py_RETURN_NONE;
  const at::Device dev = x.device();
  const int64_t rows = x.numel() / cols;
  int64_t shape[4];
  const int nd = (int)x.dim();
  for (int i = 0; i + 1 < nd; ++i) shape[i] = x.size(i);
  shape[nd - 1] = fmt == MX_E2M1 ? K / 2 : K;
  at::Tensor q = device_empty(at::IntArrayRef(shape, nd),
                              fmt == MX_E4M3 ? at::kFloat8_e4m3fn : fmt == MX_E5M2 ? at::kFloat8_e5m2 : at::kByte, dev);
  shape[nd - 1] = K / 32;
  at::Tensor s = device_empty(at::IntArrayRef(shape, nd), at::kFloat8_e8m0fnu, dev);
  mx_tensor dx{x.data_ptr(), xc, 2, {rows, cols, 0, 0}, {nd == 2 ? x.stride(0) : cols, 1, 0, 0}, -1, 0};
  mx_tensor dq{q.data_ptr(), fmt, 2, {rows, K, 0, 0}, {fmt == MX_E2M1 ? K / 2 : K, 1, 0, 0}, fmt == MX_E2M1 ? 1 : -1, 0};
  mx_tensor ds{s.data_ptr(), MX_E8M0, 2, {rows, K / 32, 0, 0}, {K / 32, 1, 0, 0}, -1, 0};
  const int mode = (int)PyLong_AsLong(a[2]);
  int rc;
  {
    NoGil nogil;
    rc = silu ? lib.p_mx_silu_mul_quantize(&dx, &dq, &ds, mode, stream_of(dev)) : lib.p_mx_quantize(&dx, &dq, &ds, mode, stream_of(dev));
  }
  if (rc != MX_OK) return PyLong_FromLong(rc);
  PyObject* res = PyTuple_New(2);
  if (!res) return nullptr;
  PyTuple_SET_ITEM(res, 0, THPVariable_Wrap(q));
  PyTuple_SET_ITEM(res, 1, THPVariable_Wrap(s));
  return res;
}

// scales of a stack of expert weights: a [E, rows, K/32] E8M0 tensor or a PackedScales of it
bool expert_scale_desc(PyObject* o, int64_t E, int64_t rows, int64_t K, const at::Device& dev, mx_tensor* d, int32_t* layout) {
  if (THPVariable_Check(o)) {
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!is_e8m0(t) || t.device() != dev || t.dim() != 3) return false;
    *d = desc(t, MX_E8M0);
    *layout = MX_SCALE_2D;
    return true;
  }
  if ((PyObject*)Py_TYPE(o) != packed_type) return false;
  PyObject* pb = PyObject_GetAttr(o, s_batch);
  const bool ok = pb && PyLong_AsLongLong(pb) == E;
  Py_XDECREF(pb);
  if (PyErr_Occurred()) { PyErr_Clear(); return false; }
  if (!ok || !scale_desc(o, rows, K, true, dev, d, layout) || *layout != MX_SCALE_NATIVE) return false;
  d->ndim = 3;
  d->shape[0] = E; d->shape[1] = rows; d->shape[2] = K / 32;
  d->stride[0] = rows * (K / 32); d->stride[1] = K / 32; d->stride[2] = 1;
  return true;
}

// moe(hidden, hidden_scale, w1, w1_scale, w2, w2_scale, topk_weights, topk_ids, out_dtype, mode, w_format, tile_m)
//   -> result, error code, or None
PyObject* py_moe(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 12) { PyErr_SetString(PyExc_TypeError, "moe takes 12 arguments"); return nullptr; }
  for (int i : {0, 1, 2, 4, 6, 7})
    if (!THPVariable_Check(a[i])) Py_RETURN_NONE;
  const at::Tensor &X = THPVariable_Unpack(a[0]), &Xs = THPVariable_Unpack(a[1]), &W1 = THPVariable_Unpack(a[2]),
                   &W2 = THPVariable_Unpack(a[4]), &wt = THPVariable_Unpack(a[6]), &ids = THPVariable_Unpack(a[7]);
  if (X.dim() != 2 || Xs.dim() != 2 || W1.dim() != 3 || W2.dim() != 3 || ids.dim() != 2 || !on_current_device(X)) Py_RETURN_NONE;
  const at::Device dev = X.device();
  if (Xs.device() != dev || W1.device() != dev || W2.device() != dev || wt.device() != dev || ids.device() != dev) Py_RETURN_NONE;
  const int f1 = elem_format(W1, a[10]), f2 = elem_format(W2, a[10]);
  if (X.scalar_type() != at::kFloat8_e4m3fn || !is_e8m0(Xs) || f1 != f2 || (f1 != MX_E4M3 && f1 != MX_E2M1)) Py_RETURN_NONE;
  if (f1 == MX_E2M1 && (W1.stride(2) != 1 || W2.stride(2) != 1)) Py_RETURN_NONE;
  const int64_t T = X.size(0), topk = ids.size(1), E = W1.size(0);
  if (ids.size(0) != T || T == 0 || topk == 0 || topk > 1 << 20 || !ids.is_contiguous() ||
      (ids.scalar_type() != at::kInt && ids.scalar_type() != at::kLong) || wt.scalar_type() != at::kFloat ||
      !wt.is_contiguous() || wt.numel() != T * topk || !THPDtype_Check(a[8]))
    Py_RETURN_NONE;
  const auto out_t = ((THPDtype*)a[8])->scalar_type;
  if (out_code(out_t) < 0) Py_RETURN_NONE;
  mx_tensor dX = desc(X, MX_E4M3), dXs = desc(Xs, MX_E8M0), dW1 = desc(W1, f1, f1 == MX_E2M1 ? 2 : -1),
            dW2 = desc(W2, f2, f2 == MX_E2M1 ? 2 : -1), dW1s, dW2s;
  const long tile_m = PyLong_AsLong(a[11]);
  if (tile_m == -1 && PyErr_Occurred()) PyErr_Clear();
  if (tile_m <= 0 || tile_m > 0x7FFFFFFF) Py_RETURN_NONE;
  // (the operator's default, 256, leaves the form of the layer to the library)
  mx_gemm_opts o = {sizeof(mx_gemm_opts), 0, 0, 0, MX_KERNEL_AUTO, 32, 0, tile_m == 256 ? 0 : (int32_t)tile_m};
  if (!expert_scale_desc(a[3], E, dW1.shape[1], dW1.shape[2], dev, &dW1s, &o.a_scale_layout) ||
      !expert_scale_desc(a[5], E, dW2.shape[1], dW2.shape[2], dev, &dW2s, &o.b_scale_layout))
    Py_RETURN_NONE;
  at::Tensor out = device_empty({T, dW2.shape[1]}, out_t, dev);
  mx_tensor dO = desc(out, out_code(out_t));
  const int mode = (int)PyLong_AsLong(a[9]);
  const int64_t need = lib.p_mx_moe_forward_workspace_bytes(T, (int32_t)topk, &dW1, &dW2, &o);
  at::Tensor ws = device_empty({need > 0 ? need : 1}, at::kByte, dev);
  int rc;
  {
    NoGil nogil;
    rc = lib.p_mx_moe_forward(&dX, &dXs, &dW1, &dW1s, &dW2, &dW2s, (const float*)wt.data_ptr(), ids.data_ptr(),
                              ids.scalar_type() == at::kLong, (int32_t)topk, &dO, mode, &o, ws.data_ptr(), need, stream_of(dev));
  }
  if (rc == MX_ERR_LAYOUT) Py_RETURN_NONE;   // nothing was enqueued: operands for the single operators
  return rc_or(rc, out);
}

// bind(handle of the loaded libmxgemm.so, PackedScales class)
PyObject* py_bind(PyObject*, PyObject* args) {
  unsigned long long h;
  PyObject* cls;
  if (!PyArg_ParseTuple(args, "KO", &h, &cls)) return nullptr;
#define MX_FN(name)                                                                      \
  if (!(lib.p_##name = (decltype(lib.p_##name))dlsym((void*)h, #name))) {                \
    PyErr_SetString(PyExc_RuntimeError, "libmxgemm.so does not export " #name);          \
    return nullptr;                                                                      \
  }
  MX_FN(mx_gemm)
  MX_FN(mx_gemm_add)
  MX_FN(mx_gemm_workspace_bytes)
  MX_FN(mx_packed_scale_bytes)
  MX_FN(mx_gemm_list)
  MX_FN(mx_gemm_list_workspace_bytes)
  MX_FN(mx_quantize)
  MX_FN(mx_silu_mul_quantize)
  MX_FN(mx_moe_forward)
  MX_FN(mx_moe_forward_workspace_bytes)
#undef MX_FN
  Py_INCREF(cls);
  Py_XDECREF(packed_type);
  packed_type = cls;
  Py_RETURN_NONE;
}

// torch and allocator errors (out of memory, ...) become Python exceptions of the same kind
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  return F(self, a, n);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, nullptr},
    {"gemm", (PyCFunction)(void (*)(void))guarded<py_gemm>, METH_FASTCALL, nullptr},
    {"gemm_list", (PyCFunction)(void (*)(void))guarded<py_gemm_list>, METH_FASTCALL, nullptr},
    {"mma", (PyCFunction)(void (*)(void))guarded<py_mma>, METH_FASTCALL, nullptr},
    {"quantize", (PyCFunction)(void (*)(void))guarded<py_quantize>, METH_FASTCALL, nullptr},
    {"moe", (PyCFunction)(void (*)(void))guarded<py_moe>, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_mxhost", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__mxhost(void) {
  s_data = PyUnicode_InternFromString("data");
  s_rows = PyUnicode_InternFromString("rows");
  s_K = PyUnicode_InternFromString("K");
  s_operand = PyUnicode_InternFromString("operand");
  s_layout = PyUnicode_InternFromString("layout");
  s_batch = PyUnicode_InternFromString("batch");
  return PyModule_Create(&module);
}
