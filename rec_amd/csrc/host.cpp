// The Python side of the smallest calls, native: a decode step's cache and
// attention call and a projection are 5-20 us on the GPU, and checking their
// tensors, allocating the result and calling through ctypes took 13-23 us of
// Python.  The functions here take the tensors themselves, make the checks of
// rec_amd.attention / rec_amd.gemv for the plain case (dtypes, shapes, strides,
// alignment, one device) and launch through the C ABI; anything else, and any
// error, returns None, and the caller's general path runs (and raises).
//
// No state is kept: the caller passes the workspace and the stream.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/rec_amd.h"

namespace {

constexpr int64_t DIM = 128, MAX_GROUP = 8;

// The float types of queries and new keys / values as C ABI codes, or -1.
int float_code(at::ScalarType t) {
  return t == at::kHalf ? REC_F16 : t == at::kBFloat16 ? REC_BF16 : t == at::kFloat ? REC_F32 : -1;
}

// A GPU tensor with memory of its own, on device `dev` (any when dev < 0).
const at::Tensor* tensor(PyObject* o, int dev) {
  if (!THPVariable_Check(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || !t.has_storage() || (dev >= 0 && t.get_device() != dev)) return nullptr;
  return &t;
}

bool aligned16(const at::Tensor& t) { return ((uintptr_t)t.data_ptr() & 15) == 0; }

// Rows the kernels read with vector loads: unit dim stride, 16-byte aligned
// start, other strides multiples of 4 elements.
bool rows_aligned(const at::Tensor& t, int64_t outer) {
  const auto s = t.strides();
  if (s.back() != 1 || !aligned16(t)) return false;
  for (int64_t i = 0; i < outer; ++i)
    if (s[i] % 4 != 0) return false;
  return true;
}

struct Step {  // one query token and one new key / value token
  const at::Tensor *q, *k, *v;
  int dev, q_code, kv_code;
  int B, Hq, H;
};

bool plain_step(PyObject* const* a, Step& s) {
  s.q = tensor(a[0], -1);
  if (!s.q || s.q->dim() != 4) return false;
  s.dev = (int)s.q->get_device();
  s.k = tensor(a[1], s.dev);
  s.v = tensor(a[2], s.dev);
  if (!s.k || !s.v || s.k->dim() != 4 || s.k->sizes() != s.v->sizes()) return false;
  s.q_code = float_code(s.q->scalar_type());
  s.kv_code = float_code(s.k->scalar_type());
  if (s.q_code < 0 || s.kv_code < 0 || s.v->scalar_type() != s.k->scalar_type()) return false;
  const auto qs = s.q->sizes(), ks = s.k->sizes();
  if (qs[2] != 1 || qs[3] != DIM || ks[2] != 1 || ks[3] != DIM || qs[0] != ks[0] || qs[0] < 1 || ks[1] < 1) return false;
  if (qs[1] % ks[1] != 0 || qs[1] / ks[1] > MAX_GROUP || qs[1] < 1) return false;
  if (!rows_aligned(*s.q, 2) || !rows_aligned(*s.k, 3) || !rows_aligned(*s.v, 3)) return false;
  s.B = (int)qs[0];
  s.Hq = (int)qs[1];
  s.H = (int)ks[1];
  return true;
}

// float32 sinks of every query head (None: no sinks); false when they need more than their pointer.
bool plain_sinks(PyObject* o, const Step& s, const float** p) {
  *p = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* t = tensor(o, s.dev);
  if (!t || t->scalar_type() != at::kFloat || !t->is_contiguous() || t->numel() != s.Hq) return false;
  *p = (const float*)t->data_ptr();
  return true;
}

// A buffer of at least the decode workspace's bytes.
const at::Tensor* decode_workspace(PyObject* o, const Step& s, int64_t T, int* splits) {
  const at::Tensor* ws = tensor(o, s.dev);
  *splits = rec_decode_default_splits(s.B, s.H, T);
  if (!ws || (size_t)ws->nbytes() < rec_decode_workspace_bytes(s.B, s.H, *splits)) return nullptr;
  return ws;
}

at::Tensor step_out(const Step& s) { return at::empty({s.B, s.Hq, 1, DIM}, s.q->options().requires_grad(false)); }

// One side of a quantized cache: codes, scales, zeros (or None).
struct Side {
  const at::Tensor *codes, *scales, *zeros;
  int code;
};
bool plain_side(PyObject* const* a, int bits, bool affine, const Step& s, Side& c) {
  c.codes = tensor(a[0], s.dev);
  c.scales = tensor(a[1], s.dev);
  c.zeros = a[2] == Py_None ? nullptr : tensor(a[2], s.dev);
  if (!c.codes || !c.scales || (a[2] != Py_None && !c.zeros) || c.codes->dim() < 2) return false;
  if (c.codes->size(0) != s.B || c.codes->size(1) != s.H) return false;
  c.code = !affine ? bits
           : c.scales->scalar_type() == at::kHalf ? (bits == 8 ? REC_AFFINE8_F16 : REC_AFFINE4_F16)
                                                  : (bits == 8 ? REC_AFFINE8 : REC_AFFINE4);
  return true;
}

// decode_quantized(q, k, v, k_codes, k_scales, k_zeros, k_bits, v_codes, v_scales, v_zeros, v_bits, affine,
//                  sinks, scale, T, capacity, workspace, stream) -> out or None
PyObject* decode_quantized(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 18) Py_RETURN_NONE;
  try {
    Step s;
    Side k, v;
    const float* sinks;
    int splits;
    if (!plain_step(a, s)) Py_RETURN_NONE;
    const bool affine = PyObject_IsTrue(a[11]) == 1;
    const double scale = PyFloat_AsDouble(a[13]);
    const int64_t T = PyLong_AsLongLong(a[14]), capacity = PyLong_AsLongLong(a[15]);
    const int kb = (int)PyLong_AsLong(a[6]), vb = (int)PyLong_AsLong(a[10]);
    void* stream = (void*)PyLong_AsUnsignedLongLong(a[17]);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    if (!plain_side(a + 3, kb, affine, s, k) || !plain_side(a + 7, vb, affine, s, v) || !plain_sinks(a[12], s, &sinks))
      Py_RETURN_NONE;
    const at::Tensor* ws = decode_workspace(a[16], s, T, &splits);
    if (!ws) Py_RETURN_NONE;
    at::Tensor out = step_out(s);
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = rec_decode_append_attn(
        s.q->data_ptr(), s.q_code, s.q->stride(0), s.q->stride(1), s.k->data_ptr(), s.v->data_ptr(), s.kv_code,
        s.k->stride(0), s.k->stride(1), s.v->stride(0), s.v->stride(1), k.code, k.codes->data_ptr(),
        (uint16_t*)k.scales->data_ptr(), k.zeros ? (uint16_t*)k.zeros->data_ptr() : nullptr, v.code,
        v.codes->data_ptr(), (uint16_t*)v.scales->data_ptr(), v.zeros ? (uint16_t*)v.zeros->data_ptr() : nullptr, sinks,
        (float)scale, s.B, s.Hq, s.H, (int)DIM, T, capacity, splits, ws->data_ptr(), ws->nbytes(), s.q_code,
        out.data_ptr(), stream);
    Py_END_ALLOW_THREADS;
    if (rc == REC_OK) return THPVariable_Wrap(out);
  } catch (const std::exception&) {
    PyErr_Clear();
  }
  Py_RETURN_NONE;
}

// decode_ring(q, k, v, ring_k, ring_v, sinks, scale, T, capacity, slot, workspace, stream) -> out or None
PyObject* decode_ring(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 12) Py_RETURN_NONE;
  try {
    Step s;
    const float* sinks;
    int splits;
    if (!plain_step(a, s)) Py_RETURN_NONE;
    const double scale = PyFloat_AsDouble(a[6]);
    const int64_t T = PyLong_AsLongLong(a[7]), capacity = PyLong_AsLongLong(a[8]), slot = PyLong_AsLongLong(a[9]);
    void* stream = (void*)PyLong_AsUnsignedLongLong(a[11]);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    const at::Tensor *rk = tensor(a[3], s.dev), *rv = tensor(a[4], s.dev);
    if (!rk || !rv || rk->dim() != 4 || rk->sizes() != rv->sizes() || rk->size(0) != s.B || rk->size(1) != s.H ||
        rk->size(2) < capacity || rk->scalar_type() != at::kBFloat16 || rv->scalar_type() != at::kBFloat16 ||
        !plain_sinks(a[5], s, &sinks))
      Py_RETURN_NONE;
    const at::Tensor* ws = decode_workspace(a[10], s, T, &splits);
    if (!ws) Py_RETURN_NONE;
    at::Tensor out = step_out(s);
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = rec_decode_bf16_ring(s.q->data_ptr(), s.q_code, s.q->stride(0), s.q->stride(1), s.k->data_ptr(),
                              s.v->data_ptr(), s.kv_code, s.k->stride(0), s.k->stride(1), s.v->stride(0),
                              s.v->stride(1), rk->data_ptr(), rk->stride(0), rk->stride(1), rv->data_ptr(),
                              rv->stride(0), rv->stride(1), sinks, (float)scale, s.B, s.Hq, s.H, (int)DIM, T, capacity,
                              slot, 0, ws->data_ptr(), ws->nbytes(), s.q_code, out.data_ptr(), stream);
    Py_END_ALLOW_THREADS;
    if (rc == REC_OK) return THPVariable_Wrap(out);
  } catch (const std::exception&) {
    PyErr_Clear();
  }
  Py_RETURN_NONE;
}

// q4_matmul(x, packed, N, K, fp32, gemm_rows, stream) -> out or None; from gemm_rows rows on one GEMM
PyObject* q4_matmul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 7) Py_RETURN_NONE;
  try {
    const at::Tensor* x = tensor(a[0], -1);
    if (!x) Py_RETURN_NONE;
    const at::Tensor* w = tensor(a[1], (int)x->get_device());
    const int64_t N = PyLong_AsLongLong(a[2]), K = PyLong_AsLongLong(a[3]), gemm_rows = PyLong_AsLongLong(a[5]);
    const bool fp32 = PyObject_IsTrue(a[4]) == 1;
    void* stream = (void*)PyLong_AsUnsignedLongLong(a[6]);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    if (!w || x->scalar_type() != at::kBFloat16 || x->dim() < 1 || x->size(-1) != K || x->numel() == 0 || !aligned16(*x))
      Py_RETURN_NONE;
    const int64_t rows = x->numel() / K;
    int64_t stride = K;
    if (x->dim() == 2) {
      stride = x->stride(0);
      if (x->stride(1) != 1 || (rows > 1 && (stride % 8 != 0 || stride < K))) Py_RETURN_NONE;
    } else if (!x->is_contiguous()) {
      Py_RETURN_NONE;
    }
    if (rows > INT32_MAX) Py_RETURN_NONE;
    auto shape = x->sizes().vec();
    shape.back() = N;
    const auto opt = x->options().requires_grad(false);
    at::Tensor out = at::empty(shape, opt.dtype(fp32 ? at::kFloat : at::kBFloat16)), ws;
    const bool gemm = rows >= gemm_rows;
    if (gemm) ws = at::empty({(int64_t)rec_q4_gemm_workspace_bytes((int)rows, K)}, opt.dtype(at::kByte));
    const int code = fp32 ? REC_F32 : REC_BF16;
    int rc = REC_OK;
    Py_BEGIN_ALLOW_THREADS;
    if (gemm) {
      rc = rec_q4_gemm(w->data_ptr(), N, K, (const uint16_t*)x->data_ptr(), stride, (int)rows, out.data_ptr(), code, N,
                       ws.data_ptr(), ws.nbytes(), stream);
    } else {
      for (int64_t r = 0; r < rows && rc == REC_OK; r += 8)
        rc = rec_q4_gemv(w->data_ptr(), N, K, (const uint16_t*)x->data_ptr() + r * stride, stride,
                         (int)(rows - r < 8 ? rows - r : 8), (char*)out.data_ptr() + r * N * (fp32 ? 4 : 2), code, N,
                         stream);
    }
    Py_END_ALLOW_THREADS;
    if (rc == REC_OK) return THPVariable_Wrap(out);
  } catch (const std::exception&) {
    PyErr_Clear();
  }
  Py_RETURN_NONE;
}

PyMethodDef METHODS[] = {
    {"decode_quantized", (PyCFunction)(void (*)(void))decode_quantized, METH_FASTCALL, nullptr},
    {"decode_ring", (PyCFunction)(void (*)(void))decode_ring, METH_FASTCALL, nullptr},
    {"q4_matmul", (PyCFunction)(void (*)(void))q4_matmul, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef MODULE = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, METHODS};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&MODULE); }
