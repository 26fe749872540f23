// The package's entry points on torch tensors, in C++: checks, output allocation and the call into libave_fp4.so.
//
// A small call (a decode step of one layer) takes 3 to 15 us on the GPU, and the Python wrapper around it -- a few dozen attribute
// reads for the checks, a device context, torch.empty, ctypes with ten arguments -- took 11 us on the host, so that a sequence of
// such calls ran at the host's pace.  Every function here takes the wrapper's positional arguments and either does the
// whole call (about 4 us with the launch) or returns None without having done anything: when an argument is not exactly what
// the kernels take -- another dtype, shape, device or layout, a tensor subclass -- the Python wrapper goes on with its own
// checks, which say what is wrong.  The checks below are therefore conditions, not messages.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>

#include "../../include/ave_fp4.h"

namespace {

using at::Tensor;

// ---- arguments ---------------------------------------------------------------------------------------------------------
const Tensor* tensor(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

bool is_byte(const Tensor& t) {   // uint8, or a 1-byte FP4 / FP8 dtype that is viewed as such
  const auto d = t.scalar_type();
  return d == at::kByte || d == at::ScalarType::Float4_e2m1fn_x2 || d == at::ScalarType::Float8_e8m0fnu || d == at::ScalarType::Float8_e4m3fn;
}
// on the GPU `dev`, contiguous, of this shape
bool matrix(const Tensor& t, c10::Device dev, int64_t d0, int64_t d1) {
  return t.dim() == 2 && t.size(0) == d0 && t.size(1) == d1 && t.device() == dev && t.is_contiguous();
}
bool cube(const Tensor& t, c10::Device dev, int64_t d0, int64_t d1, int64_t d2) {
  return t.dim() == 3 && t.size(0) == d0 && t.size(1) == d1 && t.size(2) == d2 && t.device() == dev && t.is_contiguous();
}
bool vec(const Tensor& t, c10::Device dev, int64_t n, at::ScalarType dtype) {
  return t.dim() == 1 && t.size(0) == n && t.scalar_type() == dtype && t.device() == dev && t.is_contiguous();
}
bool fits(int64_t v) { return v >= 0 && v <= INT_MAX; }
void* ptr(const Tensor& t) { return t.data_ptr(); }
template <typename T>
T* ptr_as(const Tensor& t) { return static_cast<T*>(t.data_ptr()); }

bool as_int(PyObject* o, int* v) {
  if (!PyLong_CheckExact(o)) return false;
  const long x = PyLong_AsLong(o);
  if (x == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  *v = (int)x;
  return x >= INT_MIN && x <= INT_MAX;
}

// Other Python threads run while this one is inside: an allocation may have to wait for the driver, as torch.empty's may.
struct NoGil {
  PyThreadState* const state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};
Tensor empty(at::IntArrayRef shape, at::ScalarType dtype, c10::Device dev) {
  NoGil no_gil;
  return at::empty(shape, at::TensorOptions().dtype(dtype).device(dev));
}
Tensor zeros(at::IntArrayRef shape, at::ScalarType dtype, c10::Device dev) {
  NoGil no_gil;
  return at::zeros(shape, at::TensorOptions().dtype(dtype).device(dev));
}

// `given` (None: a new tensor) as the output of this shape and dtype; false when a given one does not fit.
struct Out {
  Tensor t;
  PyObject* given = nullptr;
  bool take(PyObject* o, at::IntArrayRef shape, at::ScalarType dtype, c10::Device dev, bool zero = false) {
    if (o == Py_None) {
      t = zero ? zeros(shape, dtype, dev) : empty(shape, dtype, dev);
      return true;
    }
    const Tensor* p = tensor(o);
    if (!p || p->scalar_type() != dtype || p->device() != dev || p->sizes() != shape || !p->is_contiguous()) return false;
    t = *p;
    given = o;
    return true;
  }
  PyObject* object() const {   // a new reference
    if (given) {
      Py_INCREF(given);
      return given;
    }
    return THPVariable_Wrap(t);
  }
};

PyObject* pair_of(const Out& a, const Out& b) {
  PyObject* x = a.object();
  PyObject* y = x ? b.object() : nullptr;
  PyObject* r = y ? PyTuple_Pack(2, x, y) : nullptr;
  Py_XDECREF(x);
  Py_XDECREF(y);
  return r;
}

// ---- the call ------------------------------------------------------------------------------------------------------------
// Runs f(stream) with `dev` current and the GIL released; true when it returned 0, otherwise the exception is set.
template <typename F>
bool launch(c10::Device dev, F f) {
  int rc;
  const auto current = c10::hip::current_device();
  if (current != dev.index()) c10::hip::set_device(dev.index());
  void* stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  {
    NoGil no_gil;
    rc = f(stream);
  }
  if (current != dev.index()) c10::hip::set_device(current);
  if (rc == 0) return true;
  const char* msg = ave_fp4_last_error();
  if (rc == AVE_FP4_EINVAL) PyErr_SetString(PyExc_ValueError, msg);
  else if (msg[0]) PyErr_SetString(PyExc_RuntimeError, msg);
  else PyErr_Format(PyExc_RuntimeError, "ave-lang Error [HIP]: error %d", rc);
  return false;
}

// A workspace query runs on the device that the call will run on (plans depend on its compute units).
template <typename F>
size_t on_device(c10::Device dev, F f) {
  const auto current = c10::hip::current_device();
  if (current == dev.index()) return f();
  c10::hip::set_device(dev.index());
  const size_t r = f();
  c10::hip::set_device(current);
  return r;
}

#define NOT_MINE Py_RETURN_NONE

struct Gemm {   // A, its scales, B, its scales
  const Tensor *a, *as, *b, *bs;
  c10::Device dev{c10::kCPU};
  int64_t m = 0, n = 0, k = 0, e = 0;   // n: rows of B (of one expert)
  // group_k: elements per scale; grouped: B is [E, rows, K/2]
  bool take(PyObject* const* arg, int64_t group_k, bool grouped) {
    return take(tensor(arg[0]), tensor(arg[1]), tensor(arg[2]), tensor(arg[3]), group_k, grouped);
  }
  bool take(const Tensor* a_, const Tensor* as_, const Tensor* b_, const Tensor* bs_, int64_t group_k, bool grouped) {
    a = a_, as = as_, b = b_, bs = bs_;
    if (!a || !as || !b || !bs || !is_byte(*a) || !is_byte(*as) || !is_byte(*b) || !is_byte(*bs)) return false;
    if (a->dim() != 2 || b->dim() != (grouped ? 3 : 2) || !a->is_cuda()) return false;
    dev = a->device();
    m = a->size(0), k = 2 * a->size(1);
    e = grouped ? b->size(0) : 0;
    n = b->size(grouped ? 1 : 0);
    if (k <= 0 || k % group_k != 0 || !fits(m) || !fits(n) || !fits(k) || !fits(e)) return false;
    if (!matrix(*a, dev, m, k / 2) || !matrix(*as, dev, m, k / group_k)) return false;
    return grouped ? cube(*b, dev, e, n, k / 2) && cube(*bs, dev, e, n, k / group_k) : matrix(*b, dev, n, k / 2) && matrix(*bs, dev, n, k / group_k);
  }
};

const uint8_t* u8(const Tensor* t) { return static_cast<const uint8_t*>(t->data_ptr()); }

// A, A_scale, B, B_scale, out, variant, split_k
PyObject* gemm_mxfp4(PyObject* const* arg) {
  Gemm g;
  Out out;
  int variant;
  if (!g.take(arg, 32, false) || !as_int(arg[5], &variant) || !out.take(arg[4], {g.m, g.n}, at::kBFloat16, g.dev)) NOT_MINE;
  const int split = PyObject_IsTrue(arg[6]);
  if (split < 0) return nullptr;
  const size_t bytes = variant == AVE_FP4_AUTO && split ? on_device(g.dev, [&] { return ave_fp4_gemm_mxfp4_planned_workspace_bytes(g.m, g.n, g.k); }) : 0;
  Tensor ws;
  if (bytes) ws = empty({(int64_t)bytes}, at::kByte, g.dev);
  const bool ok = launch(g.dev, [&](void* s) {
    if (bytes) return ave_fp4_gemm_mxfp4_planned(u8(g.a), u8(g.as), u8(g.b), u8(g.bs), ptr_as<uint16_t>(out.t), g.m, g.n, g.k, ptr(ws), bytes, s);
    return ave_fp4_gemm_mxfp4_ex(u8(g.a), u8(g.as), u8(g.b), u8(g.bs), ptr_as<uint16_t>(out.t), g.m, g.n, g.k, s, variant);
  });
  return ok ? out.object() : nullptr;
}

// A, A_scale, A_global, B, B_scale, B_global, out, variant, split_k
PyObject* gemm_nvfp4(PyObject* const* arg) {
  Gemm g;
  Out out;
  int variant;
  if (!g.take(tensor(arg[0]), tensor(arg[1]), tensor(arg[3]), tensor(arg[4]), 16, false) || !as_int(arg[7], &variant)) NOT_MINE;
  const Tensor *ag = tensor(arg[2]), *bg = tensor(arg[5]);
  for (const Tensor* t : {ag, bg})
    if (!t || t->scalar_type() != at::kFloat || t->numel() != 1 || t->device() != g.dev) NOT_MINE;
  if (!out.take(arg[6], {g.m, g.n}, at::kBFloat16, g.dev)) NOT_MINE;
  const int split = PyObject_IsTrue(arg[8]);
  if (split < 0) return nullptr;
  const size_t bytes = variant == AVE_FP4_AUTO && split ? on_device(g.dev, [&] { return ave_fp4_gemm_nvfp4_workspace_bytes(g.m, g.n, g.k); }) : 0;
  Tensor ws;
  if (bytes) ws = empty({(int64_t)bytes}, at::kByte, g.dev);
  const bool ok = launch(g.dev, [&](void* s) {
    if (bytes)
      return ave_fp4_gemm_nvfp4_ws(u8(g.a), u8(g.as), ptr_as<float>(*ag), u8(g.b), u8(g.bs), ptr_as<float>(*bg), ptr_as<uint16_t>(out.t), g.m, g.n,
                                   g.k, ptr(ws), bytes, s);
    return ave_fp4_gemm_nvfp4_ex(u8(g.a), u8(g.as), ptr_as<float>(*ag), u8(g.b), u8(g.bs), ptr_as<float>(*bg), ptr_as<uint16_t>(out.t), g.m, g.n,
                                 g.k, s, variant);
  });
  return ok ? out.object() : nullptr;
}

// A, A_scale_blocked, B, B_scale_blocked, out
PyObject* gemm_mxfp4_blocked_scales(PyObject* const* arg) {
  const Tensor *a = tensor(arg[0]), *as = tensor(arg[1]), *b = tensor(arg[2]), *bs = tensor(arg[3]);
  if (!a || !as || !b || !bs || !is_byte(*a) || !is_byte(*as) || !is_byte(*b) || !is_byte(*bs)) NOT_MINE;
  if (a->dim() != 2 || b->dim() != 2 || !a->is_cuda()) NOT_MINE;
  const auto dev = a->device();
  const int64_t m = a->size(0), n = b->size(0), k = 2 * a->size(1);
  if (k <= 0 || k % 512 != 0 || !fits(m) || !fits(n) || !fits(k) || !matrix(*a, dev, m, k / 2) || !matrix(*b, dev, n, k / 2)) NOT_MINE;
  auto blocked = [&](const Tensor& t, int64_t rows) { return t.dim() == 1 && t.numel() == (rows + 127) / 128 * 128 * (k / 32) && t.device() == dev && t.is_contiguous(); };
  Out out;
  if (!blocked(*as, m) || !blocked(*bs, n) || !out.take(arg[4], {m, n}, at::kBFloat16, dev)) NOT_MINE;
  const bool ok = launch(dev, [&](void* s) {
    return ave_fp4_gemm_mxfp4_blocked_scales(u8(a), u8(as), u8(b), u8(bs), ptr_as<uint16_t>(out.t), m, n, k, s);
  });
  return ok ? out.object() : nullptr;
}

// A, A_scale, B, B_scale, out, variant
PyObject* gemm_mxfp4_swiglu(PyObject* const* arg) {
  Gemm g;
  Out out;
  int variant;
  if (!g.take(arg, 32, false) || g.n % 2 != 0 || !as_int(arg[5], &variant) || !out.take(arg[4], {g.m, g.n / 2}, at::kBFloat16, g.dev)) NOT_MINE;
  const size_t bytes = variant == AVE_FP4_AUTO ? on_device(g.dev, [&] { return ave_fp4_gemm_mxfp4_swiglu_workspace_bytes(g.m, g.n / 2, g.k, 0); }) : 0;
  Tensor ws;
  if (bytes) ws = empty({(int64_t)bytes}, at::kByte, g.dev);
  const bool ok = launch(g.dev, [&](void* s) {
    if (bytes) return ave_fp4_gemm_mxfp4_swiglu_ws(u8(g.a), u8(g.as), u8(g.b), u8(g.bs), ptr_as<uint16_t>(out.t), g.m, g.n / 2, g.k, ptr(ws), bytes, s);
    return ave_fp4_gemm_mxfp4_swiglu_ex(u8(g.a), u8(g.as), u8(g.b), u8(g.bs), ptr_as<uint16_t>(out.t), g.m, g.n / 2, g.k, s, variant);
  });
  return ok ? out.object() : nullptr;
}

bool offsets(PyObject* o, const Gemm& g, const Tensor** t) {
  *t = tensor(o);
  return *t && vec(**t, g.dev, g.e + 1, at::kInt);
}
// codes and scales of a quantising epilogue over n columns; n_pad: None or a multiple of 32 from n up
bool quantised(PyObject* q, PyObject* qs, PyObject* n_pad, const Gemm& g, int64_t n, Out* out, Out* scale, int* padded) {
  if (g.n % 2 != 0 || n % 32 != 0 || g.m == 0 || n == 0) return false;   // (nothing to launch: left to the wrapper)
  *padded = (int)n;
  if (n_pad != Py_None && (!as_int(n_pad, padded) || *padded < n || *padded % 32 != 0)) return false;
  const bool zero = *padded != n;   // the kernels leave the columns from n on alone
  return out->take(q, {g.m, *padded / 2}, at::kByte, g.dev, zero) && scale->take(qs, {g.m, *padded / 32}, at::kByte, g.dev, zero);
}

// A, A_scale, B, B_scale, out, out_scale, n_pad
PyObject* gemm_mxfp4_swiglu_quant(PyObject* const* arg) {
  Gemm g;
  Out out, scale;
  int padded;
  if (!g.take(arg, 32, false) || !quantised(arg[4], arg[5], arg[6], g, g.n / 2, &out, &scale, &padded)) NOT_MINE;
  const size_t bytes = on_device(g.dev, [&] { return ave_fp4_gemm_mxfp4_swiglu_workspace_bytes(g.m, g.n / 2, g.k, 1); });
  Tensor ws;
  if (bytes) ws = empty({(int64_t)bytes}, at::kByte, g.dev);
  const bool ok = launch(g.dev, [&](void* s) {
    return ave_fp4_gemm_mxfp4_swiglu_quant_ws(u8(g.a), u8(g.as), u8(g.b), u8(g.bs), ptr_as<uint8_t>(out.t), ptr_as<uint8_t>(scale.t), g.m, g.n / 2,
                                              padded, g.k, bytes ? ptr(ws) : nullptr, bytes, s);
  });
  return ok ? pair_of(out, scale) : nullptr;
}

// A, A_scale, B, B_scale, row_offsets, out, variant
PyObject* grouped_gemm_mxfp4(PyObject* const* arg) {
  Gemm g;
  Out out;
  const Tensor* ro;
  int variant;
  if (!g.take(arg, 32, true) || !offsets(arg[4], g, &ro) || !as_int(arg[6], &variant) || !out.take(arg[5], {g.m, g.n}, at::kBFloat16, g.dev)) NOT_MINE;
  const bool ok = launch(g.dev, [&](void* s) {
    return ave_fp4_grouped_gemm_mxfp4_ex(u8(g.a), u8(g.as), u8(g.b), u8(g.bs), ptr_as<int32_t>(*ro), ptr_as<uint16_t>(out.t), g.m, g.e, g.n, g.k, s,
                                         variant);
  });
  return ok ? out.object() : nullptr;
}

// A, A_scale, B, B_scale, row_offsets, out
PyObject* grouped_gemm_mxfp4_swiglu(PyObject* const* arg) {
  Gemm g;
  Out out;
  const Tensor* ro;
  if (!g.take(arg, 32, true) || g.n % 2 != 0 || !offsets(arg[4], g, &ro) || !out.take(arg[5], {g.m, g.n / 2}, at::kBFloat16, g.dev)) NOT_MINE;
  const bool ok = launch(g.dev, [&](void* s) {
    return ave_fp4_grouped_gemm_mxfp4_swiglu(u8(g.a), u8(g.as), u8(g.b), u8(g.bs), ptr_as<int32_t>(*ro), ptr_as<uint16_t>(out.t), g.m, g.e, g.n / 2,
                                             g.k, s);
  });
  return ok ? out.object() : nullptr;
}

// A, A_scale, B, B_scale, row_offsets, out, out_scale, n_pad
PyObject* grouped_gemm_mxfp4_swiglu_quant(PyObject* const* arg) {
  Gemm g;
  Out out, scale;
  const Tensor* ro;
  int padded;
  if (!g.take(arg, 32, true) || !offsets(arg[4], g, &ro) || !quantised(arg[5], arg[6], arg[7], g, g.n / 2, &out, &scale, &padded)) NOT_MINE;
  const bool ok = launch(g.dev, [&](void* s) {
    return ave_fp4_grouped_gemm_mxfp4_swiglu_quant_padded(u8(g.a), u8(g.as), u8(g.b), u8(g.bs), ptr_as<int32_t>(*ro), ptr_as<uint8_t>(out.t),
                                                          ptr_as<uint8_t>(scale.t), g.m, g.e, g.n / 2, padded, g.k, s);
  });
  return ok ? pair_of(out, scale) : nullptr;
}

bool activations(PyObject* o, int64_t group_k, const Tensor** x) {
  *x = tensor(o);
  if (!*x || ((*x)->scalar_type() != at::kFloat && (*x)->scalar_type() != at::kBFloat16) || (*x)->dim() != 2 || !(*x)->is_cuda()) return false;
  const int64_t k = (*x)->size(1);
  return k > 0 && k % group_k == 0 && fits((*x)->size(0)) && fits(k) && (*x)->is_contiguous();
}

// x, packed, scales, k_pad
PyObject* quantize_mxfp4(PyObject* const* arg) {
  const Tensor* x;
  if (!activations(arg[0], 32, &x)) NOT_MINE;
  const auto dev = x->device();
  const int64_t r = x->size(0), k = x->size(1);
  int padded = (int)k;
  Out packed, scales;
  if (arg[3] != Py_None && (!as_int(arg[3], &padded) || padded < k || padded % 32 != 0)) NOT_MINE;
  if (!packed.take(arg[1], {r, padded / 2}, at::kByte, dev) || !scales.take(arg[2], {r, padded / 32}, at::kByte, dev)) NOT_MINE;
  const bool ok = launch(dev, [&](void* s) {
    if (x->scalar_type() == at::kBFloat16)
      return ave_fp4_quantize_mxfp4_bf16_padded(ptr_as<uint16_t>(*x), ptr_as<uint8_t>(packed.t), ptr_as<uint8_t>(scales.t), r, k, padded, s);
    return ave_fp4_quantize_mxfp4_f32_padded(ptr_as<float>(*x), ptr_as<uint8_t>(packed.t), ptr_as<uint8_t>(scales.t), r, k, padded, s);
  });
  return ok ? pair_of(packed, scales) : nullptr;
}

// x, global_scale, packed, scales
PyObject* quantize_nvfp4(PyObject* const* arg) {
  const Tensor *x, *g = tensor(arg[1]);
  if (!activations(arg[0], 16, &x) || !g || g->scalar_type() != at::kFloat || g->numel() != 1 || g->device() != x->device()) NOT_MINE;
  const auto dev = x->device();
  const int64_t r = x->size(0), k = x->size(1);
  Out packed, scales;
  if (!packed.take(arg[2], {r, k / 2}, at::kByte, dev) || !scales.take(arg[3], {r, k / 16}, at::kByte, dev)) NOT_MINE;
  const bool ok = launch(dev, [&](void* s) {
    if (x->scalar_type() == at::kBFloat16)
      return ave_fp4_quantize_nvfp4_bf16(ptr_as<uint16_t>(*x), ptr_as<float>(*g), ptr_as<uint8_t>(packed.t), ptr_as<uint8_t>(scales.t), r, k, s);
    return ave_fp4_quantize_nvfp4_f32(ptr_as<float>(*x), ptr_as<float>(*g), ptr_as<uint8_t>(packed.t), ptr_as<uint8_t>(scales.t), r, k, s);
  });
  return ok ? pair_of(packed, scales) : nullptr;
}

// logits, token_of_row, row_offsets, row_weight, rows_of_token
PyObject* moe_route_top2(PyObject* const* arg) {
  const Tensor* l = tensor(arg[0]);
  if (!l || l->scalar_type() != at::kFloat || l->dim() != 2 || !l->is_cuda() || !l->is_contiguous()) NOT_MINE;
  const auto dev = l->device();
  const int64_t t = l->size(0), e = l->size(1);
  if (e < 2 || e > 256 || t > (1 << 29)) NOT_MINE;
  Out token, offs, weight;
  const Tensor* inv = nullptr;
  if (arg[4] != Py_None) {
    inv = tensor(arg[4]);
    if (!inv || inv->scalar_type() != at::kInt || !matrix(*inv, dev, t, 2)) NOT_MINE;
  }
  if (!token.take(arg[1], {2 * t}, at::kInt, dev) || !offs.take(arg[2], {e + 1}, at::kInt, dev) || !weight.take(arg[3], {2 * t}, at::kFloat, dev))
    NOT_MINE;
  // the choices and the counts between the two launches (torch's allocator, stream-ordered, part of a graph's pool)
  const size_t bytes = ave_fp4_moe_route_top2_workspace_bytes(t, e);
  Tensor ws;
  if (bytes) ws = empty({(int64_t)bytes}, at::kByte, dev);
  const bool ok = launch(dev, [&](void* s) {
    return ave_fp4_moe_route_top2_ws(ptr_as<float>(*l), t, e, ptr_as<int32_t>(token.t), ptr_as<int32_t>(offs.t), ptr_as<float>(weight.t),
                                     inv ? ptr_as<int32_t>(*inv) : nullptr, bytes ? ptr(ws) : nullptr, bytes, s);
  });
  if (!ok) return nullptr;
  PyObject *x = token.object(), *y = offs.object(), *z = weight.object();
  PyObject* r = x && y && z ? PyTuple_Pack(3, x, y, z) : nullptr;
  Py_XDECREF(x);
  Py_XDECREF(y);
  Py_XDECREF(z);
  return r;
}

// rows, rows_of_token, row_weight, out, renormalize
PyObject* moe_combine_top2(PyObject* const* arg) {
  const Tensor *rows = tensor(arg[0]), *inv = tensor(arg[1]), *weight = tensor(arg[2]);
  if (!rows || !inv || !weight || rows->scalar_type() != at::kBFloat16 || rows->dim() != 2 || !rows->is_cuda() || !rows->is_contiguous()) NOT_MINE;
  const auto dev = rows->device();
  const int64_t t = rows->size(0) / 2, h = rows->size(1);
  if (rows->size(0) % 2 != 0 || h <= 0 || h % 8 != 0 || !fits(2 * t) || !fits(h)) NOT_MINE;
  Out out;
  if (inv->scalar_type() != at::kInt || !matrix(*inv, dev, t, 2) || !vec(*weight, dev, 2 * t, at::kFloat) || !out.take(arg[3], {t, h}, at::kBFloat16, dev))
    NOT_MINE;
  const int renormalize = PyObject_IsTrue(arg[4]);
  if (renormalize < 0) return nullptr;
  const bool ok = launch(dev, [&](void* s) {
    return ave_fp4_moe_combine_top2(ptr_as<uint16_t>(*rows), ptr_as<int32_t>(*inv), ptr_as<float>(*weight), t, h, renormalize,
                                    ptr_as<uint16_t>(out.t), s);
  });
  return ok ? out.object() : nullptr;
}

// A, A_scale, index, out, out_scale
PyObject* gather_rows_mxfp4(PyObject* const* arg) {
  const Tensor *a = tensor(arg[0]), *as = tensor(arg[1]), *index = tensor(arg[2]);
  if (!a || !as || !index || !is_byte(*a) || !is_byte(*as) || a->dim() != 2 || !a->is_cuda()) NOT_MINE;
  const auto dev = a->device();
  const int64_t src = a->size(0), k = 2 * a->size(1);
  if (k <= 0 || k % 32 != 0 || !fits(src) || !fits(k) || !matrix(*a, dev, src, k / 2) || !matrix(*as, dev, src, k / 32) || index->dim() != 1) NOT_MINE;
  const int64_t rows = index->size(0);
  Out out, scale;
  if (!fits(rows) || !vec(*index, dev, rows, at::kInt) || !out.take(arg[3], {rows, k / 2}, at::kByte, dev) ||
      !scale.take(arg[4], {rows, k / 32}, at::kByte, dev))
    NOT_MINE;
  const bool ok = launch(dev, [&](void* s) {
    return ave_fp4_gather_rows_mxfp4(u8(a), u8(as), ptr_as<int32_t>(*index), rows, src, k, ptr_as<uint8_t>(out.t), ptr_as<uint8_t>(scale.t), s);
  });
  return ok ? pair_of(out, scale) : nullptr;
}

// ---- the module -------------------------------------------------------------------------------------------------------------
template <PyObject* (*F)(PyObject* const*), int ARGS>
PyObject* entry(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != ARGS) {
    PyErr_Format(PyExc_TypeError, "%d arguments expected, got %zd", ARGS, n);
    return nullptr;
  }
  HANDLE_TH_ERRORS   // torch's exceptions (an allocation that does not fit) become the Python ones they are elsewhere
  return F(arg);
  END_HANDLE_TH_ERRORS
}

#define ENTRY(f, args) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<&f, args>)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    ENTRY(gemm_mxfp4, 7),
    ENTRY(gemm_nvfp4, 9),
    ENTRY(gemm_mxfp4_blocked_scales, 5),
    ENTRY(gemm_mxfp4_swiglu, 6),
    ENTRY(gemm_mxfp4_swiglu_quant, 7),
    ENTRY(grouped_gemm_mxfp4, 7),
    ENTRY(grouped_gemm_mxfp4_swiglu, 6),
    ENTRY(grouped_gemm_mxfp4_swiglu_quant, 8),
    ENTRY(quantize_mxfp4, 4),
    ENTRY(quantize_nvfp4, 4),
    ENTRY(moe_route_top2, 5),
    ENTRY(moe_combine_top2, 5),
    ENTRY(gather_rows_mxfp4, 5),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_torch_calls", "the package's entry points on torch tensors, in C++", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_calls() { return PyModule_Create(&kModule); }
