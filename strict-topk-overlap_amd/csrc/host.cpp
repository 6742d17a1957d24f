// Native host path of the fused steps' Python entry points: argument checks,
// output allocation and the C-ABI call of step.speculative_step,
// paged.speculative_step, paged.speculative_signed_step and paged.exact.
//
// A small step's kernel takes 5 us and its call from Python took 26 on the
// host: about 6 us of checks, 10 of allocations, 4 of ctypes conversions and
// the current stream, 4 of launch.  Done here the same call takes a third of
// that.  A call that does not pass every check below, or whose
// arguments are not plain strided tensors (subclasses, wrappers of transforms,
// active modes), returns None, and the Python code runs it as before, with its
// own messages; nothing is kept between calls but the C entry points'
// addresses and which devices were prepared.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/strict_topk.h"

namespace {

struct Entry {
  decltype(&stk_step_supported) step_supported;
  decltype(&stk_step_workspace_bytes) step_workspace;
  decltype(&stk_speculative_step) step;
  decltype(&stk_paged_workspace_bytes) paged_workspace;
  decltype(&stk_paged_step) paged_step;
  decltype(&stk_paged_signed_step) paged_signed;
} g_entry;
bool g_bound = false;
uint64_t g_prepared = 0;   // bit per device whose step memory was looked up

const c10::DispatchKeySet kWrapped({c10::DispatchKey::FuncTorchBatched,
                                    c10::DispatchKey::FuncTorchGradWrapper,
                                    c10::DispatchKey::Functionalize, c10::DispatchKey::Python,
                                    c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                    c10::DispatchKey::ZeroTensor,
                                    c10::DispatchKey::NestedTensor});

// A plain contiguous tensor on a GPU, or null.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided ||
      t.key_set().has_any(kWrapped) || t.unsafeGetTensorImpl()->has_symbolic_sizes_strides() ||
      !t.is_contiguous())
    return nullptr;
  return &t;
}

bool no_modes() {
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !at::impl::torch_function_mode_enabled();
}

int dtype_code(const at::Tensor& t) {
  return t.scalar_type() == at::kHalf ? 1 : (t.scalar_type() == at::kBFloat16 ? 2 : -1);
}

bool aligned(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

bool small(const at::Tensor& t) {
  for (int64_t s : t.sizes())
    if (s < 1 || s > 0x7fffffff) return false;
  return true;
}

// topk as a C int when it is a plain Python int in range
bool plain_int(PyObject* o, long lo, long hi, int* out) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  const long v = PyLong_AsLongAndOverflow(o, &over);
  if (over || v < lo || v > hi) return false;
  *out = (int)v;
  return true;
}

bool plain_float(PyObject* o, double* out) {
  if (PyFloat_CheckExact(o)) *out = PyFloat_AS_DOUBLE(o);
  else if (PyLong_CheckExact(o)) *out = PyLong_AsDouble(o);
  else return false;
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

void* stream_of(const at::Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

PyObject* pack(std::initializer_list<const at::Tensor*> ts) {
  PyObject* r = PyTuple_New((Py_ssize_t)ts.size());
  if (!r) return nullptr;
  Py_ssize_t i = 0;
  for (const at::Tensor* t : ts) {
    PyObject* o;
    if (t->defined()) {
      o = THPVariable_Wrap(*t);
    } else {
      o = Py_None;
      Py_INCREF(o);
    }
    if (!o) {
      Py_DECREF(r);
      return nullptr;
    }
    PyTuple_SET_ITEM(r, i++, o);
  }
  return r;
}

// A C++ exception (a tensor kind the checks do not know, memory that ran out;
// all of them before anything is launched) means None: the Python code then
// meets the same and raises torch's own.
template <typename F>
PyObject* checked(F f) {
  try {
    return f();
  } catch (const std::exception&) {
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
}

// (q, k, v, lo, hi, predicted, topk, union): (selected, m, l, u, out), an error
// code, or None
PyObject* step_impl(PyObject* const* a, Py_ssize_t n) {
  if (!g_bound || n != 8 || !no_modes()) Py_RETURN_NONE;
  const at::Tensor* t[6];
  for (int i = 0; i < 6; ++i)
    if (!(t[i] = plain(a[i]))) Py_RETURN_NONE;
  const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &lo = *t[3], &hi = *t[4], &p = *t[5];
  if (q.dim() != 2 || k.dim() != 4 || lo.dim() != 3 || p.dim() != 2 || !small(q) || !small(k) ||
      !small(p) || v.sizes() != k.sizes() || hi.sizes() != lo.sizes())
    Py_RETURN_NONE;
  const int64_t hq = q.size(0), d = q.size(1), hkv = k.size(0), nb = k.size(1), b = k.size(2);
  const int64_t sp = p.size(1);
  const int dt = dtype_code(q);
  if (dt < 0 || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() ||
      k.size(3) != d || hq % hkv || p.size(0) != hq || p.scalar_type() != at::kInt ||
      lo.size(0) != hkv || lo.size(1) != nb || lo.size(2) != d ||
      hi.scalar_type() != lo.scalar_type() ||
      (lo.scalar_type() != at::kFloat && lo.scalar_type() != q.scalar_type()))
    Py_RETURN_NONE;
  const auto dev = q.device();
  for (int i = 1; i < 6; ++i)
    if (t[i]->device() != dev) Py_RETURN_NONE;
  for (int i = 0; i < 5; ++i)
    if (!aligned(*t[i])) Py_RETURN_NONE;
  int topk;
  const int uni = PyObject_IsTrue(a[7]);
  if (uni < 0) return nullptr;
  if (dev.index() < 0 || dev.index() > 63 || !(g_prepared >> dev.index() & 1) ||
      !plain_int(a[6], 1, nb, &topk) ||
      !g_entry.step_supported(dt, (int)hq, (int)hkv, (int)nb, (int)b, (int)d, topk, (int)sp, 0))
    Py_RETURN_NONE;
  const auto f = q.options().dtype(at::kFloat).requires_grad(false);
  const at::Tensor sel = at::empty({hq, topk}, f.dtype(at::kInt));
  const at::Tensor m = at::empty({hq, sp}, f), l = at::empty({hq, sp}, f);
  const at::Tensor u = at::empty({hq, sp, d}, f), out = at::empty({hq, d}, f);
  const size_t bytes = g_entry.step_workspace((int)hq, (int)hkv, (int)nb, (int)d, topk);
  const at::Tensor ws = at::empty({(int64_t)(bytes ? bytes : 1)}, f.dtype(at::kByte));
  void* st = stream_of(q);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_entry.step(q.data_ptr(), k.data_ptr(), v.data_ptr(), dt, (int)hq, (int)hkv, (int)nb,
                    (int)b, (int)d, lo.data_ptr(), hi.data_ptr(),
                    lo.scalar_type() == at::kFloat ? 0 : dt, topk, p.data_ptr(), 0, (int)sp, uni,
                    sel.data_ptr<int32_t>(), m.data_ptr<float>(), l.data_ptr<float>(),
                    u.data_ptr<float>(), out.data_ptr<float>(), ws.data_ptr(), bytes, st);
  Py_END_ALLOW_THREADS
  if (rc) return PyLong_FromLong(rc);
  return pack({&sel, &m, &l, &u, &out});
}

// (q, k_pages, v_pages, lo, hi, table, nblocks, ntokens or None, predicted or
// None, topk, mode, tau, min_remaining, cancellation, eps): mode 0 saved (or no
// prediction), 1 union, 2 signed saved, 3 signed hybrid.
// Returns (selected, m, l, u, out[, fallback, remaining, approx, extra, pos,
// total]), an error code, or None.
PyObject* paged_impl(PyObject* const* a, Py_ssize_t n) {
  if (!g_bound || n != 15 || !no_modes()) Py_RETURN_NONE;
  const at::Tensor* t[9] = {};
  for (int i = 0; i < 9; ++i) {
    if (i >= 7 && a[i] == Py_None) continue;
    if (!(t[i] = plain(a[i]))) Py_RETURN_NONE;
  }
  const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &lo = *t[3], &hi = *t[4], &tab = *t[5],
                   &nbk = *t[6];
  if (q.dim() != 3 || k.dim() != 3 || lo.dim() != 2 || tab.dim() != 3 || nbk.dim() != 1 ||
      !small(q) || !small(k) || !small(tab) || v.sizes() != k.sizes() ||
      hi.sizes() != lo.sizes())
    Py_RETURN_NONE;
  const int64_t r = q.size(0), hq = q.size(1), d = q.size(2), pages = k.size(0), b = k.size(1);
  const int64_t hkv = tab.size(1), width = tab.size(2);
  const int dt = dtype_code(q);
  if (dt < 0 || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() ||
      k.size(2) != d || lo.size(0) != pages || lo.size(1) != d || tab.size(0) != r || hq % hkv ||
      nbk.size(0) != r || tab.scalar_type() != at::kInt || nbk.scalar_type() != at::kInt ||
      hi.scalar_type() != lo.scalar_type() ||
      (lo.scalar_type() != at::kFloat && lo.scalar_type() != q.scalar_type()))
    Py_RETURN_NONE;
  if (t[7] && (t[7]->dim() != 1 || t[7]->size(0) != r || t[7]->scalar_type() != at::kInt))
    Py_RETURN_NONE;
  if (t[8] && (t[8]->dim() != 3 || !small(*t[8]) || t[8]->size(0) != r || t[8]->size(1) != hq ||
               t[8]->scalar_type() != at::kInt))
    Py_RETURN_NONE;
  const auto dev = q.device();
  for (int i = 1; i < 9; ++i)
    if (t[i] && t[i]->device() != dev) Py_RETURN_NONE;
  int topk, mode;
  double tau, minr, tol, eps;
  if (!plain_int(a[9], 1, 256, &topk) || !plain_int(a[10], 0, 3, &mode) ||
      !plain_float(a[11], &tau) || !plain_float(a[12], &minr) || !plain_float(a[13], &tol) ||
      !plain_float(a[14], &eps) || !(tau >= 0 && tau <= 1) || !(eps >= 0 && eps <= 1) ||
      (mode >= 2 && !t[8]))
    Py_RETURN_NONE;
  const int64_t sp = t[8] ? t[8]->size(2) : 0;
  const auto f = q.options().dtype(at::kFloat).requires_grad(false);
  const at::Tensor sel = at::empty({r, hq, topk}, f.dtype(at::kInt));
  at::Tensor m, l, u;
  if (sp) {
    m = at::empty({r, hq, sp}, f);
    l = at::empty({r, hq, sp}, f);
    u = at::empty({r, hq, sp, d}, f);
  }
  const at::Tensor out = at::empty({r, hq, d}, f);
  const size_t bytes = g_entry.paged_workspace((int)r, (int)hq, (int)width);
  const at::Tensor ws = at::empty({(int64_t)(bytes ? bytes : 1)}, f.dtype(at::kByte));
  auto fp = [](const at::Tensor& x) { return x.defined() ? x.data_ptr<float>() : nullptr; };
  const int32_t* nt = t[7] ? t[7]->data_ptr<int32_t>() : nullptr;
  const int32_t* p = t[8] ? t[8]->data_ptr<int32_t>() : nullptr;
  const int lb = lo.scalar_type() == at::kFloat ? 0 : dt;
  void* st = stream_of(q);
  int rc;
  if (mode < 2) {
    Py_BEGIN_ALLOW_THREADS
    rc = g_entry.paged_step(q.data_ptr(), k.data_ptr(), v.data_ptr(), dt, (int)r, (int)hq,
                            (int)hkv, (int)width, (int)b, (int)d, (int)pages, lo.data_ptr(),
                            hi.data_ptr(), lb, tab.data_ptr<int32_t>(),
                            nbk.data_ptr<int32_t>(), nt, topk, p, (int)sp, mode,
                            sel.data_ptr<int32_t>(), fp(m), fp(l), fp(u),
                            out.data_ptr<float>(), ws.data_ptr(), bytes, st);
    Py_END_ALLOW_THREADS
    if (rc) return PyLong_FromLong(rc);
    return pack({&sel, &m, &l, &u, &out});
  }
  const at::Tensor bad = at::empty({r, hq}, f.dtype(at::kBool)), rem = at::empty({r, hq}, f);
  at::Tensor approx, extra;
  if (eps > 0) {
    approx = at::empty({r, hq}, f.dtype(at::kBool));
    extra = at::empty({r, hq}, f);
  }
  const at::Tensor pos = at::empty({r, hq}, f.dtype(at::kInt));
  const at::Tensor tot = at::empty({r, hq}, f.dtype(at::kInt));
  Py_BEGIN_ALLOW_THREADS
  rc = g_entry.paged_signed(
      q.data_ptr(), k.data_ptr(), v.data_ptr(), dt, (int)r, (int)hq, (int)hkv, (int)width,
      (int)b, (int)d, (int)pages, lo.data_ptr(), hi.data_ptr(), lb, tab.data_ptr<int32_t>(),
      nbk.data_ptr<int32_t>(), nt, topk, p, (int)sp, mode == 3, (float)tau, (float)minr,
      (float)tol, (float)eps, sel.data_ptr<int32_t>(), fp(m), fp(l), fp(u),
      out.data_ptr<float>(), static_cast<uint8_t*>(bad.data_ptr()), rem.data_ptr<float>(),
      approx.defined() ? static_cast<uint8_t*>(approx.data_ptr()) : nullptr, fp(extra),
      pos.data_ptr<int32_t>(), tot.data_ptr<int32_t>(), ws.data_ptr(), bytes, st);
  Py_END_ALLOW_THREADS
  if (rc) return PyLong_FromLong(rc);
  return pack({&sel, &m, &l, &u, &out, &bad, &rem, &approx, &extra, &pos, &tot});
}

PyObject* speculative_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return checked([&] { return step_impl(a, n); });
}

PyObject* paged_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return checked([&] { return paged_impl(a, n); });
}

// bind(step_supported, step_workspace, step, paged_workspace, paged_step,
// paged_signed): the C entry points' addresses
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 6) {
    PyErr_SetString(PyExc_TypeError, "bind takes six addresses");
    return nullptr;
  }
  void* p[6];
  for (int i = 0; i < 6; ++i) {
    p[i] = PyLong_AsVoidPtr(a[i]);
    if (!p[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
      return nullptr;
    }
  }
  memcpy(&g_entry, p, sizeof(g_entry));
  g_bound = true;
  Py_RETURN_NONE;
}

PyObject* prepared(PyObject*, PyObject* o) {
  int idx;
  if (plain_int(o, 0, 63, &idx)) g_prepared |= 1ull << idx;
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"speculative_step", (PyCFunction)(void (*)())speculative_step, METH_FASTCALL, nullptr},
    {"paged_step", (PyCFunction)(void (*)())paged_step, METH_FASTCALL, nullptr},
    {"bind", (PyCFunction)(void (*)())bind, METH_FASTCALL, nullptr},
    {"prepared", (PyCFunction)prepared, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

// torch_version: the torch that the module was built for
PyMODINIT_FUNC PyInit__host(void) {
  PyObject* m = PyModule_Create(&kModule);
  if (m && PyModule_AddStringConstant(m, "torch_version", STK_TORCH_VERSION)) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
