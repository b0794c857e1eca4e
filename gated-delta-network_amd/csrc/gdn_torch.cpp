// Python entry of the operators for the ordinary call: the arguments of
// gdn_amd.decode.kernel / gdn_amd.prefill.kernel checked and unpacked in native
// code, then the C ABI.  A call that needs anything more -- a strided input, a
// scale tensor, a wrapped tensor, a message about what is wrong -- is not
// launched here: the functions return 1 and the Python path takes it from the
// start.
//
// The checks and the unpacking of eleven tensors took the Python path ~6 us a
// call, more than a small decode step takes on the GPU (B = 1: 8.5 -> 4.3 us
// per step back to back).
#include <Python.h>

#include <math.h>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <initializer_list>

#include "gdn_amd.h"

namespace {

constexpr int64_t kD = 128;

// The C ABI of the loaded library (bind()).
decltype(&gdn_decode_fwd) decode_fwd;
decltype(&gdn_decode_fwd_heads) decode_fwd_heads;
decltype(&gdn_decode_multi_fwd) decode_multi_fwd;
decltype(&gdn_prefill_fwd) prefill_fwd;
decltype(&gdn_prefill_fwd_heads) prefill_fwd_heads;
decltype(&gdn_prefill_workspace_bytes_heads) workspace_bytes;

// A plain tensor (no subclass but Parameter) on HIP device `dev`, or nullptr.
const at::Tensor *plain(PyObject *o) {
  return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}

// Dense, of the given type and shape, on device `dev`: its address, else nullptr.
void *address(PyObject *o, at::ScalarType type, c10::Device dev, std::initializer_list<int64_t> shape) {
  const at::Tensor *t = plain(o);
  if (t == nullptr || t->scalar_type() != type || t->device() != dev ||
      t->sizes() != c10::IntArrayRef(shape) || !t->is_contiguous())
    return nullptr;
  return t->data_ptr();
}

// scale as a Python float (0.0: the default) or None; false: something else.
bool read_scale(PyObject *o, float &scale) {
  double s = 0.0;
  if (PyFloat_CheckExact(o))
    s = PyFloat_AS_DOUBLE(o);
  else if (o != Py_None)
    return false;
  if (s == 0.0) s = 1.0 / sqrt(static_cast<double>(kD));
  if (!isfinite(s) || s <= 0.0) return false;
  scale = static_cast<float>(s);
  return true;
}

using Bf = gdn_bf16;

// decode(q, k, v, state, A_log, a, dt_bias, b, scale, output, new_state):
// 0 launched, 1 not an ordinary call, < 0 a GDN_ERR_* status.
int decode(PyObject *const *x) {
  const at::Tensor *q = plain(x[0]), *v = plain(x[2]);
  float scale;
  if (q == nullptr || v == nullptr || q->dim() != 4 || v->dim() != 4 || !q->is_cuda() ||
      !read_scale(x[8], scale))
    return 1;
  const c10::Device dev = q->device();
  const int64_t B = q->size(0), T = q->size(1), hqk = q->size(2), hv = v->size(2);
  if (T < 1 || B > INT_MAX || T > INT_MAX || hqk > INT_MAX || hv > INT_MAX) return 1;
  constexpr auto bf = at::kBFloat16, f32 = at::kFloat;
  const auto *pq = static_cast<Bf *>(address(x[0], bf, dev, {B, T, hqk, kD}));
  const auto *pk = static_cast<Bf *>(address(x[1], bf, dev, {B, T, hqk, kD}));
  const auto *pv = static_cast<Bf *>(address(x[2], bf, dev, {B, T, hv, kD}));
  const auto *ps = x[3] == Py_None ? nullptr : static_cast<float *>(address(x[3], f32, dev, {B, hv, kD, kD}));
  const auto *pA = static_cast<float *>(address(x[4], f32, dev, {hv}));
  const auto *pa = static_cast<Bf *>(address(x[5], bf, dev, {B, T, hv}));
  const auto *pd = static_cast<float *>(address(x[6], f32, dev, {hv}));
  const auto *pb = static_cast<Bf *>(address(x[7], bf, dev, {B, T, hv}));
  auto *po = static_cast<Bf *>(address(x[9], bf, dev, {B, T, hv, kD}));
  auto *pn = static_cast<float *>(address(x[10], f32, dev, {B, hv, kD, kD}));
  // (an empty batch has no addresses: the Python path)
  if (!pq || !pk || !pv || !pA || !pa || !pd || !pb || !po || !pn || (x[3] != Py_None && !ps)) return 1;
  void *stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (hqk != 4 || hv != 8)
    rc = decode_fwd_heads(pq, pk, pv, ps, pA, pa, pd, pb, scale, po, pn, static_cast<int>(B),
                          static_cast<int>(T), static_cast<int>(hqk), static_cast<int>(hv), stream, -1);
  else if (T > 1)
    rc = decode_multi_fwd(pq, pk, pv, ps, pA, pa, pd, pb, scale, po, pn, static_cast<int>(B),
                          static_cast<int>(T), stream, -1);
  else
    rc = decode_fwd(pq, pk, pv, ps, pA, pa, pd, pb, scale, po, pn, static_cast<int>(B), stream);
  Py_END_ALLOW_THREADS
  return rc;
}

// prefill(q, k, v, state, A_log, a, dt_bias, b, cu_seqlens, scale, output,
// new_state, workspace, cached): `cached(device index, stream, bytes)` gives
// the stream's workspace when `workspace` is None.  Results as decode();
// 2: `cached` raised.
int prefill(PyObject *const *x) {
  const at::Tensor *q = plain(x[0]), *v = plain(x[2]), *cu = plain(x[8]);
  float scale;
  if (q == nullptr || v == nullptr || cu == nullptr || q->dim() != 3 || v->dim() != 3 ||
      cu->dim() != 1 || cu->size(0) < 1 || !q->is_cuda() || !read_scale(x[9], scale))
    return 1;
  const c10::Device dev = q->device();
  const int64_t T = q->size(0), N = cu->size(0) - 1, hqk = q->size(1), hv = v->size(1);
  if (hqk < 1 || hv < 1 || hv % hqk != 0 || T > INT_MAX || N > INT_MAX || hv > INT_MAX) return 1;
  constexpr auto bf = at::kBFloat16, f32 = at::kFloat;
  const bool cu64 = cu->scalar_type() == at::kLong;
  const void *pcu = address(x[8], cu64 ? at::kLong : at::kInt, dev, {N + 1});
  const auto *pq = static_cast<Bf *>(address(x[0], bf, dev, {T, hqk, kD}));
  const auto *pk = static_cast<Bf *>(address(x[1], bf, dev, {T, hqk, kD}));
  const auto *pv = static_cast<Bf *>(address(x[2], bf, dev, {T, hv, kD}));
  const auto *ps = x[3] == Py_None ? nullptr : static_cast<float *>(address(x[3], f32, dev, {N, hv, kD, kD}));
  const auto *pA = static_cast<float *>(address(x[4], f32, dev, {hv}));
  const auto *pa = static_cast<Bf *>(address(x[5], bf, dev, {T, hv}));
  const auto *pd = static_cast<float *>(address(x[6], f32, dev, {hv}));
  const auto *pb = static_cast<Bf *>(address(x[7], bf, dev, {T, hv}));
  auto *po = static_cast<Bf *>(address(x[10], bf, dev, {T, hv, kD}));
  auto *pn = static_cast<float *>(address(x[11], f32, dev, {N, hv, kD, kD}));
  if (!pcu || !pq || !pk || !pv || !pA || !pa || !pd || !pb || !po || !pn || (x[3] != Py_None && !ps) ||
      reinterpret_cast<uintptr_t>(po) % 16 != 0)
    return 1;
  void *stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  const size_t need = workspace_bytes(static_cast<int>(T), static_cast<int>(N), static_cast<int>(hqk),
                                      static_cast<int>(hv));
  struct Held {  // given back on every way out, a C++ exception included
    PyObject *o = nullptr;
    ~Held() { Py_XDECREF(o); }
  } held;
  PyObject *ws = x[12];
  if (ws == Py_None) {
    ws = held.o = PyObject_CallFunction(x[13], "iKn", static_cast<int>(dev.index()),
                                        reinterpret_cast<unsigned long long>(stream),
                                        static_cast<Py_ssize_t>(need));
    if (ws == nullptr) return 2;
  }
  const at::Tensor *w = plain(ws);
  int rc = 1;
  if (w != nullptr && w->scalar_type() == at::kByte && w->dim() == 1 && w->device() == dev &&
      w->is_contiguous() && static_cast<size_t>(w->numel()) >= need &&
      reinterpret_cast<uintptr_t>(w->data_ptr()) % 256 == 0) {
    void *pw = w->data_ptr();
    const size_t bytes = static_cast<size_t>(w->numel());
    Py_BEGIN_ALLOW_THREADS
    if (hqk != 4 || hv != 8)
      rc = prefill_fwd_heads(pq, pk, pv, ps, pA, pa, pd, pb, pcu, cu64, static_cast<int>(N),
                             static_cast<int>(T), static_cast<int>(hqk), static_cast<int>(hv), scale, po,
                             pn, pw, bytes, stream, -1, -1, -1);
    else
      rc = prefill_fwd(pq, pk, pv, ps, pA, pa, pd, pb, pcu, cu64, static_cast<int>(N),
                       static_cast<int>(T), scale, po, pn, pw, bytes, stream);
    Py_END_ALLOW_THREADS
  }
  return rc;
}

// A C++ exception (a tensor without storage, ...) leaves the call to the
// Python path, which raises its own error for it.
template <int (*F)(PyObject *const *), Py_ssize_t ARGS>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
  int rc = 1;
  if (n == ARGS) {
    try {
      rc = F(args);
    } catch (...) {
      rc = 1;
    }
  }
  return rc == 2 ? nullptr : PyLong_FromLong(rc);
}

// bind(addresses): the C ABI functions, in the order below, from the library
// that gdn_amd._lib loaded.
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t n) {
  void *p[6];
  if (n != 6) {
    PyErr_SetString(PyExc_TypeError, "bind takes six addresses");
    return nullptr;
  }
  for (int i = 0; i < 6; ++i) {
    p[i] = PyLong_AsVoidPtr(args[i]);
    if (p[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
      return nullptr;
    }
  }
  decode_fwd = reinterpret_cast<decltype(decode_fwd)>(p[0]);
  decode_multi_fwd = reinterpret_cast<decltype(decode_multi_fwd)>(p[1]);
  decode_fwd_heads = reinterpret_cast<decltype(decode_fwd_heads)>(p[2]);
  prefill_fwd = reinterpret_cast<decltype(prefill_fwd)>(p[3]);
  prefill_fwd_heads = reinterpret_cast<decltype(prefill_fwd_heads)>(p[4]);
  workspace_bytes = reinterpret_cast<decltype(workspace_bytes)>(p[5]);
  Py_RETURN_NONE;
}

template <typename F>
PyCFunction method(F f) {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}

PyMethodDef methods[] = {
    {"bind", method(bind), METH_FASTCALL, "the C ABI functions to call"},
    {"decode", method(entry<decode, 11>), METH_FASTCALL, "0 launched, 1 not an ordinary call, < 0 status"},
    {"prefill", method(entry<prefill, 14>), METH_FASTCALL, "0 launched, 1 not an ordinary call, < 0 status"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "ordinary calls of the GDN operators", -1, methods};

}  // namespace

// torch_version: the torch this was compiled against.  Tensors are unpacked by
// that version's layout, so gdn_amd._lib binds the module under no other.
PyMODINIT_FUNC PyInit__native() {
  PyObject *m = PyModule_Create(&module);
  if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", GDN_TORCH_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
