// The calls that a program makes per product, without the interpreter between them: tensor checks, output and chunk
// allocation, pointer tables and the C entry point in one native call each.
//
// Every function here takes the ordinary case only (plain dense GPU tensors on the current device, lists or tuples of equal
// slices, no tracing, no capture where a workspace would have to come from the graph's pool) and returns None for everything
// else, invalid arguments among it: the caller then takes the Python path, which says what is wrong or handles the rest.
// Nothing is kept between calls but the workspaces that local_gemm.workspace() announces (workspace_set / workspace_drop).  The interpreter
// lock is released while an output is allocated and a product launched: either may wait for the device (a full queue, an allocator that has
// to free), and another Python thread may be the one that raises the flag that the device waits for.  So everything that is needed of the
// Python objects is read before, and a call holds the storage of its workspace until its launch has been queued.
#include <Python.h>

#include <ATen/Functions.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "meshslice_hip.h"

namespace {

struct Workspace {
  int device = -1;
  void *stream = nullptr;
  c10::Storage hold;
  void *ptr = nullptr;
  size_t bytes = 0;
  unsigned long long used = 0;      // when the last call took it
};
constexpr int MAX_WORKSPACES = 256;
Workspace *const g_ws = new Workspace[MAX_WORKSPACES];      // (never destroyed: the allocator may be gone by then)
int g_ws_count = 0;
unsigned long long g_clock = 0;

Workspace *find_workspace(int device, void *stream) {
  for (int i = 0; i < g_ws_count; i++)
    if (g_ws[i].device == device && g_ws[i].stream == stream) return &g_ws[i];
  return nullptr;
}

// the interpreter lock is released for the life of one of these
struct Unlocked {
  PyThreadState *state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
  Unlocked() = default;
  Unlocked(const Unlocked &) = delete;
};

int code_of(const at::Tensor &t) {
  return t.scalar_type() == at::kBFloat16 ? MS_DTYPE_BF16 : t.scalar_type() == at::kFloat ? MS_DTYPE_F32 : -1;
}

// what a call needs of a matrix once the lock is released
struct Mat {
  char *ptr;
  int64_t rows, cols;
  int ld, code;
  at::TensorOptions options;
  explicit Mat(const at::Tensor &t)
      : ptr(static_cast<char *>(t.data_ptr())), rows(t.size(0)), cols(t.size(1)), ld((int)t.stride(0)), code(code_of(t)), options(t.options().requires_grad(false)) {}
};

// a row-major matrix in plain GPU memory, or null
const at::Tensor *matrix(PyObject *o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  if (!t.is_cuda() || t.dim() != 2 || t.layout() != at::kStrided || code_of(t) < 0 || t.stride(1) != 1) return nullptr;
  if (t.stride(0) > INT32_MAX || t.size(0) > INT32_MAX || t.size(1) > INT32_MAX || t.stride(0) < 0) return nullptr;
  using c10::DispatchKey;
  const auto ks = t.key_set();
  for (DispatchKey k : {DispatchKey::Python, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper, DispatchKey::Functionalize,
                        DispatchKey::Negative, DispatchKey::Conjugate, DispatchKey::ZeroTensor, DispatchKey::Fake})
    if (ks.has(k)) return nullptr;
  return &t;
}

// `n` equal matrices of a list or tuple: their addresses go to `ptrs`; the first of them, or null
const at::Tensor *matrices(PyObject *seq, void **ptrs, int *n) {
  if (!PyList_CheckExact(seq) && !PyTuple_CheckExact(seq)) return nullptr;
  const Py_ssize_t count = PySequence_Fast_GET_SIZE(seq);
  if (count < 1 || count + *n > MS_MAX_SLICES) return nullptr;
  PyObject **items = PySequence_Fast_ITEMS(seq);
  const at::Tensor *first = nullptr;
  for (Py_ssize_t i = 0; i < count; i++) {
    const at::Tensor *t = matrix(items[i]);
    if (!t) return nullptr;
    if (!first) first = t;
    else if (t->size(0) != first->size(0) || t->size(1) != first->size(1) || t->stride(0) != first->stride(0) ||
             t->scalar_type() != first->scalar_type() || t->device() != first->device()) return nullptr;
    ptrs[(*n)++] = t->data_ptr();
  }
  return first;
}

// where a call on tensor `t` runs
struct Place {
  int device = -1;
  hipStream_t stream = nullptr;
  bool ok = false;
};
Place place_of(const at::Tensor &t) {
  Place p;
  if (at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set()) return p;
  p.device = t.device().index();
  if (p.device != c10::hip::current_device()) return p;
  p.stream = c10::hip::getCurrentHIPStream(p.device).stream();
  p.ok = true;
  return p;
}
// the workspace of that place, or one without storage: none yet, or a capture is under way (its workspaces come from the graph's pool)
Workspace workspace_of(const Place &p) {
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(p.stream, &capturing) != hipSuccess) {
    (void)hipGetLastError();      // (not for the next launch to find)
    return Workspace();
  }
  if (capturing != hipStreamCaptureStatusNone) return Workspace();
  Workspace *w = find_workspace(p.device, p.stream);
  if (!w) return Workspace();
  w->used = ++g_clock;
  return *w;
}

// the dtype named by `o` (None: `otherwise`), or -1 for one that the kernels do not write
int wanted_dtype(PyObject *o, int otherwise) {
  if (o == Py_None) return otherwise;
  if (!THPDtype_Check(o)) return -1;
  const auto st = reinterpret_cast<THPDtype *>(o)->scalar_type;
  return st == at::kBFloat16 ? MS_DTYPE_BF16 : st == at::kFloat ? MS_DTYPE_F32 : -1;
}
at::ScalarType type_of(int code) { return code == MS_DTYPE_BF16 ? at::kBFloat16 : at::kFloat; }

PyObject *chunk_list(const at::Tensor &buf) {
  const int64_t n = buf.size(0);
  PyObject *list = PyList_New(n);
  if (!list) return nullptr;
  for (int64_t i = 0; i < n; i++) PyList_SET_ITEM(list, i, THPVariable_Wrap(buf.select(0, i)));
  return list;
}
void chunk_pointers(const at::Tensor &buf, void **ptrs) {
  char *base = static_cast<char *>(buf.data_ptr());
  const int64_t step = buf.stride(0) * buf.element_size();
  for (int64_t i = 0; i < buf.size(0); i++) ptrs[i] = base + i * step;
}

// gemm_os(A_slices, B_slices, out_dtype, gelu, residual) -> Tensor or None
PyObject *gemm_os(PyObject *const *args) {
  const void *a[MS_MAX_SLICES], *b[MS_MAX_SLICES];
  int na = 0, nb = 0;
  const at::Tensor *a0 = matrices(args[0], const_cast<void **>(a), &na), *b0 = a0 ? matrices(args[1], const_cast<void **>(b), &nb) : nullptr;
  if (!b0 || na != nb || a0->size(1) != b0->size(0) || a0->scalar_type() != b0->scalar_type() || a0->device() != b0->device()) return nullptr;
  const int in = code_of(*a0), outc = wanted_dtype(args[2], in);
  if (outc < 0) return nullptr;
  const Mat A(*a0), B(*b0);
  const int64_t m = A.rows, n = B.cols;
  const void *res = nullptr;
  int ldr = 0;
  if (args[4] != Py_None) {
    const at::Tensor *r = matrix(args[4]);
    if (!r || r->size(0) != m || r->size(1) != n || code_of(*r) != outc || r->device() != a0->device()) return nullptr;
    res = r->data_ptr();
    ldr = (int)r->stride(0);
  }
  const Place p = place_of(*a0);
  const Workspace ws = p.ok ? workspace_of(p) : Workspace();
  if (!ws.ptr) return nullptr;
  at::Tensor out;
  int rc;
  {
    Unlocked u;
    out = at::empty({m, n}, A.options.dtype(type_of(outc)));
    rc = ms_gemm_os_ws(a, b, na, (int)m, (int)n, (int)A.cols, A.ld, B.ld, out.data_ptr(), (int)n, in, outc, args[3] == Py_True ? MS_ACT_GELU : MS_ACT_NONE,
                       res, ldr, nullptr, nullptr, ws.ptr, ws.bytes, p.stream);
  }
  return rc == MS_OK ? THPVariable_Wrap(std::move(out)) : nullptr;
}

// gemm_os_cyclic(A_slices, W) -> Tensor or None
PyObject *gemm_os_cyclic(PyObject *const *args) {
  const void *a[MS_MAX_SLICES];
  int S = 0;
  const at::Tensor *a0 = matrices(args[0], const_cast<void **>(a), &S), *w = a0 ? matrix(args[1]) : nullptr;
  if (!w || a0->size(1) * S != w->size(0) || a0->scalar_type() != w->scalar_type() || a0->device() != w->device()) return nullptr;
  const Place p = place_of(*a0);
  const Workspace ws = p.ok ? workspace_of(p) : Workspace();
  if (!ws.ptr) return nullptr;
  const Mat A(*a0), W(*w);
  at::Tensor out;
  int rc;
  {
    Unlocked u;
    out = at::empty({A.rows, W.cols}, W.options);
    rc = ms_gemm_os_cyclic(a, W.ptr, S, (int)A.rows, (int)W.cols, (int)A.cols, A.ld, W.ld, out.data_ptr(), (int)W.cols, W.code, W.code, ws.ptr, ws.bytes, p.stream);
  }
  return rc == MS_OK ? THPVariable_Wrap(std::move(out)) : nullptr;
}

// gemm_ls(A, W_slices, out_dtype) / gemm_rs(X_slices, W, out_dtype) -> [chunks] or None
template <bool LS>
PyObject *gemm_chunks(PyObject *const *args) {
  const void *cut[MS_MAX_SLICES];
  void *y[MS_MAX_SLICES];
  int S = 0;
  const at::Tensor *own = matrix(args[LS ? 0 : 1]), *c0 = own ? matrices(args[LS ? 1 : 0], const_cast<void **>(cut), &S) : nullptr;
  if (!c0 || own->scalar_type() != c0->scalar_type() || own->device() != c0->device() || own->size(LS ? 1 : 0) != c0->size(LS ? 1 : 0)) return nullptr;
  const int in = code_of(*own), outc = wanted_dtype(args[2], MS_DTYPE_F32);
  if (outc < 0) return nullptr;
  const Place p = place_of(*own);
  if (!p.ok) return nullptr;
  const Mat O(*own), C(*c0);
  const int64_t m = LS ? O.rows : C.cols, n = LS ? C.rows : O.cols, k = LS ? O.cols : O.rows;
  at::Tensor buf;
  int rc;
  {
    Unlocked u;
    buf = at::empty({S, m, n}, O.options.dtype(type_of(outc)));
    chunk_pointers(buf, y);
    rc = LS ? ms_gemm_ls_ex(O.ptr, O.ld, cut, C.ld, S, (int)m, (int)n, (int)k, y, (int)n, in, outc, p.stream)
            : ms_gemm_rs_ex(cut, C.ld, O.ptr, O.ld, S, (int)m, (int)n, (int)k, y, (int)n, in, outc, p.stream);
  }
  return rc == MS_OK ? chunk_list(buf) : nullptr;
}

// gemm_ls_cyclic(A, W, S) -> [chunks] or None
PyObject *gemm_ls_cyclic(PyObject *const *args) {
  void *y[MS_MAX_SLICES];
  const at::Tensor *a = matrix(args[0]), *w = a ? matrix(args[1]) : nullptr;
  const long S = PyLong_AsLong(args[2]);
  if (!w || S < 1 || S > MS_MAX_SLICES || w->size(0) % S || a->size(1) != w->size(1) || a->scalar_type() != w->scalar_type() || a->device() != w->device()) return nullptr;
  const Place p = place_of(*a);
  if (!p.ok) return nullptr;
  const Mat A(*a), W(*w);
  const int64_t n = W.rows / S;
  at::Tensor buf;
  int rc;
  {
    Unlocked u;
    buf = at::empty({S, A.rows, n}, A.options.dtype(type_of(MS_DTYPE_F32)));
    chunk_pointers(buf, y);
    rc = ms_gemm_ls_cyclic(A.ptr, A.ld, W.ptr, W.ld, (int)S, (int)A.rows, (int)n, (int)A.cols, y, (int)n, A.code, MS_DTYPE_F32, p.stream);
  }
  return rc == MS_OK ? chunk_list(buf) : nullptr;
}

// gemm_ls_sum(X, W, P) / gemm_rs_sum(X, W, P) -> Tensor or None
template <bool LS>
PyObject *gemm_sum(PyObject *const *args) {
  const at::Tensor *x = matrix(args[0]), *w = x ? matrix(args[1]) : nullptr;
  const long P = PyLong_AsLong(args[2]);
  constexpr int C = LS ? 1 : 0;      // the contracted extent of both
  if (!w || P < 1 || P > MS_MAX_SLICES || x->size(C) != w->size(C) || x->size(C) % P || x->scalar_type() != w->scalar_type() || x->device() != w->device())
    return nullptr;
  const Place p = place_of(*x);
  const Workspace ws = p.ok ? workspace_of(p) : Workspace();
  if (!ws.ptr) return nullptr;
  const Mat X(*x), W(*w);
  const int64_t k = x->size(C) / P, m = x->size(1 - C), n = w->size(1 - C), es = x->element_size();
  const void *xs[MS_MAX_SLICES], *wsh[MS_MAX_SLICES];
  for (long i = 0; i < P; i++) {
    xs[i] = X.ptr + i * k * es * (LS ? 1 : X.ld);
    wsh[i] = W.ptr + i * k * es * (LS ? 1 : W.ld);
  }
  at::Tensor out;
  int rc;
  {
    Unlocked u;
    out = at::empty({m, n}, X.options);
    rc = (LS ? ms_gemm_ls_sum : ms_gemm_rs_sum)(xs, X.ld, wsh, W.ld, (int)P, (int)m, (int)n, (int)k, out.data_ptr(), (int)n, X.code, X.code, ws.ptr, ws.bytes, p.stream);
  }
  return rc == MS_OK ? THPVariable_Wrap(std::move(out)) : nullptr;
}

// prefers_sum(rs, P, S, m, n, k) -> bool
PyObject *prefers_sum(PyObject *const *args) {
  int v[6];
  for (int i = 0; i < 6; i++) {
    const long x = PyLong_AsLong(args[i]);
    if (x < 0 || x > INT32_MAX) return nullptr;
    v[i] = (int)x;
  }
  return PyBool_FromLong(ms_prefers_sum(v[0], v[1], v[2], v[3], v[4], v[5]));
}

// pack_slices(block, S, B, axis) -> [slices] or None
PyObject *pack_slices(PyObject *const *args) {
  const at::Tensor *t = matrix(args[0]);
  const long S = PyLong_AsLong(args[1]), B = PyLong_AsLong(args[2]), axis = PyLong_AsLong(args[3]);
  if (!t || S < 1 || S > MS_MAX_SLICES || B < 1 || B > INT32_MAX || (axis != 0 && axis != 1)) return nullptr;
  const int64_t r = t->size(0), c = t->size(1), cut = axis == 1 ? c : r;
  if (r < 1 || c < 1 || cut % (S * B)) return nullptr;
  const Place p = place_of(*t);
  if (!p.ok) return nullptr;
  const Mat T(*t);
  void *d[MS_MAX_SLICES];
  at::Tensor buf;
  int rc;
  {
    Unlocked u;
    buf = at::empty({S, axis == 1 ? r : r / S, axis == 1 ? c / S : c}, T.options);
    chunk_pointers(buf, d);
    rc = ms_pack_slices(T.ptr, T.ld, (int)r, (int)c, (int)axis, (int)S, (int)B, d, (int)buf.size(2), T.code, p.stream);
  }
  return rc == MS_OK ? chunk_list(buf) : nullptr;
}

// unpack_chunks(chunks_by_peer, B, axis, window, parts, out_dtype) -> Tensor or None
PyObject *unpack_chunks(PyObject *const *args) {
  if (!PyList_CheckExact(args[0]) && !PyTuple_CheckExact(args[0])) return nullptr;
  const Py_ssize_t P = PySequence_Fast_GET_SIZE(args[0]);
  PyObject **peers = PySequence_Fast_ITEMS(args[0]);
  const long B = PyLong_AsLong(args[1]), axis = PyLong_AsLong(args[2]), window = PyLong_AsLong(args[3]), parts = PyLong_AsLong(args[4]);
  if (P < 1 || B < 1 || (axis != 0 && axis != 1) || parts < 1 || window < 0 || window >= parts) return nullptr;
  void *src[MS_MAX_SLICES];
  int n = 0, S = 0;
  const at::Tensor *c0 = nullptr;
  for (Py_ssize_t q = 0; q < P; q++) {
    const int before = n;
    const at::Tensor *c = matrices(peers[q], src, &n);
    if (!c) return nullptr;
    if (q == 0) { c0 = c; S = n; }
    else if (n - before != S || c->size(0) != c0->size(0) || c->size(1) != c0->size(1) || c->stride(0) != c0->stride(0) ||
             c->scalar_type() != c0->scalar_type() || c->device() != c0->device()) return nullptr;
  }
  const int in = code_of(*c0), outc = wanted_dtype(args[5], in);
  const int64_t cr = c0->size(0), cc = c0->size(1), cut = axis == 1 ? cc : cr;
  if (outc < 0 || cr < 1 || cc < 1 || cut % parts || (cut / parts) % B) return nullptr;
  const int64_t keep = cut / parts, rows = axis == 1 ? cr : keep * S, cols = axis == 1 ? keep * S : cc;
  if (rows > INT32_MAX || cols > INT32_MAX || rows < 1 || cols < 1) return nullptr;
  const Place p = place_of(*c0);
  if (!p.ok) return nullptr;
  const Mat C(*c0);
  at::Tensor out;
  int rc;
  {
    Unlocked u;
    out = at::empty({rows, cols}, C.options.dtype(type_of(outc)));
    rc = ms_unpack_chunks(src, (int)P, S, C.ld, axis == 1 ? 0 : (int)(window * keep), axis == 1 ? (int)(window * keep) : 0, (int)rows, (int)cols, (int)axis, (int)B,
                          out.data_ptr(), (int)cols, in, outc, p.stream);
  }
  return rc == MS_OK ? THPVariable_Wrap(std::move(out)) : nullptr;
}

// One Python entry per function: argument count, the conversion of C++ exceptions (an allocation that does not fit, say) to
// "not taken" -- the Python path then meets them itself -- and of a missing result to None.
typedef PyObject *(*Impl)(PyObject *const *);
template <Impl F, int NARGS>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != NARGS) {
    PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", NARGS, n);
    return nullptr;
  }
  PyObject *r = nullptr;
  try {
    r = F(args);
  } catch (...) {
    r = nullptr;
  }
  if (r) return r;
  PyErr_Clear();
  Py_RETURN_NONE;
}

// workspace_set(device, stream, tensor); workspace_drop(device, stream); workspace_touch(device, stream, touch = True) -> when it was used last
PyObject *workspace_set(PyObject *, PyObject *args) {
  int device;
  unsigned long long stream;
  PyObject *o;
  if (!PyArg_ParseTuple(args, "iKO", &device, &stream, &o)) return nullptr;
  if (!THPVariable_Check(o)) {
    PyErr_SetString(PyExc_TypeError, "a workspace is a tensor");
    return nullptr;
  }
  const at::Tensor &t = THPVariable_Unpack(o);
  Workspace *w = find_workspace(device, reinterpret_cast<void *>(stream));
  if (!w && g_ws_count < MAX_WORKSPACES) w = &g_ws[g_ws_count++];
  if (w) *w = Workspace{device, reinterpret_cast<void *>(stream), t.storage(), t.data_ptr(), (size_t)t.nbytes(), ++g_clock};
  Py_RETURN_NONE;
}
PyObject *workspace_drop(PyObject *, PyObject *args) {
  int device;
  unsigned long long stream;
  if (!PyArg_ParseTuple(args, "iK", &device, &stream)) return nullptr;
  if (Workspace *w = find_workspace(device, reinterpret_cast<void *>(stream))) {
    *w = g_ws[--g_ws_count];
    g_ws[g_ws_count] = Workspace();
  }
  Py_RETURN_NONE;
}
PyObject *workspace_touch(PyObject *, PyObject *args) {
  int device, touch = 1;
  unsigned long long stream;
  if (!PyArg_ParseTuple(args, "iK|p", &device, &stream, &touch)) return nullptr;
  Workspace *w = find_workspace(device, reinterpret_cast<void *>(stream));
  if (w && touch) w->used = ++g_clock;
  return PyLong_FromUnsignedLongLong(w ? w->used : 0);
}

#define MS_ENTRY(name, impl, nargs) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<impl, nargs>)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {
    MS_ENTRY("gemm_os", gemm_os, 5),
    MS_ENTRY("gemm_os_cyclic", gemm_os_cyclic, 2),
    MS_ENTRY("gemm_ls", gemm_chunks<true>, 3),
    MS_ENTRY("gemm_rs", gemm_chunks<false>, 3),
    MS_ENTRY("gemm_ls_cyclic", gemm_ls_cyclic, 3),
    MS_ENTRY("gemm_ls_sum", gemm_sum<true>, 3),
    MS_ENTRY("gemm_rs_sum", gemm_sum<false>, 3),
    MS_ENTRY("prefers_sum", prefers_sum, 6),
    MS_ENTRY("pack_slices", pack_slices, 4),
    MS_ENTRY("unpack_chunks", unpack_chunks, 6),
    {"workspace_set", workspace_set, METH_VARARGS, nullptr},
    {"workspace_drop", workspace_drop, METH_VARARGS, nullptr},
    {"workspace_touch", workspace_touch, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host", "native call path of meshslice_amd", -1, g_methods};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&g_module); }
