// The host side of the launches that a prompt step makes most, in C++: what `HipKernels.linear`, `linear_swiglu`, `rmsnorm`,
// `attention` (prompts) and `rope_store_pieces` check of their tensors before they call the library.  A prompt of a few words to a
// small model is bound by this: 138 launches of 10 to 20 microseconds of Python each.
//
// Every function returns 1 when it has launched, 0 when something is not as the launch wants it (the caller's Python checks then
// say what, or take another way: nothing was launched), or the library's negative code.  It keeps nothing of its arguments and
// nothing between calls but the library's addresses, given once.
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>

namespace {

typedef int (*LinearFn)(const void*, const void*, void*, int, int, int, int, int, int, int, int, int, long long, int, int, void*);
typedef int (*SplitsFn)(int, int, int, int, int);
typedef int (*SwigluFn)(const void*, const void*, void*, int, int, int, int, int, int, int, int, int, int, void*);
typedef int (*RmsnormFn)(void*, const void*, int, int, long long, const void*, float, void*, int, int, int, void*);
typedef int (*AttentionFn)(const void*, int, void*, int, int, int, int, int, int, int, const void*, const void*, const void*, const void*,
                           const void*, int, const void*, const void*, int, float, int, int, int, void*, long long, void*, long long,
                           const void*, const void*, int, int, const void*, int, int, long long, int, void*);
typedef int (*RopePiecesFn)(const void*, int, int, long long, void*, int, int, int, int, int, const void*, const void*, const void*,
                            const void*, const void*, int, void*, void*, int, void*);

LinearFn lq_linear;
SplitsFn lq_linear_splits, lq_linear_narrow_splits;
SwigluFn lq_linear_swiglu;
RmsnormFn lq_rmsnorm;
AttentionFn lq_attention;
RopePiecesFn lq_rope_store_pieces;
PyObject *str_data, *str_packed, *str_shape, *str_whole;

// A tensor on the GPU that a kernel can read by address.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_Check(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() ? &t : nullptr;
}

int code(const at::Tensor& t) { return t.scalar_type() == at::kFloat ? 0 : t.scalar_type() == at::kBFloat16 ? 1 : -1; }

struct Matrix {  // dense rows `ld` entries apart
  char* at = nullptr;
  long long rows = 0, cols = 0, ld = 0;
  int type = -1;
  bool packed = false;
};

bool matrix(const at::Tensor& t, Matrix& m) {
  if (t.dim() != 2 || (t.stride(1) != 1 && t.size(1) != 1)) return false;
  m.rows = t.size(0), m.cols = t.size(1), m.type = code(t), m.at = (char*)t.data_ptr();
  m.ld = m.rows > 1 ? t.stride(0) : std::max<long long>(t.stride(0), m.cols);
  const long long most = 0x7fffffff;
  return m.type >= 0 && m.rows <= most && m.cols <= most && m.ld <= most;
}
bool matrix(PyObject* o, Matrix& m) {
  const at::Tensor* t = plain(o);
  return t != nullptr && matrix(*t, m);
}

// A weight: a tensor, or the object that holds one in the packed order (its data, shape and the whole matrix's columns).
bool weight(PyObject* o, Matrix& m) {
  if (THPVariable_Check(o)) return matrix(o, m);
  PyObject *packed = PyObject_GetAttr(o, str_packed), *data = packed ? PyObject_GetAttr(o, str_data) : nullptr,
           *shape = data ? PyObject_GetAttr(o, str_shape) : nullptr, *whole = shape ? PyObject_GetAttr(o, str_whole) : nullptr;
  bool ok = whole != nullptr && packed == Py_True && PyTuple_Check(shape) && PyTuple_GET_SIZE(shape) == 2;
  const at::Tensor* t = ok ? plain(data) : nullptr;
  if (t != nullptr) {
    m.at = (char*)t->data_ptr(), m.type = code(*t), m.packed = true;
    m.rows = PyLong_AsLongLong(PyTuple_GET_ITEM(shape, 0)), m.cols = PyLong_AsLongLong(PyTuple_GET_ITEM(shape, 1));
    m.ld = PyLong_AsLongLong(whole);
    if (m.rows == 1) m.ld = std::max(m.ld, m.cols);
    ok = m.type >= 0;
  } else {
    ok = false;
  }
  Py_XDECREF(packed), Py_XDECREF(data), Py_XDECREF(shape), Py_XDECREF(whole);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return ok;
}

bool ints(PyObject* o, long long n, const void*& at) {  // a dense int32 tensor of n entries or more
  const at::Tensor* t = plain(o);
  if (t == nullptr || t->scalar_type() != at::kInt || !t->is_contiguous() || t->numel() < n) return false;
  at = t->data_ptr();
  return true;
}

bool is(const at::Tensor& t, std::initializer_list<long long> sizes) {
  return t.dim() == (long long)sizes.size() && std::equal(sizes.begin(), sizes.end(), t.sizes().begin());
}

// A delta shaped like x [rows, width], or pieces of one: its address, how many and how far apart.
bool pieces_of(PyObject* o, const Matrix& x, const void*& at, int& type, int& n, long long& apart) {
  at = nullptr, type = 0, n = 0, apart = 0;
  if (o == Py_None) return true;
  const at::Tensor* t = plain(o);
  if (t == nullptr || !t->is_contiguous() || t->dim() < 2 || t->dim() > 3 || t->size(-1) != x.cols || t->size(-2) != x.rows) return false;
  at = t->data_ptr(), type = code(*t), n = t->dim() == 3 ? (int)t->size(0) : 1, apart = t->dim() == 3 ? x.rows * x.cols : 0;
  return type >= 0;
}

// Python's lock, given back while a launch is made (it waits where the stream's queue is full).
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename F>
int launch(F f) {
  Unlocked unlocked;
  return f() ?: 1;
}

long long number(PyObject* o) { return PyLong_AsLongLong(o); }
void* address(PyObject* o) { return (void*)PyLong_AsUnsignedLongLong(o); }

// linear(x, w, out, generic, stream)
int linear(PyObject* const* a) {
  Matrix x, w, out;
  if (!matrix(a[0], x) || !weight(a[1], w)) return 0;
  const at::Tensor* o = plain(a[2]);
  const int generic = (int)number(a[3]);
  void* stream = address(a[4]);
  if (o == nullptr || PyErr_Occurred()) return 0;
  int pieces = 1;
  long long apart = 0;
  if (o->dim() == 3) {
    if (!o->is_contiguous() || code(*o) < 0) return 0;
    pieces = (int)o->size(0), apart = x.rows * w.rows;
    out.at = (char*)o->data_ptr(), out.type = code(*o), out.rows = o->size(1), out.cols = out.ld = o->size(2);
    if (pieces != lq_linear_splits(x.type, (int)x.rows, (int)w.rows, (int)x.cols, generic) &&
        pieces != lq_linear_narrow_splits(x.type, (int)x.rows, (int)w.rows, (int)x.cols, generic))
      return 0;
  } else if (!matrix(*o, out)) {
    return 0;
  }
  if (w.cols != x.cols || out.rows != x.rows || out.cols != w.rows || x.type != w.type) return 0;
  return launch([&] {
    return lq_linear(x.at, w.at, out.at, x.type, out.type, (int)x.rows, (int)w.rows, (int)x.cols, (int)x.ld, (int)w.ld, (int)out.ld, pieces,
                     apart, generic, w.packed, stream);
  });
}

// linear_swiglu(x, w, out, form, stream)
int linear_swiglu(PyObject* const* a) {
  Matrix x, w, out;
  const int form = (int)number(a[3]);
  void* stream = address(a[4]);
  if (PyErr_Occurred() || !matrix(a[0], x) || !weight(a[1], w) || !matrix(a[2], out)) return 0;
  if (w.cols != x.cols || out.rows != x.rows || out.cols != w.rows / 2 || w.rows % 16 != 0 || x.type != w.type) return 0;
  return launch([&] {
    return lq_linear_swiglu(x.at, w.at, out.at, x.type, out.type, (int)x.rows, (int)w.rows, (int)x.cols, (int)x.ld, (int)w.ld, (int)out.ld,
                            w.packed, form, stream);
  });
}

// rmsnorm(x, weight, eps, out, delta, stream)
int rmsnorm(PyObject* const* a) {
  Matrix x, out;
  const at::Tensor* w = plain(a[1]);
  const void* delta;
  int type, n;
  long long apart;
  const float eps = (float)PyFloat_AsDouble(a[2]);
  void* stream = address(a[5]);
  if (PyErr_Occurred() || !matrix(a[0], x) || !matrix(a[3], out) || w == nullptr || !pieces_of(a[4], x, delta, type, n, apart)) return 0;
  if (x.type != 0 || (x.ld != x.cols && x.rows > 1) || w->scalar_type() != at::kFloat || w->numel() != x.cols || !w->is_contiguous() ||
      out.rows != x.rows || out.cols != x.cols || (out.ld != x.cols && x.rows > 1))
    return 0;
  return launch([&, gain = w->data_ptr()] {
    return lq_rmsnorm(x.at, delta, type, n, apart, gain, eps, out.at, out.type, (int)x.rows, (int)x.cols, stream);
  });
}

// Keys and values in the paged layout, [blocks, kv_heads, block, head] and [blocks, kv_heads, head, block].
bool paged(PyObject* k, PyObject* v, long long kv_heads, long long head, long long block, at::ScalarType type, void*& kp, void*& vp) {
  const at::Tensor *kt = plain(k), *vt = plain(v);
  if (kt == nullptr || vt == nullptr || kt->dim() != 4 || !is(*kt, {kt->size(0), kv_heads, block, head}) ||
      !is(*vt, {kt->size(0), kv_heads, head, block}) || !kt->is_contiguous() || !vt->is_contiguous() || kt->scalar_type() != type ||
      vt->scalar_type() != type)
    return false;
  kp = kt->data_ptr(), vp = vt->data_ptr();
  return true;
}

// attention(q, out, heads, kv_heads, head_dim, row_pos, row_seq, seq_slot, cu_rows, block_table, k, v, block, scale, window, max_len,
// tickets, generic, stream): a prompt's
int attention(PyObject* const* a) {
  Matrix q, out;
  const long long heads = number(a[2]), kv_heads = number(a[3]), head = number(a[4]), block = number(a[12]);
  const long long window = number(a[14]), max_len = number(a[15]), generic = number(a[17]);
  const float scale = (float)PyFloat_AsDouble(a[13]);
  void* stream = address(a[18]);
  if (PyErr_Occurred()) return 0;
  const at::Tensor *slots = plain(a[7]), *table = plain(a[9]), *tickets = plain(a[16]);
  const void *pos, *seq, *cu;
  void *k, *v;
  if (!matrix(a[0], q) || !matrix(a[1], out) || slots == nullptr || table == nullptr || tickets == nullptr) return 0;
  const long long batch = slots->numel();
  if (slots->scalar_type() != at::kInt || (slots->dim() > 0 && slots->stride(-1) != 1 && slots->size(-1) != 1) ||
      table->scalar_type() != at::kInt || table->dim() != 2 || (table->stride(1) != 1 && table->size(1) != 1) ||
      !ints(a[5], q.rows, pos) || !ints(a[6], q.rows, seq) || !ints(a[8], batch + 1, cu) || out.rows != q.rows ||
      out.cols < heads * head || q.cols < heads * head || q.type != out.type ||
      !paged(a[10], a[11], kv_heads, head, block, out.type ? at::kBFloat16 : at::kFloat, k, v))
    return 0;
  void *slot = slots->data_ptr(), *blocks = table->data_ptr(), *counters = tickets->data_ptr();
  const long long ld = table->stride(0), room = tickets->numel();
  return launch([&] {
    return lq_attention(q.at, (int)q.ld, out.at, (int)out.ld, out.type, (int)q.rows, (int)batch, (int)heads, (int)kv_heads, (int)head, pos,
                        seq, slot, cu, blocks, (int)ld, k, v, (int)block, scale, (int)window, 0, (int)max_len, nullptr, 0, counters, room,
                        nullptr, nullptr, 0, 0, nullptr, 0, 1, 0, (int)generic, stream);
  });
}

// rope_store_pieces(qkv, q_out, heads, kv_heads, head_dim, freqs, row_pos, row_seq, seq_slot, block_table, k, v, block, stream)
int rope_store_pieces(PyObject* const* a) {
  Matrix q;
  const long long heads = number(a[2]), kv_heads = number(a[3]), head = number(a[4]), block = number(a[12]);
  void* stream = address(a[13]);
  if (PyErr_Occurred()) return 0;
  const at::Tensor *qkv = plain(a[0]), *freqs = plain(a[5]), *slots = plain(a[8]), *table = plain(a[9]);
  const void *pos, *seq;
  void *k, *v;
  if (qkv == nullptr || freqs == nullptr || slots == nullptr || table == nullptr || !matrix(a[1], q) || qkv->dim() != 3 ||
      qkv->scalar_type() != at::kFloat || !qkv->is_contiguous() || qkv->size(2) != (heads + 2 * kv_heads) * head || q.type != 1 ||
      q.rows != qkv->size(1) || q.cols != heads * head || freqs->scalar_type() != at::kDouble || freqs->numel() != head / 2 ||
      !freqs->is_contiguous() || !ints(a[6], q.rows, pos) || !ints(a[7], q.rows, seq) || slots->scalar_type() != at::kInt ||
      (slots->dim() > 0 && slots->stride(-1) != 1 && slots->size(-1) != 1) || table->scalar_type() != at::kInt || table->dim() != 2 ||
      (table->stride(1) != 1 && table->size(1) != 1) || !paged(a[10], a[11], kv_heads, head, block, at::kBFloat16, k, v))
    return 0;
  void *in = qkv->data_ptr(), *angles = freqs->data_ptr(), *slot = slots->data_ptr(), *blocks = table->data_ptr();
  const long long n = qkv->size(2), pieces = qkv->size(0), apart = qkv->stride(0), ld = table->stride(0);
  return launch([&] {
    return lq_rope_store_pieces(in, (int)n, (int)pieces, apart, q.at, (int)q.ld, (int)q.rows, (int)heads, (int)kv_heads, (int)head, angles,
                                pos, seq, slot, blocks, (int)ld, k, v, (int)block, stream);
  });
}

// A function of N arguments.  What torch throws means "not as the launch wants it": the caller's own checks meet it again.
template <int (*FN)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  int got = 0;
  if (n == N && lq_linear != nullptr) {
    try {
      got = FN(args);
    } catch (...) {
      got = 0;
    }
  }
  PyErr_Clear();  // (a number that was none: nothing was launched)
  return PyLong_FromLong(got);
}

// use(addresses of the seven functions above, in their order)
PyObject* use(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 7) {
    PyErr_SetString(PyExc_TypeError, "seven addresses");
    return nullptr;
  }
  lq_linear_splits = (SplitsFn)address(args[1]), lq_linear_narrow_splits = (SplitsFn)address(args[2]);
  lq_linear_swiglu = (SwigluFn)address(args[3]), lq_rmsnorm = (RmsnormFn)address(args[4]);
  lq_attention = (AttentionFn)address(args[5]), lq_rope_store_pieces = (RopePiecesFn)address(args[6]);
  lq_linear = (LinearFn)address(args[0]);
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

#define LQ_METHOD(NAME, N) {#NAME, (PyCFunction)(void*)(entry<NAME, N>), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {LQ_METHOD(linear, 5),     LQ_METHOD(linear_swiglu, 5),
                         LQ_METHOD(rmsnorm, 6),    LQ_METHOD(attention, 19),
                         LQ_METHOD(rope_store_pieces, 14), {"use", (PyCFunction)(void*)use, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "lqhost", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_lqhost() {
  str_data = PyUnicode_InternFromString("data"), str_packed = PyUnicode_InternFromString("packed");
  str_shape = PyUnicode_InternFromString("shape"), str_whole = PyUnicode_InternFromString("whole");
  return PyModule_Create(&module);
}
