// The entry points of a token step's kernels as Python functions.
//
// A step of one token a sequence is bound by the host: through ctypes an entry point of some thirty arguments
// cost 6 to 7 us, 4 of them for turning Python's numbers and addresses into C's. Here the conversions follow from the entry
// point's own type, and a pointer argument takes the tensor itself (its data_ptr()), a number or None. Two launches of a windowed
// token with the checks before them: 24.5 us through ctypes, 14.4 through this. Latent attention's steps, which are short prompts as
// well, come through here too.
//
// The symbols are libloqa_seqmix.so's, which is loaded before this module; signatures() lets the loader compare the
// types here with those it knows.
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>

#include <exception>
#include <string>
#include <utility>

typedef void* stream_t;

extern "C" {
int loqa_qk_prep_append(const void*, int, long, int, int, int, int, int, const void*, int, int, float, float, int, const void*, void*,
                        void*, int, int, const void*, void*, int, const void*, const void*, int, const void*, long, float, const void*,
                        long, void*, long, int, int, int, int, stream_t);
int loqa_window_attention(const void*, int, const void*, const void*, int, int, const void*, const void*, const void*, int, const void*,
                          const void*, long, float, float, int, int, int, int, int, int, int, int, int, int, void*, long, int, void*,
                          const void*, const void*, stream_t);
int loqa_window_attention_parts(const void*, int, const void*, const void*, int, int, const void*, const void*, const void*, int,
                                const void*, const void*, long, float, float, int, int, int, int, int, int, int, int, int, int, void*,
                                long, int, void*, const void*, const void*, int, long, void*, long, stream_t);
int loqa_delta_prep(const void*, int, long, const void*, const void*, long, int, int, int, int, int, const void*, int, const void*, int,
                    const void*, const void*, const void*, const void*, const void*, int, int, void*, void*, stream_t);
int loqa_delta_scan(const void*, long, int, int, int, int, int, int, int, int, void*, int, const void*, const void*, const void*,
                    const void*, void*, int, int, stream_t);
int loqa_seq_state_save(const void*, int, const void*, int, int, void*, void*, int, int, int, const void*, const void*, const void*, int,
                        stream_t);
int loqa_gated_rmsnorm(const void*, const void*, const void*, int, long, float, void*, int, int, int, int, int, stream_t);
int loqa_latent_attention(const void*, long, long, const void*, long, long, int, const void*, int, int, const void*, const void*,
                          const void*, int, const void*, const void*, int, const void*, float, int, int, int, int, int, int, void*, int,
                          void*, int, int, stream_t);
int loqa_latent_kv(const void*, long, int, int, const void*, int, const void*, const void*, int, int, const void*, int, int, int, int,
                   int, void*, void*, int, stream_t);
int loqa_latent_prefill(const void*, long, const void*, const void*, void*, long, const void*, const void*, const void*, const void*,
                        const void*, float, int, const void*, long, int, int, int, int, int, int, const void*, int, int, int, int,
                        void*, long, void*, long, stream_t);
int loqa_sigmoid_gate(const void*, long, long, int, const void*, long, void*, long, long, int, int, int, stream_t);
int loqa_head_product(const void*, long, long, const void*, int, int, int, int, void*, long, long, stream_t);
int loqa_moe_route(const void*, const void*, const void*, int, int, int, int, int, int, int, float, void*, void*, int, stream_t);
}

namespace {

bool tensor_of(PyObject* o, const at::Tensor** t) {
  if (!THPVariable_CheckExact(o) && !THPVariable_Check(o)) return false;
  *t = &THPVariable_Unpack(o);
  return true;
}

template <typename T> struct Arg;
template <> struct Arg<void*> {
  static constexpr char code = 'p';
  static bool get(PyObject* o, void** v) {
    const at::Tensor* t;
    if (o == Py_None) *v = nullptr;
    else if (PyLong_Check(o)) *v = PyLong_AsVoidPtr(o);
    else if (tensor_of(o, &t)) *v = t->data_ptr();
    else PyErr_SetString(PyExc_TypeError, "a tensor, an address or None");
    return !PyErr_Occurred();
  }
};
template <> struct Arg<const void*> : Arg<void*> {
  static bool get(PyObject* o, const void** v) { return Arg<void*>::get(o, const_cast<void**>(v)); }
};
template <> struct Arg<long> {
  static constexpr char code = 'l';
  static bool get(PyObject* o, long* v) {
    *v = PyLong_AsLong(o);
    return *v != -1 || !PyErr_Occurred();
  }
};
template <> struct Arg<int> {
  static constexpr char code = 'i';
  static bool get(PyObject* o, int* v) {
    long x;
    if (!Arg<long>::get(o, &x)) return false;
    *v = (int)x;
    if (*v != x) PyErr_SetString(PyExc_OverflowError, "an argument is out of the range of an int");
    return *v == x;
  }
};
template <> struct Arg<float> {
  static constexpr char code = 'f';
  static bool get(PyObject* o, float* v) {
    const double x = PyFloat_AsDouble(o);
    *v = (float)x;
    return x != -1.0 || !PyErr_Occurred();
  }
};

template <auto F> struct Entry;
template <typename... A, int (*F)(A...)> struct Entry<F> {
  static std::string signature() { return {Arg<A>::code...}; }
  template <size_t... I> static PyObject* run(PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<A...> v;
    if (!(Arg<A>::get(args[I], &std::get<I>(v)) && ...)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = F(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
  }
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "takes %d arguments, got %d", (int)sizeof...(A), (int)n);
    try {
      return run(args, std::index_sequence_for<A...>{});
    } catch (const std::exception& e) {          // a tensor without storage
      PyErr_SetString(PyExc_RuntimeError, e.what());
      return nullptr;
    }
  }
};

// Pairs of a tensor and its name, all of them contiguous and of one type.
template <at::ScalarType T> PyObject* contiguous(PyObject*, PyObject* const* args, Py_ssize_t n) {
  for (Py_ssize_t i = 0; i + 1 < n; i += 2) {
    const at::Tensor* t;
    if (!tensor_of(args[i], &t)) return PyErr_Format(PyExc_TypeError, "%U must be a tensor", args[i + 1]);
    try {
      if (t->scalar_type() == T && t->is_contiguous()) continue;
    } catch (const std::exception& e) {
      PyErr_SetString(PyExc_RuntimeError, e.what());
      return nullptr;
    }
    return PyErr_Format(PyExc_TypeError, T == at::kInt ? "%U must be contiguous int32" : "%U must be contiguous float32", args[i + 1]);
  }
  Py_RETURN_NONE;
}

// What ops/seqmix.py asserts of its tensors before these launches, in one call: fifty attributes of tensors took 5 us from Python.
struct Bad { const char* what; };
void need(bool ok, const char* what) {
  if (!ok) throw Bad{what};
}
void need_i32(const at::Tensor& t, const char* name) {
  if (t.scalar_type() == at::kInt && t.is_contiguous()) return;
  PyErr_Format(PyExc_TypeError, "%s must be contiguous int32", name);
  throw Bad{nullptr};
}

// f(tensors, numbers) with the first N arguments as tensors (null for None) and the others as numbers
template <int N, int M, typename Fn> PyObject* checked(PyObject* const* args, Py_ssize_t n, Fn&& f) {
  if (n != N + M) return PyErr_Format(PyExc_TypeError, "takes %d arguments, got %d", N + M, (int)n);
  const at::Tensor* t[N] = {};
  long v[M];
  for (int i = 0; i < N; ++i)
    if (args[i] != Py_None && !tensor_of(args[i], &t[i])) return PyErr_Format(PyExc_TypeError, "argument %d must be a tensor", i);
  for (int i = 0; i < M; ++i)
    if (!Arg<long>::get(args[N + i], &v[i])) return nullptr;
  try {
    return f(t, v);
  } catch (const Bad& b) {
    if (b.what) PyErr_SetString(PyExc_AssertionError, b.what);
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  return nullptr;
}

void need_caches(const at::Tensor& k, const at::Tensor& v, const at::Tensor& x, long G, long D, long Dv) {
  need(k.dim() >= 3 && v.dim() == 3 && k.is_contiguous() && v.is_contiguous(), "contiguous caches [blocks, block, columns]");
  need(k.scalar_type() == x.scalar_type() && v.scalar_type() == x.scalar_type(), "caches of the rows' type");
  need(k.size(2) == G * D && v.size(0) == k.size(0) && v.size(1) == k.size(1) && v.size(2) == G * Dv, "cache columns");
}

// (T, row stride of u, blocks, block, rows of the rotation table) of qk_prep_append
PyObject* qk_shapes(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return checked<6, 6>(args, n, [](const at::Tensor* const* t, const long* v) {
    for (int i = 0; i < 5; ++i) need(t[i], "tensors");
    const at::Tensor &u = *t[0], &k = *t[1], &vc = *t[2], &pos = *t[3], &slots = *t[4];
    const long H = v[0], G = v[1], D = v[2], Dv = v[3], v_off = v[4], dims = v[5];
    need(u.dim() == 2 && u.stride(1) == 1 && (H + G) * D <= u.size(1), "rows with q and k");
    need((v_off < 0 && Dv == D) || (v_off >= (H + G) * D && v_off + G * Dv <= u.size(1)), "values' columns");
    need(dims % 2 == 0 && 0 <= dims && dims <= D, "rotated entries");
    long rows = 0;
    if (dims) {
      need(t[5] && t[5]->dim() >= 2, "a table of rotations");
      if (t[5]->scalar_type() != at::kFloat || !t[5]->is_contiguous()) {
        PyErr_SetString(PyExc_TypeError, "cos_sin must be contiguous float32");
        throw Bad{nullptr};
      }
      need(t[5]->size(1) * 2 == dims, "a table of these rotations");
      rows = t[5]->size(0);
    }
    need_caches(k, vc, u, G, D, Dv);
    need_i32(pos, "positions");
    need_i32(slots, "slots");
    need(pos.numel() >= u.size(0) && slots.numel() >= u.size(0), "a position and a slot for every row");
    return Py_BuildValue("lllll", (long)u.size(0), (long)u.stride(0), (long)k.size(0), (long)k.size(1), rows);
  });
}

// (T, blocks, block, B, columns of the block table, whether the matrix-core token form takes the rows) of window_attention
PyObject* window_shapes(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return checked<7, 4>(args, n, [](const at::Tensor* const* t, const long* v) {
    for (int i = 0; i < 7; ++i) need(t[i], "tensors");
    const at::Tensor &q = *t[0], &k = *t[1], &vc = *t[2], &cu = *t[3], &ctx = *t[4], &bt = *t[5], &pos = *t[6];
    const long H = v[0], G = v[1], D = v[2], Dv = v[3];
    need(q.dim() >= 2 && q.is_contiguous() && q.size(1) == H * D && G > 0 && H % G == 0, "rows of H heads");
    need_caches(k, vc, q, G, D, Dv);
    need(D <= 512 && Dv <= 512, "heads up to 512");
    need_i32(cu, "cu_q");
    need_i32(ctx, "ctx_lens");
    need_i32(bt, "block_tables");
    need_i32(pos, "positions");
    const long B = ctx.numel();
    need(cu.numel() == B + 1 && bt.dim() >= 2 && bt.size(0) == B && pos.numel() >= q.size(0), "feeds, block table and positions");
    // attn_window_token.hip's rule
    const bool token = q.scalar_type() == at::kBFloat16 && D <= 128 && Dv <= 128 && D % 8 == 0 && Dv % 8 == 0 && H / G <= 16 &&
                       (long)k.size(0) * k.size(1) < (1L << 31) &&
                       (((size_t)q.data_ptr() | (size_t)k.data_ptr() | (size_t)vc.data_ptr()) & 15) == 0;
    return Py_BuildValue("lllllO", (long)q.size(0), (long)k.size(0), (long)k.size(1), B, (long)bt.size(1), token ? Py_True : Py_False);
  });
}

#define ENTRIES(X)                                                                                                                \
  X(loqa_qk_prep_append) X(loqa_window_attention) X(loqa_window_attention_parts) X(loqa_delta_prep) X(loqa_delta_scan) \
  X(loqa_seq_state_save) X(loqa_gated_rmsnorm) X(loqa_moe_route) X(loqa_latent_attention) X(loqa_latent_kv) \
  X(loqa_latent_prefill) X(loqa_sigmoid_gate) X(loqa_head_product)

PyObject* signatures(PyObject*, PyObject*) {
  PyObject* d = PyDict_New();
#define SIG(F)                                                                \
  if (d) {                                                                    \
    PyObject* s = PyUnicode_FromString(Entry<&F>::signature().c_str());       \
    if (!s || PyDict_SetItemString(d, #F, s) != 0) Py_CLEAR(d);               \
    Py_XDECREF(s);                                                            \
  }
  ENTRIES(SIG)
#undef SIG
  return d;
}

#define METHOD(F) {#F, (PyCFunction)(void (*)(void))Entry<&F>::call, METH_FASTCALL, nullptr},
PyMethodDef methods[] = {
    ENTRIES(METHOD)
    {"i32c", (PyCFunction)(void (*)(void))contiguous<at::kInt>, METH_FASTCALL, nullptr},
    {"f32c", (PyCFunction)(void (*)(void))contiguous<at::kFloat>, METH_FASTCALL, nullptr},
    {"qk_shapes", (PyCFunction)(void (*)(void))qk_shapes, METH_FASTCALL, nullptr},
    {"window_shapes", (PyCFunction)(void (*)(void))window_shapes, METH_FASTCALL, nullptr},
    {"signatures", signatures, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
#undef METHOD

PyModuleDef module = {PyModuleDef_HEAD_INIT, "libloqa_launch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_libloqa_launch(void) { return PyModule_Create(&module); }
