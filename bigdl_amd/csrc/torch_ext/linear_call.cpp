// The host side of a few-row product in one native call.  A call of one row lasts 4 us on the GPU and took the host 12.8: 5.8 of
// them were checks, an output and 26 arguments in Python.  Module calls of 1 x 2048 sym_int4, us: [1, 2048] 12.8 -> 7.2, [1, 1, 2048]
// 14.3 -> 9.3 (two views more).  What is not an ordinary tensor, or does not fit a kernel as it lies, comes
// back as None and takes the Python way (transformers/low_bit_linear.py), which also raises the errors.
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <ATen/ATen.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <mutex>
#include <string>
#include <tuple>
#include <unordered_map>
#include <utility>

namespace {

// entry points of libbigdl_hip.so (csrc/hip), handed over by bind()
typedef int (*GemvFn)(const void*, const void*, const void*, void*, const void*, const void*, const void*, const void*, float, float, int,
                      int, int, int, int, int, int, int, const void*, int, int, int, int, int, int, hipStream_t);
typedef int (*GemmFn)(const void*, const void*, void*, const void*, const void*, float*, int64_t, int, int, int, int, int, int, int, int,
                      hipStream_t);
typedef int (*FragRuleFn)(int, int, int, int, int, int, int, int);
typedef int64_t (*FragFloatsFn)(int, int, int, int, int, int);
typedef int64_t (*GemmFloatsFn)(int, int, int, int, int, int, int, int);
typedef int (*FragFn)(const void*, const void*, const void*, void*, const void*, const void*, const void*, float*, int64_t, int, int, int,
                      int, int, int, int, int, int, hipStream_t);
typedef int (*RowsFn)(const void*, const void*, const void*, void*, const void*, const void*, const void*, const void*, float, float,
                      float*, int64_t, int, int, int, int, int, int, int, int, int, int, hipStream_t);
GemvFn gemv_lowbit;
GemmFn gemm_lowbit;
FragRuleFn frag_rule;
FragFloatsFn frag_floats;
GemmFloatsFn gemm_floats;
FragFn frag_dense;
RowsFn gemm_rows;
bool bound = false;

constexpr int Q_Q6_K = 26;

// A signature as text, the result in front: p an address (of any type, a stream too), i int, l int64_t, f float.  The entry points' addresses are
// cast to types that stand here, where no compiler sees csrc/hip: Python holds the texts against the ones it calls them by and binds no other.
template <class T> constexpr char KIND = 0;
template <class T> constexpr char KIND<T*> = 'p';
template <> constexpr char KIND<int> = 'i';
template <> constexpr char KIND<int64_t> = 'l';
template <> constexpr char KIND<float> = 'f';
template <class F> struct Signature;
template <class R, class... A>
struct Signature<R (*)(A...)> {
  static_assert(KIND<R> != 0 && ((KIND<A> != 0) && ...), "a type without a letter");
  static constexpr char text[] = {KIND<R>, KIND<A>..., 0};
};

// an ordinary tensor in GPU memory that nothing but the caller looks at: no subclass, wrapper, graph, tangent.  (Views are: the rows of a
// [batch, tokens, hidden] input are one, and outside inference mode it knows its base.)
bool plain(const at::Tensor& t) {
  const auto keys = t.key_set();
  return t.is_cuda() && t.layout() == at::kStrided && !t.is_conj() && !t.is_neg() && !t.requires_grad() && !t._fw_grad(0).defined() &&
         !keys.has_any(c10::python_ks) &&
         !keys.has(c10::DispatchKey::FuncTorchBatched) && !keys.has(c10::DispatchKey::FuncTorchGradWrapper) &&
         !keys.has(c10::DispatchKey::Functionalize) && !keys.has(c10::DispatchKey::BatchedNestedTensor);
}

// scratch of a dense call by its sizes (floats; frag: on the kernel that takes x in fragment order).  Asking takes a microsecond.
struct Sizes {
  int m, n, k, qtype, ldx;
  bool operator==(const Sizes& o) const { return m == o.m && n == o.n && k == o.k && qtype == o.qtype && ldx == o.ldx; }
};
struct SizesHash {
  size_t operator()(const Sizes& s) const {
    size_t h = (size_t)s.m;
    for (int v : {s.n, s.k, s.qtype, s.ldx}) h = h * 1000003u ^ (size_t)v;
    return h;
  }
};
struct Way { bool frag; int64_t floats; };
std::mutex ways_lock;
std::unordered_map<Sizes, Way, SizesHash> ways;

Way way_of(const Sizes& s) {
  std::lock_guard<std::mutex> hold(ways_lock);
  const auto it = ways.find(s);
  if (it != ways.end()) return it->second;
  Way w;
  w.frag = s.m > 32 && frag_rule(s.m, s.n, s.k, s.ldx, s.qtype, 0, 0, 0) == 1;
  w.floats = w.frag ? frag_floats(s.m, s.n, s.k, s.qtype, 0, 0) : gemm_floats(s.m, s.n, s.k, s.ldx, s.qtype, 0, 0, 0);
  if (ways.size() >= 4096) ways.clear();
  ways.emplace(s, w);
  return w;
}

PyObject* rejected(const char* what, int rc) {
  PyErr_Format(PyExc_RuntimeError, "%s: native launcher rejected the call (code %d)", what, rc);
  return nullptr;
}

// product(x, w, n, k, qtype, nbytes, gemv_rows, gemm_rows) -> y [m, n] of x's type, or None.  x fp16 [m, k] on the GPU; w: nbytes bytes,
// tiled for the device, or q6_k blocks.  Up to gemv_rows rows on the skinny kernel, up to gemm_rows on the others.  bf16 up to 32 rows
// of a tiled weight and 64 Ki values, converted by PyTorch's operation as the Python way does (18 rows of 2048: 18.6 -> 13 us of host time).
PyObject* product(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 8 || !bound || !THPVariable_CheckExact(args[0]) || !THPVariable_Check(args[1])) Py_RETURN_NONE;
  long v[6];
  for (int i = 0; i < 6; ++i) {
    v[i] = PyLong_AsLong(args[2 + i]);
    if (v[i] == -1 && PyErr_Occurred()) return nullptr;
  }
  const at::Tensor& x = THPVariable_Unpack(args[0]);
  const at::Tensor& w = THPVariable_Unpack(args[1]);
  const int64_t n = v[0], k = v[1];
  const int qtype = (int)v[2];
  const bool bf16 = x.scalar_type() == at::kBFloat16, q6k = qtype == Q_Q6_K;
  if (!plain(x) || (x.scalar_type() != at::kHalf && !bf16) || x.dim() != 2 || x.size(1) != k || x.stride(1) != 1 || x.stride(0) % 8 != 0 ||
      !w.is_cuda() || w.device() != x.device() || w.key_set().has_any(c10::python_ks) || (int64_t)w.nbytes() != v[3] ||
      c10::impl::TorchDispatchModeTLS::any_modes_set() || torch::jit::tracer::isTracing())
    Py_RETURN_NONE;
  const int64_t m = x.size(0), ldx = bf16 ? k : x.stride(0);
  if (bf16 && (q6k || m > 32 || m * k >= 65536 || x.stride(0) != k)) Py_RETURN_NONE;
  if (m < 1 || m > v[5] || n < 1 || n > INT32_MAX || k < 1 || k > INT32_MAX || ldx > INT32_MAX || ldx < 0) Py_RETURN_NONE;
  at::Tensor half;
  if (bf16) half = x.to(at::kHalf);
  const void* xp = bf16 ? half.const_data_ptr() : x.const_data_ptr();
  const void* wp = w.const_data_ptr();
  if ((uintptr_t)xp % 16 != 0 || (q6k && (k % 256 != 0 || (uintptr_t)wp % 4 != 0 || !w.is_contiguous()))) Py_RETURN_NONE;
  at::Tensor y = at::empty({m, n}, x.options());
  void* yp = y.data_ptr();
  at::Tensor scratch;
  const hipStream_t stream = c10::hip::getCurrentHIPStream().stream();
  const char* what;
  const int out_type = bf16 ? 1 : 0;                  // (csrc/hip/common.h)
  int rc;
  if (q6k) {
    what = "gemm_rows";
    Py_BEGIN_ALLOW_THREADS
    rc = gemm_rows(xp, wp, nullptr, yp, nullptr, nullptr, nullptr, nullptr, 0.0f, 1e-6f, nullptr, 0, (int)m, (int)n, (int)k, (int)ldx, (int)n,
                   qtype, 0, 0, 0, 1, stream);
    Py_END_ALLOW_THREADS
  } else if (m <= v[4]) {
    what = "gemv_lowbit";
    Py_BEGIN_ALLOW_THREADS
    rc = gemv_lowbit(xp, wp, nullptr, yp, nullptr, nullptr, nullptr, nullptr, 1e-6f, 0.0f, (int)m, (int)n, (int)k, (int)ldx, (int)n, qtype, 0,
                     out_type, nullptr, 0, 0, 0, 0, 0, 0, stream);
    Py_END_ALLOW_THREADS
  } else {
    const Way way = way_of({(int)m, (int)n, (int)k, qtype, (int)ldx});
    // (allocated by the call, never kept: a captured call's scratch belongs to its graph, calls on different streams share none)
    float* sp = nullptr;
    if (way.floats > 0) {
      scratch = at::empty({way.floats}, x.options().dtype(at::kFloat));
      sp = (float*)scratch.data_ptr();
    }
    what = way.frag ? "gemm_frag_dense" : "gemm_lowbit";
    Py_BEGIN_ALLOW_THREADS
    rc = way.frag ? frag_dense(xp, wp, nullptr, yp, nullptr, nullptr, nullptr, sp, way.floats, (int)m, (int)n, (int)k, (int)ldx, (int)n, qtype, 0,
                               0, 0, stream)
                  : gemm_lowbit(xp, wp, yp, nullptr, nullptr, sp, way.floats, (int)m, (int)n, (int)k, (int)ldx, (int)n, qtype, 0, out_type, stream);
    Py_END_ALLOW_THREADS
  }
  if (rc != 0) return rejected(what, rc);
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// the seven entry points above
struct Bound { const char* name; void** to; const char* signature; };
template <class F>
Bound bound_to(const char* name, F* to) {
  return {name, (void**)to, Signature<F>::text};
}
const Bound bound_of[] = {
    bound_to("bigdl_gemv_lowbit", &gemv_lowbit), bound_to("bigdl_gemm_lowbit", &gemm_lowbit), bound_to("bigdl_gemm_lowbit_frag", &frag_rule),
    bound_to("bigdl_gemm_frag_workspace", &frag_floats), bound_to("bigdl_gemm_lowbit_workspace", &gemm_floats),
    bound_to("bigdl_gemm_frag_dense", &frag_dense), bound_to("bigdl_gemm_rows", &gemm_rows)};

// bind({name: address}) of all of them
PyObject* bind(PyObject*, PyObject* table) {
  for (auto& e : bound_of) {
    PyObject* at = PyDict_Check(table) ? PyDict_GetItemString(table, e.name) : nullptr;
    void* p = at ? PyLong_AsVoidPtr(at) : nullptr;
    if (p == nullptr) {
      if (!PyErr_Occurred()) PyErr_Format(PyExc_ValueError, "no address for %s", e.name);
      return nullptr;
    }
    *e.to = p;
  }
  bound = true;
  Py_RETURN_NONE;
}

// ---- launchers: entry points of libbigdl_hip.so called with Python's arguments as they are ----
// A prompt of 77 tokens is forty launches of a few microseconds each, and ctypes takes 2.5 us of the host for the 19 arguments of a
// product (pointers asked for in Python included): the pass waits for the host.  Here a call converts by the C signature, with tensors in
// place of their pointers: 0.5 us.  Four layers, 77 tokens: host 521 -> 417 us, the pass 520 -> 446 (450 of kernels), on a faster host 483 -> 453.
template <class T>
struct From {                                        // int, int64_t
  static bool get(PyObject* o, T& v) {
    const long long x = PyLong_AsLongLong(o);
    v = (T)x;
    return x != -1 || !PyErr_Occurred();
  }
};
template <>
struct From<float> {
  static bool get(PyObject* o, float& v) {
    const double x = PyFloat_AsDouble(o);
    v = (float)x;
    return x != -1.0 || !PyErr_Occurred();
  }
};
// None, an address, a tensor, or what has a data_ptr() of its own
template <class T>
struct From<T*> {
  static bool get(PyObject* o, T*& v) {
    if (o == Py_None) {
      v = nullptr;
    } else if (PyLong_Check(o)) {
      v = (T*)PyLong_AsVoidPtr(o);
      return v != nullptr || !PyErr_Occurred();
    } else if (THPVariable_Check(o) && !THPVariable_Unpack(o).key_set().has_any(c10::python_ks)) {
      v = (T*)THPVariable_Unpack(o).data_ptr();
    } else {
      PyObject* at = PyObject_CallMethod(o, "data_ptr", nullptr);
      if (at == nullptr) return false;
      v = (T*)PyLong_AsVoidPtr(at);
      Py_DECREF(at);
      return v != nullptr || !PyErr_Occurred();
    }
    return true;
  }
};

template <class F, int ID>
struct Launcher;
template <class... A, int ID>
struct Launcher<int (*)(A...), ID> {
  static inline int (*entry)(A...) = nullptr;

  template <size_t... I>
  static PyObject* run(PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<A...> v;
    if (!(From<A>::get(args[I], std::get<I>(v)) && ...)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = entry(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
  }
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "%zd arguments, %zd expected", n, (Py_ssize_t)sizeof...(A));
    return run(args, std::index_sequence_for<A...>{});
    END_HANDLE_TH_ERRORS
  }
};

typedef const void* In;
typedef void* Out;
typedef hipStream_t St;
typedef int64_t L;
struct Known { const char* name; void** entry; PyCFunction call; const char* signature; };
template <int ID, class F>
Known known(const char* name) {
  return {name, (void**)&Launcher<F, ID>::entry, (PyCFunction)(void (*)(void))Launcher<F, ID>::call, Signature<F>::text};
}
template <class... A> using Fn = int (*)(A...);
// (the signatures of csrc/hip)
const Known launchers_of[] = {
    known<0, Fn<In, In, In, Out, Out, L, int, L, float, float, int, int, St>>("bigdl_rms_norm"),
    known<1, Fn<const float*, int, In, In, In, Out, Out, L, int, float, float, int, St>>("bigdl_rms_norm_parts"),
    known<2, Fn<Out, Out, Out, Out, const float*, const L*, int, int, int, int, int, int, int, int, int, int, L, L, int, St>>("bigdl_prefill_rope_append"),
    known<3, Fn<In, In, In, Out, In, int, int, int, int, int, int, L, L, L, L, L, L, L, L, L, L, L, L, L, L, const float*, float, float, int, int, int,
                int, int, St>>("bigdl_attn_prefill"),
    known<4, Fn<In, In, In, Out, In, In, In, In, float, float, const float*, float*, float*, L, int, int, int, int, int, int, int, int, St>>(
        "bigdl_gemm_lowbit_ex"),
    known<5, Fn<In, In, float*, L, int, int, int, int, int, int, St>>("bigdl_gemm_parts_run"),
    known<6, FragFn>("bigdl_gemm_frag_dense"),
    known<7, Fn<In, In, Out, In, In, float*, L, int, int, int, int, int, int, int, int, St>>("bigdl_gemm_prompt"),
    known<8, Fn<In, In, In, Out, In, In, int, int, int, int, int, int, int, int, St>>("bigdl_gemm_prompt_pair"),
    known<9, GemvFn>("bigdl_gemv_lowbit"),
    known<10, GemmFn>("bigdl_gemm_lowbit"),
    known<11, Fn<In, In, Out, int, int, int, L, L, int, float, int, St>>("bigdl_lora_down"),
    known<12, Fn<In, In, Out, In, int, int, int, L, L, L, int, float, int, int, St>>("bigdl_lora_up"),
    known<13, Fn<In, Out, int, int, L, int, int, int, int, St>>("bigdl_dequant_t16"),
};
constexpr int LAUNCHERS = sizeof(launchers_of) / sizeof(launchers_of[0]);
PyMethodDef launcher_defs[LAUNCHERS];

// launchers({name: address}) -> {name: callable}, of those it has an address for
PyObject* launchers(PyObject*, PyObject* table) {
  if (!PyDict_Check(table)) return PyErr_Format(PyExc_TypeError, "a dict of addresses");
  PyObject* out = PyDict_New();
  for (int i = 0; out != nullptr && i < LAUNCHERS; ++i) {
    const Known& k = launchers_of[i];
    PyObject* at = PyDict_GetItemString(table, k.name);
    if (at == nullptr) continue;
    *k.entry = PyLong_AsVoidPtr(at);
    launcher_defs[i] = {k.name, k.call, METH_FASTCALL, nullptr};
    PyObject* fn = *k.entry ? PyCFunction_New(&launcher_defs[i], nullptr) : nullptr;
    if (fn == nullptr || PyDict_SetItemString(out, k.name, fn) != 0) {
      if (!PyErr_Occurred()) PyErr_Format(PyExc_ValueError, "no address for %s", k.name);
      Py_CLEAR(out);
    }
    Py_XDECREF(fn);
  }
  return out;
}

// signatures() -> {name: text} of all that bind and launchers take
PyObject* signatures(PyObject*, PyObject*) {
  PyObject* out = PyDict_New();
  auto add = [&](const char* name, const char* text) {
    PyObject* t = out != nullptr ? PyUnicode_FromString(text) : nullptr;
    if (t == nullptr || PyDict_SetItemString(out, name, t) != 0) Py_CLEAR(out);
    Py_XDECREF(t);
  };
  for (auto& e : bound_of) add(e.name, e.signature);
  for (auto& k : launchers_of) add(k.name, k.signature);
  return out;
}

PyMethodDef methods[] = {{"signatures", signatures, METH_NOARGS, nullptr},
                         {"launchers", launchers, METH_O, nullptr},
                         {"product", (PyCFunction)(void (*)(void))product, METH_FASTCALL, nullptr}, {"bind", bind, METH_O, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "bigdl_linear_call", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_bigdl_linear_call() { return PyModule_Create(&module); }
