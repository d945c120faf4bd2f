// CPython extension behind capi.py: the per-step calls of SearchContext and BeamScorer in native code.
//
// A decoding step's kernels run for 7 to 60 us, so what the host spends per call decides the step rate of a small
// batch.  Marshalled through ctypes a call costs 8 to 11 us (a dozen tensor attribute lookups, fifteen argument
// conversions), plus 2 to 4 us per output tensor made by torch's Python entry points and per fill of one; here a call
// reads the tensors' C++ objects directly, makes its outputs in the caching allocator without the dispatcher and
// costs about 1 us beside the launches themselves (2.4 us each).
//
// The library owns no tensors: device memory belongs to the caller's torch tensors, this file passes pointers on.
#include <Python.h>
#include <structmember.h>
#include <ATen/EmptyTensor.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <cstring>
#include <vector>
#include "mi355x_search.h"

// Entry points of libmi355x_search.so that have no place in the C ABI: mi355x_sample* whose kept sets are padded with
// (id -1, probability 0) up to their capacity, and a copy of one of a scorer's arrays to `dst` that is done on return.
extern "C" int ms_sample_padded(mi355x_search_ctx* ctx, void* stream, const void* logits, const void* const* row_ptrs, int dtype,
                                int64_t row_stride, int rows, int vocab, const mi355x_logits_xform* xf,
                                mi355x_sample_params params, const mi355x_sample_params* per_row_params, const double* uniforms,
                                int32_t* out_tokens, int32_t* kept_count, int32_t* kept_ids, float* kept_probs,
                                int kept_capacity);
extern "C" int ms_scorer_copy_words(mi355x_beam_scorer* s, void* stream, void* dst, const void* src, size_t words);
extern "C" int ms_scorer_is_done(mi355x_beam_scorer* s, void* stream, int* done);

namespace {

using at::Tensor;

// ---- errors and argument parsing ------------------------------------------------------------------------------

// A Python exception is set; unwinds to the entry point, which returns null.
struct PyFailed {};

[[noreturn]] void Raise(PyObject* type, const char* text) {
  PyErr_SetString(type, text);
  throw PyFailed{};
}

void Require(bool ok, const char* text) {
  if (!ok) Raise(PyExc_AssertionError, text);
}

void Check(int rc) {
  if (rc == MI355X_OK) return;
  PyErr_Format(PyExc_RuntimeError, "mi355x_search error %d: %s", rc, mi355x_search_last_error());
  throw PyFailed{};
}

// Owns a reference.
struct Ref {
  PyObject* o;
  explicit Ref(PyObject* p) : o(p) {
    if (!p) throw PyFailed{};
  }
  ~Ref() { Py_XDECREF(o); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
  PyObject* release() {
    PyObject* p = o;
    o = nullptr;
    return p;
  }
};

// The parameters of one entry point: names in order, the first `required` of them without a default.  Arguments land
// in out[], absent ones stay null.  Keyword names arrive interned, so the pointers nearly always decide.
struct Signature {
  const char* function;
  int required;
  std::vector<const char*> names;
  std::vector<PyObject*> interned;

  Signature(const char* f, int req, std::vector<const char*> n) : function(f), required(req), names(std::move(n)) {}

  void Parse(PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames, PyObject** out) {
    const int n = static_cast<int>(names.size());
    if (interned.empty())
      for (const char* s : names) interned.push_back(PyUnicode_InternFromString(s));
    if (nargs > n) {
      PyErr_Format(PyExc_TypeError, "%s() takes at most %d arguments (%zd given)", function, n, nargs);
      throw PyFailed{};
    }
    for (int i = 0; i < n; ++i) out[i] = i < nargs ? args[i] : nullptr;
    const Py_ssize_t nk = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
    for (Py_ssize_t k = 0; k < nk; ++k) {
      PyObject* name = PyTuple_GET_ITEM(kwnames, k);
      int at = -1;
      for (int i = 0; i < n && at < 0; ++i)
        if (interned[i] == name) at = i;
      for (int i = 0; i < n && at < 0; ++i)
        if (PyUnicode_Compare(interned[i], name) == 0) at = i;
      if (at < 0) {
        PyErr_Format(PyExc_TypeError, "%s() got an unexpected keyword argument '%U'", function, name);
        throw PyFailed{};
      }
      if (out[at]) {
        PyErr_Format(PyExc_TypeError, "%s() got multiple values for argument '%U'", function, name);
        throw PyFailed{};
      }
      out[at] = args[nargs + k];
    }
    for (int i = 0; i < required; ++i)
      if (!out[i]) {
        PyErr_Format(PyExc_TypeError, "%s() missing required argument '%s'", function, names[i]);
        throw PyFailed{};
      }
  }
};

bool Given(PyObject* o) { return o && o != Py_None; }

const Tensor& TensorOf(PyObject* o) {
  if (!o || !THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "expected a torch.Tensor, got %s", o ? Py_TYPE(o)->tp_name : "nothing");
    throw PyFailed{};
  }
  return THPVariable_Unpack(o);
}

long LongOf(PyObject* o) {  // int(o)
  if (PyLong_Check(o)) {
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) throw PyFailed{};
    return v;
  }
  Ref i(PyNumber_Long(o));
  const long v = PyLong_AsLong(i.o);
  if (v == -1 && PyErr_Occurred()) throw PyFailed{};
  return v;
}
long LongOr(PyObject* o, long fallback) { return o ? LongOf(o) : fallback; }

double DoubleOf(PyObject* o) {  // float(o)
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyFailed{};
  return v;
}
double DoubleOr(PyObject* o, double fallback) { return o ? DoubleOf(o) : fallback; }

bool TruthOf(PyObject* o) {
  if (!o) return false;
  const int t = PyObject_IsTrue(o);
  if (t < 0) throw PyFailed{};
  return t != 0;
}

int DtypeCode(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return MI355X_F32;
    case at::kInt: return MI355X_I32;
    case at::kLong: return MI355X_I64;
    case at::kHalf: return MI355X_F16;
    case at::kBFloat16: return MI355X_BF16;
    default: PyErr_SetString(PyExc_KeyError, c10::toString(t)); throw PyFailed{};
  }
}

at::ScalarType ScalarTypeOf(PyObject* o) {
  if (!THPDtype_Check(o)) Raise(PyExc_TypeError, "expected a torch.dtype");
  return reinterpret_cast<THPDtype*>(o)->scalar_type;
}

// Everything between here and the call's outputs runs without the interpreter lock, as a foreign call does.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

void* CurrentStream() { return static_cast<void*>(c10::hip::getCurrentHIPStream().stream()); }

// A new contiguous tensor on `device`.
Tensor Empty(at::IntArrayRef sizes, at::ScalarType type, c10::Device device) {
  static c10::Allocator* const allocator = c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get();
  constexpr c10::DispatchKeySet keys(c10::DispatchKey::CUDA);
  if (device.index() == c10::hip::current_device()) return at::detail::empty_generic(sizes, allocator, keys, type, std::nullopt);
  const c10::DeviceGuard guard(device);
  return at::detail::empty_generic(sizes, allocator, keys, type, std::nullopt);
}

template <typename T>
T* Data(const Tensor& t) {
  return static_cast<T*>(t.data_ptr());
}

PyObject* Wrap(const Tensor& t) {
  PyObject* o = THPVariable_Wrap(t);
  if (!o) throw PyFailed{};
  return o;
}
PyObject* WrapAll(std::initializer_list<PyObject*> items) {  // steals the references
  PyObject* tuple = PyTuple_New(static_cast<Py_ssize_t>(items.size()));
  if (!tuple) throw PyFailed{};
  Py_ssize_t i = 0;
  for (PyObject* o : items) PyTuple_SET_ITEM(tuple, i++, o);
  return tuple;
}
PyObject* NewRef(PyObject* o) {
  Py_INCREF(o);
  return o;
}

// The ctypes structure a LogitsXform holds (its address is taken when the object is made), or null.
const mi355x_logits_xform* XformOf(PyObject* o) {
  if (!Given(o)) return nullptr;
  static PyObject* const name = PyUnicode_InternFromString("_addr");
  Ref a(PyObject_GetAttr(o, name));
  void* p = PyLong_AsVoidPtr(a.o);
  if (!p && PyErr_Occurred()) throw PyFailed{};
  return static_cast<const mi355x_logits_xform*>(p);
}

// [rows, vocab] logits whose rows are contiguous.
struct Rows {
  int rows, vocab;
  int64_t stride;
  void* data;
  int dtype;
  explicit Rows(const Tensor& t) {
    Require(t.is_cuda() && t.dim() == 2 && t.stride(1) == 1, "logits must be a 2-d device tensor with contiguous rows");
    rows = static_cast<int>(t.size(0));
    vocab = static_cast<int>(t.size(1));
    stride = t.stride(0);
    data = t.data_ptr();
    dtype = DtypeCode(t.scalar_type());
  }
};

// The items of a list or tuple.
struct Items {
  Ref seq;
  explicit Items(PyObject* o, const char* what) : seq(PySequence_Fast(o, what)) {}
  Py_ssize_t size() const { return PySequence_Fast_GET_SIZE(seq.o); }
  PyObject* operator[](Py_ssize_t i) const { return PySequence_Fast_GET_ITEM(seq.o, i); }
};

template <typename F>
PyObject* Guarded(F f) {
  try {
    return f();
  } catch (const PyFailed&) {
    return nullptr;
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// ---- Context: what SearchContext derives from -----------------------------------------------------------------

struct Context {
  PyObject_HEAD
  mi355x_search_ctx* handle;
  c10::DeviceIndex device;
};
Context* Ctx(PyObject* self) { return reinterpret_cast<Context*>(self); }

#define MS_METHOD(NAME) PyObject* NAME(PyObject* self, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames)
#define MS_PARSE(REQUIRED, ...)                                       \
  static Signature sig(__func__, REQUIRED, {__VA_ARGS__});            \
  PyObject* a[sizeof((const char*[]){__VA_ARGS__}) / sizeof(char*)];  \
  sig.Parse(args, nargs, kwnames, a)

MS_METHOD(_attach) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(2, "handle", "device");
    Ctx(self)->handle = static_cast<mi355x_search_ctx*>(PyLong_AsVoidPtr(a[0]));
    Ctx(self)->device = static_cast<c10::DeviceIndex>(LongOf(a[1]));
    return NewRef(Py_None);
  });
}

MS_METHOD(process_logits) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(2, "logits", "xf");
    const Tensor& t = TensorOf(a[0]);
    const Rows r(t);
    Require(r.dtype == MI355X_F32, "logits must be float32");
    const mi355x_logits_xform* xf = XformOf(a[1]);
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_process_logits(Ctx(self)->handle, s, static_cast<float*>(r.data), r.stride, r.rows, r.vocab, xf);
    }
    Check(rc);
    return NewRef(a[0]);
  });
}

MS_METHOD(argmax) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(1, "logits", "xf", "out");
    const Tensor& t = TensorOf(a[0]);
    const Rows r(t);
    const mi355x_logits_xform* xf = TruthOf(a[1]) ? XformOf(a[1]) : nullptr;
    Ref out(Given(a[2]) ? NewRef(a[2]) : Wrap(Empty({r.rows}, at::kInt, t.device())));
    int32_t* const tokens = Data<int32_t>(TensorOf(out.o));
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_argmax(Ctx(self)->handle, s, r.data, r.dtype, r.stride, r.rows, r.vocab, xf, tokens);
    }
    Check(rc);
    return out.release();
  });
}

MS_METHOD(sample) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(2, "logits", "uniforms", "k", "p", "temperature", "per_row", "xf", "out", "kept_capacity");
    std::vector<const void*> row_ptrs;
    int rows, vocab, dtype;
    int64_t stride;
    void* data = nullptr;
    c10::Device device(c10::DeviceType::CUDA);
    if (PyList_Check(a[0]) || PyTuple_Check(a[0])) {  // scattered rows: 1-d tensors of one type and length
      const Items list(a[0], "logits");
      rows = static_cast<int>(list.size());
      if (rows == 0) Raise(PyExc_IndexError, "no rows");
      const Tensor& first = TensorOf(list[0]);
      device = first.device();
      vocab = static_cast<int>(first.numel());
      stride = vocab;
      dtype = DtypeCode(first.scalar_type());
      row_ptrs.resize(rows);
      for (int i = 0; i < rows; ++i) {
        const Tensor& t = TensorOf(list[i]);
        Require(t.is_cuda() && t.dim() == 1 && t.stride(0) == 1 && t.scalar_type() == first.scalar_type() && t.numel() == vocab,
                "rows must be contiguous 1-d device tensors of one type and length");
        row_ptrs[i] = t.data_ptr();
      }
    } else {
      const Tensor& t = TensorOf(a[0]);
      const Rows r(t);
      rows = r.rows, vocab = r.vocab, stride = r.stride, data = r.data, dtype = r.dtype;
      device = t.device();
    }
    const Tensor& uniforms = TensorOf(a[1]);
    Require(uniforms.scalar_type() == at::kDouble && uniforms.numel() >= rows, "uniforms must be float64, one per row");
    const mi355x_sample_params prm{static_cast<int32_t>(LongOr(a[2], 0)), static_cast<float>(DoubleOr(a[3], 0.0)),
                                   static_cast<float>(DoubleOr(a[4], 1.0))};
    std::vector<mi355x_sample_params> table;
    if (Given(a[5])) {
      table.resize(rows, mi355x_sample_params{0, 0.0f, 0.0f});
      const Items list(a[5], "per_row must be a sequence");
      if (list.size() > rows) Raise(PyExc_IndexError, "more entries in per_row than rows");
      for (Py_ssize_t i = 0; i < list.size(); ++i) {
        const Items row(list[i], "an entry of per_row must be a sequence");
        if (row.size() != 3) Raise(PyExc_ValueError, "an entry of per_row is (k, p, temperature)");
        table[i] = {static_cast<int32_t>(LongOf(row[0])), static_cast<float>(DoubleOf(row[1])), static_cast<float>(DoubleOf(row[2]))};
      }
    }
    const mi355x_logits_xform* xf = TruthOf(a[6]) ? XformOf(a[6]) : nullptr;
    Ref out(Given(a[7]) ? NewRef(a[7]) : Wrap(Empty({rows}, at::kInt, device)));
    int32_t* const tokens = Data<int32_t>(TensorOf(out.o));
    const int cap = static_cast<int>(LongOr(a[8], 0));
    Tensor kc, ki, kp;
    if (cap != 0) {
      kc = Empty({rows}, at::kInt, device);
      ki = Empty({rows, cap}, at::kInt, device);
      kp = Empty({rows, cap}, at::kFloat, device);
    }
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = ms_sample_padded(Ctx(self)->handle, s, data, row_ptrs.empty() ? nullptr : row_ptrs.data(), dtype, stride, rows, vocab, xf,
                            prm, table.empty() ? nullptr : table.data(), Data<double>(uniforms), tokens,
                            cap ? Data<int32_t>(kc) : nullptr, cap ? Data<int32_t>(ki) : nullptr, cap ? Data<float>(kp) : nullptr, cap);
    }
    Check(rc);
    if (!cap) return out.release();
    return WrapAll({out.release(), Wrap(kc), Wrap(ki), Wrap(kp)});
  });
}

MS_METHOD(topk_scores) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(2, "logits", "k");
    const Tensor& t = TensorOf(a[0]);
    const Rows r(t);
    const int k = static_cast<int>(LongOf(a[1]));
    const Tensor tok = Empty({r.rows, k}, at::kInt, t.device()), sc = Empty({r.rows, k}, at::kFloat, t.device());
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_topk_scores(Ctx(self)->handle, s, r.data, r.dtype, r.stride, r.rows, r.vocab, k, Data<int32_t>(tok), Data<float>(sc));
    }
    Check(rc);
    return WrapAll({Wrap(tok), Wrap(sc)});
  });
}

MS_METHOD(softmax) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(1, "scores", "temperature", "log");
    const Rows r(TensorOf(a[0]));
    Require(r.dtype == MI355X_F32, "scores must be float32");
    const float temperature = static_cast<float>(DoubleOr(a[1], 1.0));
    const int log = TruthOf(a[2]) ? 1 : 0;
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_softmax(Ctx(self)->handle, s, static_cast<float*>(r.data), r.stride, r.rows, r.vocab, temperature, log);
    }
    Check(rc);
    return NewRef(a[0]);
  });
}

MS_METHOD(beam_select) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(4, "logits", "batch", "beams", "beam_scores");
    const Tensor& t = TensorOf(a[0]);
    const Rows r(t);
    const int batch = static_cast<int>(LongOf(a[1])), beams = static_cast<int>(LongOf(a[2]));
    const Tensor& scores = TensorOf(a[3]);
    Require(r.rows == batch * beams && scores.scalar_type() == at::kFloat && scores.numel() == r.rows,
            "batch * beams rows of logits and as many float32 beam scores");
    const int64_t k = 2 * beams;
    const Tensor sc = Empty({batch, k}, at::kFloat, t.device()), tok = Empty({batch, k}, at::kInt, t.device()),
                 idx = Empty({batch, k}, at::kInt, t.device());
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_beam_select(Ctx(self)->handle, s, r.data, r.dtype, r.stride, batch, beams, r.vocab, Data<float>(scores),
                              Data<float>(sc), Data<int32_t>(tok), Data<int32_t>(idx));
    }
    Check(rc);
    return WrapAll({Wrap(sc), Wrap(tok), Wrap(idx)});
  });
}

MS_METHOD(kv_gather) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(3, "present", "past", "beam_indices");
    const Items present(a[0], "present must be a sequence"), past(a[1], "past must be a sequence");
    const Tensor& idx = TensorOf(a[2]);
    const Py_ssize_t n = present.size();
    Require(n == past.size() && idx.scalar_type() == at::kInt, "as many past as present tensors, int32 beam indices");
    if (n == 0) Raise(PyExc_IndexError, "no tensors");
    const Tensor& first = TensorOf(present[0]);
    if (first.dim() == 0 || first.size(0) == 0) Raise(PyExc_IndexError, "tensors have a row for every beam");
    const size_t block = static_cast<size_t>(first.numel() / first.size(0)) * first.element_size();
    std::vector<const void*> src(n);
    std::vector<void*> dst(n);
    for (Py_ssize_t i = 0; i < n; ++i) {
      const Tensor &p = TensorOf(present[i]), &q = TensorOf(past[i]);
      Require(p.is_contiguous() && q.is_contiguous() && p.dim() > 0 && p.size(0) > 0 &&
                  static_cast<size_t>(p.numel() / p.size(0)) * p.element_size() == block,
              "contiguous tensors of one shape");
      src[i] = p.data_ptr();
      dst[i] = q.data_ptr();
    }
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_kv_gather(Ctx(self)->handle, s, src.data(), dst.data(), static_cast<int>(n), Data<int32_t>(idx),
                            static_cast<int>(idx.numel()), block);
    }
    Check(rc);
    return NewRef(a[1]);
  });
}

MS_METHOD(spec_verify) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(5, "p_target", "p_draft", "draft_tokens", "accept_u", "sample_u");
    const Tensor &pt = TensorOf(a[0]), &pd = TensorOf(a[1]), &dt = TensorOf(a[2]), &au = TensorOf(a[3]), &su = TensorOf(a[4]);
    if (pt.dim() != 3) Raise(PyExc_ValueError, "p_target is [batch, K + 1, vocab]");
    for (const Tensor* t : {&pt, &pd, &dt, &au, &su}) Require(t->is_cuda() && t->is_contiguous(), "contiguous device tensors");
    Require(pt.scalar_type() == at::kFloat && au.scalar_type() == at::kFloat && su.scalar_type() == at::kDouble,
            "float32 probabilities and accept draws, float64 sample draws");
    const int b = static_cast<int>(pt.size(0)), k = static_cast<int>(pt.size(1)) - 1, v = static_cast<int>(pt.size(2));
    const Tensor acc = Empty({b}, at::kInt, pt.device()), tok = Empty({b}, at::kInt, pt.device());
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_spec_verify(Ctx(self)->handle, s, Data<float>(pt), Data<float>(pd), Data<int32_t>(dt), Data<float>(au), Data<double>(su),
                              b, k, v, Data<int32_t>(acc), Data<int32_t>(tok));
    }
    Check(rc);
    return WrapAll({Wrap(acc), Wrap(tok)});
  });
}

MS_METHOD(spec_verify_sparse) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(5, "target", "draft", "proposal", "accept_u", "sample_u", "mode");
    auto fit = [](const Tensor& t) { Require(t.is_cuda() && t.is_contiguous(), "contiguous device tensors"); };
    auto optional = [&](PyObject* o) -> void* {
      if (!Given(o)) return nullptr;
      const Tensor& t = TensorOf(o);
      fit(t);
      return t.data_ptr();
    };
    const Items target(a[0], "target is (count, ids, probs)");
    if (target.size() != 3) Raise(PyExc_ValueError, "target is (count, ids, probs)");
    const Tensor &tc = TensorOf(target[0]), &ti = TensorOf(target[1]), &prop = TensorOf(a[2]);
    if (prop.dim() != 2) Raise(PyExc_ValueError, "proposal is [batch, K]");
    const int b = static_cast<int>(prop.size(0)), k = static_cast<int>(prop.size(1));
    Require(tc.dim() == 2 && tc.size(0) == b && tc.size(1) == k + 1 && ti.dim() == 3 && ti.size(0) == b && ti.size(1) == k + 1,
            "the targets have a row per proposal and one more");
    fit(tc), fit(ti), fit(prop);
    void* const tp = optional(target[2]);
    void* const au = optional(a[3]);
    void* const su = optional(a[4]);
    const void *dc = nullptr, *di = nullptr, *dp = nullptr;
    int dcap = 0;
    if (Given(a[1])) {
      const Items draft(a[1], "draft is (count, ids, probs)");
      if (draft.size() != 3) Raise(PyExc_ValueError, "draft is (count, ids, probs)");
      const Tensor& t = TensorOf(draft[1]);
      fit(TensorOf(draft[0])), fit(t), fit(TensorOf(draft[2]));
      if (t.dim() != 3) Raise(PyExc_IndexError, "draft ids are [batch, K, capacity]");
      dc = TensorOf(draft[0]).data_ptr(), di = t.data_ptr(), dp = TensorOf(draft[2]).data_ptr();
      dcap = static_cast<int>(t.size(2));
    }
    const int mode = static_cast<int>(LongOr(a[5], 0));
    const Tensor acc = Empty({b}, at::kInt, prop.device()), tok = Empty({b}, at::kInt, prop.device()), used = Empty({b}, at::kInt, prop.device());
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_spec_verify_sparse(Ctx(self)->handle, s, Data<int32_t>(tc), Data<int32_t>(ti), static_cast<float*>(tp),
                                     static_cast<int>(ti.size(2)), static_cast<const int32_t*>(dc), static_cast<const int32_t*>(di),
                                     static_cast<const float*>(dp), dcap, Data<int32_t>(prop), static_cast<float*>(au),
                                     static_cast<double*>(su), b, k, mode, Data<int32_t>(acc), Data<int32_t>(tok), Data<int32_t>(used));
    }
    Check(rc);
    return WrapAll({Wrap(acc), Wrap(tok), Wrap(used)});
  });
}

MS_METHOD(greedy_tail) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(7, "next_tokens", "eos_seen", "eos_ids", "pad", "sequences", "current_length", "done", "allow_host");
    const bool allow_host = TruthOf(a[7]);
    const Tensor &next = TensorOf(a[0]), &seen = TensorOf(a[1]), &seq = TensorOf(a[4]), &done = TensorOf(a[6]);
    for (const Tensor* t : {&next, &seen, &seq, &done}) {
      Require(t->is_contiguous() && t->scalar_type() == at::kInt, "contiguous int32 tensors");
      Require(t->is_cuda() || (allow_host && t->is_pinned()), "device tensors (or, with allow_host, pinned ones)");
    }
    if (seq.dim() < 2) Raise(PyExc_IndexError, "sequences are [batch, max_length]");
    const Items eos(a[2], "eos_ids must be a sequence");
    std::vector<int32_t> ids(eos.size() ? eos.size() : 1);
    for (Py_ssize_t i = 0; i < eos.size(); ++i) ids[i] = static_cast<int32_t>(LongOf(eos[i]));
    const int pad = static_cast<int>(LongOf(a[3])), length = static_cast<int>(LongOf(a[5]));
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_greedy_tail(Ctx(self)->handle, s, Data<int32_t>(next), Data<int32_t>(seen), static_cast<int>(next.numel()), ids.data(),
                              static_cast<int>(eos.size()), pad, Data<int32_t>(seq), static_cast<int>(seq.size(1)), length,
                              Data<int32_t>(done));
    }
    Check(rc);
    return NewRef(Py_None);
  });
}

MS_METHOD(draw_in_order) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(4, "kept_count", "kept_ids", "kept_probs", "uniform_pool", "skip_rows");
    const Tensor &kc = TensorOf(a[0]), &ki = TensorOf(a[1]), &kp = TensorOf(a[2]), &pool = TensorOf(a[3]);
    if (ki.dim() != 2) Raise(PyExc_ValueError, "kept_ids are [rows, capacity]");
    const int rows = static_cast<int>(ki.size(0)), cap = static_cast<int>(ki.size(1));
    Require(kc.scalar_type() == at::kInt && ki.scalar_type() == at::kInt && kp.scalar_type() == at::kFloat, "int32 counts and ids, float32 probabilities");
    Require(pool.scalar_type() == at::kDouble && pool.numel() >= rows, "float64 draws, one per row");
    for (const Tensor* t : {&kc, &ki, &kp, &pool}) Require(t->is_cuda() && t->is_contiguous(), "contiguous device tensors");
    const int32_t* skip = Given(a[4]) ? Data<int32_t>(TensorOf(a[4])) : nullptr;
    const c10::Device device(c10::DeviceType::CUDA, Ctx(self)->device);
    const Tensor out = Empty({rows}, at::kInt, device), used = Empty({1}, at::kInt, device);  // (the kernel writes both)
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_draw_in_order(Ctx(self)->handle, s, Data<int32_t>(kc), Data<int32_t>(ki), Data<float>(kp), cap, rows, skip, Data<double>(pool),
                                Data<int32_t>(out), Data<int32_t>(used));
    }
    Check(rc);
    return WrapAll({Wrap(out), Wrap(used)});
  });
}

MS_METHOD(cast) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(2, "src", "dtype");
    const Tensor& src = TensorOf(a[0]);
    Require(src.is_cuda() && src.is_contiguous(), "a contiguous device tensor");
    const at::ScalarType to = ScalarTypeOf(a[1]);
    const int in_code = DtypeCode(src.scalar_type()), out_code = DtypeCode(to);
    const Tensor out = Empty(src.sizes(), to, src.device());
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_cast(Ctx(self)->handle, s, src.data_ptr(), in_code, out.data_ptr(), out_code, static_cast<size_t>(src.numel()));
    }
    Check(rc);
    return Wrap(out);
  });
}

MS_METHOD(logits_handoff) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(1, "raw", "token_index", "out");
    const Tensor& raw = TensorOf(a[0]);
    Require(raw.is_cuda() && raw.is_contiguous() && raw.dim() == 3, "raw is a contiguous [rows, seq_len, vocab] device tensor");
    const int rows = static_cast<int>(raw.size(0)), seq = static_cast<int>(raw.size(1)), vocab = static_cast<int>(raw.size(2));
    const int dtype = DtypeCode(raw.scalar_type());
    std::vector<int32_t> index;
    if (Given(a[1])) {
      const Items list(a[1], "token_index must be a sequence");
      if (list.size() > rows) Raise(PyExc_IndexError, "more entries in token_index than rows");
      index.resize(rows, 0);
      for (Py_ssize_t i = 0; i < list.size(); ++i) index[i] = static_cast<int32_t>(LongOf(list[i]));
    }
    Ref out(Given(a[2]) ? NewRef(a[2]) : Wrap(Empty({rows, vocab}, at::kFloat, raw.device())));
    const Tensor& o = TensorOf(out.o);
    if (o.dim() < 1) Raise(PyExc_IndexError, "out is [rows, vocab]");
    float* const dst = Data<float>(o);
    const int64_t out_stride = o.stride(0);
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_logits_handoff(Ctx(self)->handle, s, raw.data_ptr(), dtype, rows, seq, vocab, index.empty() ? nullptr : index.data(), dst,
                                 out_stride);
    }
    Check(rc);
    return out.release();
  });
}

// ---- Issue: a mi355x_sample call whose arguments stay what they are (SearchContext.prepared_sample) ------------

struct Issue {
  PyObject_HEAD
  vectorcallfunc call;
  PyObject* keep;  // the tensors, the xform and the stream the pointers below belong to
  mi355x_search_ctx* handle;
  void* stream;
  const void* logits;
  int dtype;
  int64_t stride;
  int rows, vocab;
  const mi355x_logits_xform* xf;
  mi355x_sample_params prm;
  const double* uniforms;
  int32_t* out;
};
PyObject* CallIssue(PyObject* self, PyObject* const*, size_t nargsf, PyObject* kwnames) {
  if (PyVectorcall_NARGS(nargsf) != 0 || (kwnames && PyTuple_GET_SIZE(kwnames) != 0)) {
    PyErr_SetString(PyExc_TypeError, "a prepared call takes no arguments");
    return nullptr;
  }
  const Issue& i = *reinterpret_cast<Issue*>(self);
  return Guarded([&]() -> PyObject* {
    int rc;
    {
      Unlocked u;
      rc = mi355x_sample_typed(i.handle, i.stream, i.logits, i.dtype, i.stride, i.rows, i.vocab, i.xf, i.prm, nullptr, i.uniforms, i.out,
                               nullptr, nullptr, nullptr, 0);
    }
    Check(rc);
    return NewRef(Py_None);
  });
}
void FreeIssue(PyObject* self) {
  PyTypeObject* type = Py_TYPE(self);
  Py_XDECREF(reinterpret_cast<Issue*>(self)->keep);
  type->tp_free(self);
  Py_DECREF(type);
}
PyMemberDef kIssueMembers[] = {
    {const_cast<char*>("__vectorcalloffset__"), T_PYSSIZET, offsetof(Issue, call), READONLY, nullptr},
    {nullptr, 0, 0, 0, nullptr},
};
PyType_Slot kIssueSlots[] = {
    {Py_tp_dealloc, reinterpret_cast<void*>(FreeIssue)},
    {Py_tp_call, reinterpret_cast<void*>(PyVectorcall_Call)},
    {Py_tp_members, kIssueMembers},
    {Py_tp_doc, const_cast<char*>("A prepared mi355x_sample call: calling it, without arguments, issues it.")},
    {0, nullptr},
};
PyType_Spec kIssueSpec = {"_binding.Issue", sizeof(Issue), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL, kIssueSlots};
PyTypeObject* g_issue_type = nullptr;

MS_METHOD(prepared_sample) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(3, "logits", "uniforms", "out", "k", "p", "temperature", "xf", "stream");
    const Rows r(TensorOf(a[0]));
    const Tensor &uniforms = TensorOf(a[1]), &out = TensorOf(a[2]);
    Require(uniforms.scalar_type() == at::kDouble && uniforms.numel() >= r.rows && out.scalar_type() == at::kInt && out.numel() >= r.rows,
            "float64 uniforms and an int32 output, one per row");
    void* stream = CurrentStream();
    if (Given(a[7])) {
      Ref s(PyObject_GetAttrString(a[7], "cuda_stream"));
      stream = PyLong_AsVoidPtr(s.o);
      if (!stream && PyErr_Occurred()) throw PyFailed{};
    }
    const mi355x_logits_xform* xf = TruthOf(a[6]) ? XformOf(a[6]) : nullptr;
    const mi355x_sample_params prm{static_cast<int32_t>(LongOr(a[3], 0)), static_cast<float>(DoubleOr(a[4], 0.0)),
                                   static_cast<float>(DoubleOr(a[5], 1.0))};
    Ref keep(PyTuple_Pack(6, self, a[0], a[1], a[2], a[6] ? a[6] : Py_None, a[7] ? a[7] : Py_None));
    PyObject* o = g_issue_type->tp_alloc(g_issue_type, 0);
    if (!o) throw PyFailed{};
    Issue& i = *reinterpret_cast<Issue*>(o);
    i.call = CallIssue;
    i.keep = keep.release();
    i.handle = Ctx(self)->handle;
    i.stream = stream;
    i.logits = r.data, i.dtype = r.dtype, i.stride = r.stride, i.rows = r.rows, i.vocab = r.vocab;
    i.xf = xf, i.prm = prm, i.uniforms = Data<double>(uniforms), i.out = Data<int32_t>(out);
    return o;
  });
}

#define MS_ENTRY(NAME, DOC) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(NAME)), METH_FASTCALL | METH_KEYWORDS, DOC}
PyMethodDef kContextMethods[] = {
    MS_ENTRY(_attach, "Takes the address of the mi355x_search_ctx and its device index."),
    MS_ENTRY(process_logits, "process_logits(logits, xf): in-place logits processing; returns logits."),
    MS_ENTRY(argmax, "argmax(logits, xf=None, out=None): the argmax of every row, int32."),
    MS_ENTRY(sample,
             "sample(logits, uniforms, k=0, p=0.0, temperature=1.0, per_row=None, xf=None, out=None, kept_capacity=0)\n\n"
             "logits: a [rows, vocab] tensor, or a list of rows (1-D tensors of one dtype and length, anywhere in\n"
             "device memory).  Returns the tokens, or (tokens, kept_count, kept_ids, kept_probs) with kept_capacity."),
    MS_ENTRY(prepared_sample,
             "prepared_sample(logits, uniforms, out, k=0, p=0.0, temperature=1.0, xf=None, stream=None)\n\n"
             "Marshals one mi355x_sample call once and returns a callable that issues it: what a serving loop with fixed\n"
             "buffers does (the tensors, `xf` and the stream -- default: the stream current now -- must stay alive and\n"
             "where they are; the callable takes no arguments and raises on an error code).  `out` may be pinned host\n"
             "memory.  As with every call, one context serves one stream at a time: calls prepared for different streams\n"
             "must not overlap."),
    MS_ENTRY(topk_scores, "topk_scores(logits, k): the k best (token ids, raw fp32 scores) per row, best first."),
    MS_ENTRY(softmax, "softmax(scores, temperature=1.0, log=False): in place; returns scores."),
    MS_ENTRY(beam_select, "beam_select(logits, batch, beams, beam_scores): the 2*beams best (scores, tokens, beams) per batch entry."),
    MS_ENTRY(kv_gather,
             "kv_gather(present, past, beam_indices): lists of equally shaped contiguous device tensors [rows, ...];\n"
             "past[t][j] = present[t][beam_indices[j]].  Returns past."),
    MS_ENTRY(spec_verify, "spec_verify(p_target, p_draft, draft_tokens, accept_u, sample_u): (accepted_len, final_token)."),
    MS_ENTRY(spec_verify_sparse,
             "spec_verify_sparse(target, draft, proposal, accept_u, sample_u, mode=0)\n\n"
             "target = (count [b, K+1], ids [b, K+1, cap], probs [b, K+1, cap]) as sample returns them; draft likewise with\n"
             "K rows (None unless mode 0).  Returns (accepted_len, final_token, engine_draws)."),
    MS_ENTRY(greedy_tail,
             "greedy_tail(next_tokens, eos_seen, eos_ids, pad, sequences, current_length, done, allow_host=False)\n\n"
             "EOS padding / marking, append at column current_length, all-rows-finished flag; all in place.\n"
             "allow_host: next_tokens and done may be pinned host tensors, which the kernel reads and writes in place."),
    MS_ENTRY(draw_in_order,
             "draw_in_order(kept_count, kept_ids, kept_probs, uniform_pool, skip_rows=None)\n\n"
             "SampleCategoricalToken for a batch served by one engine, rows in order: (tokens [rows], draws used)."),
    MS_ENTRY(cast, "cast(src, dtype): a new tensor of `dtype` with the reference CPU path's conversion."),
    MS_ENTRY(logits_handoff,
             "logits_handoff(raw, token_index=None, out=None)\n\n"
             "Logits::Get: raw [rows, seq_len, vocab] (fp32 / fp16 / bf16) -> fp32 [rows, vocab] of each row's\n"
             "token_index (a host sequence; the last token when None)."),
    {nullptr, nullptr, 0, nullptr},
};
PyType_Slot kContextSlots[] = {
    {Py_tp_methods, kContextMethods},
    {Py_tp_doc, const_cast<char*>("The calls of a search context; capi.SearchContext creates and destroys the context.")},
    {0, nullptr},
};
PyType_Spec kContextSpec = {"_binding.Context", sizeof(Context), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE, kContextSlots};

// ---- Scorer: what BeamScorer derives from ---------------------------------------------------------------------

struct Scorer {
  PyObject_HEAD
  mi355x_beam_scorer* handle;
  c10::DeviceIndex device;
  int rows, max_length;
};
Scorer* Scr(PyObject* self) { return reinterpret_cast<Scorer*>(self); }

PyObject* scorer_attach(PyObject* self, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(4, "handle", "device", "rows", "max_length");
    Scr(self)->handle = static_cast<mi355x_beam_scorer*>(PyLong_AsVoidPtr(a[0]));
    Scr(self)->device = static_cast<c10::DeviceIndex>(LongOf(a[1]));
    Scr(self)->rows = static_cast<int>(LongOf(a[2]));
    Scr(self)->max_length = static_cast<int>(LongOf(a[3]));
    return NewRef(Py_None);
  });
}

MS_METHOD(step) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(3, "cand_scores", "cand_tokens", "cand_indices");
    const Tensor &sc = TensorOf(a[0]), &tok = TensorOf(a[1]), &idx = TensorOf(a[2]);
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_beam_scorer_step(Scr(self)->handle, s, Data<float>(sc), Data<int32_t>(tok), Data<int32_t>(idx));
    }
    Check(rc);
    return NewRef(Py_None);
  });
}

MS_METHOD(search_step) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(1, "logits");
    const Tensor& t = TensorOf(a[0]);
    Require(t.dim() == 2 && t.stride(1) == 1 && t.size(0) == Scr(self)->rows, "batch * beams rows of logits");
    const int dtype = DtypeCode(t.scalar_type());
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_beam_search_step(Scr(self)->handle, s, t.data_ptr(), dtype, t.stride(0), static_cast<int>(t.size(1)));
    }
    Check(rc);
    return NewRef(Py_None);
  });
}

MS_METHOD(is_done) {
  return Guarded([&]() -> PyObject* {
    if (nargs || (kwnames && PyTuple_GET_SIZE(kwnames))) Raise(PyExc_TypeError, "is_done() takes no arguments");
    void* const s = CurrentStream();
    int rc, done = 0;
    {
      Unlocked u;
      rc = ms_scorer_is_done(Scr(self)->handle, s, &done);
    }
    Check(rc);
    return PyBool_FromLong(done);
  });
}

// A copy of one of the scorer's arrays as the work of the current stream leaves it (later steps overwrite the scorer's
// own).  It is complete when the caller has it, whichever stream goes on with it.
Tensor CopyOf(const Scorer& s, const void* from, at::IntArrayRef sizes, at::ScalarType type) {
  Require(from != nullptr, "the scorer is closed");
  const Tensor out = Empty(sizes, type, c10::Device(c10::DeviceType::CUDA, s.device));
  void* const stream = CurrentStream();
  int rc;
  {
    Unlocked u;
    rc = ms_scorer_copy_words(s.handle, stream, out.data_ptr(), from, out.nbytes() / 4);
  }
  Check(rc);
  return out;
}
PyObject* get_next_scores(PyObject* self, void*) {
  return Guarded([&]() -> PyObject* { return Wrap(CopyOf(*Scr(self), mi355x_beam_scorer_next_scores(Scr(self)->handle), {Scr(self)->rows}, at::kFloat)); });
}
PyObject* get_next_tokens(PyObject* self, void*) {
  return Guarded([&]() -> PyObject* { return Wrap(CopyOf(*Scr(self), mi355x_beam_scorer_next_tokens(Scr(self)->handle), {Scr(self)->rows}, at::kInt)); });
}
PyObject* get_next_indices(PyObject* self, void*) {
  return Guarded([&]() -> PyObject* { return Wrap(CopyOf(*Scr(self), mi355x_beam_scorer_next_indices(Scr(self)->handle), {Scr(self)->rows}, at::kInt)); });
}

MS_METHOD(sequences) {
  return Guarded([&]() -> PyObject* {
    if (nargs || (kwnames && PyTuple_GET_SIZE(kwnames))) Raise(PyExc_TypeError, "sequences() takes no arguments");
    int length = 0;
    const int32_t* from = mi355x_beam_scorer_sequences(Scr(self)->handle, &length);
    const Tensor full = CopyOf(*Scr(self), from, {Scr(self)->rows, Scr(self)->max_length}, at::kInt);
    Ref view(Wrap(full.narrow(1, 0, length)));
    Ref n(PyLong_FromLong(length));
    return WrapAll({view.release(), n.release()});
  });
}

PyMethodDef kScorerMethods[] = {
    {"_attach", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(scorer_attach)), METH_FASTCALL | METH_KEYWORDS,
     "Takes the address of the mi355x_beam_scorer, its device index, batch * beams and max_length."},
    MS_ENTRY(step, "step(cand_scores, cand_tokens, cand_indices): Process + append on the candidates of beam_select."),
    MS_ENTRY(search_step, "search_step(logits): selection and scorer step in one call (BeamSearch_Cpu::SelectTop); logits\n"
                          "[batch*beams, vocab] fp32, fp16 or bf16."),
    MS_ENTRY(is_done, "is_done(): synchronises the current stream and tells whether every batch entry is done."),
    MS_ENTRY(sequences, "sequences(): (a copy of the sequences so far [batch*beams, length], length)."),
    {nullptr, nullptr, 0, nullptr},
};
PyGetSetDef kScorerGetSet[] = {
    {"next_scores", get_next_scores, nullptr, "A copy of the running scores, [batch*beams] float32.", nullptr},
    {"next_tokens", get_next_tokens, nullptr, "A copy of the tokens of the last step, [batch*beams] int32.", nullptr},
    {"next_indices", get_next_indices, nullptr, "A copy of the rows the beams continue, [batch*beams] int32.", nullptr},
    {nullptr, nullptr, nullptr, nullptr, nullptr},
};
PyType_Slot kScorerSlots[] = {
    {Py_tp_methods, kScorerMethods},
    {Py_tp_getset, kScorerGetSet},
    {Py_tp_doc, const_cast<char*>("The per-step calls of a beam scorer; capi.BeamScorer creates and destroys it.")},
    {0, nullptr},
};
PyType_Spec kScorerSpec = {"_binding.Scorer", sizeof(Scorer), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE, kScorerSlots};

// ---- module -----------------------------------------------------------------------------------------------------

PyObject* argmax_static(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
  return Guarded([&]() -> PyObject* {
    MS_PARSE(2, "logits", "out", "xf");
    const Tensor &t = TensorOf(a[0]), &out = TensorOf(a[1]);
    const Rows r(t);
    Require(out.is_cuda() && out.scalar_type() == at::kInt && out.numel() >= r.rows && out.is_contiguous(), "out is a contiguous int32 device tensor, one per row");
    const mi355x_logits_xform* xf = TruthOf(a[2]) ? XformOf(a[2]) : nullptr;
    void* const s = CurrentStream();
    int rc;
    {
      Unlocked u;
      rc = mi355x_argmax_static(s, r.data, r.dtype, r.stride, r.rows, r.vocab, xf, Data<int32_t>(out));
    }
    Check(rc);
    return NewRef(a[1]);
  });
}

PyMethodDef kModuleMethods[] = {
    MS_ENTRY(argmax_static,
             "argmax_static(logits, out, xf=None)\n\n"
             "mi355x_argmax_static: argmax of every row into the caller's `out` ([rows] int32 on the same device), on the\n"
             "current stream of the current device; needs no context and allocates nothing."),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_binding", "Native side of capi.py.", -1, kModuleMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding(void) {
  PyObject* m = PyModule_Create(&kModule);
  if (!m) return nullptr;
  PyObject* context = PyType_FromSpec(&kContextSpec);
  PyObject* scorer = PyType_FromSpec(&kScorerSpec);
  g_issue_type = reinterpret_cast<PyTypeObject*>(PyType_FromSpec(&kIssueSpec));
  if (!context || !scorer || !g_issue_type || PyModule_AddObject(m, "Context", context) < 0 || PyModule_AddObject(m, "Scorer", scorer) < 0) return nullptr;
  return m;
}
