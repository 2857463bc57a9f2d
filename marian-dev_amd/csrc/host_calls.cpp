// The host path of the operators as native code (Python module _host_calls): argument checks, output
// tensors and the call into the C ABI for one operator, without Python code in between.
//
// What bounds the small calls is the host: a decoding step is some sixty launches whose kernels run
// 3 - 12 us each, and the same checks and allocations written in Python took 15 - 20 us per call
// (transformer-big step, beam 4 x batch 32: 990 us of host work for 445 us of kernels).  Here a call
// costs its output tensors (about half a microsecond each) and the launch itself.
//
// Every function takes the arguments of the operator in its normal form - float32 tensors on the GPU,
// contiguous, quantized weights in prepared order - and returns None when it is handed anything
// else; the Python mirror (integer.py, ops.py) then checks what is wrong, raises the operator's error
// or brings the arguments into normal form and calls again.  Nothing is computed here: the kernels
// are reached through the C ABI of the library that use() was given (the shipped build, or the tuning
// build inside _lib.forced_kernel()).
//
// The interpreter lock is released around every ABI call, as ctypes does.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/as_strided_native.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <optional>
#include <utility>
#include <vector>

#include "../../include/marian_hip_int16.h"
#include "../../include/marian_hip_int8.h"
#include "../../include/marian_hip_ops.h"
#include "stream_recorded.h"

namespace {

// ---- the library in use -------------------------------------------------------------------------
#define MH_FUNCTIONS(F)                                                                                  \
  F(int8_workspace_bytes) F(int8_prepare_a) F(int8_prepare_b) F(int8_prepare_b_quantized_transposed)     \
  F(int8_affine_f32) F(int8_affine_f32_chained) F(int8_affine_f32_grouped) F(int8_proj_attention)        \
  F(int16_prepare_a) F(int16_prepare_b) F(int16_prepare_b_quantized_transposed) F(int16_affine_f32)      \
  F(int16_scratch_bytes) F(int8_affine_f32_normed) F(int8_proj_attention_normed) F(int8_proj_attention_ancestors)                                                                                 \
  F(layer_norm) F(embed) F(attention_cached) F(attention_rows) F(attention_ancestors) F(ancestors_advance)                 \
  F(select_state) F(nbest) F(nbest_words) F(nbest_beams) F(nbest_beams_workspace_bytes) F(nbest_beams_workspace_init)   \
  F(logsoftmax_nbest_beams)

struct Library {
#define F(name) decltype(&marian_hip_##name) name;
  MH_FUNCTIONS(F)
#undef F
};
Library L{};

// ---- what Python registered ---------------------------------------------------------------------
PyTypeObject* QTensorType = nullptr;
PyTypeObject* AbsMaxType = nullptr;
PyObject *type8 = nullptr, *type16 = nullptr, *raise_status = nullptr, *no_args = nullptr;
PyObject *s_data, *s_shape, *s_type, *s_prepared;

// A new reference that is dropped at the end of the scope.
struct Ref {
  PyObject* p;
  explicit Ref(PyObject* o = nullptr) : p(o) {}
  ~Ref() { Py_XDECREF(p); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
  Ref(Ref&& o) noexcept : p(o.p) { o.p = nullptr; }
  PyObject* release() { PyObject* o = p; p = nullptr; return o; }
  explicit operator bool() const { return p != nullptr; }
};

struct PyFailed {};   // a Python error is set

PyObject* ok(PyObject* o) {
  if(!o) throw PyFailed();
  return o;
}

inline bool none(PyObject* o) { return o == Py_None; }

// The tensor behind a Python object, or null.
inline const at::Tensor* tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// The tensor behind o if it is in normal form: float32, on the GPU, contiguous.
inline const at::Tensor* f32c(PyObject* o) {
  const at::Tensor* t = tensor(o);
  return t && t->scalar_type() == at::kFloat && t->is_cuda() && t->is_contiguous() ? t : nullptr;
}
// None, or a tensor in normal form; false when it is neither.
inline bool f32c_or_none(PyObject* o, const at::Tensor** t) {
  *t = nullptr;
  return none(o) || (*t = f32c(o)) != nullptr;
}
inline bool ids_type(at::ScalarType s) { return s == at::kInt || s == at::kUInt32; }

inline const float* fptr(const at::Tensor* t) { return t ? static_cast<const float*>(t->const_data_ptr()) : nullptr; }
inline float* fptr_mut(const at::Tensor& t) { return static_cast<float*>(t.data_ptr()); }

inline at::Tensor empty(at::IntArrayRef size, at::ScalarType type, c10::Device device) {
  return at::Tensor(at::detail::empty_cuda(size, type, device, std::nullopt));
}
inline PyObject* wrap(at::Tensor t) { return ok(THPVariable_Wrap(std::move(t))); }

inline hipStream_t stream_of(c10::Device d) { return c10::hip::getCurrentHIPStream(d.index()).stream(); }

inline double number(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if(v == -1.0 && PyErr_Occurred()) throw PyFailed();
  return v;
}
inline int64_t whole(PyObject* o) {
  const long long v = PyLong_AsLongLong(o);
  if(v == -1 && PyErr_Occurred()) throw PyFailed();
  return v;
}
inline bool truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if(v < 0) throw PyFailed();
  return v != 0;
}

// Calls f without the interpreter lock, and with `turn` if it is given; a status is raised as an error of `where`, or of what f
// left in *which.
template <typename F>
inline void call(const char* where, F f, const char** which = nullptr, std::mutex* turn = nullptr) {
  int status;
  {
    struct Unlocked {
      PyThreadState* s = PyEval_SaveThread();
      ~Unlocked() { PyEval_RestoreThread(s); }
    } unlocked;
    std::unique_lock<std::mutex> held;
    if(turn) held = std::unique_lock<std::mutex>(*turn);
    status = f();
  }
  if(status != MARIAN_HIP_OK) {
    if(which && **which) where = *which;
    Ref r(PyObject_CallFunction(raise_status, "is", status, where));
    if(!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, where);
    throw PyFailed();
  }
}

// ---- what stays with a stream: workspaces, for good (a graph may have recorded one), and scratch ---------
struct PerStream {
  at::Tensor workspace;              // abs-max partials, one-pass exchange
  std::mutex turn;                   // held while a call makes its launches over the workspace
  std::vector<at::Tensor> nbest;     // the last one the largest
  at::Tensor scratch;                // of the calls, not lent at the moment
};
std::map<std::pair<int, hipStream_t>, PerStream> per_stream;   // (looked up with the interpreter lock held)

PerStream& with_workspace(c10::Device d, hipStream_t st) {
  PerStream& p = per_stream[{d.index(), st}];
  if(!p.workspace.defined()) {
    at::Tensor made = empty({(int64_t)L.int8_workspace_bytes()}, at::kByte, d);
    if(!p.workspace.defined()) p.workspace = std::move(made);
  }
  return p;
}

// A call whose launches hand each other something in the workspace of its stream.  They follow each other on the stream: where threads
// share one, the launches of another thread's call would otherwise come in between and write over it.
template <typename F>
inline void call_over(PerStream& p, const char* where, F f, const char** which = nullptr) {
  void* const ws = p.workspace.data_ptr();
  const size_t bytes = (size_t)p.workspace.numel();
  call(where, [&] { return f(ws, bytes); }, which, &p.turn);
}

// Memory of one call that nobody sees afterwards: what the stream's last call gave back if that is large enough, which spares the call
// an allocation (0.45 us of a small call's 4.7), or new.  Calls of one stream run one after the other, so the next may have it as soon
// as the launches are made; a call that another thread makes meanwhile finds none and takes new memory.  A stream keeps
// one piece, the largest of up to kScratchBytes, kScratchStreams of them do, and release_scratch gives all back.
// A call that is recorded has memory of its own: its graph may be replayed on another stream.
constexpr int64_t kScratchBytes = 1 << 20;
constexpr int kScratchStreams = 16;
int scratch_kept = 0;
class Scratch {   // (made and dropped with the interpreter lock held)
 public:
  Scratch(int64_t bytes, c10::Device d, hipStream_t st) {
    int64_t size = bytes;
    if(bytes <= kScratchBytes && !marian_hip::recorded(st)) {
      home_ = &per_stream[{d.index(), st}];
      if(home_->scratch.defined()) {
        t_ = std::move(home_->scratch);
        --scratch_kept;
      }
      for(size = 4096; size < bytes;) size *= 2;
    }
    if(!t_.defined() || t_.numel() < bytes) t_ = empty({size}, at::kByte, d);
  }
  ~Scratch() {
    if(!home_) return;
    at::Tensor& kept = home_->scratch;
    if(kept.defined() ? kept.numel() >= t_.numel() : scratch_kept >= kScratchStreams) return;
    scratch_kept += !kept.defined();
    kept = std::move(t_);
  }
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;
  void* data() const { return t_.data_ptr(); }

 private:
  PerStream* home_ = nullptr;
  at::Tensor t_;
};

at::Tensor nbest_workspace(int64_t beam, int64_t batch, int64_t vocab, int64_t N, c10::Device d, hipStream_t st) {
  const int64_t need = (int64_t)L.nbest_beams_workspace_bytes(beam, batch, vocab, N);
  {
    std::vector<at::Tensor>& held = per_stream[{d.index(), st}].nbest;
    if(!held.empty() && held.back().numel() >= need) return held.back();
  }
  at::Tensor made = empty({need > 4 ? need : 4}, at::kByte, d);
  call("getNBestListOfBeams", [&] { return L.nbest_beams_workspace_init(made.data_ptr(), (size_t)made.numel(), st); });
  per_stream[{d.index(), st}].nbest.push_back(made);
  return made;
}

// ---- quantized tensors --------------------------------------------------------------------------
struct Quantized {
  Ref data, shape;
  const at::Tensor* t = nullptr;
  int64_t rows = 0, cols = 0;
  int width = 0;
};

// A matrix in q: Type::intgemm8 or Type::intgemm16, two dimensions.  prepared: 8-bit weights have to be in
// prepared order (true) or in file order (false).
bool matrix(PyObject* q, Quantized& m, bool prepared) {
  if(Py_TYPE(q) != QTensorType) return false;
  Ref type(ok(PyObject_GetAttr(q, s_type)));
  m.width = type.p == type8 ? 1 : (type.p == type16 ? 2 : 0);
  if(m.width == 0) return false;
  if(m.width == 1 || !prepared) {
    Ref p(ok(PyObject_GetAttr(q, s_prepared)));
    if(truth(p.p) != prepared) return false;
  }
  Ref shape(ok(PyObject_GetAttr(q, s_shape)));
  if(!PyTuple_Check(shape.p) || PyTuple_GET_SIZE(shape.p) != 2) return false;
  m.rows = whole(PyTuple_GET_ITEM(shape.p, 0));
  m.cols = whole(PyTuple_GET_ITEM(shape.p, 1));
  Ref data(ok(PyObject_GetAttr(q, s_data)));
  m.t = tensor(data.p);
  if(!m.t || !m.t->is_cuda() || m.t->numel() < m.rows * m.cols * m.width + 4) return false;
  std::swap(m.data.p, data.p);
  std::swap(m.shape.p, shape.p);
  return true;
}

at::Tensor quantized_buffer(int64_t elements, int width, c10::Device d) {
  return empty({(elements * width + 4 + 255) / 256 * 256}, at::kChar, d);
}

PyObject* make_quantized(at::Tensor data, PyObject* shape_tuple, PyObject* type, bool prepared) {
  Ref q(ok(QTensorType->tp_new(QTensorType, no_args, nullptr)));
  Ref d(wrap(std::move(data)));
  if(PyObject_SetAttr(q.p, s_data, d.p) || PyObject_SetAttr(q.p, s_shape, shape_tuple) ||
     PyObject_SetAttr(q.p, s_type, type) || PyObject_SetAttr(q.p, s_prepared, prepared ? Py_True : Py_False))
    throw PyFailed();
  return q.release();
}

PyObject* shape_tuple(at::IntArrayRef s) {
  Ref t(ok(PyTuple_New((Py_ssize_t)s.size())));
  for(size_t i = 0; i < s.size(); ++i) PyTuple_SET_ITEM(t.p, (Py_ssize_t)i, ok(PyLong_FromLongLong(s[i])));
  return t.release();
}

// ---- abs-max hand-over --------------------------------------------------------------------------
// None, or the slots of an AbsMax; false when it is neither.
bool absmax_in(PyObject* o, const float** p) {
  *p = nullptr;
  if(none(o)) return true;
  if(Py_TYPE(o) != AbsMaxType) return false;
  Ref data(ok(PyObject_GetAttr(o, s_data)));
  const at::Tensor* t = f32c(data.p);
  if(!t || t->numel() < MARIAN_HIP_ABSMAX_SLOTS) return false;
  *p = fptr(t);
  return true;
}
inline at::Tensor absmax_slots(c10::Device d) { return empty({MARIAN_HIP_ABSMAX_SLOTS}, at::kFloat, d); }
PyObject* make_absmax(at::Tensor slots) {
  Ref o(ok(AbsMaxType->tp_new(AbsMaxType, no_args, nullptr)));
  Ref d(wrap(std::move(slots)));
  if(PyObject_SetAttr(o.p, s_data, d.p)) throw PyFailed();
  return o.release();
}

inline at::DimVector with_last(at::IntArrayRef s, int64_t last) {
  at::DimVector v(s.begin(), s.end());
  v.back() = last;
  return v;
}

#define MH_TRY \
  HANDLE_TH_ERRORS try {
#define MH_END                       \
  }                                  \
  catch(const PyFailed&) {           \
    return nullptr;                  \
  }                                  \
  END_HANDLE_TH_ERRORS
#define MH_ARGS(count, name)                                                        \
  if(nargs != (count)) {                                                            \
    PyErr_SetString(PyExc_TypeError, name " takes another number of arguments");    \
    return nullptr;                                                                 \
  }

// ---- affine -------------------------------------------------------------------------------------
// prepareA and the multiplication: out and the quantized activations in aq.
struct Affine {
  const at::Tensor *a = nullptr, *bias = nullptr, *idx = nullptr;
  Quantized b;
  int64_t M = 0, K = 0, n_out = 0;
};

bool affine_args(PyObject* a, PyObject* bq, PyObject* bias, PyObject* shortlist, Affine& x) {
  x.a = f32c(a);
  if(!x.a || x.a->dim() < 1 || !matrix(bq, x.b, true)) return false;
  x.K = x.a->size(-1);
  if(x.b.rows != x.K) return false;
  x.M = x.K ? x.a->numel() / x.K : 0;
  x.n_out = x.b.cols;
  if(!f32c_or_none(bias, &x.bias) || (x.bias && x.bias->numel() != x.b.cols)) return false;
  if(!none(shortlist)) {
    x.idx = tensor(shortlist);
    if(!x.idx || x.b.width != 1 || !ids_type(x.idx->scalar_type()) || !x.idx->is_cuda() || !x.idx->is_contiguous()) return false;
    x.n_out = x.idx->numel();
  }
  return true;
}

// affine_or_dot(a, bQuant, bias, scale, relu, shortlist) -> out
PyObject* py_affine_or_dot(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(6, "affine_or_dot");
  Affine x;
  if(!affine_args(args[0], args[1], args[2], args[5], x)) Py_RETURN_NONE;
  const float scale = (float)number(args[3]);
  const int relu = truth(args[4]);
  const c10::Device d = x.a->device();
  at::Tensor out = empty(with_last(x.a->sizes(), x.n_out), at::kFloat, d);
  const hipStream_t st = stream_of(d);
  if(x.b.width == 2) {   // Type::intgemm16
    std::optional<Scratch> scratch;
    if(const size_t bytes = L.int16_scratch_bytes(x.M, x.K, x.b.cols)) scratch.emplace((int64_t)bytes, d, st);
    call("affineOrDot", [&] {
      return L.int16_affine_f32(fptr(x.a), scratch ? static_cast<int16_t*>(scratch->data()) : nullptr,
                                static_cast<const int16_t*>(x.b.t->const_data_ptr()), fptr(x.bias), fptr_mut(out), x.M, x.K, x.b.cols,
                                scale, relu, st);
    });
    return wrap(std::move(out));
  }
  const Scratch aq(x.M * x.K + 4, d, st);
  PerStream& ps = with_workspace(d, st);
  call_over(ps, "affineOrDot", [&](void* ws, size_t ws_bytes) {
    return L.int8_affine_f32(fptr(x.a), static_cast<int8_t*>(aq.data()), static_cast<const int8_t*>(x.b.t->const_data_ptr()),
                             fptr(x.bias), x.idx ? static_cast<const uint32_t*>(x.idx->const_data_ptr()) : nullptr,
                             x.idx ? x.n_out : 0, fptr_mut(out), x.M, x.K, x.b.cols, scale, relu, ws, ws_bytes, st);
  });
  return wrap(std::move(out));
  MH_END
}

// affine_f32(a, bQuant, bias, scale, relu, shortlist, absmax, want_absmax) -> (out, aQuant[, absmax of out])
PyObject* py_affine_f32(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(8, "affine_f32");
  Affine x;
  const float* amax = nullptr;
  if(!affine_args(args[0], args[1], args[2], args[5], x) || x.b.width != 1 || !absmax_in(args[6], &amax)) Py_RETURN_NONE;
  const float scale = (float)number(args[3]);
  const int relu = truth(args[4]);
  const bool want = truth(args[7]);
  const c10::Device d = x.a->device();
  at::Tensor out = empty(with_last(x.a->sizes(), x.n_out), at::kFloat, d);
  at::Tensor aq = quantized_buffer(x.M * x.K, 1, d);
  at::Tensor omax;
  if(want) omax = absmax_slots(d);
  const hipStream_t st = stream_of(d);
  PerStream& ps = with_workspace(d, st);
  call_over(ps, "affineOrDot", [&](void* ws, size_t ws_bytes) {
    return L.int8_affine_f32_chained(
        fptr(x.a), static_cast<int8_t*>(aq.data_ptr()), static_cast<const int8_t*>(x.b.t->const_data_ptr()), fptr(x.bias),
        x.idx ? static_cast<const uint32_t*>(x.idx->const_data_ptr()) : nullptr, x.idx ? x.n_out : 0, fptr_mut(out), x.M, x.K,
        x.b.cols, scale, relu, amax, want ? fptr_mut(omax) : nullptr, ws, ws_bytes, st);
  });
  Ref r(ok(PyTuple_New(want ? 3 : 2)));
  PyTuple_SET_ITEM(r.p, 0, wrap(std::move(out)));
  Ref shape(shape_tuple(x.a->sizes()));
  PyTuple_SET_ITEM(r.p, 1, make_quantized(std::move(aq), shape.p, type8, false));
  if(want) PyTuple_SET_ITEM(r.p, 2, make_absmax(std::move(omax)));
  return r.release();
  MH_END
}

// A list or tuple of (bQuant, bias or None) with K rows each, biases of one value a column (exact_bias: and no more);
// false when it is anything else.
constexpr int kMaxMatrices = 4;
struct Matrices {
  int n = 0;
  Quantized b[kMaxMatrices];
  const int8_t* Bq[kMaxMatrices];
  const float* bias[kMaxMatrices];
};
bool matrices(PyObject* weights, int64_t K, bool exact_bias, Matrices& m) {
  if(!PyList_Check(weights) && !PyTuple_Check(weights)) return false;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(weights);
  if(n < 1 || n > kMaxMatrices) return false;
  m.n = (int)n;
  for(int g = 0; g < m.n; ++g) {
    PyObject* w = PySequence_Fast_GET_ITEM(weights, g);
    if((!PyTuple_Check(w) && !PyList_Check(w)) || PySequence_Fast_GET_SIZE(w) != 2) return false;
    if(!matrix(PySequence_Fast_GET_ITEM(w, 0), m.b[g], true) || m.b[g].width != 1 || m.b[g].rows != K) return false;
    const at::Tensor* bias;
    if(!f32c_or_none(PySequence_Fast_GET_ITEM(w, 1), &bias) || (bias && (exact_bias ? bias->numel() != m.b[g].cols : bias->numel() < m.b[g].cols)))
      return false;
    m.Bq[g] = static_cast<const int8_t*>(m.b[g].t->const_data_ptr());
    m.bias[g] = fptr(bias);
  }
  return true;
}

// affine_f32_grouped(a, weights, scale, relu, absmax) -> ([out, ..], aQuant)
PyObject* py_affine_f32_grouped(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(5, "affine_f32_grouped");
  const at::Tensor* a = f32c(args[0]);
  Matrices w;
  const float* amax = nullptr;
  if(!a || a->dim() < 1 || !matrices(args[1], a->size(-1), true, w) || !absmax_in(args[4], &amax)) Py_RETURN_NONE;
  const float scale = (float)number(args[2]);
  const int relu = truth(args[3]);
  const int64_t K = a->size(-1), M = K ? a->numel() / K : 0;
  const c10::Device d = a->device();
  at::Tensor aq = quantized_buffer(M * K, 1, d), outs[kMaxMatrices];
  float* out[kMaxMatrices];
  int64_t N[kMaxMatrices];
  for(int g = 0; g < w.n; ++g) {
    outs[g] = empty(with_last(a->sizes(), w.b[g].cols), at::kFloat, d);
    out[g] = fptr_mut(outs[g]);
    N[g] = w.b[g].cols;
  }
  const hipStream_t st = stream_of(d);
  PerStream& ps = with_workspace(d, st);
  call_over(ps, "affineOrDot", [&](void* ws, size_t ws_bytes) {
    return L.int8_affine_f32_grouped(fptr(a), static_cast<int8_t*>(aq.data_ptr()), w.n, w.Bq, w.bias, out, N, M, K, scale, relu, amax,
                                     ws, ws_bytes, st);
  });
  Ref list(ok(PyList_New(w.n)));
  for(int g = 0; g < w.n; ++g) PyList_SET_ITEM(list.p, g, wrap(std::move(outs[g])));
  Ref shape(shape_tuple(a->sizes()));
  Ref q(make_quantized(std::move(aq), shape.p, type8, false));
  return PyTuple_Pack(2, list.p, q.p);
  MH_END
}

// The layer norm of a + add in front of a multiplication that does it itself; false when the call is not one of
// those (too many or too long rows, another form): the caller then makes two calls.
struct Normed {
  const at::Tensor* a = nullptr;
  int64_t M = 0, K = 0;
  at::Tensor x;
  marian_hip_norm_input n{};
};
bool normed(PyObject* a, PyObject* add, PyObject* ln, PyObject* eps, Normed& r) {
  r.a = f32c(a);
  const at::Tensor* s = f32c(add);
  if(!r.a || !s || r.a->dim() < 1 || r.a->sizes() != s->sizes() || !PyTuple_Check(ln) || PyTuple_GET_SIZE(ln) != 2) return false;
  const at::Tensor *gamma = f32c(PyTuple_GET_ITEM(ln, 0)), *beta = f32c(PyTuple_GET_ITEM(ln, 1));
  r.K = r.a->size(-1);
  r.M = r.K ? r.a->numel() / r.K : 0;
  if(!gamma || !beta || gamma->numel() != r.K || beta->numel() != r.K || r.M < 1 || r.M > MARIAN_HIP_NORM_MAX_ROWS ||
     r.K > MARIAN_HIP_NORM_MAX_COLS || r.K % 64 != 0)
    return false;
  for(const at::Tensor* t : {r.a, s, gamma, beta})
    if(reinterpret_cast<uintptr_t>(t->const_data_ptr()) % 16 != 0) return false;
  r.x = empty(r.a->sizes(), at::kFloat, r.a->device());
  r.n = marian_hip_norm_input{fptr(s), fptr(gamma), fptr(beta), fptr_mut(r.x), (float)number(eps)};
  return true;
}

// affine_f32_normed(a, add, (gamma, beta), eps, weights, scale, relu, want_absmax) -> (x, [out, ..], absmax or None)
PyObject* py_affine_f32_normed(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(8, "affine_f32_normed");
  Normed r;
  Matrices w;
  if(!normed(args[0], args[1], args[2], args[3], r) || !matrices(args[4], r.K, true, w)) Py_RETURN_NONE;
  const float scale = (float)number(args[5]);
  const int relu = truth(args[6]);
  const bool want = truth(args[7]);
  if(want && w.n != 1) Py_RETURN_NONE;
  const c10::Device d = r.a->device();
  at::Tensor outs[kMaxMatrices], omax;
  float* out[kMaxMatrices];
  int64_t N[kMaxMatrices], columns = 0;
  for(int g = 0; g < w.n; ++g) {
    outs[g] = empty(with_last(r.a->sizes(), w.b[g].cols), at::kFloat, d);
    out[g] = fptr_mut(outs[g]);
    N[g] = w.b[g].cols;
    columns += N[g];
  }
  if(columns == 0) Py_RETURN_NONE;
  if(want) omax = absmax_slots(d);
  const hipStream_t st = stream_of(d);
  call("affineOrDot", [&] {
    return L.int8_affine_f32_normed(fptr(r.a), &r.n, w.n, w.Bq, w.bias, out, N, r.M, r.K, scale, relu, want ? fptr_mut(omax) : nullptr, st);
  });
  Ref x(wrap(std::move(r.x))), list(ok(PyList_New(w.n)));
  for(int g = 0; g < w.n; ++g) PyList_SET_ITEM(list.p, g, wrap(std::move(outs[g])));
  if(!want) return PyTuple_Pack(3, x.p, list.p, Py_None);
  Ref m(make_absmax(std::move(omax)));
  return PyTuple_Pack(3, x.p, list.p, m.p);
  MH_END
}

// ---- quantizers ---------------------------------------------------------------------------------
// prepare_a(a, width) -> QTensor
PyObject* py_prepare_a(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(2, "prepare_a");
  const at::Tensor* a = f32c(args[0]);
  const int64_t width = whole(args[1]);
  if(!a || a->dim() < 1 || (width != 1 && width != 2)) Py_RETURN_NONE;
  const int64_t K = a->size(-1), M = K ? a->numel() / K : 0;
  const c10::Device d = a->device();
  at::Tensor out = quantized_buffer(a->numel(), (int)width, d);
  const hipStream_t st = stream_of(d);
  PerStream& ps = with_workspace(d, st);
  call_over(ps, "prepareA", [&](void* ws, size_t ws_bytes) {
    return width == 2 ? L.int16_prepare_a(fptr(a), static_cast<int16_t*>(out.data_ptr()), M, K, st)
                      : L.int8_prepare_a(fptr(a), static_cast<int8_t*>(out.data_ptr()), M, K, ws, ws_bytes, st);
  });
  Ref shape(shape_tuple(a->sizes()));
  return make_quantized(std::move(out), shape.p, width == 2 ? type16 : type8, false);
  MH_END
}

// prepare_b(w, width) -> QTensor
PyObject* py_prepare_b(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(2, "prepare_b");
  const at::Tensor* w = f32c(args[0]);
  const int64_t width = whole(args[1]);
  if(!w || w->dim() != 2 || (width != 1 && width != 2)) Py_RETURN_NONE;
  const int64_t K = w->size(0), N = w->size(1);
  const c10::Device d = w->device();
  at::Tensor out = quantized_buffer(K * N, (int)width, d);
  const hipStream_t st = stream_of(d);
  PerStream& ps = with_workspace(d, st);
  call_over(ps, "prepareB", [&](void* ws, size_t ws_bytes) {
    return width == 2 ? L.int16_prepare_b(fptr(w), static_cast<int16_t*>(out.data_ptr()), K, N, st)
                      : L.int8_prepare_b(fptr(w), static_cast<int8_t*>(out.data_ptr()), K, N, ws, ws_bytes, st);
  });
  Ref shape(shape_tuple(w->sizes()));
  return make_quantized(std::move(out), shape.p, width == 2 ? type16 : type8, true);
  MH_END
}

// prepare_stored(q) -> QTensor in prepared order
PyObject* py_prepare_stored(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(1, "prepare_stored");
  Quantized q;
  if(!matrix(args[0], q, false)) Py_RETURN_NONE;
  const c10::Device d = q.t->device();
  at::Tensor out = quantized_buffer(q.rows * q.cols, q.width, d);
  const hipStream_t st = stream_of(d);
  call("prepareAndTransposeB", [&] {
    return q.width == 2 ? L.int16_prepare_b_quantized_transposed(static_cast<const int16_t*>(q.t->const_data_ptr()),
                                                                 static_cast<int16_t*>(out.data_ptr()), q.rows, q.cols, st)
                        : L.int8_prepare_b_quantized_transposed(static_cast<const int8_t*>(q.t->const_data_ptr()),
                                                                static_cast<int8_t*>(out.data_ptr()), q.rows, q.cols, st);
  });
  return make_quantized(std::move(out), q.shape.p, q.width == 2 ? type16 : type8, true);
  MH_END
}

// ---- float operators ----------------------------------------------------------------------------
// (out, absmax of out) when it was asked for, else out
PyObject* with_absmax(at::Tensor out, at::Tensor omax) {
  if(!omax.defined()) return wrap(std::move(out));
  Ref o(wrap(std::move(out))), m(make_absmax(std::move(omax)));
  return PyTuple_Pack(2, o.p, m.p);
}

// layer_norm(x, gamma, beta, eps, add, want_absmax)
PyObject* py_layer_norm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(6, "layer_norm");
  const at::Tensor *x = f32c(args[0]), *gamma = f32c(args[1]), *beta, *add;
  if(!x || x->dim() < 1 || !gamma || !f32c_or_none(args[2], &beta) || !f32c_or_none(args[4], &add)) Py_RETURN_NONE;
  const int64_t cols = x->size(-1), rows = cols ? x->numel() / cols : 0;
  if((gamma->numel() != 1 && gamma->numel() != cols) || (beta && beta->numel() != 1 && beta->numel() != cols) ||
     (add && add->sizes() != x->sizes()))
    Py_RETURN_NONE;
  const float eps = (float)number(args[3]);
  const c10::Device d = x->device();
  at::Tensor out = empty(x->sizes(), at::kFloat, d), omax;
  if(truth(args[5])) omax = absmax_slots(d);
  const hipStream_t st = stream_of(d);
  call("layerNorm", [&] {
    return L.layer_norm(fptr(x), fptr(add), fptr(gamma), gamma->numel(), fptr(beta), beta ? beta->numel() : 0, fptr_mut(out), rows,
                        cols, eps, omax.defined() ? fptr_mut(omax) : nullptr, st);
  });
  return with_absmax(std::move(out), std::move(omax));
  MH_END
}

// embed(E, ids, scale, signal, rowsPerSignal, want_absmax, out)
PyObject* py_embed(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(7, "embed");
  const at::Tensor *E = f32c(args[0]), *ids = tensor(args[1]), *signal, *given;
  if(!E || E->dim() != 2 || !ids || !ids_type(ids->scalar_type()) || !ids->is_contiguous() || ids->device() != E->device() ||
     !f32c_or_none(args[3], &signal) || !f32c_or_none(args[6], &given))
    Py_RETURN_NONE;
  const int64_t vocab = E->size(0), dim = E->size(1), rows = ids->numel();
  if(signal && (dim == 0 || signal->numel() % dim != 0)) Py_RETURN_NONE;
  const c10::Device d = E->device();
  at::Tensor out;
  if(given) {
    if(given->device() != d || given->numel() != rows * dim) Py_RETURN_NONE;
    const float *lo = fptr(given), *table = fptr(E);
    if(lo < table + E->numel() && table < lo + given->numel()) Py_RETURN_NONE;
    out = *given;
  } else {
    at::DimVector size(ids->sizes().begin(), ids->sizes().end());
    size.push_back(dim);
    out = empty(size, at::kFloat, d);
  }
  const float scale = (float)number(args[2]);
  const int64_t per = whole(args[4]);
  at::Tensor omax;
  if(truth(args[5])) omax = absmax_slots(d);
  const hipStream_t st = stream_of(d);
  call("scaledEmbeddings", [&] {
    return L.embed(fptr(E), static_cast<const uint32_t*>(ids->const_data_ptr()), rows, vocab, dim, scale, fptr(signal), per,
                   signal ? signal->numel() / dim : 0, fptr_mut(out), omax.defined() ? fptr_mut(omax) : nullptr, st);
  });
  return with_absmax(std::move(out), std::move(omax));
  MH_END
}

// select_state(state, ids, out, used)
PyObject* py_select_state(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(4, "select_state");
  const at::Tensor *s = f32c(args[0]), *ids = tensor(args[1]), *out = f32c(args[2]);
  if(!s || !out || s->dim() != 3 || out->dim() != 3 || !ids || !ids_type(ids->scalar_type()) || !ids->is_contiguous() ||
     ids->device() != s->device() || out->size(0) != ids->numel() || out->size(1) != s->size(1) || out->size(2) != s->size(2))
    Py_RETURN_NONE;
  const int64_t used = none(args[3]) ? s->size(2) : whole(args[3]);
  const hipStream_t st = stream_of(s->device());
  call("selectState", [&] {
    return L.select_state(fptr(s), static_cast<const uint32_t*>(ids->const_data_ptr()), ids->numel(), s->size(0), s->size(1), s->size(2),
                          used, fptr_mut(*out), st);
  });
  Py_INCREF(args[2]);
  return args[2];
  MH_END
}

// attention(q, k, v, mask, rowsPerMask, want_absmax, kNew, vNew, kvLen) -> out or (out, absmax)
PyObject* py_attention(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(9, "attention");
  const at::Tensor *q = f32c(args[0]), *k = f32c(args[1]), *v = f32c(args[2]), *mask, *kn, *vn;
  if(!q || !k || !v || q->dim() < 2 || k->dim() < 2 || k->sizes() != v->sizes() || !f32c_or_none(args[3], &mask) ||
     !f32c_or_none(args[6], &kn) || !f32c_or_none(args[7], &vn))
    Py_RETURN_NONE;
  const int64_t dk = q->size(-1), m = q->size(-2), cap = k->size(-2), len = none(args[8]) ? cap : whole(args[8]);
  if(k->size(-1) != dk || len <= 0 || len > cap || m * dk == 0 || (mask && mask->numel() % len != 0)) Py_RETURN_NONE;
  for(const at::Tensor* t : {kn, vn})   // (a row for every query row)
    if(t && t->numel() < q->numel()) Py_RETURN_NONE;
  const int64_t per = whole(args[4]);
  const bool want = truth(args[5]);
  const c10::Device d = q->device();
  at::Tensor out = empty(q->sizes(), at::kFloat, d), omax;
  if(want) omax = absmax_slots(d);
  const hipStream_t st = stream_of(d);
  call("Attention", [&] {
    return L.attention_cached(fptr(q), fptr_mut(*k), fptr_mut(*v), fptr(mask), mask ? mask->numel() / len : 0, per, fptr_mut(out),
                              q->numel() / (m * dk), k->numel() / (cap * dk), m, len, cap, dk, (float)(1.0 / std::pow((double)dk, 0.5)),
                              want ? fptr_mut(omax) : nullptr, fptr(kn), fptr(vn), st);
  });
  return with_absmax(std::move(out), std::move(omax));
  MH_END
}

// ---- heads --------------------------------------------------------------------------------------
// split_heads(x [beam, batch, steps, model], heads) -> [batch * beam, heads, steps, model / heads], the same memory
PyObject* py_split_heads(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(2, "split_heads");
  const at::Tensor* x = f32c(args[0]);
  const int64_t heads = whole(args[1]);
  if(!x || x->dim() != 4 || heads <= 0 || x->size(3) % heads != 0) Py_RETURN_NONE;
  const int64_t entries = x->size(0) * x->size(1), steps = x->size(2), model = x->size(3), depth = model / heads;
  const int64_t size[4] = {entries, heads, steps, depth};
  const int64_t stride[4] = {steps * model, steps == 1 ? depth : (heads == 1 ? steps * depth : depth), steps == 1 ? depth : model, 1};
  return wrap(at::native::as_strided_tensorimpl(*x, size, stride, x->storage_offset()));
  MH_END
}

// join_heads(x [batch * beam, heads, steps, depth], beam) -> [beam, batch, steps, heads * depth] where x lies in
// memory as that tensor does; None otherwise
PyObject* py_join_heads(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(2, "join_heads");
  const at::Tensor* x = tensor(args[0]);
  const int64_t beam = whole(args[1]);
  if(!x || x->scalar_type() != at::kFloat || !x->is_cuda() || x->dim() != 4 || beam <= 0 || x->size(0) % beam != 0) Py_RETURN_NONE;
  const int64_t entries = x->size(0), heads = x->size(1), steps = x->size(2), depth = x->size(3), model = heads * depth;
  if(x->numel() == 0 || x->stride(3) != 1 || (heads > 1 && x->stride(1) != depth) || (steps > 1 && x->stride(2) != model) ||
     (entries > 1 && x->stride(0) != steps * model))
    Py_RETURN_NONE;
  const int64_t size[4] = {beam, entries / beam, steps, model};
  const int64_t stride[4] = {entries / beam * steps * model, steps * model, model, 1};
  return wrap(at::native::as_strided_tensorimpl(*x, size, stride, x->storage_offset()));
  MH_END
}

// The strides of t as [batch, heads, positions, dk]; false when it has none, or when they are not multiples of
// sixteen bytes.
bool head_strides(const at::Tensor& t, int64_t heads, int64_t (&st)[3]) {
  if(reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 != 0) return false;
  if(t.is_contiguous()) {   // (heads one behind the other, however they are counted)
    st[2] = t.size(-1);
    st[1] = t.size(-2) * st[2];
    st[0] = heads * st[1];
  } else {
    if(t.dim() != 4 || t.size(1) != heads || t.stride(3) != 1) return false;
    for(int i = 0; i < 3; ++i) st[i] = t.stride(i);
  }
  return st[0] >= 0 && st[1] >= 0 && st[2] >= 0 && (st[0] | st[1] | st[2]) % 4 == 0;
}

// attention_rows(q, k, v, mask, rowsPerMask, kvLen, want_absmax) -> out or (out, absmax): several positions per
// head, or tensors that are not contiguous.  out lies in memory as q does: head by head, or the heads of a
// position side by side.
PyObject* py_attention_rows(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(7, "attention_rows");
  const at::Tensor *q = tensor(args[0]), *k = tensor(args[1]), *v = tensor(args[2]), *mask;
  int64_t heads = 1;   // of the tensors that are not contiguous
  for(const at::Tensor* t : {q, k, v}) {
    if(!t || t->scalar_type() != at::kFloat || !t->is_cuda() || t->dim() < 3 || t->dim() > 4 || t->numel() == 0) Py_RETURN_NONE;
    if(t->dim() == 4 && !t->is_contiguous()) heads = t->size(1);
  }
  if(k->sizes() != v->sizes() || !f32c_or_none(args[3], &mask)) Py_RETURN_NONE;
  const int64_t dk = q->size(-1), m = q->size(-2), cap = k->size(-2), len = none(args[5]) ? cap : whole(args[5]), entries = q->numel() / (m * dk);
  if(k->size(-1) != dk || len <= 0 || len > cap || (mask && mask->numel() % len != 0)) Py_RETURN_NONE;
  const bool blocks = m >= MARIAN_HIP_ATTENTION_ROWS_MIN, want = truth(args[6]);
  if(blocks && (dk != 64 || len > MARIAN_HIP_ATTENTION_ROWS_MAX_LEN)) Py_RETURN_NONE;
  if(want && entries * m > MARIAN_HIP_ABSMAX_SLOTS) Py_RETURN_NONE;
  const int64_t per = whole(args[4]);
  int64_t qs[3], ks[3], vs[3], os[3];
  if(!head_strides(*q, heads, qs) || !head_strides(*k, heads, ks) || !head_strides(*v, heads, vs)) Py_RETURN_NONE;
  const c10::Device d = q->device();
  at::Tensor out, omax;
  if(q->is_contiguous()) {
    out = empty(q->sizes(), at::kFloat, d);
    head_strides(out, heads, os);
  } else {
    os[0] = m * heads * dk;
    os[1] = dk;
    os[2] = heads * dk;
    const int64_t stride[4] = {os[0], os[1], os[2], 1};
    out = at::Tensor(at::detail::empty_strided_cuda(q->sizes(), stride, at::kFloat, d));
  }
  if(want) omax = absmax_slots(d);
  const hipStream_t st = stream_of(d);
  call("Attention", [&] {
    return L.attention_rows(fptr(q), qs, fptr(k), ks, fptr(v), vs, fptr(mask), mask ? mask->numel() / len : 0, per, fptr_mut(out), os,
                            entries, k->numel() / (cap * dk), heads, m, len, dk, (float)(1.0 / std::pow((double)dk, 0.5)),
                            want ? fptr_mut(omax) : nullptr, st);
  });
  return with_absmax(std::move(out), std::move(omax));
  MH_END
}

// proj_attention(x, weights, k, v, heads, kvLen, mask, absmax, want_absmax, want_projections)
//   -> (out, aQuant[, absmax][, projections])
PyObject* py_proj_attention(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(10, "proj_attention");
  const at::Tensor *x = f32c(args[0]), *k = f32c(args[2]), *v = f32c(args[3]), *mask;
  Matrices w;
  const float* amax = nullptr;
  if(!x || x->dim() < 1 || !k || !v || k->dim() < 2 || k->size(-1) != 64 || k->sizes() != v->sizes() ||
     !matrices(args[1], x->size(-1), false, w) || (w.n != 1 && w.n != 3) || !f32c_or_none(args[6], &mask) || !absmax_in(args[7], &amax))
    Py_RETURN_NONE;
  const int64_t heads = whole(args[4]), N = heads * 64, K = x->size(-1), M = K ? x->numel() / K : 0;
  const int64_t cap = k->size(-2), len = none(args[5]) ? cap : whole(args[5]);
  for(int g = 0; g < w.n; ++g)
    if(w.b[g].cols != N) Py_RETURN_NONE;
  if(cap <= 0 || len <= 0 || (mask && mask->numel() % len != 0)) Py_RETURN_NONE;
  const bool want = truth(args[8]), want_proj = truth(args[9]);
  const c10::Device d = x->device();
  const at::DimVector size = with_last(x->sizes(), N);
  at::Tensor out = empty(size, at::kFloat, d), aq = quantized_buffer(M * K, 1, d), omax, projections[3];
  float* proj[3] = {nullptr, nullptr, nullptr};
  if(want) omax = absmax_slots(d);
  if(want_proj)
    for(int g = 0; g < w.n; ++g) {
      projections[g] = empty(size, at::kFloat, d);
      proj[g] = fptr_mut(projections[g]);
    }
  const hipStream_t st = stream_of(d);
  PerStream& ps = with_workspace(d, st);
  call_over(ps, "ProjectedAttention", [&](void* ws, size_t ws_bytes) {
    return L.int8_proj_attention(fptr(x), static_cast<int8_t*>(aq.data_ptr()), w.n, w.Bq, w.bias, proj, M, K, heads, fptr_mut(*k),
                                 fptr_mut(*v), k->numel() / (cap * 64), len, cap, fptr(mask), mask ? mask->numel() / len : 0, 1.0f / 8.0f,
                                 fptr_mut(out), amax, want ? fptr_mut(omax) : nullptr, ws, ws_bytes, st);
  });
  Ref r(ok(PyTuple_New(2 + (want ? 1 : 0) + (want_proj ? 1 : 0))));
  PyTuple_SET_ITEM(r.p, 0, wrap(std::move(out)));
  Ref shape(shape_tuple(x->sizes()));
  PyTuple_SET_ITEM(r.p, 1, make_quantized(std::move(aq), shape.p, type8, false));
  if(want) PyTuple_SET_ITEM(r.p, 2, make_absmax(std::move(omax)));
  if(want_proj) {
    Ref list(ok(PyList_New(w.n)));
    for(int g = 0; g < w.n; ++g) PyList_SET_ITEM(list.p, g, wrap(std::move(projections[g])));
    PyTuple_SET_ITEM(r.p, want ? 3 : 2, list.release());
  }
  return r.release();
  MH_END
}

// proj_attention_normed(a, add, (gamma, beta), eps, weights, k, v, heads, kvLen, mask, want_projections)
//   -> (x, out, absmax of out, [projections] or None)
PyObject* py_proj_attention_normed(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(11, "proj_attention_normed");
  Normed r;
  const at::Tensor *k = f32c(args[5]), *v = f32c(args[6]), *mask;
  Matrices w;
  if(!normed(args[0], args[1], args[2], args[3], r) || r.K % 128 != 0 || !k || !v || k->dim() < 2 || k->size(-1) != 64 ||
     k->sizes() != v->sizes() || !matrices(args[4], r.K, true, w) || (w.n != 1 && w.n != 3) || !f32c_or_none(args[9], &mask))
    Py_RETURN_NONE;
  const int64_t heads = whole(args[7]), N = heads * 64, cap = k->size(-2), len = none(args[8]) ? cap : whole(args[8]);
  for(int g = 0; g < w.n; ++g)
    if(w.b[g].cols != N) Py_RETURN_NONE;
  if(cap <= 0 || len <= 0 || (mask && mask->numel() % len != 0)) Py_RETURN_NONE;
  const bool want_proj = truth(args[10]);
  const c10::Device d = r.a->device();
  const at::DimVector size = with_last(r.a->sizes(), N);
  at::Tensor out = empty(size, at::kFloat, d), omax = absmax_slots(d), projections[3];
  float* proj[3] = {nullptr, nullptr, nullptr};
  if(want_proj)
    for(int g = 0; g < w.n; ++g) {
      projections[g] = empty(size, at::kFloat, d);
      proj[g] = fptr_mut(projections[g]);
    }
  const hipStream_t st = stream_of(d);
  call("ProjectedAttention", [&] {
    return L.int8_proj_attention_normed(fptr(r.a), &r.n, w.n, w.Bq, w.bias, proj, r.M, r.K, heads, fptr_mut(*k), fptr_mut(*v),
                                        k->numel() / (cap * 64), len, cap, fptr(mask), mask ? mask->numel() / len : 0, 1.0f / 8.0f,
                                        fptr_mut(out), fptr_mut(omax), st);
  });
  Ref x(wrap(std::move(r.x))), o(wrap(std::move(out))), m(make_absmax(std::move(omax)));
  if(!want_proj) return PyTuple_Pack(4, x.p, o.p, m.p, Py_None);
  Ref list(ok(PyList_New(w.n)));
  for(int g = 0; g < w.n; ++g) PyList_SET_ITEM(list.p, g, wrap(std::move(projections[g])));
  return PyTuple_Pack(4, x.p, o.p, m.p, list.p);
  MH_END
}

// proj_attention_ancestors(a, add or None, (gamma, beta), eps, weights, k, v, ancestors, kvLen, absmax, want_projections)
//   -> (x, out, absmax of out, [projections] or None); add None: x is a itself
PyObject* py_proj_attention_ancestors(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(11, "proj_attention_ancestors");
  const bool with_norm = !none(args[1]);
  Normed r;
  const at::Tensor *k = f32c(args[5]), *v = f32c(args[6]), *anc = tensor(args[7]);
  const float* amax = nullptr;
  if(with_norm ? !normed(args[0], args[1], args[2], args[3], r) : !(r.a = f32c(args[0]))) Py_RETURN_NONE;
  if(r.a->dim() < 1) Py_RETURN_NONE;
  r.K = r.a->size(-1);
  r.M = r.K ? r.a->numel() / r.K : 0;
  Matrices w;
  const int64_t heads = r.K / 64;
  if(r.M < 1 || r.K % 128 != 0 || r.K > 1024 || r.M * heads > MARIAN_HIP_ABSMAX_SLOTS || !k || !v || k->dim() != 3 || k->size(-1) != 64 ||
     k->sizes() != v->sizes() || k->size(0) != r.M * heads || !anc || !ids_type(anc->scalar_type()) || anc->device() != r.a->device() ||
     !anc->is_contiguous() || anc->dim() != 2 || anc->size(0) != r.M || anc->size(1) != k->size(1) ||
     !matrices(args[4], r.K, true, w) || w.n != 3 || !absmax_in(args[9], &amax))
    Py_RETURN_NONE;
  for(int g = 0; g < 3; ++g)
    if(w.b[g].cols != r.K) Py_RETURN_NONE;
  const int64_t len = whole(args[8]), cap = k->size(1);
  if(len < 1 || len > cap || len > 512) Py_RETURN_NONE;
  const bool want_proj = truth(args[10]);
  const c10::Device d = r.a->device();
  at::Tensor out = empty(r.a->sizes(), at::kFloat, d), omax = absmax_slots(d), projections[3], aq;
  if(!with_norm) aq = quantized_buffer(r.M * r.K, 1, d);
  float* proj[3] = {nullptr, nullptr, nullptr};
  if(want_proj)
    for(int g = 0; g < 3; ++g) {
      projections[g] = empty(r.a->sizes(), at::kFloat, d);
      proj[g] = fptr_mut(projections[g]);
    }
  const hipStream_t st = stream_of(d);
  PerStream& ps = with_workspace(d, st);
  call_over(ps, "ProjectedAttention", [&](void* ws, size_t ws_bytes) {
    return L.int8_proj_attention_ancestors(fptr(r.a), with_norm ? &r.n : nullptr, with_norm ? nullptr : static_cast<int8_t*>(aq.data_ptr()),
                                           w.Bq, w.bias, proj, r.M, r.K, heads, fptr_mut(*k), fptr_mut(*v), len, cap,
                                           static_cast<const uint32_t*>(anc->const_data_ptr()), 1.0f / 8.0f, fptr_mut(out), amax,
                                           fptr_mut(omax), ws, ws_bytes, st);
  });
  Ref x(with_norm ? wrap(std::move(r.x)) : (Py_INCREF(args[0]), args[0])), o(wrap(std::move(out))), m(make_absmax(std::move(omax)));
  if(!want_proj) return PyTuple_Pack(4, x.p, o.p, m.p, Py_None);
  Ref list(ok(PyList_New(3)));
  for(int g = 0; g < 3; ++g) PyList_SET_ITEM(list.p, g, wrap(std::move(projections[g])));
  return PyTuple_Pack(4, x.p, o.p, m.p, list.p);
  MH_END
}

// ---- the layers of a decoding step ---------------------------------------------------------------
// The calls of a decoding step's layers, one after the other, as decoder_step.py makes them one by one: the same entry
// points of the library on the same values.  Made from Python, each cost 5.5 us of host time (arguments, three tensors, two
// objects, the launch), more than the kernels of a small step take; here everything is looked at first, what lies between the
// layers is one allocation, and the launches follow each other without the interpreter lock.
struct DecoderMatrix {
  Quantized b;
  at::Tensor bias;
  const int8_t* weights() const { return static_cast<const int8_t*>(b.t->const_data_ptr()); }
  const float* shift() const { return bias.defined() ? static_cast<const float*>(bias.const_data_ptr()) : nullptr; }
};
struct DecoderNorm {
  at::Tensor gamma, beta;
};
struct DecoderLayer {
  DecoderMatrix qkv[3], o, cq, co, w1, w2;
  DecoderNorm ln1, ln2, ln3;
  at::Tensor k, v, kc, vc;   // caches of the target positions, and the source's
};

// Whether a layer's vector can be read as the kernels do: n values on device d, from an address of whole vectors.
inline bool decoder_vector(const at::Tensor* t, int64_t n, c10::Device d) {
  return t && t->numel() == n && t->device() == d && reinterpret_cast<uintptr_t>(t->const_data_ptr()) % 16 == 0;
}
// A (bQuant, bias or None) with K rows and N columns (0: any number), the bias of one value a column.
bool decoder_matrix(PyObject* w, int64_t K, int64_t N, c10::Device d, DecoderMatrix& m) {
  if(!w || !PyTuple_Check(w) || PyTuple_GET_SIZE(w) != 2) return false;
  const at::Tensor* bias;
  if(!matrix(PyTuple_GET_ITEM(w, 0), m.b, true) || m.b.width != 1 || m.b.rows != K || (N && m.b.cols != N) ||
     m.b.t->device() != d || !f32c_or_none(PyTuple_GET_ITEM(w, 1), &bias) || (bias && !decoder_vector(bias, m.b.cols, d)))
    return false;
  if(bias) m.bias = *bias;
  return true;
}
bool decoder_norm(PyObject* ln, int64_t n, c10::Device d, DecoderNorm& out) {
  if(!ln || !PyTuple_Check(ln) || PyTuple_GET_SIZE(ln) != 2) return false;
  const at::Tensor *gamma = f32c(PyTuple_GET_ITEM(ln, 0)), *beta = f32c(PyTuple_GET_ITEM(ln, 1));
  if(!decoder_vector(gamma, n, d) || !decoder_vector(beta, n, d)) return false;
  out.gamma = *gamma;
  out.beta = *beta;
  return true;
}
// A cache of `entries` entries of [.., 64] (all of one size) at place i of a list.
bool decoder_cache(PyObject* list, Py_ssize_t i, int64_t entries, c10::Device d, int64_t& capacity, at::Tensor& out) {
  const at::Tensor* t = f32c(PyList_GET_ITEM(list, i));
  if(!t || t->device() != d || t->dim() != 3 || t->size(2) != 64 || (entries && t->size(0) != entries) || (capacity && t->size(1) != capacity)) return false;
  capacity = t->size(1);
  out = *t;
  return true;
}

// decoder_layers(x, absmax of x, layers, Kself, Vself, Kenc, Venc, mask, ancestors or None, heads, kvLen, eps, (output matrix, bias))
//   -> scores [M, vocabulary]; layers: dicts of Wq, Wk, Wv, Wo, cWq, cWo, W1, W2 (bQuant, bias) and ln1, ln2, ln3 (gamma, beta)
PyObject* py_decoder_layers(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(13, "decoder_layers");
  const at::Tensor *x = f32c(args[0]), *mask, *anc = nullptr;
  const float* amax = nullptr;
  for(int i : {2, 3, 4, 5, 6})
    if(!PyList_Check(args[i]) || PyList_GET_SIZE(args[i]) != PyList_GET_SIZE(args[2])) Py_RETURN_NONE;
  const Py_ssize_t n = PyList_GET_SIZE(args[2]);
  if(!x || x->dim() != 2 || n < 1 || !absmax_in(args[1], &amax) || !amax || !f32c_or_none(args[7], &mask)) Py_RETURN_NONE;
  const int64_t M = x->size(0), d = x->size(1), heads = whole(args[9]), len = whole(args[10]);
  const float eps = (float)number(args[11]);
  if(M < 1 || d % 128 != 0 || d > 1024 || d != heads * 64 || M * heads > MARIAN_HIP_ABSMAX_SLOTS || len < 1 || len > 512 ||
     reinterpret_cast<uintptr_t>(x->const_data_ptr()) % 16 != 0)
    Py_RETURN_NONE;
  if(!none(args[8])) {
    anc = tensor(args[8]);
    if(M > 256 || !anc || !ids_type(anc->scalar_type()) || anc->device() != x->device() || !anc->is_contiguous() || anc->dim() != 2 || anc->size(0) != M)
      Py_RETURN_NONE;
  }
  const c10::Device dev = x->device();
  if(mask && mask->device() != dev) Py_RETURN_NONE;
  const bool few = M <= MARIAN_HIP_NORM_MAX_ROWS;   // the layer norms need no launches of their own
  int64_t cap = anc ? anc->size(1) : 0, source = 0, widest = d;
  std::vector<DecoderLayer> layers((size_t)n);
  for(Py_ssize_t i = 0; i < n; ++i) {
    DecoderLayer& l = layers[(size_t)i];
    PyObject* dict = PyList_GET_ITEM(args[2], i);
    if(!PyDict_Check(dict)) Py_RETURN_NONE;
    auto item = [&](const char* name) { return PyDict_GetItemString(dict, name); };
    int64_t source_cap = source;
    if(!decoder_matrix(item("Wq"), d, d, dev, l.qkv[0]) || !decoder_matrix(item("Wk"), d, d, dev, l.qkv[1]) || !decoder_matrix(item("Wv"), d, d, dev, l.qkv[2]) ||
       !decoder_matrix(item("Wo"), d, d, dev, l.o) || !decoder_matrix(item("cWq"), d, d, dev, l.cq) || !decoder_matrix(item("cWo"), d, d, dev, l.co) ||
       !decoder_matrix(item("W1"), d, 0, dev, l.w1) || !decoder_matrix(item("W2"), l.w1.b.cols, d, dev, l.w2) ||
       !decoder_norm(item("ln1"), d, dev, l.ln1) || !decoder_norm(item("ln2"), d, dev, l.ln2) || !decoder_norm(item("ln3"), d, dev, l.ln3) ||
       !decoder_cache(args[3], i, M * heads, dev, cap, l.k) || !decoder_cache(args[4], i, M * heads, dev, cap, l.v) ||
       !decoder_cache(args[5], i, i ? layers[0].kc.size(0) : 0, dev, source_cap, l.kc) || !decoder_cache(args[6], i, l.kc.size(0), dev, source_cap, l.vc))
      Py_RETURN_NONE;
    source = source_cap;
    widest = std::max(widest, l.w1.b.cols);
  }
  DecoderMatrix last;
  if(!decoder_matrix(args[12], d, 0, dev, last) || len > cap || source < 1 || source > 512 || widest % 64 != 0 || last.b.cols < 1 ||
     layers[0].kc.size(0) < 1 || (mask && (mask->numel() < 1 || mask->numel() % source != 0)))
    Py_RETURN_NONE;
  const int64_t entries = layers[0].kc.size(0), masks = mask ? mask->numel() / source : 0;
  // what lies between the calls: rows of d (x twice, for one layer's and the next's), of the widest, slots, quantized activations
  enum { kO, kA, kX1, kCo, kCa, kX2, kF2, kXa, kXb, kRows };
  const int64_t row_bytes = (M * d * 4 + 255) / 256 * 256, wide_bytes = (M * widest * 4 + 255) / 256 * 256;
  const int64_t slot_bytes = MARIAN_HIP_ABSMAX_SLOTS * 4;
  enum { kOMax, kX1Max, kCoMax, kX2Max, kF1Max, kXMax, kSlots };
  at::Tensor arena = empty({kRows * row_bytes + wide_bytes + kSlots * slot_bytes + M * widest + 256}, at::kByte, dev);
  char* const base = static_cast<char*>(arena.data_ptr());
  auto rows = [&](int i) { return reinterpret_cast<float*>(base + i * row_bytes); };
  auto slots = [&](int i) { return reinterpret_cast<float*>(base + kRows * row_bytes + wide_bytes + i * slot_bytes); };
  float* const f1 = reinterpret_cast<float*>(base + kRows * row_bytes);
  int8_t* const aq = reinterpret_cast<int8_t*>(base + kRows * row_bytes + wide_bytes + kSlots * slot_bytes);
  at::Tensor scores = empty({M, last.b.cols}, at::kFloat, dev);
  float* const out = fptr_mut(scores);
  const hipStream_t st = stream_of(dev);
  PerStream& ps = with_workspace(dev, st);
  const uint32_t* const table = anc ? static_cast<const uint32_t*>(anc->const_data_ptr()) : nullptr;
  const char* where = "";
  call_over(ps, "decoder step", [&](void* wp, size_t wn) {
    auto affine = [&](const float* a, const DecoderMatrix& w, float* to, int relu, const float* in_max, float* out_max) {
      return L.int8_affine_f32_chained(a, aq, w.weights(), w.shift(), nullptr, 0, to, M, w.b.rows, w.b.cols, 1.0f, relu, in_max, out_max, wp, wn, st);
    };
    auto norm = [&](const float* a, const float* add, const DecoderNorm& ln, float* to, float* out_max) {
      return L.layer_norm(a, add, fptr(&ln.gamma), d, fptr(&ln.beta), d, to, M, d, eps, out_max, st);
    };
    auto normed = [&](const float* add, const DecoderNorm& ln, float* to) {
      return marian_hip_norm_input{add, fptr(&ln.gamma), fptr(&ln.beta), to, eps};
    };
    auto affine_of_norm = [&](const float* a, const marian_hip_norm_input& ln, const DecoderMatrix& w, float* to, int relu, float* out_max) {
      const int8_t* Bq = w.weights();
      const float* bias = w.shift();
      const int64_t N = w.b.cols;
      return L.int8_affine_f32_normed(a, &ln, 1, &Bq, &bias, &to, &N, M, d, 1.0f, relu, out_max, st);
    };
    const float* now = fptr(x);
    const float* now_max = amax;
    float* none_out[3] = {nullptr, nullptr, nullptr};
    int status = MARIAN_HIP_OK;
#define MH_STEP(name, expr)                      \
  do {                                           \
    status = (expr);                             \
    if(status != MARIAN_HIP_OK) {                \
      where = name;                              \
      return status;                             \
    }                                            \
  } while(0)
    for(size_t i = 0; i < layers.size(); ++i) {
      const DecoderLayer& l = layers[i];
      const int8_t* Bq[3] = {l.qkv[0].weights(), l.qkv[1].weights(), l.qkv[2].weights()};
      const float* bias[3] = {l.qkv[0].shift(), l.qkv[1].shift(), l.qkv[2].shift()};
      float *k = fptr_mut(l.k), *v = fptr_mut(l.v), *next = rows(i % 2 ? kXb : kXa);
      // self-attention; behind a layer of few rows its input is that layer's last norm, taken on the way
      const bool pending = few && i > 0;
      const marian_hip_norm_input last_norm = pending ? normed(rows(kX2), layers[i - 1].ln3, next) : marian_hip_norm_input{};
      const float* in = pending ? rows(kF2) : now;
      if(anc)
        MH_STEP("ProjectedAttention", L.int8_proj_attention_ancestors(in, pending ? &last_norm : nullptr, pending ? nullptr : aq, Bq, bias, none_out, M, d,
                                                                     heads, k, v, len, cap, table, 1.0f / 8.0f, rows(kO), pending ? nullptr : now_max,
                                                                     slots(kOMax), wp, wn, st));
      else if(pending)
        MH_STEP("ProjectedAttention", L.int8_proj_attention_normed(in, &last_norm, 3, Bq, bias, none_out, M, d, heads, k, v, M * heads, len, cap, nullptr,
                                                                  0, 1.0f / 8.0f, rows(kO), slots(kOMax), st));
      else
        MH_STEP("ProjectedAttention", L.int8_proj_attention(in, aq, 3, Bq, bias, none_out, M, d, heads, k, v, M * heads, len, cap, nullptr, 0,
                                                           1.0f / 8.0f, rows(kO), now_max, slots(kOMax), wp, wn, st));
      if(pending) now = next;
      MH_STEP("affineOrDot", affine(rows(kO), l.o, rows(kA), 0, slots(kOMax), nullptr));
      // attention over the source
      const int8_t* cBq = l.cq.weights();
      const float* cbias = l.cq.shift();
      float *kc = fptr_mut(l.kc), *vc = fptr_mut(l.vc);
      if(few) {
        const marian_hip_norm_input ln = normed(now, l.ln1, rows(kX1));
        MH_STEP("ProjectedAttention", L.int8_proj_attention_normed(rows(kA), &ln, 1, &cBq, &cbias, none_out, M, d, heads, kc, vc, entries, source, source,
                                                                  fptr(mask), masks, 1.0f / 8.0f, rows(kCo), slots(kCoMax), st));
      } else {
        MH_STEP("layerNorm", norm(rows(kA), now, l.ln1, rows(kX1), slots(kX1Max)));
        MH_STEP("ProjectedAttention", L.int8_proj_attention(rows(kX1), aq, 1, &cBq, &cbias, none_out, M, d, heads, kc, vc, entries, source, source,
                                                           fptr(mask), masks, 1.0f / 8.0f, rows(kCo), slots(kX1Max), slots(kCoMax), wp, wn, st));
      }
      MH_STEP("affineOrDot", affine(rows(kCo), l.co, rows(kCa), 0, slots(kCoMax), nullptr));
      // feed-forward block
      if(few) {
        MH_STEP("affineOrDot", affine_of_norm(rows(kCa), normed(rows(kX1), l.ln2, rows(kX2)), l.w1, f1, 1, slots(kF1Max)));
      } else {
        MH_STEP("layerNorm", norm(rows(kCa), rows(kX1), l.ln2, rows(kX2), slots(kX2Max)));
        MH_STEP("affineOrDot", affine(rows(kX2), l.w1, f1, 1, slots(kX2Max), slots(kF1Max)));
      }
      MH_STEP("affineOrDot", affine(f1, l.w2, rows(kF2), 0, slots(kF1Max), nullptr));
      if(!few) {
        MH_STEP("layerNorm", norm(rows(kF2), rows(kX2), l.ln3, next, slots(kXMax)));
        now = next;
        now_max = slots(kXMax);
      }
    }
    if(few) MH_STEP("affineOrDot", affine_of_norm(rows(kF2), normed(rows(kX2), layers.back().ln3, rows(layers.size() % 2 ? kXb : kXa)), last, out, 0, nullptr));
    else MH_STEP("affineOrDot", affine(now, last, out, 0, now_max, nullptr));
#undef MH_STEP
    return status;
  }, &where);
  return wrap(std::move(scores));
  MH_END
}

// attention_ancestors(q, k, v, ancestors, kvLen, kNew, vNew, want_absmax) -> out or (out, absmax)
PyObject* py_attention_ancestors(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(8, "attention_ancestors");
  const at::Tensor *q = f32c(args[0]), *k = f32c(args[1]), *v = f32c(args[2]), *anc = tensor(args[3]), *kn = f32c(args[5]), *vn = f32c(args[6]);
  if(!q || !k || !v || !kn || !vn || k->dim() != 3 || k->sizes() != v->sizes() || !anc || !ids_type(anc->scalar_type()) ||
     !anc->is_cuda() || !anc->is_contiguous() || anc->dim() != 2 || anc->size(1) != k->size(1) || anc->size(0) <= 0 ||
     k->size(0) % anc->size(0) != 0)
    Py_RETURN_NONE;
  const int64_t entries = k->size(0), cap = k->size(1), dk = k->size(2), hyps = anc->size(0), len = whole(args[4]);
  if(q->numel() != entries * dk || kn->numel() != entries * dk || vn->numel() != entries * dk) Py_RETURN_NONE;
  const c10::Device d = q->device();
  at::Tensor out = empty(q->sizes(), at::kFloat, d), omax;
  if(truth(args[7])) omax = absmax_slots(d);
  const hipStream_t st = stream_of(d);
  call("AttentionByAncestors", [&] {
    return L.attention_ancestors(fptr(q), fptr_mut(*k), fptr_mut(*v), fptr_mut(out), hyps, entries / hyps, len, cap, dk,
                                 (float)(1.0 / std::pow((double)dk, 0.5)), omax.defined() ? fptr_mut(omax) : nullptr, fptr(kn), fptr(vn),
                                 static_cast<const uint32_t*>(anc->const_data_ptr()), st);
  });
  return with_absmax(std::move(out), std::move(omax));
  MH_END
}

// ancestors_advance(prev, parents, lenPrev, out)
PyObject* py_ancestors_advance(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(4, "ancestors_advance");
  const at::Tensor *prev = tensor(args[0]), *par = tensor(args[1]), *out = tensor(args[3]);
  if(!prev || !par || !out || prev->scalar_type() != at::kInt || out->scalar_type() != at::kInt || prev->dim() != 2 ||
     prev->sizes() != out->sizes() || !prev->is_cuda() || !prev->is_contiguous() || !out->is_contiguous() ||
     !ids_type(par->scalar_type()) || !par->is_contiguous() || par->numel() != prev->size(0) ||
     par->device() != prev->device() || out->device() != prev->device())
    Py_RETURN_NONE;
  const int64_t len = whole(args[2]);
  const hipStream_t st = stream_of(prev->device());
  call("advanceAncestors", [&] {
    return L.ancestors_advance(static_cast<const uint32_t*>(prev->const_data_ptr()), static_cast<const uint32_t*>(par->const_data_ptr()),
                               prev->size(0), prev->size(1), len, static_cast<uint32_t*>(out->data_ptr()), st);
  });
  Py_INCREF(args[3]);
  return args[3];
  MH_END
}

// ---- n-best -------------------------------------------------------------------------------------
// nbest(scores, N): scores [dimBatch, ..]
PyObject* py_nbest(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(2, "nbest");
  const at::Tensor* s = f32c(args[0]);
  if(!s || s->dim() < 1) Py_RETURN_NONE;
  const int64_t N = whole(args[1]), batch = s->size(0), row = batch ? s->numel() / batch : 0;
  const c10::Device d = s->device();
  at::Tensor vals = empty({batch * N}, at::kFloat, d), keys = empty({batch * N}, at::kInt, d);
  const hipStream_t st = stream_of(d);
  call("getNBestList", [&] {
    return L.nbest(fptr(s), batch, row, N, fptr_mut(vals), static_cast<uint32_t*>(keys.data_ptr()), st);
  });
  Ref a(wrap(std::move(vals))), b(wrap(std::move(keys)));
  return PyTuple_Pack(2, a.p, b.p);
  MH_END
}

// nbest_words(scores, N, ids): scores [.., cols], ids [cols] or None
PyObject* py_nbest_words(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(3, "nbest_words");
  const at::Tensor *s = f32c(args[0]), *ids = nullptr;
  if(!s || s->dim() < 1) Py_RETURN_NONE;
  const int64_t N = whole(args[1]), cols = s->size(-1), rows = cols ? s->numel() / cols : 0;
  if(!none(args[2]) && (!(ids = tensor(args[2])) || !ids_type(ids->scalar_type()) || ids->device() != s->device() ||
                        !ids->is_contiguous() || ids->numel() != cols))
    Py_RETURN_NONE;
  const c10::Device d = s->device();
  at::Tensor vals = empty({rows, N}, at::kFloat, d), words = empty({rows, N}, at::kLong, d);
  const hipStream_t st = stream_of(d);
  call("getNBestList", [&] {   // (no rows: refused)
    return L.nbest_words(fptr(s), rows, rows ? cols : 0, N, ids ? static_cast<const uint32_t*>(ids->const_data_ptr()) : nullptr,
                         fptr_mut(vals), static_cast<int64_t*>(words.data_ptr()), st);
  });
  Ref a(wrap(std::move(vals))), b(wrap(std::move(words)));
  return PyTuple_Pack(2, a.p, b.p);
  MH_END
}

// nbest_beams(scores, N): scores [beam, .., vocab]
PyObject* py_nbest_beams(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(2, "nbest_beams");
  const at::Tensor* s = f32c(args[0]);
  if(!s || s->dim() < 2) Py_RETURN_NONE;
  const int64_t N = whole(args[1]), beam = s->size(0), vocab = s->size(-1), batch = beam * vocab != 0 ? s->numel() / (beam * vocab) : 0;
  const c10::Device d = s->device();
  at::Tensor vals = empty({batch * N}, at::kFloat, d), keys = empty({batch * N}, at::kInt, d);
  const hipStream_t st = stream_of(d);
  const at::Tensor ws = nbest_workspace(beam, batch, vocab, N, d, st);
  call("getNBestListOfBeams", [&] {
    return L.nbest_beams(fptr(s), beam, batch, vocab, N, fptr_mut(vals), static_cast<uint32_t*>(keys.data_ptr()), ws.data_ptr(),
                         (size_t)ws.numel(), st);
  });
  Ref a(wrap(std::move(vals))), b(wrap(std::move(keys)));
  return PyTuple_Pack(2, a.p, b.p);
  MH_END
}

// logsoftmax_nbest_beams(logits, N, pathScores, want_logprobs): the sizes of the one-launch form only
PyObject* py_logsoftmax_nbest_beams(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(4, "logsoftmax_nbest_beams");
  const at::Tensor *s = f32c(args[0]), *add;
  if(!s || s->dim() < 2 || !f32c_or_none(args[2], &add)) Py_RETURN_NONE;
  const int64_t N = whole(args[1]), beam = s->size(0), vocab = s->size(-1), batch = beam * vocab != 0 ? s->numel() / (beam * vocab) : 0;
  if(vocab % 4 != 0 || vocab <= 4096 || vocab > 32768 || reinterpret_cast<uintptr_t>(s->const_data_ptr()) % 16 != 0 ||
     (add && add->numel() != beam * batch))
    Py_RETURN_NONE;
  const c10::Device d = s->device();
  at::Tensor vals = empty({batch * N}, at::kFloat, d), keys = empty({batch * N}, at::kInt, d), lp;
  if(truth(args[3])) lp = empty(s->sizes(), at::kFloat, d);
  const hipStream_t st = stream_of(d);
  const at::Tensor ws = nbest_workspace(beam, batch, vocab, N, d, st);
  call("logsoftmaxNBestOfBeams", [&] {
    return L.logsoftmax_nbest_beams(fptr(s), fptr(add), lp.defined() ? fptr_mut(lp) : nullptr, beam, batch, vocab, N, fptr_mut(vals),
                                    static_cast<uint32_t*>(keys.data_ptr()), ws.data_ptr(), (size_t)ws.numel(), st);
  });
  Ref a(wrap(std::move(vals))), b(wrap(std::move(keys)));
  if(!lp.defined()) return PyTuple_Pack(2, a.p, b.p);
  Ref c(wrap(std::move(lp)));
  return PyTuple_Pack(3, a.p, b.p, c.p);
  MH_END
}

// ---- module -------------------------------------------------------------------------------------
// workspace(device index) -> the workspace of that device's current stream
PyObject* py_workspace(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(1, "workspace");
  const c10::Device d(c10::kCUDA, (c10::DeviceIndex)whole(args[0]));
  return wrap(with_workspace(d, stream_of(d)).workspace);
  MH_END
}

// release_scratch(): the scratch of all streams goes back to torch's allocator
PyObject* py_release_scratch(PyObject*, PyObject* const*, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(0, "release_scratch");
  for(auto& p : per_stream) p.second.scratch = at::Tensor();
  scratch_kept = 0;
  Py_RETURN_NONE;
  MH_END
}

// use(handle): takes the C ABI's functions from a loaded library (a dlopen handle)
PyObject* py_use(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(1, "use");
  void* h = PyLong_AsVoidPtr(args[0]);
  if(!h && PyErr_Occurred()) return nullptr;
  Library n{};
#define F(name)                                                                          \
  n.name = reinterpret_cast<decltype(&marian_hip_##name)>(dlsym(h, "marian_hip_" #name)); \
  if(!n.name) {                                                                          \
    PyErr_SetString(PyExc_ImportError, "marian_hip_" #name " is not in the library");     \
    return nullptr;                                                                      \
  }
  MH_FUNCTIONS(F)
#undef F
  L = n;
  Py_RETURN_NONE;
  MH_END
}

// setup(QTensor, AbsMax, Type.intgemm8, Type.intgemm16, check)
PyObject* py_setup(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  MH_TRY MH_ARGS(5, "setup");
  if(!PyType_Check(args[0]) || !PyType_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "setup expects two classes first");
    return nullptr;
  }
  for(int i = 0; i < 5; ++i) Py_INCREF(args[i]);   // (kept for good)
  QTensorType = reinterpret_cast<PyTypeObject*>(args[0]);
  AbsMaxType = reinterpret_cast<PyTypeObject*>(args[1]);
  type8 = args[2];
  type16 = args[3];
  raise_status = args[4];
  Py_RETURN_NONE;
  MH_END
}

#define MH_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&py_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    MH_METHOD(setup), MH_METHOD(use), MH_METHOD(workspace), MH_METHOD(release_scratch), MH_METHOD(affine_or_dot), MH_METHOD(affine_f32),
    MH_METHOD(affine_f32_grouped), MH_METHOD(affine_f32_normed), MH_METHOD(proj_attention_normed), MH_METHOD(proj_attention_ancestors), MH_METHOD(prepare_a), MH_METHOD(prepare_b), MH_METHOD(prepare_stored), MH_METHOD(layer_norm),
    MH_METHOD(embed), MH_METHOD(select_state), MH_METHOD(attention), MH_METHOD(attention_rows), MH_METHOD(split_heads), MH_METHOD(join_heads), MH_METHOD(proj_attention), MH_METHOD(attention_ancestors), MH_METHOD(decoder_layers),
    MH_METHOD(ancestors_advance), MH_METHOD(nbest), MH_METHOD(nbest_words), MH_METHOD(nbest_beams), MH_METHOD(logsoftmax_nbest_beams),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_calls", "host path of the operators", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// This module calls functions of torch's that have no stable binary interface: it works in the torch it was built
// against and no other.  (Python's own interface only, until that is known.)
static bool built_for_this_torch() {
  Ref torch(PyImport_ImportModule("torch"));
  if(!torch) return false;
  Ref version(PyObject_GetAttrString(torch.p, "__version__"));
  if(!version) return false;
  Ref text(PyObject_Str(version.p));
  if(!text) return false;
  if(PyUnicode_CompareWithASCIIString(text.p, MARIAN_BUILT_FOR_TORCH) == 0) return true;
  PyErr_Format(PyExc_ImportError, "_host_calls.so was built for torch %s and this is torch %U; run make -C marian-dev_amd/csrc -B python",
               MARIAN_BUILT_FOR_TORCH, text.p);
  return false;
}

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__host_calls() {
  if(!built_for_this_torch()) return nullptr;
  s_data = PyUnicode_InternFromString("data");
  s_shape = PyUnicode_InternFromString("shape");
  s_type = PyUnicode_InternFromString("type");
  s_prepared = PyUnicode_InternFromString("prepared");
  no_args = PyTuple_New(0);
  if(!s_data || !s_shape || !s_type || !s_prepared || !no_args) return nullptr;
  return PyModule_Create(&module);
}
