// The host side of small calls: checks, output tensors and the library call of one Python method in one native function.
//
// A decode token of one sequence, a token of the cache object or a few thousand keys to codes are two to eight launches of a few
// microseconds each; the tensor attributes, allocations and foreign-function conversions around them took longer than the launches.  Host time
// through the Python methods, through here, and the kernels' time, us: a chat token (ring, decode step) 47, 25, 22; a token of the cache object
// (append, scores, softmax, weighted values; 8 heads of 128, 4096 tokens) 101, 53, 38; 4096 keys of 128 to codes, scores with 32 queries and back 43, 23, 31.
// Every function here takes the case that the Python method in front of it meets in a decode loop - plain dense tensors of the current
// device, contiguous where the library wants it - and returns None (ring_write: False) for everything else, before it allocates or launches
// anything: the Python method then goes on as if it had not been called.  What the library refuses comes back as None too, with the outputs and
// the workspace made for it dropped again and nothing launched, and the Python method meets the refusal itself.
// The library is bound by the addresses of its functions (bind), so the module has no link to it.

#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/GradMode.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <optional>
#include <vector>

#include "../../include/tq_hip.h"

// The Python, the torch and the interface that this file is compiled for (_ffi.host_stamp): it reads their structures through their headers, and
// its calls take their arguments by position.
#ifndef TQ_HOST_STAMP
#error "TQ_HOST_STAMP is not defined"
#endif

namespace {

struct Library {
  decltype(&tq_quantize_keys) quantize_keys;
  decltype(&tq_dequant_keys) dequant_keys;
  decltype(&tq_score) score;
  decltype(&tq_ring_write) ring_write;
  decltype(&tq_append_kv_paged) append_kv_paged;
  decltype(&tq_append_kv_newest) append_kv_newest;
  decltype(&tq_decode_workspace_bytes) decode_workspace_bytes;
  decltype(&tq_decode_attn_paged) decode_attn_paged;
  decltype(&tq_decode_attn_paged_by_length) decode_attn_paged_by_length;
  decltype(&tq_decode_attn_paged_ring) decode_attn_paged_ring;
  decltype(&tq_decode_attn_paged_ring_by_length) decode_attn_paged_ring_by_length;
  decltype(&tq_cache_append_bytes) cache_append_bytes;
  decltype(&tq_cache_append) cache_append;
  decltype(&tq_cache_scores_rows) cache_scores_rows;
  decltype(&tq_cache_attend_bytes) cache_attend_bytes;
  decltype(&tq_cache_attend) cache_attend;
} g_lib{};
constexpr const char* kNames[] = {"tq_quantize_keys", "tq_dequant_keys", "tq_score", "tq_ring_write", "tq_append_kv_paged",
                                  "tq_append_kv_newest", "tq_decode_workspace_bytes", "tq_decode_attn_paged", "tq_decode_attn_paged_by_length",
                                  "tq_decode_attn_paged_ring", "tq_decode_attn_paged_ring_by_length", "tq_cache_append_bytes",
                                  "tq_cache_append", "tq_cache_scores_rows", "tq_cache_attend_bytes", "tq_cache_attend"};
static_assert(sizeof(Library) == sizeof(kNames) / sizeof(kNames[0]) * sizeof(void*), "a pointer per name, in order");
bool g_bound = false;

// Whether torch would run an operation as it stands: no dispatch or function mode, transform, trace or autocast (all of which include or
// exclude dispatch keys of this thread) that has to see it.
bool nothing_watches() {
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  c10::DispatchKeySet inc = c10::default_included_set, exc = c10::default_excluded_set;
  if (c10::InferenceMode::is_enabled()) {
    inc = inc.remove(c10::DispatchKey::ADInplaceOrView);
    exc = exc | c10::autograd_dispatch_keyset;
  }
  return tls.included_ == inc && tls.excluded_ == exc && c10::impl::TorchDispatchModeTLS::stack_len() == 0 &&
         at::impl::PythonTorchFunctionTLS::stack_len() == 0 && !at::globalContext().deterministicAlgorithms();      // (which fills new tensors)
}

// The arguments' tensors: plain ones (torch.Tensor itself; dense, its memory holding its values: no lazy conjugation or negation,
// zero tensor, wrapper), of one device, the current one, with nothing to differentiate.
struct Plain {
  c10::DeviceIndex device = -1;
  bool ok = nothing_watches() && g_bound;

  static const std::array<c10::DispatchKeySet, 2>& dense() {      // key sets of an ordinary and of an inference tensor
    static const std::array<c10::DispatchKeySet, 2> sets = [] {
      auto opt = at::TensorOptions().device(at::kCUDA, c10::hip::current_device());
      c10::InferenceMode off(false);
      const auto normal = at::empty({0}, opt).key_set();
      c10::InferenceMode on(true);
      return std::array<c10::DispatchKeySet, 2>{normal, at::empty({0}, opt).key_set()};
    }();
    return sets;
  }
  at::Tensor take(PyObject* o) {
    if (!ok || !THPVariable_CheckExact(o)) { ok = false; return {}; }
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda()) { ok = false; return {}; }
    const auto ks = t.key_set();
    if (!(ks == dense()[0]) && !(ks == dense()[1])) { ok = false; return {}; }
    if (t.unsafeGetTensorImpl()->autograd_meta() != nullptr &&
        ((c10::GradMode::is_enabled() && t.requires_grad()) || t._fw_grad(0).defined())) { ok = false; return {}; }
    const auto at = t.get_device();
    if (device < 0) ok = (device = at) == c10::hip::current_device();
    else ok = device == at;
    return t;
  }
  void* stream() const { return (void*)c10::hip::getCurrentHIPStream(device).stream(); }
  // (nothing watches: the dispatcher, half of an allocation's time, has nothing to do)
  at::Tensor fresh(at::IntArrayRef size, at::ScalarType dt) const {
    return at::Tensor(at::detail::empty_cuda(size, dt, c10::Device(at::kCUDA, device), std::nullopt));
  }
};

int dtype_tag(at::ScalarType t) {
  return t == at::kFloat ? TQ_F32 : t == at::kHalf ? TQ_F16 : t == at::kBFloat16 ? TQ_BF16 : -1;
}
int code_bits(int mse_bits) { return mse_bits == 1 ? 1 : mse_bits == 2 ? 2 : mse_bits <= 4 ? 4 : 8; }
int64_t int_arg(PyObject* o) { return PyLong_AsLongLong(o); }
// The memory of a descriptor (a ctypes structure), and a reference to it: the library reads it while the interpreter's lock is given up, and
// another thread may make its owner build a new one meanwhile.
template <class T> class Held {
  Py_buffer view_{};

 public:
  explicit Held(PyObject* o) {
    if (PyObject_GetBuffer(o, &view_, PyBUF_SIMPLE) == 0 && view_.len != (Py_ssize_t)sizeof(T)) PyErr_SetString(PyExc_TypeError, "not that descriptor");
  }
  ~Held() { PyBuffer_Release(&view_); }
  Held(const Held&) = delete;
  Held& operator=(const Held&) = delete;
  const T* get() const { return (const T*)view_.buf; }
};
bool dense_as(const at::Tensor& t, at::ScalarType dt) { return t.scalar_type() == dt && t.is_contiguous(); }
std::vector<int64_t> shape(at::IntArrayRef lead, std::initializer_list<int64_t> tail = {}) {
  std::vector<int64_t> s(lead.begin(), lead.end());
  s.insert(s.end(), tail);
  return s;
}
PyObject* tuple(std::initializer_list<at::Tensor> ts) {
  PyObject* r = PyTuple_New((Py_ssize_t)ts.size());
  if (!r) return nullptr;
  Py_ssize_t i = 0;
  for (const auto& t : ts) PyTuple_SET_ITEM(r, i++, THPVariable_Wrap(t));
  return r;
}

// The library call runs without the interpreter's lock (a launch may wait for room in its queue)
template <class F, class... A>
int unlocked(F f, A... args) {
  PyThreadState* s = PyEval_SaveThread();
  const int rc = f(args...);
  PyEval_RestoreThread(s);
  return rc;
}

// None, and nothing raised, for whatever goes wrong before the launch (an argument that is no number, no memory): the Python method
// that goes on raises it as it always did
template <int N, class F>
PyObject* entry(PyObject* const* a, Py_ssize_t n, F&& f) {
  if (n != N) { PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n); return nullptr; }
  PyObject* r = nullptr;
  try {
    r = f(a);
  } catch (const std::exception&) {
  }
  if (PyErr_Occurred()) { PyErr_Clear(); Py_XDECREF(r); r = nullptr; }
  if (r) return r;
  Py_RETURN_NONE;
}

// ---- keys <-> codes ---------------------------------------------------------------------------------------------------------

// quantize(x, layer, d, mse_bits) -> (indices, signs, residual norms, norms)
PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return entry<4>(args, n_args, [](PyObject* const* a) -> PyObject* {
    Plain p;
    const at::Tensor x = p.take(a[0]);
    const int64_t d = int_arg(a[2]);
    const int mb = (int)int_arg(a[3]);
    const Held<tq_layer> layer(a[1]);
    if (!p.ok || PyErr_Occurred() || d <= 0 || x.dim() < 1 || x.size(-1) != d || x.numel() == 0 || !x.is_contiguous()) return nullptr;
    const int tag = dtype_tag(x.scalar_type()), per = 8 / code_bits(mb);
    if (tag < 0) return nullptr;
    const auto lead = x.sizes().slice(0, x.dim() - 1);
    constexpr auto bytes = at::kByte;
    at::Tensor idx = p.fresh(shape(lead, {(d + per - 1) / per}), bytes), sgn = p.fresh(shape(lead, {(d + 7) / 8}), bytes);
    at::Tensor nrm = p.fresh(lead, x.scalar_type()), rn = p.fresh(lead, at::kFloat);
    if (unlocked(g_lib.quantize_keys, x.data_ptr(), tag, x.numel() / d, d, layer.get(), (uint8_t*)idx.data_ptr(), (uint8_t*)sgn.data_ptr(),
                            nrm.data_ptr(), (float*)rn.data_ptr(), nullptr, nullptr, 0, p.stream()) != TQ_OK)
      return nullptr;
    return tuple({idx, sgn, rn, nrm});
  });
}

// codes of vectors: sections that belong together, norms of shape `lead`
struct Codes {
  at::Tensor idx, sgn, rn, nrm;
  int64_t n = 0;
  bool take(Plain& p, PyObject* const* a, int64_t d, int mb) {     // indices, signs, residual norms, norms
    idx = p.take(a[0]); sgn = p.take(a[1]); rn = p.take(a[2]); nrm = p.take(a[3]);
    if (!p.ok) return false;
    const int per = 8 / code_bits(mb);
    n = nrm.numel();
    auto rows = [&](const at::Tensor& t, int64_t w) {
      return t.dim() == nrm.dim() + 1 && t.size(-1) == w && t.sizes().slice(0, nrm.dim()) == nrm.sizes() && dense_as(t, at::kByte);
    };
    return n > 0 && nrm.dim() > 0 && dtype_tag(nrm.scalar_type()) >= 0 && nrm.is_contiguous() && dense_as(rn, at::kFloat) &&
           rn.sizes() == nrm.sizes() && rows(idx, (d + per - 1) / per) && rows(sgn, (d + 7) / 8);
  }
};

// dequantize(indices, signs, residual norms, norms, layer, d, mse_bits) -> vectors
PyObject* dequantize(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return entry<7>(args, n_args, [](PyObject* const* a) -> PyObject* {
    Plain p;
    Codes c;
    const int64_t d = int_arg(a[5]);
    const int mb = (int)int_arg(a[6]);
    const Held<tq_layer> layer(a[4]);
    if (PyErr_Occurred() || !c.take(p, a, d, mb)) return nullptr;
    at::Tensor out = p.fresh(shape(c.nrm.sizes(), {d}), at::kFloat);
    if (unlocked(g_lib.dequant_keys, (const uint8_t*)c.idx.data_ptr(), (const uint8_t*)c.sgn.data_ptr(), c.nrm.data_ptr(), dtype_tag(c.nrm.scalar_type()),
                           (const float*)c.rn.data_ptr(), c.n, layer.get(), (float*)out.data_ptr(), p.stream()) != TQ_OK)
      return nullptr;
    return THPVariable_Wrap(out);
  });
}

// score(query, indices, signs, residual norms, norms, layer, d, mse_bits) -> (..., queries, keys)
PyObject* score(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return entry<8>(args, n_args, [](PyObject* const* a) -> PyObject* {
    Plain p;
    const at::Tensor q = p.take(a[0]);
    Codes c;
    const int64_t d = int_arg(a[6]);
    const int mb = (int)int_arg(a[7]);
    const Held<tq_layer> layer(a[5]);
    if (PyErr_Occurred() || !c.take(p, a + 1, d, mb)) return nullptr;
    const int tag = dtype_tag(q.scalar_type());
    if (tag < 0 || !q.is_contiguous() || q.dim() != c.nrm.dim() + 1 || q.size(-1) != d || q.numel() == 0) return nullptr;
    const auto lead = c.nrm.sizes().slice(0, c.nrm.dim() - 1);
    if (q.sizes().slice(0, q.dim() - 2) != lead) return nullptr;
    const int64_t n_q = q.size(-2), n_k = c.nrm.size(-1), batch = c.n / n_k;
    at::Tensor out = p.fresh(shape(lead, {n_q, n_k}), at::kFloat), work = p.fresh({2 * batch * n_q * d}, at::kFloat);
    if (unlocked(g_lib.score, q.data_ptr(), tag, batch, n_q, (const uint8_t*)c.idx.data_ptr(), (const uint8_t*)c.sgn.data_ptr(), c.nrm.data_ptr(),
                    dtype_tag(c.nrm.scalar_type()), (const float*)c.rn.data_ptr(), n_k, layer.get(), (float*)out.data_ptr(),
                    (float*)work.data_ptr(), p.stream()) != TQ_OK)
      return nullptr;
    return THPVariable_Wrap(out);
  });
}

// ---- ring and pages ---------------------------------------------------------------------------------------------------------

// ring_write(rows (2, capacity, H, d), key, value, src, n, held) -> bool: rows src .. src + n - 1 behind the `held` ones
PyObject* ring_write(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  PyObject* r = entry<6>(args, n_args, [](PyObject* const* a) -> PyObject* {
    Plain p;
    const at::Tensor rows = p.take(a[0]), key = p.take(a[1]), value = p.take(a[2]);
    const int64_t src = int_arg(a[3]), n = int_arg(a[4]), held = int_arg(a[5]);
    if (!p.ok || PyErr_Occurred() || rows.dim() != 4 || key.dim() != 3 || key.sizes() != value.sizes()) return nullptr;
    const int64_t H = rows.size(2), d = rows.size(3);
    if (src < 0 || n <= 0 || held < 0 || held + n > rows.size(1) || key.size(0) < src + n || key.size(1) != H || key.size(2) != d) return nullptr;
    if (key.scalar_type() != rows.scalar_type() || value.scalar_type() != rows.scalar_type() || !rows.is_contiguous()) return nullptr;
    for (const at::Tensor* t : {&key, &value})
      if (t->stride(2) != 1 || (H > 1 && t->stride(1) != d)) return nullptr;
    const bool inference = rows.is_inference();
    if (inference && !c10::InferenceMode::is_enabled()) return nullptr;       // (torch refuses the copy)
    const int64_t size = rows.element_size(), row = H * d * size;
    const uintptr_t base = (uintptr_t)rows.data_ptr(), end = base + rows.nbytes();
    const uintptr_t kp = (uintptr_t)key.data_ptr() + src * key.stride(0) * size, vp = (uintptr_t)value.data_ptr() + src * value.stride(0) * size;
    const int64_t kr = n > 1 ? key.stride(0) * size : row, vr = n > 1 ? value.stride(0) * size : row;
    if ((kp | vp | (uintptr_t)kr | (uintptr_t)vr | (uintptr_t)row | base) & 15) return nullptr;
    if ((kp < end && kp + (n - 1) * kr + row > base) || (vp < end && vp + (n - 1) * vr + row > base)) return nullptr;      // the ring's own rows
    const uintptr_t dst = base + held * row;
    if (unlocked(g_lib.ring_write, (const void*)kp, (const void*)vp, kr, vr, (void*)dst, (void*)(dst + rows.size(1) * row), row, n, p.stream()) != TQ_OK)
      return nullptr;
    if (!inference) rows.unsafeGetTensorImpl()->bump_version();
    Py_RETURN_TRUE;
  });
  if (r == Py_None) { Py_DECREF(r); Py_RETURN_FALSE; }
  return r;
}

// append(key, value (B, T, H, d), block table, start positions or None, pool, pages, H, d, dtype tag, layer, layout, newest) -> True; newest: the
// positions are the lengths with the new tokens
PyObject* append(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return entry<12>(args, n_args, [](PyObject* const* a) -> PyObject* {
    Plain p;
    const at::Tensor key = p.take(a[0]), value = p.take(a[1]), table = p.take(a[2]), pool = p.take(a[4]);
    const bool from_zero = a[3] == Py_None, newest = a[11] == Py_True;
    at::Tensor start;
    if (!from_zero) start = p.take(a[3]);
    const int64_t pages = int_arg(a[5]), H = int_arg(a[6]), d = int_arg(a[7]), tag = int_arg(a[8]);
    const Held<tq_layer> layer(a[9]);
    const Held<tq_page_layout> layout(a[10]);
    if (!p.ok || PyErr_Occurred() || key.dim() != 4 || key.sizes() != value.sizes() || key.strides() != value.strides()) return nullptr;
    if (key.size(2) != H || key.size(3) != d || key.stride(3) != 1 || key.numel() == 0) return nullptr;
    if (dtype_tag(key.scalar_type()) != tag || value.scalar_type() != key.scalar_type()) return nullptr;
    const int64_t B = key.size(0), T = key.size(1);
    if (B > INT_MAX || T > INT_MAX || table.dim() != 2 || table.size(0) != B || table.size(1) > INT_MAX || !dense_as(table, at::kInt)) return nullptr;
    if (!from_zero && (start.dim() != 1 || start.size(0) != B || !dense_as(start, at::kInt))) return nullptr;
    if (unlocked(newest ? g_lib.append_kv_newest : g_lib.append_kv_paged, key.data_ptr(), value.data_ptr(), (int)tag, (int)B, (int)T, (int)H, key.stride(0), key.stride(1), key.stride(2),
                              from_zero ? nullptr : (const int32_t*)start.data_ptr(), (const int32_t*)table.data_ptr(), (int)table.size(1),
                              layer.get(), layout.get(), (uint8_t*)pool.data_ptr(), pages, p.stream()) != TQ_OK)
      return nullptr;
    Py_RETURN_TRUE;
  });
}

// A decode step's common arguments: query (B, Hq, d), block table (B, n) or (n,), lengths (int32, from element `at` on)
struct Step {
  at::Tensor q, table, lens, pool;
  int64_t B = 0, Hq = 0, bt_stride = 0;
  int tag = -1;
  const int32_t* len_ptr = nullptr;
  bool take(Plain& p, PyObject* query, PyObject* bt, PyObject* seq, int64_t at, PyObject* data, int64_t H, int64_t d) {
    q = p.take(query); table = p.take(bt); lens = p.take(seq); pool = p.take(data);
    if (!p.ok || q.dim() != 3 || q.size(2) != d || H <= 0 || q.size(1) % H || q.numel() == 0 || !q.is_contiguous()) return false;
    B = q.size(0); Hq = q.size(1);
    tag = dtype_tag(q.scalar_type());
    if (tag < 0 || B > INT_MAX || Hq > INT_MAX || !dense_as(table, at::kInt) || !dense_as(lens, at::kInt)) return false;
    if (table.dim() == 2 ? table.size(0) != B : table.dim() != 1) return false;
    bt_stride = table.dim() == 1 ? -table.size(0) : table.size(1);      // negative: one shared row of that length
    if (bt_stride == 0 || bt_stride > INT_MAX || bt_stride < -INT_MAX || lens.dim() != 1 || at < 0 || at + B > lens.size(0)) return false;
    len_ptr = (const int32_t*)lens.data_ptr() + at;
    return true;
  }
  at::Tensor workspace(const Plain& p, int64_t d, int n_split) const {
    return p.fresh({(int64_t)(g_lib.decode_workspace_bytes((int)B, (int)Hq, (int)d, n_split) / 4)}, at::kFloat);
  }
};

// decode(query, block table, lengths, first length, pool, pages, H, d, scale, recent keys or None, recent values, layer, layout, splits,
// by length) -> attention.  Recent rows (B, R, H, d), or (R, H, d) of one sequence.
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return entry<15>(args, n_args, [](PyObject* const* a) -> PyObject* {
    Plain p;
    Step s;
    const int64_t at = int_arg(a[3]), pages = int_arg(a[5]), H = int_arg(a[6]), d = int_arg(a[7]);
    const double scale = PyFloat_AsDouble(a[8]);
    const int n_split = (int)int_arg(a[13]), by_length = PyObject_IsTrue(a[14]);
    const Held<tq_layer> layer(a[11]);
    const Held<tq_page_layout> layout(a[12]);
    if (PyErr_Occurred() || !s.take(p, a[0], a[1], a[2], at, a[4], H, d)) return nullptr;
    const void *rk = nullptr, *rv = nullptr;
    int64_t R = 0, rs[3] = {0, 0, 0};
    at::Tensor k, v;
    if (a[9] != Py_None) {
      k = p.take(a[9]); v = p.take(a[10]);
      if (!p.ok || (k.dim() != 4 && !(k.dim() == 3 && s.B == 1)) || k.sizes() != v.sizes() || k.strides() != v.strides()) return nullptr;
      const int64_t i = k.dim() - 3;                              // dimension of the rows
      if (k.scalar_type() != s.q.scalar_type() || v.scalar_type() != k.scalar_type() || k.stride(i + 2) != 1) return nullptr;
      if (k.size(i + 1) != H || k.size(i + 2) != d || (i == 1 && k.size(0) != s.B) || k.size(i) > INT_MAX) return nullptr;
      if ((R = k.size(i)) > 0) {
        rk = k.data_ptr(); rv = v.data_ptr();
        rs[0] = i == 1 ? k.stride(0) : R * k.stride(0);
        rs[1] = k.stride(i); rs[2] = k.stride(i + 1);
      }
    }
    const at::Tensor ws = s.workspace(p, d, by_length ? -n_split : n_split), out = p.fresh(s.q.sizes(), s.q.scalar_type());
    const auto call = by_length ? g_lib.decode_attn_paged_by_length : g_lib.decode_attn_paged;
    if (unlocked(call, s.q.data_ptr(), s.tag, (int)s.B, (int)s.Hq, (int)H, (const uint8_t*)s.pool.data_ptr(), pages, (const int32_t*)s.table.data_ptr(),
             (int)s.bt_stride, s.len_ptr, (float)scale, layer.get(), layout.get(), rk, rv, (int)R, rs[0], rs[1],
             rs[2], nullptr, out.data_ptr(), (float*)ws.data_ptr(), n_split, p.stream()) != TQ_OK)
      return nullptr;
    return THPVariable_Wrap(out);
  });
}

// decode_ring(query, block table, lengths, pool, pages, H, d, scale, key cache, value cache (blocks, 16, H, d), ring rows, layer, layout,
// splits, by length) -> attention
PyObject* decode_ring(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return entry<15>(args, n_args, [](PyObject* const* a) -> PyObject* {
    Plain p;
    Step s;
    const int64_t pages = int_arg(a[4]), H = int_arg(a[5]), d = int_arg(a[6]), ring = int_arg(a[10]);
    const double scale = PyFloat_AsDouble(a[7]);
    const int n_split = (int)int_arg(a[13]), by_length = PyObject_IsTrue(a[14]);
    const Held<tq_layer> layer(a[11]);
    const Held<tq_page_layout> layout(a[12]);
    if (PyErr_Occurred() || ring > INT_MAX || ring < INT_MIN || !s.take(p, a[0], a[1], a[2], 0, a[3], H, d)) return nullptr;
    const at::Tensor k = p.take(a[8]), v = p.take(a[9]);
    if (!p.ok || k.dim() != 4 || k.sizes() != v.sizes() || k.strides() != v.strides() || k.size(1) != TQ_PAGE_TOKENS || k.size(2) != H ||
        k.size(3) != d || k.stride(3) != 1 || k.scalar_type() != s.q.scalar_type() || v.scalar_type() != k.scalar_type())
      return nullptr;
    if (k.element_size() == 2 && ((k.stride(0) | k.stride(1) | k.stride(2)) % 2 || (((uintptr_t)k.data_ptr() | (uintptr_t)v.data_ptr()) & 3)))
      return nullptr;
    const at::Tensor ws = s.workspace(p, d, by_length ? -n_split : n_split), out = p.fresh(s.q.sizes(), s.q.scalar_type());
    const auto call = by_length ? g_lib.decode_attn_paged_ring_by_length : g_lib.decode_attn_paged_ring;
    if (unlocked(call, s.q.data_ptr(), s.tag, (int)s.B, (int)s.Hq, (int)H, (const uint8_t*)s.pool.data_ptr(), pages, (const int32_t*)s.table.data_ptr(),
             (int)s.bt_stride, s.len_ptr, (float)scale, layer.get(), layout.get(), k.data_ptr(), v.data_ptr(),
             k.stride(0), k.stride(1), k.stride(2), (int)ring, out.data_ptr(), (float*)ws.data_ptr(), n_split, p.stream()) != TQ_OK)
      return nullptr;
    return THPVariable_Wrap(out);
  });
}

// ---- the cache object: a decode token in fp32 -----------------------------------------------------------------------------------

// Its compressed part as it writes it itself: seven contiguous sections over norms (B, H, n)
struct Part {
  at::Tensor idx, sgn, rn, nrm, data, scales, zeros;
  int64_t B = 0, H = 0, n = 0;
  bool take(Plain& p, PyObject* const* a, int64_t d, int mb, int bits, int64_t gs) {     // indices, signs, residual norms, norms, data, scales, zeros
    idx = p.take(a[0]); sgn = p.take(a[1]); rn = p.take(a[2]); nrm = p.take(a[3]);
    data = p.take(a[4]); scales = p.take(a[5]); zeros = p.take(a[6]);
    if (!p.ok || d <= 0 || gs <= 0 || nrm.dim() != 3) return false;
    B = nrm.size(0); H = nrm.size(1); n = nrm.size(2);
    auto is = [&](const at::Tensor& t, at::ScalarType dt, int64_t w) { return dense_as(t, dt) && t.numel() == nrm.numel() * w; };
    auto rows = [&](const at::Tensor& t) { return t.dim() == 4 && t.size(0) == B && t.size(1) == H && t.size(2) == n; };
    return n > 0 && is(nrm, at::kFloat, 1) && is(rn, at::kFloat, 1) && is(idx, at::kByte, d * code_bits(mb) / 8) && is(sgn, at::kByte, d / 8) &&
           is(data, at::kByte, d * bits / 8) && is(scales, at::kFloat, d / gs) && is(zeros, at::kFloat, d / gs) && rows(idx) && rows(sgn) &&
           rows(data) && rows(scales) && rows(zeros) && rn.sizes() == nrm.sizes();
  }
};
bool rows4(const at::Tensor& t) { return t.scalar_type() == at::kFloat && t.dim() == 4 && t.stride(3) == 1; }

// cache_append(seven sections, key, value (B, H, 1, d), key buffer, value buffer (B, H, n, d), layer, d, mse bits, value bits, group size)
// -> the nine tensors after it
PyObject* cache_append(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return entry<16>(args, n_args, [](PyObject* const* a) -> PyObject* {
    Plain p;
    Part c;
    const int64_t d = int_arg(a[12]), gs = int_arg(a[15]);
    const int mb = (int)int_arg(a[13]), bits = (int)int_arg(a[14]);
    const Held<tq_layer> layer(a[11]);
    if (PyErr_Occurred() || !c.take(p, a, d, mb, bits, gs)) return nullptr;
    const at::Tensor key = p.take(a[7]), value = p.take(a[8]), kb = p.take(a[9]), vb = p.take(a[10]);
    if (!p.ok || !rows4(key) || !rows4(value) || !rows4(kb) || !rows4(vb)) return nullptr;
    const int64_t B = c.B, H = c.H, n_buf = kb.size(2);
    if (kb.size(0) != B || kb.size(1) != H || kb.size(3) != d || n_buf < 1 || n_buf > INT_MAX || vb.sizes() != kb.sizes() || B * H > 65535 || c.n >= 1 << 20)
      return nullptr;
    for (const at::Tensor* t : {&key, &value})
      if (t->size(0) != B || t->size(1) != H || t->size(2) != 1 || t->size(3) != d || t->stride(1) < d || (B > 1 && t->stride(0) != H * t->stride(1)))
        return nullptr;
    for (const at::Tensor* t : {&kb, &vb})
      if (t->stride(2) != d || t->stride(1) < d || (B > 1 && t->stride(0) != H * t->stride(1))) return nullptr;
    auto grown = [&](const at::Tensor& t) {
      auto s = t.sizes().vec();
      s[2] = c.n + 1;
      return p.fresh(s, t.scalar_type());
    };
    const at::Tensor idx = grown(c.idx), sgn = grown(c.sgn), rn = grown(c.rn), nrm = grown(c.nrm), data = grown(c.data), scales = grown(c.scales),
                     zeros = grown(c.zeros), nk = p.fresh(kb.sizes(), at::kFloat), nv = p.fresh(kb.sizes(), at::kFloat);
    const at::Tensor work = p.fresh({(int64_t)g_lib.cache_append_bytes(B * H, (int)d, mb, bits, (int)gs)}, at::kByte);
    if (unlocked(g_lib.cache_append, (const float*)key.data_ptr(), (const float*)value.data_ptr(), key.stride(1), value.stride(1), (const float*)kb.data_ptr(),
                           (const float*)vb.data_ptr(), kb.stride(0), kb.stride(1), kb.stride(2), vb.stride(0), vb.stride(1), vb.stride(2), B * H, (int)H,
                           (int)n_buf, layer.get(), bits, (int)gs, c.n, (const uint8_t*)c.idx.data_ptr(), (const uint8_t*)c.sgn.data_ptr(),
                           (const float*)c.nrm.data_ptr(), (const float*)c.rn.data_ptr(), (const uint8_t*)c.data.data_ptr(),
                           (const float*)c.scales.data_ptr(), (const float*)c.zeros.data_ptr(), (uint8_t*)idx.data_ptr(), (uint8_t*)sgn.data_ptr(),
                           (float*)nrm.data_ptr(), (float*)rn.data_ptr(), (uint8_t*)data.data_ptr(), (float*)scales.data_ptr(), (float*)zeros.data_ptr(),
                           (float*)nk.data_ptr(), (float*)nv.data_ptr(), work.data_ptr(), p.stream()) != TQ_OK)
      return nullptr;
    return tuple({idx, sgn, rn, nrm, data, scales, zeros, nk, nv});
  });
}

// cache_scores(seven sections, query (B, H, n, d), key buffer, layer, d, mse bits, value bits, group size, scale) -> (B, H, n, tokens)
PyObject* cache_scores(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return entry<15>(args, n_args, [](PyObject* const* a) -> PyObject* {
    Plain p;
    Part c;
    const int64_t d = int_arg(a[10]), gs = int_arg(a[13]);
    const int mb = (int)int_arg(a[11]), bits = (int)int_arg(a[12]);
    const double scale = PyFloat_AsDouble(a[14]);
    const Held<tq_layer> layer(a[9]);
    if (PyErr_Occurred() || !c.take(p, a, d, mb, bits, gs)) return nullptr;
    const at::Tensor query = p.take(a[7]), kb = p.take(a[8]);
    if (!p.ok || !rows4(query) || !rows4(kb) || kb.size(0) != c.B || kb.size(1) != c.H || kb.size(3) != d || kb.size(2) < 1 || kb.size(2) > INT_MAX) return nullptr;
    const int64_t n_q = query.size(2), n_buf = kb.size(2), batch = c.B * c.H;
    if (query.size(0) != c.B || query.size(1) != c.H || query.size(3) != d || n_q < 1 || batch > 65535) return nullptr;
    // rows that lie evenly apart are read where they are (a token's slice of all queries)
    const bool even = (n_q == 1 || query.stride(1) == n_q * query.stride(2)) && (c.B == 1 || query.stride(0) == c.H * query.stride(1));
    const int64_t apart = n_q == 1 ? query.stride(1) : query.stride(2);
    const bool in_place = even && apart >= d;
    const at::Tensor q = in_place ? query : query.contiguous(), out = p.fresh({c.B, c.H, n_q, c.n + n_buf}, at::kFloat);
    const at::Tensor work = p.fresh({2 * batch * n_q * d}, at::kFloat);
    if (unlocked(g_lib.cache_scores_rows, (const float*)q.data_ptr(), in_place ? apart : d, batch, (int)c.H, n_q, (const uint8_t*)c.idx.data_ptr(), (const uint8_t*)c.sgn.data_ptr(),
                           (const float*)c.nrm.data_ptr(), (const float*)c.rn.data_ptr(), c.n, layer.get(), (const float*)kb.data_ptr(),
                           kb.stride(0), kb.stride(1), kb.stride(2), (int)n_buf, (float)scale, (float*)out.data_ptr(), (float*)work.data_ptr(),
                           p.stream()) != TQ_OK)
      return nullptr;
    return THPVariable_Wrap(out);
  });
}

// cache_attend(seven sections, weights (B, H, n, tokens), value buffer, d, mse bits, value bits, group size) -> (B, H, n, d)
PyObject* cache_attend(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return entry<13>(args, n_args, [](PyObject* const* a) -> PyObject* {
    Plain p;
    Part c;
    const int64_t d = int_arg(a[9]), gs = int_arg(a[12]);
    const int mb = (int)int_arg(a[10]), bits = (int)int_arg(a[11]);
    if (PyErr_Occurred() || !c.take(p, a, d, mb, bits, gs)) return nullptr;
    const at::Tensor weights = p.take(a[7]), vb = p.take(a[8]);
    if (!p.ok || !rows4(weights) || !rows4(vb) || vb.size(0) != c.B || vb.size(1) != c.H || vb.size(3) != d || vb.size(2) < 1 || vb.size(2) > INT_MAX) return nullptr;
    const int64_t n_q = weights.size(2), n_buf = vb.size(2), batch = c.B * c.H;
    if (weights.size(0) != c.B || weights.size(1) != c.H || weights.size(3) != c.n + n_buf || n_q < 1 || n_q > 65535 || batch > 65535) return nullptr;
    const at::Tensor w = weights.contiguous(), out = p.fresh({c.B, c.H, n_q, d}, at::kFloat);
    const at::Tensor work = p.fresh({(int64_t)(g_lib.cache_attend_bytes(batch, n_q, (int)d, c.n, (int)n_buf) / 4)}, at::kFloat);
    if (unlocked(g_lib.cache_attend, (const float*)w.data_ptr(), batch, (int)c.H, n_q, (const uint8_t*)c.data.data_ptr(), (const float*)c.scales.data_ptr(),
                           (const float*)c.zeros.data_ptr(), c.n, (int)d, (int)gs, bits, (const float*)vb.data_ptr(), vb.stride(0), vb.stride(1),
                           vb.stride(2), (int)n_buf, (float*)out.data_ptr(), (float*)work.data_ptr(), p.stream()) != TQ_OK)
      return nullptr;
    return THPVariable_Wrap(out);
  });
}

// bind({name: address}): the library's functions
PyObject* bind(PyObject*, PyObject* arg) {
  if (!PyDict_Check(arg)) { PyErr_SetString(PyExc_TypeError, "bind takes a dict of addresses"); return nullptr; }
  void** to = (void**)&g_lib;
  for (size_t i = 0; i < sizeof(kNames) / sizeof(kNames[0]); ++i) {
    PyObject* o = PyDict_GetItemString(arg, kNames[i]);
    if (!o) { PyErr_SetString(PyExc_KeyError, kNames[i]); return nullptr; }
    to[i] = PyLong_AsVoidPtr(o);
    if (PyErr_Occurred()) return nullptr;
  }
  g_bound = true;
  Py_RETURN_NONE;
}

#define TQ_FAST(f, doc) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, doc}
PyMethodDef kMethods[] = {
    {"bind", bind, METH_O, "addresses of the library's functions, by name"},
    TQ_FAST(quantize, "keys to codes"), TQ_FAST(dequantize, "codes to keys"), TQ_FAST(score, "inner products with codes"),
    TQ_FAST(ring_write, "rows into the ring"), TQ_FAST(append, "tokens into pages"), TQ_FAST(decode, "a decode step"),
    TQ_FAST(decode_ring, "a decode step, exact tokens in place"), TQ_FAST(cache_append, "a token into the cache object"),
    TQ_FAST(cache_scores, "scores of the cache object"), TQ_FAST(cache_attend, "weighted values of the cache object"),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_tq_host", "host side of small calls", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tq_host(void) {
  PyObject* m = PyModule_Create(&kModule);
  if (m && PyModule_AddStringConstant(m, "built_for", TQ_HOST_STAMP) < 0) { Py_DECREF(m); m = nullptr; }
  return m;
}
