// The host side of the calls that a sub-block step makes, in native code: checks, output
// allocation, descriptor, workspace lookup and launch of one call of libfdllm_hip.so.
//
// Each function takes the tensors of its ops.py namesake and returns its result, or None
// where the call is not in the plain form (a tensor to convert or copy, a wrong shape or
// type, a CPU, traced or wrapped tensor): the Python function then converts, refuses or
// computes as it did. So nothing is refused or accepted here that is not there; this is the
// path of the calls that need no change. The Python statement of such a call took 15-25 us of
// host time (40 descriptor fields through ctypes), more than its kernels; this one takes 3-5.
//
// The C ABI's entry points arrive as addresses (init), so the library in use is the one that
// _ffi loaded. The per-stream workspaces stay ops._Workspace's: its dictionary is read here,
// its `get` called where a buffer is missing or too small.
#include <Python.h>

#include <cmath>
#include <cstring>
#include <initializer_list>

#include <ATen/ATen.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/fdllm_hip.h"

namespace {

using at::Tensor;

struct Api {
  decltype(&fdllm_last_error) last_error;
  decltype(&fdllm_kv_attn_workspace_size) attn_size;
  decltype(&fdllm_kv_attn_fwd) attn;
  decltype(&fdllm_gather_rmsnorm) gather;
  decltype(&fdllm_scatter_rows) scatter;
  decltype(&fdllm_add_rmsnorm) add_norm;
  decltype(&fdllm_qkv_rope_workspace_size) qkv_size;
  decltype(&fdllm_qkv_rope_kv_write_ws) qkv;
  decltype(&fdllm_linear_workspace_size) linear_size;
  decltype(&fdllm_linear) linear;
  decltype(&fdllm_unmask_workspace_size) unmask_size;
  decltype(&fdllm_unmask_step_ws) unmask;
} api;
constexpr int kApis = 12;

PyObject* g_stream = nullptr;   // torch's raw stream lookup: device index -> handle
PyObject* g_buffers = nullptr;  // ops._Workspace's dictionary: (device index, stream) -> tensor
PyObject* g_get = nullptr;      // ops._Workspace.get

// Raised inside a call for "not the plain form".
struct NotPlain {};
struct PyFailed {};  // a Python error is set

void plain(bool ok) {
  if (!ok) throw NotPlain{};
}

// A strided GPU tensor that is what it says: no subclass, no wrapper of a transform.
const Tensor& tensor(PyObject* o) {
  plain(THPVariable_CheckExact(o) || (THPVariable_Check(o) && Py_TYPE(o) == reinterpret_cast<PyTypeObject*>(ParameterClass)));
  const Tensor& t = THPVariable_Unpack(o);
  static const c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                        c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                        c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                        c10::DispatchKey::ZeroTensor});
  plain(t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() &&
        !t.unsafeGetTensorImpl()->key_set().has_any(odd) && !t.unsafeGetTensorImpl()->has_symbolic_sizes_strides());
  return t;
}

struct Opt {  // a tensor or None
  const Tensor* t = nullptr;
  explicit Opt(PyObject* o) {
    if (o != Py_None) t = &tensor(o);
  }
  explicit operator bool() const { return t != nullptr; }
  const Tensor* operator->() const { return t; }
  const Tensor& operator*() const { return *t; }
  void* ptr() const { return t ? t->data_ptr() : nullptr; }
};

int dtype_code(at::ScalarType s) {
  if (s == at::kBFloat16) return FDLLM_DTYPE_BF16;
  if (s == at::kHalf) return FDLLM_DTYPE_F16;
  plain(s == at::kFloat);
  return FDLLM_DTYPE_F32;
}

bool half_type(at::ScalarType s) { return s == at::kBFloat16 || s == at::kHalf; }

bool same(const Tensor& a, const Tensor& b) { return a.device() == b.device() && a.scalar_type() == b.scalar_type(); }

long integer(PyObject* o) {
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw NotPlain{};
  }
  return v;
}

double number(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    throw NotPlain{};
  }
  return v;
}

struct Ref {  // owned reference
  PyObject* o;
  explicit Ref(PyObject* p) : o(p) {
    if (!p) throw PyFailed{};
  }
  ~Ref() { Py_XDECREF(o); }
  Ref(const Ref&) = delete;
};

// A call's workspace, held until its kernels are launched.
struct Workspace {
  Tensor buf;
  void* ptr = nullptr;
  size_t bytes = 0;
};

// The current stream of a device, and its workspace.
struct Stream {
  Ref index, handle;
  void* ptr;
  explicit Stream(const Tensor& t)
      : index(PyLong_FromLong(t.device().index())), handle(PyObject_CallOneArg(g_stream, index.o)),
        ptr(PyLong_AsVoidPtr(handle.o)) {}
  // at least `bytes` (nothing for 0)
  Workspace workspace(size_t bytes, const Tensor& t) const {
    Workspace w;
    if (bytes == 0) return w;
    Ref key(PyTuple_Pack(2, index.o, handle.o));
    PyObject* have = PyDict_GetItemWithError(g_buffers, key.o);
    if (!have && PyErr_Occurred()) throw PyFailed{};
    if (have && static_cast<size_t>(THPVariable_Unpack(have).numel()) >= bytes) {
      w.buf = THPVariable_Unpack(have);
    } else {
      Ref dev(THPDevice_New(t.device()));
      Ref size(PyLong_FromSize_t(bytes));
      Ref made(PyObject_CallFunctionObjArgs(g_get, size.o, dev.o, nullptr));
      w.buf = THPVariable_Unpack(made.o);
    }
    w.ptr = w.buf.data_ptr();
    w.bytes = w.buf.numel();
    return w;
  }
};

// The interpreter is free for other threads while memory is allocated and while a launch
// waits for room in its queue.
struct NoGil {
  PyThreadState* s = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(s); }
};

Tensor empty(at::IntArrayRef sizes, const Tensor& like) {
  NoGil free;
  return at::empty(sizes, like.options().requires_grad(false));
}

template <typename F>
int launch(F f) {
  NoGil free;
  return f();
}

void check(int rc, const char* what) {
  if (rc == FDLLM_OK) return;
  PyErr_Format(PyExc_RuntimeError, "%s failed (code %d): %s", what, rc, api.last_error());
  throw PyFailed{};
}

PyObject* wrap(Tensor t) {
  PyObject* o = THPVariable_Wrap(std::move(t));
  if (!o) throw PyFailed{};
  return o;
}

void arity(Py_ssize_t got, Py_ssize_t want) {
  if (got != want) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, got);
    throw PyFailed{};
  }
}

using Body = PyObject* (*)(PyObject* const*, Py_ssize_t);

// No C++ exception leaves a call.
template <Body body>
PyObject* call(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  try {
    plain(!c10::impl::TorchDispatchModeTLS::any_modes_set());
    return body(a, n);
  } catch (const NotPlain&) {
    Py_RETURN_NONE;
  } catch (const PyFailed&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// q, k, v, seqlens, scale | None, mask_mode, mask_block, q_start, page_table, page_size,
// k_new, v_new, flags
PyObject* attn(PyObject* const* a, Py_ssize_t n) {
  arity(n, 13);
  const Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &len = tensor(a[3]);
  const Opt qs(a[7]), table(a[8]), kn(a[10]), vn(a[11]);
  const int64_t page = integer(a[9]);
  plain(q.dim() == 4 && k.dim() == 4 && v.dim() == 4 && same(q, k) && same(q, v) && k.sizes() == v.sizes());
  const int64_t B = q.size(0), S = q.size(1), Hq = q.size(2), D = q.size(3), Hkv = k.size(2);
  plain(k.size(3) == D && Hkv > 0 && Hq % Hkv == 0 && (table || k.size(0) == B) && q.stride(3) == 1 &&
        k.stride(3) == 1 && v.stride(3) == 1);
  auto ints = [&](const Tensor& t) { return t.device() == q.device() && t.scalar_type() == at::kInt && t.is_contiguous(); };
  plain(ints(len) && (!qs || ints(*qs)) && (!table || (ints(*table) && table->dim() == 2 && page > 0 && k.size(1) == page)));
  plain(static_cast<bool>(kn) == static_cast<bool>(vn));
  if (kn)
    plain(same(q, *kn) && same(q, *vn) && half_type(q.scalar_type()) && kn->dim() == 4 && kn->size(0) == B &&
          kn->size(1) == S && kn->size(2) == Hkv && kn->size(3) == D && vn->sizes() == kn->sizes() &&
          vn->strides() == kn->strides() && kn->stride(3) == 1);
  fdllm_kv_attn_desc d = {};
  d.dtype = dtype_code(q.scalar_type());
  d.softmax_scale = a[4] == Py_None ? static_cast<float>(std::pow(static_cast<double>(D), -0.5)) : static_cast<float>(number(a[4]));
  d.mask_mode = static_cast<int>(integer(a[5]));
  d.mask_block = static_cast<int>(integer(a[6]));
  d.flags = static_cast<int>(integer(a[12]));
  const int64_t most = table ? table->size(1) * page : k.size(1);
  plain(most <= INT32_MAX && B <= INT32_MAX && S <= INT32_MAX && Hq <= INT32_MAX && D <= INT32_MAX);
  Tensor out = empty({B, S, Hq, D}, q);
  d.q = q.data_ptr();
  d.q_stride_b = q.stride(0), d.q_stride_s = q.stride(1), d.q_stride_h = q.stride(2);
  d.k = k.data_ptr();
  d.k_stride_page = k.stride(0), d.k_stride_slot = k.stride(1), d.k_stride_h = k.stride(2);
  d.v = v.data_ptr();
  d.v_stride_page = v.stride(0), d.v_stride_slot = v.stride(1), d.v_stride_h = v.stride(2);
  d.out = out.data_ptr();
  d.out_stride_b = out.stride(0), d.out_stride_s = out.stride(1), d.out_stride_h = out.stride(2);
  d.seqlens = static_cast<const int32_t*>(len.data_ptr());
  d.q_start = static_cast<const int32_t*>(qs.ptr());
  if (table) {
    d.page_table = static_cast<const int32_t*>(table.ptr());
    d.max_pages = static_cast<int>(table->size(1));
    d.page_size = static_cast<int>(page);
  }
  d.max_seqlen = static_cast<int>(most);
  d.batch = static_cast<int>(B), d.q_len = static_cast<int>(S), d.num_q_heads = static_cast<int>(Hq);
  d.num_kv_heads = static_cast<int>(Hkv), d.head_dim = static_cast<int>(D);
  if (kn) {
    d.k_new = kn.ptr();
    d.v_new = vn.ptr();
    d.new_stride_b = kn->stride(0), d.new_stride_s = kn->stride(1), d.new_stride_h = kn->stride(2);
  }
  size_t need = 0;
  check(api.attn_size(&d, &need), "fdllm_kv_attn_workspace_size");
  const Stream s(q);
  const Workspace ws = s.workspace(need, q);
  check(launch([&] { return api.attn(&d, ws.ptr, ws.bytes, s.ptr); }), "fdllm_kv_attn_fwd");
  return wrap(std::move(out));
}

// hidden, indices, weight | None, eps, mode, with_gathered -> (normed, gathered | None)
PyObject* gather(PyObject* const* a, Py_ssize_t n) {
  arity(n, 6);
  const Tensor &h = tensor(a[0]), &idx = tensor(a[1]);
  const Opt w(a[2]);
  const int mode = static_cast<int>(integer(a[4]));
  const float eps = static_cast<float>(number(a[3]));
  const int both = PyObject_IsTrue(a[5]);
  if (both < 0) throw PyFailed{};
  plain(h.dim() == 3 && idx.dim() == 2 && idx.size(0) == h.size(0) && h.stride(2) == 1 && idx.device() == h.device() &&
        idx.scalar_type() == at::kLong && idx.stride(1) == 1);
  const int64_t B = h.size(0), S = h.size(1), H = h.size(2), T = idx.size(1);
  plain(B <= INT32_MAX && S <= INT32_MAX && H <= INT32_MAX && T <= INT32_MAX);
  if (w) plain(w->device() == h.device() && w->is_contiguous() && w->numel() == H);
  else plain(mode == FDLLM_NORM_PLAIN);
  const int dt = dtype_code(h.scalar_type()), wdt = w ? dtype_code(w->scalar_type()) : 0;
  Tensor normed = empty({B, T, H}, h), gathered;
  if (both) gathered = empty({B, T, H}, h);
  const Stream s(h);
  check(launch([&] { return api.gather(h.data_ptr(), h.stride(0), h.stride(1), static_cast<const int64_t*>(idx.data_ptr()), idx.stride(0),
                   w.ptr(), wdt, normed.data_ptr(), gathered.defined() ? gathered.data_ptr() : nullptr,
                   static_cast<int>(B), static_cast<int>(S), static_cast<int>(T), static_cast<int>(H),
                   eps, dt, mode, s.ptr); }),
        "fdllm_gather_rmsnorm");
  Ref x(wrap(std::move(normed)));
  if (!gathered.defined()) return PyTuple_Pack(2, x.o, Py_None);
  Ref y(wrap(std::move(gathered)));
  return PyTuple_Pack(2, x.o, y.o);
}

// values, indices, cache, current | None -> True
PyObject* scatter(PyObject* const* a, Py_ssize_t n) {
  arity(n, 4);
  const Tensor &v = tensor(a[0]), &idx = tensor(a[1]), &c = tensor(a[2]);
  const Opt cur(a[3]);
  plain(v.dim() == 3 && v.is_contiguous() && idx.dim() == 2 && idx.device() == v.device() &&
        idx.scalar_type() == at::kLong && idx.stride(1) == 1 && idx.size(0) == v.size(0) && idx.size(1) == v.size(1) &&
        c.dim() == 3 && same(v, c) && c.size(0) == v.size(0) && c.size(2) == v.size(2) && c.stride(2) == 1);
  if (cur) plain(same(v, *cur) && cur->sizes() == c.sizes() && cur->stride(2) == 1);
  plain(c.size(1) <= INT32_MAX && v.size(1) <= INT32_MAX && v.size(2) <= INT32_MAX && v.size(0) <= INT32_MAX);
  const int dt = dtype_code(v.scalar_type());
  const Stream s(v);
  check(launch([&] { return api.scatter(v.data_ptr(), static_cast<const int64_t*>(idx.data_ptr()), idx.stride(0), c.data_ptr(), c.stride(0),
                    c.stride(1), cur.ptr(), cur ? cur->stride(0) : 0, cur ? cur->stride(1) : 0,
                    static_cast<int>(v.size(0)), static_cast<int>(c.size(1)), static_cast<int>(v.size(1)),
                    static_cast<int>(v.size(2)), dt, s.ptr); }),
        "fdllm_scatter_rows");
  Py_RETURN_TRUE;
}

// x, residual, weight | None, eps, mode -> (sum, normed)
PyObject* add_norm(PyObject* const* a, Py_ssize_t n) {
  arity(n, 5);
  const Tensor &x = tensor(a[0]), &r = tensor(a[1]);
  const Opt w(a[2]);
  const int mode = static_cast<int>(integer(a[4]));
  const float eps = static_cast<float>(number(a[3]));
  plain(x.dim() >= 1 && same(x, r) && half_type(x.scalar_type()) && x.sizes() == r.sizes() && x.is_contiguous() &&
        r.is_contiguous() && x.size(-1) > 0);
  const int64_t H = x.size(-1);
  if (w) plain(w->device() == x.device() && w->is_contiguous() && w->numel() == H);
  else plain(mode == FDLLM_NORM_PLAIN);
  plain(H <= INT32_MAX && x.numel() / H <= INT32_MAX);
  const int wdt = w ? dtype_code(w->scalar_type()) : 0;
  Tensor sum = empty(x.sizes(), x), normed = empty(x.sizes(), x);
  const Stream s(x);
  check(launch([&] { return api.add_norm(x.data_ptr(), r.data_ptr(), w.ptr(), wdt, sum.data_ptr(), normed.data_ptr(),
                     static_cast<int>(x.numel() / H), static_cast<int>(H), eps,
                     dtype_code(x.scalar_type()), mode, s.ptr); }),
        "fdllm_add_rmsnorm");
  Ref p(wrap(std::move(sum)));
  Ref q(wrap(std::move(normed)));
  return PyTuple_Pack(2, p.o, q.o);
}

// A gradient to record, or a forward-mode tangent to carry.
bool differentiates(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t && t->_fw_grad(0).defined()) return true;
  if (!c10::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t && t->requires_grad()) return true;
  return false;
}

// What ops.linear_fits accepts (with x's rows in place).
bool fits(const Tensor& x, const Tensor& w, const Tensor* up, const Tensor* bias) {
  if (!half_type(x.scalar_type()) || x.dim() < 2 || w.dim() != 2) return false;
  const int64_t N = w.size(0), K = w.size(1);
  if (x.size(-1) != K || K % 64 || K < 64 || K > 65536 || N % 8 || N <= 0 || N > (1 << 24) || x.numel() <= 0 ||
      x.numel() > 128 * K || differentiates({&x, &w, up, bias}))
    return false;
  auto rows = [&](const Tensor& t) {
    return same(x, t) && t.sizes() == w.sizes() && t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  if (!rows(w) || (up && !rows(*up))) return false;
  return !bias || (same(x, *bias) && bias->dim() == 1 && bias->size(0) == N && bias->is_contiguous() &&
                   reinterpret_cast<uintptr_t>(bias->data_ptr()) % 16 == 0);
}

// x, weight, bias | None -> whether ops.linear takes them
PyObject* linear_takes(PyObject* const* a, Py_ssize_t n) {
  arity(n, 3);
  const Opt bias(a[2]);
  plain(fits(tensor(a[0]), tensor(a[1]), nullptr, bias.t));
  Py_RETURN_TRUE;
}

// x, weight, up weight | None, bias | None
PyObject* linear(PyObject* const* a, Py_ssize_t n) {
  arity(n, 4);
  const Tensor &x = tensor(a[0]), &w = tensor(a[1]);
  const Opt up(a[2]), bias(a[3]);
  plain(fits(x, w, up.t, bias.t) && x.is_contiguous() && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0);
  const int N = static_cast<int>(w.size(0)), K = static_cast<int>(w.size(1)), m = static_cast<int>(x.numel() / K);
  auto sizes = x.sizes().vec();
  sizes.back() = N;
  Tensor out = empty(sizes, x);
  size_t need = 0;
  check(api.linear_size(m, N, K, up ? 1 : 0, &need), "fdllm_linear_workspace_size");
  const Stream s(x);
  const Workspace ws = s.workspace(need, x);
  check(launch([&] { return api.linear(x.data_ptr(), K, w.data_ptr(), up.ptr(), bias.ptr(), out.data_ptr(), m, N, K,
                   dtype_code(x.scalar_type()), ws.ptr, ws.bytes, s.ptr); }),
        "fdllm_linear");
  return wrap(std::move(out));
}

// x, wq, bq, wk, bk, wv, bv, cos, sin, k_cache, v_cache, write_start, write_offset, k_block,
// v_block, block_offset, head_dim -> q
PyObject* qkv(PyObject* const* a, Py_ssize_t n) {
  arity(n, 17);
  const Tensor& x = tensor(a[0]);
  const Tensor *w[3], *bias[3];
  plain(x.dim() == 3 && half_type(x.scalar_type()) && x.stride(2) == 1);
  const int64_t B = x.size(0), S = x.size(1), H = x.size(2), D = integer(a[16]);
  plain(D > 0 && x.stride(1) % 8 == 0 && (B <= 1 || x.stride(0) == S * x.stride(1)));
  for (int i = 0; i < 3; ++i) {
    w[i] = &tensor(a[1 + 2 * i]);
    const Opt b(a[2 + 2 * i]);
    bias[i] = b.t;
    plain(w[i]->dim() == 2 && same(x, *w[i]) && w[i]->size(1) == H && w[i]->size(0) % D == 0 && w[i]->is_contiguous());
    if (b) plain(same(x, *b) && b->dim() == 1 && b->size(0) == w[i]->size(0) && b->is_contiguous());
  }
  plain(w[1]->size(0) == w[2]->size(0));
  const int64_t Hq = w[0]->size(0) / D, Hkv = w[1]->size(0) / D;
  const Tensor &cos = tensor(a[7]), &sin = tensor(a[8]);
  plain(same(x, cos) && same(x, sin) && cos.dim() == 3 && cos.sizes() == sin.sizes() && cos.strides() == sin.strides() &&
        cos.size(1) == S && cos.size(2) == D && (cos.size(0) == 1 || cos.size(0) == B) && cos.stride(2) == 1 &&
        cos.stride(0) % 8 == 0 && cos.stride(1) % 8 == 0);
  auto pair = [&](PyObject* ok, PyObject* ov, const Tensor** k, const Tensor** v) {
    plain((ok == Py_None) == (ov == Py_None));
    if (ok == Py_None) return false;
    *k = &tensor(ok);
    *v = &tensor(ov);
    for (const Tensor* t : {*k, *v})
      plain(same(x, *t) && t->dim() == 4 && t->size(0) == B && t->size(2) == Hkv && t->size(3) == D && t->stride(3) == 1 &&
            t->size(1) <= INT32_MAX);
    plain((*k)->strides() == (*v)->strides());
    return true;
  };
  const Tensor *kc, *vc, *kb, *vb;
  const bool cache = pair(a[9], a[10], &kc, &vc), block = pair(a[13], a[14], &kb, &vb);
  const Opt start(a[11]);
  if (start) plain(start->device() == x.device() && start->scalar_type() == at::kInt && start->is_contiguous());
  plain(B <= INT32_MAX && S <= INT32_MAX && H <= INT32_MAX && Hq <= INT32_MAX && D <= INT32_MAX);
  Tensor out = empty({B, S, Hq, D}, x);
  fdllm_qkv_rope_desc d = {};
  fdllm_rope_kv_desc& r = d.rope;
  d.x = x.data_ptr();
  d.x_stride_row = x.stride(1);
  d.hidden = static_cast<int>(H);
  d.wq = w[0]->data_ptr(), d.wk = w[1]->data_ptr(), d.wv = w[2]->data_ptr();
  d.bq = bias[0] ? bias[0]->data_ptr() : nullptr;
  d.bk = bias[1] ? bias[1]->data_ptr() : nullptr;
  d.bv = bias[2] ? bias[2]->data_ptr() : nullptr;
  r.cos = cos.data_ptr(), r.sin = sin.data_ptr();
  r.cs_stride_b = cos.size(0) == B && B > 1 ? cos.stride(0) : 0;
  r.cs_stride_s = cos.stride(1);
  r.q_out = out.data_ptr();
  r.qo_stride_b = out.stride(0), r.qo_stride_s = out.stride(1), r.qo_stride_h = out.stride(2);
  if (cache) {
    r.k_cache = kc->data_ptr(), r.v_cache = vc->data_ptr();
    r.c_stride_b = kc->stride(0), r.c_stride_s = kc->stride(1), r.c_stride_h = kc->stride(2);
    r.cache_len = static_cast<int>(kc->size(1));
    r.write_start = static_cast<const int32_t*>(start.ptr());
    r.write_offset = static_cast<int>(integer(a[12]));
  }
  if (block) {
    r.k_block = kb->data_ptr(), r.v_block = vb->data_ptr();
    r.bc_stride_b = kb->stride(0), r.bc_stride_s = kb->stride(1), r.bc_stride_h = kb->stride(2);
    r.block_len = static_cast<int>(kb->size(1));
    r.block_offset = static_cast<int>(integer(a[15]));
  }
  r.batch = static_cast<int>(B), r.seq_len = static_cast<int>(S), r.num_q_heads = static_cast<int>(Hq);
  r.num_kv_heads = static_cast<int>(Hkv), r.head_dim = static_cast<int>(D);
  r.dtype = dtype_code(x.scalar_type());
  size_t need = 0;
  if (B * S <= 128) check(api.qkv_size(&d, &need), "fdllm_qkv_rope_workspace_size");
  const Stream s(x);
  const Workspace ws = s.workspace(need, x);
  check(launch([&] { return api.qkv(&d, ws.ptr, ws.bytes, s.ptr); }), "fdllm_qkv_rope_kv_write");
  return wrap(std::move(out));
}

// logits, tokens, mask_id, threshold, row_offset, shift, finished | None, stop (-1: none),
// row_tok, row_conf, counts, parts -> True
PyObject* unmask(PyObject* const* a, Py_ssize_t n) {
  arity(n, 12);
  const Tensor &lg = tensor(a[0]), &tok = tensor(a[1]), &rt = tensor(a[8]), &rc = tensor(a[9]), &cn = tensor(a[10]), &parts = tensor(a[11]);
  const Opt fin(a[6]);
  plain(lg.dim() == 3 && tok.dim() == 2 && tok.size(0) == lg.size(0) && tok.device() == lg.device() &&
        half_type(lg.scalar_type()) && lg.stride(2) == 1 && tok.scalar_type() == at::kLong && tok.stride(1) == 1);
  const int64_t B = tok.size(0), L = tok.size(1), V = lg.size(2);
  if (fin)
    plain(fin->device() == lg.device() && (fin->scalar_type() == at::kBool || fin->scalar_type() == at::kByte) &&
          fin->is_contiguous() && fin->numel() == B);
  plain(rt.device() == lg.device() && rt.dim() == 2 && rt.size(0) == B && rt.size(1) == L && V <= INT32_MAX &&
        B <= INT32_MAX && L <= INT32_MAX);
  const long offset = integer(a[4]), shift = integer(a[5]), mask = integer(a[2]), stop = integer(a[7]);
  const float threshold = static_cast<float>(number(a[3]));
  plain(offset >= INT32_MIN && offset <= INT32_MAX && shift >= INT32_MIN && shift <= INT32_MAX);
  size_t need = 0;
  check(api.unmask_size(static_cast<int>(V), static_cast<int>(B), static_cast<int>(L), &need), "fdllm_unmask_workspace_size");
  plain(parts.device() == lg.device() && parts.scalar_type() == at::kByte && static_cast<size_t>(parts.numel()) >= need);
  const Stream s(lg);
  check(launch([&] { return api.unmask(lg.data_ptr(), lg.stride(0), lg.stride(1), static_cast<int>(V), static_cast<int>(offset),
                   static_cast<int>(shift), static_cast<int64_t*>(tok.data_ptr()), tok.stride(0),
                   static_cast<uint8_t*>(fin.ptr()), mask, threshold, stop,
                   static_cast<int64_t*>(rt.data_ptr()), static_cast<float*>(rc.data_ptr()),
                   static_cast<int32_t*>(cn.data_ptr()), static_cast<int>(B), static_cast<int>(L),
                   dtype_code(lg.scalar_type()), parts.data_ptr(), need, s.ptr); }),
        "fdllm_unmask_step_ws");
  Py_RETURN_TRUE;
}

// entry point addresses in Api's order, stream lookup, workspace dictionary, its get
PyObject* init(PyObject*, PyObject* args) {
  PyObject *addr, *stream, *buffers, *get;
  if (!PyArg_ParseTuple(args, "O!OO!O", &PyTuple_Type, &addr, &stream, &PyDict_Type, &buffers, &get)) return nullptr;
  static_assert(sizeof(Api) == kApis * sizeof(void*), "entry points");
  if (PyTuple_Size(addr) != kApis) {
    PyErr_SetString(PyExc_ValueError, "entry points");
    return nullptr;
  }
  void* p[kApis];
  for (int i = 0; i < kApis; ++i) {
    p[i] = PyLong_AsVoidPtr(PyTuple_GetItem(addr, i));
    if (!p[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
      return nullptr;
    }
  }
  memcpy(&api, p, sizeof(api));
  for (PyObject* o : {stream, buffers, get}) Py_INCREF(o);
  g_stream = stream;
  g_buffers = buffers;
  g_get = get;
  Py_RETURN_NONE;
}

#define FDLLM_CALL(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&call<name>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FDLLM_CALL(attn),   FDLLM_CALL(gather), FDLLM_CALL(scatter), FDLLM_CALL(add_norm),
                         FDLLM_CALL(linear), FDLLM_CALL(linear_takes), FDLLM_CALL(qkv),    FDLLM_CALL(unmask),  {"init", init, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "fdllm_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" PyObject* PyInit_fdllm_host() {
  PyObject* m = PyModule_Create(&module);
  // torch's C++ API has no stable layout: the loader compares
  if (m && PyModule_AddStringConstant(m, "torch_version", FDLLM_TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
