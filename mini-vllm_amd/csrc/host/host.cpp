// The host side of the decode step's ops in native code: argument checks, plan, output
// allocation and the library call of an op in one C function each.
//
// What bounds a small eager call is the host, not the GPU: in Python the same work (some eighty
// attribute reads, two ctypes calls of up to thirty arguments) took 8-11 us a call. Measured in
// back-to-back eager calls, with the Python body and with this one: a lone sequence's fused
// decode attention 21.1 -> 16.3 us (its kernels alone: 16.2), the MLP's three
// launches of 32 rows 22 -> 13.4 us (kernels alone: 13.2), four float32 sequences' decode
// attention 16.7 -> 15.2 us (kernels: 14.9).
//
// Every function serves the calls whose arguments are exactly what the kernels take and
// answers None to anything else - another type, dtype, shape, stride, device or integer kind, a
// tensor subclass or wrapper, a workspace not there yet - without having done anything: the
// caller then runs the Python path, which converts, allocates or refuses as it always did.
// Nothing is kept between calls: the library's entries and the workspaces are the extension
// object's and come with each call, the workspaces as its dict by (device, stream).

#include <Python.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include "minivllm_hip.h"

namespace {

using PlanFn = decltype(&mvllm_paged_attention_plan);
using PagedFn = decltype(&mvllm_paged_attention);
using FreshFn = decltype(&mvllm_paged_decode_qk_norm_rope);
using BytesFn = decltype(&mvllm_linear_workspace_bytes);
using SwigluFn = decltype(&mvllm_linear_swiglu);
using NormFn = decltype(&mvllm_linear_residual_rmsnorm);
using ErrorFn = decltype(&mvllm_last_error);

// One library's entries; the extension object that loaded the library holds them as a capsule.
struct Entries {
  PlanFn plan;
  PagedFn paged;
  FreshFn fresh;
  BytesFn linear_bytes;
  SwigluFn swiglu;
  NormFn norm;
  ErrorFn error;
};

constexpr const char* kCapsule = "mvllm_host.entries";

const Entries* entries_of(PyObject* o) {
  return static_cast<const Entries*>(PyCapsule_GetPointer(o, kCapsule));
}

// An active dispatch or function mode sees the Python path's calls; it has none to see here.
bool modes() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() ||
         at::impl::torch_function_mode_enabled();
}

// A plain strided device tensor or parameter (no subclass, no transform's wrapper, no lazy
// negation), or null.
const at::Tensor* tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet kWrapped(
      {c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
       c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
       c10::DispatchKey::Negative, c10::DispatchKey::Conjugate});
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() ||
      t.key_set().has_any(kWrapped)) {
    return nullptr;
  }
  return &t;
}

bool integer(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return v > INT32_MIN && v < INT32_MAX;
}

bool number(PyObject* o, double& v) {
  if (!PyFloat_CheckExact(o)) return false;
  v = PyFloat_AS_DOUBLE(o);
  return true;
}

int code_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return MVLLM_DTYPE_F32;
    case at::kHalf: return MVLLM_DTYPE_F16;
    case at::kBFloat16: return MVLLM_DTYPE_BF16;
    case at::kFloat8_e4m3fn: return MVLLM_DTYPE_FP8_E4M3;
    default: return -1;
  }
}

bool sixteen_bit(const at::Tensor& t) {
  return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16;
}

bool aligned(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// The extension's workspace of (device, stream), at least `need` bytes, or false.
// `held` keeps it alive over the launch, as the Python path's own reference does.
bool workspace(PyObject* dict, int device, void* stream, uint64_t need, at::Tensor& held) {
  PyObject* key = Py_BuildValue("(iK)", device,
                                static_cast<unsigned long long>(reinterpret_cast<uintptr_t>(stream)));
  if (key == nullptr) {
    PyErr_Clear();
    return false;
  }
  PyObject* found = PyDict_GetItem(dict, key);  // borrowed
  Py_DECREF(key);
  if (found == nullptr || !THPVariable_Check(found)) return false;
  held = THPVariable_Unpack(found);
  return static_cast<uint64_t>(held.numel()) >= need;
}

void* pointer(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
uint64_t bytes(const at::Tensor& t) { return t.defined() ? static_cast<uint64_t>(t.numel()) : 0; }

PyObject* none() { Py_RETURN_NONE; }

PyObject* finish(const Entries* e, int rc, PyObject* result) {
  if (rc == 0) return result;
  Py_XDECREF(result);
  const char* message = e->error();
  PyErr_SetString(PyExc_RuntimeError,
                  message != nullptr && message[0] ? message : "libminivllm_hip call failed");
  return nullptr;
}

// The tensors of a paged call and whether the kernels take them as they are.
struct Paged {
  const at::Tensor *q, *kp, *vp, *tables, *cu, *ctx, *lens, *ks = nullptr, *vs = nullptr;
  int64_t max_q = 1, max_ctx = 0;
  double scale = 0;
  int device = 0, q_code = -1, kv_code = -1;

  // q's rows may be strided when the caller checks them (`rows` false)
  bool check(bool rows) {
    if (!q || !kp || !vp || !tables || !cu || !ctx || !lens) return false;
    if (q->dim() != 3 || kp->dim() != 4 || kp->sizes() != vp->sizes() || tables->dim() != 2 ||
        cu->dim() != 1 || ctx->dim() != 1 || lens->dim() != 1) {
      return false;
    }
    if ((rows && !q->is_contiguous()) || !kp->is_contiguous() || !vp->is_contiguous()) return false;
    q_code = code_of(q->scalar_type());
    kv_code = code_of(kp->scalar_type());
    if (q_code < 0 || q_code == MVLLM_DTYPE_FP8_E4M3 || kv_code < 0 ||
        vp->scalar_type() != kp->scalar_type()) {
      return false;
    }
    const bool fp8 = kv_code == MVLLM_DTYPE_FP8_E4M3;
    if (!fp8 && kv_code != q_code) return false;
    const int64_t d = q->size(2), hk = kp->size(2), bs = kp->size(1), n = lens->size(0);
    if (d != kp->size(3) || (d != 32 && d != 64 && d != 128 && d != 256) || hk <= 0 ||
        q->size(1) <= 0 || q->size(1) % hk != 0 || bs <= 0 || (bs & (bs - 1)) != 0) {
      return false;
    }
    if (n <= 0 || q->size(0) <= 0 || tables->size(0) != n || ctx->size(0) != n || cu->size(0) != n + 1) {
      return false;
    }
    device = q->get_device();
    for (const at::Tensor* t : {tables, cu, ctx, lens}) {
      if (t->scalar_type() != at::kInt || !t->is_contiguous() || t->get_device() != device) return false;
    }
    if (kp->get_device() != device || vp->get_device() != device) return false;
    if (fp8 != (ks != nullptr) || fp8 != (vs != nullptr)) return false;
    if (fp8) {
      for (const at::Tensor* t : {ks, vs}) {
        if (t->scalar_type() != at::kFloat || t->dim() != 2 || t->size(0) != kp->size(0) ||
            t->size(1) != hk || !t->is_contiguous() || t->get_device() != device) {
          return false;
        }
      }
    }
    return max_q >= 1 && max_ctx >= max_q && q->size(0) < INT32_MAX && n < INT32_MAX &&
           tables->size(1) < INT32_MAX;
  }

  bool plan(const Entries* e, mvllm_paged_plan& out) const {
    return e->plan(static_cast<int32_t>(q->size(0)), static_cast<int32_t>(lens->size(0)),
                  static_cast<int32_t>(q->size(1)), static_cast<int32_t>(kp->size(2)),
                  static_cast<int32_t>(q->size(2)), static_cast<int32_t>(kp->size(1)),
                  static_cast<int32_t>(max_q), static_cast<int32_t>(max_ctx), q_code, kv_code,
                  nullptr, &out) == 0;
  }
};

bool optional(PyObject* o, const at::Tensor*& t) {
  if (o == Py_None) return true;
  t = tensor(o);
  return t != nullptr;
}

// (q, key_pool, value_pool, block_tables, cu_seqlens_q, context_lens, seq_lens, max_query_len,
//  max_context_len, scale, k_scale, v_scale)
bool read_paged(PyObject* const* a, Paged& p) {
  p.q = tensor(a[0]);
  p.kp = tensor(a[1]);
  p.vp = tensor(a[2]);
  p.tables = tensor(a[3]);
  p.cu = tensor(a[4]);
  p.ctx = tensor(a[5]);
  p.lens = tensor(a[6]);
  return integer(a[7], p.max_q) && integer(a[8], p.max_ctx) && number(a[9], p.scale) &&
         optional(a[10], p.ks) && optional(a[11], p.vs) && p.check(true);
}

PyObject* paged_served(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Paged p;
  return PyBool_FromLong(n == 12 && !modes() && read_paged(a, p));
  END_HANDLE_TH_ERRORS
}

// (entries, workspaces, then the arguments above)
PyObject* paged_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Paged p;
  if (n != 14 || !PyDict_CheckExact(a[1]) || modes() || !read_paged(a + 2, p)) return none();
  const Entries* e = entries_of(a[0]);
  if (e == nullptr) return nullptr;
  mvllm_paged_plan plan;
  if (!p.plan(e, plan)) return none();
  void* stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(p.device)).stream();
  at::Tensor ws;
  if (plan.workspace_bytes > 0 &&
      !workspace(a[1], p.device, stream, plan.workspace_bytes, ws)) {
    return none();
  }
  at::Tensor out = at::empty(p.q->sizes(), p.q->options());
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = e->paged(out.data_ptr(), p.q->data_ptr(), p.kp->data_ptr(), p.vp->data_ptr(),
               p.ks ? static_cast<const float*>(p.ks->data_ptr()) : nullptr,
               p.vs ? static_cast<const float*>(p.vs->data_ptr()) : nullptr,
               static_cast<const int32_t*>(p.tables->data_ptr()),
               static_cast<const int32_t*>(p.cu->data_ptr()),
               static_cast<const int32_t*>(p.ctx->data_ptr()),
               static_cast<const int32_t*>(p.lens->data_ptr()),
               static_cast<int32_t>(p.q->size(0)), static_cast<int32_t>(p.lens->size(0)),
               static_cast<int32_t>(p.q->size(1)), static_cast<int32_t>(p.kp->size(2)),
               static_cast<int32_t>(p.q->size(2)), static_cast<int32_t>(p.kp->size(1)),
               p.kp->size(0), static_cast<int32_t>(p.tables->size(1)),
               static_cast<int32_t>(p.max_q), static_cast<int32_t>(p.max_ctx),
               static_cast<float>(p.scale), p.q_code, p.kv_code, nullptr, pointer(ws), bytes(ws), stream);
  Py_END_ALLOW_THREADS
  return finish(e, rc, rc == 0 ? THPVariable_Wrap(std::move(out)) : nullptr);
  END_HANDLE_TH_ERRORS
}

// (entries, workspaces, q, k, v, q_weight, k_weight, cos, sin, eps, key_pool, value_pool,
//  block_tables, cu_seqlens_q, context_lens, seq_lens, max_context_len, scale)
PyObject* paged_decode_qk_norm_rope(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 18 || !PyDict_CheckExact(args[1]) || modes()) return none();
  const Entries* e = entries_of(args[0]);
  if (e == nullptr) return nullptr;
  PyObject* const* a = args + 2;
  Paged p;
  double eps;
  p.q = tensor(a[0]);
  p.kp = tensor(a[8]);
  p.vp = tensor(a[9]);
  p.tables = tensor(a[10]);
  p.cu = tensor(a[11]);
  p.ctx = tensor(a[12]);
  p.lens = tensor(a[13]);
  const at::Tensor *k = tensor(a[1]), *v = tensor(a[2]), *qw = tensor(a[3]), *kw = tensor(a[4]),
                   *cos = tensor(a[5]), *sin = tensor(a[6]);
  if (!k || !v || !qw || !kw || !cos || !sin || !number(a[7], eps) || !integer(a[14], p.max_ctx) ||
      !number(a[15], p.scale) || !p.check(false)) {
    return none();
  }
  const at::Tensor& q = *p.q;
  const int64_t d = q.size(2), seqs = p.lens->size(0), hk = p.kp->size(2), group = q.size(1) / hk;
  const int64_t chunk = group % 4 == 0 ? 4 : (group % 2 == 0 ? 2 : 1);
  if (!sixteen_bit(q) || p.kv_code != p.q_code || d != 128 || q.size(0) != seqs || seqs > 4096 ||
      hk * (group / chunk) > 8) {
    return none();
  }
  for (const at::Tensor* t : {k, v, qw, kw}) {
    if (t->scalar_type() != q.scalar_type() || t->get_device() != p.device) return none();
  }
  if (k->dim() != 3 || k->size(0) != seqs || k->size(1) != hk || k->size(2) != d ||
      v->sizes() != k->sizes() || k->stride(0) != v->stride(0)) {
    return none();
  }
  for (const at::Tensor* t : {p.q, k, v}) {  // heads contiguous within each token
    if (t->stride(2) != 1 || t->stride(1) != d) return none();
  }
  for (const at::Tensor* t : {qw, kw}) {
    if (t->dim() != 1 || t->size(0) != d || !t->is_contiguous()) return none();
  }
  for (const at::Tensor* t : {cos, sin}) {
    if (t->scalar_type() != at::kFloat || t->dim() != 2 || t->size(1) != d ||
        t->size(0) != cos->size(0) || !t->is_contiguous() || t->get_device() != p.device) {
      return none();
    }
  }
  mvllm_paged_plan plan;
  if (!p.plan(e, plan) || plan.decode_mode != MVLLM_DECODE_STREAM) return none();
  void* stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(p.device)).stream();
  at::Tensor ws;
  const uint64_t need = plan.workspace_bytes > 256 ? plan.workspace_bytes : 256;
  if (!workspace(args[1], p.device, stream, need, ws)) return none();
  at::Tensor out = at::empty(q.sizes(), q.options());
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = e->fresh(out.data_ptr(), q.data_ptr(), k->data_ptr(), v->data_ptr(), q.stride(0),
               k->stride(0), qw->data_ptr(), kw->data_ptr(),
               static_cast<const float*>(cos->data_ptr()),
               static_cast<const float*>(sin->data_ptr()), cos->size(0), static_cast<float>(eps),
               p.kp->data_ptr(), p.vp->data_ptr(),
               static_cast<const int32_t*>(p.tables->data_ptr()),
               static_cast<const int32_t*>(p.cu->data_ptr()),
               static_cast<const int32_t*>(p.ctx->data_ptr()),
               static_cast<const int32_t*>(p.lens->data_ptr()), static_cast<int32_t>(seqs),
               static_cast<int32_t>(q.size(1)), static_cast<int32_t>(hk), static_cast<int32_t>(d),
               static_cast<int32_t>(p.kp->size(1)), p.kp->size(0),
               static_cast<int32_t>(p.tables->size(1)), static_cast<int32_t>(p.max_ctx),
               static_cast<float>(p.scale), p.q_code, nullptr, pointer(ws), bytes(ws), stream);
  Py_END_ALLOW_THREADS
  return finish(e, rc, rc == 0 ? THPVariable_Wrap(std::move(out)) : nullptr);
  END_HANDLE_TH_ERRORS
}

// x [m, k] against a packed weight of n rows: the skinny kernels take it as it is.
bool skinny(const at::Tensor* x, const at::Tensor* w, int64_t n) {
  if (!x || !w || x->dim() != 2 || !sixteen_bit(*x) || w->scalar_type() != x->scalar_type() ||
      w->get_device() != x->get_device()) {
    return false;
  }
  const int64_t m = x->size(0), k = x->size(1);
  return m >= 1 && m <= 64 && k >= 1 && k % 64 == 0 && k <= 65536 && n >= 1 &&
         w->numel() == (n + 31) / 32 * 32 * k && x->is_contiguous() && w->is_contiguous() &&
         aligned(*x) && aligned(*w);
}

// (entries, workspaces, x, packed, n), n the packed rows: twice the outputs
PyObject* linear_swiglu(PyObject*, PyObject* const* a, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  int64_t n;
  if (count != 5 || !PyDict_CheckExact(a[1]) || modes() || !integer(a[4], n)) return none();
  const Entries* e = entries_of(a[0]);
  if (e == nullptr) return nullptr;
  const at::Tensor *x = tensor(a[2]), *w = tensor(a[3]);
  if (n % 32 != 0 || !skinny(x, w, n)) return none();
  const int device = x->get_device();
  void* stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device)).stream();
  const int64_t m = x->size(0), k = x->size(1);
  const uint64_t need = e->linear_bytes(m, n, k);
  at::Tensor ws;
  if (need > 0 && !workspace(a[1], device, stream, need, ws)) return none();
  at::Tensor y = at::empty({m, n / 2}, x->options());
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = e->swiglu(y.data_ptr(), x->data_ptr(), w->data_ptr(), m, n / 2, k,
                code_of(x->scalar_type()), pointer(ws), bytes(ws), stream);
  Py_END_ALLOW_THREADS
  return finish(e, rc, rc == 0 ? THPVariable_Wrap(std::move(y)) : nullptr);
  END_HANDLE_TH_ERRORS
}

// (entries, workspaces, x, packed, n, residual, norm_weight, eps)
PyObject* linear_residual_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  int64_t n;
  double eps;
  if (count != 8 || !PyDict_CheckExact(a[1]) || modes() || !integer(a[4], n) || !number(a[7], eps)) {
    return none();
  }
  const Entries* e = entries_of(a[0]);
  if (e == nullptr) return nullptr;
  const at::Tensor *x = tensor(a[2]), *w = tensor(a[3]), *r = tensor(a[5]), *g = tensor(a[6]);
  if (!skinny(x, w, n) || !r || !g || x->size(1) <= 1024 || n % 512 != 0 || n > 4096) return none();
  const int64_t m = x->size(0), k = x->size(1);
  const int device = x->get_device();
  if (r->dim() != 2 || r->size(0) != m || r->size(1) != n || !r->is_contiguous() ||
      r->scalar_type() != x->scalar_type() || r->get_device() != device || g->dim() != 1 ||
      g->size(0) != n || !g->is_contiguous() || g->scalar_type() != x->scalar_type() ||
      g->get_device() != device) {
    return none();
  }
  void* stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device)).stream();
  const uint64_t need = e->linear_bytes(m, n, k);
  at::Tensor ws;
  if (need > 0 && !workspace(a[1], device, stream, need, ws)) return none();
  at::Tensor h = at::empty(r->sizes(), r->options()), normed = at::empty(r->sizes(), r->options());
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = e->norm(h.data_ptr(), normed.data_ptr(), x->data_ptr(), w->data_ptr(), r->data_ptr(),
              g->data_ptr(), m, n, k, static_cast<float>(eps), code_of(x->scalar_type()), pointer(ws),
              bytes(ws), stream);
  Py_END_ALLOW_THREADS
  if (rc != 0) return finish(e, rc, nullptr);
  PyObject* first = THPVariable_Wrap(std::move(h));
  PyObject* second = THPVariable_Wrap(std::move(normed));
  PyObject* both = first != nullptr && second != nullptr ? PyTuple_Pack(2, first, second) : nullptr;
  Py_XDECREF(first);
  Py_XDECREF(second);
  return both;
  END_HANDLE_TH_ERRORS
}

// A capsule of the library's entries, given by address: plan, paged attention, the fused decode, the projections'
// workspace size, gate/up with SwiGLU, residual with RMSNorm, the error text.
PyObject* entries(PyObject*, PyObject* args) {
  unsigned long long f[7];
  if (!PyArg_ParseTuple(args, "KKKKKKK", &f[0], &f[1], &f[2], &f[3], &f[4], &f[5], &f[6])) {
    return nullptr;
  }
  auto* e = new Entries{reinterpret_cast<PlanFn>(f[0]),   reinterpret_cast<PagedFn>(f[1]),
                        reinterpret_cast<FreshFn>(f[2]),  reinterpret_cast<BytesFn>(f[3]),
                        reinterpret_cast<SwigluFn>(f[4]), reinterpret_cast<NormFn>(f[5]),
                        reinterpret_cast<ErrorFn>(f[6])};
  PyObject* capsule = PyCapsule_New(e, kCapsule, [](PyObject* c) {
    delete static_cast<Entries*>(PyCapsule_GetPointer(c, kCapsule));
  });
  if (capsule == nullptr) delete e;
  return capsule;
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(name), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    {"entries", entries, METH_VARARGS, nullptr}, FAST(paged_served),   FAST(paged_attention),
    FAST(paged_decode_qk_norm_rope),       FAST(linear_swiglu),  FAST(linear_residual_rmsnorm),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "mvllm_host", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

// The build's identity, also to be read off the file before it is loaded.
extern "C" __attribute__((used, visibility("default"))) const char mvllm_host_id[] =
    "mvllm-host-id:" MVLLM_SOURCE_HASH;

PyMODINIT_FUNC PyInit_mvllm_host() {
  PyObject* m = PyModule_Create(&kModule);
  if (m != nullptr) PyModule_AddStringConstant(m, "source_hash", MVLLM_SOURCE_HASH);
  return m;
}
