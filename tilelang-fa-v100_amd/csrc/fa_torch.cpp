// Call marshalling for the Python entry points: tensor checks, argument structs
// and output allocation in one native call instead of ~60 Python-level ones.
//
// Bounds: small calls are limited by the host.  Through ctypes, filling an
// argument struct, the per-tensor checks and the stream lookup took 12-15 us
// of a 19 us forward ([1, 512, 16, 64], 7 us of GPU work) and of each call of
// an append + decode step.
//
// Every function takes the plain case only: exact torch.Tensor objects with
// storage on the current device, matching dtypes, shapes and strides the
// kernels address as they are, index tensors already int32 (int64 for slots),
// no dispatch mode.  Anything else returns None before any work, and the
// Python path, which converts, copies or raises, takes the call.  Otherwise
// the result is the outputs, or the library's negative status for the caller
// to raise.  Nothing is kept between calls except the library's entry points.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include <climits>
#include <cmath>

#include "fa355.h"

namespace {

struct Entries {
  decltype(&fa_fwd) fwd;
  decltype(&fa_decode_workspace_bytes) decode_workspace;
  decltype(&fa_paged_decode) decode;
  decltype(&fa_paged_prefill_num_splits) paged_splits;
  decltype(&fa_paged_prefill_splitkv_workspace_bytes) paged_workspace;
  decltype(&fa_paged_prefill_splitkv) paged;
  decltype(&fa_reshape_and_cache) cache_write;
} lib;

struct Call {
  int device;
  void* stream;
};

// A plain tensor on the call's device, or nullptr.
const at::Tensor* plain(PyObject* o, const Call& c, int64_t dim) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.dim() != dim || t.get_device() != c.device ||
      t.layout() != at::kStrided || !t.has_storage() || t.numel() == 0)
    return nullptr;
  return &t;
}

// The kernels can address it as it is: contiguous last dimension, 16-byte
// aligned, other strides multiples of 8 elements.
bool rows_ready(const at::Tensor& t) {
  const auto size = t.sizes(), stride = t.strides();
  const int64_t n = t.dim();
  if (stride[n - 1] != 1 || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0) return false;
  for (int64_t i = 0; i + 1 < n; ++i)
    if (size[i] > 1 && (stride[i] % 8 != 0 || stride[i] < 0)) return false;
  return true;
}

template <size_t N>
void set_strides(int64_t (&dst)[N], const at::Tensor& t) {
  for (size_t i = 0; i < N; ++i) dst[i] = t.size(i) == 1 ? 0 : t.stride(i);
}

bool half_code(const at::Tensor& t, int32_t* code) {
  if (t.scalar_type() == at::kHalf)
    *code = FA_DTYPE_F16;
  else if (t.scalar_type() == at::kBFloat16)
    *code = FA_DTYPE_BF16;
  else
    return false;
  return true;
}

bool fits(int64_t v) { return v <= INT_MAX; }

// int32 tensor of `dim` dimensions whose rows are contiguous.
bool index_ready(const at::Tensor* t) {
  return t && t->scalar_type() == at::kInt && t->is_contiguous();
}

bool call_of(PyObject* device, PyObject* stream, Call* c) {
  if (c10::impl::TorchDispatchModeTLS::any_modes_set()) return false;
  c->device = (int)PyLong_AsLong(device);
  c->stream = PyLong_AsVoidPtr(stream);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool number(PyObject* o, float* out) {
  if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  *out = (float)v;
  return true;
}

bool integer(PyObject* o, int64_t* out) {
  if (!PyLong_Check(o)) return false;
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  *out = v;
  return true;
}

// softmax_scale argument: None is 1 / sqrt(D).
bool scale_of(PyObject* o, int64_t D, float* out) {
  if (o == Py_None) {
    *out = (float)(1.0 / std::sqrt((double)D));
    return true;
  }
  return number(o, out);
}

PyObject* none() { Py_RETURN_NONE; }

// Allocations and launches can block (a full queue, hipMalloc): other threads
// run meanwhile, as they do under ctypes and torch's own calls.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// C++ exceptions (an allocation that fails, say) become Python ones, by torch's
// own translation.
template <class F>
PyObject* guarded(F f) {
  HANDLE_TH_ERRORS
  return f();
  END_HANDLE_TH_ERRORS
}

// dense_forward(q, k, v, scale, causal, left, right, with_lse, device, stream)
//   -> (out, lse or None) | status | None
PyObject* dense_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Call c;
    int64_t left, right;
    fa_fwd_args p = {};
    if (n != 10 || !call_of(a[8], a[9], &c) || !integer(a[5], &left) || !integer(a[6], &right) ||
        !number(a[3], &p.softmax_scale))
      return none();
    const at::Tensor *q = plain(a[0], c, 4), *k = plain(a[1], c, 4), *v = plain(a[2], c, 4);
    if (!q || !k || !v || !half_code(*q, &p.dtype) || k->scalar_type() != q->scalar_type() ||
        v->scalar_type() != q->scalar_type() || !rows_ready(*q) || !rows_ready(*k) ||
        !rows_ready(*v))
      return none();
    const int64_t B = q->size(0), Sq = q->size(1), H = q->size(2), D = q->size(3);
    const int64_t Sk = k->size(1), Hk = k->size(2), lim = int64_t(1) << 24;
    if (k->sizes() != v->sizes() || k->size(0) != B || k->size(3) != D || H % Hk != 0 ||
        (D != 64 && D != 128 && D != 256) || k->stride(1) >= lim || v->stride(1) >= lim ||
        !fits(B) || !fits(Sq) || !fits(Sk) || !fits(H) || left < -1 || right < -1 || !fits(left) ||
        !fits(right))
      return none();
    const bool with_lse = a[7] == Py_True;
    const bool causal = a[4] == Py_True;
    at::Tensor out, lse;
    int status;
    {
      NoGil no_gil;
      out = at::empty({B, Sq, H, D}, q->options().requires_grad(false));
      if (with_lse) lse = at::empty({B, H, Sq}, out.options().dtype(at::kFloat));
      p.q = q->data_ptr();
      p.k = k->data_ptr();
      p.v = v->data_ptr();
      p.out = out.data_ptr();
      p.lse = with_lse ? lse.data_ptr<float>() : nullptr;
      set_strides(p.q_stride, *q);
      set_strides(p.k_stride, *k);
      set_strides(p.v_stride, *v);
      set_strides(p.o_stride, out);
      p.batch = (int32_t)B;
      p.seqlen_q = (int32_t)Sq;
      p.seqlen_k = (int32_t)Sk;
      p.num_heads = (int32_t)H;
      p.num_heads_k = (int32_t)Hk;
      p.head_dim = (int32_t)D;
      p.causal = causal;
      p.has_window = left != -1 || right != -1;
      p.window_left = (int32_t)left;
      p.window_right = (int32_t)right;
      status = lib.fwd(&p, c.stream);
    }
    if (status != FA_OK) return PyLong_FromLong(status);
    PyObject* l = with_lse ? THPVariable_Wrap(lse) : (Py_INCREF(Py_None), Py_None);
    return Py_BuildValue("NN", THPVariable_Wrap(out), l);
  });
}

// Caches [num_pages, page_size, kv_heads, head_dim] of q's dtype and head_dim,
// and the scalars every paged entry point shares.
template <class Args>
bool caches(const at::Tensor* q, const at::Tensor* kc, const at::Tensor* vc, PyObject* block_size,
            PyObject* num_kv_heads, PyObject* scale, Args* p) {
  int64_t page, heads;
  if (!q || !kc || !vc || !half_code(*q, &p->dtype) || kc->scalar_type() != q->scalar_type() ||
      vc->scalar_type() != q->scalar_type() || !rows_ready(*q) || !rows_ready(*kc) ||
      !rows_ready(*vc) || kc->sizes() != vc->sizes())
    return false;
  const int64_t H = q->size(1), D = q->size(2), Hk = kc->size(2), P = kc->size(1);
  if (!integer(block_size, &page) || page != P || (P & (P - 1)) != 0 || kc->size(3) != D ||
      (D != 64 && D != 128 && D != 256 && D != 512) || H % Hk != 0 || !fits(kc->size(0)) ||
      !fits(P) || !fits(H) || !scale_of(scale, D, &p->softmax_scale))
    return false;
  if (num_kv_heads != Py_None && !(integer(num_kv_heads, &heads) && (heads == 0 || heads == Hk)))
    return false;
  p->q = q->data_ptr();
  p->k_cache = kc->data_ptr();
  p->v_cache = vc->data_ptr();
  set_strides(p->q_stride, *q);
  set_strides(p->k_stride, *kc);
  set_strides(p->v_stride, *vc);
  p->num_heads = (int32_t)H;
  p->num_kv_heads = (int32_t)Hk;
  p->head_dim = (int32_t)D;
  p->page_size = (int32_t)P;
  p->num_pages = (int32_t)kc->size(0);
  return true;
}

template <class Args>
bool block_table(const at::Tensor* bt, const at::Tensor* seq_lens, int64_t batch, Args* p) {
  if (!index_ready(bt) || !index_ready(seq_lens) || bt->size(0) != batch ||
      seq_lens->size(0) != batch || !fits(batch) || !fits(bt->size(1) * p->page_size))
    return false;
  p->block_table = bt->data_ptr<int32_t>();
  p->seq_lens = seq_lens->data_ptr<int32_t>();
  p->block_table_stride = bt->size(1);
  p->max_blocks = (int32_t)bt->size(1);
  p->batch = (int32_t)batch;
  return true;
}

// decode(q, k_cache, v_cache, block_table, seq_lens, block_size, num_kv_heads, scale,
//        device, stream) -> out | status | None
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Call c;
    fa_decode_args p = {};
    if (n != 10 || !call_of(a[8], a[9], &c)) return none();
    const at::Tensor* q = plain(a[0], c, 3);
    if (!caches(q, plain(a[1], c, 4), plain(a[2], c, 4), a[5], a[6], a[7], &p) ||
        !block_table(plain(a[3], c, 2), plain(a[4], c, 1), q->size(0), &p))
      return none();
    at::Tensor out;
    int status = FA_E_INVALID;
    {
      NoGil no_gil;
      out = at::empty(q->sizes(), q->options().requires_grad(false));
      p.out = out.data_ptr();
      set_strides(p.o_stride, out);
      p.max_seq_len = p.max_blocks * p.page_size;
      if (const size_t bytes = lib.decode_workspace(&p)) {
        at::Tensor ws = at::empty({(int64_t)bytes}, out.options().dtype(at::kByte));
        status = lib.decode(&p, ws.data_ptr(), bytes, c.stream);
      }
    }
    if (status != FA_OK) return PyLong_FromLong(status);
    return THPVariable_Wrap(out);
  });
}

// paged_forward(q, k_cache, v_cache, block_table, seq_lens, query_start_loc,
//               prefix_kv_lens, block_size, num_kv_heads, scale, causal, window_q, window_k,
//               device, stream) -> (out, lse) | status | None
PyObject* paged_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Call c;
    fa_paged_args p = {};
    int64_t wq, wk;
    if (n != 15 || !call_of(a[13], a[14], &c) || !integer(a[11], &wq) || !integer(a[12], &wk) ||
        !fits(wq) || !fits(wk) || wq < INT_MIN || wk < INT_MIN)
      return none();
    const at::Tensor *q = plain(a[0], c, 3), *bt = plain(a[3], c, 2);
    if (!bt || !caches(q, plain(a[1], c, 4), plain(a[2], c, 4), a[7], a[8], a[9], &p) ||
        !block_table(bt, plain(a[4], c, 1), bt->size(0), &p) || !q->is_contiguous())
      return none();
    const at::Tensor *qsl = plain(a[5], c, 1), *prefix = plain(a[6], c, 1);
    if (!index_ready(qsl) || !index_ready(prefix) || qsl->size(0) != bt->size(0) + 1 ||
        prefix->size(0) != bt->size(0) || !fits(q->size(0)))
      return none();
    const bool causal = a[10] == Py_True;
    at::Tensor out, lse;
    int status;
    {
      NoGil no_gil;
      out = at::empty(q->sizes(), q->options().requires_grad(false));
      lse = at::empty({q->size(1), q->size(0)}, out.options().dtype(at::kFloat));
      p.out = out.data_ptr();
      p.lse = lse.data_ptr<float>();
      set_strides(p.o_stride, out);
      p.query_start_loc = qsl->data_ptr<int32_t>();
      p.prefix_kv_lens = prefix->data_ptr<int32_t>();
      p.num_tokens = (int32_t)q->size(0);
      p.causal = causal;
      p.window_q = (int32_t)wq;
      p.window_k = (int32_t)wk;
      status = lib.paged_splits(&p);
      if (status > 0) {
        const int splits = status;
        const size_t bytes = lib.paged_workspace(&p, splits);
        at::Tensor ws;
        if (bytes) ws = at::empty({(int64_t)bytes}, out.options().dtype(at::kByte));
        status = lib.paged(&p, splits, bytes ? ws.data_ptr() : nullptr, bytes, c.stream);
      }
    }
    if (status != FA_OK) return PyLong_FromLong(status);
    return Py_BuildValue("NN", THPVariable_Wrap(out), THPVariable_Wrap(lse));
  });
}

// cache_write(key, value, key_cache, value_cache, slot_mapping, device, stream)
//   -> 0 | status | None
PyObject* cache_write(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Call c;
    fa_cache_write_args p = {};
    if (n != 7 || !call_of(a[5], a[6], &c)) return none();
    const at::Tensor *k = plain(a[0], c, 3), *v = plain(a[1], c, 3), *kc = plain(a[2], c, 4),
                     *vc = plain(a[3], c, 4), *slots = plain(a[4], c, 1);
    if (!k || !v || !kc || !vc || !slots || !half_code(*k, &p.dtype) ||
        v->scalar_type() != k->scalar_type() || kc->scalar_type() != k->scalar_type() ||
        vc->scalar_type() != k->scalar_type() || k->sizes() != v->sizes() ||
        kc->sizes() != vc->sizes() || kc->size(2) != k->size(1) || kc->size(3) != k->size(2) ||
        slots->scalar_type() != at::kLong || !slots->is_contiguous() ||
        slots->size(0) != k->size(0) || k->size(2) % 8 != 0 || k->size(2) > 1024 ||
        !rows_ready(*k) || !rows_ready(*v) || !rows_ready(*kc) || !rows_ready(*vc) ||
        !fits(k->size(0)) || !fits(k->size(1)) || !fits(kc->size(0)) || !fits(kc->size(1)))
      return none();
    p.key = k->data_ptr();
    p.value = v->data_ptr();
    p.k_cache = kc->data_ptr();
    p.v_cache = vc->data_ptr();
    p.slot_mapping = slots->data_ptr<int64_t>();
    set_strides(p.key_stride, *k);
    set_strides(p.value_stride, *v);
    set_strides(p.k_stride, *kc);
    set_strides(p.v_stride, *vc);
    p.num_tokens = (int32_t)k->size(0);
    p.num_kv_heads = (int32_t)k->size(1);
    p.head_dim = (int32_t)k->size(2);
    p.page_size = (int32_t)kc->size(1);
    p.num_pages = (int32_t)kc->size(0);
    int status;
    {
      NoGil no_gil;
      status = lib.cache_write(&p, c.stream);
    }
    return PyLong_FromLong(status);
  });
}

// bind(fa_fwd, fa_decode_workspace_bytes, fa_paged_decode, fa_paged_prefill_num_splits,
//      fa_paged_prefill_splitkv_workspace_bytes, fa_paged_prefill_splitkv,
//      fa_reshape_and_cache): the library's entry points, as addresses.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  void* f[7];
  if (n != 7) {
    PyErr_SetString(PyExc_TypeError, "bind takes seven addresses");
    return nullptr;
  }
  for (int i = 0; i < 7; ++i) {
    f[i] = PyLong_AsVoidPtr(a[i]);
    if (PyErr_Occurred()) return nullptr;
  }
  lib = {reinterpret_cast<decltype(lib.fwd)>(f[0]),
         reinterpret_cast<decltype(lib.decode_workspace)>(f[1]),
         reinterpret_cast<decltype(lib.decode)>(f[2]),
         reinterpret_cast<decltype(lib.paged_splits)>(f[3]),
         reinterpret_cast<decltype(lib.paged_workspace)>(f[4]),
         reinterpret_cast<decltype(lib.paged)>(f[5]),
         reinterpret_cast<decltype(lib.cache_write)>(f[6])};
  Py_RETURN_NONE;
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyMethodDef method(const char* name) {
  return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)), METH_FASTCALL,
          nullptr};
}

PyMethodDef methods[] = {method<bind>("bind"),
                         method<dense_forward>("dense_forward"),
                         method<decode>("decode"),
                         method<paged_forward>("paged_forward"),
                         method<cache_write>("cache_write"),
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_fa_torch", nullptr, -1, methods};

}  // namespace

// FA_TORCH_VERSION: the torch whose headers this was compiled against; another
// one's tensors may be laid out differently, so the loader compares it.
PyMODINIT_FUNC PyInit__fa_torch(void) {
  PyObject* m = PyModule_Create(&module_def);
  if (m && PyModule_AddStringConstant(m, "torch_version", FA_TORCH_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
