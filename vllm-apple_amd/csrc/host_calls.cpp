// Native host path of the functional wrappers (vllm_apple_amd/kernels.py and
// backend.py): each function reads the tensors' metadata, makes the same
// checks as its Python wrapper and calls the C ABI, in 1 to 3 us instead of 10
// to 40 (one decode step through the vLLM backend: 43 us of Python for two
// launches before).  A function returns
//   True          the work is enqueued;
//   False         something is not the plain accepted case: nothing is
//                 enqueued that the wrapper's own path does not repeat, and
//                 the wrapper goes on from its first line, which converts,
//                 or raises the same error as ever;
//   an int n > 0  nothing is enqueued and n bytes of workspace are needed.
// No state is kept between calls.  The library's entry points are looked up in
// the handle that _lib.py loaded (bind), so both use one library.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_variable.h>

#include <initializer_list>

#include "vllm_apple_amd.h"

namespace {

#define VAA_FUNCS(X)                                                                      \
  X(vaa_kv_write_slots) X(vaa_paged_attention_decode)                                     \
  X(vaa_paged_attention_decode_workspace_size) X(vaa_paged_attention_prefill)             \
  X(vaa_paged_attention_prefill_split) X(vaa_paged_attention_prefill_tiles)               \
  X(vaa_paged_attention_prefill_workspace_size) X(vaa_prefill_step)                       \
  X(vaa_prefill_step_workspace_size) X(vaa_rmsnorm) X(vaa_add_rmsnorm) X(vaa_silu_mul)    \
  X(vaa_qkv_epilogue) X(vaa_topk_logits) X(vaa_topk_workspace_size)                       \
  X(vaa_gate_up_silu_split) X(vaa_gate_up_silu_workspace_size) X(vaa_linear)        \
  X(vaa_linear_workspace_size) X(vaa_attention_no_cache)                            \
  X(vaa_attention_no_cache_workspace_size)
#define VAA_DECL(f) decltype(&::f) p_##f = nullptr;
VAA_FUNCS(VAA_DECL)
#undef VAA_DECL

using at::Tensor;

// args[i] as a tensor, or null for None (or anything else).
const Tensor* ten(PyObject* o) {
  return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr;
}
bool none_or_ten(PyObject* o) { return o == Py_None || THPVariable_Check(o); }

// As Tensor.data_ptr(): a lazy clone that still shares its memory gets its own
// first, also where the kernel only reads (two views of one storage then agree).
void* ptr(const Tensor& t) { return t.mutable_data_ptr(); }
uint16_t* p16(const Tensor& t) { return static_cast<uint16_t*>(ptr(t)); }

bool on_gpu(const Tensor& t) { return t.is_cuda() && t.layout() == at::kStrided; }
// Whether the tensors (null: absent) are all on one device.  A kernel given
// another device's pointers would read them over the peer mapping or fault.
bool one_device(std::initializer_list<const Tensor*> ts) {
  const Tensor* first = nullptr;
  for (const Tensor* t : ts) {
    if (!t) continue;
    if (!first) first = t;
    if (t->device() != first->device()) return false;
  }
  return true;
}
// Whether ws is a workspace of `need` bytes on the tensor's device.
bool room(const Tensor* ws, size_t need, const Tensor& like) {
  return ws && on_gpu(*ws) && ws->device() == like.device() && ws->nbytes() >= need;
}

// VAA_DTYPE_* of a GPU tensor of the two 16-bit types, else -1.
int dt16(const Tensor& t) {
  if (!on_gpu(t)) return -1;
  if (t.scalar_type() == at::kHalf) return VAA_DTYPE_F16;
  if (t.scalar_type() == at::kBFloat16) return VAA_DTYPE_BF16;
  return -1;
}
bool is_i32(const Tensor& t) {
  return on_gpu(t) && t.scalar_type() == at::kInt && t.is_contiguous();
}
// A slot mapping of at least n entries: VAA_INDEX_*, else -1.
int slot_type(const Tensor& t, int64_t n) {
  if (!on_gpu(t) || !t.is_contiguous() || t.numel() < n) return -1;
  if (t.scalar_type() == at::kLong) return VAA_INDEX_I64;
  if (t.scalar_type() == at::kInt) return VAA_INDEX_I32;
  return -1;
}
// [tokens, heads, head_size] with a contiguous last dim.
bool rows3(const Tensor& t) { return t.dim() == 3 && t.stride(2) == 1; }
bool small(int64_t v) { return v >= 0 && v < (int64_t{1} << 31); }

// Cache fields of p from one K and one V cache tensor of four dims (kernel
// layout [nb, KV, bs, D], vLLM layout [nb, bs, KV, D]); false when they are not
// what the wrappers take.
bool cache4(const Tensor& k, const Tensor& v, bool vllm, vaa_attn_params* p) {
  if (k.dim() != 4 || v.dim() != 4 || k.stride(3) != 1 || v.stride(3) != 1 ||
      k.sizes() != v.sizes())
    return false;
  const int h = vllm ? 2 : 1, t = vllm ? 1 : 2;
  if (!small(k.size(h)) || !small(k.size(t)) || !small(k.size(3)) || k.size(h) == 0) return false;
  p->num_blocks = k.size(0);
  p->num_kv_heads = k.size(h);
  p->block_size = k.size(t);
  p->head_size = k.size(3);
  p->k_stride_block = k.stride(0);
  p->k_stride_head = k.stride(h);
  p->k_stride_token = k.stride(t);
  p->v_stride_block = v.stride(0);
  p->v_stride_head = v.stride(h);
  p->v_stride_token = v.stride(t);
  return true;
}
bool heads(int64_t H, vaa_attn_params* p) {
  if (!small(H) || H == 0 || H % p->num_kv_heads) return false;
  p->num_query_heads = H;
  p->queries_per_kv = H / p->num_kv_heads;
  return true;
}
bool same_rows(const Tensor& a, const Tensor& b) {
  return a.sizes() == b.sizes() && a.strides() == b.strides();
}

// Entry points are called without the interpreter lock, as by ctypes: a launch
// into a full queue blocks until the GPU takes one, and other Python threads run
// meanwhile.  The arguments are evaluated before, with the lock; the tensors live
// as long as the caller's argument list.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename... P, typename... A>
int launch(int (*f)(P...), A... args) {
  Unlocked unlocked;
  return f(args...);
}

PyObject* yes(int status) {
  if (status != VAA_OK) Py_RETURN_FALSE;  // the wrapper repeats the call and raises
  Py_RETURN_TRUE;
}

// Arguments by position; any conversion error or exception falls back.
struct Args {
  PyObject* const* a;
  int64_t i(int k) const {
    const long long v = PyLong_AsLongLong(a[k]);
    if (v == -1 && PyErr_Occurred()) throw 0;
    return v;
  }
  double f(int k) const {
    const double v = PyFloat_AsDouble(a[k]);
    if (v == -1.0 && PyErr_Occurred()) throw 0;
    return v;
  }
  bool b(int k) const { return a[k] == Py_True; }
  void* s(int k) const { return reinterpret_cast<void*>(static_cast<intptr_t>(i(k))); }
  const Tensor* t(int k) const { return ten(a[k]); }
};

template <int N, PyObject* (*F)(const Args&)>
PyObject* guarded(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
    return nullptr;
  }
  if (!p_vaa_rmsnorm) Py_RETURN_FALSE;  // not bound
  try {
    return F(Args{args});
  } catch (...) {
    PyErr_Clear();
    Py_RETURN_FALSE;
  }
}

// ------------------------------------------------------------ layer ops --

// (x, w, residual or None, out, eps, stream, add)
PyObject* norm(const Args& a) {
  const Tensor *x = a.t(0), *w = a.t(1), *r = a.t(2), *o = a.t(3);
  const bool add = a.b(6);
  if (!x || !w || !o || !none_or_ten(a.a[2]) || (add && !r) || !one_device({x, w, r, o}))
    Py_RETURN_FALSE;
  const int dt = dt16(*x);
  if (dt < 0 || dt16(*w) != dt || dt16(*o) != dt || (r && dt16(*r) != dt)) Py_RETURN_FALSE;
  if (x->dim() != 2 || x->stride(1) != 1 || !w->is_contiguous() || w->numel() != x->size(1) ||
      o->sizes() != x->sizes() || o->stride(1) != 1 ||
      (r && (r->sizes() != x->sizes() || r->stride(1) != 1)) || !small(x->size(0)) ||
      !small(x->size(1)))
    Py_RETURN_FALSE;
  const float eps = static_cast<float>(a.f(4));
  if (add)
    return yes(launch(p_vaa_add_rmsnorm, p16(*x), p16(*r), p16(*w), p16(*o), x->size(0), x->size(1),
                      x->stride(0), r->stride(0), o->stride(0), eps, dt, a.s(5)));
  return yes(launch(p_vaa_rmsnorm, p16(*x), p16(*o), p16(*w), r ? p16(*r) : nullptr, x->size(0),
                    x->size(1), x->stride(0), o->stride(0), r ? r->stride(0) : 0, eps, dt, a.s(5)));
}

// (gate, up, out, stream): contiguous tensors
PyObject* silu(const Args& a) {
  const Tensor *g = a.t(0), *u = a.t(1), *o = a.t(2);
  if (!g || !u || !o || !one_device({g, u, o})) Py_RETURN_FALSE;
  const int dt = dt16(*g);
  if (dt < 0 || dt16(*u) != dt || dt16(*o) != dt || g->sizes() != u->sizes() ||
      o->sizes() != g->sizes() || !g->is_contiguous() || !u->is_contiguous() ||
      !o->is_contiguous())
    Py_RETURN_FALSE;
  return yes(launch(p_vaa_silu_mul, p16(*g), p16(*u), p16(*o), g->numel(), dt, a.s(3)));
}

// (q, k, v, pos, cos, sin, slots, k_cache, v_cache, bias or None, rot, vllm, stream)
PyObject* epilogue(const Args& a) {
  const Tensor *q = a.t(0), *k = a.t(1), *v = a.t(2), *pos = a.t(3), *c = a.t(4), *s = a.t(5),
               *sl = a.t(6), *kc = a.t(7), *vc = a.t(8), *b = a.t(9);
  if (!q || !k || !v || !pos || !c || !s || !sl || !kc || !vc || !none_or_ten(a.a[9]) ||
      !one_device({q, k, v, pos, c, s, sl, kc, vc, b}))
    Py_RETURN_FALSE;
  const int dt = dt16(*q);
  if (dt < 0 || dt16(*k) != dt || dt16(*v) != dt || dt16(*kc) != dt || dt16(*vc) != dt ||
      (b && dt16(*b) != dt))
    Py_RETURN_FALSE;
  for (const Tensor* t : {q, k, v})
    if (!rows3(*t) || t->stride(1) != t->size(2)) Py_RETURN_FALSE;
  if (!same_rows(*k, *v)) Py_RETURN_FALSE;
  const int64_t T = q->size(0), H = q->size(1), D = q->size(2), KV = k->size(1), rot = a.i(10);
  vaa_attn_params p{};
  if (k->size(0) != T || k->size(2) != D || !small(T) || !is_i32(*pos) || pos->numel() < T ||
      slot_type(*sl, T) < 0 || !on_gpu(*c) || !on_gpu(*s) || c->scalar_type() != at::kFloat ||
      s->scalar_type() != at::kFloat || c->dim() != 2 || c->sizes() != s->sizes() ||
      rot <= 0 || c->size(1) != rot / 2 || !c->is_contiguous() || !s->is_contiguous() ||
      !small(c->size(0)) || !small(rot) ||
      (b && (b->dim() != 1 || b->numel() != (H + 2 * KV) * D || !b->is_contiguous())) ||
      !cache4(*kc, *vc, a.b(11), &p) || !heads(H, &p) || KV != p.num_kv_heads ||
      D != p.head_size)
    Py_RETURN_FALSE;
  p.dtype = dt;
  p.scale = 1.f;
  p.q_stride_token = q->stride(0);
  p.q_stride_head = q->stride(1);
  p.new_kv_stride_token = k->stride(0);
  p.new_kv_stride_head = k->stride(1);
  return yes(launch(p_vaa_qkv_epilogue, &p, p16(*q), p16(*k), p16(*v), b ? p16(*b) : nullptr,
                    static_cast<float*>(ptr(*c)), static_cast<float*>(ptr(*s)), rot, c->size(0),
                    static_cast<int32_t*>(ptr(*pos)), ptr(*sl), slot_type(*sl, T), p16(*kc),
                    p16(*vc), T, a.s(12)));
}

// (logits, k, indices, values, workspace or None, stream)
PyObject* topk(const Args& a) {
  const Tensor *x = a.t(0), *idx = a.t(2), *val = a.t(3), *ws = a.t(4);
  if (!x || !idx || !val || !none_or_ten(a.a[4]) || !one_device({x, idx, val, ws}))
    Py_RETURN_FALSE;
  const int64_t k = a.i(1);
  if (dt16(*x) < 0 || dt16(*val) != dt16(*x) || x->dim() != 2 || x->stride(1) != 1 ||
      !on_gpu(*idx) || idx->scalar_type() != at::kInt || idx->dim() != 2 || val->dim() != 2 ||
      idx->strides() != val->strides() || idx->stride(1) != 1 || idx->sizes() != val->sizes() ||
      idx->size(0) != x->size(0) || idx->size(1) != k || k < 1 || k > 256 || k > x->size(1) ||
      !small(x->size(0)) || !small(x->size(1)))
    Py_RETURN_FALSE;
  size_t need = 0;
  if (p_vaa_topk_workspace_size(x->size(0), x->size(1), k, &need) != VAA_OK) Py_RETURN_FALSE;
  if (need && !room(ws, need, *x)) return PyLong_FromSize_t(need);
  return yes(launch(p_vaa_topk_logits, p16(*x), x->size(0), x->size(1), x->stride(0), k,
                    static_cast<int32_t*>(ptr(*idx)), p16(*val), idx->stride(0),
                    ws ? ptr(*ws) : nullptr, ws ? ws->nbytes() : 0, a.s(5)));
}

bool mat16(const Tensor& t, int dt) {
  return dt16(t) == dt && t.dim() == 2 && t.stride(1) == 1 && small(t.size(0)) &&
         small(t.size(1));
}

// (x, gate weight or fused gate/up weight, up weight or None, out, workspace or
// None, stream)
PyObject* gate_up(const Args& a) {
  const Tensor *x = a.t(0), *g = a.t(1), *u = a.t(2), *o = a.t(3), *ws = a.t(4);
  if (!x || !g || !o || !none_or_ten(a.a[2]) || !none_or_ten(a.a[4]) ||
      !one_device({x, g, u, o}))
    Py_RETURN_FALSE;
  const int dt = dt16(*x);
  if (dt < 0 || !mat16(*x, dt) || !mat16(*g, dt) || !mat16(*o, dt) || (u && !mat16(*u, dt)))
    Py_RETURN_FALSE;
  const int64_t T = x->size(0), H = x->size(1);
  int64_t I = g->size(0);
  const uint16_t* up;
  if (u) {
    if (u->sizes() != g->sizes() || u->stride(0) != g->stride(0)) Py_RETURN_FALSE;
    up = p16(*u);
  } else {
    if (I % 2) Py_RETURN_FALSE;
    I /= 2;
    up = p16(*g) + I * g->stride(0);
  }
  if (g->size(1) != H || o->size(0) != T || o->size(1) != I) Py_RETURN_FALSE;
  const size_t need = p_vaa_gate_up_silu_workspace_size(T, H, I);
  if (need && !room(ws, need, *x)) return PyLong_FromSize_t(need);
  return yes(launch(p_vaa_gate_up_silu_split, p16(*x), x->stride(0), p16(*g), up, g->stride(0),
                    p16(*o), o->stride(0), T, H, I, dt, ws ? ptr(*ws) : nullptr,
                    ws ? ws->nbytes() : 0, a.s(5)));
}

// Whether torch.matmul(out=) would do nothing but the product on these: no
// gradient to record or refuse (reverse or forward mode), no tensor whose
// operations Python or a transform implements, no dispatch mode that would see
// the call.
bool plain_matmul(std::initializer_list<const Tensor*> ts) {
  if (c10::impl::dispatch_mode_enabled()) return false;
  const bool grad = c10::GradMode::is_enabled();
  for (const Tensor* t : ts)
    if ((grad && t->requires_grad()) || t->_fw_grad(0).defined() ||
        t->key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python,
                                                  c10::DispatchKey::FuncTorchBatched,
                                                  c10::DispatchKey::FuncTorchGradWrapper})))
      return false;
  return true;
}

// (x, weight, out, workspace or None, stream); what linear_ok accepts, in a call
// that stands in for torch.matmul(out=): like it, it counts as a write to out.
PyObject* linear(const Args& a) {
  const Tensor *x = a.t(0), *w = a.t(1), *o = a.t(2), *ws = a.t(3);
  if (!x || !w || !o || !none_or_ten(a.a[3]) || !one_device({x, w, o}) ||
      !plain_matmul({x, w, o}))
    Py_RETURN_FALSE;
  const int dt = dt16(*x);
  if (dt < 0 || !mat16(*x, dt) || !mat16(*w, dt) || !mat16(*o, dt)) Py_RETURN_FALSE;
  const int64_t T = x->size(0), K = x->size(1), N = w->size(0);
  if (w->size(1) != K || o->size(0) != T || o->size(1) != N) Py_RETURN_FALSE;
  const size_t need = p_vaa_linear_workspace_size(T, K, N);
  if (!need) Py_RETURN_FALSE;
  if (!room(ws, need, *x)) return PyLong_FromSize_t(need);
  void* const stream = a.s(4);
  if (launch(p_vaa_linear, p16(*x), x->stride(0), p16(*w), w->stride(0), p16(*o), o->stride(0), T,
             K, N, dt, ptr(*ws), ws->nbytes(), stream) != VAA_OK)
    Py_RETURN_FALSE;
  if (!o->is_inference()) o->unsafeGetTensorImpl()->bump_version();
  Py_RETURN_TRUE;
}

// ------------------------------------------------------------ attention --

// Fields and slot type of a write of K/V rows key/value[:n]; false: fall back.
bool write_params(const Tensor& k, const Tensor& v, const Tensor& slots, int64_t n,
                  vaa_attn_params* p, int* it) {
  *it = slot_type(slots, n);
  if (*it < 0 || !rows3(k) || !same_rows(k, v) || k.size(0) < n || k.size(1) != p->num_kv_heads ||
      k.size(2) != p->head_size)
    return false;
  p->num_query_heads = p->num_kv_heads;
  p->queries_per_kv = 1;
  p->scale = 1.f;
  p->new_kv_stride_token = k.stride(0);
  p->new_kv_stride_head = k.stride(1);
  return true;
}

// (key, value, key_cache, value_cache, slots, vllm, stream)
PyObject* kv_write(const Args& a) {
  const Tensor *k = a.t(0), *v = a.t(1), *kc = a.t(2), *vc = a.t(3), *sl = a.t(4);
  if (!k || !v || !kc || !vc || !sl || !one_device({k, v, kc, vc, sl})) Py_RETURN_FALSE;
  const int dt = dt16(*k);
  vaa_attn_params p{};
  if (dt < 0 || dt16(*v) != dt || dt16(*kc) != dt || dt16(*vc) != dt || k->dim() != 3 ||
      !small(k->size(0)) || !cache4(*kc, *vc, a.b(5), &p))
    Py_RETURN_FALSE;
  p.dtype = dt;
  int it;
  if (!write_params(*k, *v, *sl, k->size(0), &p, &it)) Py_RETURN_FALSE;
  return yes(launch(p_vaa_kv_write_slots, &p, p16(*kc), p16(*vc), ptr(*sl), it, p16(*k), p16(*v),
                    k->size(0), a.s(6)));
}

// Fills the query, output, table and length fields of a decode over the first
// n sequences; false: fall back.
bool decode_params(const Tensor& q, const Tensor& o, const Tensor& bt, const Tensor& sl, int64_t n,
                   double scale, int64_t max_len, int64_t part, vaa_attn_params* p) {
  if (!rows3(q) || !rows3(o) || q.size(0) < n || o.size(0) < n || q.size(2) != p->head_size ||
      !heads(q.size(1), p) || !is_i32(bt) || bt.dim() != 2 || bt.size(0) < n || !is_i32(sl) ||
      sl.numel() < n || !small(n) || !small(bt.size(1)) || !small(max_len) ||
      part != static_cast<int32_t>(part))
    return false;
  p->scale = static_cast<float>(scale);
  p->num_seqs = n;
  p->max_seq_len = max_len;
  p->max_blocks_per_seq = bt.size(1);
  p->partition_size = part;
  p->q_stride_token = q.stride(0);
  p->q_stride_head = q.stride(1);
  p->o_stride_token = o.stride(0);
  p->o_stride_head = o.stride(1);
  return true;
}

// (query, key_cache, value_cache, block_table, seq_lens, output, new_keys or
// None, new_values or None, vllm, scale, max_seq_len, partition_size,
// workspace or None, stream)
PyObject* decode(const Args& a) {
  const Tensor *q = a.t(0), *kc = a.t(1), *vc = a.t(2), *bt = a.t(3), *sl = a.t(4), *o = a.t(5),
               *nk = a.t(6), *nv = a.t(7), *ws = a.t(12);
  if (!q || !kc || !vc || !bt || !sl || !o || !none_or_ten(a.a[6]) || !none_or_ten(a.a[7]) ||
      !none_or_ten(a.a[12]) || !nk != !nv || !one_device({q, kc, vc, bt, sl, o, nk, nv}))
    Py_RETURN_FALSE;
  const int dt = dt16(*q);
  vaa_attn_params p{};
  const int64_t n = sl->numel();
  if (dt < 0 || dt16(*kc) != dt || dt16(*vc) != dt || dt16(*o) != dt ||
      !cache4(*kc, *vc, a.b(8), &p) ||
      !decode_params(*q, *o, *bt, *sl, n, a.f(9), a.i(10), a.i(11), &p))
    Py_RETURN_FALSE;
  if (nk) {
    // The wrapper checks neither the rows' count nor their shape; only the
    // plain case is taken here.
    if (dt16(*nk) != dt || dt16(*nv) != dt || !rows3(*nk) || !same_rows(*nk, *nv) ||
        nk->size(0) < n || nk->size(1) != p.num_kv_heads || nk->size(2) != p.head_size)
      Py_RETURN_FALSE;
    p.new_kv_stride_token = nk->stride(0);
    p.new_kv_stride_head = nk->stride(1);
  }
  p.dtype = dt;
  const size_t need = p_vaa_paged_attention_decode_workspace_size(&p, nullptr);
  if (need && !room(ws, need, *q)) return PyLong_FromSize_t(need);
  return yes(launch(p_vaa_paged_attention_decode, &p, p16(*q), p16(*kc), p16(*vc),
                    static_cast<int32_t*>(ptr(*bt)), static_cast<int32_t*>(ptr(*sl)), p16(*o),
                    nk ? p16(*nk) : nullptr, nv ? p16(*nv) : nullptr, need ? ptr(*ws) : nullptr,
                    need ? ws->nbytes() : 0, a.s(13)));
}

// Cache fields of p from vLLM's [2, nb, bs, KV, D] tensor.
bool cache5(const Tensor& c, vaa_attn_params* p, uint16_t** kc, uint16_t** vc) {
  if (c.dim() != 5 || c.size(0) != 2 || c.stride(4) != 1 || !small(c.size(2)) ||
      !small(c.size(3)) || !small(c.size(4)) || c.size(3) == 0)
    return false;
  p->num_blocks = c.size(1);
  p->block_size = c.size(2);
  p->num_kv_heads = c.size(3);
  p->head_size = c.size(4);
  p->k_stride_block = p->v_stride_block = c.stride(1);
  p->k_stride_token = p->v_stride_token = c.stride(2);
  p->k_stride_head = p->v_stride_head = c.stride(3);
  *kc = p16(c);
  *vc = *kc + c.stride(0);
  return true;
}

// One decode step of the backend: the K/V rows of the first n tokens (with
// write) go to the cache, then n sequences attend.
// (query, key, value, kv_cache, output, block_table, seq_lens, slots, n, write,
//  head_size, scale, max_seq_len, partition_size, workspace or None, stream)
PyObject* step_decode(const Args& a) {
  const Tensor *q = a.t(0), *k = a.t(1), *v = a.t(2), *c = a.t(3), *o = a.t(4), *bt = a.t(5),
               *sl = a.t(6), *slots = a.t(7), *ws = a.t(14);
  const bool write = a.b(9);
  if (!q || !c || !o || !bt || !sl || (write && (!k || !v || !slots)) || !none_or_ten(a.a[14]) ||
      !one_device({q, c, o, bt, sl}) || (write && !one_device({q, k, v, slots})))
    Py_RETURN_FALSE;
  const int dt = dt16(*q);
  const int64_t n = a.i(8);
  vaa_attn_params p{};
  uint16_t *kc, *vc;
  if (dt < 0 || n <= 0 || dt16(*c) != dt || dt16(*o) != dt ||
      (write && (dt16(*k) != dt || dt16(*v) != dt)) || !cache5(*c, &p, &kc, &vc) ||
      p.head_size != a.i(10) ||
      !decode_params(*q, *o, *bt, *sl, n, a.f(11), a.i(12), a.i(13), &p))
    Py_RETURN_FALSE;
  p.dtype = dt;
  const size_t need = p_vaa_paged_attention_decode_workspace_size(&p, nullptr);
  if (need && !room(ws, need, *q)) return PyLong_FromSize_t(need);
  vaa_attn_params wp = p;
  int it = 0;
  if (write && !write_params(*k, *v, *slots, n, &wp, &it)) Py_RETURN_FALSE;
  const uint16_t *kp = write ? p16(*k) : nullptr, *vp = write ? p16(*v) : nullptr;
  const void* slp = write ? ptr(*slots) : nullptr;
  auto *btp = static_cast<int32_t*>(ptr(*bt)), *lp = static_cast<int32_t*>(ptr(*sl));
  uint16_t *qp = p16(*q), *op = p16(*o);
  void *wsp = need ? ptr(*ws) : nullptr, *stream = a.s(15);
  const size_t ws_bytes = need ? ws->nbytes() : 0;
  int st = VAA_OK;
  {
    Unlocked unlocked;
    if (write) st = p_vaa_kv_write_slots(&wp, kc, vc, slp, it, kp, vp, n, stream);
    if (st == VAA_OK)
      st = p_vaa_paged_attention_decode(&p, qp, kc, vc, btp, lp, op, nullptr, nullptr, wsp,
                                        ws_bytes, stream);
  }
  return yes(st);
}

// Fields of an unsplit prefill of tokens [0, n).
bool prefill_params(const Tensor& q, const Tensor& o, const Tensor& bt, int64_t n, double scale,
                    vaa_attn_params* p) {
  if (!rows3(q) || !rows3(o) || q.size(0) < n || o.size(0) < n || q.size(2) != p->head_size ||
      o.size(1) != q.size(1) || o.size(2) != q.size(2) || !heads(q.size(1), p) || !is_i32(bt) ||
      bt.dim() != 2 || !small(bt.size(0)) || !small(bt.size(1)) || !small(n))
    return false;
  p->scale = static_cast<float>(scale);
  p->num_seqs = bt.size(0);
  p->max_blocks_per_seq = bt.size(1);
  p->q_stride_token = q.stride(0);
  p->q_stride_head = q.stride(1);
  p->o_stride_token = o.stride(0);
  p->o_stride_head = o.stride(1);
  return true;
}

// One prefill-only step of the backend: K/V rows, indices (and, with own_tiles,
// query tiles of one sequence each) and the unsplit prefill of the first n tokens.
// (query, key, value, kv_cache, output, block_table, seq_lens, slots,
//  query_start_loc, n, write, head_size, scale, own_tiles, workspace or None,
//  stream)
PyObject* step_prefill(const Args& a) {
  const Tensor *q = a.t(0), *k = a.t(1), *v = a.t(2), *c = a.t(3), *o = a.t(4), *bt = a.t(5),
               *sl = a.t(6), *slots = a.t(7), *qsl = a.t(8), *ws = a.t(14);
  const bool write = a.b(10);
  if (!q || !c || !o || !bt || !sl || !qsl || (write && (!k || !v || !slots)) ||
      !none_or_ten(a.a[14]) || !one_device({q, c, o, bt, sl, qsl}) ||
      (write && !one_device({q, k, v, slots})))
    Py_RETURN_FALSE;
  const int dt = dt16(*q);
  const int64_t n = a.i(9);
  vaa_attn_params p{};
  uint16_t *kc, *vc;
  if (dt < 0 || n <= 0 || dt16(*c) != dt || dt16(*o) != dt ||
      (write && (dt16(*k) != dt || dt16(*v) != dt)) || !cache5(*c, &p, &kc, &vc) ||
      p.head_size != a.i(11) || !prefill_params(*q, *o, *bt, n, a.f(12), &p) || !is_i32(*qsl) ||
      !is_i32(*sl) || qsl->numel() < 1 || !small(qsl->numel()) ||
      sl->numel() < qsl->numel() - 1)
    Py_RETURN_FALSE;
  p.dtype = dt;
  int it = 0;
  if (write) {
    it = slot_type(*slots, n);
    if (it < 0 || !rows3(*k) || !same_rows(*k, *v) || k->size(0) < n ||
        k->size(1) != p.num_kv_heads || k->size(2) != p.head_size)
      Py_RETURN_FALSE;
    p.new_kv_stride_token = k->stride(0);
    p.new_kv_stride_head = k->stride(1);
  }
  const int S = static_cast<int>(qsl->numel() - 1);
  const size_t need = p_vaa_prefill_step_workspace_size(&p, n, S);
  if (!room(ws, need, *q)) return PyLong_FromSize_t(need);
  return yes(launch(p_vaa_prefill_step, &p, p16(*q), kc, vc, static_cast<int32_t*>(ptr(*bt)),
                    static_cast<int32_t*>(ptr(*sl)), static_cast<int32_t*>(ptr(*qsl)), S,
                    write ? p16(*k) : nullptr, write ? p16(*v) : nullptr,
                    write ? ptr(*slots) : nullptr, it, p16(*o), n, a.b(13), ptr(*ws), ws->nbytes(),
                    a.s(15)));
}

// (query, key_cache, value_cache, block_table, token_to_seq, positions, output,
//  vllm, scale, tiles or None, split_keys, max_seq_len, workspace or None, stream)
PyObject* prefill(const Args& a) {
  const Tensor *q = a.t(0), *kc = a.t(1), *vc = a.t(2), *bt = a.t(3), *tok = a.t(4),
               *pos = a.t(5), *o = a.t(6), *tiles = a.t(9), *ws = a.t(12);
  if (!q || !kc || !vc || !bt || !tok || !pos || !o || !none_or_ten(a.a[9]) ||
      !none_or_ten(a.a[12]) || !one_device({q, kc, vc, bt, tok, pos, o, tiles}))
    Py_RETURN_FALSE;
  const int dt = dt16(*q);
  const int64_t split = a.i(10), max_len = a.i(11);
  vaa_attn_params p{};
  if (dt < 0 || dt16(*kc) != dt || dt16(*vc) != dt || dt16(*o) != dt || q->dim() != 3 ||
      !cache4(*kc, *vc, a.b(7), &p) || !prefill_params(*q, *o, *bt, q->size(0), a.f(8), &p) ||
      !is_i32(*tok) || !is_i32(*pos) || tok->numel() < q->size(0) || pos->numel() < q->size(0) ||
      !small(split) || !small(max_len) || (split && !max_len) ||
      (tiles && (!is_i32(*tiles) || tiles->dim() != 2 || tiles->size(1) != 2 ||
                 !small(tiles->size(0)))))
    Py_RETURN_FALSE;
  p.dtype = dt;
  const int n = static_cast<int>(q->size(0));
  size_t need = 0;
  if (split) {
    p.max_seq_len = max_len;
    need = p_vaa_paged_attention_prefill_workspace_size(&p, n, split);
    if (need && !room(ws, need, *q)) return PyLong_FromSize_t(need);
  }
  auto* btp = static_cast<int32_t*>(ptr(*bt));
  auto* tp = static_cast<int32_t*>(ptr(*tok));
  auto* pp = static_cast<int32_t*>(ptr(*pos));
  void* wp = need ? ptr(*ws) : nullptr;
  if (tiles)
    return yes(launch(p_vaa_paged_attention_prefill_tiles, &p, p16(*q), p16(*kc), p16(*vc), btp, tp,
                      pp, p16(*o), n, static_cast<int32_t*>(ptr(*tiles)),
                      static_cast<int>(tiles->size(0)), split, wp, need ? ws->nbytes() : 0,
                      a.s(13)));
  if (split)
    return yes(launch(p_vaa_paged_attention_prefill_split, &p, p16(*q), p16(*kc), p16(*vc), btp, tp,
                      pp, p16(*o), n, split, wp, need ? ws->nbytes() : 0, a.s(13)));
  return yes(launch(p_vaa_paged_attention_prefill, &p, p16(*q), p16(*kc), p16(*vc), btp, tp, pp,
                    p16(*o), n, a.s(13)));
}

// 16-byte aligned rows, which the attention kernels read directly.
bool aligned_rows(const Tensor& t) {
  return rows3(t) && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 && t.stride(0) >= 0 &&
         t.stride(1) >= 0 && (reinterpret_cast<uintptr_t>(ptr(t)) & 15u) == 0;
}
// Whether the address ranges of two tensors' first T rows meet.
bool overlap(const Tensor& a, const Tensor& b, int64_t T) {
  auto end = [T](const Tensor& t) {
    return p16(t) + (T - 1) * t.stride(0) + (t.size(1) - 1) * t.stride(1) + t.size(2);
  };
  return p16(a) < end(b) && p16(b) < end(a);
}

// Attention of T tokens inside their sequences, K and V read in place; the
// caller knows that query_start_loc runs from 0 to T without decreasing.
// (query, key, value, output, query_start_loc, T, num_seqs, head_size, scale,
//  max_seq_len, causal, workspace or None, stream)
PyObject* no_cache(const Args& a) {
  const Tensor *q = a.t(0), *k = a.t(1), *v = a.t(2), *o = a.t(3), *qsl = a.t(4), *ws = a.t(11);
  if (!q || !k || !v || !o || !qsl || !none_or_ten(a.a[11]) || !one_device({q, k, v, o, qsl}))
    Py_RETURN_FALSE;
  const int dt = dt16(*q);
  const int64_t T = a.i(5), S = a.i(6), L = a.i(9);
  if (dt < 0 || dt16(*k) != dt || dt16(*v) != dt || dt16(*o) != dt || !small(T) || T == 0 ||
      !small(S) || S == 0 || !small(L) || !is_i32(*qsl) || qsl->numel() != S + 1)
    Py_RETURN_FALSE;
  for (const Tensor* t : {q, k, v, o})
    if (!aligned_rows(*t) || t->size(0) < T || t->size(2) != a.i(7) || t->size(1) == 0)
      Py_RETURN_FALSE;
  if (k->sizes() != v->sizes() || k->strides() != v->strides() || o->size(1) != q->size(1) ||
      q->size(1) % k->size(1) || overlap(*o, *k, T) || overlap(*o, *v, T))
    Py_RETURN_FALSE;
  vaa_attn_params p{};
  p.dtype = dt;
  p.scale = static_cast<float>(a.f(8));
  p.num_seqs = S;
  p.max_seq_len = L;
  p.head_size = q->size(2);
  p.num_kv_heads = k->size(1);
  p.num_query_heads = q->size(1);
  p.queries_per_kv = q->size(1) / k->size(1);
  p.k_stride_token = p.v_stride_token = k->stride(0);
  p.k_stride_head = p.v_stride_head = k->stride(1);
  p.q_stride_token = q->stride(0);
  p.q_stride_head = q->stride(1);
  p.o_stride_token = o->stride(0);
  p.o_stride_head = o->stride(1);
  const size_t need = p_vaa_attention_no_cache_workspace_size(S, T, L);
  if (!room(ws, need, *q)) return PyLong_FromSize_t(need);
  return yes(launch(p_vaa_attention_no_cache, &p, p16(*q), p16(*k), p16(*v),
                    static_cast<int32_t*>(ptr(*qsl)), p16(*o), T, a.b(10), ptr(*ws), ws->nbytes(),
                    a.s(12)));
}

// bind(handle): the entry points of the library that _lib.py loaded.
PyObject* bind(PyObject*, PyObject* arg) {
  void* h = PyLong_AsVoidPtr(arg);
  if (PyErr_Occurred()) return nullptr;
  // The entry points are found by name and called by this build's signatures.
  auto* version = reinterpret_cast<decltype(&::vaa_abi_version)>(dlsym(h, "vaa_abi_version"));
  if (!version || version() != VAA_ABI_VERSION) {
    PyErr_Format(PyExc_RuntimeError, "ABI version mismatch: the library has %d, _host needs %d",
                 version ? version() : 0, VAA_ABI_VERSION);
    return nullptr;
  }
#define VAA_BIND(f)                                                    \
  p_##f = reinterpret_cast<decltype(p_##f)>(dlsym(h, #f));             \
  if (!p_##f) {                                                        \
    p_vaa_rmsnorm = nullptr;                                           \
    PyErr_SetString(PyExc_RuntimeError, "missing entry point " #f);    \
    return nullptr;                                                    \
  }
  VAA_FUNCS(VAA_BIND)
#undef VAA_BIND
  Py_RETURN_NONE;
}

#define VAA_METHOD(name, n) \
  {#name, reinterpret_cast<PyCFunction>(guarded<n, name>), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"bind", bind, METH_O, nullptr},
                         VAA_METHOD(norm, 7),
                         VAA_METHOD(silu, 4),
                         VAA_METHOD(epilogue, 13),
                         VAA_METHOD(topk, 6),
                         VAA_METHOD(gate_up, 6),
                         VAA_METHOD(linear, 5),
                         VAA_METHOD(kv_write, 7),
                         VAA_METHOD(decode, 14),
                         VAA_METHOD(step_decode, 16),
                         VAA_METHOD(step_prefill, 16),
                         VAA_METHOD(prefill, 14),
                         VAA_METHOD(no_cache, 13),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods,
                      nullptr,               nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
