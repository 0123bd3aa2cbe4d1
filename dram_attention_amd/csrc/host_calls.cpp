// The host's part of a decode step and of a token through the model, as calls of one Python module
// (_host): the operands' checks, the outputs' allocation and the library's entry point in one
// native call each.  Nothing is kept from call to call: every operand is looked at every time.
//
// Bound: the interpreter.  A check of a tensor costs 0.1 us an attribute from Python, 17 tensors
// of 4 to 8 attributes a step, which made a step of a small layer wait for its caller.  us of a host
// thread, from Python / from here: a paged layer's step 29 / 22, a static one's 26 / 12, a token of a
// 4-layer model 331 / 218, of which 3 us a launch are the runtime's.
//
// A call that finds an operand other than the kernels take it returns None (or false): the
// caller then goes the general way, which takes or refuses it.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <initializer_list>
#include <string>
#include <vector>

#include "../../include/dram_attention_amd.h"

namespace {

PyObject *parameter_class;   // torch.nn.Parameter

// Plain tensors only: what a subclass does when it is read is its own.
const at::Tensor *tensor_of(PyObject *o) {
  if (Py_TYPE(o) != (PyTypeObject *)THPVariableClass && (PyObject *)Py_TYPE(o) != parameter_class) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  return t.layout() == at::kStrided ? &t : nullptr;
}

int dtype_code(const at::Tensor &t) {
  switch (t.scalar_type()) {
    case at::kFloat: return DA_F32;
    case at::kHalf: return DA_F16;
    case at::kBFloat16: return DA_BF16;
    default: return -1;
  }
}

bool like(const at::Tensor &t, const at::Tensor &x) {
  return t.scalar_type() == x.scalar_type() && t.device() == x.device() && t.is_contiguous();
}
bool aligned(const at::Tensor &t) { return (uintptr_t)t.data_ptr() % 16 == 0; }
bool is_shape(const at::Tensor &t, at::IntArrayRef want) { return t.sizes() == want; }

// A whole number of any kind (numpy's too); `ok` is left false by anything else.
int64_t whole_number(PyObject *o, bool &ok) {
  PyObject *n = PyNumber_Index(o);
  const long long v = n ? PyLong_AsLongLong(n) : -1;
  Py_XDECREF(n);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    ok = false;
  }
  return v;
}

// Positional arguments, read in order; what is not what it should be leaves `ok` false.
struct Args {
  PyObject *const *at;
  Py_ssize_t left;
  bool ok = true;
  PyObject *next() {
    if (left <= 0) {
      ok = false;
      return Py_None;
    }
    --left;
    return *at++;
  }
  const at::Tensor *tensor() {
    const at::Tensor *t = tensor_of(next());
    ok = ok && t != nullptr;
    return t;
  }
  const at::Tensor *tensor_or_none() {
    PyObject *o = next();
    if (o == Py_None) return nullptr;
    const at::Tensor *t = tensor_of(o);
    ok = ok && t != nullptr;
    return t;
  }
  int64_t integer() { return whole_number(next(), ok); }
  double number() {
    PyObject *o = next();
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
    return v;
  }
  void *pointer() {
    PyObject *o = next();
    if (!PyLong_Check(o)) {
      ok = false;
      return nullptr;
    }
    void *p = PyLong_AsVoidPtr(o);
    if (p == nullptr && PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
    return p;
  }
};

PyObject *raise(int rc, const char *what) {
  PyErr_Format(PyExc_RuntimeError, "%s failed (code %d): %s", what, rc, da_last_error_string());
  return nullptr;
}
// Other Python threads run while this one allocates or launches: either may wait, an allocation for
// another thread that holds the allocator, a launch for room in its queue.
struct Released {
  PyThreadState *state = PyEval_SaveThread();
  ~Released() { PyEval_RestoreThread(state); }
};
template <typename F>
int unlocked(F call) {
  const Released others;
  return call();
}
at::Tensor empty_like(at::IntArrayRef sizes, const at::Tensor &x) {
  const Released others;
  return at::empty(sizes, x.options().requires_grad(false));
}
PyObject *wrap(at::Tensor t) { return THPVariable_Wrap(std::move(t)); }
// A tuple that takes these over; null, with the error that is set, if one is.
PyObject *tuple_of(std::initializer_list<PyObject *> items) {
  PyObject *result = PyTuple_New((Py_ssize_t)items.size());
  bool whole = result != nullptr;
  Py_ssize_t n = 0;
  for (PyObject *o : items) {
    whole = whole && o != nullptr;
    if (result)
      PyTuple_SET_ITEM(result, n++, o);
    else
      Py_XDECREF(o);
  }
  if (!whole) Py_CLEAR(result);
  return result;
}

// The position of the token: a Python int, or one int32 on the device.
struct Position {
  int64_t len;
  const int32_t *len_dev;
};
bool position(PyObject *o, int64_t paged, const at::Tensor &x, Position &p) {
  if (PyLong_CheckExact(o)) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
    p = {v - paged, nullptr};
    return true;
  }
  const at::Tensor *t = tensor_of(o);
  if (!t || t->scalar_type() != at::kInt || t->device() != x.device() || t->numel() < 1) return false;
  p = {-paged, (const int32_t *)t->data_ptr()};
  return true;
}

// step_args(xq, xk, xv, start_pos, minmax, dram, hbm, times, d2h, h2d, counter, cache_k, cache_v, n_slots,
// page, top_k, paged, dram_ptr, stream_blocks, score_flags, link_gbps, block_gbps, scratch, idx, scores, topk_ws,
// workspace) -> (argument block of da_decode_step, output); None: not a step for one call; an
// int, the query rows of a kv head: the operands are, but the last five are not there yet.
PyObject *step_args(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Args in{argv, argc};
  const at::Tensor *xq = in.tensor(), *xk = in.tensor(), *xv = in.tensor();
  PyObject *start = in.next();
  const at::Tensor *minmax = in.tensor(), *dram = in.tensor(), *hbm = in.tensor(), *times = in.tensor(),
                   *d2h = in.tensor(), *h2d = in.tensor(), *counter = in.tensor(), *cache_k = in.tensor(),
                   *cache_v = in.tensor();
  const int64_t N = in.integer(), page = in.integer(), top_k = in.integer(), paged = in.integer();
  void *dram_ptr = in.pointer();
  const int64_t stream_blocks = in.integer(), flags = in.integer();
  const double link = in.number(), block = in.number();
  PyObject *scratch = in.next();
  if (!in.ok) Py_RETURN_NONE;
  const int dtype = dtype_code(*xq);
  if (dtype < 0 || !xq->is_cuda() || xq->dim() != 4 || minmax->dim() != 4) Py_RETURN_NONE;
  const int64_t H = minmax->size(0), P = minmax->size(1), D = minmax->size(3), Hq = xq->size(2);
  if (H < 1 || cache_k->dim() != 4) Py_RETURN_NONE;
  const int64_t rep = Hq / H, kp = top_k < P ? top_k : P, capacity = cache_k->size(1), page_dim = page * 2 * D;
  if (!(is_shape(*xq, {1, 1, rep * H, D}) && is_shape(*xk, {1, 1, H, D}) && is_shape(*xv, {1, 1, H, D}) && kp > 0 &&
        N > 0 && minmax->size(2) == 2 && is_shape(*hbm, {H, N, page_dim}) && is_shape(*dram, {H, P, page_dim}) &&
        is_shape(*times, {H, N}) && is_shape(*h2d, {H, N}) && is_shape(*d2h, {H, P}) &&
        is_shape(*cache_k, {1, capacity, H, D}) && is_shape(*cache_v, {1, capacity, H, D}) &&
        times->scalar_type() == at::kFloat && d2h->scalar_type() == at::kLong && h2d->scalar_type() == at::kLong &&
        counter->scalar_type() == at::kInt && counter->numel() == 1))
    Py_RETURN_NONE;
  // (what the attending page stream takes)
  const int64_t row = D * xq->element_size();
  if (!((row == 64 || row == 128 || row == 256 || row == 512) && rep >= 1 && rep <= 8 && page * 2 * row <= 16384 &&
        H <= 64))
    Py_RETURN_NONE;
  for (const at::Tensor *t : {xq, xk, xv, minmax, hbm, cache_k, cache_v})
    if (!like(*t, *xq)) Py_RETURN_NONE;
  for (const at::Tensor *t : {times, d2h, h2d, counter})
    if (t->device() != xq->device() || !t->is_contiguous()) Py_RETURN_NONE;
  if (dram->scalar_type() != xq->scalar_type() || !dram->is_contiguous()) Py_RETURN_NONE;
  Position pos;
  if (!position(start, paged, *xq, pos)) Py_RETURN_NONE;
  if (!pos.len_dev && (pos.len < 0 || pos.len >= capacity)) Py_RETURN_NONE;

  // (the room is looked at like the operands: the kernels write to all of it)
  const int64_t total = rep * kp;
  auto fits = [&](const at::Tensor *t, at::IntArrayRef shape, at::ScalarType type) {
    return t && t->scalar_type() == type && t->device() == xq->device() && t->is_contiguous() && is_shape(*t, shape);
  };
  const at::Tensor *idx = in.tensor_or_none(), *scores = in.tensor_or_none(), *topk_ws = in.tensor_or_none(),
                   *workspace = in.tensor_or_none();
  if (!in.ok) Py_RETURN_NONE;
  const size_t topk_need = da_topk_pages_workspace_bytes((int)rep, (int)H, P, (int)kp);
  if (!PyTuple_Check(scratch) || PyTuple_GET_SIZE(scratch) != 7 || !fits(idx, {H, total}, at::kLong) ||
      !fits(scores, {rep, H, P}, at::kFloat) || !workspace || !fits(workspace, workspace->sizes(), at::kFloat) ||
      (topk_need && (!topk_ws || !fits(topk_ws, topk_ws->sizes(), at::kByte) ||
                     (size_t)topk_ws->nbytes() < topk_need)))
    return PyLong_FromLongLong(rep);
  const at::Tensor *room[7];   // miss_page, miss_slot, miss_count, hit_mask, workspace, slot_epoch, candidates
  for (int i = 0; i < 7; ++i)
    if (!(room[i] = tensor_of(PyTuple_GET_ITEM(scratch, i)))) Py_RETURN_NONE;
  if (room[0]->dim() != 2 || room[0]->size(1) != total) return PyLong_FromLongLong(rep);
  const at::Tensor &list = *room[6];
  if (list.dim() != 2 || list.size(1) < 1) Py_RETURN_NONE;
  const int64_t stamps_end = list.storage_offset() + H * (list.size(1) + 1);   // (a word per head behind the lists)
  if (!(fits(room[0], {H, total}, at::kInt) && fits(room[1], {H, total}, at::kInt) && fits(room[2], {H}, at::kInt) &&
        fits(room[3], {H, total}, at::kByte) && fits(room[4], room[4]->sizes(), at::kByte) &&
        fits(room[5], {H, N}, at::kInt) && fits(&list, {H, list.size(1)}, at::kInt) &&
        (int64_t)list.storage().nbytes() >= stamps_end * 4))
    Py_RETURN_NONE;

  at::Tensor out = empty_like({1, 1, Hq, D}, *xq);
  da_decode_step_args a = {};
  a.q = xq->data_ptr();
  a.new_k = xk->data_ptr();
  a.new_v = xv->data_ptr();
  a.out = out.data_ptr();
  a.minmax = minmax->data_ptr();
  a.scores = (float *)scores->data_ptr();
  a.idx = (int64_t *)idx->data_ptr();
  if (topk_need) {
    a.topk_workspace = topk_ws->data_ptr();
    a.topk_workspace_bytes = (int64_t)topk_ws->nbytes();
  }
  a.access_time = (float *)times->data_ptr();
  a.candidates = (int32_t *)room[6]->data_ptr();
  a.step = (int32_t *)counter->data_ptr();
  a.d2h = (int64_t *)d2h->data_ptr();
  a.h2d = (int64_t *)h2d->data_ptr();
  a.miss_page = (int32_t *)room[0]->data_ptr();
  a.miss_slot = (int32_t *)room[1]->data_ptr();
  a.miss_count = (int32_t *)room[2]->data_ptr();
  a.hit_mask = (uint8_t *)room[3]->data_ptr();
  a.lru_workspace = room[4]->data_ptr();
  a.lru_workspace_bytes = (int64_t)room[4]->nbytes();
  a.slot_epoch = (int32_t *)room[5]->data_ptr();
  a.dram = dram_ptr;
  a.hbm = hbm->data_ptr();
  a.cache_k = cache_k->data_ptr();
  a.cache_v = cache_v->data_ptr();
  a.cache_len_dev = pos.len_dev;
  a.workspace = workspace->data_ptr();
  a.workspace_bytes = (int64_t)workspace->nbytes();
  a.q_head_stride = D;
  a.n_pages = P;
  a.cache_rows = capacity;
  a.cache_len = pos.len;
  a.n_q_heads = (int32_t)Hq;
  a.n_kv_heads = (int32_t)H;
  a.head_dim = (int32_t)D;
  a.dtype = dtype;
  a.page_size = (int32_t)page;
  a.kp = (int32_t)kp;
  a.n_slots = (int32_t)N;
  a.k_cand = (int32_t)room[6]->size(1);
  a.score_flags = (int32_t)flags;
  const int64_t blocks = stream_blocks / H < total ? stream_blocks / H : total;
  a.gather_blocks = (int32_t)(blocks > 1 ? blocks : 1);
  a.scale = (float)(1.0 / std::sqrt((double)D));
  a.link_gbps = (float)link;
  a.block_gbps = (float)block;
  return tuple_of({PyBytes_FromStringAndSize((const char *)&a, sizeof(a)), wrap(std::move(out))});
  END_HANDLE_TH_ERRORS
}

// static_step(xq, xk, xv, start_pos, prefix_k, prefix_v, cache_k, cache_v, paged, workspace, stream) -> output of
// a step over a static prefix, or None.
PyObject *static_step(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Args in{argv, argc};
  const at::Tensor *xq = in.tensor(), *xk = in.tensor(), *xv = in.tensor();
  PyObject *start = in.next();
  const at::Tensor *pk = in.tensor(), *pv = in.tensor(), *ck = in.tensor(), *cv = in.tensor();
  const int64_t paged = in.integer();
  const at::Tensor *workspace = in.tensor_or_none();
  void *stream = in.pointer();
  if (!in.ok || !workspace) Py_RETURN_NONE;
  const int dtype = dtype_code(*xq);
  if (dtype < 0 || !xq->is_cuda() || xq->dim() != 4 || pk->dim() != 3 || ck->dim() != 4) Py_RETURN_NONE;
  const int64_t Hq = xq->size(2), D = xq->size(3), H = ck->size(2), capacity = ck->size(1), T = pk->size(1);
  if (!(is_shape(*xq, {1, 1, Hq, D}) && is_shape(*xk, {1, 1, H, D}) && is_shape(*xv, {1, 1, H, D}) &&
        is_shape(*pk, {H, T, D}) && is_shape(*pv, {H, T, D}) && is_shape(*ck, {1, capacity, H, D}) &&
        is_shape(*cv, {1, capacity, H, D}) && T > 0 && capacity > 0 && pk->strides() == pv->strides() &&
        ck->strides() == cv->strides() && xk->strides() == xv->strides() && workspace->is_contiguous()))
    Py_RETURN_NONE;
  for (const at::Tensor *t : {xq, xk, xv, pk, pv, ck, cv})
    if (t->scalar_type() != xq->scalar_type() || t->device() != xq->device() || t->stride(-1) != 1) Py_RETURN_NONE;
  if (workspace->device() != xq->device()) Py_RETURN_NONE;
  Position pos;
  if (!position(start, paged, *xq, pos)) Py_RETURN_NONE;
  at::Tensor out = empty_like({1, 1, Hq, D}, *xq);
  const int rc = unlocked([&] {
    return da_decode_attention(
        xq->data_ptr(), xq->stride(2), (int)Hq, (int)H, (int)D, dtype, pk->data_ptr(), pv->data_ptr(), pk->stride(1),
        pk->stride(0), T, ck->data_ptr(), cv->data_ptr(), ck->stride(1), ck->stride(2), capacity, pos.len, pos.len_dev,
        xk->data_ptr(), xv->data_ptr(), xk->stride(2), (float)(1.0 / std::sqrt((double)D)), out.data_ptr(), D, nullptr,
        workspace->data_ptr(), workspace->nbytes(), stream);
  });
  if (rc) return raise(rc, "da_decode_attention");
  return wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// alike(x, ...) -> whether all are plain, contiguous, aligned GPU tensors of x's type and device.
PyObject *alike(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Args in{argv, argc};
  const at::Tensor *x = in.tensor();
  if (!in.ok || !x->is_cuda() || dtype_code(*x) < 0 || !like(*x, *x) || !aligned(*x)) Py_RETURN_FALSE;
  while (in.left > 0) {
    const at::Tensor *t = in.tensor();
    if (!in.ok || !like(*t, *x) || !aligned(*t)) Py_RETURN_FALSE;
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// linears(x, nn.Linear, longest_row, module, out, in, module, out, in, ...) -> the modules' weights as a tuple, or
// None: each is an nn.Linear (no kind of its own) without bias, that nobody hooked and whose forward
// nobody exchanged, its weight a plain contiguous aligned tensor of x's type and device, of shape
// (out, in) (-1: whatever the module says) and with rows that the one-token layers hold.
PyObject *linears(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  static PyObject *hooks = PyUnicode_InternFromString("_forward_hooks");
  static PyObject *pre_hooks = PyUnicode_InternFromString("_forward_pre_hooks");
  static PyObject *forward = PyUnicode_InternFromString("forward");
  static PyObject *parameters = PyUnicode_InternFromString("_parameters");
  static PyObject *weight_name = PyUnicode_InternFromString("weight");
  static PyObject *bias_name = PyUnicode_InternFromString("bias");
  static PyObject *out_name = PyUnicode_InternFromString("out_features");
  static PyObject *in_name = PyUnicode_InternFromString("in_features");
  Args in{argv, argc};
  const at::Tensor *x = in.tensor();
  PyObject *linear = in.next();
  const int64_t longest = in.integer();
  if (!in.ok || in.left % 3) Py_RETURN_NONE;
  const Py_ssize_t n = in.left / 3;
  PyObject *weights = PyTuple_New(n);
  if (!weights) return nullptr;
  auto item = [](PyObject *dict, PyObject *name) -> PyObject * {
    PyObject *o = dict && PyDict_Check(dict) ? PyDict_GetItemWithError(dict, name) : nullptr;
    if (!o) PyErr_Clear();
    return o;
  };
  auto features = [&](PyObject *dict, PyObject *name) -> int64_t {
    PyObject *o = item(dict, name);
    bool ok = o != nullptr;
    const int64_t n = ok ? whole_number(o, ok) : 0;
    return ok ? n : -2;
  };
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject *m = in.next();
    const int64_t want_out = in.integer(), want_in = in.integer();
    bool fits = in.ok && (PyObject *)Py_TYPE(m) == linear;
    PyObject **dict_at = fits ? _PyObject_GetDictPtr(m) : nullptr;
    PyObject *dict = dict_at ? *dict_at : nullptr;
    PyObject *h = item(dict, hooks), *p = item(dict, pre_hooks), *params = item(dict, parameters);
    PyObject *w = item(params, weight_name), *b = item(params, bias_name);
    fits = fits && h && p && PyDict_Check(h) && PyDict_Check(p) && PyDict_Size(h) == 0 && PyDict_Size(p) == 0 &&
           !item(dict, forward) && w && b == Py_None;
    const at::Tensor *t = fits ? tensor_of(w) : nullptr;
    if (t) {
      const int64_t rows = features(dict, out_name), cols = features(dict, in_name);
      const int64_t row_bytes = cols * (int64_t)x->element_size();
      fits = like(*t, *x) && aligned(*t) && is_shape(*t, {rows, cols}) && (want_out < 0 || want_out == rows) &&
             (want_in < 0 || want_in == cols) && row_bytes % 16 == 0 && row_bytes <= longest;
    }
    if (!t || !fits) {
      Py_DECREF(weights);
      Py_RETURN_NONE;
    }
    Py_INCREF(w);
    PyTuple_SET_ITEM(weights, i, w);
  }
  return weights;
  END_HANDLE_TH_ERRORS
}

// qkv_rope(x, norm_weight, eps, wq, wk, wv, n_heads, n_kv_heads, head_dim, rope_row, stream) -> (q, k, v); the
// operands are checked.
PyObject *qkv_rope(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Args in{argv, argc};
  const at::Tensor *x = in.tensor(), *norm = in.tensor();
  const double eps = in.number();
  const at::Tensor *wq = in.tensor(), *wk = in.tensor(), *wv = in.tensor();
  const int64_t Hq = in.integer(), H = in.integer(), D = in.integer();
  const at::Tensor *rope = in.tensor();
  void *stream = in.pointer();
  if (!in.ok) return PyErr_Format(PyExc_TypeError, "qkv_rope: bad argument");
  at::Tensor q = empty_like({1, 1, Hq, D}, *x), k = empty_like({1, 1, H, D}, *x), v = empty_like({1, 1, H, D}, *x);
  const int rc = unlocked([&] {
    return da_linear_qkv_rope(x->data_ptr(), norm->data_ptr(), (float)eps, (int)x->size(-1), wq->data_ptr(),
                              wk->data_ptr(), wv->data_ptr(), (int)Hq, (int)H, (int)D,
                              (const float *)rope->data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                              dtype_code(*x), stream);
  });
  if (rc) return raise(rc, "da_linear_qkv_rope");
  return tuple_of({wrap(std::move(q)), wrap(std::move(k)), wrap(std::move(v))});
  END_HANDLE_TH_ERRORS
}

// block_tail(attended, wo, x, norm_weight, eps, w1, w3, w2, stream) -> the block's output; the operands
// are checked.
PyObject *block_tail(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Args in{argv, argc};
  const at::Tensor *attended = in.tensor(), *wo = in.tensor(), *x = in.tensor(), *norm = in.tensor();
  const double eps = in.number();
  const at::Tensor *w1 = in.tensor(), *w3 = in.tensor(), *w2 = in.tensor();
  void *stream = in.pointer();
  if (!in.ok) return PyErr_Format(PyExc_TypeError, "block_tail: bad argument");
  const int64_t dim = w2->size(0), hidden = w2->size(1);
  at::Tensor room = empty_like({dim + hidden}, *x), out = empty_like(x->sizes(), *x);
  char *h = (char *)room.data_ptr();
  const int rc = unlocked([&] {
    return da_linear_block_tail(attended->data_ptr(), (int)wo->size(1), wo->data_ptr(), x->data_ptr(), (int)dim,
                                norm->data_ptr(), (float)eps, w1->data_ptr(), w3->data_ptr(), (int)hidden,
                                w2->data_ptr(), h, h + dim * x->element_size(), out.data_ptr(), dtype_code(*x),
                                stream);
  });
  if (rc) return raise(rc, "da_linear_block_tail");
  return wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

#define DA_CALL(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {DA_CALL(step_args), DA_CALL(static_step), DA_CALL(alike), DA_CALL(linears),
                         DA_CALL(qkv_rope),  DA_CALL(block_tail),  {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  PyObject *nn = PyImport_ImportModule("torch.nn");
  if (!nn) return nullptr;
  parameter_class = PyObject_GetAttrString(nn, "Parameter");
  Py_DECREF(nn);
  return parameter_class ? PyModule_Create(&module) : nullptr;
}
