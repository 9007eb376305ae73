// The per-layer calls of an engine step, from torch tensors to libkvhot's
// entry points without Python in between: paged_flash_attention, the append
// (_PagedKVCache.write) and the two together (a model's layer).
//
// Every function here answers the ordinary call only, after checking all that
// the Python function of the same name checks, and returns None before it has
// done anything when a check fails, when something it needs (a launch list,
// a workspace) is not there yet or when the library refuses the launch; the
// Python function then takes the call, does that preparation or raises.  (Where
// layer()'s attention is refused its append is queued already, and its answer
// says so.)  Nothing is kept between calls: pointers, shapes
// and strides are read from the tensors each time.
//
// Measured, Python with ctypes before -> here, calls queued back to back on one
// MI355X: an append of 16 tokens 8.2 -> 4.3 us, attention of one row of 1001
// keys 20.2 -> 12.1, a layer (append and attention) of 8 decode rows 33 -> 16,
// of 4 short fp32 rows 31.5 -> 12.2, 16 layers of 16 rows with their step's
// metadata and launch list 770 -> 360 to 450.  From here on the GPU's own time bounds
// all of these but the last two.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/kvhot.h"

namespace {

using at::Tensor;

decltype(&kvhot_paged_attention) g_attention = nullptr;
decltype(&kvhot_paged_attention_workspace_bytes) g_workspace_bytes = nullptr;
decltype(&kvhot_reshape_and_cache) g_append = nullptr;

// Keys of the metadata dict and of its launch lists.
struct Names {
  PyObject *q_lens, *k_lens, *q_starts, *q_pos_offsets, *block_table, *block_table_row_stride, *max_q_len, *max_k_len,
      *host_q_lens, *schedules, *schedule_streams;
} g_names;

// The plain torch.Tensor behind o, with memory on a GPU.  (Subclasses and
// functorch's wrappers, which have no storage of their own, are not taken.)
bool gpu_tensor(PyObject* o, Tensor& t) {
  if (!o || !THPVariable_CheckExact(o)) return false;
  t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() &&
         !t.unsafeGetTensorImpl()->key_set().has(c10::DispatchKey::Python) && !t.is_conj() && !t.is_neg();
}

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return KVHOT_F32;
    case at::kHalf: return KVHOT_F16;
    case at::kBFloat16: return KVHOT_BF16;
    default: return -1;
  }
}

// An integer that fits int64 (bool excluded: the Python path's business).
bool as_int(PyObject* o, int64_t& x) {
  if (!o || PyBool_Check(o) || !PyIndex_Check(o)) return false;
  PyObject* i = PyNumber_Index(o);
  if (!i) return false;
  int overflow = 0;
  x = PyLong_AsLongLongAndOverflow(i, &overflow);
  Py_DECREF(i);
  return overflow == 0;
}

// An int32 contiguous metadata tensor of n rows on device d.
bool meta_tensor(PyObject* meta, PyObject* name, c10::Device d, int64_t n, Tensor& t) {
  return gpu_tensor(PyDict_GetItemWithError(meta, name), t) && t.scalar_type() == at::kInt && t.device() == d &&
         t.is_contiguous() && t.dim() >= 1 && t.size(0) == n;
}

// One layer's append: K and V new rows [1, Hkv, S, D] into the pool.
struct Append {
  Tensor kv, key, value, slots;
  int64_t layer, heads, dim;

  bool check(PyObject* kv_o, PyObject* heads_o, PyObject* dim_o, PyObject* key_o, PyObject* value_o, PyObject* layer_o,
             PyObject* slots_o) {
    if (!gpu_tensor(kv_o, kv) || !gpu_tensor(key_o, key) || !gpu_tensor(value_o, value) || !gpu_tensor(slots_o, slots) ||
        !as_int(heads_o, heads) || !as_int(dim_o, dim) || !as_int(layer_o, layer))
      return false;
    return kv.dim() == 6 && kv.size(1) == 2 && key.dim() == 4 && key.size(0) == 1 && value.sizes() == key.sizes() &&
           key.size(1) == heads && key.size(3) == dim && key.size(2) > 0 && heads > 0 && dim > 0 &&
           kv.size(4) == heads && kv.size(5) == dim && dtype_code(kv) >= 0 && key.scalar_type() == kv.scalar_type() &&
           value.scalar_type() == kv.scalar_type() && slots.dim() == 1 && slots.size(0) == key.size(2) &&
           (slots.scalar_type() == at::kLong || slots.scalar_type() == at::kInt) && slots.is_contiguous() &&
           key.device() == kv.device() && value.device() == kv.device() && slots.device() == kv.device() && layer >= 0 &&
           layer < kv.size(0);
  }
  char* pool(int64_t which) const {
    return static_cast<char*>(kv.data_ptr()) + (layer * kv.stride(0) + which * kv.stride(1)) * kv.element_size();
  }
  int launch(void* stream) const {
    const int64_t ks[3] = {key.stride(2), key.stride(1), key.stride(3)};
    const int64_t vs[3] = {value.stride(2), value.stride(1), value.stride(3)};
    const int64_t cs[4] = {kv.stride(2), kv.stride(3), kv.stride(4), kv.stride(5)};
    return g_append(key.data_ptr(), ks, value.data_ptr(), vs, pool(0), cs, pool(1), cs, slots.data_ptr(),
                    slots.scalar_type() == at::kLong ? 1 : 0, key.size(2), heads, dim, kv.size(3), kv.size(2),
                    dtype_code(kv), stream);
  }
};

// One attention call: q [T, Hq, D] over the pool's blocks.
struct Attention {
  Tensor q, k_lens, q_lens, q_starts, q_offs, bt, units, ws;
  const void *k = nullptr, *v = nullptr;
  int64_t kst[4], vst[4], num_blocks, block_size, hkv;
  int64_t bt_stride, max_q, max_k, counts[4], need, pt;
  bool listed = false;
  float scale;
  int flags;
  void* stream;

  // Whether the stream comes after the copy of the launch list of `key`
  // (_order_list's record; a list without one is taken as it is).
  bool list_ordered(PyObject* meta, PyObject* key) const {
    PyObject* all = PyDict_GetItemWithError(meta, g_names.schedule_streams);
    PyObject* rec = all && PyDict_CheckExact(all) ? PyDict_GetItemWithError(all, key) : nullptr;
    if (!rec) return !PyErr_Occurred();
    if (!PyTuple_CheckExact(rec) || PyTuple_GET_SIZE(rec) != 2 || !PySet_Check(PyTuple_GET_ITEM(rec, 1))) return false;
    PyObject* h = PyLong_FromLongLong(static_cast<long long>(reinterpret_cast<intptr_t>(stream)));
    if (!h) return false;
    const int in = PySet_Contains(PyTuple_GET_ITEM(rec, 1), h);
    Py_DECREF(h);
    return in == 1;
  }

  // q, the pool and hkv are set; the rest from the metadata.
  bool check(PyObject* meta, PyObject* scale_o, int64_t pt_, bool causal, int flags_, PyObject* workspaces) {
    if (!PyDict_CheckExact(meta) || !PyDict_CheckExact(workspaces) || !PyFloat_Check(scale_o)) return false;
    scale = static_cast<float>(PyFloat_AS_DOUBLE(scale_o));
    pt = pt_;
    flags = flags_;
    const c10::Device d = q.device();
    const int64_t hq = q.size(1), dim = q.size(2);
    stream = c10::hip::getCurrentHIPStream(d.index()).stream();
    const int dt = dtype_code(q);
    if (dt < 0 || hkv <= 0 || hq <= 0 || hq % hkv != 0 || q.size(0) == 0 || dim == 0) return false;
    if (!gpu_tensor(PyDict_GetItemWithError(meta, g_names.q_lens), q_lens) || q_lens.dim() < 1) return false;
    const int64_t rows = q_lens.size(0);
    if (rows == 0 || q_lens.scalar_type() != at::kInt || q_lens.device() != d || !q_lens.is_contiguous() ||
        !meta_tensor(meta, g_names.k_lens, d, rows, k_lens) || !meta_tensor(meta, g_names.q_starts, d, rows, q_starts) ||
        !meta_tensor(meta, g_names.q_pos_offsets, d, rows, q_offs) || !meta_tensor(meta, g_names.block_table, d, rows, bt))
      return false;
    PyObject* st = PyDict_GetItemWithError(meta, g_names.block_table_row_stride);
    if (st) {
      if (!as_int(st, bt_stride)) return false;
    } else {
      bt_stride = bt.dim() == 2 ? bt.size(1) : 0;
    }
    if (!as_int(PyDict_GetItemWithError(meta, g_names.max_q_len), max_q) ||
        !as_int(PyDict_GetItemWithError(meta, g_names.max_k_len), max_k))
      return false;
    PyObject* host = PyDict_GetItemWithError(meta, g_names.host_q_lens);
    if (host && host != Py_None) {
      // The step's launch list, built by the first call of its shape.
      PyObject* lists = PyDict_GetItemWithError(meta, g_names.schedules);
      if (!lists || !PyDict_CheckExact(lists)) return false;
      char name[16];
      snprintf(name, sizeof name, "cuda:%d", static_cast<int>(d.index()));
      PyObject* key = Py_BuildValue("(LLLLLOis)", (long long)hq, (long long)hkv, (long long)dim, (long long)block_size,
                                    (long long)pt, causal ? Py_True : Py_False, dt, name);
      if (!key) return false;
      PyObject* hit = PyDict_GetItemWithError(lists, key);
      const bool ordered = hit && (hit == Py_None || list_ordered(meta, key));
      Py_DECREF(key);
      if (!ordered) return false;
      if (hit != Py_None) {
        if (!PyTuple_CheckExact(hit) || PyTuple_GET_SIZE(hit) != 6) return false;
        // (device units, decode, prefill, merge units, workspace bytes, prefix units)
        if (!as_int(PyTuple_GET_ITEM(hit, 1), counts[0]) || !as_int(PyTuple_GET_ITEM(hit, 2), counts[1]) ||
            !as_int(PyTuple_GET_ITEM(hit, 3), counts[2]) || !as_int(PyTuple_GET_ITEM(hit, 4), need) ||
            !as_int(PyTuple_GET_ITEM(hit, 5), counts[3]) || !gpu_tensor(PyTuple_GET_ITEM(hit, 0), units))
          return false;
        listed = counts[0] + counts[1] > 0;
      }
    }
    if (!listed) {
      counts[0] = counts[1] = counts[2] = counts[3] = 0;
      need = g_workspace_bytes(rows, q.size(0), max_q, max_k, hq, hkv, dim, block_size, pt, dt);
      if (need < 0) return false;
    }
    if (need > 0) {  // the stream's workspace, made by the first call that needs it
      hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing(static_cast<hipStream_t>(stream), &capture) != hipSuccess)
        (void)hipGetLastError();
      if (capture != hipStreamCaptureStatusNone)
        return false;  // a graph's calls have workspaces of their own
      PyObject* key = Py_BuildValue("(iL)", static_cast<int>(d.index()),
                                    static_cast<long long>(reinterpret_cast<intptr_t>(stream)));
      if (!key) return false;
      PyObject* w = PyDict_GetItemWithError(workspaces, key);
      Py_DECREF(key);
      if (!gpu_tensor(w, ws) || ws.numel() < need) return false;
    }
    return true;
  }

  int launch(const Tensor& o, const Tensor& l) const {
    const int64_t qs[3] = {q.stride(0), q.stride(1), q.stride(2)}, os[3] = {o.stride(0), o.stride(1), o.stride(2)};
    const int64_t ls[2] = {l.stride(0), l.stride(1)};
    const auto i32 = [](const Tensor& t) { return static_cast<const int32_t*>(t.data_ptr()); };
    return g_attention(q.data_ptr(), qs, k, kst, v, vst, o.data_ptr(), os, static_cast<float*>(l.data_ptr()), ls, i32(bt),
                       bt_stride, i32(q_lens), i32(k_lens), i32(q_starts), i32(q_offs), q_lens.size(0), q.size(0), max_q,
                       max_k, q.size(1), hkv, q.size(2), block_size, num_blocks, scale, flags, dtype_code(q), pt,
                       listed ? i32(units) : nullptr, counts[0], counts[1], counts[2], counts[3], listed ? need : 0,
                       ws.defined() ? ws.data_ptr() : nullptr, ws.defined() ? ws.numel() : 0, stream);
  }
};

// The call's Python result, or None with no error set.
template <class F>
PyObject* or_none(F f) {
  PyObject* r = nullptr;
  try {
    r = f();
  } catch (...) {
    r = nullptr;
  }
  if (!r) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  return r;
}

// f() without the GIL, which is taken again whichever way f ends.
template <class F>
int without_gil(F f) {
  struct Released {
    PyThreadState* state = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(state); }
  } released;
  return f();
}

Tensor lse_of(const Tensor& q) {
  return at::empty({q.size(0), q.size(1)}, q.options().dtype(at::kFloat).requires_grad(false).memory_format(c10::nullopt));
}

// attention(q, k_cache, v_cache, metadata, hq, hkv, scale, causal, pt, flags, workspaces) -> (o, l) | None
PyObject* py_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return or_none([&]() -> PyObject* {
    Tensor k, v;
    Attention at_;
    int64_t hq, pt, flags;
    if (n != 11 || !g_attention || !gpu_tensor(a[0], at_.q) || !gpu_tensor(a[1], k) || !gpu_tensor(a[2], v) ||
        !as_int(a[4], hq) || !as_int(a[5], at_.hkv) || !as_int(a[8], pt) || !as_int(a[9], flags) || !PyBool_Check(a[7]))
      return nullptr;
    const Tensor& q = at_.q;
    if (q.dim() != 3 || k.dim() != 4 || v.sizes() != k.sizes() || q.size(1) != hq || k.size(2) != at_.hkv ||
        k.size(3) != q.size(2) || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() ||
        k.device() != q.device() || v.device() != q.device())
      return nullptr;
    for (int i = 0; i < 4; ++i) {
      at_.kst[i] = k.stride(i);
      at_.vst[i] = v.stride(i);
    }
    at_.k = k.data_ptr();
    at_.v = v.data_ptr();
    at_.num_blocks = k.size(0);
    at_.block_size = k.size(1);
    if (!at_.check(a[3], a[6], pt, a[7] == Py_True, static_cast<int>(flags), a[10])) return nullptr;
    const Tensor o = at::empty_like(q, q.options().requires_grad(false)), l = lse_of(q);
    if (without_gil([&] { return at_.launch(o, l); }) != 0) return nullptr;
    PyObject* r = PyTuple_New(2);
    if (!r) return nullptr;
    PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(o));
    PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(l));
    return r;
  });
}

// append(kv_cache, heads, dim, key, value, layer, slots) -> True | None
PyObject* py_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return or_none([&]() -> PyObject* {
    Append ap;
    if (n != 7 || !g_append || !ap.check(a[0], a[1], a[2], a[3], a[4], a[5], a[6])) return nullptr;
    void* stream = c10::hip::getCurrentHIPStream(ap.kv.device().index()).stream();
    if (without_gil([&] { return ap.launch(stream); }) != 0) return nullptr;
    Py_RETURN_TRUE;
  });
}

// layer(kv_cache, heads, dim, key, value, layer, slots, query, metadata, scale, pt, flags, workspaces)
//   -> o [1, S, Hq, D] | None | False: the append, then causal attention; False
//   where the append is queued and the library then refused the attention.
PyObject* py_layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return or_none([&]() -> PyObject* {
    Append ap;
    Attention at_;
    Tensor query;
    int64_t pt, flags;
    if (n != 13 || !g_append || !g_attention || !ap.check(a[0], a[1], a[2], a[3], a[4], a[5], a[6]) ||
        !gpu_tensor(a[7], query) || !as_int(a[10], pt) || !as_int(a[11], flags))
      return nullptr;
    const Tensor& kv = ap.kv;
    if (query.dim() != 4 || query.size(0) != 1 || query.size(3) != ap.dim ||
        query.scalar_type() != kv.scalar_type() || query.device() != kv.device())
      return nullptr;
    at_.q = query.transpose(1, 2).squeeze(0);
    if (at_.q.dim() != 3) return nullptr;
    for (int i = 0; i < 4; ++i) at_.kst[i] = at_.vst[i] = kv.stride(2 + i);
    at_.k = ap.pool(0);
    at_.v = ap.pool(1);
    at_.num_blocks = kv.size(2);
    at_.block_size = kv.size(3);
    at_.hkv = ap.heads;
    if (!at_.check(a[8], a[9], pt, true, static_cast<int>(flags), a[12])) return nullptr;
    const Tensor o = at::empty_like(at_.q, at_.q.options().requires_grad(false)), l = lse_of(at_.q);
    if (without_gil([&] { return ap.launch(at_.stream); }) != 0) return nullptr;
    // (An exception here, from a library call that could not form its message,
    // is such a refusal too.)
    int status = -1;
    try {
      status = without_gil([&] { return at_.launch(o, l); });
    } catch (...) {
    }
    if (status != 0) Py_RETURN_FALSE;
    return THPVariable_Wrap(o.unsqueeze(0));
  });
}

// bind(attention, workspace_bytes, append): addresses of libkvhot's entry points.
PyObject* py_bind(PyObject*, PyObject* args) {
  unsigned long long at, ws, ap;
  if (!PyArg_ParseTuple(args, "KKK", &at, &ws, &ap)) return nullptr;
  g_attention = reinterpret_cast<decltype(g_attention)>(static_cast<uintptr_t>(at));
  g_workspace_bytes = reinterpret_cast<decltype(g_workspace_bytes)>(static_cast<uintptr_t>(ws));
  g_append = reinterpret_cast<decltype(g_append)>(static_cast<uintptr_t>(ap));
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_attention)), METH_FASTCALL, nullptr},
    {"append", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_append)), METH_FASTCALL, nullptr},
    {"layer", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_layer)), METH_FASTCALL, nullptr},
    {"bind", py_bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "kvhot_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_kvhot_torch(void) {
  Names& g = g_names;
  g.q_lens = PyUnicode_InternFromString("q_lens");
  g.k_lens = PyUnicode_InternFromString("k_lens");
  g.q_starts = PyUnicode_InternFromString("q_starts");
  g.q_pos_offsets = PyUnicode_InternFromString("q_pos_offsets");
  g.block_table = PyUnicode_InternFromString("block_table");
  g.block_table_row_stride = PyUnicode_InternFromString("block_table_row_stride");
  g.max_q_len = PyUnicode_InternFromString("max_q_len");
  g.max_k_len = PyUnicode_InternFromString("max_k_len");
  g.host_q_lens = PyUnicode_InternFromString("host_q_lens");
  g.schedules = PyUnicode_InternFromString("_schedules");
  g.schedule_streams = PyUnicode_InternFromString("_schedule_streams");
  return PyModule_Create(&kModule);
}
