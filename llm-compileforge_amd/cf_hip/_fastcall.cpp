// CPython extension: the tensor entry points' call path in native code.
//
// A call through ctypes costs 15-20 us of host time (a descriptor per tensor
// built in Python, two foreign calls, an output allocation through the Python
// API), more than the kernels of a small step take; the same call from here
// costs the launches plus about 2 us.  Each function checks what its ops.py
// wrapper checks, fills the descriptors from the tensors, allocates outputs
// and calls the library with the GIL released.  It returns
//   - the result (or 0 for calls without one) when the library accepted it,
//   - the library's negative status otherwise (ops.py raises from it),
//   - None when an argument is not an ordinary tensor on the current device
//     (another type or device, a rank or dtype without a descriptor, a tensor
//     without storage, ...): ops.py then takes its own path, which raises or
//     handles the case.
// No C++ exception leaves a function: one thrown by torch ends in None.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "cf_hip.h"

namespace {

struct Lib {
  decltype(&cf_paged_decode_workspace_bytes) decode_ws = nullptr;
  decltype(&cf_paged_decode_shared) decode = nullptr;
  decltype(&cf_prefill_chunk_workspace_bytes) prefill_ws = nullptr;
  decltype(&cf_prefill_chunk_fp8) prefill = nullptr;
  decltype(&cf_paged_write) paged_write = nullptr;
  decltype(&cf_paged_gather) paged_gather = nullptr;
  decltype(&cf_kv_write_fp8) kv_write = nullptr;
  decltype(&cf_fp8_scale_quantize) scale_quantize = nullptr;
  decltype(&cf_fp8_dequantize_kv) dequantize_kv = nullptr;
  decltype(&cf_stage_from_host) stage = nullptr;
};
Lib g_lib;
PyObject* g_raw_stream = nullptr;        // device index -> hipStream_t of the current stream
PyObject* g_current_device = nullptr;    // () -> current device index
PyObject* g_workspaces = nullptr;        // {(device index, stream): workspace tensor}, shared with ops.py
PyObject* g_cached_workspace = nullptr;  // (bytes, device) -> workspace tensor

// Thrown to leave a call for ops.py's own path.
struct Slow {};

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return CF_F32;
    case at::kHalf: return CF_F16;
    case at::kBFloat16: return CF_BF16;
    case at::kLong: return CF_I64;
    case at::kInt: return CF_I32;
    case at::kChar: return CF_I8;
    case at::kByte: return CF_U8;
    case at::kFloat8_e4m3fn: return CF_F8E4M3FN;
    default: throw Slow{};
  }
}

// The plain tensor in `o` (torch.Tensor or Parameter, strided).
const at::Tensor& tensor_of(PyObject* o) {
  if (!THPVariable_CheckExact(o)) throw Slow{};
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided) throw Slow{};
  return t;
}

CfTensor describe(const at::Tensor& t) {
  const int64_t rank = t.dim();
  if (rank < 1 || rank > 4) throw Slow{};
  CfTensor d{};
  d.t.device = SFA_ROCM;
  d.t.rank = (int32_t)rank;
  d.t.elem_size = (int32_t)t.element_size();
  const int64_t off = t.storage_offset();
  char* base = (char*)t.data_ptr() - off * t.element_size();
  SFATensorRaw4& r = d.t.r4;  // the union members share their first three fields
  r.allocated = base;
  r.aligned = base;
  r.offset = off;
  int64_t* sizes = &r.offset + 1;
  for (int64_t i = 0; i < rank; ++i) {
    sizes[i] = t.size(i);
    sizes[rank + i] = t.stride(i);
  }
  d.dtype = dtype_code(t.scalar_type());
  return d;
}

// The device of a call: every tensor must be on it and it must be current.
struct Call {
  int device = -1;
  void* stream = nullptr;

  explicit Call(const at::Tensor& first) {
    if (g_raw_stream == nullptr) throw Slow{};
    device = first.get_device();
    PyObject* cur = PyObject_CallNoArgs(g_current_device);
    if (cur == nullptr) throw Slow{};
    const long now = PyLong_AsLong(cur);
    Py_DECREF(cur);
    if (now != device) throw Slow{};
    PyObject* idx = PyLong_FromLong(device);
    if (idx == nullptr) throw Slow{};
    PyObject* s = PyObject_CallOneArg(g_raw_stream, idx);
    Py_DECREF(idx);
    if (s == nullptr) throw Slow{};
    stream = (void*)PyLong_AsUnsignedLongLong(s);
    Py_DECREF(s);
    if (PyErr_Occurred()) throw Slow{};
  }
  CfTensor in(PyObject* o) const {
    const at::Tensor& t = tensor_of(o);
    if (t.get_device() != device) throw Slow{};
    return describe(t);
  }
  // [n] view of a scale tensor of any shape
  CfTensor flat(PyObject* o) const {
    const at::Tensor& t = tensor_of(o);
    if (t.get_device() != device) throw Slow{};
    if (t.dim() == 1) return describe(t);
    if (!t.is_contiguous()) throw Slow{};
    CfTensor d{};
    d.t.device = SFA_ROCM;
    d.t.rank = 1;
    d.t.elem_size = (int32_t)t.element_size();
    d.t.r1.allocated = d.t.r1.aligned = t.data_ptr();
    d.t.r1.sizes[0] = t.numel();
    d.t.r1.strides[0] = 1;
    d.dtype = dtype_code(t.scalar_type());
    return d;
  }
};

int64_t as_int(PyObject* o) {
  if (!PyLong_CheckExact(o)) throw Slow{};
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw Slow{};
  return v;
}

double as_float(PyObject* o) {
  if (!PyFloat_CheckExact(o)) throw Slow{};
  return PyFloat_AS_DOUBLE(o);
}

at::Tensor new_tensor(at::IntArrayRef sizes, at::ScalarType dtype, const at::Tensor& like) {
  return at::empty(sizes, at::TensorOptions().dtype(dtype).device(like.device()));
}

// A workspace of `need` bytes for this device and stream: the caller's, or
// ops.py's cached one (held by a new reference while the call runs).  `any`: the
// caller's may be of another size, for the library to judge.
struct Workspace {
  PyObject* held = nullptr;
  void* ptr = nullptr;
  uint64_t bytes = 0;

  Workspace(PyObject* given, uint64_t need, const Call& call, PyObject* tensor_on_device, bool any = false) {
    if (need == 0) return;
    bytes = need;
    if (given != Py_None) {
      const at::Tensor& t = tensor_of(given);
      const uint64_t has = (uint64_t)(t.numel() * t.element_size());
      if (any) bytes = has;
      else if (has < need) throw Slow{};
      ptr = t.data_ptr();
      return;
    }
    PyObject* key = Py_BuildValue("(iK)", call.device, (unsigned long long)(uintptr_t)call.stream);
    if (key == nullptr) throw Slow{};
    PyObject* ws = PyDict_GetItem(g_workspaces, key);  // borrowed
    Py_DECREF(key);
    if (ws != nullptr && THPVariable_Check(ws) && (uint64_t)THPVariable_Unpack(ws).numel() >= need) {
      Py_INCREF(ws);
      held = ws;
    } else {
      PyObject* dev = PyObject_GetAttrString(tensor_on_device, "device");
      if (dev == nullptr) throw Slow{};
      held = PyObject_CallFunction(g_cached_workspace, "KO", (unsigned long long)need, dev);
      Py_DECREF(dev);
      if (held == nullptr) throw Slow{};
    }
    ptr = THPVariable_Unpack(held).data_ptr();
  }
  ~Workspace() { Py_XDECREF(held); }
  Workspace(const Workspace&) = delete;
  Workspace& operator=(const Workspace&) = delete;
};

// Runs f with the GIL released; held again also where f throws.
template <class F>
int32_t without_gil(F f) {
  struct Release {
    PyThreadState* st = PyEval_SaveThread();
    ~Release() { PyEval_RestoreThread(st); }
  } release;
  return f();
}

// Runs a call body: Slow, torch's exceptions and Python errors become None.
template <class F>
PyObject* guarded(PyObject* const* args, Py_ssize_t n, Py_ssize_t want, F f) {
  if (n != want) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
    return nullptr;
  }
  try {
    return f(args);
  } catch (...) {
    PyErr_Clear();
  }
  Py_RETURN_NONE;
}

const CfTensor* opt(PyObject* o, const CfTensor& d) { return o == Py_None ? nullptr : &d; }

// (q, k_cache, v_cache, block_tables, seq_lens, scale, block_size, k_scale,
// v_scale, partition_tokens, out, workspace, shared_prefix_lens) -> out
PyObject* paged_decode(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded(args, n, 13, [](PyObject* const* a) -> PyObject* {
    const at::Tensor& q = tensor_of(a[0]);
    const at::Tensor& k = tensor_of(a[1]);
    const at::Tensor& bt = tensor_of(a[3]);
    if (q.dim() != 3 || k.dim() != 4 || bt.dim() != 2) throw Slow{};
    const Call call(q);
    const CfTensor dq = call.in(a[0]), dk = call.in(a[1]), dv = call.in(a[2]), dt = call.in(a[3]), dl = call.in(a[4]);
    const double scale = as_float(a[5]);
    const int64_t bs = as_int(a[6]), pt = as_int(a[9]);
    if (bs != (int32_t)bs || pt != (int32_t)pt) throw Slow{};
    CfTensor dks{}, dvs{}, dsh{};
    if (a[7] != Py_None) dks = call.in(a[7]);
    if (a[8] != Py_None) dvs = call.in(a[8]);
    if (a[12] != Py_None) dsh = call.in(a[12]);
    uint64_t need = 0;
    if (g_lib.decode_ws(q.size(0), q.size(1), k.size(2), q.size(2), bt.size(1), (int32_t)bs, (int32_t)pt, &need) !=
        CF_OK)
      throw Slow{};
    const Workspace ws(a[11], need, call, a[0]);
    at::Tensor fresh;
    CfTensor dout;
    if (a[10] == Py_None) {
      fresh = new_tensor(q.sizes(), q.scalar_type(), q);
      dout = describe(fresh);
    } else {
      dout = call.in(a[10]);
    }
    const int32_t rc = without_gil([&] {
      return g_lib.decode(&dq, &dk, &dv, &dt, &dl, opt(a[12], dsh), opt(a[7], dks), opt(a[8], dvs), (float)scale,
                          (int32_t)bs, (int32_t)pt, &dout, ws.ptr, need, call.stream);
    });
    if (rc != CF_OK) return PyLong_FromLong(rc);
    if (a[10] == Py_None) return THPVariable_Wrap(fresh);
    Py_INCREF(a[10]);
    return a[10];
  });
}

// (q, k_cache, v_cache, block_tables, seq_lens, q_start, scale, block_size,
// k_scale, v_scale, out, workspace) -> out
PyObject* prefill_chunk(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded(args, n, 12, [](PyObject* const* a) -> PyObject* {
    const at::Tensor& q = tensor_of(a[0]);
    const at::Tensor& k = tensor_of(a[1]);
    const at::Tensor& bt = tensor_of(a[3]);
    if (q.dim() != 3 || k.dim() != 4 || bt.dim() != 2) throw Slow{};
    const Call call(q);
    const CfTensor dq = call.in(a[0]), dk = call.in(a[1]), dv = call.in(a[2]), dt = call.in(a[3]), dl = call.in(a[4]),
                   ds = call.in(a[5]);
    const double scale = as_float(a[6]);
    const int64_t bs = as_int(a[7]);
    if (bs != (int32_t)bs) throw Slow{};
    CfTensor dks{}, dvs{};
    if (a[8] != Py_None) dks = call.in(a[8]);
    if (a[9] != Py_None) dvs = call.in(a[9]);
    uint64_t need = 0;
    if (g_lib.prefill_ws(q.size(0), bt.size(0), q.size(1), k.size(2), q.size(2), (int32_t)bs, &need) != CF_OK)
      throw Slow{};
    const Workspace ws(a[11], need, call, a[0], true);
    at::Tensor fresh;
    CfTensor dout;
    if (a[10] == Py_None) {
      fresh = new_tensor(q.sizes(), q.scalar_type(), q);
      dout = describe(fresh);
    } else {
      dout = call.in(a[10]);
    }
    const int32_t rc = without_gil([&] {
      return g_lib.prefill(&dq, &dk, &dv, &dt, &dl, &ds, opt(a[8], dks), opt(a[9], dvs), (float)scale, (int32_t)bs,
                           &dout, ws.ptr, ws.bytes, call.stream);
    });
    if (rc != CF_OK) return PyLong_FromLong(rc);
    if (a[10] == Py_None) return THPVariable_Wrap(fresh);
    Py_INCREF(a[10]);
    return a[10];
  });
}

// (x_new, slot_mapping, cache, scale) -> 0
PyObject* paged_write(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded(args, n, 4, [](PyObject* const* a) -> PyObject* {
    const Call call(tensor_of(a[0]));
    const CfTensor dx = call.in(a[0]), ds = call.in(a[1]);
    CfTensor dc = call.in(a[2]), dsc{};
    if (a[3] != Py_None) dsc = call.flat(a[3]);
    return PyLong_FromLong(
        without_gil([&] { return g_lib.paged_write(&dx, &ds, &dc, opt(a[3], dsc), call.stream); }));
  });
}

// (cache, block_tables, seq_len, out_dtype, scale, out) -> out
PyObject* paged_gather(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded(args, n, 6, [](PyObject* const* a) -> PyObject* {
    const at::Tensor& cache = tensor_of(a[0]);
    const at::Tensor& bt = tensor_of(a[1]);
    if (cache.dim() != 4 || bt.dim() != 2) throw Slow{};
    const Call call(cache);
    const CfTensor dc = call.in(a[0]), dt = call.in(a[1]);
    const int64_t seq = as_int(a[2]);
    if (seq < 0) throw Slow{};
    CfTensor dsc{}, dout;
    if (a[4] != Py_None) dsc = call.flat(a[4]);
    at::Tensor fresh;
    if (a[5] == Py_None) {
      at::ScalarType dtype = cache.scalar_type() == at::kFloat8_e4m3fn ? at::kFloat : cache.scalar_type();
      if (a[3] != Py_None) {
        if (!THPDtype_Check(a[3])) throw Slow{};
        dtype = reinterpret_cast<THPDtype*>(a[3])->scalar_type;
      }
      fresh = new_tensor({bt.size(0), seq, cache.size(2), cache.size(3)}, dtype, cache);
      dout = describe(fresh);
    } else {
      dout = call.in(a[5]);
    }
    const int32_t rc =
        without_gil([&] { return g_lib.paged_gather(&dc, &dt, opt(a[4], dsc), &dout, call.stream); });
    if (rc != CF_OK) return PyLong_FromLong(rc);
    if (a[5] == Py_None) return THPVariable_Wrap(fresh);
    Py_INCREF(a[5]);
    return a[5];
  });
}

// (k_new, v_new, slot_mapping, k_cache, v_cache, k_scale, v_scale) -> 0
PyObject* kv_write_fp8(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded(args, n, 7, [](PyObject* const* a) -> PyObject* {
    const Call call(tensor_of(a[0]));
    const CfTensor dk = call.in(a[0]), dv = call.in(a[1]), ds = call.in(a[2]);
    CfTensor dkc = call.in(a[3]), dvc = call.in(a[4]);
    const CfTensor dks = call.flat(a[5]), dvs = call.flat(a[6]);
    return PyLong_FromLong(
        without_gil([&] { return g_lib.kv_write(&dk, &dv, &ds, &dkc, &dvc, &dks, &dvs, call.stream); }));
  });
}

// A contiguous tensor of n elements as [n / (heads * row), heads, row].
CfTensor rows3(const at::Tensor& t, int64_t heads, int64_t row) {
  CfTensor d{};
  d.t.device = SFA_ROCM;
  d.t.rank = 3;
  d.t.elem_size = (int32_t)t.element_size();
  SFATensorRaw3& r = d.t.r3;
  r.allocated = r.aligned = t.data_ptr();
  r.sizes[0] = t.numel() / (heads * row);
  r.sizes[1] = heads;
  r.sizes[2] = row;
  r.strides[0] = heads * row;
  r.strides[1] = row;
  r.strides[2] = 1;
  d.dtype = dtype_code(t.scalar_type());
  return d;
}

// (x, y or None, per_head) -> ((codes, scales), ...) for contiguous tensors of
// one shape and dtype
PyObject* scale_quantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded(args, n, 3, [](PyObject* const* a) -> PyObject* {
    const int count = a[1] == Py_None ? 1 : 2;
    const bool per_head = a[2] == Py_True;
    const at::Tensor& x0 = tensor_of(a[0]);
    const int64_t total = x0.numel();
    if (total == 0 || total % 16 != 0) throw Slow{};
    // (2-D: one head; the library takes 64 heads, and its workspace grows with them)
    if (per_head && (x0.dim() < 3 || x0.size(-1) % 16 != 0 || x0.size(-2) > 64)) throw Slow{};
    const Call call(x0);
    const int64_t heads = per_head ? x0.size(-2) : 1, row = per_head ? x0.size(-1) : 16;
    at::Tensor codes[2], scales[2];
    CfTensor dx[2], dc[2], ds[2];
    for (int i = 0; i < count; ++i) {
      const at::Tensor& x = tensor_of(a[i]);
      if (x.get_device() != call.device || !x.is_contiguous() || x.scalar_type() != x0.scalar_type() ||
          x.sizes() != x0.sizes())
        throw Slow{};
      codes[i] = new_tensor(x.sizes(), at::kFloat8_e4m3fn, x);
      scales[i] = new_tensor({heads}, at::kFloat, x);
      dx[i] = rows3(x, heads, row);
      dc[i] = rows3(codes[i], heads, row);
      ds[i] = describe(scales[i]);
    }
    const at::Tensor ws = new_tensor({4096 * heads}, at::kByte, x0);
    const int32_t rc = without_gil([&] {
      return g_lib.scale_quantize(&dx[0], count == 2 ? &dx[1] : nullptr, &ds[0], count == 2 ? &ds[1] : nullptr, &dc[0],
                                  count == 2 ? &dc[1] : nullptr, ws.data_ptr(), (uint64_t)ws.numel(), call.stream);
    });
    if (rc == CF_ERR_UNSUPPORTED) throw Slow{};
    if (rc != CF_OK) return PyLong_FromLong(rc);
    PyObject* out = PyTuple_New(count);
    if (out == nullptr) throw Slow{};
    for (int i = 0; i < count; ++i)
      PyTuple_SET_ITEM(out, i, Py_BuildValue("(NN)", THPVariable_Wrap(codes[i]), THPVariable_Wrap(scales[i])));
    return out;
  });
}

// (k, v, k_scales, v_scales) -> (f32 k, f32 v) for contiguous tensors of one
// shape with one scale each
PyObject* dequantize_kv(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded(args, n, 4, [](PyObject* const* a) -> PyObject* {
    const at::Tensor& k = tensor_of(a[0]);
    const at::Tensor& v = tensor_of(a[1]);
    const Call call(k);
    if (v.get_device() != call.device || k.sizes() != v.sizes() || !k.is_contiguous() || !v.is_contiguous() ||
        k.numel() % 16 != 0 || k.numel() == 0)
      throw Slow{};
    const CfTensor dks = call.flat(a[2]), dvs = call.flat(a[3]);
    if (dks.t.r1.sizes[0] != 1 || dvs.t.r1.sizes[0] != 1) throw Slow{};
    at::Tensor out[2] = {new_tensor(k.sizes(), at::kFloat, k), new_tensor(k.sizes(), at::kFloat, k)};
    const CfTensor dk = rows3(k, 1, 16), dv = rows3(v, 1, 16);
    CfTensor dko = rows3(out[0], 1, 16), dvo = rows3(out[1], 1, 16);
    const int32_t rc =
        without_gil([&] { return g_lib.dequantize_kv(&dk, &dv, &dks, &dvs, &dko, &dvo, call.stream); });
    if (rc != CF_OK) return PyLong_FromLong(rc);
    return Py_BuildValue("(NN)", THPVariable_Wrap(out[0]), THPVariable_Wrap(out[1]));
  });
}

// (pinned host int32, device int32, requests, blocks): uploads the packed
// tables [requests, blocks] | lengths [requests] | shared-prefix lengths
// [requests] and returns their views of the device buffer
PyObject* stage_tables(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded(args, n, 4, [](PyObject* const* a) -> PyObject* {
    if (!THPVariable_CheckExact(a[0])) throw Slow{};
    const at::Tensor& host = THPVariable_Unpack(a[0]);
    const at::Tensor& dev = tensor_of(a[1]);
    const Call call(dev);
    const int64_t reqs = as_int(a[2]), mb = as_int(a[3]), used = reqs * (mb + 2), words = (used + 3) / 4;
    if (!host.is_cpu() || host.scalar_type() != at::kInt || dev.scalar_type() != at::kInt || !host.is_contiguous() ||
        !dev.is_contiguous() || reqs < 1 || mb < 1 || host.numel() < 4 * words || dev.numel() < 4 * words)
      throw Slow{};
    const int32_t rc = without_gil(
        [&] { return g_lib.stage(host.data_ptr(), dev.data_ptr(), (uint64_t)words * 16, call.stream); });
    if (rc == CF_ERR_INVALID) throw Slow{};
    if (rc != CF_OK) return PyLong_FromLong(rc);
    const int64_t at = dev.storage_offset();
    return Py_BuildValue("(NNN)", THPVariable_Wrap(dev.as_strided({reqs, mb}, {mb, 1}, at)),
                         THPVariable_Wrap(dev.as_strided({reqs}, {1}, at + reqs * mb)),
                         THPVariable_Wrap(dev.as_strided({reqs}, {1}, at + reqs * (mb + 1))));
  });
}

template <class T>
bool take_address(PyObject* addrs, const char* name, T* fn) {
  PyObject* v = PyDict_GetItemString(addrs, name);
  if (v == nullptr) {
    PyErr_Format(PyExc_KeyError, "%s", name);
    return false;
  }
  *fn = (T)(uintptr_t)PyLong_AsUnsignedLongLong(v);
  return !PyErr_Occurred();
}

// bind({entry point: address}, raw_stream, current_device, workspaces, cached_workspace)
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *addrs, *raw, *cur, *wss, *cached;
  if (!PyArg_ParseTuple(args, "O!OOO!O", &PyDict_Type, &addrs, &raw, &cur, &PyDict_Type, &wss, &cached)) return nullptr;
  Lib l;
  if (!take_address(addrs, "cf_paged_decode_workspace_bytes", &l.decode_ws) ||
      !take_address(addrs, "cf_paged_decode_shared", &l.decode) ||
      !take_address(addrs, "cf_prefill_chunk_workspace_bytes", &l.prefill_ws) ||
      !take_address(addrs, "cf_prefill_chunk_fp8", &l.prefill) ||
      !take_address(addrs, "cf_paged_write", &l.paged_write) ||
      !take_address(addrs, "cf_paged_gather", &l.paged_gather) ||
      !take_address(addrs, "cf_kv_write_fp8", &l.kv_write) ||
      !take_address(addrs, "cf_fp8_scale_quantize", &l.scale_quantize) ||
      !take_address(addrs, "cf_fp8_dequantize_kv", &l.dequantize_kv) ||
      !take_address(addrs, "cf_stage_from_host", &l.stage))
    return nullptr;
  g_lib = l;
  for (auto [slot, obj] : {std::pair{&g_raw_stream, raw}, std::pair{&g_current_device, cur},
                           std::pair{&g_workspaces, wss}, std::pair{&g_cached_workspace, cached}}) {
    Py_INCREF(obj);
    Py_XDECREF(*slot);
    *slot = obj;
  }
  Py_RETURN_NONE;
}

#define CF_FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    CF_FAST(paged_decode),
    CF_FAST(prefill_chunk),
    CF_FAST(paged_write),
    CF_FAST(paged_gather),
    CF_FAST(kv_write_fp8),
    CF_FAST(scale_quantize),
    CF_FAST(dequantize_kv),
    CF_FAST(stage_tables),
    {nullptr, nullptr, 0, nullptr},
};
#undef CF_FAST

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fastcall", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fastcall(void) { return PyModule_Create(&kModule); }
