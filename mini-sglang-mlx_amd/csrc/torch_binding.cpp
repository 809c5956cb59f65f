// The Python call path of the operators: argument checks, output and workspace allocation and the
// call into the C ABI (include/msgl_paged_attention.h), as one CPython extension module
// (mini_sglang_amd_kernel/_native.so).  Host code only, compiled by g++ against torch's headers.
//
// Why it is native: at serving's small sizes a layer's kernels take 10-30 us, and the same steps
// written in Python over ctypes took 13-29 us of host time per operator (some twenty attribute
// reads, two torch.empty calls and twenty argument conversions each), so a decode step waited for
// Python and not for the GPU.  The functions here take their arguments positionally, straight from
// mini_sglang_amd_kernel/__init__.py, which holds the documented signatures.
//
// Checks, their order and their texts are the reference's (paged_decode_attention.cpp:25-62,
// paged_prefill_attention.cpp:31-76, store_kv_cache.cpp:22-63, gdn_state.cpp:26-126).
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <initializer_list>
#include <optional>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/msgl_paged_attention.h"

namespace {

using at::Tensor;

[[noreturn]] void fail(const char* op, const std::string& msg) { throw std::runtime_error(std::string(op) + ": " + msg); }

void check_rc(const char* op, int rc) {
  if (rc != MSGL_OK) fail(op, msgl_strerror(rc));
}

const Tensor& tensor(PyObject* o, const char* name) {
  if (!THPVariable_Check(o)) throw c10::TypeError({__func__, __FILE__, __LINE__}, std::string(name) + " must be a torch.Tensor");
  return THPVariable_Unpack(o);
}

struct PyFailure {};  // a Python exception is set

int64_t integer(PyObject* o) {  // what int(o) gives
  PyObject* n = PyNumber_Long(o);
  if (!n) throw PyFailure();
  const long long v = PyLong_AsLongLong(n);
  Py_DECREF(n);
  if (v == -1 && PyErr_Occurred()) throw PyFailure();
  return v;
}

double real(PyObject* o) {  // what float(o) gives
  PyObject* n = PyFloat_CheckExact(o) ? (Py_INCREF(o), o) : PyNumber_Float(o);
  if (!n) throw PyFailure();
  const double v = PyFloat_AS_DOUBLE(n);
  Py_DECREF(n);
  return v;
}

bool truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PyFailure();
  return v != 0;
}

struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// The launch device current (nothing to do in the usual case of one process per GPU) and its stream.
struct OnDevice {
  std::optional<c10::DeviceGuard> guard;
  c10::hip::HIPStream stream;
  explicit OnDevice(const c10::Device& d) : stream(c10::hip::getCurrentHIPStream(d.index())) {
    if (c10::hip::current_device() != d.index()) guard.emplace(d);
  }
  void* ptr() const { return stream.stream(); }
};

c10::Device require_device(const char* op, std::initializer_list<const Tensor*> ts) {
  const c10::Device dev = (*ts.begin())->device();
  if (!dev.is_cuda()) fail(op, "tensors must live on a ROCm GPU device (no CPU implementation exists)");
  for (const Tensor* t : ts)
    if (t->device() != dev) fail(op, "all tensors must be on the same device");
  return dev;
}

int64_t pool_stride0(const char* op, const Tensor& pool, const char* name) {
  if (pool.stride(2) != 1 || pool.stride(1) != pool.size(2))
    fail(op, std::string(name) + " must be contiguous in its (num_kv_heads, head_dim) dimensions");
  // a one-slot pool may report any leading stride
  return pool.size(0) > 1 ? pool.stride(0) : pool.size(1) * pool.size(2);
}

void require_int32(const char* op, const Tensor& t, const char* name) {
  if (t.scalar_type() != at::kInt) fail(op, std::string(name) + " must be int32");
}

Tensor empty(c10::IntArrayRef size, at::ScalarType dtype, const c10::Device& dev) {
  return at::detail::empty_cuda(size, dtype, dev, std::nullopt);
}

// Scratch from torch's caching allocator, taken on the launch stream: safe to drop right after the
// launch because the allocator reuses a block in stream order.
Tensor scratch(size_t bytes, const c10::Device& dev) {
  return bytes ? empty({static_cast<int64_t>(bytes)}, at::kByte, dev) : Tensor();
}

void* data_or_null(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
const int32_t* ints(const Tensor& t) { return static_cast<const int32_t*>(t.data_ptr()); }

// ---- opt-in index validation: mini_sglang_amd_kernel._run_checks, given at import ---------------
PyObject* g_run_checks = nullptr;

// `validate` as the caller wrote it; None asks the environment.  No Python runs unless it is on.
void debug_checks(PyObject* validate, const char* op, std::initializer_list<PyObject*> args) {
  if (validate == Py_None) {
    const char* env = std::getenv("MSGL_DEBUG_CHECKS");
    if (!env || !*env || std::strcmp(env, "0") == 0) return;
  } else if (!truth(validate)) {
    return;
  }
  if (!g_run_checks) return;
  PyObject* tuple = PyTuple_New(static_cast<Py_ssize_t>(args.size()) + 2);
  if (!tuple) throw PyFailure();
  Py_INCREF(validate);
  PyTuple_SET_ITEM(tuple, 0, validate);
  PyTuple_SET_ITEM(tuple, 1, PyUnicode_FromString(op));
  Py_ssize_t i = 2;
  for (PyObject* a : args) {
    Py_INCREF(a);
    PyTuple_SET_ITEM(tuple, i++, a);
  }
  PyObject* r = PyObject_CallObject(g_run_checks, tuple);
  Py_DECREF(tuple);
  if (!r) throw PyFailure();
  Py_DECREF(r);
}

template <typename F>
PyObject* guarded(PyObject* const* args, Py_ssize_t n, Py_ssize_t want, F&& f) {
  HANDLE_TH_ERRORS
  if (n != want) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
    return nullptr;
  }
  try {
    return f(args);
  } catch (const PyFailure&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

PyObject* none() { Py_RETURN_NONE; }

// ---- store_kv_cache(k_cache, v_cache, indices, k, v, validate) ----------------------------------
PyObject* store_kv_cache(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 6, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "store_kv_cache";
    const Tensor &kc = tensor(a[0], "k_cache"), &vc = tensor(a[1], "v_cache"), &idx = tensor(a[2], "indices");
    const Tensor &k = tensor(a[3], "k"), &v = tensor(a[4], "v");
    if (kc.dim() != 3 || vc.dim() != 3) fail(op, "k_cache and v_cache must be 3D (num_pages, num_kv_heads, head_dim)");
    if (idx.dim() != 1) fail(op, "indices must be 1D");
    if (k.dim() != 3 || v.dim() != 3) fail(op, "k and v must be 3D (length, num_kv_heads, head_dim)");
    const auto dt = kc.scalar_type();
    if (vc.scalar_type() != dt || k.scalar_type() != dt || v.scalar_type() != dt)
      fail(op, "k_cache, v_cache, k, v must have the same dtype");
    require_int32(op, idx, "indices");
    const int64_t pages = kc.size(0), heads = kc.size(1), d = kc.size(2), length = idx.size(0);
    if (d % 4 != 0) fail(op, "head_dim must be a multiple of 4");
    if (vc.sizes() != kc.sizes()) fail(op, "v_cache shape must match k_cache");
    if (k.size(0) != length || k.size(1) != heads || k.size(2) != d || v.sizes() != k.sizes())
      fail(op, "k and v shape must be (length, num_kv_heads, head_dim)");
    const int64_t esz = kc.element_size();
    if (esz != 2 && esz != 4) fail(op, "unsupported dtype, must be float16, bfloat16 or float32");
    const c10::Device dev = require_device(op, {&kc, &vc, &idx, &k, &v});
    if (length == 0) return none();
    debug_checks(a[5], op, {a[2], a[0]});
    const int64_t row = heads * d, kcs = pool_stride0(op, kc, "k_cache"), vcs = pool_stride0(op, vc, "v_cache");
    int rc;
    {
      NoGil nogil;
      OnDevice on(dev);
      auto source = [d](const Tensor& t) { return t.stride(2) != 1 || t.stride(1) != d ? t.contiguous() : t; };
      const Tensor ks = source(k), vs = source(v), ix = idx.contiguous();
      rc = msgl_store_kv_cache(kc.data_ptr(), vc.data_ptr(), ints(ix), ks.data_ptr(), vs.data_ptr(), length, heads, d,
                               pages, kcs, vcs, length > 1 ? ks.stride(0) : row, length > 1 ? vs.stride(0) : row,
                               static_cast<int32_t>(esz), on.ptr());
    }
    check_rc(op, rc);
    return none();
  });
}

int32_t attention_dtype(const char* op, const Tensor& q, const Tensor& kc, const Tensor& vc, bool half_ok) {
  const auto dt = q.scalar_type();
  if (dt != at::kBFloat16 && dt != at::kHalf) fail(op, "unsupported dtype, must be float16 or bfloat16");
  if (kc.scalar_type() != dt || vc.scalar_type() != dt) fail(op, "q, k_cache and v_cache must have the same dtype");
  // float16 exists for decode only, as in the reference: its prefill kernel is instantiated for
  // bfloat16 alone (paged_prefill_attention.metal:646-647)
  if (dt == at::kHalf && !half_ok) fail(op, "unsupported dtype, the prefill kernel is bfloat16 only");
  return dt == at::kHalf ? MSGL_DTYPE_F16 : MSGL_DTYPE_BF16;
}

// ---- paged_decode_attention(q, k_cache, v_cache, kv_indptr, kv_indices, num_kv_splits, sm_scale,
//                             max_kv_splits, validate) -> out --------------------------------------
PyObject* paged_decode_attention(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 9, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "paged_decode_attention";
    const Tensor &q = tensor(a[0], "q"), &kc = tensor(a[1], "k_cache"), &vc = tensor(a[2], "v_cache");
    const Tensor &ip = tensor(a[3], "kv_indptr"), &ix = tensor(a[4], "kv_indices"), &ns = tensor(a[5], "num_kv_splits");
    if (q.dim() != 3) fail(op, "q must be 3D (batch, num_q_heads, head_dim)");
    if (kc.dim() != 3 || vc.dim() != 3) fail(op, "k_cache and v_cache must be 3D (num_pages, num_kv_heads, head_dim)");
    if (ip.dim() != 1 || ix.dim() != 1 || ns.dim() != 1) fail(op, "kv_indptr, kv_indices, num_kv_splits must be 1D");
    const int64_t batch = q.size(0), n_q = q.size(1), d = q.size(2), n_kv = kc.size(1);
    if (d != 128 && d != 256) fail(op, "head_dim must be 128 or 256");
    if (n_kv == 0 || n_q % n_kv != 0) fail(op, "num_q_heads must be a multiple of num_kv_heads");
    if (n_q / n_kv > 16) fail(op, "only q_heads/kv_heads <= 16 is supported");
    if (kc.size(2) != d || vc.size(2) != d) fail(op, "cache head_dim must match q head_dim");
    if (vc.size(1) != n_kv) fail(op, "v_cache shape must match k_cache");
    const int32_t dtype = attention_dtype(op, q, kc, vc, true);
    require_int32(op, ip, "kv_indptr");
    require_int32(op, ix, "kv_indices");
    require_int32(op, ns, "num_kv_splits");
    if (ip.size(0) != batch + 1) fail(op, "kv_indptr must have batch + 1 entries");
    if (ns.size(0) != batch) fail(op, "num_kv_splits must have batch entries");
    const c10::Device dev = require_device(op, {&q, &kc, &vc, &ip, &ix, &ns});
    const float scale = static_cast<float>(real(a[6]));
    const int32_t max_splits = static_cast<int32_t>(integer(a[7]));
    if (batch > 0) debug_checks(a[8], op, {a[3], a[4], a[1]});
    const int64_t total_kv = ix.size(0);
    Tensor out;
    int rc = MSGL_OK;
    {
      NoGil nogil;
      OnDevice on(dev);
      out = empty({batch, n_q, d}, q.scalar_type(), dev);
      if (batch > 0) {
        const int64_t kcs = pool_stride0(op, kc, "k_cache"), vcs = pool_stride0(op, vc, "v_cache");
        const Tensor qc = q.contiguous(), ipc = ip.contiguous(), ixc = ix.contiguous(), nsc = ns.contiguous();
        const size_t bytes = msgl_paged_decode_workspace_bytes(batch, total_kv, n_q, n_kv, d);
        const Tensor ws = scratch(bytes, dev);
        rc = msgl_paged_decode_attention(qc.data_ptr(), kc.data_ptr(), vc.data_ptr(), ints(ipc), ints(ixc), ints(nsc),
                                         out.data_ptr(), data_or_null(ws), bytes, batch, total_kv, n_q, n_kv, d,
                                         kc.size(0), kcs, vcs, scale, max_splits, dtype, on.ptr());
      }
    }
    check_rc(op, rc);
    return THPVariable_Wrap(std::move(out));
  });
}

// ---- paged_prefill_attention(q, k_cache, v_cache, qo_indptr, kv_indptr, kv_indices, prefix_lens,
//        sm_scale, max_len_extend, is_cross_attention, sliding_window_size, validate) -> out -------
PyObject* paged_prefill_attention(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 12, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "paged_prefill_attention";
    const Tensor &q = tensor(a[0], "q"), &kc = tensor(a[1], "k_cache"), &vc = tensor(a[2], "v_cache");
    const Tensor &qp = tensor(a[3], "qo_indptr"), &ip = tensor(a[4], "kv_indptr"), &ix = tensor(a[5], "kv_indices");
    const Tensor& pl = tensor(a[6], "prefix_lens");
    if (q.dim() != 3) fail(op, "q must be 3D (total_q_tokens, num_q_heads, head_dim)");
    if (kc.dim() != 3 || vc.dim() != 3) fail(op, "k_cache and v_cache must be 3D (num_pages, num_kv_heads, head_dim)");
    if (qp.dim() != 1 || ip.dim() != 1 || ix.dim() != 1 || pl.dim() != 1)
      fail(op, "qo_indptr, kv_indptr, kv_indices, prefix_lens must be 1D");
    const int64_t total_q = q.size(0), n_q = q.size(1), d = q.size(2), n_kv = kc.size(1);
    if (d != 128 && d != 256) fail(op, "head_dim must be 128 or 256");
    if (n_kv == 0 || n_q % n_kv != 0) fail(op, "num_q_heads must be a multiple of num_kv_heads");
    if (kc.size(2) != d || vc.size(2) != d) fail(op, "cache head_dim must match q head_dim");
    const int64_t window = integer(a[10]);
    if (window < 0) fail(op, "sliding_window_size must be >= 0");
    const int64_t batch = qp.size(0) - 1;
    if (batch <= 0) fail(op, "batch must be > 0");
    if (vc.size(1) != n_kv) fail(op, "v_cache shape must match k_cache");
    const int32_t dtype = attention_dtype(op, q, kc, vc, false);
    require_int32(op, qp, "qo_indptr");
    require_int32(op, ip, "kv_indptr");
    require_int32(op, ix, "kv_indices");
    require_int32(op, pl, "prefix_lens");
    if (ip.size(0) != batch + 1 || pl.size(0) != batch) fail(op, "kv_indptr / prefix_lens length must match qo_indptr");
    const c10::Device dev = require_device(op, {&q, &kc, &vc, &qp, &ip, &ix, &pl});
    const float scale = static_cast<float>(real(a[7]));
    const int64_t max_extend = integer(a[8]);
    const bool cross = truth(a[9]);
    if (total_q > 0) debug_checks(a[11], op, {a[3], a[4], a[5], a[0], a[1]});
    const int64_t total_kv = ix.size(0);
    Tensor out;
    int rc = MSGL_OK;
    {
      NoGil nogil;
      OnDevice on(dev);
      out = empty({total_q, n_q, d}, q.scalar_type(), dev);
      if (total_q > 0) {
        const int64_t kcs = pool_stride0(op, kc, "k_cache"), vcs = pool_stride0(op, vc, "v_cache");
        const Tensor qc = q.contiguous(), qpc = qp.contiguous(), ipc = ip.contiguous(), ixc = ix.contiguous(),
                     plc = pl.contiguous();
        const size_t bytes = msgl_paged_prefill_workspace_bytes(batch, total_q, total_kv, n_q, n_kv, d, max_extend);
        const Tensor ws = scratch(bytes, dev);
        rc = msgl_paged_prefill_attention(qc.data_ptr(), kc.data_ptr(), vc.data_ptr(), ints(qpc), ints(ipc), ints(ixc),
                                          ints(plc), out.data_ptr(), data_or_null(ws), bytes, batch, total_q, total_kv,
                                          n_q, n_kv, d, kc.size(0), kcs, vcs, scale, static_cast<int32_t>(max_extend),
                                          cross ? 1 : 0, static_cast<int32_t>(window), dtype, on.ptr());
      }
    }
    check_rc(op, rc);
    return THPVariable_Wrap(std::move(out));
  });
}

// ---- attention metadata ---------------------------------------------------------------------------
// One allocation, six views (an allocation per array costs more host time than the kernel).
struct MetadataOut {
  Tensor buf;
  int64_t batch, total_q, total_kv;
  MetadataOut(int64_t b, int64_t tq, int64_t tkv, const c10::Device& dev) : batch(b), total_q(tq), total_kv(tkv) {
    buf = empty({2 * (b + 1) + 2 * b + tq + tkv}, at::kInt, dev);
  }
  // kv_indptr, qo_indptr, prefix_lens, num_kv_splits, positions, kv_indices
  int64_t offset(int i) const {
    const int64_t at[6] = {0, batch + 1, 2 * (batch + 1), 2 * (batch + 1) + batch, 2 * (batch + 1) + 2 * batch,
                           2 * (batch + 1) + 2 * batch + total_q};
    return at[i];
  }
  int64_t count(int i) const { return i < 2 ? batch + 1 : i < 4 ? batch : i == 4 ? total_q : total_kv; }
  int32_t* ptr(int i) const { return static_cast<int32_t*>(buf.data_ptr()) + offset(i); }
  PyObject* dict() const {
    static const char* const names[6] = {"kv_indptr", "qo_indptr", "prefix_lens", "num_kv_splits", "positions", "kv_indices"};
    PyObject* d = PyDict_New();
    if (!d) throw PyFailure();
    for (int i = 0; i < 6; ++i) {
      PyObject* t = THPVariable_Wrap(buf.narrow(0, offset(i), count(i)));
      const int rc = t ? PyDict_SetItemString(d, names[i], t) : -1;
      Py_XDECREF(t);
      if (rc < 0) {
        Py_DECREF(d);
        throw PyFailure();
      }
    }
    return d;
  }
};

void check_table(const char* op, const Tensor& table) {
  if (table.dim() != 2) fail(op, "page_table must be 2D (rows, max_seq_len)");
  require_int32(op, table, "page_table");
  if (table.stride(1) != 1) fail(op, "page_table must be contiguous in its last dimension");
}

// build_attention_metadata(page_table, table_rows, kv_lens, extend_lens | None, total_kv, total_q | None,
//                          max_kv_splits) -> dict
PyObject* build_attention_metadata(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 7, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "build_attention_metadata";
    const Tensor &table = tensor(a[0], "page_table"), &rows = tensor(a[1], "table_rows"), &kv = tensor(a[2], "kv_lens");
    check_table(op, table);
    const bool has_ext = a[3] != Py_None;
    const Tensor& ext = has_ext ? tensor(a[3], "extend_lens") : kv;
    if (rows.dim() != 1) fail(op, "table_rows must be 1D");
    if (kv.dim() != 1) fail(op, "kv_lens must be 1D");
    if (ext.dim() != 1) fail(op, "extend_lens must be 1D");
    const c10::Device dev = require_device(op, {&table, &rows, &kv, &ext});
    require_int32(op, rows, "table_rows");
    require_int32(op, kv, "kv_lens");
    require_int32(op, ext, "extend_lens");
    const int64_t batch = kv.size(0);
    if (rows.size(0) != batch) fail(op, "table_rows and kv_lens must have the same length");
    if (ext.size(0) != batch) fail(op, "extend_lens and kv_lens must have the same length");
    const int64_t total_kv = integer(a[4]);
    const int64_t total_q = a[5] != Py_None ? integer(a[5]) : has_ext ? 0 : batch;
    if (total_kv < 0 || total_q < 0) fail(op, "total_kv and total_q must be >= 0");
    const int32_t max_splits = static_cast<int32_t>(integer(a[6]));
    std::optional<MetadataOut> out;
    int rc;
    {
      NoGil nogil;
      OnDevice on(dev);
      out.emplace(batch, total_q, total_kv, dev);
      const Tensor rc_ = rows.contiguous(), kvc = kv.contiguous(), exc = ext.contiguous();
      const int64_t n_rows = table.size(0), width = table.size(1);
      rc = msgl_build_attention_metadata(ints(table), n_rows > 1 ? table.stride(0) : width, n_rows, width, ints(rc_),
                                         ints(kvc), has_ext ? ints(exc) : nullptr, batch, out->ptr(0), out->ptr(5),
                                         total_kv, out->ptr(1), out->ptr(2), out->ptr(4), total_q, out->ptr(3),
                                         max_splits, on.ptr());
    }
    check_rc(op, rc);
    return out->dict();
  });
}

void int_list(PyObject* o, std::vector<int32_t>& to) {
  PyObject* fast = PySequence_Fast(o, "a sequence of ints is wanted");
  if (!fast) throw PyFailure();
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(fast);
  for (Py_ssize_t i = 0; i < n; ++i) {
    const long v = PyLong_AsLong(PySequence_Fast_GET_ITEM(fast, i));
    if ((v == -1 && PyErr_Occurred()) || v != static_cast<int32_t>(v)) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_OverflowError, "length or table row out of int32 range");
      Py_DECREF(fast);
      throw PyFailure();
    }
    to.push_back(static_cast<int32_t>(v));
  }
  Py_DECREF(fast);
}

// build_metadata_from_host(page_table, table_rows, kv_lens, extend_lens | None, max_kv_splits) -> dict
// The same arrays from the scheduler's own lists of ints.  Up to MSGL_METADATA_HOST_BATCH requests
// travel as kernel arguments (no copy, nothing waited for); more go through pinned memory.
PyObject* build_metadata_from_host(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 5, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "build_attention_metadata";
    const Tensor& table = tensor(a[0], "page_table");
    check_table(op, table);
    const c10::Device dev = require_device(op, {&table});
    const bool has_ext = a[3] != Py_None;
    std::vector<int32_t> host;
    int_list(a[1], host);
    const int64_t batch = static_cast<int64_t>(host.size());
    host.reserve(3 * batch);
    int_list(a[2], host);
    if (static_cast<int64_t>(host.size()) != 2 * batch) fail(op, "table_rows and kv_lens must have the same length");
    if (has_ext) int_list(a[3], host);
    if (has_ext && static_cast<int64_t>(host.size()) != 3 * batch) fail(op, "extend_lens and kv_lens must have the same length");
    const int32_t max_splits = static_cast<int32_t>(integer(a[4]));
    int64_t total_kv = 0, total_q = has_ext ? 0 : batch;
    for (int64_t i = 0; i < batch; ++i) {
      total_kv += host[batch + i];
      if (has_ext) total_q += host[2 * batch + i];
    }
    if (total_kv < 0 || total_q < 0) fail(op, "total_kv and total_q must be >= 0");
    std::optional<MetadataOut> out;
    int rc;
    {
      NoGil nogil;
      OnDevice on(dev);
      out.emplace(batch, total_q, total_kv, dev);
      const int64_t n_rows = table.size(0), width = table.size(1), stride0 = n_rows > 1 ? table.stride(0) : width;
      if (batch <= MSGL_METADATA_HOST_BATCH) {
        rc = msgl_build_attention_metadata_host(ints(table), stride0, n_rows, width, host.data(), host.data() + batch,
                                                has_ext ? host.data() + 2 * batch : nullptr, batch, out->ptr(0),
                                                out->ptr(5), total_kv, out->ptr(1), out->ptr(2), out->ptr(4), total_q,
                                                out->ptr(3), max_splits, on.ptr());
      } else {
        const int64_t n = static_cast<int64_t>(host.size());
        const Tensor pinned = at::empty({n}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
        std::memcpy(pinned.data_ptr(), host.data(), n * sizeof(int32_t));
        const Tensor up = pinned.to(dev, at::kInt, /*non_blocking=*/true);
        rc = msgl_build_attention_metadata(ints(table), stride0, n_rows, width, ints(up), ints(up) + batch,
                                           has_ext ? ints(up) + 2 * batch : nullptr, batch, out->ptr(0), out->ptr(5),
                                           total_kv, out->ptr(1), out->ptr(2), out->ptr(4), total_q, out->ptr(3),
                                           max_splits, on.ptr());
      }
    }
    check_rc(op, rc);
    return out->dict();
  });
}

int64_t heads_stride0(const char* op, const Tensor& t, const char* name) {
  if (t.dim() != 3) fail(op, std::string(name) + " must be 3D (tokens, heads, head_dim)");
  if (t.stride(2) != 1 || t.stride(1) != t.size(2))
    fail(op, std::string(name) + " must be contiguous in its (heads, head_dim) dimensions");
  return t.size(0) > 1 ? t.stride(0) : t.size(1) * t.size(2);
}

// ---- qk_norm_rope_store(q, k, v, q_weight, k_weight, positions, out_loc, k_cache, v_cache, eps,
//                         rope_base, validate) -> rotated q -----------------------------------------
PyObject* qk_norm_rope_store(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 12, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "qk_norm_rope_store";
    const Tensor &q = tensor(a[0], "q"), &k = tensor(a[1], "k"), &v = tensor(a[2], "v"), &qw = tensor(a[3], "q_weight");
    const Tensor &kw = tensor(a[4], "k_weight"), &pos = tensor(a[5], "positions"), &loc = tensor(a[6], "out_loc");
    const Tensor &kc = tensor(a[7], "k_cache"), &vc = tensor(a[8], "v_cache");
    const c10::Device dev = require_device(op, {&q, &k, &v, &qw, &kw, &pos, &loc, &kc, &vc});
    const int64_t qs = heads_stride0(op, q, "q"), ks = heads_stride0(op, k, "k"), vs = heads_stride0(op, v, "v");
    const int64_t tokens = q.size(0), n_q = q.size(1), d = q.size(2), n_kv = k.size(1);
    if (d != 128 && d != 256) fail(op, "head_dim must be 128 or 256");
    if (k.size(0) != tokens || k.size(2) != d || v.sizes() != k.sizes())
      fail(op, "k and v shape must be (tokens, num_kv_heads, head_dim)");
    if (kc.dim() != 3 || kc.size(1) != n_kv || kc.size(2) != d || vc.sizes() != kc.sizes())
      fail(op, "k_cache and v_cache must be (num_pages, num_kv_heads, head_dim)");
    const std::pair<const Tensor*, const char*> typed[] = {{&q, "q"}, {&k, "k"}, {&v, "v"}, {&kc, "k_cache"},
                                                           {&vc, "v_cache"}, {&qw, "q_weight"}, {&kw, "k_weight"}};
    for (const auto& [t, name] : typed)
      if (t->scalar_type() != at::kBFloat16) fail(op, std::string(name) + " must be bfloat16");
    if (qw.dim() != 1 || qw.size(0) != d || kw.dim() != 1 || kw.size(0) != d) fail(op, "q_weight and k_weight must be (head_dim,)");
    require_int32(op, pos, "positions");
    require_int32(op, loc, "out_loc");
    if (pos.dim() < 1 || loc.dim() < 1 || pos.size(0) != tokens || loc.size(0) != tokens)
      fail(op, "positions and out_loc length must match q length");
    const float eps = static_cast<float>(real(a[9])), base = static_cast<float>(real(a[10]));
    debug_checks(a[11], op, {a[6], a[7]});
    const int64_t kcs = pool_stride0(op, kc, "k_cache"), vcs = pool_stride0(op, vc, "v_cache");
    Tensor out;
    int rc;
    {
      NoGil nogil;
      OnDevice on(dev);
      out = empty({tokens, n_q, d}, at::kBFloat16, dev);
      const Tensor qwc = qw.contiguous(), kwc = kw.contiguous(), pc = pos.contiguous(), lc = loc.contiguous();
      rc = msgl_qk_norm_rope_store(q.data_ptr(), k.data_ptr(), v.data_ptr(), qs, ks, vs, qwc.data_ptr(), kwc.data_ptr(),
                                   ints(pc), ints(lc), out.data_ptr(), kc.data_ptr(), vc.data_ptr(), kcs, vcs, kc.size(0),
                                   tokens, n_q, n_kv, d, eps, base, MSGL_DTYPE_BF16, on.ptr());
    }
    check_rc(op, rc);
    return THPVariable_Wrap(std::move(out));
  });
}

// ---- decode_step(q, k, v, q_weight | None, k_weight | None, positions | None, out_loc, k_cache, v_cache, kv_indptr,
//                  kv_indices, num_kv_splits, sm_scale, eps, rope_base) -> out or None ------------------
// Decode attention with the store (or norm, rotary embedding and store) inside, None where that is not the way: the
// caller then makes the two calls, which check what is refused here and say why, and take every form.
PyObject* decode_step(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 15, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "decode_step";
    const bool norm = a[3] != Py_None;
    for (int i = 0; i < 12; ++i)
      if (!THPVariable_Check(a[i]) && (norm || i < 3 || i > 5)) return none();
    if (const char* env = std::getenv("MSGL_DEBUG_CHECKS"); env && *env && std::strcmp(env, "0") != 0) return none();
    auto t = [&](int i) -> const Tensor& { return THPVariable_Unpack(a[i]); };
    const Tensor &q = t(0), &k = t(1), &v = t(2), &loc = t(6), &kc = t(7), &vc = t(8), &ip = t(9), &ix = t(10), &ns = t(11);
    if (q.dim() != 3 || k.dim() != 3 || kc.dim() != 3 || vc.dim() != 3) return none();
    const int64_t batch = q.size(0), n_q = q.size(1), d = q.size(2), n_kv = k.size(1), slots = kc.size(0);
    const auto dt = q.scalar_type();
    if (batch == 0 || slots == 0 || n_kv == 0 || n_q == 0 || (dt != at::kBFloat16 && (norm || dt != at::kHalf))) return none();
    const c10::Device dev = q.device();
    if (!dev.is_cuda()) return none();
    auto same = [&](const Tensor& x) { return x.scalar_type() == dt && x.device() == dev; };
    auto ints_of = [&](const Tensor& x, int64_t n) {
      return x.dim() == 1 && x.size(0) == n && x.scalar_type() == at::kInt && x.device() == dev && x.is_contiguous();
    };
    auto rows = [&](const Tensor& x) {
      return x.stride(2) == 1 && x.stride(1) == d && (batch == 1 || (x.stride(0) >= x.size(1) * d && x.stride(0) % 8 == 0)) &&
             reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0;
    };
    auto pool = [&](const Tensor& x) {
      return x.stride(2) == 1 && x.stride(1) == d && (slots == 1 || (x.stride(0) >= n_kv * d && x.stride(0) % 8 == 0)) &&
             reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0;
    };
    const c10::IntArrayRef pool_size = kc.sizes();
    if (!same(k) || !same(v) || !same(kc) || !same(vc) || k.size(0) != batch || k.size(2) != d || v.sizes() != k.sizes() ||
        pool_size[1] != n_kv || pool_size[2] != d || vc.sizes() != pool_size || !rows(q) || !rows(k) || !rows(v) || !pool(kc) ||
        !pool(vc) || !ints_of(loc, batch) || !ints_of(ip, batch + 1) || !ints_of(ix, ix.numel()) || !ints_of(ns, batch))
      return none();
    float eps = 0.f, base = 0.f;
    if (norm) {
      auto weight = [&](const Tensor& x) {
        return same(x) && x.dim() == 1 && x.size(0) == d && x.is_contiguous() && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0;
      };
      if (!weight(t(3)) || !weight(t(4)) || !ints_of(t(5), batch)) return none();
      eps = static_cast<float>(real(a[13]));
      base = static_cast<float>(real(a[14]));
      if (!(base > 1.0f) || !(eps >= 0.0f)) return none();
    }
    const size_t bytes = msgl_decode_step_workspace_bytes(batch, ix.size(0), n_q, n_kv, d, norm ? 1 : 0);
    if (bytes == 0) return none();
    const float scale = static_cast<float>(real(a[12]));
    auto stride0 = [](const Tensor& x) { return x.size(0) > 1 ? x.stride(0) : x.size(1) * x.size(2); };
    Tensor out;
    int rc;
    {
      NoGil nogil;
      OnDevice on(dev);
      out = empty({batch, n_q, d}, dt, dev);
      const Tensor ws = scratch(bytes, dev);
      rc = msgl_decode_step(q.data_ptr(), k.data_ptr(), v.data_ptr(), stride0(q), stride0(k), stride0(v),
                            norm ? t(3).data_ptr() : nullptr, norm ? t(4).data_ptr() : nullptr, norm ? ints(t(5)) : nullptr,
                            ints(loc), kc.data_ptr(), vc.data_ptr(), ints(ip), ints(ix), out.data_ptr(), ws.data_ptr(), bytes,
                            batch, ix.size(0), n_q, n_kv, d, slots, stride0(kc), stride0(vc), scale, eps, base,
                            dt == at::kHalf ? MSGL_DTYPE_F16 : MSGL_DTYPE_BF16, on.ptr());
    }
    check_rc(op, rc);
    return THPVariable_Wrap(std::move(out));
  });
}

// ---- extend_step(q, k, v, out_loc, k_cache, v_cache, qo_indptr, kv_indptr, kv_indices, prefix_lens, sm_scale,
//                  max_len_extend, is_cross_attention, sliding_window_size, own_slots) -> out or None ----
// As decode_step, for prefill metadata; the two launches are made here too where one is not the way, and always
// without own_slots.
PyObject* extend_step(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 15, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "extend_step";
    for (int i = 0; i < 10; ++i)
      if (!THPVariable_Check(a[i])) return none();
    auto t = [&](int i) -> const Tensor& { return THPVariable_Unpack(a[i]); };
    const Tensor &q = t(0), &k = t(1), &v = t(2), &loc = t(3), &kc = t(4), &vc = t(5), &qp = t(6), &ip = t(7), &ix = t(8), &pl = t(9);
    if (q.dim() != 3 || k.dim() != 3 || kc.dim() != 3 || vc.dim() != 3 || qp.dim() != 1 || ix.dim() != 1) return none();
    const int64_t total = q.size(0), n_q = q.size(1), d = q.size(2), n_kv = k.size(1), slots = kc.size(0), batch = qp.size(0) - 1;
    const c10::Device dev = q.device();
    if (total == 0 || batch <= 0 || slots == 0 || q.scalar_type() != at::kBFloat16 || !dev.is_cuda()) return none();
    const int64_t max_extend = integer(a[11]), window = integer(a[13]);
    const bool cross = truth(a[12]), own_slots = truth(a[14]);
    if (window < 0 || window > 0x7fffffff || max_extend <= 0 || max_extend > 0x7fffffff || (d != 128 && d != 256) || n_kv == 0 ||
        n_q == 0 || n_q % n_kv != 0)
      return none();
    if (const char* env = std::getenv("MSGL_DEBUG_CHECKS"); env && *env && std::strcmp(env, "0") != 0) return none();
    auto same = [&](const Tensor& x) { return x.scalar_type() == at::kBFloat16 && x.device() == dev; };
    auto ints_of = [&](const Tensor& x, int64_t n) {
      return x.dim() == 1 && x.size(0) == n && x.scalar_type() == at::kInt && x.device() == dev && x.is_contiguous();
    };
    auto rows = [&](const Tensor& x) {
      return x.stride(2) == 1 && x.stride(1) == d && (x.size(0) == 1 || (x.stride(0) >= x.size(1) * d && x.stride(0) % 8 == 0)) &&
             reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0;
    };
    const c10::IntArrayRef pool_size = kc.sizes();
    if (!same(k) || !same(v) || !same(kc) || !same(vc) || k.size(0) != total || k.size(2) != d || v.sizes() != k.sizes() ||
        pool_size[1] != n_kv || pool_size[2] != d || vc.sizes() != pool_size || !q.is_contiguous() || !rows(q) || !rows(k) ||
        !rows(v) || !rows(kc) || !rows(vc) || !ints_of(loc, total) || !ints_of(qp, batch + 1) || !ints_of(ip, batch + 1) ||
        !ints_of(ix, ix.numel()) || !ints_of(pl, batch))
      return none();
    const float scale = static_cast<float>(real(a[10]));
    auto stride0 = [](const Tensor& x) { return x.size(0) > 1 ? x.stride(0) : x.size(1) * x.size(2); };
    Tensor out;
    int rc;
    {
      NoGil nogil;
      OnDevice on(dev);
      out = empty({total, n_q, d}, at::kBFloat16, dev);
      const int64_t ks0 = stride0(k), vs0 = stride0(v), kcs = stride0(kc), vcs = stride0(vc);
      size_t bytes = !own_slots ? 0 : msgl_extend_step_workspace_bytes(batch, total, ix.size(0), n_q, n_kv, d, max_extend, cross,
                                                                       static_cast<int32_t>(window));
      if (bytes > 0) {
        const Tensor ws = scratch(bytes, dev);
        rc = msgl_extend_step(q.data_ptr(), k.data_ptr(), v.data_ptr(), ks0, vs0, ints(loc), kc.data_ptr(), vc.data_ptr(), ints(qp),
                              ints(ip), ints(ix), ints(pl), out.data_ptr(), ws.data_ptr(), bytes, batch, total, ix.size(0), n_q,
                              n_kv, d, slots, kcs, vcs, scale, static_cast<int32_t>(max_extend), cross ? 1 : 0,
                              static_cast<int32_t>(window), MSGL_DTYPE_BF16, on.ptr());
      } else {
        rc = msgl_store_kv_cache(kc.data_ptr(), vc.data_ptr(), ints(loc), k.data_ptr(), v.data_ptr(), total, n_kv, d, slots, kcs,
                                 vcs, ks0, vs0, 2, on.ptr());
        if (rc == MSGL_OK) {
          bytes = msgl_paged_prefill_workspace_bytes(batch, total, ix.size(0), n_q, n_kv, d, max_extend);
          const Tensor ws = scratch(bytes, dev);
          rc = msgl_paged_prefill_attention(q.data_ptr(), kc.data_ptr(), vc.data_ptr(), ints(qp), ints(ip), ints(ix), ints(pl),
                                            out.data_ptr(), data_or_null(ws), bytes, batch, total, ix.size(0), n_q, n_kv, d, slots,
                                            kcs, vcs, scale, static_cast<int32_t>(max_extend), cross ? 1 : 0,
                                            static_cast<int32_t>(window), MSGL_DTYPE_BF16, on.ptr());
        }
      }
    }
    check_rc(op, rc);
    return THPVariable_Wrap(std::move(out));
  });
}

// ---- gdn_state_inplace(q, k, v, g, beta, state, slot_ids, qo_indptr, single_token_mode) -> y -------
PyObject* gdn_state_inplace(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 9, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "gdn_state_inplace";
    const Tensor &q = tensor(a[0], "q"), &k = tensor(a[1], "k"), &v = tensor(a[2], "v"), &g = tensor(a[3], "g");
    const Tensor &beta = tensor(a[4], "beta"), &state = tensor(a[5], "state"), &slots = tensor(a[6], "slot_ids");
    const bool single = truth(a[8]);
    if (q.dim() != 3 || k.dim() != 3) fail(op, "q and k must be 3D");
    if (v.dim() != 3) fail(op, "v must be 3D");
    if (g.dim() != 2 || beta.dim() != 2) fail(op, "g and beta must be 2D");
    if (state.dim() != 4) fail(op, "state must be 4D");
    if (slots.dim() != 1 || slots.scalar_type() != at::kInt) fail(op, "slot_ids must be int32 1D");
    for (const Tensor* t : {&q, &k, &v, &g, &beta})
      if (t->scalar_type() != at::kBFloat16) fail(op, "q/k/v/g/beta must be bfloat16");
    if (state.scalar_type() != at::kFloat) fail(op, "state must be float32");
    const int64_t tokens = q.size(0), hk = q.size(1), dk = q.size(2), hv = v.size(1), dv = v.size(2);
    for (const Tensor* t : {&k, &v, &g, &beta})
      if (t->size(0) != tokens) fail(op, "leading dimensions must match");
    if (k.size(1) != hk || k.size(2) != dk) fail(op, "q and k shapes must match");
    if (g.size(1) != hv || beta.size(1) != hv) fail(op, "hv dimension mismatch");
    if (state.size(1) != hv || state.size(2) != dv || state.size(3) != dk) fail(op, "state shape must be (slots, hv, dv, dk)");
    if (hk == 0 || hv % hk != 0) fail(op, "hv must be a multiple of hk");
    if (dk != 128 || dv != 128) fail(op, "this specialized kernel requires dk=dv=128");
    const int64_t batch = slots.size(0);
    if (single && tokens != batch) fail(op, "decode mode expects one token per request");
    if (!single) {
      const Tensor& ip = tensor(a[7], "qo_indptr");
      if (ip.dim() != 1 || ip.scalar_type() != at::kInt) fail(op, "qo_indptr must be int32 1D");
      if (ip.size(0) != batch + 1) fail(op, "qo_indptr must have shape (batch + 1,)");
    }
    const c10::Device dev = require_device(op, {&q, &k, &v, &g, &beta, &state, &slots});
    if (!single && tensor(a[7], "qo_indptr").device() != dev) fail(op, "all tensors must be on the same device");
    const int64_t qs = heads_stride0(op, q, "q"), ks = heads_stride0(op, k, "k"), vs = heads_stride0(op, v, "v");
    if (state.stride(3) != 1 || state.stride(2) != dk || state.stride(1) != dv * dk)
      fail(op, "state must be contiguous in its (hv, dv, dk) dimensions");
    const int64_t ss = state.size(0) > 1 ? state.stride(0) : hv * dv * dk;
    Tensor y;
    int rc;
    {
      NoGil nogil;
      OnDevice on(dev);
      y = empty({tokens, hv, dv}, at::kBFloat16, dev);
      const Tensor gc = g.contiguous(), bc = beta.contiguous(), sc = slots.contiguous();
      const Tensor ipc = single ? Tensor() : THPVariable_Unpack(a[7]).contiguous();
      rc = msgl_gdn_state_inplace(q.data_ptr(), k.data_ptr(), v.data_ptr(), gc.data_ptr(), bc.data_ptr(), state.data_ptr(),
                                  ints(sc), single ? nullptr : ints(ipc), y.data_ptr(), tokens, batch, hk, hv, dk, dv,
                                  state.size(0), ss, qs, ks, vs, single ? 1 : 0, on.ptr());
    }
    check_rc(op, rc);
    return THPVariable_Wrap(std::move(y));
  });
}

PyObject* set_checks(PyObject*, PyObject* fn) {
  Py_INCREF(fn);
  Py_XSETREF(g_run_checks, fn);
  Py_RETURN_NONE;
}

#define MSGL_FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {MSGL_FAST(store_kv_cache),
                           MSGL_FAST(paged_decode_attention),
                           MSGL_FAST(paged_prefill_attention),
                           MSGL_FAST(build_attention_metadata),
                           MSGL_FAST(build_metadata_from_host),
                           MSGL_FAST(qk_norm_rope_store),
                           MSGL_FAST(decode_step),
                           MSGL_FAST(extend_step),
                           MSGL_FAST(gdn_state_inplace),
                           {"set_checks", set_checks, METH_O, nullptr},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&g_module); }
