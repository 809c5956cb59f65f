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
#include <c10/hip/HIPCachingAllocator.h>
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
#include <utility>
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

// What is wrong with an operator's arguments, if anything.  An operator raises it; a step that is two operators in one
// asks both (decode_step, extend_step), and leaves it to them to say so.
struct Wrong {
  const char *name = nullptr, *text = nullptr;  // the message: one behind the other
  Wrong() = default;
  Wrong(const char* t) : name(""), text(t) {}
  Wrong(const char* n, const char* t) : name(n), text(t) {}
  explicit operator bool() const { return text != nullptr; }
};

void require(const char* op, const Wrong& w) {
  if (w) fail(op, std::string(w.name) + w.text);
}

Wrong device_of(std::initializer_list<const Tensor*> ts, c10::Device* dev) {
  *dev = (*ts.begin())->device();
  if (!dev->is_cuda()) return "tensors must live on a ROCm GPU device (no CPU implementation exists)";
  for (const Tensor* t : ts)
    if (t->device() != *dev) return "all tensors must be on the same device";
  return {};
}

c10::Device require_device(const char* op, std::initializer_list<const Tensor*> ts) {
  c10::Device dev = c10::kCPU;
  require(op, device_of(ts, &dev));
  return dev;
}

bool whole_rows(const Tensor& t) { return t.stride(2) == 1 && t.stride(1) == t.size(2); }  // of a 3D tensor
// one row may report any leading stride
int64_t row_stride(const Tensor& t) { return t.size(0) > 1 ? t.stride(0) : t.size(1) * t.size(2); }

Wrong pool_form(const Tensor& pool, const char* name) {
  return whole_rows(pool) ? Wrong() : Wrong(name, " must be contiguous in its (num_kv_heads, head_dim) dimensions");
}
int64_t pool_stride0(const char* op, const Tensor& pool, const char* name) {
  require(op, pool_form(pool, name));
  return row_stride(pool);
}

Wrong int32_of(const Tensor& t, const char* name) {
  return t.scalar_type() == at::kInt ? Wrong() : Wrong(name, " must be int32");
}
void require_int32(const char* op, const Tensor& t, const char* name) { require(op, int32_of(t, name)); }

Tensor empty(c10::IntArrayRef size, at::ScalarType dtype, const c10::Device& dev) {
  return at::detail::empty_cuda(size, dtype, dev, std::nullopt);
}

// Scratch from torch's caching allocator, taken on the launch stream (the device is current): safe to give back right after
// the launch because the allocator reuses a block in stream order.  Memory alone: a tensor around it takes as long again (0.3 us).
class Scratch {
 public:
  Scratch() = default;
  Scratch(size_t bytes, const OnDevice& on) : at_(bytes ? c10::hip::HIPCachingAllocator::raw_alloc_with_stream(bytes, on.stream) : nullptr) {}
  Scratch(Scratch&& o) noexcept : at_(std::exchange(o.at_, nullptr)) {}
  Scratch& operator=(Scratch&& o) noexcept {
    std::swap(at_, o.at_);
    return *this;
  }
  ~Scratch() {
    if (at_) c10::hip::HIPCachingAllocator::raw_delete(at_);
  }
  void* ptr() const { return at_; }

 private:
  void* at_ = nullptr;
};

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
Wrong store_args(const Tensor& kc, const Tensor& vc, const Tensor& idx, const Tensor& k, const Tensor& v, c10::Device* dev) {
  if (kc.dim() != 3 || vc.dim() != 3) return "k_cache and v_cache must be 3D (num_pages, num_kv_heads, head_dim)";
  if (idx.dim() != 1) return "indices must be 1D";
  if (k.dim() != 3 || v.dim() != 3) return "k and v must be 3D (length, num_kv_heads, head_dim)";
  const auto dt = kc.scalar_type();
  if (vc.scalar_type() != dt || k.scalar_type() != dt || v.scalar_type() != dt)
    return "k_cache, v_cache, k, v must have the same dtype";
  if (const Wrong w = int32_of(idx, "indices")) return w;
  if (kc.size(2) % 4 != 0) return "head_dim must be a multiple of 4";
  if (vc.sizes() != kc.sizes()) return "v_cache shape must match k_cache";
  if (k.size(0) != idx.size(0) || k.size(1) != kc.size(1) || k.size(2) != kc.size(2) || v.sizes() != k.sizes())
    return "k and v shape must be (length, num_kv_heads, head_dim)";
  if (kc.element_size() != 2 && kc.element_size() != 4) return "unsupported dtype, must be float16, bfloat16 or float32";
  return device_of({&kc, &vc, &idx, &k, &v}, dev);
}

PyObject* store_kv_cache(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 6, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "store_kv_cache";
    const Tensor &kc = tensor(a[0], "k_cache"), &vc = tensor(a[1], "v_cache"), &idx = tensor(a[2], "indices");
    const Tensor &k = tensor(a[3], "k"), &v = tensor(a[4], "v");
    c10::Device dev = c10::kCPU;
    require(op, store_args(kc, vc, idx, k, v, &dev));
    const int64_t pages = kc.size(0), heads = kc.size(1), d = kc.size(2), length = idx.size(0), esz = kc.element_size();
    if (length == 0) return none();
    debug_checks(a[5], op, {a[2], a[0]});
    const int64_t kcs = pool_stride0(op, kc, "k_cache"), vcs = pool_stride0(op, vc, "v_cache");
    int rc;
    {
      NoGil nogil;
      OnDevice on(dev);
      auto source = [](const Tensor& t) { return whole_rows(t) ? t : t.contiguous(); };
      const Tensor ks = source(k), vs = source(v), ix = idx.contiguous();
      rc = msgl_store_kv_cache(kc.data_ptr(), vc.data_ptr(), ints(ix), ks.data_ptr(), vs.data_ptr(), length, heads, d,
                               pages, kcs, vcs, row_stride(ks), row_stride(vs), static_cast<int32_t>(esz), on.ptr());
    }
    check_rc(op, rc);
    return none();
  });
}

Wrong attention_dtype(const Tensor& q, const Tensor& kc, const Tensor& vc, bool half_ok) {
  const auto dt = q.scalar_type();
  if (dt != at::kBFloat16 && dt != at::kHalf) return "unsupported dtype, must be float16 or bfloat16";
  if (kc.scalar_type() != dt || vc.scalar_type() != dt) return "q, k_cache and v_cache must have the same dtype";
  // float16 exists for decode only, as in the reference: its prefill kernel is instantiated for
  // bfloat16 alone (paged_prefill_attention.metal:646-647)
  if (dt == at::kHalf && !half_ok) return "unsupported dtype, the prefill kernel is bfloat16 only";
  return {};
}
int32_t dtype_code(const Tensor& q) { return q.scalar_type() == at::kHalf ? MSGL_DTYPE_F16 : MSGL_DTYPE_BF16; }

// ---- paged_decode_attention(q, k_cache, v_cache, kv_indptr, kv_indices, num_kv_splits, sm_scale,
//                             max_kv_splits, validate) -> out --------------------------------------
Wrong decode_args(const Tensor& q, const Tensor& kc, const Tensor& vc, const Tensor& ip, const Tensor& ix, const Tensor& ns,
                  c10::Device* dev) {
  if (q.dim() != 3) return "q must be 3D (batch, num_q_heads, head_dim)";
  if (kc.dim() != 3 || vc.dim() != 3) return "k_cache and v_cache must be 3D (num_pages, num_kv_heads, head_dim)";
  if (ip.dim() != 1 || ix.dim() != 1 || ns.dim() != 1) return "kv_indptr, kv_indices, num_kv_splits must be 1D";
  const int64_t batch = q.size(0), n_q = q.size(1), d = q.size(2), n_kv = kc.size(1);
  if (d != 128 && d != 256) return "head_dim must be 128 or 256";
  if (n_kv == 0 || n_q % n_kv != 0) return "num_q_heads must be a multiple of num_kv_heads";
  if (n_q / n_kv > 16) return "only q_heads/kv_heads <= 16 is supported";
  if (kc.size(2) != d || vc.size(2) != d) return "cache head_dim must match q head_dim";
  if (vc.size(1) != n_kv) return "v_cache shape must match k_cache";
  if (const Wrong w = attention_dtype(q, kc, vc, true)) return w;
  if (const Wrong w = int32_of(ip, "kv_indptr")) return w;
  if (const Wrong w = int32_of(ix, "kv_indices")) return w;
  if (const Wrong w = int32_of(ns, "num_kv_splits")) return w;
  if (ip.size(0) != batch + 1) return "kv_indptr must have batch + 1 entries";
  if (ns.size(0) != batch) return "num_kv_splits must have batch entries";
  return device_of({&q, &kc, &vc, &ip, &ix, &ns}, dev);
}

PyObject* paged_decode_attention(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 9, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "paged_decode_attention";
    const Tensor &q = tensor(a[0], "q"), &kc = tensor(a[1], "k_cache"), &vc = tensor(a[2], "v_cache");
    const Tensor &ip = tensor(a[3], "kv_indptr"), &ix = tensor(a[4], "kv_indices"), &ns = tensor(a[5], "num_kv_splits");
    c10::Device dev = c10::kCPU;
    require(op, decode_args(q, kc, vc, ip, ix, ns, &dev));
    const int64_t batch = q.size(0), n_q = q.size(1), d = q.size(2), n_kv = kc.size(1);
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
        const Scratch ws(bytes, on);
        rc = msgl_paged_decode_attention(qc.data_ptr(), kc.data_ptr(), vc.data_ptr(), ints(ipc), ints(ixc), ints(nsc),
                                         out.data_ptr(), ws.ptr(), bytes, batch, total_kv, n_q, n_kv, d,
                                         kc.size(0), kcs, vcs, scale, max_splits, dtype_code(q), on.ptr());
      }
    }
    check_rc(op, rc);
    return THPVariable_Wrap(std::move(out));
  });
}

// ---- paged_prefill_attention(q, k_cache, v_cache, qo_indptr, kv_indptr, kv_indices, prefix_lens,
//        sm_scale, max_len_extend, is_cross_attention, sliding_window_size, validate) -> out -------
Wrong prefill_args(const Tensor& q, const Tensor& kc, const Tensor& vc, const Tensor& qp, const Tensor& ip, const Tensor& ix,
                   const Tensor& pl, PyObject* sliding_window_size, int64_t* window, c10::Device* dev) {
  if (q.dim() != 3) return "q must be 3D (total_q_tokens, num_q_heads, head_dim)";
  if (kc.dim() != 3 || vc.dim() != 3) return "k_cache and v_cache must be 3D (num_pages, num_kv_heads, head_dim)";
  if (qp.dim() != 1 || ip.dim() != 1 || ix.dim() != 1 || pl.dim() != 1)
    return "qo_indptr, kv_indptr, kv_indices, prefix_lens must be 1D";
  const int64_t n_q = q.size(1), d = q.size(2), n_kv = kc.size(1);
  if (d != 128 && d != 256) return "head_dim must be 128 or 256";
  if (n_kv == 0 || n_q % n_kv != 0) return "num_q_heads must be a multiple of num_kv_heads";
  if (kc.size(2) != d || vc.size(2) != d) return "cache head_dim must match q head_dim";
  *window = integer(sliding_window_size);
  if (*window < 0) return "sliding_window_size must be >= 0";
  const int64_t batch = qp.size(0) - 1;
  if (batch <= 0) return "batch must be > 0";
  if (vc.size(1) != n_kv) return "v_cache shape must match k_cache";
  if (const Wrong w = attention_dtype(q, kc, vc, false)) return w;
  if (const Wrong w = int32_of(qp, "qo_indptr")) return w;
  if (const Wrong w = int32_of(ip, "kv_indptr")) return w;
  if (const Wrong w = int32_of(ix, "kv_indices")) return w;
  if (const Wrong w = int32_of(pl, "prefix_lens")) return w;
  if (ip.size(0) != batch + 1 || pl.size(0) != batch) return "kv_indptr / prefix_lens length must match qo_indptr";
  return device_of({&q, &kc, &vc, &qp, &ip, &ix, &pl}, dev);
}

PyObject* paged_prefill_attention(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 12, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "paged_prefill_attention";
    const Tensor &q = tensor(a[0], "q"), &kc = tensor(a[1], "k_cache"), &vc = tensor(a[2], "v_cache");
    const Tensor &qp = tensor(a[3], "qo_indptr"), &ip = tensor(a[4], "kv_indptr"), &ix = tensor(a[5], "kv_indices");
    const Tensor& pl = tensor(a[6], "prefix_lens");
    int64_t window;
    c10::Device dev = c10::kCPU;
    require(op, prefill_args(q, kc, vc, qp, ip, ix, pl, a[10], &window, &dev));
    const int64_t total_q = q.size(0), n_q = q.size(1), d = q.size(2), n_kv = kc.size(1), batch = qp.size(0) - 1;
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
        const Scratch ws(bytes, on);
        rc = msgl_paged_prefill_attention(qc.data_ptr(), kc.data_ptr(), vc.data_ptr(), ints(qpc), ints(ipc), ints(ixc),
                                          ints(plc), out.data_ptr(), ws.ptr(), bytes, batch, total_q, total_kv,
                                          n_q, n_kv, d, kc.size(0), kcs, vcs, scale, static_cast<int32_t>(max_extend),
                                          cross ? 1 : 0, static_cast<int32_t>(window), dtype_code(q), on.ptr());
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

Wrong heads_form(const Tensor& t, const char* name) {
  if (t.dim() != 3) return {name, " must be 3D (tokens, heads, head_dim)"};
  return whole_rows(t) ? Wrong() : Wrong(name, " must be contiguous in its (heads, head_dim) dimensions");
}
int64_t heads_stride0(const char* op, const Tensor& t, const char* name) {
  require(op, heads_form(t, name));
  return row_stride(t);
}

// ---- qk_norm_rope_store(q, k, v, q_weight, k_weight, positions, out_loc, k_cache, v_cache, eps,
//                         rope_base, validate) -> rotated q -----------------------------------------
Wrong norm_rope_args(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& qw, const Tensor& kw, const Tensor& pos,
                     const Tensor& loc, const Tensor& kc, const Tensor& vc, c10::Device* dev) {
  if (const Wrong w = device_of({&q, &k, &v, &qw, &kw, &pos, &loc, &kc, &vc}, dev)) return w;
  const std::pair<const Tensor*, const char*> typed[] = {{&q, "q"}, {&k, "k"}, {&v, "v"}, {&kc, "k_cache"},
                                                         {&vc, "v_cache"}, {&qw, "q_weight"}, {&kw, "k_weight"}};
  for (int i = 0; i < 3; ++i)
    if (const Wrong w = heads_form(*typed[i].first, typed[i].second)) return w;
  const int64_t tokens = q.size(0), d = q.size(2), n_kv = k.size(1);
  if (d != 128 && d != 256) return "head_dim must be 128 or 256";
  if (k.size(0) != tokens || k.size(2) != d || v.sizes() != k.sizes()) return "k and v shape must be (tokens, num_kv_heads, head_dim)";
  if (kc.dim() != 3 || kc.size(1) != n_kv || kc.size(2) != d || vc.sizes() != kc.sizes())
    return "k_cache and v_cache must be (num_pages, num_kv_heads, head_dim)";
  for (const auto& [t, name] : typed)
    if (t->scalar_type() != at::kBFloat16) return {name, " must be bfloat16"};
  if (qw.dim() != 1 || qw.size(0) != d || kw.dim() != 1 || kw.size(0) != d) return "q_weight and k_weight must be (head_dim,)";
  if (const Wrong w = int32_of(pos, "positions")) return w;
  if (const Wrong w = int32_of(loc, "out_loc")) return w;
  if (pos.dim() < 1 || loc.dim() < 1 || pos.size(0) != tokens || loc.size(0) != tokens)
    return "positions and out_loc length must match q length";
  return {};
}

PyObject* qk_norm_rope_store(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 12, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "qk_norm_rope_store";
    const Tensor &q = tensor(a[0], "q"), &k = tensor(a[1], "k"), &v = tensor(a[2], "v"), &qw = tensor(a[3], "q_weight");
    const Tensor &kw = tensor(a[4], "k_weight"), &pos = tensor(a[5], "positions"), &loc = tensor(a[6], "out_loc");
    const Tensor &kc = tensor(a[7], "k_cache"), &vc = tensor(a[8], "v_cache");
    c10::Device dev = c10::kCPU;
    require(op, norm_rope_args(q, k, v, qw, kw, pos, loc, kc, vc, &dev));
    const int64_t qs = row_stride(q), ks = row_stride(k), vs = row_stride(v);
    const int64_t tokens = q.size(0), n_q = q.size(1), d = q.size(2), n_kv = k.size(1);
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
// caller then makes the two calls, which say what is wrong with their arguments, and take every form.
//
// What is refused here is what one of the two operators refuses (their own checks), what one of them would copy first,
// and what the C ABI refuses before it launches anything (strides, alignment, constants).
bool steps_are_checked() {  // index validation is the operators'
  const char* env = std::getenv("MSGL_DEBUG_CHECKS");
  return env && *env && std::strcmp(env, "0") != 0;
}
bool as_they_are(std::initializer_list<const Tensor*> rows, std::initializer_list<const Tensor*> indices) {
  for (const Tensor* t : rows)
    if (!whole_rows(*t)) return false;
  for (const Tensor* t : indices)
    if (t->dim() != 1 || !t->is_contiguous()) return false;
  return true;
}
PyObject* step_result(const char* op, int rc, Tensor&& out) {
  if (rc == MSGL_ERR_SHAPE || rc == MSGL_ERR_ALIGNMENT) return none();  // the two kinds that are left to the C ABI
  check_rc(op, rc);
  return THPVariable_Wrap(std::move(out));
}

PyObject* decode_step(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 15, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "decode_step";
    const bool norm = a[3] != Py_None;
    for (int i = 0; i < 12; ++i)
      if (!THPVariable_Check(a[i]) && (norm || i < 3 || i > 5)) return none();
    if (steps_are_checked()) return none();
    auto t = [&](int i) -> const Tensor& { return THPVariable_Unpack(a[i]); };
    const Tensor &q = t(0), &k = t(1), &v = t(2), &loc = t(6), &kc = t(7), &vc = t(8), &ip = t(9), &ix = t(10), &ns = t(11);
    c10::Device dev = c10::kCPU, again = c10::kCPU;
    if (decode_args(q, kc, vc, ip, ix, ns, &dev) || !as_they_are({&q, &kc, &vc}, {&ip, &ix, &ns})) return none();
    if (norm ? bool(norm_rope_args(q, k, v, t(3), t(4), t(5), loc, kc, vc, &again)) : bool(store_args(kc, vc, loc, k, v, &again)))
      return none();
    const int64_t batch = q.size(0), n_q = q.size(1), d = q.size(2), n_kv = kc.size(1), slots = kc.size(0);
    if (again != dev || loc.size(0) != batch || !as_they_are({&k, &v}, {&loc})) return none();
    if (norm && !as_they_are({}, {&t(3), &t(4), &t(5)})) return none();
    const size_t bytes = msgl_decode_step_workspace_bytes(batch, ix.size(0), n_q, n_kv, d, norm ? 1 : 0);
    if (bytes == 0) return none();
    const float scale = static_cast<float>(real(a[12]));
    const float eps = norm ? static_cast<float>(real(a[13])) : 0.f, base = norm ? static_cast<float>(real(a[14])) : 0.f;
    Tensor out;
    int rc;
    {
      NoGil nogil;
      OnDevice on(dev);
      out = empty({batch, n_q, d}, q.scalar_type(), dev);
      const Scratch ws(bytes, on);
      rc = msgl_decode_step(q.data_ptr(), k.data_ptr(), v.data_ptr(), row_stride(q), row_stride(k), row_stride(v),
                            norm ? t(3).data_ptr() : nullptr, norm ? t(4).data_ptr() : nullptr, norm ? ints(t(5)) : nullptr,
                            ints(loc), kc.data_ptr(), vc.data_ptr(), ints(ip), ints(ix), out.data_ptr(), ws.ptr(), bytes,
                            batch, ix.size(0), n_q, n_kv, d, slots, row_stride(kc), row_stride(vc), scale, eps, base,
                            dtype_code(q), on.ptr());
    }
    return step_result(op, rc, std::move(out));
  });
}

// ---- extend_step(q, k, v, out_loc, k_cache, v_cache, qo_indptr, kv_indptr, kv_indices, prefix_lens, sm_scale,
//                  max_len_extend, is_cross_attention, sliding_window_size, own_slots) -> out or None ----
// As decode_step, for prefill metadata; the two launches are made here too where one is not the way, and always
// without own_slots.  (Where the second of them is refused, the rows are stored as the first call would have.)
PyObject* extend_step(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 15, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "extend_step";
    for (int i = 0; i < 10; ++i)
      if (!THPVariable_Check(a[i])) return none();
    if (steps_are_checked()) return none();
    auto t = [&](int i) -> const Tensor& { return THPVariable_Unpack(a[i]); };
    const Tensor &q = t(0), &k = t(1), &v = t(2), &loc = t(3), &kc = t(4), &vc = t(5), &qp = t(6), &ip = t(7), &ix = t(8), &pl = t(9);
    int64_t window = 0;
    c10::Device dev = c10::kCPU, again = c10::kCPU;
    if (prefill_args(q, kc, vc, qp, ip, ix, pl, a[13], &window, &dev) || store_args(kc, vc, loc, k, v, &again)) return none();
    if (again != dev || !q.is_contiguous() || !as_they_are({&k, &v, &kc, &vc}, {&loc, &qp, &ip, &ix, &pl})) return none();
    const int64_t total = q.size(0), n_q = q.size(1), d = q.size(2), n_kv = kc.size(1), slots = kc.size(0), batch = qp.size(0) - 1;
    const int64_t max_extend = integer(a[11]);
    const bool cross = truth(a[12]), own_slots = truth(a[14]);
    if (total == 0 || loc.size(0) != total || max_extend <= 0 || std::max(max_extend, window) > 0x7fffffff) return none();
    const float scale = static_cast<float>(real(a[10]));
    Tensor out;
    int rc;
    {
      NoGil nogil;
      OnDevice on(dev);
      out = empty({total, n_q, d}, q.scalar_type(), dev);
      const int64_t ks0 = row_stride(k), vs0 = row_stride(v), kcs = row_stride(kc), vcs = row_stride(vc);
      size_t bytes = !own_slots ? 0 : msgl_extend_step_workspace_bytes(batch, total, ix.size(0), n_q, n_kv, d, max_extend, cross,
                                                                       static_cast<int32_t>(window));
      if (bytes > 0) {
        const Scratch ws(bytes, on);
        rc = msgl_extend_step(q.data_ptr(), k.data_ptr(), v.data_ptr(), ks0, vs0, ints(loc), kc.data_ptr(), vc.data_ptr(), ints(qp),
                              ints(ip), ints(ix), ints(pl), out.data_ptr(), ws.ptr(), bytes, batch, total, ix.size(0), n_q,
                              n_kv, d, slots, kcs, vcs, scale, static_cast<int32_t>(max_extend), cross ? 1 : 0,
                              static_cast<int32_t>(window), dtype_code(q), on.ptr());
      } else {
        rc = msgl_store_kv_cache(kc.data_ptr(), vc.data_ptr(), ints(loc), k.data_ptr(), v.data_ptr(), total, n_kv, d, slots, kcs,
                                 vcs, ks0, vs0, static_cast<int32_t>(kc.element_size()), on.ptr());
        if (rc == MSGL_OK) {
          bytes = msgl_paged_prefill_workspace_bytes(batch, total, ix.size(0), n_q, n_kv, d, max_extend);
          const Scratch ws(bytes, on);
          rc = msgl_paged_prefill_attention(q.data_ptr(), kc.data_ptr(), vc.data_ptr(), ints(qp), ints(ip), ints(ix), ints(pl),
                                            out.data_ptr(), ws.ptr(), bytes, batch, total, ix.size(0), n_q, n_kv, d, slots,
                                            kcs, vcs, scale, static_cast<int32_t>(max_extend), cross ? 1 : 0,
                                            static_cast<int32_t>(window), dtype_code(q), on.ptr());
        }
      }
    }
    return step_result(op, rc, std::move(out));
  });
}

// ---- gdn_state_inplace(q, k, v, g, beta, state, slot_ids, qo_indptr, single_token_mode, longest) -> y -----
PyObject* gdn_state_inplace(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  return guarded(args, n_args, 10, [](PyObject* const* a) -> PyObject* {
    static const char op[] = "gdn_state_inplace";
    const Tensor &q = tensor(a[0], "q"), &k = tensor(a[1], "k"), &v = tensor(a[2], "v"), &g = tensor(a[3], "g");
    const Tensor &beta = tensor(a[4], "beta"), &state = tensor(a[5], "state"), &slots = tensor(a[6], "slot_ids");
    const bool single = truth(a[8]);
    const int64_t longest = a[9] == Py_None ? 0 : std::max<int64_t>(integer(a[9]), 0);
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
      // the forms whose scratch memory would not be used (see the header)
      const bool plain = reinterpret_cast<uintptr_t>(v.data_ptr()) % 16 == 0 && vs % 8 == 0 && std::max({qs, ks, vs}) < (1 << 24) && hv < (1 << 17);
      size_t bytes = plain ? msgl_gdn_state_workspace_bytes(tokens, batch, hv, single ? 1 : 0) : 0;
      Scratch ws;
      if (bytes > 0) {
        try {
          ws = Scratch(bytes, on);
        } catch (const c10::OutOfMemoryError&) {  // it is an optimisation: the call goes without
          bytes = 0;
        }
      }
      rc = msgl_gdn_state_inplace_longest(q.data_ptr(), k.data_ptr(), v.data_ptr(), gc.data_ptr(), bc.data_ptr(), state.data_ptr(),
                                  ints(sc), single ? nullptr : ints(ipc), y.data_ptr(), tokens, batch, hk, hv, dk, dv,
                                  state.size(0), ss, qs, ks, vs, single ? 1 : 0, longest, ws.ptr(), bytes, on.ptr());
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
