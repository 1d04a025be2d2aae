// Python binding of the C ABI (include/we_attn.h): tensors in, validation, output allocation and the
// library call in native code.
//
// The kernels of a 256-token frame take 25 us per layer; reading shapes, strides and pointers of a
// dozen tensors through Python and ctypes took 35 us, and checking the position ids with torch
// operations another 120 us (15 launches, three synchronisations).  Here the tensors are read where
// they live, and the position ids are checked by the call's own first kernel: the host waits for
// that kernel's verdict only, while the attention behind it is already running.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/core/grad_mode.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_strided.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <chrono>
#include <cmath>
#include <mutex>
#include <stdexcept>
#include <typeinfo>
#include <string>

#include "../../include/we_attn.h"
#include "record_slots.h"

namespace {

using at::Tensor;

[[noreturn]] void fail(const std::string& what) { throw std::runtime_error(what); }
[[noreturn]] void fail_code(const char* fn, int code) {
  fail(std::string(fn) + " failed: " + we_error_string(code) + " (code " + std::to_string(code) + ")");
}

// Without the interpreter's lock for as long as it lives: around everything that can wait (a launch
// into a full queue, a verdict, a free record), so that other threads of the program go on.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
  NoGil() = default;
  NoGil(const NoGil&) = delete;
  NoGil& operator=(const NoGil&) = delete;
};

// ---- arguments -----------------------------------------------------------------------------

struct Args {
  const char* fn;
  PyObject* const* v;
  Py_ssize_t n;
  Py_ssize_t i = 0;
  Args(const char* fn_, PyObject* const* v_, Py_ssize_t n_, Py_ssize_t want) : fn(fn_), v(v_), n(n_) {
    if (n != want) fail(std::string(fn) + ": wrong number of arguments");
  }
  const Tensor& tensor() {
    PyObject* o = v[i++];
    if (!THPVariable_Check(o)) fail(std::string(fn) + ": expected a tensor");
    return THPVariable_Unpack(o);
  }
  const Tensor* opt_tensor() {
    if (v[i] == Py_None) { ++i; return nullptr; }
    return &tensor();
  }
  int64_t integer() {
    const long long r = PyLong_AsLongLong(v[i++]);
    if (r == -1 && PyErr_Occurred()) throw std::bad_cast();
    return r;
  }
  bool flag() {
    const int r = PyObject_IsTrue(v[i++]);
    if (r < 0) throw std::bad_cast();
    return r != 0;
  }
  double number() {
    const double r = PyFloat_AsDouble(v[i++]);
    if (r == -1.0 && PyErr_Occurred()) throw std::bad_cast();
    return r;
  }
  // None = the default
  double scale(int64_t d_head) {
    if (v[i] == Py_None) { ++i; return 1.0 / std::sqrt((double)d_head); }
    return number();
  }
};

// ---- devices -------------------------------------------------------------------------------

c10::Device need_device(std::initializer_list<const Tensor*> ts) {
  c10::Device dev(c10::DeviceType::CPU);
  bool first = true;
  for (const Tensor* t : ts) {
    if (t == nullptr) continue;
    const c10::Device d = t->device();
    if (d.type() != c10::DeviceType::CUDA)
      fail("world_engine_amd kernels run on a ROCm GPU only; got a tensor on " + d.str() + " (there is no CPU path)");
    if (first) dev = d;
    else if (d != dev) fail("all tensors must be on the same device");
    first = false;
  }
  return dev;
}

// The library launches on the device that is current: the tensors' device for the time of a call.
struct OnDevice {
  int back = -1;
  explicit OnDevice(c10::Device dev) {
    int cur = -1;
    if (hipGetDevice(&cur) != hipSuccess) fail("no current device");
    if (cur == dev.index()) return;
    if (hipSetDevice(dev.index()) != hipSuccess) fail("cannot select the tensors' device");
    back = cur;
  }
  ~OnDevice() {
    if (back >= 0) (void)hipSetDevice(back);
  }
};

hipStream_t stream_of(c10::Device dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

bool capturing(hipStream_t st) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cs) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return cs != hipStreamCaptureStatusNone;
}

// ---- tensors -------------------------------------------------------------------------------

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return WE_DTYPE_BF16;
    case at::kHalf: return WE_DTYPE_F16;
    case at::kFloat: return WE_DTYPE_F32;
    default: fail(std::string("unsupported element type ") + c10::toString(t.scalar_type()));
  }
}

struct Strides {
  int64_t s[3] = {0, 0, 0};
  Strides() = default;
  Strides(const Tensor& t, const char* what) {
    if (t.dim() != 4 || t.stride(3) != 1)
      fail(std::string(what) + " must be [B, H, T, Dh] with a contiguous last dimension");
    s[0] = t.stride(0); s[1] = t.stride(1); s[2] = t.stride(2);
  }
};

bool is_shape(const Tensor& t, std::initializer_list<int64_t> shape) {
  return t.sizes().equals(c10::IntArrayRef(shape));
}

// Position ids [B, T] with one row stride (copies are made where the layout needs it).
struct PosIds {
  Tensor t, y, x;
  int64_t row_stride = 0;
  PosIds(const Tensor& t_, const Tensor* y_, const Tensor* x_, int64_t B, int64_t T) : t(t_) {
    if (!is_shape(t, {B, T})) fail("t_pos must be [B, T]");
    if (t.scalar_type() != at::kLong) fail("position ids must be int64");
    if (y_ == nullptr) {
      if (t.stride(1) != 1 && T > 1) t = t.contiguous();
    } else {
      y = *y_; x = *x_;
      for (const Tensor* p : {&y, &x})
        if (!is_shape(*p, {B, T}) || p->scalar_type() != at::kLong) fail("y_pos / x_pos must be int64 [B, T]");
      const int64_t rs = t.stride(0);
      if (t.stride(1) != 1 || y.stride(1) != 1 || x.stride(1) != 1 || y.stride(0) != rs || x.stride(0) != rs) {
        t = t.contiguous(); y = y.contiguous(); x = x.contiguous();
      }
    }
    row_stride = t.stride(0);
  }
  const int64_t* tp() const { return t.const_data_ptr<int64_t>(); }
  const int64_t* yp() const { return y.defined() ? y.const_data_ptr<int64_t>() : nullptr; }
  const int64_t* xp() const { return x.defined() ? x.const_data_ptr<int64_t>() : nullptr; }
};

void check_cache(const Tensor& kv, const Tensor& written, int64_t B, int64_t Hkv, int64_t T, int64_t Dh, int64_t L) {
  if (kv.dim() != 5 || !is_shape(kv, {2, B, Hkv, L + T, Dh}) || !kv.is_contiguous())
    fail("kv must be a contiguous [2, B, Hkv, L+T, Dh] buffer; KV cache expects exactly one frame per upsert");
  if (written.scalar_type() != at::kBool || written.numel() != L + T || !written.is_contiguous())
    fail("written must be a contiguous bool [L+T] tensor");
}

void check_tables(const Tensor& cos, const Tensor& sin, int64_t Dh) {
  if (cos.scalar_type() != at::kFloat || sin.scalar_type() != at::kFloat || cos.dim() != 2 || cos.sizes() != sin.sizes() ||
      cos.size(1) != Dh / 2 || !cos.is_contiguous() || !sin.is_contiguous())
    fail("cos/sin tables must be contiguous fp32 [rows, Dh/2]");
}

Tensor new_heads(const Tensor& like, int64_t B, int64_t H, int64_t T, int64_t Dh) {
  return at::empty({B, H, T, Dh}, like.options());
}
// [B, H, T, Dh] whose memory is [B, T, H, Dh]
Tensor new_token_major(const Tensor& like, int64_t B, int64_t H, int64_t T, int64_t Dh) {
  return at::empty_strided({B, H, T, Dh}, {T * H * Dh, Dh, H * Dh, 1}, like.options());
}

Tensor output_or_new(const Tensor* out, bool token_major, const Tensor& like, c10::Device dev, int64_t B, int64_t H,
                     int64_t T, int64_t Dh) {
  if (out == nullptr) return token_major ? new_token_major(like, B, H, T, Dh) : new_heads(like, B, H, T, Dh);
  if (!is_shape(*out, {B, H, T, Dh}) || out->scalar_type() != like.scalar_type() || out->device() != dev)
    fail("out must be [B, H, T, Dh] of q's element type on q's device");
  return *out;
}

// The caller's split-context workspace where it is long enough and in one piece, else a new one.
struct Workspace {
  Tensor t;
  void* ptr = nullptr;
  size_t bytes = 0;
  Workspace(const Tensor* given, int64_t B, int64_t H, int64_t Hkv, int64_t T, int64_t Dh, int64_t L, int64_t dilation, int splits,
            int q_tile, const Tensor& like) {
    if (like.scalar_type() == at::kFloat) {  // (no caller has to know of it: a given one that does not do is passed over)
      const size_t wanted = splits == 0 ? we_attn_f32_workspace_bytes((int)B, (int)H, (int)Hkv, (int)T, (int)Dh, L, (int)dilation) : 0;
      if (wanted == 0) return;
      const bool fits = given != nullptr && given->device() == like.device() && given->is_contiguous() &&
                        (size_t)given->numel() * given->element_size() >= wanted && ((uintptr_t)given->data_ptr() & 15u) == 0;
      t = fits ? *given : at::empty({(int64_t)wanted}, like.options().dtype(at::kByte));
      ptr = t.data_ptr();
      bytes = (size_t)t.numel() * t.element_size();
      return;
    }
    const size_t need = we_attn_workspace_bytes_for((int)B, (int)H, (int)Hkv, (int)T, (int)Dh, L, splits, q_tile, dtype_code(like));
    if (need == 0) return;
    if (given != nullptr && given->device() != like.device()) fail("workspace must be on the call's device, " + like.device().str());
    if (given != nullptr && given->is_contiguous() && (size_t)given->numel() * given->element_size() >= need) t = *given;
    else t = at::empty({(int64_t)need}, like.options().dtype(at::kByte));
    ptr = t.data_ptr();
    bytes = (size_t)t.numel() * t.element_size();
  }
};

// The attention module's element-wise neighbours (we_attn_extras); has = whether any is asked for.
struct Extras {
  we_attn_extras e{};
  bool has = false;
  const we_attn_extras* ptr() const { return has ? &e : nullptr; }
  Extras(double eps, const Tensor* v1, const Tensor* v_lamb, const Tensor* gate, const Tensor* gate_x,
         const Tensor* gate_w, at::ScalarType dtype, int64_t B, int64_t H, int64_t Hkv, int64_t T, int64_t Dh) {
    has = eps != 0.0 || v1 != nullptr || gate != nullptr || gate_w != nullptr;
    if (!has) return;
    e.qk_norm_eps = (float)eps;
    if (v1 != nullptr) {
      if (v_lamb == nullptr || v_lamb->numel() != 1 || v_lamb->scalar_type() != dtype || !is_shape(*v1, {B, Hkv, T, Dh}) ||
          v1->scalar_type() != dtype)
        fail("v1 must match v and v_lamb must be one element of the same type");
      need_device({v1, v_lamb});
      const Strides s(*v1, "v1");
      e.v1 = v1->data_ptr(); e.v_lamb = v_lamb->data_ptr();
      for (int i = 0; i < 3; ++i) e.v1_strides[i] = s.s[i];
    }
    if (gate != nullptr) {
      if (!is_shape(*gate, {B, H, T}) || gate->scalar_type() != dtype) fail("gate must be [B, H, T] of q's element type");
      need_device({gate});
      e.gate = gate->data_ptr();
      for (int i = 0; i < 3; ++i) e.gate_strides[i] = gate->stride(i);
    }
    if (gate_w != nullptr) {
      if (gate != nullptr) fail("give either gate or gate_x / gate_w");
      if (gate_x == nullptr || !is_shape(*gate_x, {B, T, H}) || gate_x->stride(2) != 1 || gate_x->scalar_type() != dtype ||
          !is_shape(*gate_w, {H, H}) || gate_w->scalar_type() != dtype || !gate_w->is_contiguous())
        fail("gate_x must be [B, T, H] (contiguous channels) and gate_w a contiguous [H, H], both of q's element type");
      need_device({gate_x, gate_w});
      e.gate_x = gate_x->data_ptr(); e.gate_w = gate_w->data_ptr();
      e.gate_x_strides[0] = gate_x->stride(0); e.gate_x_strides[1] = gate_x->stride(1);
    }
  }
};

// ---- verdicts of the position-id check -------------------------------------------------------
// A call that checks holds one of a device's records until it has its verdict: a word of host-coherent
// memory, which one of the call's kernels writes once.  The records are made on a device's first
// checked call and live as long as the process; a call that finds all of them out waits for one,
// without the interpreter's lock.
// The device word in which the verdict goes on to the call's later kernels is read long after the
// host has had its report, so it cannot be a record's: it is memory from torch's allocator, which
// hands it out again only to work that the stream runs behind this call's.
constexpr int kVerdicts = we::RecordSlots::kCount;
constexpr int kMaxDevices = 64;
struct Verdicts {
  we::RecordSlots slots;
  uint64_t* report = nullptr;   // kVerdicts words, one per 64 bytes
  uint64_t ticket[kVerdicts] = {};
};
std::atomic<Verdicts*> g_verdicts[kMaxDevices];
std::mutex g_mu;

Verdicts& verdicts(c10::Device dev) {
  const int d = dev.index();
  if (d < 0 || d >= kMaxDevices) fail("device index out of range");
  Verdicts* p = g_verdicts[d].load(std::memory_order_acquire);
  if (p != nullptr) return *p;
  std::lock_guard<std::mutex> lock(g_mu);
  p = g_verdicts[d].load(std::memory_order_acquire);
  if (p != nullptr) return *p;
  void* host = nullptr;
  if (hipHostMalloc(&host, kVerdicts * 64, hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess)
    fail("cannot allocate the position-id check's records");
  Verdicts* made = new Verdicts;
  made->report = static_cast<uint64_t*>(host);
  for (int i = 0; i < kVerdicts * 8; ++i) made->report[i] = 0;
  g_verdicts[d].store(made, std::memory_order_release);
  return *made;
}

class PosCheck {
 public:
  // what: WE_CHECK_* bits, for a call on B x T ids on dev's current stream st; nothing is checked under
  // stream capture (the verdict could not be waited for)
  PosCheck(int what, c10::Device dev, hipStream_t st, int64_t B, int64_t T, bool with_projection) : st_(st) {
    if (what == 0 || capturing(st)) return;
    const size_t bytes = we_pos_check_guard_bytes((int)B, (int)T, with_projection ? 1 : 0);
    if (bytes != 0) guard_ = at::empty({(int64_t)bytes}, at::TensorOptions().dtype(at::kByte).device(dev));
    v_ = &verdicts(dev);
    slot_ = v_->slots.take([](auto&& wait) {
      const NoGil off;
      wait();
    });
    c_.what = what;
    c_.report = v_->report + slot_ * 8;
    c_.guard = guard_.defined() ? reinterpret_cast<uint32_t*>(guard_.data_ptr()) : nullptr;
    c_.ticket = ++v_->ticket[slot_];
  }
  ~PosCheck() {
    if (v_ == nullptr) return;
    if (!awaited_) {  // (a call that failed half-way: nothing may report to the record later)
      const NoGil off;
      (void)hipStreamSynchronize(st_);
    }
    v_->slots.give_back(slot_);
  }
  PosCheck(const PosCheck&) = delete;
  PosCheck& operator=(const PosCheck&) = delete;
  const we_pos_check* arg() const { return v_ != nullptr ? &c_ : nullptr; }
  // Waits for the verdict of the launched call (not under the interpreter's lock); true = refused.
  bool refused() {
    if (v_ == nullptr) return false;
    awaited_ = true;
    const volatile uint64_t* word = c_.report;
    uint64_t got = 0;
    const auto began = std::chrono::steady_clock::now();
    bool there = false;
    for (int spin = 1; !there; ++spin) {
      got = *word;
      there = (got >> 1) == c_.ticket;
      if (there) break;
      __builtin_ia32_pause();
      // the queue in front is long (or the device is in trouble): let the runtime do the waiting
      if ((spin & 1023) == 0 && std::chrono::steady_clock::now() - began > std::chrono::milliseconds(20)) break;
    }
    hipError_t e = hipSuccess;
    if (!there) {
      e = hipStreamSynchronize(st_);
      got = *word;
      there = (got >> 1) == c_.ticket;
    }
    if (!there) fail(std::string("the position-id check did not report: ") + hipGetErrorString(e));
    std::atomic_thread_fence(std::memory_order_acquire);
    return (got & 1u) != 0;
  }

 private:
  hipStream_t st_;
  Verdicts* v_ = nullptr;
  int slot_ = 0;
  bool awaited_ = false;
  Tensor guard_;
  we_pos_check c_{};
};

// A library call and, where it checks, the wait for its verdict, without the interpreter's lock; true = refused.
template <typename F>
bool run(const char* fn, PosCheck* check, F&& call) {
  const NoGil off;
  const int rc = call();
  if (rc != WE_OK) fail_code(fn, rc);
  return check != nullptr && check->refused();
}

// A tensor that is its memory and nothing else: no Python subclass or functorch wrapper that would
// see the operation, no tangent, no lazily negated view.
bool plain_memory(const Tensor& t) {
  return t.has_storage() && !t.unsafeGetTensorImpl()->is_python_dispatch() && !t.is_neg() && !t._fw_grad(/*level=*/0).defined();
}
// Somebody sees every operation of this thread (dispatch and function modes).
bool watched() { return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled(); }
bool to_record(const Tensor& t) { return at::GradMode::is_enabled() && t.requires_grad(); }

// ---- results -------------------------------------------------------------------------------

PyObject* wrap(const Tensor& t) { return THPVariable_Wrap(t); }
PyObject* wrap_or_none(const Tensor& t) {
  if (t.defined()) return THPVariable_Wrap(t);
  Py_RETURN_NONE;
}
PyObject* none() { Py_RETURN_NONE; }
PyObject* pack(std::initializer_list<const Tensor*> ts) {
  PyObject* r = PyTuple_New((Py_ssize_t)ts.size());
  if (r == nullptr) throw std::bad_cast();
  Py_ssize_t i = 0;
  for (const Tensor* t : ts) PyTuple_SET_ITEM(r, i++, wrap_or_none(*t));
  return r;
}
PyObject* refused_result() { Py_RETURN_FALSE; }

template <typename F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (const std::bad_cast&) {
    return nullptr;  // (the Python error is set)
  } catch (const c10::Error& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    return nullptr;
  } catch (const std::exception& e) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// ---- entry points ----------------------------------------------------------------------------
// Positional arguments only; world_engine_amd/ops.py documents them.  `check` is the set of
// WE_CHECK_* rules; a call whose position ids break one returns False.

PyObject* rope_kv_store(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a("rope_kv_store", argv, n, 17);
    const Tensor* q = a.opt_tensor();
    const Tensor &k = a.tensor(), &v = a.tensor(), &tp = a.tensor();
    const Tensor *yp = a.opt_tensor(), *xp = a.opt_tensor(), *cos = a.opt_tensor(), *sin = a.opt_tensor();
    const int64_t gh = a.integer(), gw = a.integer();
    const Tensor &kv = a.tensor(), &written = a.tensor();
    const int64_t L = a.integer(), dilation = a.integer();
    const bool frozen = a.flag();
    const int what = (int)a.integer();
    const int64_t tpf = a.integer();
    const bool rotate = cos != nullptr;
    if (rotate && (sin == nullptr || yp == nullptr || xp == nullptr))
      fail("a rotation takes the cos and sin tables and y_pos and x_pos together");
    const c10::Device dev = need_device({&k, &v, &kv, &written, q, cos, sin, &tp, rotate ? yp : nullptr, rotate ? xp : nullptr});
    if (k.dim() != 4 || k.sizes() != v.sizes()) fail("k and v must both be [B, Hkv, T, Dh]");
    const int64_t B = k.size(0), Hkv = k.size(1), T = k.size(2), Dh = k.size(3);
    if (tpf > 0 && T != tpf) fail("KV cache expects exactly one frame per upsert");
    if (k.scalar_type() != kv.scalar_type() || v.scalar_type() != kv.scalar_type() ||
        (q != nullptr && q->scalar_type() != kv.scalar_type()))
      fail("q/k/v must have the cache's element type");
    check_cache(kv, written, B, Hkv, T, Dh, L);
    if (q != nullptr && (q->dim() != 4 || q->size(0) != B || q->size(2) != T || q->size(3) != Dh))
      fail("q must be [B, H, T, Dh] matching k");
    if (rotate) check_tables(*cos, *sin, Dh);
    const PosIds pos(tp, rotate ? yp : nullptr, rotate ? xp : nullptr, B, T);
    const Strides qs = q != nullptr ? Strides(*q, "q") : Strides(), ks(k, "k"), vs(v, "v");
    const int code_t = dtype_code(kv);
    const OnDevice on(dev);
    const hipStream_t st = stream_of(dev);
    const int64_t H = q != nullptr ? q->size(1) : Hkv;
    Tensor q_out;
    if (q != nullptr) q_out = new_heads(*q, B, H, T, Dh);
    PosCheck check(what, dev, st, B, T, false);
    const bool refused = run("we_rope_kv_store", &check, [&] { return we_rope_kv_store_checked(
        q != nullptr ? q->data_ptr() : nullptr, k.data_ptr(), v.data_ptr(), q != nullptr ? qs.s : nullptr, ks.s, vs.s,
        q != nullptr ? q_out.data_ptr() : nullptr, rotate ? cos->const_data_ptr<float>() : nullptr,
        rotate ? sin->const_data_ptr<float>() : nullptr, rotate ? cos->size(0) : 0, pos.tp(), pos.yp(), pos.xp(),
        pos.row_stride, gh, gw, kv.data_ptr(), static_cast<uint8_t*>(written.data_ptr()), (int)B, (int)H, (int)Hkv,
        (int)T, (int)Dh, L, (int)dilation, frozen ? 1 : 0, code_t, check.arg(), st); });
    if (refused) return refused_result();
    return q != nullptr ? wrap(q_out) : none();
  });
}

PyObject* rope_apply(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a("rope_apply", argv, n, 9);
    const Tensor &x = a.tensor(), &tp = a.tensor(), &yp = a.tensor(), &xp = a.tensor();
    const Tensor &cos_in = a.tensor(), &sin_in = a.tensor();
    const int64_t gh = a.integer(), gw = a.integer();
    const int what = (int)a.integer();
    const c10::Device dev = need_device({&x, &cos_in, &sin_in, &tp, &yp, &xp});
    if (x.dim() != 4) fail("x must be [B, H, T, Dh]");
    const int64_t B = x.size(0), H = x.size(1), T = x.size(2), Dh = x.size(3);
    if (cos_in.scalar_type() != at::kFloat || sin_in.scalar_type() != at::kFloat) fail("cos/sin tables must be fp32");
    if (cos_in.sizes() != sin_in.sizes() || cos_in.dim() != 2 || cos_in.size(1) != Dh / 2)
      fail("cos/sin tables must be [rows, Dh/2]");
    const PosIds pos(tp, &yp, &xp, B, T);
    const Strides xs(x, "x");
    const int code_t = dtype_code(x);
    const OnDevice on(dev);
    const hipStream_t st = stream_of(dev);
    const Tensor cos = cos_in.contiguous(), sin = sin_in.contiguous();
    const Tensor out = new_heads(x, B, H, T, Dh);
    PosCheck check(what, dev, st, B, T, false);
    const bool refused = run("we_rope_apply", &check, [&] { return we_rope_apply_checked(x.data_ptr(), xs.s, out.data_ptr(), cos.const_data_ptr<float>(),
                                         sin.const_data_ptr<float>(), cos.size(0), pos.tp(), pos.yp(), pos.xp(),
                                         pos.row_stride, gh, gw, (int)B, (int)H, (int)T, (int)Dh, code_t, check.arg(), st); });
    if (refused) return refused_result();
    return wrap(out);
  });
}

// what every attention call asks of its cache and frame index
void check_attn(const Tensor& q, const Tensor& kv, const Tensor& written, const Tensor& t_pos, int64_t L) {
  if (q.dim() != 4) fail("q must be [B, H, T, Dh]");
  const int64_t B = q.size(0), T = q.size(2), Dh = q.size(3);
  if (kv.dim() != 5 || kv.size(0) != 2 || kv.size(1) != B || kv.size(3) != L + T || kv.size(4) != Dh)
    fail("kv must be [2, B, Hkv, L+T, Dh] matching q");
  if (!kv.is_contiguous() || kv.scalar_type() != q.scalar_type()) fail("kv must be contiguous and of q's element type");
  if (written.scalar_type() != at::kBool || written.numel() != L + T || !written.is_contiguous())
    fail("written must be a contiguous bool [L+T] tensor");
  if (t_pos.scalar_type() != at::kLong || t_pos.numel() < 1) fail("t_pos must be a non-empty int64 tensor");
}

PyObject* attn_ring(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a("attn_ring", argv, n, 12);
    const Tensor &q = a.tensor(), &kv = a.tensor(), &written = a.tensor(), &t_pos = a.tensor();
    const int64_t L = a.integer(), dilation = a.integer();
    const c10::Device dev = need_device({&q, &kv, &written, &t_pos});
    check_attn(q, kv, written, t_pos, L);
    const int64_t B = q.size(0), H = q.size(1), T = q.size(2), Dh = q.size(3), Hkv = kv.size(2);
    const float scale = (float)a.scale(Dh);
    const int splits = (int)a.integer(), q_tile = (int)a.integer();
    const Tensor *out_in = a.opt_tensor(), *ws_in = a.opt_tensor();
    const bool token_major = a.flag();
    const Strides qs(q, "q");
    const OnDevice on(dev);
    const Workspace ws(ws_in, B, H, Hkv, T, Dh, L, dilation, splits, q_tile, q);
    const Tensor out = output_or_new(out_in, token_major, q, dev, B, H, T, Dh);
    const Strides os(out, "out");
    run("we_attn_ring_fwd", nullptr, [&] { return we_attn_ring_fwd(q.data_ptr(), qs.s, kv.data_ptr(), static_cast<const uint8_t*>(written.data_ptr()),
                                    t_pos.const_data_ptr<int64_t>(), out.data_ptr(), os.s, ws.ptr, ws.bytes, (int)B, (int)H,
                                    (int)Hkv, (int)T, (int)Dh, L, (int)dilation, scale, splits, q_tile, dtype_code(q),
                                    stream_of(dev)); });
    return wrap(out);
  });
}

PyObject* attn_ring_static(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a("attn_ring_static", argv, n, 10);
    const Tensor &q = a.tensor(), &kv = a.tensor(), &written = a.tensor(), &t_pos = a.tensor();
    const int64_t L = a.integer(), dilation = a.integer();
    const Tensor& out = a.tensor();
    const c10::Device dev = need_device({&q, &kv, &written, &t_pos, &out});
    check_attn(q, kv, written, t_pos, L);
    const int64_t B = q.size(0), H = q.size(1), T = q.size(2), Dh = q.size(3), Hkv = kv.size(2);
    const float scale = (float)a.scale(Dh);
    const int splits = (int)a.integer(), q_tile = (int)a.integer();
    if (!is_shape(out, {B, H, T, Dh}) || out.scalar_type() != q.scalar_type())
      fail("out must be [B, H, T, Dh] of q's element type on q's device");
    const Strides qs(q, "q"), os(out, "out");
    const OnDevice on(dev);
    run("we_attn_ring_fwd_static", nullptr, [&] { return we_attn_ring_fwd_static(q.data_ptr(), qs.s, kv.data_ptr(), static_cast<const uint8_t*>(written.data_ptr()),
                                           t_pos.const_data_ptr<int64_t>(), out.data_ptr(), os.s, (int)B, (int)H, (int)Hkv,
                                           (int)T, (int)Dh, L, (int)dilation, scale, splits, q_tile, dtype_code(q),
                                           stream_of(dev)); });
    return none();
  });
}

PyObject* rope_kv_attn(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a("rope_kv_attn", argv, n, 30);
    const Tensor &q = a.tensor(), &k = a.tensor(), &v = a.tensor(), &tp = a.tensor(), &yp = a.tensor(), &xp = a.tensor();
    const Tensor &cos = a.tensor(), &sin = a.tensor();
    const int64_t gh = a.integer(), gw = a.integer();
    const Tensor &kv = a.tensor(), &written = a.tensor();
    const int64_t L = a.integer(), dilation = a.integer();
    const bool frozen = a.flag();
    const c10::Device dev = need_device({&q, &k, &v, &kv, &written, &cos, &sin, &tp, &yp, &xp});
    if (k.dim() != 4 || k.sizes() != v.sizes()) fail("k and v must both be [B, Hkv, T, Dh]");
    const int64_t B = k.size(0), Hkv = k.size(1), T = k.size(2), Dh = k.size(3);
    const float scale = (float)a.scale(Dh);
    const int splits = (int)a.integer(), q_tile = (int)a.integer();
    const Tensor *out_in = a.opt_tensor(), *ws_in = a.opt_tensor(), *q_rot_in = a.opt_tensor();
    const bool token_major = a.flag();
    const double eps = a.number();
    const Tensor *v1 = a.opt_tensor(), *v_lamb = a.opt_tensor(), *gate = a.opt_tensor();
    const Tensor *gate_x = a.opt_tensor(), *gate_w = a.opt_tensor();
    const int what = (int)a.integer();
    const int64_t tpf = a.integer();
    if (tpf > 0 && T != tpf) fail("KV cache expects exactly one frame per upsert");
    if (q.dim() != 4 || q.size(0) != B || q.size(2) != T || q.size(3) != Dh) fail("q must be [B, H, T, Dh] matching k");
    const int64_t H = q.size(1);
    if (k.scalar_type() != kv.scalar_type() || v.scalar_type() != kv.scalar_type() || q.scalar_type() != kv.scalar_type())
      fail("q/k/v must have the cache's element type");
    check_cache(kv, written, B, Hkv, T, Dh, L);
    check_tables(cos, sin, Dh);
    const PosIds pos(tp, &yp, &xp, B, T);
    const Strides qs(q, "q"), ks(k, "k"), vs(v, "v");
    const int code_t = dtype_code(kv);
    const Extras extras(eps, v1, v_lamb, gate, gate_x, gate_w, q.scalar_type(), B, H, Hkv, T, Dh);
    const OnDevice on(dev);
    const hipStream_t st = stream_of(dev);
    const Workspace ws(ws_in, B, H, Hkv, T, Dh, L, dilation, splits, q_tile, q);
    Tensor q_rot;
    if (q_rot_in == nullptr) {
      q_rot = new_heads(q, B, H, T, Dh);
    } else {
      q_rot = *q_rot_in;
      if (!is_shape(q_rot, {B, H, T, Dh}) || q_rot.scalar_type() != q.scalar_type() || q_rot.device() != dev ||
          !q_rot.is_contiguous())
        fail("q_rot must be a contiguous [B, H, T, Dh] tensor of q's element type on q's device");
    }
    const Tensor out = output_or_new(out_in, token_major, q, dev, B, H, T, Dh);
    const Strides os(out, "out");
    PosCheck check(what, dev, st, B, T, false);
    const bool refused = run("we_rope_kv_attn_fwd", &check, [&] { return we_rope_kv_attn_fwd_checked(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), qs.s, ks.s, vs.s, q_rot.data_ptr(), cos.const_data_ptr<float>(),
        sin.const_data_ptr<float>(), cos.size(0), pos.tp(), pos.yp(), pos.xp(), pos.row_stride, gh, gw, kv.data_ptr(),
        static_cast<uint8_t*>(written.data_ptr()), out.data_ptr(), os.s, ws.ptr, ws.bytes, (int)B, (int)H, (int)Hkv, (int)T,
        (int)Dh, L, (int)dilation, frozen ? 1 : 0, scale, splits, q_tile, code_t, extras.ptr(), check.arg(), st); });
    if (refused) return refused_result();
    return pack({&out, &q_rot});
  });
}

PyObject* qkv_rope_kv_attn(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a("qkv_rope_kv_attn", argv, n, 32);
    const Tensor &x = a.tensor(), &w = a.tensor();
    const int64_t H = a.integer(), Hkv = a.integer();
    const Tensor &tp = a.tensor(), &yp = a.tensor(), &xp = a.tensor(), &cos = a.tensor(), &sin = a.tensor();
    const int64_t gh = a.integer(), gw = a.integer();
    const Tensor &kv = a.tensor(), &written = a.tensor();
    const int64_t L = a.integer(), dilation = a.integer();
    const bool frozen = a.flag();
    const c10::Device dev = need_device({&x, &w, &kv, &written, &cos, &sin, &tp, &yp, &xp});
    if (x.dim() != 3 || x.stride(2) != 1) fail("x must be [B, T, d_model] with contiguous channels");
    const int64_t B = x.size(0), T = x.size(1), d_model = x.size(2);
    if (kv.dim() != 5) fail("kv must be [2, B, Hkv, L+T, Dh]");
    const int64_t Dh = kv.size(4);
    const float scale = (float)a.scale(Dh);
    const int splits = (int)a.integer(), q_tile = (int)a.integer();
    const bool attend = a.flag(), want_v = a.flag();
    const double eps = a.number();
    const Tensor *v1 = a.opt_tensor(), *v_lamb = a.opt_tensor(), *gate = a.opt_tensor();
    const Tensor *gate_x = a.opt_tensor(), *gate_w = a.opt_tensor();
    const Tensor *out_in = a.opt_tensor(), *ws_in = a.opt_tensor(), *q_rot_in = a.opt_tensor();
    const int what = (int)a.integer();
    const int64_t tpf = a.integer();
    if (tpf > 0 && T != tpf) fail("KV cache expects exactly one frame per upsert");
    if (!attend && what != 0) fail("qkv_rope_kv_attn: a call without attention has no check of its position ids");
    if (w.dim() != 2 || !is_shape(w, {(H + 2 * Hkv) * Dh, d_model}) || w.stride(1) != 1)
      fail("w_qkv must be [(H + 2 Hkv) * Dh, d_model] with contiguous rows");
    if (x.scalar_type() != kv.scalar_type() || w.scalar_type() != kv.scalar_type())
      fail("x and w_qkv must have the cache's element type");
    check_cache(kv, written, B, Hkv, T, Dh, L);
    check_tables(cos, sin, Dh);
    const PosIds pos(tp, &yp, &xp, B, T);
    const int code_t = dtype_code(kv);
    const Extras extras(eps, v1, v_lamb, gate, gate_x, gate_w, x.scalar_type(), B, H, Hkv, T, Dh);
    const OnDevice on(dev);
    const hipStream_t st = stream_of(dev);
    const Tensor q_rot = q_rot_in != nullptr ? *q_rot_in : new_heads(x, B, H, T, Dh);
    we_qkv_proj proj{};
    proj.x = x.data_ptr(); proj.w = w.data_ptr(); proj.d_model = (int)d_model;
    proj.x_strides[0] = x.stride(0); proj.x_strides[1] = x.stride(1);
    proj.w_row_stride = w.stride(0);
    Tensor v_raw;
    if (want_v) {  // token-major like the projection output the module would have sliced it from
      v_raw = new_token_major(x, B, Hkv, T, Dh);
      const Strides s(v_raw, "v_out");
      proj.v_out = v_raw.data_ptr();
      for (int i = 0; i < 3; ++i) proj.v_out_strides[i] = s.s[i];
    }
    Tensor out;
    PosCheck check(what, dev, st, B, T, true);
    if (!attend) {
      run("we_qkv_rope_kv_store", nullptr, [&] { return we_qkv_rope_kv_store(&proj, q_rot.data_ptr(), cos.const_data_ptr<float>(), sin.const_data_ptr<float>(),
                                          cos.size(0), pos.tp(), pos.yp(), pos.xp(), pos.row_stride, gh, gw, kv.data_ptr(),
                                          static_cast<uint8_t*>(written.data_ptr()), (int)B, (int)H, (int)Hkv, (int)T, (int)Dh,
                                          L, (int)dilation, frozen ? 1 : 0, code_t, extras.ptr(), st); });
    } else {
      const Workspace ws(ws_in, B, H, Hkv, T, Dh, L, dilation, splits, q_tile, x);
      out = output_or_new(out_in, true, x, dev, B, H, T, Dh);
      const Strides os(out, "out");
      const bool refused = run("we_qkv_rope_kv_attn_fwd", &check, [&] { return we_qkv_rope_kv_attn_fwd_checked(
          &proj, q_rot.data_ptr(), cos.const_data_ptr<float>(), sin.const_data_ptr<float>(), cos.size(0), pos.tp(), pos.yp(),
          pos.xp(), pos.row_stride, gh, gw, kv.data_ptr(), static_cast<uint8_t*>(written.data_ptr()), out.data_ptr(), os.s,
          ws.ptr, ws.bytes, (int)B, (int)H, (int)Hkv, (int)T, (int)Dh, L, (int)dilation, frozen ? 1 : 0, scale, splits, q_tile,
          code_t, extras.ptr(), check.arg(), st); });
      if (refused) return refused_result();
    }
    return pack({&out, &q_rot, &v_raw});
  });
}

// plain(t, ...): whether an operation on these tensors can be done on their memory without anybody
// missing it - tensors (or parameters) of no other class, of one element type and device, nobody
// watching, no gradient or tangent to carry on.
PyObject* plain(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a("plain", argv, n, n);
    bool ok = !watched();
    const Tensor* first = nullptr;
    for (Py_ssize_t i = 0; i < n && ok; ++i) {
      const Tensor& t = a.tensor();
      if (first == nullptr) first = &t;
      ok = THPVariable_CheckExact(argv[i]) && plain_memory(t) && !to_record(t) && t.scalar_type() == first->scalar_type() &&
           t.device() == first->device();
    }
    return PyBool_FromLong(ok ? 1 : 0);
  });
}

// The same for what the store kernel's blend reads: v, the value rows it is blended with (contiguous rows on
// 16-byte boundaries) and the weight.
PyObject* blend_ready(PyObject* self, PyObject* const* argv, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a("blend_ready", argv, n, 3);
    a.tensor();
    const Tensor& t = a.tensor();
    const int64_t per16 = 16 / (int64_t)t.element_size();
    if (t.dim() != 4 || t.stride(3) != 1 || t.stride(0) % per16 != 0 || t.stride(1) % per16 != 0 || t.stride(2) % per16 != 0 ||
        !t.has_storage() || (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15u) != 0)
      Py_RETURN_FALSE;
    return plain(self, argv, n);
  });
}
// And for the head gate in the attention's epilogue: x (contiguous channels), gate_proj's weight (contiguous), q; one
// half-precision type.
PyObject* gate_ready(PyObject* self, PyObject* const* argv, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a("gate_ready", argv, n, 3);
    const Tensor &x = a.tensor(), &w = a.tensor();
    if ((x.scalar_type() != at::kBFloat16 && x.scalar_type() != at::kHalf) || x.stride(-1) != 1 || !w.is_contiguous()) Py_RETURN_FALSE;
    return plain(self, argv, n);
  });
}

// And for the norm of the query and key rows in the store kernel: half-precision rows of 64 or 128 on 16-byte
// boundaries, on a GPU.
PyObject* norm_ready(PyObject* self, PyObject* const* argv, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a("norm_ready", argv, n, 2);
    for (int i = 0; i < 2; ++i) {
      const Tensor& t = a.tensor();
      if (!t.is_cuda() || (t.scalar_type() != at::kBFloat16 && t.scalar_type() != at::kHalf) || t.dim() != 4 ||
          (t.size(3) != 64 && t.size(3) != 128) || t.stride(3) != 1 || t.stride(0) % 8 != 0 || t.stride(1) % 8 != 0 ||
          t.stride(2) % 8 != 0 || !t.has_storage() || (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15u) != 0)
        Py_RETURN_FALSE;
    }
    return plain(self, argv, n);
  });
}

// x [..., K] times w [N, K] transposed; None where the kernel is not the one to use (shape, layout,
// element type, a gradient to record, somebody who watches torch's operations): the caller then takes
// its linear layer.
PyObject* linear(PyObject*, PyObject* const* argv, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a("linear", argv, n, 2);
    const Tensor &x = a.tensor(), &w = a.tensor();
    if (watched()) return none();
    if (!x.is_cuda() || w.device() != x.device() || !plain_memory(x) || !plain_memory(w) || x.dim() < 2 || w.dim() != 2) return none();
    const at::ScalarType dt = x.scalar_type();
    if ((dt != at::kBFloat16 && dt != at::kHalf) || w.scalar_type() != dt) return none();
    if (to_record(x) || to_record(w)) return none();
    const int64_t K = x.size(-1), N = w.size(0), M = K > 0 ? x.numel() / K : 0;
    const int64_t xs = x.stride(-2);
    if (w.size(1) != K || M <= 0 || M > (1 << 20) || N > (1 << 24) || x.stride(-1) != 1 || w.stride(1) != 1) return none();
    int64_t step = xs;  // rows of all leading dimensions at one distance
    for (int64_t d = x.dim() - 3; d >= 0; --d) {
      step *= x.size(d + 1);
      if (x.size(d) > 1 && x.stride(d) != step) return none();
    }
    const OnDevice on(x.device());
    if (we_linear_covers((int)M, (int)N, (int)K, dtype_code(x)) == 0) return none();
    c10::SmallVector<int64_t, 4> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = N;
    const Tensor y = at::empty(shape, x.options());
    int rc = WE_OK;
    {
      const NoGil off;
      rc = we_linear(x.data_ptr(), xs, w.data_ptr(), w.stride(0), y.data_ptr(), N, (int)M, (int)N, (int)K, dtype_code(x),
                     stream_of(x.device()));
    }
    if (rc == WE_ERR_ALIGNMENT || rc == WE_ERR_UNSUPPORTED || rc == WE_ERR_BAD_SHAPE) return none();
    if (rc != WE_OK) fail_code("we_linear", rc);
    return wrap(y);
  });
}

PyMethodDef methods[] = {
    {"plain", (PyCFunction)(void (*)(void))plain, METH_FASTCALL, nullptr},
    {"blend_ready", (PyCFunction)(void (*)(void))blend_ready, METH_FASTCALL, nullptr},
    {"gate_ready", (PyCFunction)(void (*)(void))gate_ready, METH_FASTCALL, nullptr},
    {"norm_ready", (PyCFunction)(void (*)(void))norm_ready, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void (*)(void))linear, METH_FASTCALL, nullptr},
    {"rope_kv_store", (PyCFunction)(void (*)(void))rope_kv_store, METH_FASTCALL, nullptr},
    {"rope_apply", (PyCFunction)(void (*)(void))rope_apply, METH_FASTCALL, nullptr},
    {"attn_ring", (PyCFunction)(void (*)(void))attn_ring, METH_FASTCALL, nullptr},
    {"attn_ring_static", (PyCFunction)(void (*)(void))attn_ring_static, METH_FASTCALL, nullptr},
    {"rope_kv_attn", (PyCFunction)(void (*)(void))rope_kv_attn, METH_FASTCALL, nullptr},
    {"qkv_rope_kv_attn", (PyCFunction)(void (*)(void))qkv_rope_kv_attn, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
