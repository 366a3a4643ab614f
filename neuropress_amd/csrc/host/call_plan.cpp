// CallPlan: one lowered module's forward call with everything that stays the same from call to call
// worked out once, issued from native code.
//
// What bounds a decode step of small layers is the time to issue its launches, not the kernels: through
// Python argument checks and ctypes a call took 12-19 us of host time against 3-9 us of kernel.  Through a plan it
// takes 3.4 us in a stream of calls, 2.4 of them the HIP launch itself and 0.5 the output's allocation (us per eager call, before / now:
// 2048 x 640 with a 256-row codebook 15.1 / 3.5, the nine calls of a block with hidden size 2048 132 / 36).  In other processes
// the same calls take 4.3 and 44: the first 75 or so launches behind a synchronisation then cost 6 to 12 us each, inside the
// runtime.  A bare loop over the launch shows it as well; what selects it is which CPU the scheduler gives the runtime's own
// thread, busy with the commands of the time before while this one launches (moved by hand, each process goes from one state
// to the other, whatever this file does).  (Residual VQ 4096 x 4096 18.1 / 8.2 and int4 14336 x 4096 12.6 / 8.2
// are bound by their kernels.)  The looks at what torch follows (tracked) are 0.03 of it.  A plan
// keeps the entry point's constant arguments (addresses, sizes, the kernel that serves a token count) and does
// per call only what depends on the call: check that nothing it was built from has changed, allocate the output,
// pass the addresses on.
//
// A plan never decides anything: which kernel serves how many tokens, and when a layer's derived tensors are
// stale, stays the Python module's business.  Whatever a plan has not been told about (a token count, a dtype, a
// layout, a changed buffer or threshold, an error from the library) makes the call return None, and the module
// takes its ordinary route, which checks and reports.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/index_select.h>
#include <ATen/ops/linear.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <algorithm>
#include <deque>
#include <unordered_map>
#include <vector>

#include "../../../include/npamd.h"

namespace {

enum Kind : int {
  kSliced = 0,
  kVqGemv, kVqGemvPerm, kVqTile, kVqDense,
  kRvqGemv, kRvqTile, kRvqDense,
  kQGemv, kQTile, kQDense,
  kRmsNorm, kVqEmbedding, kQEmbedding,
  kVqSlice,
  kVqBlocks, kRvqBlocks, kQBlocks,  // the *_gemv_blocks entry points: any number of tokens, rows of x that end inside the last 64 columns
  kKinds,
};

// Constant arguments each kind takes, in the order of its entry point (see issue()).
constexpr int kArgs[kKinds] = {7, 9, 10, 9, 7, 15, 15, 13, 9, 9, 9, 2, 8, 8, 9, 9, 15, 9};

// A dictionary some of whose entries the plan was built from.  CPython stamps a dictionary with a new tag on every
// change, so an unchanged tag means unchanged entries; after a change the entries themselves are compared.
struct Guard {
  PyObject* dict = nullptr;  // borrowed for the module's own __dict__, owned otherwise
  bool wrappers = false;     // entries that instrumentation replaces: the plan's own calls step aside for them, no more
  uint64_t tag = 0;
  std::vector<std::pair<PyObject*, PyObject*>> entries;  // owned; a null value: the key has to be absent
};

uint64_t dict_tag(PyObject* dict) {
#if PY_VERSION_HEX < 0x030C0000
  return reinterpret_cast<PyDictObject*>(dict)->ma_version_tag;
#else
  (void)dict;
  return 0;  // no tag in this interpreter: the entries are compared on every call
#endif
}

bool holds(Guard& g, PyObject* dict) {
  const uint64_t tag = dict_tag(dict);
  if (tag != 0 && tag == g.tag && dict == g.dict) return true;
  for (const auto& e : g.entries)
    if (PyDict_GetItemWithError(dict, e.first) != e.second) {
      PyErr_Clear();
      return false;
    }
  g.dict = dict;
  g.tag = tag;
  return true;
}

// A buffer the plan's derived tensors were made from: the same tensor, at the same place, not written to since.
struct Source {
  at::Tensor tensor;
  const void* data;
  int64_t version;  // -1: an inference tensor, which counts no versions
};

int64_t version_of(const at::Tensor& t) {
  return t.is_inference() ? -1 : (int64_t)t.unsafeGetTensorImpl()->version_counter().current_version();
}

struct Template {
  Kind kind;
  int64_t n, k;                     // output features, columns the kernel contracts (embedding lookups: row length, 1)
  int64_t k_in;                     // columns of x: fewer than k where rows are padded to whole 64-column chunks
  std::vector<int64_t> a;           // constant arguments
  double f;                         // eps of a norm, scale of an embedding
  at::ScalarType out;
  at::Tensor perm;                  // column permutation applied to x first, or undefined: int32 (16-bit x) or int64
  at::Tensor bias;                  // bias of the dense product, or undefined: float32 for the framework's own
  at::Tensor leaf;                  // dense kinds: the module's bias itself, which may ask for a gradient
  bool own;                         // dense kinds: the framework's own product, not the library's
  std::vector<at::Tensor> keep;     // what the addresses point into
};

struct Route {
  int tmpl;
  int64_t ws;  // bytes of scratch (for kSliced: bytes of the shared zero-filled one)
};

struct Plan {
  PyObject_HEAD
  vectorcallfunc call;
  PyObject* names;  // dict: what the module calls its templates
  int device;
  bool guarded;
  Guard self;  // entries of the module's own __dict__
  std::vector<Guard>* guards;
  // What `module(x)` may go straight to the plan under: the class whose forward the plan stands for (null: not at all),
  // and that torch's own call of a module would do nothing but call that forward.
  PyTypeObject* direct_type;
  Guard direct_self;                   // entries of the module's own __dict__
  std::vector<Guard>* direct_guards;   // of its class and of torch.nn.Module
  std::vector<PyObject*>* hooks;       // dictionaries of hooks, all of which have to be empty
  std::vector<PyObject*>* held;
  std::vector<Source>* sources;
  std::deque<Template>* templates;
  std::unordered_map<int64_t, Route>* routes;  // key: dtype code << 32 | tokens
  // Streams on which the plan and its templates were made -- and, just before, the tensors derived for them (a bias in the
  // activations' type, a widened index stream) -- and the other streams that have waited for those.
  std::vector<hipStream_t>* made;
  std::vector<hipStream_t>* ordered;
};

PyObject* g_workspaces = nullptr;       // {(device, stream): zero-filled scratch of the slice-list GEMV}
PyObject* g_drop_workspace = nullptr;   // called as drop(device, stream) after a call that failed part-way

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kHalf: return NPAMD_F16;
    case at::kBFloat16: return NPAMD_BF16;
    case at::kFloat: return NPAMD_F32;
    case at::kLong: return 3;
    default: return -1;
  }
}

at::ScalarType scalar_type(int code) {
  return code == NPAMD_F16 ? at::kHalf : code == NPAMD_BF16 ? at::kBFloat16 : at::kFloat;
}

at::Tensor empty(at::IntArrayRef sizes, at::ScalarType t, int device) {
  return at::Tensor(at::detail::empty_cuda(sizes, t, c10::Device(c10::kCUDA, (c10::DeviceIndex)device), std::nullopt));
}

// The slice-list GEMV's scratch on this device and stream, as the Python side allocated it; the last answer is
// reused while the dictionary is unchanged.
bool sliced_scratch(int device, hipStream_t stream, int64_t need, void** ptr, int64_t* bytes) {
  static struct { uint64_t tag; int device; hipStream_t stream; void* ptr; int64_t bytes; } last = {0, -1, nullptr, nullptr, 0};
  const uint64_t tag = dict_tag(g_workspaces);
  if (tag == 0 || tag != last.tag || device != last.device || stream != last.stream) {
    PyObject* key = Py_BuildValue("(in)", device, (Py_ssize_t)(intptr_t)stream);
    if (!key) { PyErr_Clear(); return false; }
    PyObject* ws = PyDict_GetItemWithError(g_workspaces, key);
    Py_DECREF(key);
    if (!ws || !THPVariable_Check(ws)) { PyErr_Clear(); return false; }
    const at::Tensor& t = THPVariable_Unpack(ws);
    last = {tag, device, stream, t.data_ptr(), t.numel() * (int64_t)t.element_size()};
  }
  if (last.bytes < need) return false;
  *ptr = last.ptr;
  *bytes = last.bytes;
  return true;
}

template <class T>
T ptr(int64_t v) { return reinterpret_cast<T>((uintptr_t)v); }

using U8 = const uint8_t*;
using F32 = const float*;
using I32 = const int32_t*;

hipStream_t current_stream(int device) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

bool contains(const std::vector<hipStream_t>& streams, hipStream_t st) {
  return std::find(streams.begin(), streams.end(), st) != streams.end();
}

void made_on(Plan* p, hipStream_t st) {
  if (contains(*p->made, st)) return;
  p->made->push_back(st);
  p->ordered->clear();
}

bool capturing(hipStream_t st) {
  hipStreamCaptureStatus status;
  if (hipStreamIsCapturing(st, &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;  // the legacy stream while another one is
}

// A call on a stream the plan was not made on: let that stream wait, once, for what was made on the others.  Not inside a
// capture or for a stream inside one (captures start on an idle GPU, and an event would tie the streams together).  False:
// could not be arranged.
bool order_after_making(Plan* p, hipStream_t st) {
  if (contains(*p->ordered, st) || capturing(st)) return true;
  const c10::DeviceGuard guard(c10::Device(c10::kCUDA, (c10::DeviceIndex)p->device));
  for (hipStream_t from : *p->made) {
    if (from == st || capturing(from)) continue;
    hipEvent_t done = nullptr;
    const bool ok = hipEventCreateWithFlags(&done, hipEventDisableTiming) == hipSuccess && hipEventRecord(done, from) == hipSuccess &&
                    hipStreamWaitEvent(st, done, 0) == hipSuccess;
    if (done) (void)hipEventDestroy(done);  // freed once it has happened
    if (!ok) {
      (void)hipGetLastError();
      return false;
    }
  }
  if (p->ordered->size() >= 64) p->ordered->clear();  // bounded, however many streams a program makes
  p->ordered->push_back(st);
  return true;
}

// Launches template t on x ([m, k], row stride ldx); the output in *out.  False: not issued, or it failed.
bool issue(const Template& t, const Route& r, const at::Tensor& x_in, int64_t m, int64_t ldx, int device, hipStream_t st,
           at::Tensor* out) {
  if (t.leaf.defined() && t.leaf.requires_grad() && c10::GradMode::is_enabled()) return false;
  const std::vector<int64_t>& a = t.a;
  c10::SmallVector<int64_t, 6> sizes(x_in.sizes().begin(), x_in.sizes().end());
  at::Tensor x = x_in;
  const int64_t ldx_in = ldx;
  bool with_gather = false;
  const bool blocks = t.kind == kVqBlocks || t.kind == kRvqBlocks || t.kind == kQBlocks;
  // The package's product and the blocks entries read 16 bytes at a time: rows that do not start at such addresses, or lie too far apart, are copied first.
  const bool copied = (blocks || t.own) && (ldx % 8 || ldx >= NPAMD_TILE_MAX_STRIDE || ((uintptr_t)x_in.const_data_ptr() & 15));
  if (t.perm.defined() && t.perm.scalar_type() == at::kLong) {
    x = at::index_select(x_in, -1, t.perm);
    ldx = t.k;
  } else if (t.perm.defined() || copied || (t.k_in != t.k && !blocks)) {
    sizes.back() = t.k;
    x = empty(sizes, x_in.scalar_type(), device);
    with_gather = t.kind == kVqDense && t.own;  // its decode gathers them too
    if (!with_gather && npamd_gather_columns(x_in.const_data_ptr(), ldx, t.perm.defined() ? t.perm.const_data_ptr<int32_t>() : nullptr, x.data_ptr(),
                             t.k, (int)m, (int)t.k_in, st) != NPAMD_OK)
      return false;
    ldx = t.k;
  }
  if (t.kind == kVqEmbedding || t.kind == kQEmbedding) sizes.push_back(t.n);
  else sizes.back() = t.n;

  if (t.kind == kVqDense || t.kind == kRvqDense || t.kind == kQDense) {
    const int code = dtype_code(t.out);
    at::Tensor w = empty({t.n, t.k}, t.out, device);
    int rc;
    if (with_gather)
      rc = npamd_vq_dequant_gather(ptr<U8>(a[0]), a[1], (int)a[2], ptr<void*>(a[3]), (int)a[4], (int)a[5], a[6], w.data_ptr(), code,
                                   x_in.const_data_ptr(), ldx_in, t.perm.defined() ? t.perm.const_data_ptr<int32_t>() : nullptr,
                                   x.data_ptr(), t.k, (int)m, (int)t.k_in, st);
    else if (t.kind == kVqDense)
      rc = npamd_vq_dequant(ptr<U8>(a[0]), a[1], (int)a[2], ptr<void*>(a[3]), (int)a[4], (int)a[5], a[6], w.data_ptr(), code, st);
    else if (t.kind == kRvqDense)
      rc = npamd_rvq_dequant(ptr<U8>(a[0]), a[1], (int)a[2], ptr<U8>(a[3]), a[4], (int)a[5], ptr<void*>(a[6]), (int)a[7],
                             ptr<void*>(a[8]), (int)a[9], ptr<void*>(a[10]), ptr<void*>(a[11]), (int)a[12], (int)t.n, (int)t.k,
                             w.data_ptr(), code, st);
    else
      rc = npamd_q_dequant(ptr<U8>(a[0]), ptr<void*>(a[1]), ptr<void*>(a[2]), (int)t.n, (int)t.k, (int)a[6], (int)a[7],
                           w.data_ptr(), code, st);
    if (rc != NPAMD_OK) return false;
    if (t.own) {
      at::Tensor parts;
      if (r.ws > 0) parts = empty({r.ws / 4}, at::kFloat, device);
      at::Tensor y = empty(sizes, t.out, device);
      if ((t.k % 64 ? npamd_dense_gemm_ragged : npamd_dense_gemm)(x.const_data_ptr(), ldx, w.data_ptr(), t.k, t.bias.defined() ? t.bias.const_data_ptr<float>() : nullptr,
                           y.data_ptr(), t.n, (int)m, (int)t.n, (int)t.k, code, r.ws > 0 ? parts.data_ptr() : nullptr, r.ws, st) != NPAMD_OK)
        return false;
      *out = std::move(y);
      return true;
    }
    *out = at::linear(x, w, t.bias.defined() ? std::optional<at::Tensor>(t.bias) : std::nullopt);
    return true;
  }

  void* ws = nullptr;
  int64_t ws_bytes = 0;
  at::Tensor scratch;
  if (t.kind == kSliced) {
    if (!sliced_scratch(device, st, r.ws, &ws, &ws_bytes)) return false;
  } else if (r.ws > 0) {
    scratch = empty({r.ws / 4}, at::kFloat, device);
    ws = scratch.data_ptr();
    ws_bytes = r.ws;
  }
  at::Tensor y = empty(sizes, t.out, device);
  const void* xp = x.const_data_ptr();
  void* yp = y.data_ptr();
  const int M = (int)m, N = (int)t.n, K = (int)t.k;
  // Also of a padded copy: residual rows have no filler whose product with a padded zero is sure to be one.
  const int x_columns = (int)t.k_in;
  int rc = NPAMD_ERR_INVALID;
  switch (t.kind) {
    case kSliced:
      rc = npamd_vq_gemv_sliced(xp, ldx, ptr<I32>(a[0]), ptr<const npamd_sliced_header*>(a[1]), ptr<void*>(a[2]), ptr<void*>(a[3]), (int)a[4],
                                ptr<F32>(a[5]), yp, t.n, M, (int)a[6], ws, ws_bytes, st);
      if (rc != NPAMD_OK) {  // a launch of a multi-pass call may have run: the shared buffer is not known to be zero
        PyObject* done = PyObject_CallFunction(g_drop_workspace, "in", device, (Py_ssize_t)(intptr_t)st);
        if (!done) PyErr_Clear();
        Py_XDECREF(done);
      }
      break;
    case kVqGemv:
      rc = npamd_vq_gemv(xp, ldx, ptr<U8>(a[0]), a[1], (int)a[2], ptr<void*>(a[3]), (int)a[4], (int)a[5], (int)a[6],
                         ptr<F32>(a[7]), yp, t.n, M, N, K, (int)a[8], st);
      break;
    case kVqBlocks:
      rc = npamd_vq_gemv_blocks(xp, ldx, x_columns, ptr<U8>(a[0]), a[1], (int)a[2], ptr<void*>(a[3]), (int)a[4], (int)a[5], (int)a[6],
                                ptr<F32>(a[7]), yp, t.n, M, N, K, (int)a[8], st);
      break;
    case kVqGemvPerm:
      rc = npamd_vq_gemv_perm(xp, ldx, ptr<I32>(a[9]), ptr<U8>(a[0]), a[1], (int)a[2], ptr<void*>(a[3]), (int)a[4],
                              (int)a[5], (int)a[6], ptr<F32>(a[7]), yp, t.n, M, N, K, (int)a[8], st);
      break;
    case kVqTile:
      rc = npamd_vq_gemm_tile(xp, ldx, ptr<U8>(a[0]), a[1], (int)a[2], ptr<void*>(a[3]), (int)a[4], (int)a[5], (int)a[6],
                              ptr<F32>(a[7]), yp, t.n, M, N, K, (int)a[8], ws, ws_bytes, st);
      break;
    case kVqSlice:
      rc = npamd_vq_slice_gemm(xp, ldx, ptr<U8>(a[0]), a[1], (int)a[2], ptr<void*>(a[3]), (int)a[4], (int)a[5], (int)a[6],
                               ptr<F32>(a[7]), yp, t.n, M, N, K, (int)a[8], ws, ws_bytes, st);
      break;
    case kRvqGemv:
      rc = npamd_rvq_gemv(xp, ldx, ptr<U8>(a[0]), a[1], (int)a[2], ptr<U8>(a[3]), a[4], (int)a[5], ptr<void*>(a[6]), (int)a[7],
                          ptr<void*>(a[8]), (int)a[9], ptr<void*>(a[10]), ptr<void*>(a[11]), (int)a[12], ptr<F32>(a[13]), yp,
                          t.n, M, N, K, (int)a[14], st);
      break;
    case kRvqBlocks:
      rc = npamd_rvq_gemv_blocks(xp, ldx, x_columns, ptr<U8>(a[0]), a[1], (int)a[2], ptr<U8>(a[3]), a[4], (int)a[5], ptr<void*>(a[6]),
                                 (int)a[7], ptr<void*>(a[8]), (int)a[9], ptr<void*>(a[10]), ptr<void*>(a[11]), (int)a[12],
                                 ptr<F32>(a[13]), yp, t.n, M, N, K, (int)a[14], st);
      break;
    case kRvqTile:
      rc = npamd_rvq_gemm_tile(xp, ldx, ptr<U8>(a[0]), a[1], (int)a[2], ptr<U8>(a[3]), a[4], (int)a[5], ptr<void*>(a[6]),
                               (int)a[7], ptr<void*>(a[8]), (int)a[9], ptr<void*>(a[10]), ptr<void*>(a[11]), (int)a[12],
                               ptr<F32>(a[13]), yp, t.n, M, N, K, (int)a[14], ws, ws_bytes, st);
      break;
    case kQGemv:
      rc = npamd_q_gemv(xp, ldx, ptr<U8>(a[0]), ptr<void*>(a[1]), ptr<void*>(a[2]), ptr<F32>(a[3]), yp, t.n, M, N, K,
                        (int)a[6], (int)a[7], (int)a[8], st);
      break;
    case kQBlocks:
      rc = npamd_q_gemv_blocks(xp, ldx, ptr<U8>(a[0]), ptr<void*>(a[1]), ptr<void*>(a[2]), ptr<F32>(a[3]), yp, t.n, M, N, K,
                               (int)a[6], (int)a[7], (int)a[8], st);
      break;
    case kQTile:
      rc = npamd_q_gemm_tile(xp, ldx, ptr<U8>(a[0]), ptr<void*>(a[1]), ptr<void*>(a[2]), ptr<F32>(a[3]), yp, t.n, M, N, K,
                             (int)a[6], (int)a[7], (int)a[8], ws, ws_bytes, st);
      break;
    case kRmsNorm:
      rc = npamd_rms_norm(xp, ldx, ptr<void*>(a[0]), yp, t.n, M, N, (float)t.f, (int)a[1], st);
      break;
    case kVqEmbedding:
      rc = npamd_vq_embedding((const int64_t*)xp, m, ptr<const int16_t*>(a[0]), a[1], (int)a[2], ptr<void*>(a[3]), (int)a[4], (int)a[5],
                              ptr<I32>(a[6]), (float)t.f, yp, (int)a[7], st);
      break;
    case kQEmbedding:
      rc = npamd_q_embedding((const int64_t*)xp, m, ptr<U8>(a[0]), ptr<void*>(a[1]), ptr<void*>(a[2]), (int)a[3], (int)a[4],
                             a[5], N, a[6], (float)t.f, yp, (int)a[7], st);
      break;
    default: break;
  }
  if (rc != NPAMD_OK) return false;
  *out = std::move(y);
  return true;
}

bool wrapped(Plan* p) {
  for (Guard& g : *p->guards)
    if (g.wrappers && !holds(g, g.dict)) return true;
  return false;
}

bool stale(Plan* p, PyObject* module) {
  PyObject** dictp = _PyObject_GetDictPtr(module);
  if (!dictp || !*dictp || !holds(p->self, *dictp)) return true;
  for (Guard& g : *p->guards)
    if (!g.wrappers && !holds(g, g.dict)) return true;
  for (const Source& s : *p->sources) {
    if (s.tensor.const_data_ptr() != s.data) return true;
    if (s.version >= 0 && (int64_t)s.tensor.unsafeGetTensorImpl()->version_counter().current_version() != s.version) return true;
  }
  return false;
}

// Whether x is a stack of contiguous rows at one distance (the last tokens of a batch of prompts, say).  Expanded inputs
// are not: their rows lie at distance 0, or at several.
bool rows_at_one_stride(const at::Tensor& x, int64_t* ldx) {
  if (x.stride(-1) != 1) return false;
  bool found = false;
  int64_t row = x.size(-1), next = 0;  // distance of two rows; stride the next dimension outwards must have
  for (int64_t d = x.dim() - 2; d >= 0; --d) {
    if (x.size(d) == 1) continue;
    if (!found) row = x.stride(d);
    else if (x.stride(d) != next) return false;
    found = true;
    next = x.stride(d) * x.size(d);
  }
  *ldx = row;
  return row >= x.size(-1);
}

// Whether torch follows what is done to x: it records a gradient or a trace, x carries a tangent, is a wrapper (vmap, grad
// and jvp of torch.func; a tensor without storage of its own or one that is read negated) or not strided, a dispatch
// mode looks on, or autocast gives the library's product another type than x's.  The kernels read addresses and their outputs carry nothing: no plan issues such a call, and the
// module decides between its kernels and torch's own operations.
bool tracked(const at::Tensor& x) {
  constexpr c10::DispatchKeySet own = c10::autograd_dispatch_keyset | c10::autocast_dispatch_keyset |
                                      c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView);
  const c10::DispatchKeySet keys = x.key_set() - own;
  if (keys != c10::DispatchKeySet(c10::DispatchKey::CUDA) && keys != c10::DispatchKeySet(c10::DispatchKey::CPU)) return true;
  return (x.requires_grad() && c10::GradMode::is_enabled()) || x._fw_grad(0).defined() || torch::jit::tracer::isTracing() ||
         c10::impl::TorchDispatchModeTLS::any_modes_set() ||
         (at::isReducedFloatingType(x.scalar_type()) && at::autocast::is_autocast_enabled(x.device().type()) &&
          at::autocast::get_autocast_dtype(x.device().type()) != x.scalar_type());
}

PyObject* issue_planned(Plan* p, PyObject* xo) {
  if (!THPVariable_CheckExact(xo)) Py_RETURN_NONE;
  const at::Tensor& x = THPVariable_Unpack(xo);
  if (tracked(x)) Py_RETURN_NONE;
  const int code = dtype_code(x.scalar_type());
  const int64_t dims = x.dim();
  if (code < 0 || dims < 1 || !x.is_cuda() || x.get_device() != p->device) Py_RETURN_NONE;
  const bool ids = code == 3;
  const int64_t k = ids ? 1 : x.size(-1);
  if (k == 0) Py_RETURN_NONE;
  int64_t ldx = k;
  const int64_t m = x.numel() / k;
  if (!x.is_contiguous() && (ids || !rows_at_one_stride(x, &ldx))) Py_RETURN_NONE;
  if (m < 1 || m > INT32_MAX) Py_RETURN_NONE;
  auto it = p->routes->find(((int64_t)code << 32) | m);
  if (it == p->routes->end()) {
    it = p->routes->find((int64_t)code << 32);  // a route for any number of tokens
    if (it == p->routes->end()) Py_RETURN_NONE;
  }
  const Route route = it->second;
  const Template& t = (*p->templates)[(size_t)route.tmpl];
  if (t.k_in != k) Py_RETURN_NONE;
  hipStream_t st = current_stream(p->device);
  if ((p->made->size() != 1 || p->made->front() != st) && !order_after_making(p, st)) Py_RETURN_NONE;
  at::Tensor y;
  if (!issue(t, route, x, m, ldx, p->device, st, &y)) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(y));
}

// Runs fn; a C++ exception becomes the Python one torch makes of it (torch.OutOfMemoryError for an allocation that failed).
template <class Fn>
PyObject* translated(Fn&& fn) {
  try {
    return fn();
  } catch (...) {
    torch::translate_exception_to_python(std::current_exception());
    return nullptr;
  }
}

PyObject* run(Plan* p, PyObject* xo) {
  return translated([&] { return issue_planned(p, xo); });
}

// What torch.nn.Module.__call__ looks at before it calls forward: hooks of the module and of all modules, a compiled
// call, a replaced forward (and a trace being recorded, for which tracked() sends the call the long way).
bool direct(Plan* p, PyObject* module) {
  if (Py_TYPE(module) != p->direct_type || !holds(p->direct_self, *_PyObject_GetDictPtr(module))) return false;
  for (Guard& g : *p->direct_guards)
    if (!holds(g, g.dict)) return false;
  for (PyObject* d : *p->hooks)
    if (PyDict_GET_SIZE(d) != 0) return false;
  return true;
}

// plan(module, x)
PyObject* plan_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  Plan* p = reinterpret_cast<Plan*>(self);
  if (PyVectorcall_NARGS(nargsf) != 2 || kwnames) {
    PyErr_SetString(PyExc_TypeError, "CallPlan(module, x)");
    return nullptr;
  }
  return translated([&]() -> PyObject* {
    if (!p->guarded || stale(p, args[0]) || wrapped(p)) Py_RETURN_NONE;
    return issue_planned(p, args[1]);
  });
}

void clear_guard(Guard& g, bool owns_dict) {
  for (auto& e : g.entries) {
    Py_XDECREF(e.first);
    Py_XDECREF(e.second);
  }
  g.entries.clear();
  if (owns_dict) Py_XDECREF(g.dict);
  g.dict = nullptr;
}

PyObject* plan_new(PyTypeObject* type, PyObject* args, PyObject*) {
  int device = 0;
  if (!PyArg_ParseTuple(args, "i", &device)) return nullptr;
  PyObject* names = PyDict_New();
  if (!names) return nullptr;
  Plan* p = reinterpret_cast<Plan*>(type->tp_alloc(type, 0));
  if (!p) {
    Py_DECREF(names);
    return nullptr;
  }
  // tp_alloc has handed the object to the garbage collector: from here to the last member nothing may allocate a
  // Python object.
  p->call = plan_call;
  p->device = device;
  p->guarded = false;
  new (&p->self) Guard();
  p->names = names;
  p->guards = new std::vector<Guard>();
  p->direct_type = nullptr;
  new (&p->direct_self) Guard();
  p->direct_guards = new std::vector<Guard>();
  p->hooks = new std::vector<PyObject*>();
  p->held = new std::vector<PyObject*>();
  p->sources = new std::vector<Source>();
  p->templates = new std::deque<Template>();
  p->routes = new std::unordered_map<int64_t, Route>();
  p->made = new std::vector<hipStream_t>();
  p->ordered = new std::vector<hipStream_t>();
  return reinterpret_cast<PyObject*>(p);
}

int plan_traverse(PyObject* self, visitproc visit, void* arg) {
  Plan* p = reinterpret_cast<Plan*>(self);
  for (Guard* g : {&p->self, &p->direct_self})
    for (auto& e : g->entries) {
      Py_VISIT(e.first);
      Py_VISIT(e.second);
    }
  Py_VISIT(p->direct_type);
  for (PyObject* o : *p->hooks) Py_VISIT(o);
  Py_VISIT(p->names);
  for (PyObject* o : *p->held) Py_VISIT(o);
  for (std::vector<Guard>* list : {p->guards, p->direct_guards})
    for (Guard& g : *list) {
      Py_VISIT(g.dict);
      for (auto& e : g.entries) {
        Py_VISIT(e.first);
        Py_VISIT(e.second);
      }
    }
  return 0;
}

int plan_clear(PyObject* self) {
  Plan* p = reinterpret_cast<Plan*>(self);
  p->guarded = false;
  clear_guard(p->self, false);
  for (Guard& g : *p->guards) clear_guard(g, true);
  p->guards->clear();
  clear_guard(p->direct_self, false);
  for (Guard& g : *p->direct_guards) clear_guard(g, true);
  p->direct_guards->clear();
  Py_CLEAR(p->direct_type);
  for (PyObject* o : *p->hooks) Py_DECREF(o);
  p->hooks->clear();
  Py_CLEAR(p->names);
  for (PyObject* o : *p->held) Py_DECREF(o);
  p->held->clear();
  return 0;
}

void plan_dealloc(PyObject* self) {
  PyObject_GC_UnTrack(self);
  plan_clear(self);
  Plan* p = reinterpret_cast<Plan*>(self);
  p->self.~Guard();
  p->direct_self.~Guard();
  delete p->guards;
  delete p->direct_guards;
  delete p->hooks;
  delete p->held;
  delete p->sources;
  delete p->templates;
  delete p->routes;
  delete p->made;
  delete p->ordered;
  Py_TYPE(self)->tp_free(self);
}

bool fill_guard(Guard& g, PyObject* entries) {
  PyObject *key, *value;
  Py_ssize_t at = 0;
  if (!PyDict_Check(entries)) {
    PyErr_SetString(PyExc_TypeError, "guard entries must be a dict");
    return false;
  }
  while (PyDict_Next(entries, &at, &key, &value)) {
    if (value == Py_Ellipsis) value = nullptr;  // the key has to be absent
    Py_INCREF(key);
    Py_XINCREF(value);
    g.entries.emplace_back(key, value);
  }
  return true;
}

bool make_guard(Guard& g, PyObject* where, PyObject* entries) {
  PyObject* dict = PyType_Check(where) ? reinterpret_cast<PyTypeObject*>(where)->tp_dict : where;
  if (!PyDict_Check(dict)) {
    PyErr_SetString(PyExc_TypeError, "a guard takes a dict or a class");
    return false;
  }
  if (!fill_guard(g, entries)) return false;
  Py_INCREF(dict);
  g.dict = dict;
  return true;
}

// guard(dict_or_type, {key: expected}, wrappers)
PyObject* plan_guard(PyObject* self, PyObject* args) {
  PyObject *where, *entries;
  int wrappers;
  if (!PyArg_ParseTuple(args, "OOp", &where, &entries, &wrappers)) return nullptr;
  Guard g;
  if (!make_guard(g, where, entries)) return nullptr;
  g.wrappers = wrappers != 0;
  reinterpret_cast<Plan*>(self)->guards->push_back(std::move(g));
  Py_RETURN_NONE;
}

// guard_module({attribute: expected}): entries of the calling module's __dict__.  The plan keeps no reference to
// that dictionary (it holds the plan).
PyObject* plan_guard_module(PyObject* self, PyObject* entries) {
  Plan* p = reinterpret_cast<Plan*>(self);
  if (!fill_guard(p->self, entries)) return nullptr;
  p->guarded = true;
  Py_RETURN_NONE;
}

// direct(class, {attribute: expected} of the module, ((dict_or_class, {key: expected}), ...), (dict of hooks, ...))
PyObject* plan_direct(PyObject* self, PyObject* args) {
  Plan* p = reinterpret_cast<Plan*>(self);
  PyObject *type, *own, *guards, *hooks;
  if (p->direct_type || !PyArg_ParseTuple(args, "O!OO!O!", &PyType_Type, &type, &own, &PyTuple_Type, &guards, &PyTuple_Type, &hooks))
    return nullptr;
  if (!fill_guard(p->direct_self, own)) return nullptr;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(guards); ++i) {
    PyObject *where, *entries;
    Guard g;
    if (!PyArg_ParseTuple(PyTuple_GET_ITEM(guards, i), "OO", &where, &entries) || !make_guard(g, where, entries)) return nullptr;
    p->direct_guards->push_back(std::move(g));
  }
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(hooks); ++i) {
    PyObject* d = PyTuple_GET_ITEM(hooks, i);
    if (!PyDict_Check(d)) {
      PyErr_SetString(PyExc_TypeError, "direct(): hooks are dictionaries");
      return nullptr;
    }
    Py_INCREF(d);
    p->hooks->push_back(d);
  }
  Py_INCREF(type);
  p->direct_type = reinterpret_cast<PyTypeObject*>(type);
  Py_RETURN_NONE;
}

// source(tensor or None)
PyObject* plan_source(PyObject* self, PyObject* t) {
  if (t == Py_None) Py_RETURN_NONE;
  if (!THPVariable_Check(t)) {
    PyErr_SetString(PyExc_TypeError, "source() takes a tensor");
    return nullptr;
  }
  return translated([&]() -> PyObject* {
    const at::Tensor& v = THPVariable_Unpack(t);
    Plan* p = reinterpret_cast<Plan*>(self);
    p->sources->push_back({v, v.const_data_ptr(), version_of(v)});
    made_on(p, current_stream(p->device));  // as are the derived tensors that a module prepares when it reaches the GPU
    Py_RETURN_NONE;
  });
}

// hold(object): something the template's addresses point into that is not a tensor
PyObject* plan_hold(PyObject* self, PyObject* o) {
  Py_INCREF(o);
  reinterpret_cast<Plan*>(self)->held->push_back(o);
  Py_RETURN_NONE;
}

// template(kind, n, k, k_in, args, f, out_dtype_code, perm or None, bias or None, leaf or None, own, keep) -> number
PyObject* plan_template(PyObject* self, PyObject* args) {
  Plan* p = reinterpret_cast<Plan*>(self);
  int kind, out_code, own;
  long long n, k, k_in;
  double f;
  PyObject *ints, *perm, *bias, *leaf, *keep;
  if (!PyArg_ParseTuple(args, "iLLLO!diOOOpO!", &kind, &n, &k, &k_in, &PyTuple_Type, &ints, &f, &out_code, &perm, &bias, &leaf, &own,
                        &PyTuple_Type, &keep))
    return nullptr;
  if (kind < 0 || kind >= kKinds || (int)PyTuple_GET_SIZE(ints) > kArgs[kind]) {
    PyErr_SetString(PyExc_ValueError, "template(): bad kind or argument count");
    return nullptr;
  }
  Template t;
  t.kind = (Kind)kind;
  t.n = n;
  t.k = k;
  t.k_in = k_in;
  t.f = f;
  t.own = own != 0;
  t.out = scalar_type(out_code);
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(ints); ++i) {
    PyObject* v = PyTuple_GET_ITEM(ints, i);
    const long long value = v == Py_None ? 0 : PyLong_AsLongLong(v);
    if (value == -1 && PyErr_Occurred()) return nullptr;
    t.a.push_back(value);
  }
  t.a.resize((size_t)kArgs[kind], 0);
  if (perm != Py_None) t.perm = THPVariable_Unpack(perm);
  if (bias != Py_None) t.bias = THPVariable_Unpack(bias);
  if (leaf != Py_None) t.leaf = THPVariable_Unpack(leaf);
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(keep); ++i) {
    PyObject* v = PyTuple_GET_ITEM(keep, i);
    if (v != Py_None && THPVariable_Check(v)) t.keep.push_back(THPVariable_Unpack(v));
  }
  return translated([&] {
    made_on(p, current_stream(p->device));
    p->templates->push_back(std::move(t));
    return PyLong_FromSize_t(p->templates->size() - 1);
  });
}

// route(dtype_code, tokens (0: any number), template, scratch_bytes)
PyObject* plan_route(PyObject* self, PyObject* args) {
  Plan* p = reinterpret_cast<Plan*>(self);
  int code, tmpl;
  long long m, ws;
  if (!PyArg_ParseTuple(args, "iLiL", &code, &m, &tmpl, &ws)) return nullptr;
  if (code < 0 || code > 3 || m < 0 || m > INT32_MAX || tmpl < 0 || (size_t)tmpl >= p->templates->size()) {
    PyErr_SetString(PyExc_ValueError, "route(): out of range");
    return nullptr;
  }
  if (p->routes->size() > 65536) p->routes->clear();  // bounded, whatever token counts a server sees
  (*p->routes)[((int64_t)code << 32) | m] = Route{tmpl, ws};
  Py_RETURN_NONE;
}

PyObject* plan_stale(PyObject* self, PyObject* module) {
  Plan* p = reinterpret_cast<Plan*>(self);
  return translated([&] { return PyBool_FromLong(!p->guarded || stale(p, module)); });
}

PyObject* plan_wrapped(PyObject* self, PyObject*) { return PyBool_FromLong(wrapped(reinterpret_cast<Plan*>(self))); }

PyObject* plan_run(PyObject* self, PyObject* x) { return run(reinterpret_cast<Plan*>(self), x); }

// A plan holds addresses: a copied or unpickled module starts without one.
PyObject* plan_reduce(PyObject*, PyObject*) { return Py_BuildValue("(O())", Py_TYPE(Py_None)); }

PyMethodDef plan_methods[] = {
    {"guard", plan_guard, METH_VARARGS, "guard(dict_or_class, {key: expected}, wrappers)"},
    {"guard_module", plan_guard_module, METH_O, "guard_module({attribute: expected})"},
    {"direct", plan_direct, METH_VARARGS, "direct(class, own, guards, hooks): when module(x) may go straight to the plan"},
    {"source", plan_source, METH_O, "source(tensor or None)"},
    {"hold", plan_hold, METH_O, "hold(object)"},
    {"template", plan_template, METH_VARARGS, "template(kind, n, k, k_in, args, f, out, perm, bias, leaf, own, keep) -> number"},
    {"route", plan_route, METH_VARARGS, "route(dtype, tokens, template, scratch_bytes)"},
    {"stale", plan_stale, METH_O, "stale(module): whether anything the plan was built from has changed"},
    {"wrapped", plan_wrapped, METH_NOARGS, "wrapped(): whether a wrapper function has been replaced"},
    {"run", plan_run, METH_O, "run(x): the call without the checks of the module"},
    {"__reduce__", plan_reduce, METH_NOARGS, ""},
    {nullptr, nullptr, 0, nullptr},
};

PyMemberDef plan_members[] = {
    {"names", T_OBJECT_EX, offsetof(Plan, names), READONLY, "template numbers by the module's names for them"},
    {nullptr, 0, 0, 0, nullptr},
};

PyTypeObject plan_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// `__call__` of the module classes that have plans: module(x) goes to the plan when torch's call of the module would
// only find the way to a forward that asks it (two Python frames and the checks in them: 4.7 -> 4.1 us per call),
// and is torch.nn.Module.__call__ otherwise.
struct ModuleCall {
  PyObject_HEAD
  vectorcallfunc call;
};

PyTypeObject module_call_type = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyTypeObject* g_module_class = nullptr;  // torch.nn.Module
PyObject *g_plan_key = nullptr, *g_call_key = nullptr;

PyObject* module_call(PyObject*, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  if (PyVectorcall_NARGS(nargsf) == 2 && !kwnames) {
    PyObject** dict = _PyObject_GetDictPtr(args[0]);
    PyObject* plan = dict && *dict ? PyDict_GetItemWithError(*dict, g_plan_key) : nullptr;
    if (plan && Py_TYPE(plan) == &plan_type) {
      Plan* p = reinterpret_cast<Plan*>(plan);
      Py_INCREF(plan);  // the module may drop it meanwhile
      PyObject* y = translated([&]() -> PyObject* {
        if (!p->guarded || !p->direct_type || !direct(p, args[0]) || stale(p, args[0]) || wrapped(p)) Py_RETURN_NONE;
        return issue_planned(p, args[1]);
      });
      Py_DECREF(plan);
      if (y != Py_None) return y;
      Py_DECREF(y);
    } else if (!plan && PyErr_Occurred()) {
      return nullptr;
    }
  }
  PyObject* call = g_module_class ? PyDict_GetItemWithError(g_module_class->tp_dict, g_call_key) : nullptr;
  if (!call) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "torch.nn.Module has no __call__");
    return nullptr;
  }
  return PyObject_Vectorcall(call, args, nargsf, kwnames);
}

PyObject* module_call_get(PyObject* self, PyObject* obj, PyObject*) {
  if (obj && obj != Py_None) return PyMethod_New(self, obj);
  Py_INCREF(self);
  return self;
}

// set_module_class(torch.nn.Module, call): `call` is what Python code sees as ModuleCall.__call__ -- compilers that trace
// Python source go through it -- while calls from the interpreter arrive in module_call.
PyObject* set_module_class(PyObject*, PyObject* args) {
  PyObject *type, *call;
  if (!PyArg_ParseTuple(args, "O!O", &PyType_Type, &type, &call) ||
      PyDict_SetItem(module_call_type.tp_dict, g_call_key, call) < 0)
    return nullptr;
  PyType_Modified(&module_call_type);
  Py_INCREF(type);
  Py_XDECREF(reinterpret_cast<PyObject*>(g_module_class));
  g_module_class = reinterpret_cast<PyTypeObject*>(type);
  Py_RETURN_NONE;
}

PyObject* set_workspaces(PyObject*, PyObject* args) {
  PyObject *dict, *drop;
  if (!PyArg_ParseTuple(args, "O!O", &PyDict_Type, &dict, &drop)) return nullptr;
  Py_INCREF(dict);
  Py_INCREF(drop);
  Py_XDECREF(g_workspaces);
  Py_XDECREF(g_drop_workspace);
  g_workspaces = dict;
  g_drop_workspace = drop;
  Py_RETURN_NONE;
}

// row_distance(x): elements between the rows of x that a plan would hand to a kernel, or None where it declines.
PyObject* row_distance(PyObject*, PyObject* xo) {
  if (!THPVariable_Check(xo) || THPVariable_Unpack(xo).dim() < 1) {
    PyErr_SetString(PyExc_TypeError, "row_distance() takes a tensor of one dimension or more");
    return nullptr;
  }
  return translated([&]() -> PyObject* {
    const at::Tensor& x = THPVariable_Unpack(xo);
    int64_t ldx = x.size(-1);
    if (!x.is_contiguous() && !rows_at_one_stride(x, &ldx)) Py_RETURN_NONE;
    return PyLong_FromLongLong(ldx);
  });
}

PyObject* tracked_tensor(PyObject*, PyObject* xo) {
  if (!THPVariable_Check(xo)) {
    PyErr_SetString(PyExc_TypeError, "tracked() takes a tensor");
    return nullptr;
  }
  return translated([&] { return PyBool_FromLong(tracked(THPVariable_Unpack(xo))); });
}

PyMethodDef module_methods[] = {
    {"tracked", tracked_tensor, METH_O, "tracked(x): whether torch follows what is done to x, so that no plan issues the call"},
    {"row_distance", row_distance, METH_O, "row_distance(x): elements between the rows a plan would read, or None"},
    {"set_module_class", set_module_class, METH_VARARGS, "set_module_class(torch.nn.Module, its call in Python)"},
    {"set_workspaces", set_workspaces, METH_VARARGS, "set_workspaces(dict, drop): the slice-list GEMV's scratch buffers"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "npamd_host", nullptr, -1, module_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_npamd_host(void) {
  plan_type.tp_name = "npamd_host.CallPlan";
  plan_type.tp_basicsize = sizeof(Plan);
  plan_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC | Py_TPFLAGS_HAVE_VECTORCALL;
  plan_type.tp_doc = "One lowered module's forward call, issued from native code.";
  plan_type.tp_new = plan_new;
  plan_type.tp_dealloc = plan_dealloc;
  plan_type.tp_traverse = plan_traverse;
  plan_type.tp_clear = plan_clear;
  plan_type.tp_call = PyVectorcall_Call;
  plan_type.tp_vectorcall_offset = offsetof(Plan, call);
  plan_type.tp_methods = plan_methods;
  plan_type.tp_members = plan_members;
  if (PyType_Ready(&plan_type) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  Py_INCREF(&plan_type);
  if (PyModule_AddObject(m, "CallPlan", reinterpret_cast<PyObject*>(&plan_type)) < 0) return nullptr;
  g_plan_key = PyUnicode_InternFromString("_plan");
  g_call_key = PyUnicode_InternFromString("__call__");
  module_call_type.tp_name = "npamd_host.ModuleCall";
  module_call_type.tp_basicsize = sizeof(ModuleCall);
  module_call_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL | Py_TPFLAGS_METHOD_DESCRIPTOR;
  module_call_type.tp_doc = "module(x), straight to the module's plan where nothing stands between";
  module_call_type.tp_call = PyVectorcall_Call;
  module_call_type.tp_vectorcall_offset = offsetof(ModuleCall, call);
  module_call_type.tp_descr_get = module_call_get;
  if (!g_plan_key || !g_call_key || PyType_Ready(&module_call_type) < 0) return nullptr;
  ModuleCall* call = PyObject_New(ModuleCall, &module_call_type);
  if (!call) return nullptr;
  call->call = module_call;
  if (PyModule_AddObject(m, "module_call", reinterpret_cast<PyObject*>(call)) < 0) return nullptr;
  return m;
}
