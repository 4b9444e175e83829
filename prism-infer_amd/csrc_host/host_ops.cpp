// Host side of the per-layer ops: argument checks and launches without
// Python in between.
//
// store_kvcache, paged_decode_attention and paged_prefill_attention run once
// per layer and step; checked in Python and bound through ctypes, a call costs
// the host more than the kernels of a small step take.  These functions do the
// same checks on the tensors themselves and call the C ABI (one layer's store
// and decode, B = 1, 1800 tokens: 41.8 us a step in Python, 16.1 here, where
// the GPU needs 14; a 3001-token store 13.0 and 4.9 us; a prefill reads its
// outcome from pinned memory instead of through a concatenation and a copy,
// 18 us less).  They only take calls that they can prove good: anything else
// (another device than the current one, a tensor subclass, no workspace yet, a
// contract violation, an error status) returns None, and the caller's Python
// path handles it, with its messages.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/Functions.h>
#include <ATen/core/Tensor.h>
#include <c10/hip/HIPException.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "prism_kv.h"

namespace {

constexpr int kMaxDevices = 64;
bool g_ready[kMaxDevices];  // the library's code objects are loaded (written and read under the GIL)

// A plain tensor with storage, or null.  Subclasses and wrappers (fake,
// functional, vmapped) go to the Python path.
const at::Tensor* tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.has_storage() && t.layout() == at::kStrided ? &t : nullptr;
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return PRISM_DTYPE_F32;
    case at::kBFloat16: return PRISM_DTYPE_BF16;
    case at::kHalf: return PRISM_DTYPE_F16;
    case at::kFloat8_e4m3fn: return PRISM_DTYPE_FP8_E4M3FN;
    default: return -1;
  }
}

// Every tensor on one device, which is ready and current.
template <typename... T>
bool on_current_device(int& device, const at::Tensor* first, const T*... rest) {
  if (!first->is_cuda()) return false;
  device = first->get_device();
  if (device < 0 || device >= kMaxDevices || !g_ready[device]) return false;
  return ((rest == nullptr || (rest->is_cuda() && rest->get_device() == device)) && ...) &&
         c10::hip::current_device() == device;
}

bool scale_pair(const at::Tensor& cache, const at::Tensor* ks, const at::Tensor* vs) {
  if (ks == nullptr) return true;
  const auto want = cache.sizes().slice(0, cache.dim() - 1);
  return cache.scalar_type() == at::kFloat8_e4m3fn && ks->sizes() == want && vs->sizes() == want &&
         ks->scalar_type() == at::kFloat && vs->scalar_type() == at::kFloat;
}

// An optional pair of arguments: both None, or both tensors.
bool optional_pair(PyObject* a, PyObject* b, const at::Tensor*& ta, const at::Tensor*& tb) {
  ta = tb = nullptr;
  if (a == Py_None && b == Py_None) return true;
  ta = tensor(a);
  tb = tensor(b);
  return ta != nullptr && tb != nullptr;
}

// The value at (device, stream) of a dict, borrowed, or null.
PyObject* by_stream(PyObject* dict, int device, void* stream) {
  PyObject* key = Py_BuildValue("(iK)", device, static_cast<unsigned long long>(reinterpret_cast<uintptr_t>(stream)));
  if (key == nullptr) return nullptr;
  PyObject* found = PyDict_CheckExact(dict) ? PyDict_GetItem(dict, key) : nullptr;
  Py_DECREF(key);
  return found;
}

bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }

// The kernels enqueued on this stream by the call; Python's device context is
// not needed since the tensors are on the current device.
void* current_stream(int device) { return c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device)).stream(); }

// The GIL is released over allocations and launches, which may wait (for memory,
// for room in a full queue): other Python threads run meanwhile, as they do
// under the ctypes calls.  The arguments stay alive, their caller holds them;
// what is found elsewhere (a stream's workspace) has to be held here.
class WithoutGil {
 public:
  WithoutGil() : state_(PyEval_SaveThread()) {}
  ~WithoutGil() { PyEval_RestoreThread(state_); }
  WithoutGil(const WithoutGil&) = delete;
  WithoutGil& operator=(const WithoutGil&) = delete;

 private:
  PyThreadState* state_;
};

// mark_ready(device): prism_preload has run there.
PyObject* mark_ready(PyObject*, PyObject* arg) {
  const long device = PyLong_AsLong(arg);
  if (device == -1 && PyErr_Occurred()) return nullptr;
  if (device >= 0 && device < kMaxDevices) g_ready[device] = true;
  Py_RETURN_NONE;
}

// store(key, value, k_cache, v_cache, slot_mapping, k_scale, v_scale) -> True or None
PyObject* store(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) Py_RETURN_NONE;
  const at::Tensor *key = tensor(args[0]), *value = tensor(args[1]), *kc = tensor(args[2]), *vc = tensor(args[3]),
                   *slots = tensor(args[4]), *ks, *vs;
  if (!key || !value || !kc || !vc || !slots || !optional_pair(args[5], args[6], ks, vs)) Py_RETURN_NONE;
  int device;
  if (!on_current_device(device, key, value, kc, vc, slots, ks, vs)) Py_RETURN_NONE;
  if (key->dim() != 3 || key->sizes() != value->sizes() || (kc->dim() != 3 && kc->dim() != 4) ||
      kc->sizes() != vc->sizes() || kc->scalar_type() != vc->scalar_type())
    Py_RETURN_NONE;
  const int64_t tokens = key->size(0), heads = key->size(1), dim = key->size(2);
  if (tokens <= 0 || heads <= 0 || dim <= 0 || heads > INT32_MAX || dim > INT32_MAX || kc->size(-2) != heads ||
      kc->size(-1) != dim || slots->dim() != 1 || slots->numel() != tokens || slots->scalar_type() != at::kInt ||
      !slots->is_contiguous() || !scale_pair(*kc, ks, vs))
    Py_RETURN_NONE;
  const int in = dtype_code(key->scalar_type()), out = dtype_code(kc->scalar_type());
  if (in < 0 || in == PRISM_DTYPE_FP8_E4M3FN || value->scalar_type() != key->scalar_type() || out < 0 ||
      key->stride(2) != 1 || value->stride(2) != 1 || key->stride(1) != dim || value->stride(1) != dim ||
      !kc->is_contiguous() || !vc->is_contiguous() || (ks && (!ks->is_contiguous() || !vs->is_contiguous())))
    Py_RETURN_NONE;
  const int64_t kst[3] = {key->stride(0), key->stride(1), key->stride(2)};
  const int64_t vst[3] = {value->stride(0), value->stride(1), value->stride(2)};
  int rc;
  {
    WithoutGil released;
    rc = prism_kv_store(key->data_ptr(), value->data_ptr(), in, kst, vst, kc->data_ptr(), vc->data_ptr(), out,
                        ks ? static_cast<float*>(ks->data_ptr()) : nullptr,
                        vs ? static_cast<float*>(vs->data_ptr()) : nullptr,
                        static_cast<const int32_t*>(slots->data_ptr()), tokens, static_cast<int>(heads),
                        static_cast<int>(dim), kc->numel() / (heads * dim), current_stream(device));
  }
  if (rc != PRISM_OK) Py_RETURN_NONE;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

struct Strides {
  int64_t v[4];
  explicit Strides(const at::Tensor* t) : v{0, 0, 0, 0} {
    if (t != nullptr)
      for (int64_t i = 0; i < t->dim() && i < 4; ++i) v[i] = t->stride(i);
  }
};

// A paged decode's arguments, checked: decode's of eleven (from args[0]).
struct DecodeCall {
  const at::Tensor *q, *kc, *vc, *bt, *ctx, *max_ctx, *ks, *vs;
  double scale;
  int device, qd, cd;
  int64_t batch, heads, dim, blocks, page, kv_heads, width;
  void* stream;
  int64_t need;       // workspace bytes
  at::Tensor ws_own;  // the workspace: the stream's, held over the launch (another thread may put a larger one in
                      // its place), or a captured call's from the graph's pool
  void* ws;
};

bool check_decode(PyObject* const* args, DecodeCall& d) {
  d.q = tensor(args[0]), d.kc = tensor(args[1]), d.vc = tensor(args[2]), d.bt = tensor(args[3]);
  d.ctx = tensor(args[4]), d.max_ctx = tensor(args[8]);
  if (!d.q || !d.kc || !d.vc || !d.bt || !d.ctx || !d.max_ctx || !optional_pair(args[6], args[7], d.ks, d.vs)) return false;
  if (!PyFloat_CheckExact(args[5]) || !PyLong_CheckExact(args[9])) return false;
  d.scale = PyFloat_AS_DOUBLE(args[5]);
  int overflow = 0;
  const long block_n = PyLong_AsLongAndOverflow(args[9], &overflow);
  if (overflow || block_n <= 0 || (block_n & (block_n - 1))) return false;
  const at::Tensor &q = *d.q, &kc = *d.kc;
  if (!on_current_device(d.device, d.q, d.kc, d.vc, d.bt, d.ctx, d.max_ctx, d.ks, d.vs)) return false;
  if (q.dim() != 3 || kc.dim() != 4 || kc.sizes() != d.vc->sizes() || kc.scalar_type() != d.vc->scalar_type() ||
      d.bt->dim() != 2 || d.ctx->dim() != 1 || d.bt->scalar_type() != at::kInt || d.ctx->scalar_type() != at::kInt ||
      !d.ctx->is_contiguous() || d.max_ctx->numel() != 1 || d.max_ctx->scalar_type() != at::kInt ||
      !scale_pair(kc, d.ks, d.vs))
    return false;
  d.batch = q.size(0), d.heads = q.size(1), d.dim = q.size(2);
  d.blocks = kc.size(0), d.page = kc.size(1), d.kv_heads = kc.size(2), d.width = d.bt->size(1);
  d.qd = dtype_code(q.scalar_type()), d.cd = dtype_code(kc.scalar_type());
  if (d.qd < 0 || d.qd == PRISM_DTYPE_FP8_E4M3FN || d.cd < 0 || d.batch <= 0 || d.heads <= 0 || d.dim <= 0 ||
      d.dim > 256 || kc.size(3) != d.dim || d.page <= 0 || d.kv_heads <= 0 || d.heads % d.kv_heads != 0 ||
      d.bt->size(0) < d.batch || d.ctx->size(0) < d.batch || kc.stride(3) != 1 || d.batch > INT32_MAX ||
      d.heads > INT32_MAX || d.page > INT32_MAX || d.width > INT32_MAX)
    return false;
  d.stream = current_stream(d.device);
  d.need = prism_paged_decode_workspace_bytes(static_cast<int>(d.batch), static_cast<int>(d.heads),
                                              static_cast<int>(d.kv_heads), static_cast<int>(d.dim),
                                              static_cast<int>(d.page), static_cast<int>(d.width), d.cd);
  d.ws = nullptr;
  if (d.need > 0) {
    if (capturing()) {
      WithoutGil released;
      d.ws_own = at::empty({d.need}, q.options().dtype(at::kByte));
    } else {
      PyObject* found = by_stream(args[10], d.device, d.stream);
      const at::Tensor* ws = found ? tensor(found) : nullptr;
      if (ws == nullptr || ws->numel() < d.need) return false;
      d.ws_own = *ws;
    }
    d.ws = d.ws_own.data_ptr();
  }
  return true;
}

const float* scales(const at::Tensor* t) { return t ? static_cast<const float*>(t->data_ptr()) : nullptr; }

// decode(q, k_cache, v_cache, block_tables, context_lens, scale, k_scale, v_scale, max_context_len, block_n,
//        workspaces) -> output or None
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  DecodeCall d;
  if (n != 11 || !check_decode(args, d)) Py_RETURN_NONE;
  at::Tensor out;
  int rc;
  {
    WithoutGil released;
    out = at::empty_like(*d.q);
    const Strides sq(d.q), sk(d.kc), sv(d.vc), sks(d.ks), svs(d.vs), sbt(d.bt), so(&out);
    rc = prism_paged_decode(
        d.q->data_ptr(), d.qd, sq.v, d.kc->data_ptr(), d.vc->data_ptr(), d.cd, sk.v, sv.v, scales(d.ks), scales(d.vs),
        sks.v, svs.v, static_cast<const int32_t*>(d.bt->data_ptr()), sbt.v, static_cast<const int32_t*>(d.ctx->data_ptr()),
        static_cast<const int32_t*>(d.max_ctx->data_ptr()), out.data_ptr(), so.v, static_cast<int>(d.batch),
        static_cast<int>(d.heads), static_cast<int>(d.kv_heads), static_cast<int>(d.dim), static_cast<int>(d.page),
        d.blocks, static_cast<int>(d.width), static_cast<float>(d.scale), d.ws, d.need, d.stream);
  }
  if (rc != PRISM_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// step(decode's eleven, key, value, slot_mapping) -> output or None: the store
// of the step's rows, then the decode
PyObject* step(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  DecodeCall d;
  if (n != 14 || !check_decode(args, d)) Py_RETURN_NONE;
  const at::Tensor *key = tensor(args[11]), *value = tensor(args[12]), *slots = tensor(args[13]);
  int device;
  if (!key || !value || !slots || !on_current_device(device, key, value, slots) || device != d.device) Py_RETURN_NONE;
  if (key->dim() != 3 || key->sizes() != value->sizes() || key->size(0) != d.batch || key->size(1) != d.kv_heads ||
      key->size(2) != d.dim || slots->dim() != 1 || slots->numel() != d.batch || slots->scalar_type() != at::kInt ||
      !slots->is_contiguous() || key->scalar_type() != d.q->scalar_type() ||
      value->scalar_type() != d.q->scalar_type() || key->stride(2) != 1 || value->stride(2) != 1 ||
      key->stride(1) != d.dim || value->stride(1) != d.dim || !d.kc->is_contiguous() || !d.vc->is_contiguous() ||
      (d.ks && (!d.ks->is_contiguous() || !d.vs->is_contiguous())))
    Py_RETURN_NONE;
  at::Tensor out;
  int rc;
  {
    WithoutGil released;
    out = at::empty_like(*d.q);
    const Strides skey(key), sval(value), sq(d.q), sk(d.kc), sv(d.vc), sks(d.ks), svs(d.vs), sbt(d.bt), so(&out);
    rc = prism_paged_decode_step(
        key->data_ptr(), value->data_ptr(), skey.v, sval.v, static_cast<const int32_t*>(slots->data_ptr()),
        d.q->data_ptr(), d.qd, sq.v, d.kc->data_ptr(), d.vc->data_ptr(), d.cd, sk.v, sv.v,
        const_cast<float*>(scales(d.ks)), const_cast<float*>(scales(d.vs)), sks.v, svs.v,
        static_cast<const int32_t*>(d.bt->data_ptr()), sbt.v, static_cast<const int32_t*>(d.ctx->data_ptr()),
        static_cast<const int32_t*>(d.max_ctx->data_ptr()), out.data_ptr(), so.v, static_cast<int>(d.batch),
        static_cast<int>(d.heads), static_cast<int>(d.kv_heads), static_cast<int>(d.dim), static_cast<int>(d.page),
        d.blocks, static_cast<int>(d.width), static_cast<float>(d.scale), d.ws, d.need, d.stream);
  }
  if (rc != PRISM_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// prefill(q, k_cache, v_cache, block_tables, context_lens, cu_seqlens_q, num_heads, num_kv_heads, scale, k_scale,
//         v_scale, buffers) -> (out, first bad sequence, first row, end row) or None
//
// buffers: this thread's {(device, stream): (status int32[1] on the device,
// pinned int32[3])}; status holds INT32_MAX between calls.  Waits for the
// stream, as the caller's check of the status does.
PyObject* prefill(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12) Py_RETURN_NONE;
  const at::Tensor *q = tensor(args[0]), *kc = tensor(args[1]), *vc = tensor(args[2]), *bt = tensor(args[3]),
                   *ctx = tensor(args[4]), *cu = tensor(args[5]), *ks, *vs;
  if (!q || !kc || !vc || !bt || !ctx || !cu || !optional_pair(args[9], args[10], ks, vs)) Py_RETURN_NONE;
  if (!PyLong_CheckExact(args[6]) || !PyLong_CheckExact(args[7]) || !PyFloat_CheckExact(args[8])) Py_RETURN_NONE;
  int over1 = 0, over2 = 0;
  const long heads = PyLong_AsLongAndOverflow(args[6], &over1), kv_heads = PyLong_AsLongAndOverflow(args[7], &over2);
  const double scale = PyFloat_AS_DOUBLE(args[8]);
  int device;
  if (over1 || over2 || !on_current_device(device, q, kc, vc, bt, ctx, cu, ks, vs) || capturing()) Py_RETURN_NONE;
  if (q->dim() != 3 || kc->dim() != 4 || kc->sizes() != vc->sizes() || bt->dim() != 2 ||
      kc->scalar_type() != at::kFloat8_e4m3fn || vc->scalar_type() != at::kFloat8_e4m3fn || !scale_pair(*kc, ks, vs) ||
      bt->scalar_type() != at::kInt || ctx->scalar_type() != at::kInt || cu->scalar_type() != at::kInt ||
      ctx->dim() != 1 || cu->dim() != 1 || !ctx->is_contiguous() || !cu->is_contiguous())
    Py_RETURN_NONE;
  const int64_t total = q->size(0), dim = q->size(2), batch = ctx->numel();
  const int qd = dtype_code(q->scalar_type());
  if ((qd != PRISM_DTYPE_BF16 && qd != PRISM_DTYPE_F16) || total <= 0 || total > INT32_MAX || batch <= 0 ||
      batch > INT32_MAX || heads <= 0 || kv_heads <= 0 || heads > INT32_MAX || heads % kv_heads != 0 ||
      q->size(1) != heads || dim != 128 || q->stride(2) != 1 || kc->size(2) != kv_heads || kc->size(3) != dim ||
      kc->size(0) > INT32_MAX || kc->size(1) > INT32_MAX || bt->size(1) > INT32_MAX || cu->numel() < batch + 1 ||
      bt->size(0) < batch)
    Py_RETURN_NONE;
  void* stream = current_stream(device);
  PyObject* found = by_stream(args[11], device, stream);
  if (found == nullptr || !PyTuple_CheckExact(found) || PyTuple_GET_SIZE(found) != 2) Py_RETURN_NONE;
  const at::Tensor *status = tensor(PyTuple_GET_ITEM(found, 0)), *report = tensor(PyTuple_GET_ITEM(found, 1));
  if (!status || !report) Py_RETURN_NONE;
  const int page = static_cast<int>(kc->size(1)), width = static_cast<int>(bt->size(1));
  const int64_t need = prism_paged_prefill_workspace_bytes(static_cast<int>(batch), static_cast<int>(total),
                                                           static_cast<int>(heads), static_cast<int>(kv_heads), page, width);
  at::Tensor out, ws;
  int32_t* words = static_cast<int32_t*>(report->data_ptr());
  words[0] = 0;  // (the thread's previous call on this stream has been waited for)
  int rc;
  {
    WithoutGil released;
    out = at::empty(q->sizes(), q->options());
    if (need > 0) ws = at::empty({need}, q->options().dtype(at::kByte));
    const Strides sq(q), sk(kc), sv(vc), sks(ks), svs(vs), sbt(bt), so(&out);
    rc = prism_paged_prefill_ws(
        q->data_ptr(), qd, sq.v, kc->data_ptr(), vc->data_ptr(), PRISM_DTYPE_FP8_E4M3FN, sk.v, sv.v, scales(ks),
        scales(vs), sks.v, svs.v, static_cast<const int32_t*>(bt->data_ptr()), sbt.v,
        static_cast<const int32_t*>(ctx->data_ptr()), static_cast<const int32_t*>(cu->data_ptr()), out.data_ptr(), so.v,
        static_cast<int>(batch), static_cast<int>(total), static_cast<int>(heads), static_cast<int>(kv_heads),
        static_cast<int>(dim), page, static_cast<int>(kc->size(0)), width, static_cast<float>(scale),
        static_cast<int32_t*>(status->data_ptr()), need > 0 ? ws.data_ptr() : nullptr, need, words, stream);
    if (rc == PRISM_OK) C10_HIP_CHECK(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
  }
  if (rc != PRISM_OK) Py_RETURN_NONE;
  const volatile int32_t* r = words;
  const int row0 = r[1], row1 = r[2];
  const int bad = r[0] == 0 ? INT32_MAX : status->item<int32_t>();
  PyObject* wrapped = THPVariable_Wrap(std::move(out));
  if (wrapped == nullptr) return nullptr;
  return Py_BuildValue("(Niii)", wrapped, bad, row0, row1);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"mark_ready", mark_ready, METH_O, nullptr},
    {"store", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(store)), METH_FASTCALL, nullptr},
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(decode)), METH_FASTCALL, nullptr},
    {"step", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(step)), METH_FASTCALL, nullptr},
    {"prefill", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(prefill)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_ops() { return PyModule_Create(&module); }
