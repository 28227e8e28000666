// The host side of a layer step, a decode step, the single operations and a batch's bookkeeping as one native call each: argument
// checks, output allocation (torch's caching allocator), stream lookup and the C ABI call.  The same work in Python and ctypes costs 16 us
// per layer step and 23 us per decode step against 6 us of kernel launches, which is more than the GPU needs for a short
// prompt (9 us) or a decode step of one sequence.  Nothing is computed here; every launch is an entry point of
// libenergon_hip.so.
//
// A plain CPython module (METH_FASTCALL, no pybind11): a call has up to twenty arguments, and converting them costs more
// than what the call does if each goes through a type caster.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <cmath>
#include <map>
#include <stdexcept>
#include <string>
#include <utility>

#include "energon_hip.h"

#ifndef EN_SOURCE_HASH
#define EN_SOURCE_HASH "unknown"
#endif

namespace {

using at::Tensor;

[[noreturn]] void fail(const std::string &msg) { throw std::runtime_error(msg); }

void check(int status, const char *op) {
  if (status == EN_OK) return;
  std::string msg = std::string(op) + ": " + en_status_string(status);
  if (status == EN_ERR_HIP)
    msg += std::string(": ") + en_last_hip_error_string() + " (hipError " + std::to_string(en_last_hip_error()) + ")";
  fail(msg);
}

// ---- arguments -----------------------------------------------------------------------------------------------------

const Tensor &tensor(PyObject *o, const char *name) {
  if (!THPVariable_Check(o)) fail(std::string(name) + " must be a CUDA tensor");
  return THPVariable_Unpack(o);
}

const Tensor &gpu(PyObject *o, const char *name, bool contiguous = true) {
  const Tensor &t = tensor(o, name);
  if (!t.is_cuda()) fail(std::string(name) + " must be a CUDA tensor");
  if (contiguous && !t.is_contiguous()) fail(std::string(name) + " must be contiguous");
  return t;
}

int64_t integer(PyObject *o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) fail("an integer is required");
  return v;
}

float real(PyObject *o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) fail("a number is required");
  return (float)v;
}

int dtype_tag(const Tensor &t, const char *op) {
  switch (t.scalar_type()) {
    case at::kFloat: return EN_F32;
    case at::kHalf: return EN_F16;
    case at::kBFloat16: return EN_BF16;
    default:
      fail(std::string(op) + ": Datatype not implemented (" + c10::toString(t.scalar_type()) +
           "); expected float32, float16 or bfloat16");
  }
}

hipStream_t stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

const int32_t *i32(const Tensor &t) { return t.data_ptr<int32_t>(); }

// Launches run without the interpreter lock: a launch may wait for room in the stream's queue.  `f` touches no Python object, and what
// it throws is a C++ exception, which leaves with the lock held again.  Most are the C ABI call alone, on pointers and a stream taken
// before.  One that calls ATen as well (block_prefill) may because nothing in it comes back to Python: its tensors are exact ones and
// its caller has seen that gradients and autocast are off and no dispatch or function mode is on; ATen takes the lock by itself where
// it needs it.
template <typename F> int without_gil(F &&f) {
  struct Released {
    PyThreadState *saved = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(saved); }
  } released;
  return f();
}

// ---- events (SeqInfo orders other streams behind the kernels that produced its arrays) -------------------------------

void destroy_event(PyObject *capsule) {
  void *p = PyCapsule_GetPointer(capsule, "energonai_amd.event");
  if (p) (void)hipEventDestroy(static_cast<hipEvent_t>(p));
}

PyObject *record_event(PyObject *const *a) {
  const Tensor &t = gpu(a[0], "lens");
  const c10::DeviceGuard guard(t.device());
  hipEvent_t e;
  if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) fail("record_event: hipEventCreate failed");
  PyObject *capsule = PyCapsule_New(e, "energonai_amd.event", destroy_event);
  if (!capsule) {
    (void)hipEventDestroy(e);
    return nullptr;
  }
  if (hipEventRecord(e, stream_of(t)) != hipSuccess) {
    Py_DECREF(capsule);
    fail("record_event: hipEventRecord failed");
  }
  return capsule;
}

PyObject *wait_event(PyObject *const *a) {
  void *p = PyCapsule_GetPointer(a[0], "energonai_amd.event");
  if (!p) return nullptr;
  const Tensor &t = gpu(a[1], "lens");
  const c10::DeviceGuard guard(t.device());
  if (hipStreamWaitEvent(stream_of(t), static_cast<hipEvent_t>(p), 0) != hipSuccess) fail("wait_event: hipStreamWaitEvent failed");
  Py_RETURN_NONE;
}

PyObject *tuple(std::initializer_list<Tensor> ts) {
  PyObject *r = PyTuple_New((Py_ssize_t)ts.size());
  Py_ssize_t i = 0;
  for (const Tensor &t : ts) {
    PyObject *p = r ? THPVariable_Wrap(t) : nullptr;
    if (!p) {
      Py_XDECREF(r);
      return nullptr;
    }
    PyTuple_SET_ITEM(r, i++, p);
  }
  return r;
}

// prefix_sum(lens, batch) -> (cu_seqlens [batch + 1], lens [batch]), both int32
PyObject *prefix_sum(PyObject *const *a) {
  const Tensor &lens = gpu(a[0], "seq_lens");
  const int64_t batch = integer(a[1]);
  const bool i64 = lens.scalar_type() == at::kLong;
  if ((!i64 && lens.scalar_type() != at::kInt) || lens.numel() < batch) fail("prefix_sum: lens must hold batch int32 or int64 values");
  const c10::DeviceGuard guard(lens.device());
  const auto opt = lens.options().dtype(at::kInt);
  const Tensor cu = at::empty({batch + 1}, opt), lens32 = at::empty({batch}, opt);
  const void *src = lens.data_ptr();
  int32_t *cu_out = cu.data_ptr<int32_t>(), *lens_out = lens32.data_ptr<int32_t>();
  const hipStream_t stream = stream_of(lens);
  check(without_gil([&] { return en_prefix_sum(src, i64, (int)batch, cu_out, lens_out, stream); }), "prefix_sum");
  return tuple({cu, lens32});
}

// layer_tables(lens, cu_seqlens, batch, max_seq_len, left_padded, total, heads, tiles_first)
// -> (row offsets, tile table, meeting words of en_attn_fused_norm)
PyObject *layer_tables(PyObject *const *a) {
  const Tensor &lens = gpu(a[0], "lens"), &cu = gpu(a[1], "cu_seqlens");
  const int64_t batch = integer(a[2]), S = integer(a[3]), left = integer(a[4]), total = integer(a[5]), heads = integer(a[6]),
                tiles_first = integer(a[7]);
  const c10::DeviceGuard guard(lens.device());
  const int64_t n = en_attn_tile_table_elems((int)batch, (int)heads, (int)S, 0);
  const Tensor offs = at::empty({total > 0 ? total : 1}, lens.options()), table = at::empty({n > 0 ? n : 1}, lens.options()),
               arrivals = at::empty({en_attn_fused_norm_arrivals((int)batch, (int)S)}, lens.options().dtype(at::kLong));
  const int32_t *lens_in = i32(lens), *cu_in = i32(cu);
  int32_t *table_out = table.data_ptr<int32_t>(), *offs_out = offs.data_ptr<int32_t>();
  uint64_t *words = reinterpret_cast<uint64_t *>(arrivals.data_ptr<int64_t>());
  const hipStream_t stream = stream_of(lens);
  check(without_gil([&] {
          return en_layer_tables(lens_in, cu_in, (int)batch, (int)S, (int)left, (int)heads, (int)tiles_first, table_out, offs_out,
                                 words, stream);
        }), "layer_tables");
  return tuple({offs, table, arrivals});
}

// The meeting words of en_attn_fused_norm for launches of this bucket on this stream, or an undefined tensor (SeqInfo.arrivals).
Tensor meeting_words(PyObject *arrivals, int64_t max_seq_len, hipStream_t stream) {
  if (!PyDict_Check(arrivals)) fail("arrivals must be a dict");
  PyObject *key = Py_BuildValue("(LK)", (long long)max_seq_len, (unsigned long long)reinterpret_cast<uintptr_t>(stream));
  if (!key) fail("arrivals: no key");
  PyObject *words = PyDict_GetItemWithError(arrivals, key);
  Py_DECREF(key);
  if (!words) {
    if (PyErr_Occurred()) fail("arrivals: no lookup");
    return Tensor();
  }
  return tensor(words, "arrivals");
}

// layer(hidden_padded, qkv_packed, dense_out, gamma, beta, ctx_out, cu_seqlens, lens, row offsets or None, tile table or None,
//       heads, size_per_head, total, scale, eps, causal, left_padded, form, {(bucket, stream): meeting words} or None) -> y
PyObject *layer(PyObject *const *a) {
  static const std::string who = "padding_removal_layer: ";
  const Tensor &hidden = gpu(a[0], "hidden_padded"), &qkv = gpu(a[1], "qkv_packed");
  const bool has_dense = a[2] != Py_None, has_ctx = a[5] != Py_None;
  const Tensor &gamma = tensor(a[3], "gamma"), &beta = tensor(a[4], "beta");
  const Tensor &cu = tensor(a[6], "cu_seqlens"), &lens = tensor(a[7], "lens");
  const int32_t *offs = a[8] == Py_None ? nullptr : i32(tensor(a[8], "offsets"));
  const int32_t *table = a[9] == Py_None ? nullptr : i32(tensor(a[9], "tile_table"));
  const int64_t H = integer(a[10]), D = integer(a[11]), T = integer(a[12]);
  const float scale = real(a[13]), eps = real(a[14]);
  const int causal = (int)integer(a[15]), left = (int)integer(a[16]), form = (int)integer(a[17]);
  const int64_t B = hidden.size(0), S = hidden.size(1), hid = hidden.size(2);
  const auto dt = hidden.scalar_type();
  if (qkv.numel() != T * H * 3 * D || qkv.scalar_type() != dt) fail(who + "qkv_packed must be [1,T,H,3D] of the activation dtype");
  if (gamma.scalar_type() != dt || beta.scalar_type() != dt || gamma.numel() != hid || beta.numel() != hid)
    fail(who + "gamma and beta must be [hidden] of the activation dtype");
  const void *dense = nullptr;
  if (has_dense) {
    const Tensor &d = gpu(a[2], "dense_out");
    if (d.numel() != T * hid || d.scalar_type() != dt) fail(who + "dense_out must be [1,T,hidden] of the activation dtype");
    dense = d.data_ptr();
  } else if (hid != H * D) {
    fail(who + "without dense_out the LayerNorm width must equal heads * size_per_head");
  }
  const int tag = dtype_tag(hidden, "padding_removal_layer");
  if (form == 4 && dt == at::kFloat) fail(who + "the packed scores are for float16 and bfloat16");
  if ((form == 1 || form == 2) && dt == at::kFloat && D > 64) fail(who + "the fused kernel takes float32 heads of up to 64 channels");
  if (form == 5 && (dt != at::kFloat || D <= 64 || D > 128)) fail(who + "packed_f32_wide is for float32 heads of 65..128 channels");
  if (form == 4 && !causal) fail(who + "the packed score layout is that of a causal mask");
  const c10::DeviceGuard guard(hidden.device());
  const auto opt = hidden.options();
  const Tensor y = at::empty({1, T, hid}, opt);
  Tensor x, padded, ctx, scores, ctx_packed;
  if (!offs) x = at::empty({1, T, hid}, opt);
  if (has_ctx) {
    const Tensor &c = gpu(a[5], "ctx_out", false);
    if (c.numel() != T * H * D || c.scalar_type() != dt || !c.is_contiguous())
      fail(who + "ctx_out must be a contiguous [1,T,H,D] tensor of the activation dtype");
    ctx_packed = c;
  } else {
    ctx_packed = at::empty({1, T, H, D}, opt);
  }
  if (form < 2) {
    padded = at::empty({B, H, S, 3 * D}, opt);
    ctx = at::empty({B, H, S, D}, opt);
  }
  if (form == 0 || form == 3) scores = at::empty({B, H, S, S}, opt);
  if (form == 4) {
    const int64_t n = en_packed_scores_elems((int)B, (int)H, (int)S, tag);
    if (n <= 0) fail("packed_scores_elems: bad arguments");
    scores = at::empty({n}, opt);
  }
  auto ptr = [](const Tensor &t) -> void * { return t.defined() ? t.data_ptr() : nullptr; };
  const void *hidden_p = hidden.data_ptr(), *qkv_p = qkv.data_ptr(), *gamma_p = gamma.data_ptr(), *beta_p = beta.data_ptr();
  void *x_p = ptr(x), *padded_p = ptr(padded), *scores_p = ptr(scores), *ctx_p = ptr(ctx), *packed_p = ctx_packed.data_ptr(), *y_p = y.data_ptr();
  const int32_t *lens_p = i32(lens), *cu_p = i32(cu);
  const hipStream_t stream = stream_of(hidden);
  Tensor arrivals;      // small enough: one launch
  if (form == 2 && !has_dense && offs && a[18] != Py_None && en_attn_fused_norm_pays((int)B, (int)H, (int)S, (int)D, T, tag))
    arrivals = meeting_words(a[18], S, stream);
  if (arrivals.defined()) {
    uint64_t *words = reinterpret_cast<uint64_t *>(arrivals.data_ptr<int64_t>());
    const int rc = without_gil([&] {
      return en_attn_fused_norm(qkv_p, packed_p, lens_p, cu_p, (int)B, (int)H, (int)S, (int)D, T, scale, causal, tag, table, hidden_p, offs,
                                gamma_p, beta_p, y_p, eps, words, -1, stream);
    });
    if (rc != EN_ERR_UNSUPPORTED) {
      check(rc, "padding_removal_layer");
      return THPVariable_Wrap(y);
    }
  }
  check(without_gil([&] {
          return en_padding_removal_layer(hidden_p, qkv_p, dense, gamma_p, beta_p, x_p, padded_p, scores_p, ctx_p, packed_p, y_p, cu_p, lens_p,
                                          (int)B, (int)S, (int)H, (int)D, hid, T, scale, eps, causal, left, form, offs, tag, table, stream);
        }), "padding_removal_layer");
  return THPVariable_Wrap(y);
}

// The words of en_decode_layer_norm for a launch on torch's current stream of a device, or null.  They belong to the stream: its
// order keeps launches apart that share them, and torch's own streams (a fixed pool a device, which bounds this) live as long as the
// process.  An external stream's handle may come back as another stream's while the first one's work still runs, so it gets none;
// nor does a capture, whose launches may run again beside others.  A launch whose lengths are changed under it may leave its words
// off zero, and they are to spoil no later step: launches take turns on 64 sets, 1 MB a stream, all cleared before the first is taken
// again (2 us every 64 launches).  Counting every workgroup, so that lengths do not matter, costs 10 ns for each share without keys: 1
// sequence x 16 heads x 64, up to 100 keys in caches of 16000, 5.6 -> 10.7 us a layer.
constexpr int kWordSets = 64;
struct WordSets {
  Tensor sets;
  int next = kWordSets;
};
uint32_t *next_decode_words(const Tensor &t) {
  typedef std::map<std::pair<int, hipStream_t>, WordSets> Pool;
  static Pool &pool = *new Pool;     // under the interpreter lock
  const auto stream = c10::hip::getCurrentHIPStream(t.device().index());
  if (stream.id() != 0 && stream.id() == (c10::StreamId) reinterpret_cast<intptr_t>(stream.stream())) return nullptr;   // external
  WordSets &w = pool[std::make_pair((int)t.device().index(), stream.stream())];
  const int64_t words = en_decode_layer_norm_words();
  if (w.next == kWordSets) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream.stream(), &capture) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    if (capture != hipStreamCaptureStatusNone) return nullptr;
    if (!w.sets.defined()) w.sets = at::empty({kWordSets, words}, t.options().dtype(at::kInt));
    if (hipMemsetAsync(w.sets.data_ptr(), 0, (size_t)w.sets.nbytes(), stream.stream()) != hipSuccess) fail("decode_layer: hipMemsetAsync failed");
    w.next = 0;
  }
  return reinterpret_cast<uint32_t *>(w.sets.data_ptr<int32_t>()) + words * w.next++;
}

// decode_words(tensor) -> address of the words that the next decode layer on the tensor's device and current stream would take, a
// turn of theirs, or None
PyObject *decode_words(PyObject *const *a) {
  const Tensor &t = gpu(a[0], "tensor", false);
  const c10::DeviceGuard guard(t.device());
  uint32_t *words = next_decode_words(t);
  if (!words) Py_RETURN_NONE;
  return PyLong_FromVoidPtr(words);
}

// decode_layer(q, k_cache, v_cache, lens, residual, gamma, beta, dense_out, eps, scale) -> y
PyObject *decode_layer(PyObject *const *a) {
  const Tensor &q_in = gpu(a[0], "q", false), &k = gpu(a[1], "k_cache", false), &v = gpu(a[2], "v_cache", false);
  const Tensor &lens = tensor(a[3], "lens"), &residual = gpu(a[4], "residual", false), &gamma_in = gpu(a[5], "gamma", false),
               &beta_in = gpu(a[6], "beta", false);
  const float eps = real(a[8]), scale = real(a[9]);
  for (const Tensor *c : {&k, &v}) {
    const char *name = c == &k ? "k_cache" : "v_cache";
    if (c->dim() != 4) fail(std::string(name) + " must be [batch, head, seq, size_per_head]");
    if (c->stride(3) != 1) fail(std::string(name) + ": the last dimension must be contiguous");
  }
  const int64_t B = k.size(0), H = k.size(1), S = k.size(2), D = k.size(3), hid = gamma_in.numel();
  const auto dt = q_in.scalar_type();
  if (v.sizes() != k.sizes() || v.scalar_type() != k.scalar_type()) fail("decode_attn: k_cache and v_cache must share shape and dtype");
  if (q_in.numel() != B * H * D || dt != k.scalar_type()) fail("decode_attn: q must be [B,H,1,D] of the caches' dtype");
  // the kernels read one length per sequence of the caches
  if (q_in.dim() < 1 || q_in.size(0) != B || !lens.is_cuda() || lens.scalar_type() != at::kInt || lens.numel() < B || !lens.is_contiguous() ||
      lens.device() != k.device())
    fail("decode_attn: kv_lens must hold one int32 length for each of the caches' " + std::to_string(B) + " sequences");
  const int tag = dtype_tag(q_in, "decode_attn"), out_tag = dtype_tag(gamma_in, "layer_norm");
  if (gamma_in.scalar_type() != beta_in.scalar_type()) fail("gamma and beta must share one dtype");
  if (gamma_in.dim() != 1 || beta_in.sizes() != gamma_in.sizes()) fail("gamma and beta must have normalized_shape");
  Tensor dense;
  if (a[7] != Py_None) dense = gpu(a[7], "dense_out", false).contiguous();
  const auto in_dt = dense.defined() ? dense.scalar_type() : dt;
  if (in_dt != dt || (tag != out_tag && tag != EN_F32))
    fail("layer_norm: unsupported (input, output) dtypes (" + std::string(c10::toString(in_dt)) + ", " + c10::toString(gamma_in.scalar_type()) + ")");
  if (dense.defined() ? (dense.dim() < 1 || dense.size(-1) != hid || dense.numel() != B * hid) : H * D != hid)
    fail("Given normalized_shape=[" + std::to_string(hid) + "], the LayerNorm input must have that last dimension and batch rows");
  const int64_t rows[3] = {1, B, hid};
  if (residual.scalar_type() != dt || residual.sizes() != (dense.defined() ? dense.sizes() : c10::IntArrayRef(rows)))
    fail("residual must match input in shape and dtype");
  const c10::DeviceGuard guard(k.device());
  const Tensor q = q_in.contiguous(), res = residual.contiguous(), gamma = gamma_in.contiguous(), beta = beta_in.contiguous();
  const Tensor ctx = at::empty({B, H, 1, D}, q.options());
  const Tensor y = at::empty(dense.defined() ? dense.sizes() : c10::IntArrayRef(rows), gamma.options());
  const int64_t need = en_decode_attn_workspace_bytes((int)B, (int)H, (int)S, (int)D);
  Tensor ws;
  if (need > 0) ws = at::empty({need}, q.options().dtype(at::kByte));
  const int64_t ks[3] = {k.stride(0), k.stride(1), k.stride(2)}, vs[3] = {v.stride(0), v.stride(1), v.stride(2)};
  const void *q_p = q.data_ptr(), *k_p = k.data_ptr(), *v_p = v.data_ptr(), *dense_p = dense.defined() ? dense.data_ptr() : nullptr,
             *res_p = res.data_ptr(), *gamma_p = gamma.data_ptr(), *beta_p = beta.data_ptr();
  void *ctx_p = ctx.data_ptr(), *y_p = y.data_ptr(), *ws_p = need > 0 ? ws.data_ptr() : nullptr;
  const int32_t *lens_p = i32(lens);
  const hipStream_t stream = stream_of(k);
  // small enough: one launch
  uint32_t *words = !dense_p && tag == out_tag && en_decode_layer_norm_pays((int)B, (int)H, (int)S, (int)D, tag) ? next_decode_words(k) : nullptr;
  if (words) {
    const int rc = without_gil([&] {
      return en_decode_layer_norm(q_p, k_p, v_p, ctx_p, lens_p, (int)B, (int)H, (int)S, (int)D, ks, vs, scale, res_p, gamma_p, beta_p, y_p,
                                  eps, tag, ws_p, need, words, stream);
    });
    if (rc != EN_ERR_UNSUPPORTED) {
      check(rc, "decode_layer");
      return THPVariable_Wrap(y);
    }
  }
  check(without_gil([&] {
          return en_decode_layer(q_p, k_p, v_p, ctx_p, lens_p, (int)B, (int)H, (int)S, (int)D, ks, vs, scale, dense_p, res_p, gamma_p, beta_p,
                                 y_p, hid, eps, tag, out_tag, ws_p, need, stream);
        }), "decode_layer");
  return THPVariable_Wrap(y);
}

// ---- single operations -------------------------------------------------------------------------------------------------
// What the Python calls of kernel/ do with plain operands: tensors of torch's own class on one GPU, contiguous where the entry point
// takes no strides, shapes and types as the call wants them, no function or dispatch mode on.  Anything else returns None with nothing
// launched, and the Python call goes on: it names what is wrong, copies, or has a mode see what it does.  A call takes 9..11 us of host time
// in Python and ctypes, more than most of these kernels do on a small batch.  us a layer where the host bounds it, before / now: paged
// decode (append, attention, LayerNorm: three calls) 32 / 14, the reference's sequence of operations (six calls) 72 / 48.

struct Lens {
  const Tensor *lens = nullptr, *cu = nullptr;
  int64_t batch = 0;
};

bool modes_on() { return at::impl::PythonTorchFunctionTLS::stack_len() > 0 || c10::impl::TorchDispatchModeTLS::any_modes_set(); }

const Tensor *plain(PyObject *o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor &t = THPVariable_Unpack(o);
  return t.is_cuda() && t.layout() == at::kStrided && t.numel() > 0 ? &t : nullptr;
}
const Tensor *plain_contiguous(PyObject *o) {
  const Tensor *t = plain(o);
  return t && t->is_contiguous() ? t : nullptr;
}
const Tensor *plain_rows(PyObject *o, int64_t dim) {      // the last dimension is contiguous
  const Tensor *t = plain(o);
  return t && t->dim() == dim && t->stride(dim - 1) == 1 ? t : nullptr;
}

int known_tag(const Tensor &t) {
  switch (t.scalar_type()) {
    case at::kFloat: return EN_F32;
    case at::kHalf: return EN_F16;
    case at::kBFloat16: return EN_BF16;
    default: return -1;
  }
}

// An attribute of a SeqInfo, which holds it on.
PyObject *held(PyObject *info, PyObject *key) {
  PyObject *v = PyObject_GetAttr(info, key);
  if (!v) fail("SeqInfo: attribute missing");
  Py_DECREF(v);
  return v;
}

// Lengths and prefix of a SeqInfo on t's device for `batch` sequences.
bool lens_of(PyObject *info, const Tensor &t, int64_t batch, bool with_cu, Lens &out) {
  static PyObject *const lens = PyUnicode_InternFromString("lens"), *const cu = PyUnicode_InternFromString("cu_seqlens"),
                         *const size = PyUnicode_InternFromString("batch_size");
  out.batch = integer(held(info, size));
  PyObject *l = held(info, lens), *c = held(info, cu);
  if (out.batch != batch || !THPVariable_CheckExact(l) || (with_cu && !THPVariable_CheckExact(c))) return false;
  out.lens = &THPVariable_Unpack(l);
  out.cu = with_cu ? &THPVariable_Unpack(c) : nullptr;
  for (const Tensor *x : {out.lens, out.cu})
    if (x && (x->device() != t.device() || x->scalar_type() != at::kInt || !x->is_contiguous())) return false;
  return out.lens->numel() >= batch && (!with_cu || out.cu->numel() > batch);
}

// SeqInfo.order_current_stream, looked at natively: most calls find their stream among the ordered ones.
void order_stream(PyObject *info, const Tensor &t) {
  static PyObject *const ready = PyUnicode_InternFromString("_ready"), *const ordered = PyUnicode_InternFromString("_ordered"),
                         *const order = PyUnicode_InternFromString("order_current_stream");
  const int pending = PyObject_IsTrue(held(info, ready));
  if (pending == 0) return;
  PyObject *raw = PyLong_FromVoidPtr(stream_of(t));
  const int there = pending < 0 || !raw ? -1 : PySet_Contains(held(info, ordered), raw);
  Py_XDECREF(raw);
  if (there < 0) fail("SeqInfo: streams");
  if (there) return;
  PyObject *done = PyObject_CallMethodNoArgs(info, order);
  if (!done) fail("SeqInfo: order_current_stream");
  Py_DECREF(done);
}

// Numbers and flags of a plain call.  False, with no Python error left, for what is none or does not fit: the Python call names it.
bool whole(PyObject *o, int64_t &v) {
  if (!PyLong_Check(o)) return false;
  int overflow = 0;
  v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}
bool number(PyObject *o, float &v) {
  if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
  const double d = PyFloat_AsDouble(o);
  if (d == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  v = (float)d;
  return true;
}
bool flag(PyObject *o, int &v) {      // True, False or a plain int: asking others may run their code, fail, or wait for a GPU
  if (!PyBool_Check(o) && !PyLong_CheckExact(o)) return false;
  v = PyObject_IsTrue(o);
  return true;
}

bool is_width(PyObject *shape, int64_t n) {      // n, or (n,)
  if (PyTuple_Check(shape) && PyTuple_GET_SIZE(shape) == 1) shape = PyTuple_GET_ITEM(shape, 0);
  int64_t width;
  return PyLong_CheckExact(shape) && whole(shape, width) && width == n;
}

// layer_norm(input, weight, bias, normalized_shape, eps, residual or None) -> y or None
PyObject *layer_norm(PyObject *const *a) {
  const Tensor *x = plain_contiguous(a[0]), *w = plain_contiguous(a[1]), *b = plain_contiguous(a[2]), *r = nullptr;
  if (!x || !w || !b || modes_on() || w->dim() != 1 || b->sizes() != w->sizes() || b->scalar_type() != w->scalar_type()) Py_RETURN_NONE;
  const int64_t n2 = w->numel();
  const int in = known_tag(*x), out = known_tag(*w);
  float eps;
  if (in < 0 || out < 0 || (in != out && in != EN_F32) || x->dim() < 1 || x->size(-1) != n2 || !is_width(a[3], n2) || !number(a[4], eps)) Py_RETURN_NONE;
  if (a[5] != Py_None) {
    r = plain_contiguous(a[5]);
    if (!r || r->scalar_type() != x->scalar_type() || r->sizes() != x->sizes() || r->device() != x->device()) Py_RETURN_NONE;
  }
  if (w->device() != x->device() || b->device() != x->device()) Py_RETURN_NONE;
  const c10::DeviceGuard guard(x->device());
  const Tensor y = at::empty(x->sizes(), w->options());
  void *y_p = y.data_ptr();
  const void *x_p = x->data_ptr(), *r_p = r ? r->data_ptr() : nullptr, *w_p = w->data_ptr(), *b_p = b->data_ptr();
  const int64_t n1 = x->numel() / n2;
  const hipStream_t stream = stream_of(*x);
  check(without_gil([&] { return en_layernorm_fwd(y_p, nullptr, nullptr, nullptr, x_p, r_p, nullptr, w_p, b_p, n1, n2, eps, in, out, stream); }),
        "layer_norm");
  return THPVariable_Wrap(y);
}

const Tensor *page_table(PyObject *o, const Tensor &pool, int64_t batch) {
  const Tensor *t = plain_contiguous(o);
  return t && t->dim() == 2 && t->size(0) == batch && t->scalar_type() == at::kInt && t->device() == pool.device() ? t : nullptr;
}

// kv_pages_append(k_new, v_new, k_pool, v_pool, SeqInfo, page_table, overflow or None) -> True or None
PyObject *kv_pages_append(PyObject *const *a) {
  const Tensor *kn = plain_rows(a[0], 3), *vn = plain_rows(a[1], 3), *kp = plain_rows(a[2], 4), *vp = plain_rows(a[3], 4), *over = nullptr;
  if (!kn || !vn || !kp || !vp || modes_on()) Py_RETURN_NONE;
  const int64_t N = kp->size(0), H = kp->size(1), P = kp->size(2), D = kp->size(3), B = kn->size(0), rows[3] = {B, H, D};
  Lens info;
  if (vp->sizes() != kp->sizes() || vp->strides() != kp->strides() || kn->sizes() != c10::IntArrayRef(rows) || vn->sizes() != kn->sizes() ||
      vn->strides() != kn->strides() || !lens_of(a[4], *kp, B, false, info))
    Py_RETURN_NONE;
  for (const Tensor *t : {kn, vn, vp})
    if (t->scalar_type() != kp->scalar_type() || t->device() != kp->device()) Py_RETURN_NONE;
  const Tensor *table = page_table(a[5], *kp, B);
  if (a[6] != Py_None) {
    over = plain_contiguous(a[6]);
    if (!over || over->scalar_type() != at::kInt || over->device() != kp->device()) Py_RETURN_NONE;
  }
  if (!table) Py_RETURN_NONE;
  const c10::DeviceGuard guard(kp->device());
  order_stream(a[4], *kp);
  const int64_t strides[3] = {kp->stride(0), kp->stride(1), kp->stride(2)}, n_sb = kn->stride(0), n_sh = kn->stride(1), pages = table->size(1);
  const void *kn_p = kn->data_ptr(), *vn_p = vn->data_ptr();
  void *kp_p = kp->data_ptr(), *vp_p = vp->data_ptr();
  const int32_t *lens_p = i32(*info.lens), *table_p = i32(*table);
  int32_t *over_p = over ? over->data_ptr<int32_t>() : nullptr;
  const int es = (int)kp->element_size();
  const hipStream_t stream = stream_of(*kp);
  check(without_gil([&] {
          return en_kv_append_paged(kn_p, vn_p, kp_p, vp_p, lens_p, table_p, (int)B, (int)H, (int)pages, (int)P, (int)N, (int)D, n_sb, n_sh,
                                    strides, es, over_p, stream);
        }), "kv_pages_append");
  Py_RETURN_TRUE;
}

// decode_attn_paged(q, k_pool, v_pool, SeqInfo, page_table, scale or None) -> ctx or None
PyObject *decode_attn_paged(PyObject *const *a) {
  const Tensor *q = plain_contiguous(a[0]), *kp = plain_rows(a[1], 4), *vp = plain_rows(a[2], 4);
  if (!q || !kp || !vp || modes_on()) Py_RETURN_NONE;
  const int64_t N = kp->size(0), H = kp->size(1), P = kp->size(2), D = kp->size(3), B = q->numel() / (H * D);
  const int tag = known_tag(*q);
  Lens info;
  if (tag < 0 || q->dim() < 2 || q->numel() != B * H * D || vp->sizes() != kp->sizes() || !lens_of(a[3], *q, B, false, info)) Py_RETURN_NONE;
  for (const Tensor *t : {kp, vp})
    if (t->scalar_type() != q->scalar_type() || t->device() != q->device()) Py_RETURN_NONE;
  const Tensor *table = page_table(a[4], *q, B);
  float scale = (float)std::pow((double)D, -0.5);
  if (!table || (a[5] != Py_None && !number(a[5], scale))) Py_RETURN_NONE;
  const c10::DeviceGuard guard(q->device());
  order_stream(a[3], *q);
  const int64_t pages = table->size(1), need = en_decode_attn_workspace_bytes((int)B, (int)H, (int)(pages * P), (int)D);
  const Tensor out = at::empty({B, H, 1, D}, q->options());
  Tensor ws;
  if (need > 0) ws = at::empty({need}, q->options().dtype(at::kByte));
  const int64_t ks[3] = {kp->stride(0), kp->stride(1), kp->stride(2)}, vs[3] = {vp->stride(0), vp->stride(1), vp->stride(2)};
  const void *q_p = q->data_ptr(), *k_p = kp->data_ptr(), *v_p = vp->data_ptr();
  void *out_p = out.data_ptr(), *ws_p = need > 0 ? ws.data_ptr() : nullptr;
  const int32_t *lens_p = i32(*info.lens), *table_p = i32(*table);
  const hipStream_t stream = stream_of(*q);
  check(without_gil([&] {
          return en_decode_attn_paged(q_p, k_p, v_p, out_p, lens_p, table_p, (int)B, (int)H, (int)pages, (int)P, (int)N, (int)D, ks, vs, scale,
                                      tag, ws_p, need, stream);
        }), "decode_attn_paged");
  return THPVariable_Wrap(out);
}

bool fits_int(std::initializer_list<int64_t> values) {
  for (const int64_t v : values)
    if (v < 1 || v > INT32_MAX) return false;
  return true;
}

// depad(src, SeqInfo, batch, left_padded, total) -> packed rows or None
PyObject *depad(PyObject *const *a) {
  const Tensor *src = plain_contiguous(a[0]);
  if (!src || modes_on() || src->dim() != 3) Py_RETURN_NONE;
  const int64_t S = src->size(1), hid = src->size(2);
  const int es = (int)src->element_size();
  int64_t batch, total;
  int left;
  Lens info;
  if ((es != 2 && es != 4) || !whole(a[2], batch) || !flag(a[3], left) || !whole(a[4], total) || !fits_int({batch, S, total}) || src->size(0) < batch || !lens_of(a[1], *src, batch, true, info)) Py_RETURN_NONE;
  const c10::DeviceGuard guard(src->device());
  order_stream(a[1], *src);
  const Tensor dst = at::empty({1, total, hid}, src->options());
  const void *src_p = src->data_ptr();
  void *dst_p = dst.data_ptr();
  const int32_t *cu_p = i32(*info.cu);
  const hipStream_t stream = stream_of(*src);
  check(without_gil([&] { return en_depad(src_p, dst_p, cu_p, (int)batch, (int)S, hid, es, left, stream); }), "depad");
  return THPVariable_Wrap(dst);
}

// transpose_pad(src, SeqInfo, batch, max_seq_len, heads, size_per_head) -> padded tensor or None
PyObject *transpose_pad(PyObject *const *a) {
  const Tensor *src = plain_contiguous(a[0]);
  if (!src || modes_on()) Py_RETURN_NONE;
  const int es = (int)src->element_size();
  int64_t batch, S, H, D;
  Lens info;
  if ((es != 2 && es != 4) || !whole(a[2], batch) || !whole(a[3], S) || !whole(a[4], H) || !whole(a[5], D) || !fits_int({batch, S, H, D}) || src->numel() % (H * D) || !lens_of(a[1], *src, batch, true, info)) Py_RETURN_NONE;
  const c10::DeviceGuard guard(src->device());
  order_stream(a[1], *src);
  const Tensor dst = at::empty({batch, H, S, D}, src->options());
  const void *src_p = src->data_ptr();
  void *dst_p = dst.data_ptr();
  const int32_t *cu_p = i32(*info.cu);
  const hipStream_t stream = stream_of(*src);
  check(without_gil([&] { return en_transpose_pad(src_p, dst_p, cu_p, (int)batch, (int)S, (int)H, (int)D, es, stream); }), "transpose_pad");
  return THPVariable_Wrap(dst);
}

// transpose_depad(src, SeqInfo, batch, total, max_seq_len, heads, size_per_head) -> packed tensor or None
PyObject *transpose_depad(PyObject *const *a) {
  const Tensor *src = plain_contiguous(a[0]);
  if (!src || modes_on()) Py_RETURN_NONE;
  const int es = (int)src->element_size();
  int64_t batch, total, S, H, D;
  Lens info;
  if ((es != 2 && es != 4) || !whole(a[2], batch) || !whole(a[3], total) || !whole(a[4], S) || !whole(a[5], H) || !whole(a[6], D) || !fits_int({batch, total, S, H, D}) || src->numel() / batch / H / S != D || src->numel() != batch * H * S * D ||
      !lens_of(a[1], *src, batch, true, info))
    Py_RETURN_NONE;
  const c10::DeviceGuard guard(src->device());
  order_stream(a[1], *src);
  const Tensor dst = at::empty({1, total, H, D}, src->options());
  const void *src_p = src->data_ptr();
  void *dst_p = dst.data_ptr();
  const int32_t *cu_p = i32(*info.cu);
  const hipStream_t stream = stream_of(*src);
  check(without_gil([&] { return en_transpose_depad(src_p, dst_p, cu_p, (int)batch, (int)S, (int)H, (int)D, es, stream); }), "transpose_depad");
  return THPVariable_Wrap(dst);
}

// scale_mask_softmax(src, SeqInfo, batch, max_seq_len, heads, scale, causal, tail_rows) -> True (in place) or None
PyObject *scale_mask_softmax(PyObject *const *a) {
  const Tensor *src = plain_contiguous(a[0]);
  if (!src || modes_on()) Py_RETURN_NONE;
  const int tag = known_tag(*src);
  int64_t batch, S, H, tail;
  int causal;
  float scale;
  Lens info;
  if (tag < 0 || !whole(a[2], batch) || !whole(a[3], S) || !whole(a[4], H) || !number(a[5], scale) || !flag(a[6], causal) || !whole(a[7], tail) ||
      !fits_int({batch, S, H}) || tail < 0 || tail > INT32_MAX || src->numel() / batch / H / S != S ||
      src->numel() != batch * H * S * S || !lens_of(a[1], *src, batch, false, info))
    Py_RETURN_NONE;
  const c10::DeviceGuard guard(src->device());
  order_stream(a[1], *src);
  void *src_p = src->data_ptr();
  const int32_t *lens_p = i32(*info.lens);
  const hipStream_t stream = stream_of(*src);
  check(without_gil([&] {
          return en_scale_mask_softmax(src_p, lens_p, nullptr, (int)batch, (int)H, (int)S, (int)S, scale, causal, (int)tail, tag, stream);
        }), "scale_mask_softmax");
  Py_RETURN_TRUE;
}

// The workgroup order of an attention call (SeqInfo.tile_table), None for a SeqInfo of one call.  It lives on in the SeqInfo, or in
// `keep` until the launch.
const int32_t *tile_table(PyObject *info, int64_t heads, int64_t q_len, int64_t k_len, int64_t channels, int64_t elem, bool causal, Tensor &keep) {
  static PyObject *const ephemeral = PyUnicode_InternFromString("ephemeral"), *const get = PyUnicode_InternFromString("tile_table");
  const int once = PyObject_IsTrue(held(info, ephemeral));
  if (once) {
    if (once < 0) fail("SeqInfo: ephemeral");
    return nullptr;
  }
  PyObject *args[6] = {info, PyLong_FromLongLong(heads), PyLong_FromLongLong(q_len), PyLong_FromLongLong(2 * k_len * channels * elem),
                       PyLong_FromLong(128), causal ? Py_True : Py_False};
  PyObject *t = args[1] && args[2] && args[3] && args[4] ? PyObject_VectorcallMethod(get, args, 6, nullptr) : nullptr;
  for (int i = 1; i < 5; ++i) Py_XDECREF(args[i]);
  if (!t) fail("SeqInfo: tile_table");
  if (THPVariable_Check(t)) keep = THPVariable_Unpack(t);
  Py_DECREF(t);
  if (!keep.defined()) fail("SeqInfo: tile_table gives no tensor");
  return i32(keep);
}

// attn_qk(q, k, SeqInfo, alpha, causal) -> scores or None
PyObject *attn_qk(PyObject *const *a) {
  const Tensor *q = plain_rows(a[0], 4), *k = plain_rows(a[1], 4);
  if (!q || !k || modes_on()) Py_RETURN_NONE;
  const int64_t B = q->size(0), H = q->size(1), Sq = q->size(2), D = q->size(3), Sk = k->size(2);
  const int tag = known_tag(*q);
  int causal;
  float alpha;
  Lens info;
  if (tag < 0 || !number(a[3], alpha) || !flag(a[4], causal) || k->size(0) != B || k->size(1) != H || k->size(3) != D || k->scalar_type() != q->scalar_type() ||
      k->device() != q->device() || !fits_int({B, H, Sq, Sk, D}) || !lens_of(a[2], *q, B, false, info))
    Py_RETURN_NONE;
  const c10::DeviceGuard guard(q->device());
  order_stream(a[2], *q);
  Tensor keep;
  const int32_t *table = tile_table(a[2], H, Sq, Sk, D, q->element_size(), causal, keep), *lens_p = i32(*info.lens);
  const Tensor out = at::empty({B, H, Sq, Sk}, q->options());
  const void *q_p = q->data_ptr(), *k_p = k->data_ptr();
  void *out_p = out.data_ptr();
  const int64_t q0 = q->stride(0), q1 = q->stride(1), q2 = q->stride(2), k0 = k->stride(0), k1 = k->stride(1), k2 = k->stride(2);
  const hipStream_t stream = stream_of(*q);
  check(without_gil([&] {
          return en_attn_qk(q_p, k_p, out_p, lens_p, nullptr, (int)B, (int)H, (int)Sq, (int)Sk, (int)D, q0, q1, q2, k0, k1, k2, alpha, causal, tag,
                            nullptr, nullptr, 0, table, stream);
        }), "attn_qk");
  return THPVariable_Wrap(out);
}

// attn_pv(p, v, SeqInfo, causal) -> context or None
PyObject *attn_pv(PyObject *const *a) {
  const Tensor *p = plain_contiguous(a[0]), *v = plain_rows(a[1], 4);
  if (!p || !v || modes_on() || p->dim() != 4) Py_RETURN_NONE;
  const int64_t B = p->size(0), H = p->size(1), Sq = p->size(2), Sk = p->size(3), D = v->size(3);
  const int tag = known_tag(*p);
  int causal;
  Lens info;
  if (tag < 0 || !flag(a[3], causal) || v->size(0) != B || v->size(1) != H || v->size(2) != Sk || v->scalar_type() != p->scalar_type() ||
      v->device() != p->device() || !fits_int({B, H, Sq, Sk, D}) || !lens_of(a[2], *p, B, false, info))
    Py_RETURN_NONE;
  const c10::DeviceGuard guard(p->device());
  order_stream(a[2], *p);
  Tensor keep;
  const int32_t *table = tile_table(a[2], H, Sq, Sk, D, p->element_size(), causal, keep), *lens_p = i32(*info.lens);
  const Tensor out = at::empty({B, H, Sq, D}, p->options());
  const void *p_p = p->data_ptr(), *v_p = v->data_ptr();
  void *out_p = out.data_ptr();
  const int64_t v0 = v->stride(0), v1 = v->stride(1), v2 = v->stride(2), c0 = H * Sq * D, c1 = Sq * D, c2 = D;
  const hipStream_t stream = stream_of(*p);
  check(without_gil([&] {
          return en_attn_pv(p_p, v_p, out_p, lens_p, nullptr, (int)B, (int)H, (int)Sq, (int)Sk, (int)D, v0, v1, v2, c0, c1, c2, causal, 0, tag,
                            nullptr, nullptr, 0, table, stream);
        }), "attn_pv");
  return THPVariable_Wrap(out);
}

// ---- the look at a block's modules in front of block_decode ------------------------------------------------------------

PyObject *name(const char *s) { return PyUnicode_InternFromString(s); }

// A module without hooks, without a compiled call and without any of the methods `own` set on the instance.  `dict`: its
// __dict__, borrowed.  -1 with a Python error set, 0 no, 1 yes.
int plain_module(PyObject *module, std::initializer_list<PyObject *> own, PyObject *&dict) {
  static PyObject *const hooks = name("_forward_hooks"), *const pre_hooks = name("_forward_pre_hooks"), *const compiled = name("_compiled_call_impl");
  PyObject **at = _PyObject_GetDictPtr(module);
  if (!at || !*at) return 0;
  dict = *at;
  for (PyObject *key : {hooks, pre_hooks}) {
    PyObject *d = PyDict_GetItemWithError(dict, key);
    if (!d) return PyErr_Occurred() ? -1 : 0;
    const int used = PyObject_IsTrue(d);
    if (used) return used < 0 ? -1 : 0;
  }
  for (PyObject *key : own) {
    const int there = PyDict_Contains(dict, key);
    if (there) return there < 0 ? -1 : 0;
  }
  PyObject *c = PyObject_GetAttr(module, compiled);
  if (!c) return -1;
  const bool none = c == Py_None;
  Py_DECREF(c);
  return none;
}

// plain_step(attention, MLP, activation or None, norm1, qkv, dense, norm2, mlp1, mlp2)
// -> [norm1 w, b, eps, qkv w, b, dense w, b, norm2 w, b, eps, mlp1 w, b, mlp2 w, b], or None where a module is hooked or
// compiled, has a method of its own, or holds weight or bias otherwise than as a parameter
PyObject *plain_step(PyObject *const *a) {
  static PyObject *const forward = name("forward"), *const last = name("forward_last"), *const project = name("_project"),
                         *const rows = name("forward_rows"), *const parameters = name("_parameters"), *const weight = name("weight"),
                         *const bias = name("bias"), *const eps = name("eps");
  PyObject *dict = nullptr;
  for (int i = 0; i < 3; ++i) {
    if (a[i] == Py_None) continue;
    const int ok = plain_module(a[i], {forward, last, project, rows}, dict);
    if (ok < 0) return nullptr;
    if (!ok) Py_RETURN_NONE;
  }
  PyObject *out = PyList_New(0);
  auto done = [&](bool error) -> PyObject * {
    Py_XDECREF(out);
    if (error) return nullptr;
    Py_RETURN_NONE;
  };
  if (!out) return nullptr;
  for (int i = 3; i < 9; ++i) {
    const int ok = plain_module(a[i], {forward, weight, bias}, dict);
    if (ok != 1) return done(ok < 0);
    PyObject *p = PyDict_GetItemWithError(dict, parameters);
    if (!p || !PyDict_Check(p)) return done(PyErr_Occurred());
    for (PyObject *key : {weight, bias}) {
      PyObject *t = PyDict_GetItemWithError(p, key);
      if (!t) return done(PyErr_Occurred());
      if (PyList_Append(out, t)) return done(true);
    }
    if (i == 3 || i == 6) {
      PyObject *e = PyObject_GetAttr(a[i], eps);
      if (!e) return done(true);
      const int failed = PyList_Append(out, e);
      Py_DECREF(e);
      if (failed) return done(true);
    }
  }
  return out;
}

// block_decode(hidden, norm1 w, b, eps, qkv w, b, dense w, b, norm2 w, b, eps, mlp1 w, b, mlp2 w, b, activation, heads, scale,
//              k_cache, v_cache, lens, page_table or None, cache_len, out [B, positions, hidden], position)
// -> out[:, :position + 1] with the block's output for the newest position of `hidden` at `position`, or None, with nothing
// done, where en_block_decode has no kernel for these tensors.
PyObject *block_decode(PyObject *const *a) {
  // a tensor subclass computes in its own way (quantised weights behind a plain Linear): the general path asks it
  for (int i : {0, 1, 2, 4, 5, 6, 7, 8, 9, 11, 12, 13, 14})
    if (a[i] != Py_None && !THPVariable_CheckExact(a[i])) Py_RETURN_NONE;
  const Tensor &x = gpu(a[0], "hidden_states", false);
  const Tensor &out = gpu(a[23], "out", false);
  const Tensor &k = gpu(a[18], "k_cache", false), &v = gpu(a[19], "v_cache", false), &lens = gpu(a[20], "lens");
  const auto dt = x.scalar_type();
  const int64_t heads = integer(a[16]);
  if ((dt != at::kHalf && dt != at::kBFloat16) || x.dim() != 3 || x.numel() == 0 || x.stride(2) != 1 || out.scalar_type() != dt || out.stride(2) != 1 ||
      k.scalar_type() != dt || k.dim() != 4 || k.stride(3) != 1 || v.sizes() != k.sizes() || v.strides() != k.strides())
    Py_RETURN_NONE;
  const int64_t B = x.size(0), hid = x.size(2), D = k.size(3), position = integer(a[24]);
  if (heads * D != hid || k.size(1) != heads || out.size(0) != B || out.size(2) != hid || position < 0 || position >= out.size(1) ||
      lens.numel() != B || lens.scalar_type() != at::kInt)
    Py_RETURN_NONE;
  for (const Tensor *t : {&out, &k, &v, &lens})
    if (t->device() != x.device()) Py_RETURN_NONE;
  bool usable = true;
  // [rows, cols] or, with rows = 1, [cols]: a weight laid out another way is the general path's to refuse
  auto weight = [&](int i, int64_t rows, int64_t cols) -> const void * {
    if (a[i] == Py_None) return nullptr;
    const Tensor &t = tensor(a[i], "weight");
    const int64_t shape[2] = {rows, cols};
    if (!t.is_cuda() || t.device() != x.device() || t.scalar_type() != dt || !t.is_contiguous() ||
        t.sizes() != (rows == 1 ? c10::IntArrayRef(&cols, 1) : c10::IntArrayRef(shape, 2)))
      usable = false;
    return t.data_ptr();
  };
  const Tensor &w1 = tensor(a[11], "weight");
  if (w1.dim() != 2) Py_RETURN_NONE;
  const int64_t mlp = w1.size(0);
  en_block_decode_args p{};
  p.x = static_cast<const char *>(x.data_ptr()) + (x.size(1) - 1) * x.stride(1) * 2;
  p.x_stride = B > 1 ? x.stride(0) : hid;
  p.norm1_weight = weight(1, 1, hid); p.norm1_bias = weight(2, 1, hid); p.norm1_eps = real(a[3]);
  p.qkv_weight = weight(4, 3 * hid, hid); p.qkv_bias = weight(5, 1, 3 * hid);
  p.dense_weight = weight(6, hid, hid); p.dense_bias = weight(7, 1, hid);
  p.norm2_weight = weight(8, 1, hid); p.norm2_bias = weight(9, 1, hid); p.norm2_eps = real(a[10]);
  p.mlp1_weight = weight(11, mlp, hid); p.mlp1_bias = weight(12, 1, mlp);
  p.mlp2_weight = weight(13, hid, mlp); p.mlp2_bias = weight(14, 1, hid);
  if (!usable) Py_RETURN_NONE;
  p.activation = (int)integer(a[15]);
  p.scale = real(a[17]);
  p.dtype = dtype_tag(x, "block_decode");
  p.batch = (int)B; p.head_num = (int)heads; p.size_per_head = (int)D; p.mlp_width = mlp;
  p.k_cache = k.data_ptr(); p.v_cache = v.data_ptr();
  for (int i = 0; i < 3; ++i) p.cache_strides[i] = k.stride(i);
  p.cache_len = (int)integer(a[22]);
  p.kv_lens = lens.data_ptr<int32_t>();
  if (a[21] != Py_None) {
    const Tensor &table = gpu(a[21], "page_table");
    if (table.scalar_type() != at::kInt || table.dim() != 2 || table.size(0) != B || table.device() != x.device()) Py_RETURN_NONE;
    p.page_table = i32(table);
    p.max_pages_per_seq = (int)table.size(1); p.page_size = (int)k.size(2); p.num_pages = (int)k.size(0);
  } else if (k.size(0) != B || k.size(2) != p.cache_len) {
    Py_RETURN_NONE;
  }
  p.y = static_cast<char *>(out.data_ptr()) + position * out.stride(1) * 2;
  p.y_stride = out.stride(0);
  const c10::DeviceGuard guard(x.device());
  p.workspace_bytes = en_block_decode_workspace_bytes(p.batch, p.head_num, p.size_per_head, p.mlp_width, p.cache_len);
  const Tensor ws = at::empty({p.workspace_bytes}, x.options().dtype(at::kByte));
  p.workspace = ws.data_ptr();
  const hipStream_t stream = stream_of(x);
  const int rc = without_gil([&] { return en_block_decode(&p, stream); });
  if (rc == EN_ERR_UNSUPPORTED || rc == EN_ERR_ALIGN) Py_RETURN_NONE;      // found before anything was launched
  check(rc, "block_decode");
  if (!lens.is_inference()) lens.unsafeGetTensorImpl()->bump_version();      // the lengths have moved on
  return THPVariable_Wrap(out.narrow(1, 0, position + 1));
}

// block_prefill(x [1,T,hidden], norm1 w, b, eps, qkv w, b, dense w, b, norm2 w, b, eps, mlp1 w, b, mlp2 w, b, activation, heads, scale,
//               causal, lens, cu_seqlens, tile table or None, batch, max_seq_len, address of en_linear or 0, its workspace or None,
//               what to call with the packed projections [1,T,3 hidden] or None)
// -> block's output [1,T,hidden], or None, with nothing done, where a tensor is not what the kernels take.  The ops are those of the
// general step one by one: LayerNorm, projection, fused attention on packed rows, the call with the projections (it fills a cache),
// projection, residual + LayerNorm that keeps the sum, MLP (both GEMMs by en_linear with the activation in its epilogue, or by torch
// around exact GELU), sum.  A tensor is given up where it is last read: at its peak, the MLP, the call holds x, sum, h2 and the MLP's
// own, a row of hidden less than the general form, which keeps the first LayerNorm's output.
typedef int (*en_linear_fn)(const void *, const void *, const void *, void *, int64_t, int64_t, int64_t, int, int, int, void *, int64_t,
                            hipStream_t);
PyObject *block_prefill(PyObject *const *a) {
  for (int i : {0, 1, 2, 4, 5, 6, 7, 8, 9, 11, 12, 13, 14})
    if (a[i] != Py_None && !THPVariable_CheckExact(a[i])) Py_RETURN_NONE;
  const Tensor &x = gpu(a[0], "x", false);
  const auto dt = x.scalar_type();
  const int64_t heads = integer(a[16]), batch = integer(a[22]), S = integer(a[23]);
  if ((dt != at::kHalf && dt != at::kBFloat16) || x.dim() != 3 || x.size(0) != 1 || x.numel() == 0 || !x.is_contiguous()) Py_RETURN_NONE;
  const int64_t T = x.size(1), hid = x.size(2), D = heads > 0 ? hid / heads : 0;
  if (D * heads != hid || D % 8 || D > 128) Py_RETURN_NONE;
  bool usable = true;
  auto weight = [&](int i, int64_t rows, int64_t cols) -> Tensor {
    if (a[i] == Py_None) return Tensor();
    const Tensor &t = tensor(a[i], "weight");
    const int64_t shape[2] = {rows, cols};
    if (!t.is_cuda() || t.device() != x.device() || t.scalar_type() != dt || !t.is_contiguous() ||
        t.sizes() != (rows == 1 ? c10::IntArrayRef(&cols, 1) : c10::IntArrayRef(shape, 2)))
      usable = false;
    return t;
  };
  const Tensor &w1 = tensor(a[11], "weight");
  if (w1.dim() != 2) Py_RETURN_NONE;
  const int64_t mlp = w1.size(0);
  const Tensor n1w = weight(1, 1, hid), n1b = weight(2, 1, hid), qkv_w = weight(4, 3 * hid, hid), qkv_b = weight(5, 1, 3 * hid),
               dense_w = weight(6, hid, hid), dense_b = weight(7, 1, hid), n2w = weight(8, 1, hid), n2b = weight(9, 1, hid),
               m1w = weight(11, mlp, hid), m1b = weight(12, 1, mlp), m2w = weight(13, hid, mlp), m2b = weight(14, 1, hid);
  const float eps1 = real(a[3]), eps2 = real(a[10]), scale = real(a[17]);
  const int act = (int)integer(a[15]), causal = (int)integer(a[18]);
  const Tensor &lens = gpu(a[19], "lens"), &cu = gpu(a[20], "cu_seqlens");
  const int32_t *table = a[21] == Py_None ? nullptr : i32(gpu(a[21], "tile_table"));
  const auto linear = reinterpret_cast<en_linear_fn>((uintptr_t)PyLong_AsUnsignedLongLong(a[24]));
  Tensor ws;
  if (a[25] != Py_None) ws = gpu(a[25], "workspace");
  if (!usable || !n1w.defined() || !n1b.defined() || !n2w.defined() || !n2b.defined() || !qkv_w.defined() || !dense_w.defined() ||
      !m1w.defined() || !m2w.defined() || lens.device() != x.device() || cu.device() != x.device() || lens.numel() != batch ||
      cu.numel() != batch + 1 || !(scale > 0.f) || (linear && !ws.defined()) || (!linear && act != EN_ACT_GELU))
    Py_RETURN_NONE;
  const c10::DeviceGuard guard(x.device());
  const int tag = dtype_tag(x, "block_prefill");
  const hipStream_t stream = stream_of(x);
  const int32_t *lens_p = i32(lens), *cu_p = i32(cu);
  Tensor kvq, ctx, y;
  auto attend = [&]() -> int {
    const Tensor h = at::empty_like(x);
    check(en_layernorm_fwd(h.data_ptr(), nullptr, nullptr, nullptr, x.data_ptr(), nullptr, nullptr, n1w.data_ptr(), n1b.data_ptr(), T, hid,
                           eps1, tag, tag, stream), "layer_norm");
    kvq = at::linear(h, qkv_w, qkv_b);
    // packed rows of 3 heads x D, ordered k, v, q (attention.py:74)
    ctx = at::empty({1, T, hid}, x.options());
    const int64_t in[3] = {0, D, 3 * hid}, out[3] = {0, D, hid};
    const char *rows = static_cast<const char *>(kvq.data_ptr());
    check(en_attn_fused(rows + 2 * hid * 2, rows, rows + hid * 2, ctx.data_ptr(), lens_p, nullptr, (int)batch, (int)heads, (int)S, (int)S, (int)D,
                        in, in, in, out, cu_p, cu_p, scale, causal, tag, table, 0, stream), "attn_fused_varlen");
    return EN_OK;
  };
  (void)without_gil(attend);
  if (a[26] != Py_None) {
    PyObject *rows = THPVariable_Wrap(kvq);
    PyObject *done = rows ? PyObject_CallOneArg(a[26], rows) : nullptr;
    Py_XDECREF(rows);
    if (!done) return nullptr;
    Py_DECREF(done);
  }
  kvq.reset();      // under the lock: a Python object may belong to it
  auto rest = [&]() -> int {
    Tensor att = at::linear(ctx, dense_w, dense_b);
    ctx.reset();
    Tensor h2 = at::empty_like(x);
    const Tensor sum = at::empty_like(x);
    check(en_layernorm_fwd(h2.data_ptr(), nullptr, nullptr, sum.data_ptr(), att.data_ptr(), x.data_ptr(), nullptr, n2w.data_ptr(), n2b.data_ptr(),
                           T, hid, eps2, tag, tag, stream), "layer_norm");
    att.reset();
    Tensor m;
    if (linear) {
      const Tensor f = at::empty({1, T, mlp}, x.options());
      m = at::empty_like(x);
      auto ptr = [](const Tensor &t) -> const void * { return t.defined() ? t.data_ptr() : nullptr; };
      if (linear(h2.data_ptr(), m1w.data_ptr(), ptr(m1b), f.data_ptr(), T, hid, mlp, act, tag, -1, ws.data_ptr(), ws.numel(), stream) < 0 ||
          linear(f.data_ptr(), m2w.data_ptr(), ptr(m2b), m.data_ptr(), T, mlp, hid, 0, tag, -1, ws.data_ptr(), ws.numel(), stream) < 0)
        fail("linear: the GEMM could not be launched");
    } else {
      Tensor f = at::linear(h2, m1w, m1b);
      f = at::gelu(f);
      m = at::linear(f, m2w, m2b);
    }
    h2.reset();
    y = at::add(sum, m);
    return EN_OK;
  };
  (void)without_gil(rest);
  return THPVariable_Wrap(y);
}

// ---- module --------------------------------------------------------------------------------------------------------

template <PyObject *(*F)(PyObject *const *), int N>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "%d arguments expected, %zd given", N, n);
    return nullptr;
  }
  try {
    return F(args);
  } catch (...) {      // as torch's own calls raise it: an allocation that does not fit is torch.OutOfMemoryError
    if (!PyErr_Occurred()) torch::translate_exception_to_python(std::current_exception());
    return nullptr;
  }
}

PyObject *source_hash(PyObject *, PyObject *) { return PyUnicode_FromString(EN_SOURCE_HASH); }

#define EN_FAST(name, nargs, doc) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&entry<name, nargs>)), METH_FASTCALL, doc}

PyMethodDef kMethods[] = {
    {"source_hash", source_hash, METH_NOARGS, "digest of the sources this module was built from"},
    EN_FAST(record_event, 1, "event recorded on the current stream of the tensor's device"),
    EN_FAST(wait_event, 2, "makes the current stream of the tensor's device wait for the event"),
    EN_FAST(prefix_sum, 2, "(cu_seqlens, lens) of a batch"),
    EN_FAST(layer_tables, 8, "(row offsets, tile table, meeting words) of a batch"),
    EN_FAST(layer, 19, "en_padding_removal_layer on new outputs"),
    EN_FAST(decode_words, 1, "address of the meeting words of a decode layer on the current stream, or None"),
    EN_FAST(decode_layer, 10, "en_decode_layer on new outputs"),
    EN_FAST(layer_norm, 6, "layer_norm_forward of plain operands, or None"),
    EN_FAST(kv_pages_append, 7, "kv_pages_append of plain operands, or None"),
    EN_FAST(decode_attn_paged, 6, "decode_attn_paged of plain operands, or None"),
    EN_FAST(depad, 5, "depad of plain operands, or None"),
    EN_FAST(transpose_pad, 6, "transpose_pad of plain operands, or None"),
    EN_FAST(transpose_depad, 7, "transpose_depad of plain operands, or None"),
    EN_FAST(scale_mask_softmax, 8, "scale_mask_softmax of plain operands, or None"),
    EN_FAST(attn_qk, 5, "attn_qk of plain operands, or None"),
    EN_FAST(attn_pv, 4, "attn_pv of plain operands, or None"),
    EN_FAST(plain_step, 9, "what block_decode takes of a block's modules, or None where the general step has to see them"),
    EN_FAST(block_prefill, 27, "a pre-LN block over packed rows, its attention on the packed projections"),
    EN_FAST(block_decode, 25, "en_block_decode into a position of an output history"),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_front", "host side of the layer and decode steps", -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__front(void) { return PyModule_Create(&kModule); }
