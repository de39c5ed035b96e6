// _blr_host: the per-call host work of the triton_funcs shims in native code - look at the tensors, size and find the workspace,
// allocate the result, call the C ABI of libblr.so.
//
// An eager call at decode sizes is a few microseconds of kernels behind the host work of issuing it; in Python that work
// (attribute reads, torch.empty, the current stream, ctypes' argument conversion) was 15 us a call, here it is about one
// next to the launches themselves.  Every entry takes the regular case only - GPU tensors of one dtype, contiguous weights
// of the right shape, activations with whole rows - and returns None for anything else, whereupon the Python shim goes its
// own way and raises what it always raised.  The C ABI is reached through addresses handed over by bind(), so that libblr.so
// stays a plain C library and can be replaced (BLR_LIB) without building this again.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/Context.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <algorithm>
#include <cstdint>
#include <map>
#include <tuple>
#include <vector>
#include "../../include/blr.h"

namespace {

struct Api {
  decltype(&blr_blast_workspace_bytes) blast_ws;
  decltype(&blr_blast_fwd) blast;
  decltype(&blr_blast_fwd_ep2) blast_ep;
  decltype(&blr_blast_q_workspace_bytes) q_ws;
  decltype(&blr_blast_q_fwd) q;
  decltype(&blr_blast_q_fwd_ep2) q_ep;
  decltype(&blr_monarch_workspace_bytes) monarch_ws;
  decltype(&blr_monarch_fwd) monarch;
  decltype(&blr_monarch_fwd_ep2) monarch_ep;
  decltype(&blr_low_rank_workspace_bytes) low_rank_ws;
  decltype(&blr_low_rank_fwd) low_rank;
  decltype(&blr_low_rank_fwd_ep2) low_rank_ep;
  decltype(&blr_dense_workspace_bytes) dense_ws;
  decltype(&blr_dense_fwd) dense;
  decltype(&blr_dense_fwd_ep2) dense_ep;
  decltype(&blr_ep_workspace_bytes) ep_ws;
  decltype(&blr_ln_modulate) ln_modulate;
  decltype(&blr_attention_qkv) attention;
  decltype(&blr_silu_linear) silu_linear;
  decltype(&blr_last_error) last_error;
} api = {};
PyObject* blr_error = nullptr;                     // triton_funcs._lib.BlrError

// ---- workspaces: one per (device, stream, kind), kept until the process ends (the shims' contract; see _lib.workspace) -------
// Only touched with the interpreter lock held, and never destroyed: the process may end after the device runtime did.
using WsKey = std::tuple<int, void*, bool>;
auto& workspaces = *new std::map<WsKey, at::Tensor>;
// Outgrown ones stay as they are: a graph captured while they were in use replays into their memory, the control words of a streaming
// one among it.  Every growth doubles at least, so all of them together are smaller than the one in use.
auto& outgrown = *new std::vector<at::Tensor>;
// What a call under capture is given when none of them is large enough: memory of the graph, zeroed by every replay and by nothing
// else, so only calls of the same capture use it.
auto& captured = *new std::map<WsKey, std::pair<unsigned long long, at::Tensor>>;

// the capture that `stream` is part of, 0 outside of one (the default stream cannot be)
unsigned long long capture_of(void* stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (!stream) return 0;
  if (hipStreamGetCaptureInfo((hipStream_t)stream, &status, &id) != hipSuccess) { (void)hipGetLastError(); return 0; }
  return status == hipStreamCaptureStatusActive ? id : 0;
}

const at::Tensor& workspace(const at::Device& dev, void* stream, size_t bytes, bool streaming) {
  const WsKey key{dev.index(), stream, streaming};
  at::Tensor& ws = workspaces[key];
  const size_t have = ws.defined() ? (size_t)ws.numel() : 0;
  if (have >= bytes && have) return ws;
  auto make = [&](size_t n) { return at::zeros({(int64_t)n}, at::TensorOptions().dtype(at::kByte).device(dev)); };
  if (const unsigned long long id = capture_of(stream)) {
    auto& c = captured[key];
    if (c.first != id || (size_t)c.second.numel() < bytes) c = {id, make(bytes)};
    return c.second;
  }
  at::Tensor grown = make(std::max({bytes, 2 * have, (size_t)1 << 20}));
  if (have) outgrown.push_back(std::move(ws));
  return ws = std::move(grown);
}

// ---- what a call looks at ---------------------------------------------------------------------------------------------------
// (plain tensors and parameters with memory of their own: a subclass may mean something else by its data, and what vmap, grad and their
// like hand out has none.  Asking those for their address throws, which must not happen once the interpreter lock is given up.)
const at::Tensor* tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                         c10::DispatchKey::Functionalize});
  return t.has_storage() && !t.key_set().has_any(wrapped) ? &t : nullptr;
}

int dtype_code(at::ScalarType t) { return t == at::kHalf ? BLR_F16 : t == at::kBFloat16 ? BLR_BF16 : t == at::kFloat ? BLR_F32 : -1; }

// a contiguous weight of dtype t on x's device
bool weight(const at::Tensor* w, const at::Tensor& x, int64_t dims) {
  return w && w->is_cuda() && w->dim() == dims && w->scalar_type() == x.scalar_type() && w->device() == x.device() && w->is_contiguous();
}

struct Rows { int64_t M, ld; };
// x (.., in) as M rows of in values, ld apart; false when that takes a copy
bool rows_of(const at::Tensor& x, int64_t in, Rows& r) {
  const int64_t d = x.dim();
  if (!x.is_cuda() || d < 1 || x.size(d - 1) != in || in <= 0) return false;
  r.M = x.numel() / in;
  if (r.M < 1 || r.M > INT32_MAX) return false;
  if (x.is_contiguous()) { r.ld = in; return true; }
  if (d < 2 || x.stride(d - 1) != 1 || x.size(d - 2) != r.M || x.stride(d - 2) < in) return false;   // leading dimensions of 1 only
  r.ld = x.stride(d - 2);
  return true;
}

// no gradient or tangent, no transform and no lazy form
bool plain(const at::Tensor& t) {
  return t.is_cuda() && t.layout() == at::kStrided && !(at::GradMode::is_enabled() && t.requires_grad()) && !t._fw_grad(0).defined() &&
         !t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                                   c10::DispatchKey::Functionalize, c10::DispatchKey::Negative, c10::DispatchKey::Conjugate, c10::DispatchKey::ZeroTensor}));
}

struct Ep {
  bool on = false;
  const void* bias = nullptr; int act = 0;
  const void* gate = nullptr; int gate_rows = 0; int64_t ld_gate = 0;
  const void* resid = nullptr; int64_t ld_resid = 0;
};
// ep: None or (bias, act, gate, gate_rows, residual), as _lib.fused_epilogue leaves it
bool epilogue(PyObject* ep, const at::Tensor& x, int64_t M, int64_t out_f, Ep& e) {
  if (ep == Py_None) return true;
  if (!PyTuple_Check(ep) || PyTuple_GET_SIZE(ep) != 5) return false;
  e.on = true;
  e.act = (int)PyLong_AsLong(PyTuple_GET_ITEM(ep, 1));
  auto operand = [&](PyObject* o, int64_t rows, const void** p, int64_t* ld) {      // rows of out_f values (0: any number), *ld apart
    if (o == Py_None) return true;
    const at::Tensor* t = tensor(o);
    if (!t || !t->is_cuda() || t->scalar_type() != x.scalar_type() || t->device() != x.device() || t->numel() == 0) return false;
    if (rows ? t->numel() != rows * out_f : t->numel() % out_f != 0) return false;
    *ld = out_f;
    if (!t->is_contiguous()) {                     // whole rows of a wider matrix (a chunk of the modulation's columns)
      if (t->dim() != 2 || t->size(1) != out_f || t->stride(1) != 1 || t->stride(0) < out_f) return false;
      *ld = t->stride(0);
    }
    *p = t->data_ptr();
    return true;
  };
  int64_t ld_bias = 0;
  if (!operand(PyTuple_GET_ITEM(ep, 0), 1, &e.bias, &ld_bias) || !operand(PyTuple_GET_ITEM(ep, 2), 0, &e.gate, &e.ld_gate) ||
      !operand(PyTuple_GET_ITEM(ep, 4), M, &e.resid, &e.ld_resid)) return false;
  if (e.gate) {                                    // a row of it for every gate_rows rows of the result, the last ones too
    e.gate_rows = (int)PyLong_AsLong(PyTuple_GET_ITEM(ep, 3));
    if (e.gate_rows < 1 || tensor(PyTuple_GET_ITEM(ep, 2))->numel() / out_f * e.gate_rows < M) return false;
  }
  return !PyErr_Occurred();
}

at::Tensor empty(const at::Tensor& x, at::IntArrayRef sizes) {
  return at::Tensor(at::detail::empty_cuda(sizes, x.scalar_type(), x.device(), std::nullopt));
}
// (leading sizes of x.., columns), or (M, columns)
at::Tensor result(const at::Tensor& x, bool lead, int64_t M, int64_t columns) {
  if (!lead || x.dim() == 2) return empty(x, {M, columns});
  c10::SmallVector<int64_t, 6> s(x.sizes().begin(), x.sizes().end());
  s.back() = columns;
  return empty(x, s);
}

// The record that get_*_config() hands out: made anew only when something about the call changed.
struct Record {
  PyObject* made = nullptr;                        // the dict in `rec` that these values describe (held, so that its address stays its own)
  int64_t v[8] = {};
};
std::map<std::pair<PyObject*, PyObject*>, Record> records;
bool record(PyObject* rec, PyObject* name, const at::Tensor& x, const char* const* keys, const int64_t* v, int n, bool dtype) {
  Record& r = records[{rec, name}];
  bool same = r.made && PyDict_GetItem(rec, name) == r.made;
  for (int i = 0; same && i < n; ++i) same = r.v[i] == v[i];
  const int64_t t = (int64_t)x.scalar_type();
  if (same && r.v[7] == t) return true;
  PyObject* d = PyDict_New();
  if (!d) return false;
  auto put = [&](const char* k, PyObject* o) { const bool ok = o && PyDict_SetItemString(d, k, o) == 0; Py_XDECREF(o); return ok; };
  bool ok = put("kernel", PyUnicode_FromString("libblr"));
  for (int i = 0; ok && i < n; ++i) ok = put(keys[i], PyLong_FromLongLong(v[i]));
  if (ok && dtype) ok = put("dtype", PyUnicode_FromString(x.scalar_type() == at::kHalf ? "torch.float16" : x.scalar_type() == at::kBFloat16 ? "torch.bfloat16" : "torch.float32"));
  ok = ok && PyDict_SetItem(rec, name, d) == 0;
  Py_XDECREF(r.made);
  r.made = ok ? d : nullptr;
  for (int i = 0; i < n; ++i) r.v[i] = v[i];
  r.v[7] = t;
  if (!ok) Py_DECREF(d);
  return ok;
}

PyObject* failed(PyObject* name, int rc) {
  PyErr_Format(blr_error ? blr_error : PyExc_RuntimeError, "%U failed (%d): %s", name, rc, api.last_error());
  return nullptr;
}

bool streams(int algo, int64_t M, int dt) { return algo == BLR_ALGO_STREAM || algo == BLR_ALGO_STREAM_SPLIT || (algo == BLR_ALGO_AUTO && M <= 16 && dt != BLR_F32); }

// (held over the launches, which run without the interpreter lock: another thread's call on the stream may replace the workspace; that
// the launches of two calls do not interleave in one is the C entry points' part)
struct Ws { void* p; size_t n; void* stream; at::Tensor held; };
Ws find_ws(const at::Tensor& x, size_t need, bool streaming) {
  void* st = (void*)c10::hip::getCurrentHIPStream(x.device().index()).stream();
  const at::Tensor& ws = workspace(x.device(), st, need, streaming);
  return {ws.data_ptr(), (size_t)ws.numel(), st, ws};
}

#define INT(k) ((int)PyLong_AsLong(args[k]))
#define ENTER(n)                                                                             \
  if (nargs != (n)) { PyErr_SetString(PyExc_TypeError, "wrong number of arguments"); return nullptr; } \
  HANDLE_TH_ERRORS
#define DECLINE do { PyErr_Clear(); Py_RETURN_NONE; } while (0)

// blast(name, rec, x, U, V, S, u_layout, s_layout, algo, want, ep): the result, or (out, z, y) with want
PyObject* blast(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  ENTER(11)
  const at::Tensor *x = tensor(args[2]), *U = tensor(args[3]), *V = tensor(args[4]), *S = tensor(args[5]);
  const int ul = INT(6), sl = INT(7), want = INT(9);
  int algo = INT(8);
  if (!x || !weight(U, *x, 3) || !weight(V, *x, 3) || !weight(S, *x, 3)) DECLINE;
  const int dt = dtype_code(x->scalar_type());
  const int64_t b = V->size(0), p = V->size(1), r = V->size(2);
  const int64_t q = ul == BLR_U_RQ ? U->size(2) : U->size(1), ur = ul == BLR_U_RQ ? U->size(1) : U->size(2);
  if (dt < 0 || (dt == BLR_F32) != (want != 0) || b < 2 || U->size(0) != b || ur != r) DECLINE;   // (the *_fp32 names return the intermediates)
  if (sl == BLR_S_JIR ? S->size(0) != b || S->size(1) != b || S->size(2) != r : S->size(0) != r || S->size(1) != b || S->size(2) != b) DECLINE;
  Rows R;
  Ep e;
  const int64_t in = b * p, out_f = b * q;
  if (!rows_of(*x, in, R) || !epilogue(want ? Py_None : args[10], *x, R.M, out_f, e)) DECLINE;
  if (want) algo = BLR_ALGO_TILED;
  const int M = (int)R.M;
  const int64_t cols = e.on && e.act == BLR_ACT_SILU_MUL ? out_f / 2 : out_f;
  at::Tensor out = result(*x, true, M, cols), z, y;
  if (want) { z = empty(*x, {b, M, r}); y = empty(*x, {b, M, r}); }
  size_t need = api.blast_ws(M, (int)in, (int)out_f, (int)b, (int)r, dt, algo);
  if (e.on) need += api.ep_ws(BLR_OP_BLAST, M, (int)out_f, (int)b, dt, e.act);
  const Ws w = find_ws(*x, need, streams(algo, M, dt));
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (e.on)
    rc = api.blast_ep(x->data_ptr(), R.ld, U->data_ptr(), V->data_ptr(), S->data_ptr(), out.data_ptr(), cols, M, (int)in, (int)out_f, (int)b, (int)r, dt, ul, sl,
                      algo, w.p, w.n, w.stream, e.bias, e.act, e.gate, e.gate_rows, e.ld_gate, e.resid, e.ld_resid);
  else
    rc = api.blast(x->data_ptr(), R.ld, U->data_ptr(), V->data_ptr(), S->data_ptr(), out.data_ptr(), out_f, want ? z.data_ptr() : nullptr, want ? y.data_ptr() : nullptr,
                   M, (int)in, (int)out_f, (int)b, (int)r, dt, ul, sl, algo, w.p, w.n, w.stream);
  Py_END_ALLOW_THREADS
  if (rc) return failed(args[0], rc);
  static const char* const keys[] = {"M", "in_f", "out_f", "b", "rank", "algo"};
  const int64_t v[] = {M, in, out_f, b, r, algo};
  if (!record(args[1], args[0], *x, keys, v, 6, true)) return nullptr;
  if (!want) return THPVariable_Wrap(std::move(out));
  return Py_BuildValue("NNN", THPVariable_Wrap(std::move(out)), THPVariable_Wrap(std::move(z)), THPVariable_Wrap(std::move(y)));
  END_HANDLE_TH_ERRORS
}

// blast_q(name, rec, x, U, V, S, algo, ep): U and V are QuantFactors (codes, scales, bits, shape)
PyObject* blast_q(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  ENTER(8)
  const at::Tensor *x = tensor(args[2]), *S = tensor(args[5]);
  const int algo = INT(6);
  if (!x || !weight(S, *x, 3) || !PyTuple_Check(args[3]) || !PyTuple_Check(args[4]) || PyTuple_GET_SIZE(args[3]) != 4 || PyTuple_GET_SIZE(args[4]) != 4) DECLINE;
  const at::Tensor *uc = tensor(PyTuple_GET_ITEM(args[3], 0)), *us = tensor(PyTuple_GET_ITEM(args[3], 1));
  const at::Tensor *vc = tensor(PyTuple_GET_ITEM(args[4], 0)), *vs = tensor(PyTuple_GET_ITEM(args[4], 1));
  const long bits = PyLong_AsLong(PyTuple_GET_ITEM(args[3], 2));
  const int dt = dtype_code(x->scalar_type());
  if (!uc || !us || !vc || !vs || PyLong_AsLong(PyTuple_GET_ITEM(args[4], 2)) != bits || (bits != 8 && bits != 4) || (dt != BLR_F16 && dt != BLR_BF16)) DECLINE;
  for (const at::Tensor* t : {uc, us, vc, vs})
    if (!t->is_cuda() || t->device() != x->device() || !t->is_contiguous()) DECLINE;
  if (us->scalar_type() != at::kHalf || vs->scalar_type() != at::kHalf || uc->dim() != 3 || vc->dim() != 3 || us->dim() != 2 || vs->dim() != 2) DECLINE;
  // U codes (b, r, q[/2]) + scales (b, q), V codes (b, p, r[/2]) + scales (b, r); S (r, b, b)
  const int64_t b = vs->size(0), r = vs->size(1), q = us->size(1), p = vc->size(1), in = b * p, out_f = b * q;
  if (b < 2 || us->size(0) != b || uc->size(0) != b || vc->size(0) != b || uc->size(1) != r || uc->size(2) * 8 != q * bits || vc->size(2) * 8 != r * bits) DECLINE;
  if (uc->element_size() != 1 || vc->element_size() != 1 || S->size(0) != r || S->size(1) != b || S->size(2) != b) DECLINE;
  // the module adds a bias that this one cannot take with torch, where it may be trained
  if (args[7] != Py_None && PyTuple_Check(args[7]) && PyTuple_GET_SIZE(args[7]) == 5 && PyTuple_GET_ITEM(args[7], 0) != Py_None) {
    const at::Tensor* bias = tensor(PyTuple_GET_ITEM(args[7], 0));
    if (!bias || !plain(*bias)) DECLINE;
  }
  Rows R;
  Ep e;
  if (!rows_of(*x, in, R) || !epilogue(args[7], *x, R.M, out_f, e)) DECLINE;
  const int M = (int)R.M;
  const int64_t cols = e.on && e.act == BLR_ACT_SILU_MUL ? out_f / 2 : out_f;
  at::Tensor out = result(*x, true, M, cols);
  size_t need = api.q_ws(M, (int)in, (int)out_f, (int)b, (int)r, (int)bits);
  if (e.on) need += api.ep_ws(BLR_OP_BLAST, M, (int)out_f, (int)b, dt, e.act);
  const Ws w = find_ws(*x, need, M <= 16);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (e.on)
    rc = api.q_ep(x->data_ptr(), R.ld, uc->data_ptr(), us->data_ptr(), vc->data_ptr(), vs->data_ptr(), S->data_ptr(), out.data_ptr(), cols, M, (int)in, (int)out_f,
                  (int)b, (int)r, dt, (int)bits, algo, w.p, w.n, w.stream, e.bias, e.act, e.gate, e.gate_rows, e.ld_gate, e.resid, e.ld_resid);
  else
    rc = api.q(x->data_ptr(), R.ld, uc->data_ptr(), us->data_ptr(), vc->data_ptr(), vs->data_ptr(), S->data_ptr(), out.data_ptr(), out_f, M, (int)in, (int)out_f,
               (int)b, (int)r, dt, (int)bits, algo, w.p, w.n, w.stream);
  Py_END_ALLOW_THREADS
  if (rc) return failed(args[0], rc);
  static const char* const keys[] = {"M", "in_f", "out_f", "b", "rank", "bits"};
  const int64_t v[] = {M, in, out_f, b, r, bits};
  static PyObject* slot = PyUnicode_InternFromString("q");
  if (!record(args[1], slot, *x, keys, v, 6, false)) return nullptr;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// monarch(name, rec, x, w1, w2, w2_layout, out_order, algo, want, ep): the result, or (out, out1) with want
PyObject* monarch(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  ENTER(10)
  const at::Tensor *x = tensor(args[2]), *w1 = tensor(args[3]), *w2 = tensor(args[4]);
  const int layout = INT(5), order = INT(6), want = INT(8);
  int algo = INT(7);
  if (!x || !weight(w1, *x, 3) || !weight(w2, *x, 3)) DECLINE;
  const int dt = dtype_code(x->scalar_type());
  const int64_t k = w1->size(0), p = w1->size(1), r = w1->size(2), s = layout == BLR_W2_SR ? w2->size(1) : w2->size(2), in = k * p, out_f = k * s;
  if (dt < 0 || (dt == BLR_F32) != (want != 0) || w2->size(0) != k || (layout == BLR_W2_SR ? w2->size(2) : w2->size(1)) != r) DECLINE;
  Rows R;
  Ep e;
  if (!rows_of(*x, in, R) || !epilogue(want ? Py_None : args[9], *x, R.M, out_f, e)) DECLINE;
  if (want) algo = BLR_ALGO_TILED;
  const int M = (int)R.M;
  const int64_t cols = e.on && e.act == BLR_ACT_SILU_MUL ? out_f / 2 : out_f;
  at::Tensor out = result(*x, true, M, cols), out1;
  if (want) out1 = empty(*x, {k, M, r});
  size_t need = api.monarch_ws(M, (int)in, (int)out_f, (int)k, (int)r, dt, algo);
  if (e.on) need += api.ep_ws(BLR_OP_MONARCH, M, (int)out_f, (int)k, dt, e.act);
  const Ws w = find_ws(*x, need, streams(algo, M, dt));
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (e.on)
    rc = api.monarch_ep(x->data_ptr(), R.ld, w1->data_ptr(), w2->data_ptr(), out.data_ptr(), cols, M, (int)in, (int)out_f, (int)k, (int)r, dt, layout, order, algo,
                        w.p, w.n, w.stream, e.bias, e.act, e.gate, e.gate_rows, e.ld_gate, e.resid, e.ld_resid);
  else
    rc = api.monarch(x->data_ptr(), R.ld, w1->data_ptr(), w2->data_ptr(), out.data_ptr(), out_f, want ? out1.data_ptr() : nullptr, M, (int)in, (int)out_f, (int)k, (int)r,
                     dt, layout, order, algo, w.p, w.n, w.stream);
  Py_END_ALLOW_THREADS
  if (rc) return failed(args[0], rc);
  static const char* const keys[] = {"M", "in_f", "out_f", "b", "rank", "algo"};
  const int64_t v[] = {M, in, out_f, k, r, algo};
  if (!record(args[1], args[0], *x, keys, v, 6, false)) return nullptr;
  if (!want) return THPVariable_Wrap(std::move(out));
  return Py_BuildValue("NN", THPVariable_Wrap(std::move(out)), THPVariable_Wrap(std::move(out1)));
  END_HANDLE_TH_ERRORS
}

// low_rank(name, rec, x, a, b, algo, want, lead, ep): (N, out), with lead (.., out); (out, z) with want
PyObject* low_rank(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  ENTER(9)
  const at::Tensor *x = tensor(args[2]), *a = tensor(args[3]), *b = tensor(args[4]);
  const int algo = INT(5), want = INT(6), lead = INT(7);
  if (!x || !weight(a, *x, 2) || !weight(b, *x, 2)) DECLINE;
  const int dt = dtype_code(x->scalar_type());
  const int64_t in = a->size(0), r = a->size(1), out_f = b->size(1);
  Rows R;
  Ep e;
  if (dt < 0 || (dt == BLR_F32) != (want != 0) || b->size(0) != r || !rows_of(*x, in, R) || !epilogue(want ? Py_None : args[8], *x, R.M, out_f, e)) DECLINE;
  const int M = (int)R.M;
  const int64_t cols = e.on && e.act == BLR_ACT_SILU_MUL ? out_f / 2 : out_f;
  at::Tensor out = result(*x, lead, M, cols), z;
  if (want) z = empty(*x, {M, r});
  size_t need = api.low_rank_ws(M, (int)in, (int)out_f, (int)r, dt, algo);
  if (e.on) need += api.ep_ws(BLR_OP_LOW_RANK, M, (int)out_f, 1, dt, e.act);
  const Ws w = find_ws(*x, need, streams(algo, M, dt));
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (e.on)
    rc = api.low_rank_ep(x->data_ptr(), R.ld, a->data_ptr(), b->data_ptr(), out.data_ptr(), cols, M, (int)in, (int)out_f, (int)r, dt, algo, w.p, w.n, w.stream,
                         e.bias, e.act, e.gate, e.gate_rows, e.ld_gate, e.resid, e.ld_resid);
  else
    rc = api.low_rank(x->data_ptr(), R.ld, a->data_ptr(), b->data_ptr(), out.data_ptr(), out_f, want ? z.data_ptr() : nullptr, M, (int)in, (int)out_f, (int)r, dt, algo,
                      w.p, w.n, w.stream);
  Py_END_ALLOW_THREADS
  if (rc) return failed(args[0], rc);
  static const char* const keys[] = {"M", "in_f", "out_f", "rank", "algo"};
  const int64_t v[] = {M, in, out_f, r, algo};
  if (!record(args[1], args[0], *x, keys, v, 5, false)) return nullptr;
  if (!want) return THPVariable_Wrap(std::move(out));
  return Py_BuildValue("NN", THPVariable_Wrap(std::move(out)), THPVariable_Wrap(std::move(z)));
  END_HANDLE_TH_ERRORS
}

// dense(name, rec, x, w, algo, f32, lead, ep): (N, out), with lead (.., out); f32: the float32 name
PyObject* dense(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  ENTER(8)
  const at::Tensor *x = tensor(args[2]), *W = tensor(args[3]);
  const int algo = INT(4), f32 = INT(5), lead = INT(6);
  if (!x || !weight(W, *x, 2)) DECLINE;
  const int dt = dtype_code(x->scalar_type());
  const int64_t in = W->size(0), out_f = W->size(1);
  Rows R;
  Ep e;
  if (dt < 0 || (dt == BLR_F32) != (f32 != 0) || !rows_of(*x, in, R) || !epilogue(args[7], *x, R.M, out_f, e)) DECLINE;
  const int M = (int)R.M;
  const int64_t cols = e.on && e.act == BLR_ACT_SILU_MUL ? out_f / 2 : out_f;
  at::Tensor out = result(*x, lead, M, cols);
  size_t need = api.dense_ws(M, (int)in, (int)out_f, dt, algo);
  if (e.on) need += api.ep_ws(BLR_OP_DENSE, M, (int)out_f, 1, dt, e.act);
  const Ws w = find_ws(*x, need, streams(algo, M, dt));
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (e.on)
    rc = api.dense_ep(x->data_ptr(), R.ld, W->data_ptr(), out.data_ptr(), cols, M, (int)in, (int)out_f, dt, algo, w.p, w.n, w.stream, e.bias, e.act, e.gate, e.gate_rows,
                      e.ld_gate, e.resid, e.ld_resid);
  else
    rc = api.dense(x->data_ptr(), R.ld, W->data_ptr(), out.data_ptr(), out_f, M, (int)in, (int)out_f, dt, algo, w.p, w.n, w.stream);
  Py_END_ALLOW_THREADS
  if (rc) return failed(args[0], rc);
  static const char* const keys[] = {"M", "in_f", "out_f", "algo"};
  const int64_t v[] = {M, in, out_f, algo};
  if (!record(args[1], args[0], *x, keys, v, 4, false)) return nullptr;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// The entries below stand in for torch operators, which autograd, autocast, transforms and dispatch modes see: a call that any of
// those has a part in is left to torch.
bool torch_modes_off() {
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  return (tls.included_ - c10::default_included_set).empty() && !at::autocast::is_autocast_enabled(at::kCUDA);
}
bool aligned16(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// ln_modulate(x, shift, scale, eps): x (images, tokens, columns), shift and scale (images, columns) or column chunks of a wider matrix
PyObject* ln_modulate(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  ENTER(4)
  const at::Tensor *x = tensor(args[0]), *sh = tensor(args[1]), *sc = tensor(args[2]);
  const double eps = PyFloat_AsDouble(args[3]);
  if (PyErr_Occurred() || !x || !sh || !sc || !torch_modes_off() || !plain(*x) || !plain(*sh) || !plain(*sc)) DECLINE;
  const int dt = dtype_code(x->scalar_type());
  if ((dt != BLR_F16 && dt != BLR_BF16) || x->dim() != 3 || x->numel() == 0 || !x->is_contiguous() || !aligned16(*x)) DECLINE;
  const int64_t B = x->size(0), N = x->size(1), C = x->size(2);
  if (C % 8 || C > 2048 || B * N > INT32_MAX) DECLINE;
  for (const at::Tensor* t : {sh, sc})
    if (t->scalar_type() != x->scalar_type() || t->device() != x->device() || t->dim() != 2 || t->size(0) != B || t->size(1) != C || t->stride(1) != 1 ||
        t->stride(0) < C || t->stride(0) % 8 || !aligned16(*t)) DECLINE;
  const c10::OptionalDeviceGuard guard(x->device());
  at::Tensor out = empty(*x, {B, N, C});
  const void *xp = x->data_ptr(), *shp = sh->data_ptr(), *scp = sc->data_ptr();
  const int64_t lsh = sh->stride(0), lsc = sc->stride(0);
  void* st = (void*)c10::hip::getCurrentHIPStream(x->device().index()).stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.ln_modulate(xp, shp, lsh, scp, lsc, out.data_ptr(), (int)(B * N), (int)C, (int)N, (float)eps, dt, st);
  Py_END_ALLOW_THREADS
  static PyObject* const name = PyUnicode_InternFromString("ln_modulate");
  if (rc) return failed(name, rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// attention(qkv, heads): qkv (images, tokens, 3 * columns) as the qkv linear leaves it; (images, tokens, columns)
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  ENTER(2)
  const at::Tensor* x = tensor(args[0]);
  const int64_t H = PyLong_AsLong(args[1]);
  if (PyErr_Occurred() || !x || H < 1 || !torch_modes_off() || !plain(*x)) DECLINE;
  // (a kernel of the flash kind: a caller that has those switched off, sdpa_kernel(MATH) for one, wants another one's arithmetic)
  if (!at::globalContext().userEnabledFlashSDP()) DECLINE;
  const int dt = dtype_code(x->scalar_type());
  if ((dt != BLR_F16 && dt != BLR_BF16) || x->dim() != 3 || x->numel() == 0 || !x->is_contiguous() || !aligned16(*x) || x->size(2) % (3 * H)) DECLINE;
  const int64_t B = x->size(0), N = x->size(1), D = x->size(2) / (3 * H);
  if ((D != 64 && D != 72) || N > (1 << 20) || B * H > INT32_MAX / ((N + 127) / 128)) DECLINE;
  const c10::OptionalDeviceGuard guard(x->device());
  at::Tensor out = empty(*x, {B, N, H * D});
  const void* xp = x->data_ptr();
  void* st = (void*)c10::hip::getCurrentHIPStream(x->device().index()).stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.attention(xp, out.data_ptr(), (int)B, (int)N, (int)H, (int)D, dt, st);
  Py_END_ALLOW_THREADS
  static PyObject* const name = PyUnicode_InternFromString("attention");
  if (rc) return failed(name, rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// silu_linear(c, weight, bias): c (rows, in), weight (out, in) and bias (out) or None as an nn.Linear holds them
PyObject* silu_linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  ENTER(3)
  const at::Tensor *c = tensor(args[0]), *W = tensor(args[1]), *b = args[2] == Py_None ? nullptr : tensor(args[2]);
  if (!c || !W || (!b && args[2] != Py_None) || !torch_modes_off() || !plain(*c) || !plain(*W) || (b && !plain(*b))) DECLINE;
  const int dt = dtype_code(c->scalar_type());
  if ((dt != BLR_F16 && dt != BLR_BF16) || c->dim() != 2 || !weight(W, *c, 2) || (b && !weight(b, *c, 1))) DECLINE;
  const int64_t M = c->size(0), K = c->size(1), N = W->size(0);
  if (M < 1 || M > 16 || K < 8 || K % 8 || K > INT32_MAX || N < 4 || N % 4 || N > INT32_MAX - 16 || W->size(1) != K || (b && b->numel() != N)) DECLINE;
  if (c->stride(1) != 1 || (M > 1 && (c->stride(0) < K || c->stride(0) % 8)) || !aligned16(*c) || !aligned16(*W)) DECLINE;
  const c10::OptionalDeviceGuard guard(c->device());
  at::Tensor out = empty(*c, {M, N});
  const void *cp = c->data_ptr(), *wp = W->data_ptr(), *bp = b ? b->data_ptr() : nullptr;
  const int64_t ld = M > 1 ? c->stride(0) : K;
  void* st = (void*)c10::hip::getCurrentHIPStream(c->device().index()).stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.silu_linear(cp, ld, wp, bp, out.data_ptr(), (int)M, (int)N, (int)K, dt, st);
  Py_END_ALLOW_THREADS
  static PyObject* const name = PyUnicode_InternFromString("silu_linear");
  if (rc) return failed(name, rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// workspace(device index, stream, bytes, streaming)
PyObject* py_workspace(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  ENTER(4)
  const int dev = INT(0), streaming = INT(3);
  void* st = PyLong_AsVoidPtr(args[1]);
  const size_t bytes = PyLong_AsSize_t(args[2]);
  if (PyErr_Occurred()) return nullptr;
  return THPVariable_Wrap(workspace(at::Device(at::kCUDA, (c10::DeviceIndex)dev), st, bytes, streaming != 0));
  END_HANDLE_TH_ERRORS
}

// bind(addresses by name, BlrError)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  ENTER(2)
  auto get = [&](const char* n, auto& f) {
    PyObject* o = PyDict_GetItemString(args[0], n);
    void* p = o ? PyLong_AsVoidPtr(o) : nullptr;
    f = reinterpret_cast<std::decay_t<decltype(f)>>(p);
    return p != nullptr;
  };
  const bool ok = get("blr_blast_workspace_bytes", api.blast_ws) && get("blr_blast_fwd", api.blast) && get("blr_blast_fwd_ep2", api.blast_ep) &&
                  get("blr_blast_q_workspace_bytes", api.q_ws) && get("blr_blast_q_fwd", api.q) && get("blr_blast_q_fwd_ep2", api.q_ep) &&
                  get("blr_monarch_workspace_bytes", api.monarch_ws) && get("blr_monarch_fwd", api.monarch) && get("blr_monarch_fwd_ep2", api.monarch_ep) &&
                  get("blr_low_rank_workspace_bytes", api.low_rank_ws) && get("blr_low_rank_fwd", api.low_rank) && get("blr_low_rank_fwd_ep2", api.low_rank_ep) &&
                  get("blr_dense_workspace_bytes", api.dense_ws) && get("blr_dense_fwd", api.dense) && get("blr_dense_fwd_ep2", api.dense_ep) &&
                  get("blr_ep_workspace_bytes", api.ep_ws) && get("blr_ln_modulate", api.ln_modulate) &&
                  get("blr_attention_qkv", api.attention) && get("blr_silu_linear", api.silu_linear) && get("blr_last_error", api.last_error);
  if (!ok) { PyErr_SetString(PyExc_ValueError, "an entry point of libblr.so is missing"); return nullptr; }
  Py_INCREF(args[1]);
  Py_XDECREF(blr_error);
  blr_error = args[1];
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void*)bind, METH_FASTCALL, nullptr},
    {"workspace", (PyCFunction)(void*)py_workspace, METH_FASTCALL, nullptr},
    {"blast", (PyCFunction)(void*)blast, METH_FASTCALL, nullptr},
    {"blast_q", (PyCFunction)(void*)blast_q, METH_FASTCALL, nullptr},
    {"monarch", (PyCFunction)(void*)monarch, METH_FASTCALL, nullptr},
    {"low_rank", (PyCFunction)(void*)low_rank, METH_FASTCALL, nullptr},
    {"ln_modulate", (PyCFunction)(void*)ln_modulate, METH_FASTCALL, nullptr},
    {"attention", (PyCFunction)(void*)attention, METH_FASTCALL, nullptr},
    {"silu_linear", (PyCFunction)(void*)silu_linear, METH_FASTCALL, nullptr},
    {"dense", (PyCFunction)(void*)dense, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_blr_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__blr_host() { return PyModule_Create(&module); }
