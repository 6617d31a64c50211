// Native argument checks and calls for the kernel wrappers (infurnace_amd/kernels).
//
// A wrapper's checks and its ctypes call take 15-25 us of Python per call, more than most decode
// launches.  Each function here makes the wrapper's checks on plain torch tensors and calls the same C
// entry point.  It handles exactly the calls the checked Python path accepts in its common form and
// returns None for everything else -- an argument that is no plain contiguous torch tensor, a value out
// of range, a plan for other tensors, a workspace to grow, a call the entry point refuses -- before the
// entry point launches anything (an output cleared for a call that is then refused is dropped); the wrapper
// then takes the Python path, which raises or handles it.  A launch that failed is raised here, not made
// again.  Nothing is kept between calls but the entry points' addresses.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstdint>
#include <string>
#include <type_traits>

#include "../../include/infurnace_amd.h"

namespace {

// The C entry points of the loaded library, by address (bind()).
#define IFN_ENTRIES(X) \
  X(store_kv, ifn_store_kv) X(store_kv_layers, ifn_store_kv_layers) \
  X(decode_ws, ifn_paged_decode_workspace_bytes) X(plan_bytes, ifn_paged_decode_plan_bytes) \
  X(decode, ifn_paged_decode) X(decode_append, ifn_paged_decode_append) \
  X(decode_planned, ifn_paged_decode_planned) X(decode_append_planned, ifn_paged_decode_append_planned) \
  X(decode_planning, ifn_paged_decode_planning) X(decode_append_planning, ifn_paged_decode_append_planning) \
  X(shared_ws, ifn_paged_decode_shared_prefix_workspace_bytes) X(shared, ifn_paged_decode_shared_prefix) \
  X(prefill_ws, ifn_paged_prefill_workspace_bytes) X(prefill, ifn_paged_prefill) \
  X(prefill_append, ifn_paged_prefill_append) X(prep_append, ifn_qk_norm_rope_append) \
  X(prep_decode, ifn_paged_decode_prep_append) X(prep_decode_planning, ifn_paged_decode_prep_append_planning) \
  X(prep_prefill, ifn_paged_prefill_prep_append)
struct Entries {
#define IFN_MEMBER(name, fn) decltype(&fn) name;
  IFN_ENTRIES(IFN_MEMBER)
#undef IFN_MEMBER
};
Entries E{};
bool bound = false;

struct NotPlain {};  // the call goes to the Python path
struct Raised {};    // a Python error is set: it goes to the caller

inline void need(bool ok) {
  if (!ok) throw NotPlain{};
}

// A plain contiguous GPU tensor of this type and device (dev < 0: any).
const at::Tensor& tensor(PyObject* o, at::ScalarType type, int dev = -1) {
  need(THPVariable_CheckExact(o));
  const at::Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet odd({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                     c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::Functionalize,
                                     c10::DispatchKey::Python, c10::DispatchKey::Negative,
                                     c10::DispatchKey::Conjugate, c10::DispatchKey::ZeroTensor});
  need(t.defined() && t.scalar_type() == type && t.is_cuda() && t.layout() == at::kStrided &&
       !t.key_set().has_any(odd) && t.is_contiguous() && (dev < 0 || t.get_device() == dev));
  return t;
}

template <class... D>
const at::Tensor& shaped(PyObject* o, at::ScalarType type, int dev, D... dims) {
  const at::Tensor& t = tensor(o, type, dev);
  const int64_t want[] = {int64_t(dims)...};
  need(t.dim() == int64_t(sizeof...(D)));
  for (size_t i = 0; i < sizeof...(D); ++i) need(t.size(int64_t(i)) == want[i]);
  return t;
}

// A bool or uint8 mask of n elements, or null for None.
const uint8_t* mask(PyObject* o, int dev, int64_t n) {
  if (o == Py_None) return nullptr;
  need(THPVariable_CheckExact(o));
  const at::ScalarType s = THPVariable_Unpack(o).scalar_type();
  need(s == at::kBool || s == at::kByte);
  return static_cast<const uint8_t*>(shaped(o, s, dev, n).data_ptr());
}

int64_t integer(PyObject* o) {
  need(PyLong_CheckExact(o));
  int over = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &over);
  need(over == 0 && v >= INT32_MIN && v <= INT32_MAX);
  return v;
}

double real(PyObject* o) {
  need(PyFloat_CheckExact(o));
  return PyFloat_AS_DOUBLE(o);
}

const float* f32(PyObject* o, int dev, int64_t a) { return static_cast<const float*>(shaped(o, at::kFloat, dev, a).data_ptr()); }
const float* f32(PyObject* o, int dev, int64_t a, int64_t b, int64_t c) {
  return static_cast<const float*>(shaped(o, at::kFloat, dev, a, b, c).data_ptr());
}
const int32_t* i32(PyObject* o, int dev, int64_t n) { return static_cast<const int32_t*>(shaped(o, at::kInt, dev, n).data_ptr()); }

int32_t small(int64_t v) {
  need(v >= 0 && v <= INT32_MAX);
  return int32_t(v);
}

struct Pool {  // one layer of the pool (check_pool)
  char* p;
  int64_t pages;
  int32_t bs, hkv, d;
  int dev;
  int64_t layers;
};

Pool pool(PyObject* o, int64_t layer) {
  const at::Tensor& t = tensor(o, at::kHalf);
  need(t.dim() == 5 || t.dim() == 6);
  const int64_t k = t.dim() - 5;  // dims before [2, P, bs, Hkv, D]
  for (int64_t i = 0; i < t.dim(); ++i) need(t.size(i) >= 1);
  need(t.size(k) == 2 && layer >= 0 && layer < (k == 1 ? t.size(0) : 1));
  Pool r;
  r.layers = k == 1 ? t.size(0) : 1;
  r.pages = t.size(k + 1);
  r.bs = small(t.size(k + 2));
  r.hkv = small(t.size(k + 3));
  r.d = small(t.size(k + 4));
  r.dev = t.get_device();
  r.p = static_cast<char*>(t.data_ptr()) + layer * 2 * r.pages * r.bs * r.hkv * r.d * 2;
  return r;
}

float scale_of(PyObject* o, int32_t d) {  // None: 1 / sqrt(d)
  const double s = o == Py_None ? 1.0 / std::sqrt(double(d)) : real(o);
  need(s > 0);
  return float(s);
}

float eps_of(PyObject* o) {
  const double e = real(o);
  need(e >= 0 && std::isfinite(e));
  return float(e);
}

// Work on the device runs without the GIL: a launch (or an output's fill) can wait for room in the stream's
// queue, an allocation for the device, and other threads run meanwhile, as they do in a ctypes or torch call.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};
template <class F>
auto unlocked(F f) {
  const NoGil released;
  return f();
}
template <class F, class... A>
int launch(F fn, A... args) {
  return unlocked([&] { return fn(args...); });
}

// The fp16 output [n, hq, d]: the caller's, or a new one (cleared when rows may be inactive).
at::Tensor output(PyObject* o, const Pool& P, int64_t n, int64_t hq, bool clear) {
  if (o != Py_None) return shaped(o, at::kHalf, P.dev, n, hq, P.d);
  const auto opt = at::TensorOptions().dtype(at::kHalf).device(at::kCUDA, P.dev);
  return unlocked([&] { return clear ? at::zeros({n, hq, P.d}, opt) : at::empty({n, hq, P.d}, opt); });
}

struct Call {  // the stream and its workspace
  void* stream;
  void* ws;
  size_t bytes;
  at::Tensor held;  // (another thread may replace the workspace during the launch)
};

// An entry point's status.  It refuses a call before it launches anything: that call goes to the Python path.
// IFN_ERR_HIP is a launch that failed, possibly after another one of the same call: _capi.check raises it.
void launched(int rc, const char* name) {
  need(rc == IFN_OK || rc == IFN_ERR_HIP);
  if (rc == IFN_OK) return;
  PyObject* capi = PyImport_ImportModule("infurnace_amd._capi");
  PyObject* r = capi == nullptr ? nullptr : PyObject_CallMethod(capi, "check", "si", name, rc);
  Py_XDECREF(r);
  Py_XDECREF(capi);
  if (r != nullptr) PyErr_SetString(PyExc_RuntimeError, name);
  throw Raised{};
}

Call call_on(PyObject* workspaces, int dev, size_t nbytes) {
  Call c;
  c.stream = static_cast<void*>(c10::hip::getCurrentHIPStream(c10::DeviceIndex(dev)).stream());
  PyObject* key = Py_BuildValue("(iL)", dev, (long long)(uintptr_t)c.stream);
  need(key != nullptr);
  PyObject* ws = PyDict_GetItemWithError(workspaces, key);
  Py_DECREF(key);
  need(ws != nullptr);
  const at::Tensor& t = tensor(ws, at::kByte, dev);
  need(size_t(t.numel()) >= nbytes);
  c.ws = t.data_ptr();
  c.bytes = size_t(t.numel());
  c.held = t;
  return c;
}

void* stream_of(int dev) { return static_cast<void*>(c10::hip::getCurrentHIPStream(c10::DeviceIndex(dev)).stream()); }

bool is_int(PyObject* o, int64_t v) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  const long long x = PyLong_AsLongLongAndOverflow(o, &over);
  return over == 0 && x == v;
}
bool is_ptr(PyObject* o, const void* p) { return p == nullptr ? o == Py_None : is_int(o, int64_t(uintptr_t(p))); }
bool is_tuple(PyObject* o, std::initializer_list<int64_t> v) {
  if (!PyTuple_CheckExact(o) || PyTuple_GET_SIZE(o) != Py_ssize_t(v.size())) return false;
  Py_ssize_t i = 0;
  for (int64_t x : v)
    if (!is_int(PyTuple_GET_ITEM(o, i++), x)) return false;
  return true;
}

PyObject *s_buf, *s_nbytes, *s_pending, *s_key, *s_slots;

struct Plan {  // a DecodePlan built from this call's tensors (DecodePlan.ptr_for)
  void* p = nullptr;
  size_t bytes = 0;
  bool pending = false;
  at::Tensor held;
};

PyObject* attr(PyObject* o, PyObject* name) {  // a new reference
  PyObject* r = PyObject_GetAttr(o, name);
  need(r != nullptr);
  return r;
}

Plan plan_of(PyObject* o, const Pool& P, int64_t n, int64_t hq, const at::Tensor& bt, const void* sl, const void* act,
             const void* slots, int64_t msl) {
  Plan r;
  PyObject* key = attr(o, s_key);
  const bool same = PyTuple_CheckExact(key) && PyTuple_GET_SIZE(key) == 9 &&
                    is_tuple(PyTuple_GET_ITEM(key, 0), {n, hq, P.d}) &&
                    (slots == nullptr || is_ptr(PyTuple_GET_ITEM(key, 1), slots)) &&
                    is_tuple(PyTuple_GET_ITEM(key, 2), {2, P.pages, P.bs, P.hkv, P.d}) &&
                    is_ptr(PyTuple_GET_ITEM(key, 3), bt.data_ptr()) &&
                    is_tuple(PyTuple_GET_ITEM(key, 4), {bt.size(0), bt.size(1)}) &&
                    is_ptr(PyTuple_GET_ITEM(key, 5), sl) && is_ptr(PyTuple_GET_ITEM(key, 6), act) &&
                    is_int(PyTuple_GET_ITEM(key, 7), msl) && PyTuple_GET_ITEM(key, 8) == Py_None;
  Py_DECREF(key);
  need(same);
  PyObject* buf = attr(o, s_buf);
  PyObject* nb = PyObject_GetAttr(o, s_nbytes);
  PyObject* pend = PyObject_GetAttr(o, s_pending);
  bool ok = nb != nullptr && pend != nullptr && PyLong_CheckExact(nb) && PyBool_Check(pend);
  if (ok && buf != Py_None) {
    ok = THPVariable_CheckExact(buf);
    if (ok) {
      r.held = THPVariable_Unpack(buf);
      r.p = r.held.data_ptr();
      r.bytes = PyLong_AsSize_t(nb);
    }
  }
  if (ok) r.pending = pend == Py_True;
  Py_XDECREF(nb);
  Py_XDECREF(pend);
  Py_DECREF(buf);
  need(ok);
  return r;
}

void plan_built(PyObject* plan, bool slots) {  // DecodePlan.built of a pending plan
  need(PyObject_SetAttr(plan, s_slots, slots ? Py_True : Py_False) == 0 &&
       PyObject_SetAttr(plan, s_pending, Py_False) == 0);
}

int64_t cap_of(PyObject* msl, int64_t cap) {
  if (msl == Py_None) return cap;
  const int64_t v = std::min(integer(msl), cap);
  need(v >= 0);
  return v;
}

PyObject* done(const at::Tensor& out, PyObject* given) {
  if (given != Py_None) {
    Py_INCREF(given);
    return given;
  }
  return THPVariable_Wrap(out);
}

// decode(query, kv_pool, block_tables, sequence_lengths, active_mask, slot_mapping, new_k, new_v, layer, scale, out,
//        block_size, max_seq_len, plan, shared_prefix_pages, workspaces)
PyObject* decode(PyObject* const* a) {
  const Pool P = pool(a[1], integer(a[8]));
  need(integer(a[11]) == P.bs);
  const at::Tensor& q = tensor(a[0], at::kHalf, P.dev);
  need(q.dim() == 3 && q.size(2) == P.d && q.size(1) % P.hkv == 0 && q.size(0) >= 1 && q.size(1) >= 1);
  const int64_t n = q.size(0), hq = q.size(1);
  const at::Tensor& bt = tensor(a[2], at::kInt, P.dev);
  need(bt.dim() == 2 && bt.size(0) == n && bt.size(1) >= 1);
  const int32_t* sl = i32(a[3], P.dev, n);
  const uint8_t* act = mask(a[4], P.dev, n);
  const bool append = a[5] != Py_None;
  const int32_t* slots = append ? i32(a[5], P.dev, n) : nullptr;
  const void* nk = append ? shaped(a[6], at::kHalf, P.dev, n, P.hkv, P.d).data_ptr() : nullptr;
  const void* nv = append ? shaped(a[7], at::kHalf, P.dev, n, P.hkv, P.d).data_ptr() : nullptr;
  const float scale = scale_of(a[9], P.d);
  const int64_t cap = bt.size(1) * P.bs;
  const int32_t msl = small(cap_of(a[12], cap)), B = small(n), Q = small(hq), mp = small(bt.size(1));
  const int32_t* tab = static_cast<const int32_t*>(bt.data_ptr());
  const bool shared = a[14] != Py_None;
  Plan pl;
  int64_t sp = 0;
  const int32_t* spp = nullptr;
  if (shared) {
    need(!append && a[13] == Py_None);
    const at::Tensor& s = tensor(a[14], at::kInt, P.dev);
    need(s.dim() == 1 && s.size(0) <= mp);
    sp = s.size(0);
    spp = static_cast<const int32_t*>(s.data_ptr());
  } else if (a[13] != Py_None) {
    pl = plan_of(a[13], P, n, hq, bt, sl, act, slots, msl);
  }
  const Call c = call_on(a[15], P.dev, shared ? E.shared_ws(B, Q, P.hkv, P.d, P.bs, int32_t(sp))
                                              : E.decode_ws(B, Q, P.hkv, P.d, P.bs, msl));
  const at::Tensor out = output(a[10], P, n, hq, act != nullptr);
  void* o = out.data_ptr();
  const void* qp = q.data_ptr();
  int rc;
  if (shared)
    rc = launch(E.shared, o, qp, P.p, P.pages, spp, int32_t(sp), tab, mp, sl, act, B, Q, P.hkv, P.d, P.bs, msl, scale,
                c.ws, c.bytes, c.stream);
  else if (append)
    rc = a[13] == Py_None
             ? launch(E.decode_append, o, qp, P.p, P.pages, tab, mp, sl, act, slots, nk, nv, B, Q, P.hkv, P.d, P.bs,
                      msl, scale, c.ws, c.bytes, c.stream)
         : pl.pending ? launch(E.decode_append_planning, o, qp, P.p, P.pages, tab, mp, sl, act, slots, nk, nv, B, Q,
                               P.hkv, P.d, P.bs, msl, scale, pl.p, pl.bytes, c.ws, c.bytes, c.stream)
                      : launch(E.decode_append_planned, o, qp, P.p, P.pages, tab, mp, sl, act, slots, nk, nv, B, Q,
                               P.hkv, P.d, P.bs, msl, scale, pl.p, pl.bytes, c.ws, c.bytes, c.stream);
  else
    rc = a[13] == Py_None ? launch(E.decode, o, qp, P.p, P.pages, tab, mp, sl, act, B, Q, P.hkv, P.d, P.bs, msl,
                                   scale, c.ws, c.bytes, c.stream)
         : pl.pending     ? launch(E.decode_planning, o, qp, P.p, P.pages, tab, mp, sl, act, B, Q, P.hkv, P.d, P.bs,
                                   msl, scale, pl.p, pl.bytes, c.ws, c.bytes, c.stream)
                          : launch(E.decode_planned, o, qp, P.p, P.pages, tab, mp, sl, act, B, Q, P.hkv, P.d, P.bs,
                                   msl, scale, pl.p, pl.bytes, c.ws, c.bytes, c.stream);
  launched(rc, shared ? "ifn_paged_decode_shared_prefix" : append ? "ifn_paged_decode_append" : "ifn_paged_decode");
  if (pl.pending) plan_built(a[13], append);
  return done(out, a[10]);
}

// prep_decode(q, k, v, q_norm_weight, k_norm_weight, rope, positions, slot_mapping, active_mask, kv_pool, block_tables,
//             sequence_lengths, layer, eps, scale, out, block_size, max_seq_len, plan, workspaces)
PyObject* prep_decode(PyObject* const* a) {
  const Pool P = pool(a[9], integer(a[12]));
  need(integer(a[16]) == P.bs);
  const at::Tensor& q = tensor(a[0], at::kFloat, P.dev);
  need(q.dim() == 3 && q.size(2) == P.d && q.size(1) % P.hkv == 0 && q.size(0) >= 1 && q.size(1) >= 1);
  const int64_t n = q.size(0), hq = q.size(1);
  const float* k = f32(a[1], P.dev, n, P.hkv, P.d);
  const float* v = f32(a[2], P.dev, n, P.hkv, P.d);
  const float* qw = f32(a[3], P.dev, P.d);
  const float* kw = f32(a[4], P.dev, P.d);
  const at::Tensor& rope = tensor(a[5], at::kFloat, P.dev);
  need(rope.dim() == 2 && rope.size(1) == P.d);
  const int32_t* pos = i32(a[6], P.dev, n);
  const int32_t* slots = i32(a[7], P.dev, n);
  const uint8_t* act = mask(a[8], P.dev, n);
  const at::Tensor& bt = tensor(a[10], at::kInt, P.dev);
  need(bt.dim() == 2 && bt.size(0) == n && bt.size(1) >= 1);
  const int32_t* sl = i32(a[11], P.dev, n);
  const float eps = eps_of(a[13]), scale = scale_of(a[14], P.d);
  const int32_t msl = small(cap_of(a[17], bt.size(1) * P.bs)), B = small(n), Q = small(hq), mp = small(bt.size(1));
  // What the fused kernel does not take is declined before an output is made: it takes the calls of the whole-row
  // kernel (those that have a plan) with 2 KiB token rows, 16-token pages and head dims up to 128.
  need(P.hkv * P.d == 1024 && P.d <= 128 && P.bs == 16 && E.plan_bytes(B, Q, P.hkv, P.d, P.bs, mp, msl) > 0);
  Plan pl;
  if (a[18] != Py_None) pl = plan_of(a[18], P, n, hq, bt, sl, act, slots, msl);
  const Call c = call_on(a[19], P.dev, E.decode_ws(B, Q, P.hkv, P.d, P.bs, msl));
  const at::Tensor out = output(a[15], P, n, hq, act != nullptr);
  const auto fn = pl.pending ? E.prep_decode_planning : nullptr;
  const float* qp = static_cast<const float*>(q.data_ptr());
  const float* rp = static_cast<const float*>(rope.data_ptr());
  const int32_t* tab = static_cast<const int32_t*>(bt.data_ptr());
  const int32_t maxpos = small(rope.size(0));
  const int rc = fn != nullptr
                     ? launch(fn, out.data_ptr(), qp, k, v, qw, kw, rp, maxpos, pos, slots, P.p, P.pages, tab, mp, sl,
                              act, B, Q, P.hkv, P.d, P.bs, msl, scale, eps, pl.p, pl.bytes, c.ws, c.bytes, c.stream)
                     : launch(E.prep_decode, out.data_ptr(), qp, k, v, qw, kw, rp, maxpos, pos, slots, P.p, P.pages,
                              tab, mp, sl, act, B, Q, P.hkv, P.d, P.bs, msl, scale, eps, pl.p, pl.bytes, c.ws,
                              c.bytes, c.stream);
  launched(rc, "ifn_paged_decode_prep_append");
  if (pl.pending) plan_built(a[18], true);
  return done(out, a[15]);
}

// The block table of one sequence: [max_pages] or [1, max_pages].
const at::Tensor& table_of(PyObject* o, int dev, int64_t& pages) {
  const at::Tensor& t = tensor(o, at::kInt, dev);
  need(t.dim() == 1 || (t.dim() == 2 && t.size(0) == 1));
  pages = t.size(t.dim() - 1);
  return t;
}

// prefill(query, kv_pool, block_table, new_k, new_v, query_start, layer, scale, out, block_size, workspaces)
PyObject* prefill(PyObject* const* a) {
  const Pool P = pool(a[1], integer(a[6]));
  need(integer(a[9]) == P.bs);
  const at::Tensor& q = tensor(a[0], at::kHalf, P.dev);
  need(q.dim() == 3 && q.size(2) == P.d && q.size(1) % P.hkv == 0 && q.size(0) >= 1 && q.size(1) >= 1);
  const int64_t n = q.size(0), hq = q.size(1), start = integer(a[5]);
  int64_t mp;
  const at::Tensor& bt = table_of(a[2], P.dev, mp);
  need(start >= 0 && start + n <= mp * P.bs);
  const bool append = a[3] != Py_None;
  const void* nk = append ? shaped(a[3], at::kHalf, P.dev, n, P.hkv, P.d).data_ptr() : nullptr;
  const void* nv = append ? shaped(a[4], at::kHalf, P.dev, n, P.hkv, P.d).data_ptr() : nullptr;
  const float scale = scale_of(a[7], P.d);
  const int32_t T = small(n), Q = small(hq);
  const Call c = call_on(a[10], P.dev, E.prefill_ws(T, int32_t(start), Q, P.hkv, P.d, P.bs));
  const at::Tensor out = output(a[8], P, n, hq, false);
  const int32_t* tab = static_cast<const int32_t*>(bt.data_ptr());
  void* o = out.data_ptr();
  const void* qp = q.data_ptr();
  const int rc = append ? launch(E.prefill_append, o, qp, P.p, P.pages, tab, small(mp), int32_t(start), T, nk, nv, Q,
                                 P.hkv, P.d, P.bs, scale, c.ws, c.bytes, c.stream)
                        : launch(E.prefill, o, qp, P.p, P.pages, tab, small(mp), int32_t(start), T, Q, P.hkv, P.d,
                                 P.bs, scale, c.ws, c.bytes, c.stream);
  launched(rc, append ? "ifn_paged_prefill_append" : "ifn_paged_prefill");
  return done(out, a[8]);
}

// prep_prefill(q, k, v, q_norm_weight, k_norm_weight, rope, kv_pool, block_table, query_start, layer, eps, scale, out,
//              block_size, workspaces)
PyObject* prep_prefill(PyObject* const* a) {
  const Pool P = pool(a[6], integer(a[9]));
  need(integer(a[13]) == P.bs);
  const at::Tensor& q = tensor(a[0], at::kFloat, P.dev);
  need(q.dim() == 3 && q.size(2) == P.d && q.size(1) % P.hkv == 0 && q.size(0) >= 1 && q.size(1) >= 1);
  const int64_t n = q.size(0), hq = q.size(1), start = integer(a[8]);
  const float* k = f32(a[1], P.dev, n, P.hkv, P.d);
  const float* v = f32(a[2], P.dev, n, P.hkv, P.d);
  const float* qw = f32(a[3], P.dev, P.d);
  const float* kw = f32(a[4], P.dev, P.d);
  const at::Tensor& rope = tensor(a[5], at::kFloat, P.dev);
  need(rope.dim() == 2 && rope.size(1) == P.d);
  int64_t mp;
  const at::Tensor& bt = table_of(a[7], P.dev, mp);
  need(start >= 0 && start % 32 == 0 && start + n <= mp * P.bs && start + n <= rope.size(0));
  const float eps = eps_of(a[10]), scale = scale_of(a[11], P.d);
  const int32_t T = small(n), Q = small(hq);
  const Call c = call_on(a[14], P.dev, E.prefill_ws(T, int32_t(start), Q, P.hkv, P.d, P.bs));
  const at::Tensor out = output(a[12], P, n, hq, false);
  const int rc = launch(E.prep_prefill, out.data_ptr(), static_cast<const float*>(q.data_ptr()), k, v, qw, kw,
                        static_cast<const float*>(rope.data_ptr()), small(rope.size(0)), P.p, P.pages,
                        static_cast<const int32_t*>(bt.data_ptr()), small(mp), int32_t(start), T, Q, P.hkv, P.d,
                        P.bs, eps, scale, c.ws, c.bytes, c.stream);
  launched(rc, "ifn_paged_prefill_prep_append");
  return done(out, a[12]);
}

// prep_append(q, k, v, q_norm_weight, k_norm_weight, rope, positions, slot_mapping, active_mask, kv_pool, layer, eps,
//             q_out)
PyObject* prep_append(PyObject* const* a) {
  const Pool P = pool(a[9], integer(a[10]));
  const at::Tensor& q = tensor(a[0], at::kFloat, P.dev);
  need(q.dim() == 3 && q.size(2) == P.d && q.size(1) % P.hkv == 0 && q.size(0) >= 1 && q.size(1) >= 1);
  const int64_t n = q.size(0), hq = q.size(1);
  const float* k = f32(a[1], P.dev, n, P.hkv, P.d);
  const float* v = f32(a[2], P.dev, n, P.hkv, P.d);
  const float* qw = f32(a[3], P.dev, P.d);
  const float* kw = f32(a[4], P.dev, P.d);
  const at::Tensor& rope = tensor(a[5], at::kFloat, P.dev);
  need(rope.dim() == 2 && rope.size(1) == P.d);
  const int32_t* pos = i32(a[6], P.dev, n);
  const int32_t* slots = i32(a[7], P.dev, n);
  const uint8_t* act = mask(a[8], P.dev, n);
  const float eps = eps_of(a[11]);
  const at::Tensor out = output(a[12], P, n, hq, false);
  const int rc = launch(E.prep_append, out.data_ptr(), static_cast<const float*>(q.data_ptr()), k, v, qw, kw,
                        static_cast<const float*>(rope.data_ptr()), small(rope.size(0)), pos, slots, act, P.p,
                        P.pages, small(n), small(hq), P.hkv, P.d, P.bs, eps, stream_of(P.dev));
  launched(rc, "ifn_qk_norm_rope_append");
  return done(out, a[12]);
}

// store(kv_pool, slot_mapping, active_mask, new_k, new_v, layer)
PyObject* store(PyObject* const* a) {
  const Pool P = pool(a[0], integer(a[5]));
  const at::Tensor& k = tensor(a[3], at::kHalf, P.dev);
  need(k.dim() == 3 && k.size(0) >= 1);
  const int64_t n = k.size(0);
  shaped(a[3], at::kHalf, P.dev, n, P.hkv, P.d);
  const at::Tensor& v = shaped(a[4], at::kHalf, P.dev, n, P.hkv, P.d);
  launched(launch(E.store_kv, P.p, P.pages, i32(a[1], P.dev, n), mask(a[2], P.dev, n), k.data_ptr(), v.data_ptr(),
                  small(n), P.hkv, P.d, P.bs, stream_of(P.dev)), "ifn_store_kv");
  Py_RETURN_TRUE;
}

// store_layers(kv_pool, slot_mapping, active_mask, new_k, new_v)
PyObject* store_layers(PyObject* const* a) {
  const Pool P = pool(a[0], 0);
  const at::Tensor& k = tensor(a[3], at::kHalf, P.dev);
  need(THPVariable_Unpack(a[0]).dim() == 6 && k.dim() == 4 && k.size(1) >= 1);
  const int64_t n = k.size(1);
  shaped(a[3], at::kHalf, P.dev, P.layers, n, P.hkv, P.d);
  const at::Tensor& v = shaped(a[4], at::kHalf, P.dev, P.layers, n, P.hkv, P.d);
  launched(launch(E.store_kv_layers, P.p, small(P.layers), P.pages, i32(a[1], P.dev, n), mask(a[2], P.dev, n),
                  k.data_ptr(), v.data_ptr(), small(n), P.hkv, P.d, P.bs, stream_of(P.dev)), "ifn_store_kv_layers");
  Py_RETURN_TRUE;
}

// A call of N arguments: None when it is not one for this path (no C++ exception leaves it).
template <PyObject* (*F)(PyObject* const*), Py_ssize_t N>
PyObject* guarded(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n == N && bound && !at::impl::torch_function_mode_enabled() &&
      c10::impl::TorchDispatchModeTLS::stack_len() == 0) {
    try {
      PyObject* r = F(args);
      if (r != nullptr) return r;
    } catch (const Raised&) {
      return nullptr;
    } catch (...) {
    }
    PyErr_Clear();
  }
  Py_RETURN_NONE;
}

// The entry points' names and argument kinds in ctypes' letters, as compiled here.
template <class T>
constexpr char kind() {
  if constexpr (std::is_pointer_v<T>) return 'P';
  else if constexpr (std::is_same_v<T, float>) return 'f';
  else if constexpr (std::is_same_v<T, size_t>) return 'L';
  else if constexpr (std::is_same_v<T, int64_t>) return 'l';
  else {
    static_assert(std::is_same_v<T, int32_t>);
    return 'i';
  }
}
template <class R, class... A>
std::string signature(R (*)(A...)) {
  return {kind<R>(), kind<A>()...};
}
std::string signatures() {
  std::string all;
#define IFN_SIGNATURE(name, fn) all += std::string(#fn ":") + signature(decltype(&fn){}) + ",";
  IFN_ENTRIES(IFN_SIGNATURE)
#undef IFN_SIGNATURE
  return all;
}

// bind(signatures, *addresses): the entry points' addresses, in the order of Entries.  The signatures are those
// the library was opened with; an extension compiled for others is not bound.
PyObject* bind(PyObject*, PyObject* args) {
  constexpr Py_ssize_t n = sizeof(Entries) / sizeof(void*);
  const char* given = PyTuple_GET_SIZE(args) > 0 ? PyUnicode_AsUTF8(PyTuple_GET_ITEM(args, 0)) : nullptr;
  if (given == nullptr || PyTuple_GET_SIZE(args) != n + 1) {
    PyErr_SetString(PyExc_TypeError, "bind: the signatures and the entry points' addresses");
    return nullptr;
  }
  if (signatures() != given) {
    PyErr_SetString(PyExc_ImportError, "_fast_call was built for other entry points than the library's: rebuild it");
    return nullptr;
  }
  Entries e{};
  void** at = reinterpret_cast<void**>(&e);
  for (Py_ssize_t i = 0; i < n; ++i) {
    at[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(args, i + 1));
    if (at[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null entry point");
      return nullptr;
    }
  }
  E = e;
  bound = true;
  Py_RETURN_NONE;
}

#define IFN_FAST(NAME, N) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<NAME, N>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    IFN_FAST(decode, 16), IFN_FAST(prep_decode, 20), IFN_FAST(prefill, 11), IFN_FAST(prep_prefill, 15),
    IFN_FAST(prep_append, 13), IFN_FAST(store, 6), IFN_FAST(store_layers, 5),
    {"bind", bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast_call() {
  s_buf = PyUnicode_InternFromString("buf");
  s_nbytes = PyUnicode_InternFromString("nbytes");
  s_pending = PyUnicode_InternFromString("pending");
  s_key = PyUnicode_InternFromString("key");
  s_slots = PyUnicode_InternFromString("slots");
  for (PyObject* s : {s_buf, s_nbytes, s_pending, s_key, s_slots})
    if (s == nullptr) return nullptr;
  return PyModule_Create(&module);
}
